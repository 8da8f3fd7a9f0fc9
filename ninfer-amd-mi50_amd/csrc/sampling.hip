// Sampling on the device, one block per row of logits.
//
// Order of operations as in the reference's CPU sampler
// (src/runtime/engine.cpp:18-82): repetition penalty -> greedy if
// temperature <= 0 -> / temperature -> top-k -> softmax -> top-p -> draw.
// Differences, all deliberate: the penalty arrives as (token, count) pairs
// (a token seen c times is penalised c times, as the reference's loop over
// the history does); top-k and top-p are found by radix selection on the
// ordered bit pattern of the scaled logits instead of a sort, and of the tokens
// tied at the threshold the first ones in index order are kept, so the kept set
// is the prefix a stable sort by descending logit would give (top_k = 1 is the
// greedy choice, ties included); probabilities are held as 32.32 fixed-point
// integers so every sum is exact and the draw does not depend on the order of
// additions; the draw walks the kept tokens in index order with a uniform
// number `u` in [0,1) that the caller derives from (seed, request, draw
// index), so it does not depend on what else is in the batch. top_k <= 0
// keeps all tokens (the reference clamps to >= 1).
#include "common.h"
#include <type_traits>

namespace ninfer {

constexpr int kSampleThreads = 1024;
constexpr int kBatch = 8;   // logits that a thread loads before it uses the first
// Tokens of a row whose draw is one step, as the first of two costs more than it saves: 64 rows of 9,000 tokens
// 19.3 us in two, 17.6 in one; 14,000 tokens 21.7 in two (23.4 where one step took every row).
constexpr int kShortRow = 12288;

__device__ __forceinline__ uint32_t ordered_key(float v) {
  uint32_t b = __float_as_uint(v);
  if (b == 0x80000000u) b = 0;   // -0 and +0 are one value, as in a comparison of floats
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);  // ascending with the float order
}

// Probability of a token as 32.32 fixed point, from its scaled logit as the key has it, rounded (tokens of equal
// key have equal mass, the same in every pass and kernel); m: the largest of the row.
__device__ __forceinline__ unsigned long long token_mass(float scaled, float m) {
#pragma clang fp contract(off)   // both are products, which must not go unrounded into the difference
  return (unsigned long long)(expf(scaled - m) * 4294967296.f);
}

// Copies of the histogram that a radix pass adds into, lane by lane: the keys of logits share few
// upper bytes, and atomics of a wave's lanes on one address follow each other.
template <int COPIES>
struct RadixHist {
  unsigned long long bin[COPIES][257];   // (257: the copies of a bin lie in different banks)
  unsigned long long above;
  uint32_t chosen;
};

// Largest key t such that the sum of weight(i) over kept i with key(i) >= t
// reaches `target`. 4 passes of an 8-bit histogram; the first wave sums the bins from the
// top, four to a lane.
template <int COPIES, typename KeyFn, typename WeightFn>
__device__ uint32_t radix_select(int V, unsigned long long target, RadixHist<COPIES>& hist, KeyFn key,
                                 WeightFn weight) {
  uint32_t prefix = 0, mask = 0;
  const int copy = threadIdx.x % COPIES;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = threadIdx.x; b < COPIES * 257; b += blockDim.x) (&hist.bin[0][0])[b] = 0;
    __syncthreads();
    for (int i0 = threadIdx.x; i0 < V; i0 += kBatch * blockDim.x) {
      uint32_t k[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) k[u] = key(min(i0 + u * (int)blockDim.x, V - 1));
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int i = i0 + u * blockDim.x;
        if (i < V && (k[u] & mask) == prefix) {
          unsigned long long w = weight(i, k[u]);
          if (w) atomicAdd(&hist.bin[copy][(k[u] >> shift) & 255], w);
        }
      }
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      const int lane = threadIdx.x, top = 255 - 4 * lane;   // this lane's bins: top .. top - 3
      unsigned long long bin[4], mine = 0;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        bin[x] = 0;
#pragma unroll
        for (int c = 0; c < COPIES; ++c) bin[x] += hist.bin[c][top - x];
        mine += bin[x];
      }
      unsigned long long incl = mine;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
      }
      // the first lane whose bins reach the target (the last one if none does: the lowest bin)
      const unsigned long long hit = __ballot(incl >= target);
      const int first = hit ? __ffsll(hit) - 1 : 63;
      if (lane == first) {
        unsigned long long run = incl - mine;
        int x = 0;
        for (; x < 3; ++x) {
          if (run + bin[x] >= target) break;
          run += bin[x];
        }
        hist.chosen = (uint32_t)(top - x);
        hist.above = run;   // mass above the chosen bin no longer counts towards the target
      }
    }
    __syncthreads();
    target -= hist.above;
    prefix |= hist.chosen << shift;
    mask |= 255u << shift;
    __syncthreads();
  }
  return prefix;
}

// What a call asks of its rows.
struct SampleArgs {
  const float* logits;   // [R, ld]
  const float* temperature;
  const int* top_k;      // or null, as the next two
  const float* top_p;
  const float* rep_penalty;
  const int* pen_tokens;
  const int* pen_counts;
  const int* pen_offsets;
  const float* uniform;
  int* out;
  float* work;           // [R, V]
  int ld, V;
};

struct RowLds {
  RadixHist<8> hist;
  unsigned long long sums[2 * kSampleThreads / 64];
  float fred[kSampleThreads / 64];
  int ired[kSampleThreads / 64];
};

__device__ __forceinline__ bool row_penalised(const SampleArgs& a, int r, float& rp) {
  rp = a.rep_penalty ? a.rep_penalty[r] : 1.f;
  return rp != 1.f && a.pen_offsets && a.pen_offsets[r + 1] > a.pen_offsets[r];
}
__device__ __forceinline__ float penalise(float v, float rp, int count) {
  for (int c = 0; c < count; ++c) v = v > 0.f ? v / rp : v * rp;
  return v;
}

// Row r by one block of kSampleThreads, every option and size.
__device__ __forceinline__ void sample_whole_row(const SampleArgs& a, int r, RowLds& lds) {
  RadixHist<8>& hist = lds.hist;
  unsigned long long (&sums)[2 * kSampleThreads / 64] = lds.sums;
  float (&fred)[kSampleThreads / 64] = lds.fred;
  int (&ired)[kSampleThreads / 64] = lds.ired;
  const int* pen_tokens = a.pen_tokens;
  const int* pen_counts = a.pen_counts;
  const int* pen_offsets = a.pen_offsets;
  const int* top_k = a.top_k;
  const float* top_p = a.top_p;
  const float* uniform = a.uniform;
  int* out = a.out;
  const int V = a.V, tid = threadIdx.x;
  const float* row = a.logits + (int64_t)r * a.ld;
  float* w = a.work + (int64_t)r * V;
  const float temp = a.temperature[r];

  // repetition penalty on a copy of the row (greedy rows without a penalty read the row itself)
  float rp;
  const bool penalised = row_penalised(a, r, rp);
  if (!(temp > 0.f) && !penalised) {
    w = const_cast<float*>(row);
  } else {
    for (int i0 = tid; i0 < V; i0 += kBatch * kSampleThreads) {
      float x[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) x[u] = i0 + u * kSampleThreads < V ? row[i0 + u * kSampleThreads] : 0.f;
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (i0 + u * kSampleThreads < V) w[i0 + u * kSampleThreads] = x[u];
    }
  }
  __syncthreads();
  if (penalised) {
    for (int e = pen_offsets[r] + tid; e < pen_offsets[r + 1]; e += blockDim.x) {
      int tok = pen_tokens[e];
      if (tok < 0 || tok >= V) continue;
      w[tok] = penalise(w[tok], rp, pen_counts[e]);
    }
  }
  __syncthreads();

  // max and argmax (ties: lowest index). A greedy row does nothing else: two batches of loads at a time,
  // none for tokens that are not there (151,936 tokens, us for 8 and 64 rows: four loads at a time 16.6 and
  // 34.7, sixteen 16.6 and 20.1 with the last batch's loads clamped, 11.2 and 13.1 so).
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  auto look = [&](int i0, auto loads, auto whole) {
    constexpr int N = decltype(loads)::value;
    float v[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = i0 + u * kSampleThreads;
      v[u] = decltype(whole)::value || i < V ? w[i] : -INFINITY;
    }
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (v[u] > best) {
        best = v[u];
        best_i = i0 + u * kSampleThreads;
      }
  };
  typedef std::integral_constant<int, 2 * kBatch> Many;
  typedef std::integral_constant<int, 4> Few;   // (what is left of a row, or a short row, with no steps for nothing)
  constexpr int kLook = Many::value * kSampleThreads;
  for (int i = 0; i < V / kLook; ++i) look(tid + i * kLook, Many{}, std::true_type{});
  if (V % kLook > Few::value * kSampleThreads) look(tid + V / kLook * kLook, Many{}, std::false_type{});
  else if (V % kLook) look(tid + V / kLook * kLook, Few{}, std::false_type{});
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    float ob = __shfl_xor(best, off, 64);
    int oi = __shfl_xor(best_i, off, 64);
    if (ob > best || (ob == best && oi < best_i)) {
      best = ob;
      best_i = oi;
    }
  }
  if ((tid & 63) == 0) {
    fred[tid >> 6] = best;
    ired[tid >> 6] = best_i;
  }
  __syncthreads();
  best = fred[0];
  best_i = ired[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) {
    if (fred[i] > best || (fred[i] == best && ired[i] < best_i)) {
      best = fred[i];
      best_i = ired[i];
    }
  }
  if (best_i == 0x7fffffff) best_i = 0;   // (nothing above -infinity: the first token, as where few tokens are kept)
  if (!(temp > 0.f)) {
    if (tid == 0) out[r] = best_i;
    return;
  }
  __syncthreads();

  const float inv_t = 1.f / temp;
  const float m = best * inv_t;  // max of the scaled logits (temp > 0)
  typedef unsigned long long u64;
  auto key_of = [&](float x) { return ordered_key(x * inv_t); };
  auto key = [&](int i) { return key_of(w[i]); };
  auto mass_of = [&](float x) -> u64 { return token_mass(x * inv_t, m); };
  auto mass_at = [&](uint32_t kk) -> u64 {
    const uint32_t bits = (kk & 0x80000000u) ? (kk & 0x7fffffffu) : ~kk;   // ordered_key's inverse
    return token_mass(__uint_as_float(bits), m);
  };
  // use(x) for the numbers at first, first + step, .. below end: whole batches without a condition, then the rest,
  // with no load and no exponential for numbers that are not there (1,000 tokens, nothing cut off: 17 us with
  // them, 10.8 so; 64 rows of 151,936 146 with a condition on every number, 112 so)
  auto each = [&](int first, int step, int end, auto use) {
    int i0 = first;
    float x[kBatch];
    for (; i0 + (kBatch - 1) * step < end; i0 += kBatch * step) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) x[u] = w[i0 + u * step];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) use(x[u]);
    }
    if (i0 >= end) return;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) x[u] = i0 + u * step < end ? w[i0 + u * step] : 0.f;
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (i0 + u * step < end) use(x[u]);
  };
  auto block_sum = [&](u64 v) -> u64 {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((tid & 63) == 0) sums[tid >> 6] = v;
    __syncthreads();
    u64 t = 0;
    for (int i = 0; i < kSampleThreads / 64; ++i) t += sums[i];
    __syncthreads();
    return t;
  };
  // tokens with a key above t (their count and mass) and with key t (their count)
  auto stats = [&](uint32_t t, u64& cnt_gt, u64& mass_gt, u64& cnt_eq) {
    u64 c = 0, ms = 0, e = 0;
    each(tid, kSampleThreads, V, [&](float x) {
      const uint32_t kk = key_of(x);
      c += kk > t;
      e += kk == t;
      if (kk > t) ms += mass_of(x);
    });
    cnt_gt = block_sum(c);
    mass_gt = block_sum(ms);
    cnt_eq = block_sum(e);
  };

  // The kept set is a prefix of the tokens ordered by (logit descending, index ascending),
  // as a sort would give it: every token with a key above `thr`, and of the tokens with key
  // `thr` the first `quota` in index order. Keeping all is thr = 0 with no token at it.
  uint32_t thr = 0;
  u64 cnt_gt, mass_gt, cnt_eq;
  const int k = top_k ? top_k[r] : 0;
  if (k > 0 && k < V)   // top-k: the k-th largest key
    thr = radix_select(V, (u64)k, hist, key, [](int, uint32_t) { return 1ull; });
  stats(thr, cnt_gt, mass_gt, cnt_eq);
  u64 quota = (k > 0 && k < V) ? (u64)k - cnt_gt : cnt_eq;   // 1 .. cnt_eq with top-k
  u64 mass_thr = mass_at(thr);
  u64 total = mass_gt + quota * mass_thr;

  // top-p: the shortest prefix of that order whose mass reaches top_p of the total
  const float pp = top_p ? top_p[r] : 1.f;
  if (pp < 1.f) {
    u64 target = (u64)((double)pp * (double)total);
    if (target < 1) target = 1;
    if (target <= mass_gt) {   // it ends among the keys above thr
      const uint32_t floor_key = thr;
      thr = radix_select(V, target, hist, key, [&](int i, uint32_t kk) -> u64 {
        return kk > floor_key ? mass_of(w[i]) : 0ull;
      });
      stats(thr, cnt_gt, mass_gt, cnt_eq);
      mass_thr = mass_at(thr);
      quota = cnt_eq;
    }
    // mass_gt < target <= mass_gt + quota * mass_thr
    if (mass_thr > 0) {
      const u64 need = (target - mass_gt + mass_thr - 1) / mass_thr;
      if (need < quota) quota = need;
    }
    total = mass_gt + quota * mass_thr;
  }

  if (total == 0) {   // no token has mass (+infinity is the largest logit, or -infinity, or all are NaN): the largest
    if (tid == 0) out[r] = best_i;
    return;
  }

  // Inverse CDF over the kept tokens in index order, in two steps. First every wave sums a run of
  // V / 16 tokens, 64 neighbours at a time; then the run that holds the goal is dealt to all
  // threads, a few neighbours each (short rows: the whole row at once).
  u64 goal = (u64)((double)uniform[r] * (double)total);
  if (goal >= total) goal = total - 1;
  constexpr int kWaves = kSampleThreads / 64;
  const int lane = tid & 63, wv = tid >> 6;
  const int per_wave = (V + kWaves - 1) / kWaves;
  u64 run = 0, eq_before = 0;   // mass and ties before the run
  int r0 = 0, r1 = V;
  if (V > kShortRow) {
    u64 gt_mass = 0, eq_count = 0;
    each(min(V, wv * per_wave) + lane, 64, min(V, (wv + 1) * per_wave), [&](float x) {
      const uint32_t kk = key_of(x);
      eq_count += kk == thr;
      if (kk > thr) gt_mass += mass_of(x);
    });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      gt_mass += __shfl_xor(gt_mass, off, 64);
      eq_count += __shfl_xor(eq_count, off, 64);
    }
    if (lane == 0) {
      sums[wv] = gt_mass;
      sums[kWaves + wv] = eq_count;
    }
    __syncthreads();
    // of the tokens tied at the threshold the first `quota` are kept: a run keeps what is left of it
    int at = 0;
    for (; at < kWaves; ++at) {
      const u64 left = eq_before < quota ? quota - eq_before : 0;
      const u64 mass = sums[at] + (sums[kWaves + at] < left ? sums[kWaves + at] : left) * mass_thr;
      if (goal < run + mass || at == kWaves - 1) break;
      run += mass;
      eq_before += sums[kWaves + at];
    }
    __syncthreads();
    r0 = min(V, at * per_wave);
    r1 = min(V, r0 + per_wave);
  }
  const int chunk = (r1 - r0 + kSampleThreads - 1) / kSampleThreads;
  const int c0 = min(r1, r0 + tid * chunk), c1 = min(r1, c0 + chunk);
  auto scan = [&](u64 mine) -> u64 {   // sum over the threads before this one
    u64 incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const u64 o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) sums[wv] = incl;
    __syncthreads();
    u64 base = 0;
    for (int i = 0; i < wv; ++i) base += sums[i];   // at most 15 wave totals
    __syncthreads();
    return base + incl - mine;
  };
  u64 rank0 = eq_before;   // ties before this thread's tokens (wanted only when not all are kept)
  if (quota < cnt_eq) {
    u64 eq_mine = 0;
    for (int i = c0; i < c1; ++i) eq_mine += key(i) == thr;
    rank0 += scan(eq_mine);
  }
  auto walk = [&](u64 start, bool pick_it) -> u64 {   // mass of the tokens; or the token at `goal`
    u64 run = start, rank = rank0;
    for (int i = c0; i < c1; ++i) {
      const uint32_t kk = key(i);
      u64 ms = 0;
      if (kk > thr) ms = mass_of(w[i]);
      else if (kk == thr && rank++ < quota) ms = mass_thr;
      if (pick_it && ms && goal < run + ms) return (u64)i;
      run += ms;
    }
    return pick_it ? (u64)(c1 - 1) : run - start;
  };
  const u64 mine = walk(0, false);
  const u64 before = run + scan(mine);
  if (mine > 0 && goal >= before && goal < before + mine) out[r] = (int)walk(before, true);
}

__global__ __launch_bounds__(kSampleThreads) void sample_kernel(SampleArgs a) {
  __shared__ RowLds lds;
  sample_whole_row(a, blockIdx.x, lds);
}

// The same by the whole GPU, for rows that are greedy, keep at most kFewTokens tokens (top-k) or
// cut nothing by top-k: the same kept set, masses and token. A row is cut into slices of kSlice
// tokens, one block each.
//
// Few tokens kept, two launches. The slices' blocks apply the penalty and leave the largest key of
// every thread's 16 tokens (sample_maxima_kernel). A block per row then finds a bound that at least
// k tokens reach, from the largest keys of its own threads: the k-th largest of them. Hardly more than k
// threads' keys of the first launch reach it; their tokens alone are read again, and those that reach the bound are ranked
// among themselves, each by a thread that compares it with all others (sample_draw_kernel).
// Bound by the one read of the logits and two chains of loads: 64 rows of 151,936 tokens with top-k 50 13 + 18 us (with
// the k best of every slice found by its block, and the row's among those, 36 + 21); with top-k 200 35 in all, by
// sample_whole_row 341; one row 15 and 23.
//
// Nothing cut by top-k, four launches: between the two, the slices' blocks add their tokens' masses into a
// histogram of the row over the distance to its largest logit (sample_masses_kernel), then every
// block finds in it the bin in which top-p cuts, sums its slice's mass above and lists its tokens of that bin
// (sample_cut_kernel). The row's block finds the cut among the listed ones, the slice that holds the draw, and
// the token in it. 64 rows of 151,936 tokens at top-p 0.95 73 to 84 us, by sample_whole_row 320; one row 30 and
// 267; 32,000 tokens, one row, 30 and 74, with top-p 1 23 and 33; 6,000 tokens the same in both.
//
// Rows that fit neither, lists that do not fit (many equal logits; 151,936 normal ones of a deviation below some 0.2 once scaled)
// and rows with NaN or +infinity go through sample_whole_row: 64 that are too flat 420 us, 389 without the launches in front.
constexpr int kSlice = 4096;
constexpr int kSliceThreads = 256;
constexpr int kPerThread = kSlice / kSliceThreads;   // tokens of a subgroup: tid + kSliceThreads * u
constexpr int kFewTokens = 256;
constexpr int kSubs = 512;          // subgroups that a row's block reads again
constexpr int kSubTable = 2048;     // places to look one of them up
constexpr int kFewList = 1024;      // tokens that reach the bound
constexpr int kBins = 512;          // (450 that tokens fall into: beyond a distance of 22.2 they have no mass)
constexpr int kCutList = 4096;      // tokens of the bin that top-p cuts
constexpr int kMaxSlices = 1024;    // of a row whose draw may keep all
constexpr int kSpreadRows = 65535;  // a grid's second dimension

struct SampleScratch {
  uint32_t* maxima;             // [R, slices * kSliceThreads]
  uint32_t* slice_max;          // [R, slices]
  int* listed;                  // [R]: tokens in the row's list
  uint2* list;                  // [R, kCutList]: key, token
  unsigned long long* bins;     // [R, kBins]: masses
  unsigned long long* slice_mass;   // [R, slices]: of the tokens above the cut's bin
  int slices;
  bool wide;                    // the launches between ran
};

enum RowKind : int { kRowFew, kRowWide, kRowOther };
__device__ __forceinline__ RowKind row_kind(const SampleArgs& a, const SampleScratch& s, int r) {
  const int k = a.top_k ? a.top_k[r] : 0;
  if (!(a.temperature[r] > 0.f) || (k >= 1 && k <= kFewTokens)) return kRowFew;
  return s.wide && (k <= 0 || k >= a.V) ? kRowWide : kRowOther;
}
__device__ __forceinline__ float row_inverse_temperature(const SampleArgs& a, int r) {
  const float t = a.temperature[r];
  return t > 0.f ? 1.f / t : 1.f;
}
__device__ __forceinline__ float key_value(uint32_t key) {   // ordered_key's inverse
  return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}
// Above this key, that of the largest finite number, lie +infinity and NaN.
constexpr uint32_t kFiniteKey = 0xff7fffffu;

// The same or more for every smaller scaled logit, and the same for equal ones: `scaled` is a product, which must not go
// unrounded into the difference (token_mass). 128 bins for each doubling of the distance + 2 (its float's upper bits): 64 to a
// unit up to 2, 32 up to 6, 16 up to 14, 8 beyond, as the flatter a row, the nearer to its largest logit, and the more crowded, is
// where top-p cuts it. With 16 to a unit everywhere the cut's bin of 151,936 normal logits of deviation 0.6 (top-p 0.8) held 4,400
// tokens, more than the list: 64 such rows 420 us, 124 so.
__device__ __forceinline__ int mass_bin(float scaled, float m) {
#pragma clang fp contract(off)
  return min(kBins - 1, (int)((__float_as_uint(m - scaled + 2.f) - __float_as_uint(2.f)) >> 16));
}

// Wave-wide inclusive sums.
__device__ __forceinline__ unsigned long long wave_sums(unsigned long long v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned long long o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

__global__ __launch_bounds__(kSliceThreads) void sample_maxima_kernel(SampleArgs a, SampleScratch s) {
  __shared__ float vals[kSlice];
  __shared__ uint32_t wave_max[kSliceThreads / 64];
  const int r = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  const int s0 = b * kSlice, n = min(kSlice, a.V - s0);
  const float* row = a.logits + (int64_t)r * a.ld + s0;
  float x[kPerThread];   // every load on its way at once
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) x[u] = row[min(tid + u * kSliceThreads, n - 1)];
  const RowKind kind = row_kind(a, s, r);
  if (kind == kRowOther) return;
  float rp;
  if (row_penalised(a, r, rp)) {
    const int first = a.pen_offsets[r], end = a.pen_offsets[r + 1];
    int pen[8];   // penalised tokens, eight at a time, the first beside the slice
    auto load_pens = [&](int e0) {
#pragma unroll
      for (int u = 0; u < 8; ++u) pen[u] = a.pen_tokens[min(e0 + u * kSliceThreads, end - 1)];
    };
    load_pens(first + tid);
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) vals[tid + u * kSliceThreads] = x[u];
    __syncthreads();
    for (int e0 = first + tid; e0 < end; e0 += 8 * kSliceThreads) {
      if (e0 != first + tid) load_pens(e0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + u * kSliceThreads, t = pen[u] - s0;
        if (e < end && t >= 0 && t < n) vals[t] = penalise(vals[t], rp, a.pen_counts[e]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) x[u] = vals[tid + u * kSliceThreads];
    if (kind == kRowWide) {
      float* w = a.work + (int64_t)r * a.V + s0;
#pragma unroll
      for (int u = 0; u < kPerThread; ++u)
        if (tid + u * kSliceThreads < n) w[tid + u * kSliceThreads] = x[u];
    }
  }
  const float inv_t = row_inverse_temperature(a, r);
  uint32_t best = 0;   // (below every number's key)
#pragma unroll
  for (int u = 0; u < kPerThread; ++u)
    if (tid + u * kSliceThreads < n) best = max(best, ordered_key(x[u] * inv_t));
  s.maxima[((int64_t)r * s.slices + b) * kSliceThreads + tid] = best;
  if (kind != kRowWide) return;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) best = max(best, (uint32_t)__shfl_xor((int)best, off, 64));
  if ((tid & 63) == 0) wave_max[tid >> 6] = best;
  // the row's bins and list start empty
  for (int i = b * kSliceThreads + tid; i < kBins; i += s.slices * kSliceThreads) s.bins[(int64_t)r * kBins + i] = 0;
  if (b == 0 && tid == 0) s.listed[r] = 0;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < kSliceThreads / 64; ++w) best = max(best, wave_max[w]);
    s.slice_max[(int64_t)r * s.slices + b] = best;
  }
}

// The largest key of a row, by every wave for itself.
__device__ __forceinline__ uint32_t row_max(const SampleScratch& s, int r) {
  uint32_t best = 0;
  for (int i = threadIdx.x & 63; i < s.slices; i += 64) best = max(best, s.slice_max[(int64_t)r * s.slices + i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) best = max(best, (uint32_t)__shfl_xor((int)best, off, 64));
  return best;
}

__device__ __forceinline__ const float* wide_row(const SampleArgs& a, int r) {
  float rp;
  return row_penalised(a, r, rp) ? a.work + (int64_t)r * a.V : a.logits + (int64_t)r * a.ld;
}

__global__ __launch_bounds__(kSliceThreads) void sample_masses_kernel(SampleArgs a, SampleScratch s) {
  __shared__ unsigned long long bins[kBins];
  const int r = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  if (row_kind(a, s, r) != kRowWide) return;
  const int s0 = b * kSlice, n = min(kSlice, a.V - s0);
  const float* row = wide_row(a, r) + s0;
  float x[kPerThread];
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) x[u] = row[min(tid + u * kSliceThreads, n - 1)];
  for (int i = tid; i < kBins; i += kSliceThreads) bins[i] = 0;
  const uint32_t most = row_max(s, r);
  if (most > kFiniteKey) return;
  const float m = key_value(most), inv_t = row_inverse_temperature(a, r);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const float scaled = x[u] * inv_t;
    const unsigned long long mass = token_mass(scaled, m);
    if (tid + u * kSliceThreads < n && mass) atomicAdd(&bins[mass_bin(scaled, m)], mass);
  }
  __syncthreads();
  for (int i = tid; i < kBins; i += kSliceThreads)
    if (bins[i]) atomicAdd(&s.bins[(int64_t)r * kBins + i], bins[i]);
}

// Where top-p cuts a row, by the first wave from its bins: the bin (kBins: nothing is cut), the mass of the bins
// above it, the mass that is to be kept, and of all.
struct Cut {
  int bin;
  unsigned long long above, target, total;
};
__device__ __forceinline__ void find_cut(const SampleArgs& a, const SampleScratch& s, int r, Cut& cut) {
  typedef unsigned long long u64;
  constexpr int EACH = kBins / 64;
  const int lane = threadIdx.x & 63;
  const u64* bins = s.bins + (int64_t)r * kBins + EACH * lane;
  u64 bin[EACH], mine = 0;
#pragma unroll
  for (int i = 0; i < EACH; ++i) bin[i] = bins[i];
#pragma unroll
  for (int i = 0; i < EACH; ++i) mine += bin[i];
  const u64 incl = wave_sums(mine), total = __shfl(incl, 63, 64);
  const float pp = a.top_p ? a.top_p[r] : 1.f;
  u64 target = (u64)((double)pp * (double)total);
  if (target < 1) target = 1;
  const u64 hit = __ballot(incl >= target);
  const bool cuts = pp < 1.f && hit;
  if (lane == (cuts ? __ffsll(hit) - 1 : 63)) {
    u64 run = incl - mine;
    int x = 0;
#pragma unroll
    for (int i = 0; i < EACH - 1; ++i)
      if (x == i && run + bin[i] < target) run += bin[i], ++x;
    cut.bin = cuts ? EACH * lane + x : kBins;
    cut.above = cuts ? run : total;
    cut.target = target;
    cut.total = total;
  }
}

__global__ __launch_bounds__(kSliceThreads) void sample_cut_kernel(SampleArgs a, SampleScratch s) {
  __shared__ Cut cut;
  __shared__ unsigned long long sums[kSliceThreads / 64];
  __shared__ uint2 list[kSlice];   // (its own first: one place in the row's list is asked for a block)
  __shared__ int listed, place;
  const int r = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  if (row_kind(a, s, r) != kRowWide) return;
  if (tid == 0) listed = 0;
  const int s0 = b * kSlice, n = min(kSlice, a.V - s0);
  const float* row = wide_row(a, r) + s0;
  float x[kPerThread];
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) x[u] = row[min(tid + u * kSliceThreads, n - 1)];
  const uint32_t most = row_max(s, r);
  if (most > kFiniteKey) return;
  const float m = key_value(most), inv_t = row_inverse_temperature(a, r);
  if (tid < 64) find_cut(a, s, r, cut);
  __syncthreads();
  const int cut_bin = cut.bin;
  unsigned long long above = 0;
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const float scaled = x[u] * inv_t;
    const unsigned long long mass = token_mass(scaled, m);
    if (tid + u * kSliceThreads >= n || !mass) continue;
    const int bin = mass_bin(scaled, m);
    if (bin < cut_bin) above += mass;
    else if (bin == cut_bin) list[atomicAdd(&listed, 1)] = make_uint2(ordered_key(scaled), s0 + tid + u * kSliceThreads);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) above += __shfl_xor(above, off, 64);
  if ((tid & 63) == 0) sums[tid >> 6] = above;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < kSliceThreads / 64; ++w) above += sums[w];
    s.slice_mass[(int64_t)r * s.slices + b] = above;
    place = listed ? atomicAdd(&s.listed[r], listed) : 0;
  }
  __syncthreads();
  for (int i = tid; i < listed && place + i < kCutList; i += kSliceThreads) s.list[(int64_t)r * kCutList + place + i] = list[i];
}

union DrawLds {
  RowLds row;
  struct {
    float vals[kSubs * kPerThread];
    unsigned long long tokens[kFewList + 8];   // key, then the token's complement: in the order by which tokens are kept
    unsigned kept[kFewList + 16];              // token of a kept one, else the largest number
    unsigned long long by_rank[kFewTokens], by_place[kFewTokens];   // masses
    int place_of[kFewTokens], token_at[kFewTokens];                 // of a rank; at a place
    int sub[kSubs];
    uint32_t place_of_sub[kSubTable];       // (subgroup + 1) * kSubs + its place in `sub`, hashed, or 0
    uint4 best[kSampleThreads / 4];
    int subs, listed;
    uint32_t bound, nan;
  } few;
  struct {
    uint2 list[kCutList];
    unsigned long long slice[kMaxSlices];
    RadixHist<1> hist;
    unsigned long long sums[kSampleThreads / 64];
    int ranks[kSampleThreads / 64];
    unsigned ties[kCutList];   // tokens with the threshold's key
    Cut cut;
    unsigned long long mass_gt, before;
    int cnt_eq, cnt_before, at;
  } wide;
};

// The largest bound of 20 bits that k of the block's threads' keys reach (0 if fewer are numbers); of 17 bits, which a few tokens
// more reach, beyond 64. Of up to 64 the keys of four threads count as one, their largest.
__device__ __forceinline__ void few_bound(uint32_t mine, int k, DrawLds& lds) {
  const int tid = threadIdx.x;
  auto& l = lds.few;
  if (k <= 64) {
    mine = max(mine, (uint32_t)__shfl_xor((int)mine, 1, 64));
    mine = max(mine, (uint32_t)__shfl_xor((int)mine, 2, 64));
    if (tid % 4 == 0) ((uint32_t*)l.best)[tid / 4] = mine;
  } else {
    ((uint32_t*)l.best)[tid] = mine;
  }
  __syncthreads();
  if (tid >= 64) return;
  uint32_t bound = 0;
  if (k <= 64) {
    const uint4 m = l.best[tid];
    for (int bit = 31; bit >= 12; --bit) {
      const uint32_t at = bound | (1u << bit);
      const int reach = __popcll(__ballot(m.x >= at)) + __popcll(__ballot(m.y >= at)) +
                        __popcll(__ballot(m.z >= at)) + __popcll(__ballot(m.w >= at));
      if (reach >= k) bound = at;
    }
  } else {
    uint4 m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = l.best[tid + 64 * i];
    for (int bit = 31; bit >= 15; --bit) {
      const uint32_t at = bound | (1u << bit);
      int reach = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        reach += __popcll(__ballot(m[i].x >= at)) + __popcll(__ballot(m[i].y >= at)) +
                 __popcll(__ballot(m[i].z >= at)) + __popcll(__ballot(m[i].w >= at));
      if (reach >= k) bound = at;
    }
  }
  if (tid == 0) l.bound = bound;
}

// A row that keeps few tokens; got: the first of the row's keys that are this thread's. False: through sample_whole_row.
constexpr int kLookKeys = 12;
__device__ __forceinline__ bool draw_few(const SampleArgs& a, const SampleScratch& s, int r, DrawLds& lds,
                                         const uint32_t (&got)[kLookKeys]) {
  constexpr int LOOK = kLookKeys;
  typedef unsigned long long u64;
  auto& l = lds.few;
  const int tid = threadIdx.x, lane = tid & 63;
  const int groups = s.slices * kSliceThreads;
  if (groups >= 1 << 22) return false;   // (their numbers share 32 bits with a place)
  const uint32_t* maxima = s.maxima + (int64_t)r * groups;
  const float temp = a.temperature[r], inv_t = row_inverse_temperature(a, r);
  const int k = min(temp > 0.f ? a.top_k[r] : 1, a.V);
  float rp;
  const bool penalised = row_penalised(a, r, rp);
  const int first = penalised ? a.pen_offsets[r] : 0, end = penalised ? a.pen_offsets[r + 1] : 0;
  constexpr int PENS = 2;   // of a thread, on their way beside the keys
  int pen[PENS];
#pragma unroll
  for (int u = 0; u < PENS; ++u) pen[u] = end > first ? a.pen_tokens[min(first + tid + u * kSampleThreads, end - 1)] : 0;

  uint32_t mine = 0;
#pragma unroll
  for (int u = 0; u < LOOK; ++u) mine = max(mine, got[u]);
  for (int g = tid + LOOK * kSampleThreads; g < groups; g += kSampleThreads) mine = max(mine, maxima[g]);
  for (int i = tid; i < kSubTable; i += kSampleThreads) l.place_of_sub[i] = 0;
  if (tid == 0) l.subs = l.listed = 0, l.nan = 0;
  few_bound(mine, k, lds);
  __syncthreads();
  const uint32_t bound = l.bound;
  auto slot_of = [](int g) { return (unsigned)g * 2654435761u >> 21; };
  static_assert(kSubTable == 1 << 11, "slot_of has 11 bits");
  auto take = [&](int g, uint32_t key) {   // (key 0: no token)
    if (key < bound || key == 0) return;
    const int at = atomicAdd(&l.subs, 1);
    if (at >= kSubs) return;
    l.sub[at] = g;
    // (a quarter of the places at most is taken: the search ends)
    for (unsigned h = slot_of(g); penalised && atomicCAS(&l.place_of_sub[h], 0u, (g + 1u) * kSubs + at); h = (h + 1) % kSubTable) {}
  };
  if (mine >= bound) {
#pragma unroll
    for (int u = 0; u < LOOK; ++u) take(tid + u * kSampleThreads, got[u]);
    for (int g = tid + LOOK * kSampleThreads; g < groups; g += kSampleThreads) take(g, maxima[g]);
  }
  __syncthreads();
  const int subs = l.subs;
  if (subs > kSubs) return false;
  const float* row = a.logits + (int64_t)r * a.ld;
  auto token_of = [&](int i) {   // of place i of `vals`
    const int g = l.sub[i / kPerThread];
    return g / kSliceThreads * kSlice + g % kSliceThreads + i % kPerThread * kSliceThreads;
  };
  for (int i = tid; i < subs * kPerThread; i += kSampleThreads) l.vals[i] = row[min(token_of(i), a.V - 1)];
  __syncthreads();
  if (penalised) {
    auto apply = [&](int e, int t) {
      if (e >= end || t < 0 || t >= a.V) return;
      const int g = t / kSlice * kSliceThreads + t % kSliceThreads;
      uint32_t found = 0;
      for (unsigned h = slot_of(g); (found = l.place_of_sub[h]) != 0 && found / kSubs != g + 1u; h = (h + 1) % kSubTable) {}
      if (!found) return;
      float& v = l.vals[found % kSubs * kPerThread + t % kSlice / kSliceThreads];
      v = penalise(v, rp, a.pen_counts[e]);
    };
#pragma unroll
    for (int u = 0; u < PENS; ++u) apply(first + tid + u * kSampleThreads, pen[u]);
    for (int e = first + tid + PENS * kSampleThreads; e < end; e += kSampleThreads) apply(e, a.pen_tokens[e]);
    __syncthreads();
  }
  for (int i = tid; i < subs * kPerThread; i += kSampleThreads) {
    const int t = token_of(i);
    const uint32_t key = ordered_key(l.vals[i] * inv_t);
    if (t >= a.V || key < bound) continue;
    if (key > kFiniteKey) l.nan = 1;
    const int at = atomicAdd(&l.listed, 1);
    if (at < kFewList) l.tokens[at] = (u64)key << 32 | (0xffffffffu - (unsigned)t);
  }
  __syncthreads();
  const int count = l.listed;
  if (count > kFewList || l.nan || count < k) return false;
  if (tid < 16) {   // places that nothing follows and nothing counts
    if (tid < 8) l.tokens[count + tid] = 0;
    l.kept[count + tid] = 0xffffffffu;
  }
  __syncthreads();
  // Four threads a token: how many come before it, of every fourth pair of them each.
  const int part = tid & 3;
  auto before = [&](int mine) {
    mine += __shfl_xor(mine, 1, 64);
    return mine + __shfl_xor(mine, 2, 64);
  };
  const int rounds = (count + kSampleThreads / 4 - 1) / (kSampleThreads / 4);
  int rank[kFewList / (kSampleThreads / 4)];
#pragma unroll
  for (int i = 0; i < kFewList / (kSampleThreads / 4); ++i) {
    rank[i] = k;
    const int e = tid / 4 + i * (kSampleThreads / 4);
    if (i >= rounds || e >= count) continue;
    const u64 mine = l.tokens[e];
    int n = 0;
#pragma unroll 4
    for (int j = 2 * part; j < count; j += 8) n += (l.tokens[j] > mine) + (l.tokens[j + 1] > mine);
    rank[i] = before(n);
    if (part) continue;
    const unsigned token = 0xffffffffu - (unsigned)mine;
    if (rank[i] == 0 && !(temp > 0.f)) a.out[r] = (int)token;
    l.kept[e] = rank[i] < k ? token : 0xffffffffu;
    if (rank[i] < k) l.by_rank[rank[i]] = mine >> 32;   // (its key)
  }
  if (!(temp > 0.f)) return true;
  __syncthreads();
  const float m = key_value((uint32_t)l.by_rank[0]);   // the largest scaled logit
#pragma unroll
  for (int i = 0; i < kFewList / (kSampleThreads / 4); ++i) {
    const int e = tid / 4 + i * (kSampleThreads / 4);
    if (i >= rounds || rank[i] >= k) continue;
    const unsigned mine = l.kept[e];
    int n = 0;
#pragma unroll 4
    for (int j = 4 * part; j < count; j += 16)
      n += (l.kept[j] < mine) + (l.kept[j + 1] < mine) + (l.kept[j + 2] < mine) + (l.kept[j + 3] < mine);
    const int place = before(n);
    if (part) continue;
    l.place_of[rank[i]] = place;
    l.token_at[place] = (int)mine;
  }
  __syncthreads();
  if (tid >= 64) return true;
  // One wave: masses by rank, of which those before the target are kept, then by place, where the draw is.
  constexpr int EACH = kFewTokens / 64;
  u64 here[EACH], sum = 0;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int at = EACH * lane + i;
    here[i] = at < k ? token_mass(key_value((uint32_t)l.by_rank[at]), m) : 0;
    sum += here[i];
  }
  u64 incl = wave_sums(sum);
  u64 total = __shfl(incl, 63, 64);
  const float pp = a.top_p ? a.top_p[r] : 1.f;
  u64 target = total;
  if (pp < 1.f) {
    target = (u64)((double)pp * (double)total);
    if (target < 1) target = 1;
  }
  u64 run = incl - sum;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    if (EACH * lane + i < k) l.by_place[l.place_of[EACH * lane + i]] = run < target ? here[i] : 0;
    run += here[i];
  }
  // (one wave: its LDS accesses run in order, and the fence keeps the compiler from changing that)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  sum = 0;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    here[i] = EACH * lane + i < k ? l.by_place[EACH * lane + i] : 0;
    sum += here[i];
  }
  incl = wave_sums(sum);
  total = __shfl(incl, 63, 64);
  if (total == 0 && lane == 0) a.out[r] = l.token_at[l.place_of[0]];   // (all that is kept is -infinity)
  u64 goal = (u64)((double)a.uniform[r] * (double)total);
  if (goal >= total) goal = total - 1;
  run = incl - sum;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    if (here[i] > 0 && goal >= run && goal < run + here[i]) a.out[r] = l.token_at[EACH * lane + i];
    run += here[i];
  }
  return true;
}

// A row of which top-k cuts nothing. False: through sample_whole_row.
__device__ __forceinline__ bool draw_wide(const SampleArgs& a, const SampleScratch& s, int r, DrawLds& lds) {
  typedef unsigned long long u64;
  auto& l = lds.wide;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t most = row_max(s, r);
  if (most > kFiniteKey) return false;
  const float m = key_value(most), inv_t = row_inverse_temperature(a, r);
  const int n = s.listed[r];
  if (n > kCutList) return false;
  if (wv == 0) find_cut(a, s, r, l.cut);
  for (int i = tid; i < n; i += kSampleThreads) l.list[i] = s.list[(int64_t)r * kCutList + i];
  for (int i = tid; i < s.slices; i += kSampleThreads) l.slice[i] = s.slice_mass[(int64_t)r * s.slices + i];
  if (tid == 0) l.mass_gt = 0, l.cnt_eq = 0;
  __syncthreads();
  // Kept are the tokens above key `thr` and of those with it the first `quota` in index order.
  uint32_t thr = 0;
  u64 total = l.cut.total, quota = ~0ull, mass_thr = 0;
  if (total == 0) return false;
  auto mass_of = [&](uint32_t key) { return token_mass(key_value(key), m); };
  if (l.cut.bin < kBins) {
    thr = radix_select(n, l.cut.target - l.cut.above, l.hist, [&](int i) { return l.list[i].x; },
                       [&](int, uint32_t key) { return mass_of(key); });
    u64 gt = 0;
    for (int i = tid; i < n; i += kSampleThreads) {
      const uint2 e = l.list[i];
      if (e.x > thr) gt += mass_of(e.x);
      else if (e.x == thr) l.ties[atomicAdd(&l.cnt_eq, 1)] = e.y;
    }
    if (gt) atomicAdd(&l.mass_gt, gt);
    __syncthreads();
    mass_thr = mass_of(thr);
    quota = (u64)l.cnt_eq;
    const u64 mass_gt = l.cut.above + l.mass_gt;
    if (mass_thr > 0) {
      const u64 need = (l.cut.target - mass_gt + mass_thr - 1) / mass_thr;
      if (need < quota) quota = need;
    }
    total = mass_gt + quota * mass_thr;
    // the listed tokens that are kept count in their slices
    for (int i = tid; i < n; i += kSampleThreads) {
      const uint2 e = l.list[i];
      bool kept = e.x > thr;
      if (e.x == thr) {
        u64 rank = 0;
        if (quota < (u64)l.cnt_eq)
          for (int j = 0; j < l.cnt_eq; ++j) rank += l.ties[j] < e.y;
        kept = rank < quota;
      }
      if (kept) atomicAdd(&l.slice[e.y / kSlice], mass_of(e.x));
    }
    __syncthreads();
  }
  u64 goal = (u64)((double)a.uniform[r] * (double)total);
  if (goal >= total) goal = total - 1;
  if (wv == 0) {   // the slice that holds the goal
    u64 run = 0;
    int at = s.slices - 1;
    for (int b0 = 0; b0 < s.slices; b0 += 64) {
      const u64 mine = b0 + lane < s.slices ? l.slice[b0 + lane] : 0;
      const u64 incl = run + wave_sums(mine);
      const u64 hit = __ballot(goal < incl);
      if (hit) {
        const int first = __ffsll(hit) - 1;
        at = b0 + first;
        run = __shfl(incl - mine, first, 64);
        break;
      }
      run = __shfl(incl, 63, 64);
    }
    if (lane == 0) l.at = at, l.before = run, l.cnt_before = 0;
  }
  __syncthreads();
  const int s0 = l.at * kSlice, end = min(a.V, s0 + kSlice);
  constexpr int EACH = kSlice / kSampleThreads;   // neighbours of a thread
  const float* row = wide_row(a, r);
  uint32_t key[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int t = s0 + EACH * tid + i;
    key[i] = t < end ? ordered_key(row[t] * inv_t) : 0;
  }
  u64 rank = 0;   // tokens at the threshold before this thread's
  const bool ties = quota < (u64)l.cnt_eq;
  if (ties) {
    int before = 0, mine = 0;
    for (int i = tid; i < l.cnt_eq; i += kSampleThreads) before += (int)l.ties[i] < s0;
    if (before) atomicAdd(&l.cnt_before, before);
#pragma unroll
    for (int i = 0; i < EACH; ++i) mine += key[i] == thr && s0 + EACH * tid + i < end;
    int incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) l.ranks[wv] = incl;
    __syncthreads();
    rank = l.cnt_before + incl - mine;
    for (int i = 0; i < wv; ++i) rank += l.ranks[i];
  }
  u64 mass[EACH], mine = 0;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    mass[i] = 0;
    if (s0 + EACH * tid + i >= end) continue;
    if (key[i] > thr) mass[i] = mass_of(key[i]);
    else if (key[i] == thr && (!ties || rank++ < quota)) mass[i] = mass_thr;
    mine += mass[i];
  }
  const u64 incl = wave_sums(mine);
  if (lane == 63) l.sums[wv] = incl;
  __syncthreads();
  u64 run = l.before + incl - mine;
  for (int i = 0; i < wv; ++i) run += l.sums[i];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    if (mass[i] && goal >= run && goal < run + mass[i]) a.out[r] = s0 + EACH * tid + i;
    run += mass[i];
  }
  return true;
}

__global__ __launch_bounds__(kSampleThreads) void sample_draw_kernel(SampleArgs a, SampleScratch s) {
  __shared__ DrawLds lds;
  const int r = blockIdx.x, groups = s.slices * kSliceThreads;
  uint32_t got[kLookKeys];   // (asked for before the row's kind is known; a row of another kind has left some undefined)
#pragma unroll
  for (int u = 0; u < kLookKeys; ++u) {
    const int g = threadIdx.x + u * kSampleThreads;
    got[u] = g < groups ? s.maxima[(int64_t)r * groups + g] : 0;
  }
  const RowKind kind = row_kind(a, s, r);
  if (kind == kRowFew && draw_few(a, s, r, lds, got)) return;
  if (kind == kRowWide && draw_wide(a, s, r, lds)) return;
  __syncthreads();
  sample_whole_row(a, r, lds.row);
}

}  // namespace ninfer

using namespace ninfer;

// out[i] <- a number in [0, 1) of 24 random bits from (seeds[i], keys[i], draws[i]), on the host: sampling/sampler.py's
// `uniform`. 64 rows as whole arrays in numpy took 44 us, 27 passes; here 5 and 14 for the arrays.
extern "C" void ninfer_uniforms(const unsigned long long* seeds, const unsigned long long* keys,
                                const unsigned long long* draws, int n, float* out) {
  auto mix = [](unsigned long long x) {   // splitmix64's step and finalizer
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
  };
  for (int i = 0; i < n; ++i) out[i] = (float)(mix(mix(mix(seeds[i]) ^ keys[i]) ^ draws[i]) >> 40) * 0x1p-24f;
}

static int sample_check(const SampleArgs& a, int R) {
  NINFER_REQUIRE(R > 0 && a.V > 0, "sample: R=%d V=%d must be positive", R, a.V);
  NINFER_REQUIRE(a.ld >= a.V, "sample: row stride %d < vocabulary %d", a.ld, a.V);
  NINFER_REQUIRE(a.temperature && a.uniform && a.out, "sample: a required array is null");
  return 0;
}

// logits [R, ld] (V used); work [R, V] scratch; per-row temperature, top_k,
// top_p, rep_penalty, uniform; penalties as (token, count) pairs in
// pen_tokens/pen_counts[pen_offsets[r] .. pen_offsets[r+1]) (null: none);
// out [R] token ids.
static int sample_by_rows(const SampleArgs& a, int R, hipStream_t stream) {
  int rc = sample_check(a, R);
  if (rc) return rc;
  NINFER_REQUIRE(a.work, "sample: a required array is null");
  sample_kernel<<<R, kSampleThreads, 0, stream>>>(a);
  NINFER_LAUNCH_CHECK();
  return 0;
}
extern "C" int ninfer_sample(const float* logits, int ld, int V, int R, float* work,
                             const float* temperature, const int* top_k, const float* top_p,
                             const float* rep_penalty, const int* pen_tokens,
                             const int* pen_counts, const int* pen_offsets, const float* uniform,
                             int* out, hipStream_t stream) {
  return sample_by_rows({logits, temperature, top_k, top_p, rep_penalty, pen_tokens, pen_counts, pen_offsets,
                         uniform, out, work, ld, V}, R, stream);
}

// The scratch of ninfer_sample_spread, behind work [R, V]: offsets in bytes, and the whole.
struct SpreadLayout {
  long long maxima, slice_max, listed, list, bins, slice_mass, bytes;
  int slices;
};
static SpreadLayout spread_layout(int V, int R, bool wide) {
  SpreadLayout p;
  p.slices = (V + kSlice - 1) / kSlice;
  long long at = 0;
  auto take = [&](long long bytes) {
    const long long here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  take((long long)R * V * 4);   // work
  p.maxima = take((long long)R * p.slices * kSliceThreads * 4);
  p.slice_max = take(wide ? (long long)R * p.slices * 4 : 0);
  p.listed = take(wide ? (long long)R * 4 : 0);
  p.list = take(wide ? (long long)R * kCutList * 8 : 0);
  p.bins = take(wide ? (long long)R * kBins * 8 : 0);
  p.slice_mass = take(wide ? (long long)R * p.slices * 8 : 0);
  p.bytes = at;
  return p;
}

extern "C" int ninfer_sample_few_tokens() { return kFewTokens; }
extern "C" long long ninfer_sample_spread_bytes(int V, int R, int wide) { return spread_layout(V, R, wide).bytes; }

// The same token for every row, by the whole GPU where a row is greedy or keeps at most kFewTokens
// tokens (top_k) and, with `wide`, where top_k cuts nothing; other rows are as with ninfer_sample.
// scratch: ninfer_sample_spread_bytes(V, R, wide) bytes, aligned to 256.
static int sample_by_slices(const SampleArgs& a, int R, int wide, hipStream_t stream) {
  const int V = a.V;
  void* const scratch = a.work;
  int rc = sample_check(a, R);
  if (rc) return rc;
  NINFER_REQUIRE(scratch && (uintptr_t)scratch % 256 == 0, "sample: scratch is null or not aligned");
  NINFER_REQUIRE(R <= kSpreadRows, "sample: %d rows are too many", R);
  if ((V + kSlice - 1) / kSlice > kMaxSlices) wide = 0;
  const SpreadLayout p = spread_layout(V, R, wide);
  char* base = (char*)scratch;
  typedef unsigned long long u64;
  const SampleScratch s = {(uint32_t*)(base + p.maxima), (uint32_t*)(base + p.slice_max), (int*)(base + p.listed),
                           (uint2*)(base + p.list),      (u64*)(base + p.bins),           (u64*)(base + p.slice_mass),
                           p.slices,                     wide != 0};
  const dim3 grid(p.slices, R);
  sample_maxima_kernel<<<grid, kSliceThreads, 0, stream>>>(a, s);
  NINFER_LAUNCH_CHECK();
  if (wide) {
    sample_masses_kernel<<<grid, kSliceThreads, 0, stream>>>(a, s);
    NINFER_LAUNCH_CHECK();
    sample_cut_kernel<<<grid, kSliceThreads, 0, stream>>>(a, s);
    NINFER_LAUNCH_CHECK();
  }
  sample_draw_kernel<<<R, kSampleThreads, 0, stream>>>(a, s);
  NINFER_LAUNCH_CHECK();
  return 0;
}
extern "C" int ninfer_sample_spread(const float* logits, int ld, int V, int R, int wide, void* scratch,
                                    const float* temperature, const int* top_k, const float* top_p,
                                    const float* rep_penalty, const int* pen_tokens,
                                    const int* pen_counts, const int* pen_offsets, const float* uniform,
                                    int* out, hipStream_t stream) {
  return sample_by_slices({logits, temperature, top_k, top_p, rep_penalty, pen_tokens, pen_counts, pen_offsets,
                           uniform, out, (float*)scratch, ld, V}, R, wide, stream);
}

// Pinned host memory to the device, 16 bytes a thread and turn. (As a kernel: a copy by the runtime costs the host 5 us
// more, and the same on the device.)
__global__ __launch_bounds__(256) void sample_fetch_kernel(const int4* __restrict__ from, int4* __restrict__ to, long long n) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) to[i] = from[i];
}

// A sampler's whole call: the rows' parameters, laid out in pinned host memory (aligned to 16 bytes), go to the device, the
// kernels run (mode 0: ninfer_sample, 1 and 2: ninfer_sample_spread without and with `wide`), write the tokens back into
// pinned memory, and the host waits for them. What bounds such a call is the host: as a copy, launches and a copy back through
// tensors and events it took 62 us for one row of 151,936 tokens, 78 for 8 and 139 for 64 with 1,500 tokens of history, 40, 50 and 123 so.
// host: temperature[R], top_p[R], rep_penalty[R], uniform[R] (floats), top_k[R], and with n_pen > 0 pen_offsets[R + 1],
// pen_tokens[n_pen], pen_counts[n_pen]; `ints` numbers in all, a multiple of 4 of them reserved here and in `params` (device
// memory); tokens [R] in pinned memory. scratch: as the two ask for.
extern "C" int ninfer_sample_rows(const float* logits, int ld, int V, int R, int mode, const int* host, int* params,
                                  long long ints, int n_pen, void* scratch, int* tokens, hipStream_t stream) {
  const long long need = 5ll * R + (n_pen > 0 ? R + 1 + 2ll * n_pen : 0);
  NINFER_REQUIRE(R > 0 && host && params && tokens && n_pen >= 0 && ints == need && (uintptr_t)host % 16 == 0 &&
                 (uintptr_t)params % 16 == 0, "sample: %lld numbers of %d rows with %d penalties", ints, R, n_pen);
  const long long quads = (ints + 3) / 4;
  sample_fetch_kernel<<<(unsigned)min(256ll, (quads + 255) / 256), 256, 0, stream>>>((const int4*)host, (int4*)params, quads);
  NINFER_LAUNCH_CHECK();
  const float* f = (const float*)params;
  const int* pen = n_pen > 0 ? params + 5 * R : nullptr;
  const SampleArgs a = {logits, f, params + 4 * R, f + R, f + 2 * R, pen ? pen + R + 1 : nullptr, pen ? pen + R + 1 + n_pen : nullptr,
                        pen, f + 3 * R, tokens, (float*)scratch, ld, V};
  // (not through the two entry points above: the engine's C interface has a function by the name of one, and in a program
  // that is linked to it a call by that name would end there)
  const bool by_rows = mode == 0 || R > kSpreadRows;   // (the same tokens; the others' scratch begins with this one's)
  const int rc = by_rows ? sample_by_rows(a, R, stream) : sample_by_slices(a, R, mode == 2, stream);
  const hipError_t e = hipStreamSynchronize(stream);   // (also after an error: the caller's buffers are its own again)
  if (rc) return rc;
  if (e != hipSuccess) return set_error(-2, "sample: %s", hipGetErrorString(e));
  return 0;
}
