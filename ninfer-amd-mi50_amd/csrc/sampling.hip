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

__global__ __launch_bounds__(kSampleThreads) void sample_kernel(
    const float* __restrict__ logits, int ld, int V, float* __restrict__ work,
    const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, const float* __restrict__ rep_penalty,
    const int* __restrict__ pen_tokens, const int* __restrict__ pen_counts,
    const int* __restrict__ pen_offsets, const float* __restrict__ uniform, int* __restrict__ out) {
  __shared__ RadixHist<8> hist;
  __shared__ unsigned long long sums[2 * kSampleThreads / 64];
  __shared__ float fred[kSampleThreads / 64];
  __shared__ int ired[kSampleThreads / 64];

  const int r = blockIdx.x, tid = threadIdx.x;
  const float* row = logits + (int64_t)r * ld;
  float* w = work + (int64_t)r * V;
  const float temp = temperature[r];

  // repetition penalty on a copy of the row (greedy rows without a penalty read the row itself)
  float rp = rep_penalty ? rep_penalty[r] : 1.f;
  const bool penalised = rp != 1.f && pen_offsets && pen_offsets[r + 1] > pen_offsets[r];
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
      float v = w[tok];
      for (int c = 0; c < pen_counts[e]; ++c) v = v > 0.f ? v / rp : v * rp;
      w[tok] = v;
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

// Rows that keep few tokens (greedy, or top-k up to kCandPerSlice) in two launches that use the
// whole GPU. First the row is cut into slices of kSlice tokens, one block each, which holds its
// slice in LDS, applies the repetition penalty to it, and writes out, in index order, its own k best
// tokens under the order (scaled logit descending, index ascending). Every token of the row's k
// best is among its slice's k best, so the k best of all candidates are the row's, and the second
// launch, a block per row, finds them and draws: the same kept set, masses and token as
// sample_kernel's on the whole row.
//
// The k-th largest of n keys without a histogram: of the threads' largest keys, the k-th largest
// is a bound that at least k keys reach, and hardly more do; those are listed and ranked among
// themselves, each by a thread that compares it with all others. Lists that do not fit (many equal
// logits) go through radix_select. 64 rows of 151,936 tokens with top-k 50: candidates 126 -> 36 us
// and the draw 83 -> 21 us, against four and eight passes of a histogram (the keys share few upper
// bytes, so its atomics follow each other, and one thread added the bins up).
constexpr int kSlice = 4096;
constexpr int kCandPerSlice = 64;
constexpr int kCandThreads = 256;
constexpr int kFewList = 256;

struct FewLds {
  uint4 best[kCandThreads / 4];   // the threads' largest keys, four by four
  uint32_t key[kFewList];
  int idx[kFewList];
  int kept[kFewList];             // index of a kept one
  uint32_t bound;
  int count;
  int wave_tot[kCandThreads / 64];
  RadixHist<1> hist;
};

// The k best of keys 0 .. n - 1 (1 <= k <= kCandPerSlice, k <= n): put(place, i) is called once for
// each, places counted in index order. Every thread of the block must call.
template <typename KeyFn, typename PutFn>
__device__ void few_best(int n, int k, FewLds& l, KeyFn key, PutFn put) {
  const int tid = threadIdx.x;
  uint32_t mine = 0;
  for (int i = tid; i < n; i += kCandThreads) mine = max(mine, key(i));
  ((uint32_t*)l.best)[tid] = mine;
  if (tid == 0) l.count = 0;
  __syncthreads();
  if (tid < 64) {   // the k-th largest of the 256, bit by bit: the largest bound that k of them reach
    const uint4 m = l.best[tid];
    uint32_t bound = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t at = bound | (1u << bit);
      const int reach = __popcll(__ballot(m.x >= at)) + __popcll(__ballot(m.y >= at)) +
                        __popcll(__ballot(m.z >= at)) + __popcll(__ballot(m.w >= at));
      if (reach >= k) bound = at;
    }
    if (tid == 0) l.bound = bound;
  }
  __syncthreads();
  const uint32_t bound = l.bound;
  for (int i = tid; i < n; i += kCandThreads) {
    const uint32_t kk = key(i);
    if (kk >= bound) {
      const int at = atomicAdd(&l.count, 1);
      if (at < kFewList) {
        l.key[at] = kk;
        l.idx[at] = i;
      }
    }
  }
  __syncthreads();
  const int count = l.count;
  if (count <= kFewList) {
    const int padded = (count + 15) / 16 * 16;
    if (tid >= count && tid < padded) {   // places that nothing follows and nothing counts
      l.key[tid] = 0;
      l.idx[tid] = 0x7fffffff;
      l.kept[tid] = 0x7fffffff;
    }
    __syncthreads();
    uint32_t kk = 0;
    int i = 0, better = 0;
    if (tid < count) {
      kk = l.key[tid];
      i = l.idx[tid];
#pragma unroll 16
      for (int j = 0; j < padded; ++j) better += l.key[j] > kk || (l.key[j] == kk && l.idx[j] < i);
      l.kept[tid] = better < k ? i : 0x7fffffff;
    }
    __syncthreads();
    if (tid < count && better < k) {
      int place = 0;
#pragma unroll 16
      for (int j = 0; j < padded; ++j) place += l.kept[j] < i;
      put(place, i);
    }
    __syncthreads();
    return;
  }
  const uint32_t thr = k < n ? radix_select(n, (unsigned long long)k, l.hist, key, [](int, uint32_t) { return 1ull; }) : 0;
  auto block_count = [&](int v) -> int {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((tid & 63) == 0) l.wave_tot[tid >> 6] = v;
    __syncthreads();
    v = 0;
    for (int i = 0; i < kCandThreads / 64; ++i) v += l.wave_tot[i];
    __syncthreads();
    return v;
  };
  int above = 0;
  for (int i = tid; i < n; i += kCandThreads) above += key(i) > thr;
  const int quota = k - block_count(above);   // of the keys tied at thr, the first so many
  auto scan = [&](int v) -> int {   // sum over the threads before this one
    const int lane = tid & 63, wv = tid >> 6;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) l.wave_tot[wv] = incl;
    __syncthreads();
    int base = 0;
    for (int i = 0; i < wv; ++i) base += l.wave_tot[i];
    __syncthreads();
    return base + incl - v;
  };
  const int run = (n + kCandThreads - 1) / kCandThreads, i0 = min(n, tid * run), i1 = min(n, i0 + run);
  int eq = 0;
  for (int i = i0; i < i1; ++i) eq += key(i) == thr;
  const int rank0 = scan(eq);
  int kept = 0, tie = rank0;
  for (int i = i0; i < i1; ++i) {
    const uint32_t kk = key(i);
    kept += kk > thr || (kk == thr && tie++ < quota);
  }
  int place = scan(kept);
  tie = rank0;
  for (int i = i0; i < i1; ++i) {
    const uint32_t kk = key(i);
    if (kk > thr || (kk == thr && tie++ < quota)) put(place++, i);
  }
  __syncthreads();
}

__global__ __launch_bounds__(kCandThreads) void sample_candidates_kernel(
    const float* __restrict__ logits, int ld, int V, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ rep_penalty,
    const int* __restrict__ pen_tokens, const int* __restrict__ pen_counts,
    const int* __restrict__ pen_offsets, float* __restrict__ cand_val, int* __restrict__ cand_idx) {
  __shared__ float vals[kSlice];
  __shared__ FewLds l;
  const int r = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
  const int s0 = b * kSlice, n = min(kSlice, V - s0);
  const int C = gridDim.x * kCandPerSlice;
  const float* row = logits + (int64_t)r * ld;
  float x[kSlice / kCandThreads];   // every load on its way at once
#pragma unroll
  for (int u = 0; u < kSlice / kCandThreads; ++u) x[u] = row[s0 + min(tid + u * kCandThreads, n - 1)];
  const float rp = rep_penalty ? rep_penalty[r] : 1.f;
  const bool penalised = rp != 1.f && pen_offsets && pen_offsets[r + 1] > pen_offsets[r];
  const int first_pen = penalised ? pen_offsets[r] : 0, end_pen = penalised ? pen_offsets[r + 1] : 0;
  int pen[8];   // penalised tokens, eight at a time, the first beside the slice
  auto load_pens = [&](int e0) {
#pragma unroll
    for (int u = 0; u < 8; ++u) pen[u] = pen_tokens[min(e0 + u * kCandThreads, end_pen - 1)];
  };
  if (penalised) load_pens(first_pen + tid);
#pragma unroll
  for (int u = 0; u < kSlice / kCandThreads; ++u) vals[tid + u * kCandThreads] = x[u];
  __syncthreads();
  if (penalised) {
    for (int e0 = first_pen + tid; e0 < end_pen; e0 += 8 * kCandThreads) {
      if (e0 != first_pen + tid) load_pens(e0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = e0 + u * kCandThreads, t = pen[u] - s0;
        if (e >= end_pen || t < 0 || t >= n) continue;
        float v = vals[t];
        for (int c = 0; c < pen_counts[e]; ++c) v = v > 0.f ? v / rp : v * rp;
        vals[t] = v;
      }
    }
    __syncthreads();
  }
  const float temp = temperature[r];
  const float inv_t = temp > 0.f ? 1.f / temp : 1.f;
  int k = temp > 0.f ? top_k[r] : 1;            // greedy is the best one
  if (k < 1 || k > kCandPerSlice) k = kCandPerSlice;   // (not this entry's rows: kept in bounds)
  k = min(k, n);
  float* cv = cand_val + (int64_t)r * C + b * kCandPerSlice;
  int* ci = cand_idx + (int64_t)r * C + b * kCandPerSlice;
  few_best(n, k, l, [&](int i) { return ordered_key(vals[i] * inv_t); },
           [&](int place, int i) {
             cv[place] = vals[i];
             ci[place] = s0 + i;
           });
  // the places left over hold nothing: never the largest, no mass
  for (int i = k + tid; i < kCandPerSlice; i += kCandThreads) {
    cv[i] = -INFINITY;
    ci[i] = 0;
  }
}

// The draw among a row's C candidates (in index order); sample_kernel says what it is. STAGED: they
// fit LDS (vocabularies of up to 262,144 tokens).
template <bool STAGED>
__global__ __launch_bounds__(kCandThreads) void sample_few_kernel(
    const float* __restrict__ cand_val, const int* __restrict__ cand_idx, int C,
    const float* __restrict__ temperature, const int* __restrict__ top_k, const float* __restrict__ top_p,
    const float* __restrict__ uniform, int* __restrict__ out) {
  typedef unsigned long long u64;
  __shared__ FewLds l;
  __shared__ float fred[kCandThreads / 64];
  __shared__ int ired[kCandThreads / 64];
  __shared__ float val_s[kCandPerSlice];
  __shared__ int idx_s[kCandPerSlice];
  __shared__ u64 mass_s[kCandPerSlice];
  __shared__ uint32_t key_s[kCandPerSlice];
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  __shared__ float staged[STAGED ? kSlice : 1];
  const float* row = cand_val + (int64_t)r * C;
  const int* idx = cand_idx + (int64_t)r * C;
  if (STAGED) {
    float x[kSlice / kCandThreads];
#pragma unroll
    for (int u = 0; u < kSlice / kCandThreads; ++u) x[u] = row[min(tid + u * kCandThreads, C - 1)];
#pragma unroll
    for (int u = 0; u < kSlice / kCandThreads; ++u) staged[tid + u * kCandThreads] = x[u];
    __syncthreads();
  }
  auto value = [&](int i) { return STAGED ? staged[i] : row[i]; };
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  for (int i = tid; i < C; i += kCandThreads) {
    const float v = value(i);
    if (v > best) {
      best = v;
      best_i = i;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ob = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(best_i, off, 64);
    if (ob > best || (ob == best && oi < best_i)) {
      best = ob;
      best_i = oi;
    }
  }
  if (lane == 0) {
    fred[tid >> 6] = best;
    ired[tid >> 6] = best_i;
  }
  __syncthreads();
  best = fred[0];
  best_i = ired[0];
  for (int i = 1; i < kCandThreads / 64; ++i)
    if (fred[i] > best || (fred[i] == best && ired[i] < best_i)) {
      best = fred[i];
      best_i = ired[i];
    }
  const float temp = temperature[r];
  if (!(temp > 0.f)) {
    // (a row without a number above minus infinity: the first place)
    if (tid == 0) out[r] = idx[best_i < C ? best_i : 0];
    return;
  }
  const float inv_t = 1.f / temp, m = best * inv_t;
  int k = top_k[r];
  if (k < 1 || k > kCandPerSlice) k = kCandPerSlice;
  few_best(C, k, l, [&](int i) { return ordered_key(value(i) * inv_t); },
           [&](int place, int i) {
             val_s[place] = value(i);
             idx_s[place] = idx[i];
           });
  if (tid >= 64) return;
  // One wave: lane j has the j-th kept token in index order. Its mass, and that of the tokens before
  // it in the order (logit descending, index ascending): top-p keeps those before the target.
  const bool have = lane < k;
  const uint32_t kk = have ? ordered_key(val_s[lane] * inv_t) : 0;
  const u64 mass = have ? token_mass(val_s[lane] * inv_t, m) : 0;
  mass_s[lane] = mass;
  key_s[lane] = kk;
  // (one wave: its LDS accesses run in order, and the fence keeps the compiler from changing that)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  u64 total = 0, ahead = 0;
#pragma unroll 8
  for (int j = 0; j < kCandPerSlice; ++j) {   // (places from k on have no mass)
    const u64 o = mass_s[j];
    total += o;
    if (key_s[j] > kk || (key_s[j] == kk && j < lane)) ahead += o;
  }
  const float pp = top_p ? top_p[r] : 1.f;
  u64 target = total;
  if (pp < 1.f) {
    target = (u64)((double)pp * (double)total);
    if (target < 1) target = 1;
  }
  const u64 kept = have && ahead < target ? mass : 0;
  u64 incl = kept;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const u64 o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  total = __shfl(incl, 63, 64);
  u64 goal = (u64)((double)uniform[r] * (double)total);
  if (goal >= total) goal = total - 1;
  if (kept > 0 && goal >= incl - kept && goal < incl) out[r] = idx_s[lane];
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

// logits [R, ld] (V used); work [R, V] scratch; per-row temperature, top_k,
// top_p, rep_penalty, uniform; penalties as (token, count) pairs in
// pen_tokens/pen_counts[pen_offsets[r] .. pen_offsets[r+1]) (null: none);
// out [R] token ids.
extern "C" int ninfer_sample(const float* logits, int ld, int V, int R, float* work,
                             const float* temperature, const int* top_k, const float* top_p,
                             const float* rep_penalty, const int* pen_tokens,
                             const int* pen_counts, const int* pen_offsets, const float* uniform,
                             int* out, hipStream_t stream) {
  NINFER_REQUIRE(R > 0 && V > 0, "sample: R=%d V=%d must be positive", R, V);
  NINFER_REQUIRE(ld >= V, "sample: row stride %d < vocabulary %d", ld, V);
  NINFER_REQUIRE(temperature && uniform && work && out, "sample: a required array is null");
  sample_kernel<<<R, kSampleThreads, 0, stream>>>(logits, ld, V, work, temperature, top_k, top_p,
                                                  rep_penalty, pen_tokens, pen_counts, pen_offsets,
                                                  uniform, out);
  NINFER_LAUNCH_CHECK();
  return 0;
}

// Places per row that ninfer_sample_few needs in each of cand_val and cand_idx.
extern "C" long long ninfer_sample_few_places(int V) {
  return (long long)((V + kSlice - 1) / kSlice) * kCandPerSlice;
}

// The same for rows that all keep few tokens: every row greedy (temperature <= 0) or with
// 1 <= top_k <= 64, which the caller asserts (a row with another top_k would be cut to its 64
// best per slice). Same result as ninfer_sample, from two launches that use the whole GPU.
// cand_val, cand_idx: [R, ninfer_sample_few_places(V)].
extern "C" int ninfer_sample_few(const float* logits, int ld, int V, int R, float* cand_val,
                                 int* cand_idx, const float* temperature,
                                 const int* top_k, const float* top_p, const float* rep_penalty,
                                 const int* pen_tokens, const int* pen_counts,
                                 const int* pen_offsets, const float* uniform, int* out,
                                 hipStream_t stream) {
  NINFER_REQUIRE(R > 0 && V > 0, "sample: R=%d V=%d must be positive", R, V);
  NINFER_REQUIRE(ld >= V, "sample: row stride %d < vocabulary %d", ld, V);
  NINFER_REQUIRE(temperature && top_k && uniform && cand_val && cand_idx && out,
                 "sample: a required array is null");
  const int slices = (V + kSlice - 1) / kSlice, C = slices * kCandPerSlice;
  NINFER_REQUIRE(R <= 65535, "sample: %d rows are too many", R);
  sample_candidates_kernel<<<dim3(slices, R), kCandThreads, 0, stream>>>(
      logits, ld, V, temperature, top_k, rep_penalty, pen_tokens, pen_counts, pen_offsets, cand_val,
      cand_idx);
  NINFER_LAUNCH_CHECK();
  if (C <= kSlice)
    sample_few_kernel<true><<<R, kCandThreads, 0, stream>>>(cand_val, cand_idx, C, temperature, top_k, top_p,
                                                            uniform, out);
  else
    sample_few_kernel<false><<<R, kCandThreads, 0, stream>>>(cand_val, cand_idx, C, temperature, top_k, top_p,
                                                             uniform, out);
  NINFER_LAUNCH_CHECK();
  return 0;
}
