// Paged attention of prompt portions in 32-bit: the plain kernel's sums (attention_generic.hip), several rows of a
// request at a time.
//
// A block of four waves owns 8 consecutive rows of a request and one query head, a wave two of them; the keys and
// values of a tile of 64 positions come into LDS once for all 8. As in the plain kernel a lane is a key in the scores (d
// ascending in one chain) and a value's number in the output (keys ascending), the softmax between them runs over the
// wave, and tiles are aligned to absolute positions: every row's bits are the plain kernel's, whatever block it is
// in. A row's weights come by lane reads, the two chains of products of a wave's rows share every read of keys and values.
// What bounds the plain kernel is that its lanes each walk a key's row of their own through L1, once per row; here a
// tile's chain of some 1,100 instructions a wave, 4.3 us for two rows. us there and here, 16 heads of 128: a prompt of
// 173 tokens 39 and 24, of 600 250 and 110, of 2,048 2,420 and 850; 64 rows behind 2,000 keys 360 and 148, 2 rows of four
// requests 321 and 140. Within one tile of keys the plain kernel (16 tokens 8.1 and 9.4).
#include "attention.h"
#include "gemm.h"
#include <type_traits>

namespace ninfer {

constexpr int kRowsPerWave = 2, kRowsPerBlock = 4 * kRowsPerWave, kRowsKeys = 64;

// Maximum and sum over a wave's 64 lanes, in every lane, by lane moves of the vector unit: the pairs of common.h's
// exchanges through LDS in the same order (32 lanes apart, 16, .. 1), so the same bits.
template <typename Op> __device__ __forceinline__ float rows_reduce(float v, Op op) {
  auto both = [&](auto pair) { return op(__int_as_float(pair[0]), __int_as_float(pair[1])); };
  v = both(__builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false));
  v = both(__builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false));
  auto moved = [](float x, auto ctrl, auto banks, float old) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), decltype(ctrl)::value, 0xf,
                                                      decltype(banks)::value, false));
  };
  typedef std::integral_constant<int, 0xf> all;
  v = op(v, moved(v, std::integral_constant<int, 0x128>{}, all{}, v));   // 8 lanes round the row of 16
  // four up for the even fours of lanes, four down for the odd ones
  v = op(v, moved(v, std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xa>{},
                  moved(v, std::integral_constant<int, 0x104>{}, std::integral_constant<int, 0x5>{}, v)));
  v = op(v, moved(v, std::integral_constant<int, 0x4e>{}, all{}, v));    // two, within four
  v = op(v, moved(v, std::integral_constant<int, 0xb1>{}, all{}, v));    // the neighbour
  return v;
}
__device__ __forceinline__ float rows_max(float v) { return rows_reduce(v, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ float rows_sum(float v) { return rows_reduce(v, [](float a, float b) { return a + b; }); }

typedef float quad __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void attention_rows_f32_kernel(AttnArgs a) {
  constexpr int R = kRowsPerWave;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ int info[3];
  __shared__ int64_t place_s[2][kRowsKeys];   // (page * Hkv + g) * page_size + slot of each key of a tile
  const int D = a.D, Dv = a.Dv, Hkv = a.Hkv, KROW = D + 4;   // (padded: 16 lanes' pieces in as many banks)
  float* Ks = smem;                       // [64][KROW]
  float* Vs = smem + kRowsKeys * KROW;    // [64][Dv], and 128 behind it that idle lanes may read
  float* qs = Vs + kRowsKeys * Dv + 128;  // [8][D]
  const int h = blockIdx.y, g = h / (a.Hq / Hkv);
  if (!find_tile(a.seq_row_start, a.S, kRowsPerBlock, gridDim.x - 1 - blockIdx.x, info)) return;
  const int row0 = info[0], seq = info[2], n_rows = min(kRowsPerBlock, info[1] - row0);
  const int pos0 = a.positions[row0], pos_last = pos0 + n_rows - 1;
  const int lo_first = a.window > 0 ? max(0, pos0 - a.window + 1) : 0;
  const int* bt = a.block_table + (int64_t)seq * a.bt_stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float slope = a.slopes ? a.slopes[h] : 0.f;

  int pos[R], lo[R];
  bool live[R];
  const float* q[R];   // in LDS
  float m[R], l[R], acc[R][2];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = wave * R + i;
    live[i] = r < n_rows;
    pos[i] = pos0 + r;
    lo[i] = a.window > 0 ? max(0, pos[i] - a.window + 1) : 0;
    q[i] = qs + r * D;
    m[i] = a.sink ? attention_sink(a, h) : -INFINITY;
    l[i] = a.sink ? 1.f : 0.f;
    acc[i][0] = acc[i][1] = 0.f;
  }

  // Pieces of 16 bytes that this thread moves: keys' and values', from registers that the next tile's loads fill while
  // this one is multiplied. Where a tile's keys lie is looked up a tile earlier still. A key that no row of the block
  // sees is the nearest that one does (it meets no weight).
  constexpr int PIECES = kRowsKeys * 32 / 256;
  int k_key[PIECES], k_at[PIECES], v_key[PIECES], v_at[PIECES];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int p = tid + 256 * i, kp = min(p, kRowsKeys * D / 4 - 1), vp = min(p, kRowsKeys * Dv / 4 - 1);
    k_key[i] = kp / (D / 4);
    k_at[i] = 4 * (kp % (D / 4));
    v_key[i] = vp / (Dv / 4);
    v_at[i] = 4 * (vp % (Dv / 4));
  }
  auto look_up = [&](int buf, int tile) {
    if (tid < kRowsKeys) {
      const int j = max(min(tile + tid, pos_last), lo_first);
      place_s[buf][tid] = ((int64_t)bt[j / a.page_size] * Hkv + g) * a.page_size + j % a.page_size;
    }
  };
  quad k_reg[PIECES], v_reg[PIECES];
  auto load = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      k_reg[i] = *(const quad*)((const float*)a.kpool + place_s[buf][k_key[i]] * D + k_at[i]);
      v_reg[i] = *(const quad*)((const float*)a.vpool + place_s[buf][v_key[i]] * Dv + v_at[i]);
    }
  };
  const int tile0 = (lo_first / kRowsKeys) * kRowsKeys;
  for (int i = tid; i < n_rows * D; i += 256) qs[i] = ((const float*)a.q)[(int64_t)(row0 + i / D) * a.q_stride + h * D + i % D];
  look_up(0, tile0);
  __syncthreads();
  load(0);
  look_up(1, tile0 + kRowsKeys);
  for (int tile = tile0, buf = 0; tile <= pos_last; tile += kRowsKeys, buf ^= 1) {
    __syncthreads();   // the tile before is read
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {   // (pieces behind the last are the last again, by the same bytes)
      *(quad*)(Ks + k_key[i] * KROW + k_at[i]) = k_reg[i];
      *(quad*)(Vs + v_key[i] * Dv + v_at[i]) = v_reg[i];
    }
    __syncthreads();
    if (tile + kRowsKeys <= pos_last) {
      load(buf ^ 1);
      look_up(buf, tile + 2 * kRowsKeys);
    }

    bool sees[R], any = false, whole = true;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      sees[i] = live[i] && tile <= pos[i] && tile + kRowsKeys > lo[i];
      any |= sees[i];
      whole &= sees[i] && lo[i] <= tile && tile + kRowsKeys - 1 <= pos[i];
    }
    if (!any) continue;
    float dot[R];
#pragma unroll
    for (int i = 0; i < R; ++i) dot[i] = 0.f;
    const float* kr = Ks + lane * KROW;
#pragma unroll 8
    for (int d = 0; d < D; d += 4) {
      const quad k = *(const quad*)(kr + d);
#pragma unroll
      for (int i = 0; i < R; ++i) {   // (a row that is not there: whatever LDS holds, never used)
        const quad x = *(const quad*)(q[i] + d);
        dot[i] = fmaf(x[0], k[0], dot[i]);
        dot[i] = fmaf(x[1], k[1], dot[i]);
        dot[i] = fmaf(x[2], k[2], dot[i]);
        dot[i] = fmaf(x[3], k[3], dot[i]);
      }
    }
    // (without a branch a row, so that the rows' chains run side by side; what a row that does not see the tile holds
    // stays as it is)
    const int j = tile + lane;
    float p[R], s[R], top[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bool valid = sees[i] && j >= lo[i] && j <= pos[i];
      s[i] = valid ? fmaf(slope, (float)(j - pos[i]), dot[i] * a.scale) : -INFINITY;
      top[i] = fmaxf(m[i], rows_max(s[i]));
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bool valid = sees[i] && j >= lo[i] && j <= pos[i];
      p[i] = valid ? expf(s[i] - top[i]) : 0.f;
      const float alpha = sees[i] ? expf(m[i] - top[i]) : 1.f;   // 0 on the first tile (m = -inf)
      l[i] = l[i] * alpha + rows_sum(p[i]);
      m[i] = top[i];
      acc[i][0] *= alpha;
      acc[i][1] *= alpha;
    }
    const float* v0 = Vs + lane;   // (lanes behind a value's end read what follows; they store nothing)
    auto weigh = [&](int i, int jj, float x, float y) {
      const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p[i]), jj));
      acc[i][0] = fmaf(pj, x, acc[i][0]);
      acc[i][1] = fmaf(pj, y, acc[i][1]);
    };
    if (whole) {
#pragma unroll 16
      for (int jj = 0; jj < kRowsKeys; ++jj) {
        const float x = v0[jj * Dv], y = v0[jj * Dv + 64];
#pragma unroll
        for (int i = 0; i < R; ++i) weigh(i, jj, x, y);
      }
    } else {
      // (a key that a row does not see is passed over, whatever its value is: the keys that all rows see, side by side,
      // between those that single rows see)
      int first[R], end[R], from = 0, to = kRowsKeys;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        first[i] = sees[i] ? max(0, lo[i] - tile) : 0;
        end[i] = sees[i] ? min(kRowsKeys, pos[i] - tile + 1) : 0;
        from = max(from, first[i]);
        to = min(to, end[i]);
      }
      to = max(to, from);
      auto alone = [&](int i, int begin, int stop) {
        for (int jj = begin; jj < stop; ++jj) weigh(i, jj, v0[jj * Dv], v0[jj * Dv + 64]);
      };
#pragma unroll
      for (int i = 0; i < R; ++i) alone(i, first[i], min(end[i], from));
#pragma unroll 8
      for (int jj = from; jj < to; ++jj) {
        const float x = v0[jj * Dv], y = v0[jj * Dv + 64];
#pragma unroll
        for (int i = 0; i < R; ++i) weigh(i, jj, x, y);
      }
#pragma unroll
      for (int i = 0; i < R; ++i) alone(i, max(to, first[i]), end[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (!live[i]) continue;
    const int64_t t = row0 + wave * R + i;
    const float inv = 1.f / l[i];
    const float* gate = a.gate ? (const float*)a.gate + t * a.gate_stride + h * Dv : nullptr;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int d = lane + 64 * c;
      if (d >= Dv) continue;
      float x = acc[i][c] * inv;
      if (gate) x /= 1.f + expf(-gate[d]);
      ((float*)a.out)[(t * a.Hq + h) * Dv + d] = x;
    }
  }
}

// Keys and values of up to 128 numbers in whole pieces of 16 bytes, no blocks before the window; and steps whose
// requests bring blocks enough rows, so that these pay for their start (some 5 us, one block to a CU) beside the plain
// kernel's waves, one a row. Single rows of such a step share the launch. us there and here:
// - heads of more than 64: 16 heads, 7 rows at 2,500 keys beside 505 new ones 425 and 190; 16 requests of 2 rows at 66 keys 18
//   and 14; 63 rows at 200 keys beside 17 of a prompt 50 and 59 (45 and 59 on 4 kv heads), beside 2,048 2,430 and 880. Sizes
//   that fill no whole pieces of 128 bytes: 32 heads of 100, 16 requests of 2 rows 19 and 24, of 5 rows 38 and 33.
// - of 33 to 64: 8 heads, 505 rows 77 and 46 (39 and 27 in a window of 200), 64 requests of 8 rows at 300 keys 91 and 38,
//   but of 40 of 100 rows 83 and 90, 600 rows in a window of 70 22 and 27; 64 rows at 2,000 keys 193 and 133, 9 at 500 35
//   and 39, 17 beside a single row at 2,000 127 and 142. Smaller ones: 600 rows of 16 heads 80 and 86.
bool attention_rows_f32_takes(const AttnArgs& a) {
  const int dv = a.Dv > 0 ? a.Dv : a.D, most = max(a.D, dv);
  if (a.dtype != kF32 || a.max_qlen <= 1 || a.max_kv_len <= kRowsKeys || a.kblk || a.krot || !a.seq_row_start || a.D % 4 || dv % 4 ||
      most > 128 || most <= 32 || ((uintptr_t)a.kpool | (uintptr_t)a.vpool) % 16)
    return false;
  const long blocks = (long)a.S * a.Hq, cus = device_cu_count();   // (one a request and head at the least)
  if (most > 64) return a.D % 32 || dv % 32 ? blocks <= cus || a.T >= 8L * a.S : blocks <= 2 * cus || a.T >= 4L * a.S;
  const bool windowed = a.window > 0 && a.window < a.max_kv_len;
  if (a.T >= 256 && a.T >= (a.single_rows > 0 ? 16L : 8L) * a.S && a.max_kv_len >= 200) return !windowed || a.window >= 128;
  return !windowed && a.single_rows == 0 && a.max_kv_len >= 1000 && a.T >= 32L * a.S && blocks <= cus;
}

static size_t rows_lds(int D, int Dv) {
  return ((size_t)kRowsKeys * (D + 4 + Dv) + 128 + kRowsPerBlock * D) * sizeof(float);
}

int attention_rows_f32(const AttnArgs& args, hipStream_t stream) {
  AttnArgs a = args;
  if (a.Dv <= 0) a.Dv = a.D;
  const size_t lds = rows_lds(a.D, a.Dv);
  static bool raised = false;
  if (lds > 64 * 1024 && !raised) {
    hipError_t e = hipFuncSetAttribute((const void*)attention_rows_f32_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)rows_lds(128, 128));
    if (e != hipSuccess) return set_error(-2, "paged_attention: %zu bytes of LDS refused: %s", lds, hipGetErrorString(e));
    raised = true;
  }
  const dim3 grid((unsigned)((a.T + kRowsPerBlock - 1) / kRowsPerBlock + a.S), a.Hq);
  attention_rows_f32_kernel<<<grid, 256, lds, stream>>>(a);
  NINFER_LAUNCH_CHECK();
  return 0;
}

}  // namespace ninfer
