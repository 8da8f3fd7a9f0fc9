// C = A W^T in true 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32), dense or grouped by
// expert, with the epilogues of the product family.
//
// What every output is, whatever the batch: K is cut into 8 segments of whole chunks of 16, one
// wave each; a segment is summed chunk by chunk on the matrix instruction and the 8 sums are
// added in the segments' order. Nothing of that depends on M, on the tile's size or on where a
// row lies in its tile, so a row's bits are the same under every cut of the work (which is what
// the 32-bit path promises), and chains of K / 8 terms round less than one of K.
//
// Few rows are bound by the weights' bytes, many by the matrix cores and, below them, by the
// operands' way from L2: a wave meets its RT x CT tiles of 16 x 16 with (RT + CT) KB of operands
// per chunk, straight from global memory in the instruction's own layout (a lane holds four
// neighbouring k of one row, so a chunk is four instructions with k dealt alike to both
// operands): no LDS and no barrier before the last chunk. LDS only carries the 8 partial sums.
// RT follows the rows (per group), CT the number of blocks that the output makes.
// Measured on Qwen1.5-MoE-A2.7B's shapes, a prompt of 173 tokens: the plain tiled kernel spent
// 79.8 ms in its 169 products, this one 20.3: the experts' gate/up (1.4 GB of weights) 290 us,
// 4.8 TB/s; their down products 175 us, 4.0 TB/s; the dense ones 23 to 27 TFLOP/s before and 47 to
// 54 now (at 1,024 rows 84 of the 155 that a large matrix product reaches). One row: 24 us for
// 92 MB of gate/up, 3.9 TB/s.
#include "gemm.h"

namespace ninfer {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kF32Waves = 8;    // segments of K
constexpr int kF32Chunk = 16;   // k of a chunk: four matrix instructions

template <int RT, int CT, bool GATED>
__global__ __launch_bounds__(64 * kF32Waves) void gemm_f32_kernel(GemmArgs a, int n_tiles, int m_tiles) {
  constexpr int BM = 16 * RT;                       // rows of a block
  constexpr int BN = 16 * (GATED ? CT / 2 : CT);    // output features of a block
  constexpr int COLS = 16 * CT + 4;                 // partial sums of a row in LDS (padded)
  // chunks loaded at a time: enough bytes on their way where a wave has little else to do
  constexpr int U = RT + CT <= 2 ? 8 : RT + CT <= 4 ? 4 : 2;
  __shared__ float part[kF32Waves][16][COLS];
  __shared__ int tile_info[3];

  // The row tiles that read the same weights follow each other on one XCD.
  const int xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
  const int n_tile = slot / m_tiles * kXcds + xcd, m_tile = slot % m_tiles;
  if (n_tile >= n_tiles) return;
  int row0, row_end, group = 0;
  if (a.offsets) {
    if (!find_tile(a.offsets, a.groups, BM, m_tile, tile_info)) return;
    row0 = tile_info[0];
    row_end = tile_info[1];
    group = tile_info[2];
  } else {
    row0 = m_tile * BM;
    row_end = a.M;
  }
  const int n0 = n_tile * BN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int in = lane & 15, k_lane = (lane >> 4) * 4;

  // Rows that are not there read the last one that is; nothing of them is stored.
  const float* ap[RT];
  const float* wp[CT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = min(row0 + i * 16 + in, row_end - 1);
    ap[i] = (const float*)a.A + (int64_t)(a.a_index ? a.a_index[r] / a.a_div : r) * a.lda + k_lane;
  }
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    const bool up = GATED && j >= CT / 2;
    const int n = min(n0 + (up ? j - CT / 2 : j) * 16 + in, a.N - 1) + (up ? a.N : 0);
    wp[j] = (const float*)a.W + (int64_t)group * a.w_group_stride + (int64_t)n * a.K + k_lane;
  }

  floatx4 acc[RT][CT] = {};
  const int chunks = (a.K + kF32Chunk - 1) / kF32Chunk;
  const int per = (chunks + kF32Waves - 1) / kF32Waves;
  const int c0 = min(wave * per, chunks), c_all = min(c0 + per, chunks);
  // (a last chunk that K does not fill is done on its own)
  const int c1 = c_all == chunks && a.K % kF32Chunk != 0 && c_all > c0 ? c_all - 1 : c_all;

  auto multiply = [&](const floatx4 (&av)[RT], const floatx4 (&wv)[CT]) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i][k], wv[j][k], acc[i][j], 0, 0, 0);
  };
  floatx4 av[U][RT], wv[U][CT], av2[U][RT], wv2[U][CT];
  auto fetch = [&](int c, floatx4 (&x)[U][RT], floatx4 (&y)[U][CT]) {
    // a row's neighbouring chunks one after the other: the two halves of a 128-byte line
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int u = 0; u < U; ++u) y[u][j] = *(const floatx4*)(wp[j] + (int64_t)min(c + u, c1 - 1) * kF32Chunk);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int u = 0; u < U; ++u) x[u][i] = *(const floatx4*)(ap[i] + (int64_t)min(c + u, c1 - 1) * kF32Chunk);
  };
  auto use = [&](int c, const floatx4 (&x)[U][RT], const floatx4 (&y)[U][CT]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c + u < c1) multiply(x[u], y[u]);
  };
  if (c0 < c1) {
    fetch(c0, av, wv);
    for (int c = c0; c < c1; c += 2 * U) {
      fetch(min(c + U, c1 - 1), av2, wv2);
      use(c, av, wv);
      if (c + U >= c1) break;
      fetch(min(c + 2 * U, c1 - 1), av, wv);
      use(c + U, av2, wv2);
    }
  }
  if (c1 < c_all) {
    const int64_t k = (int64_t)c1 * kF32Chunk;
    const bool in_k = k + k_lane < a.K;   // K is a multiple of 4
#pragma unroll
    for (int j = 0; j < CT; ++j) wv[0][j] = in_k ? *(const floatx4*)(wp[j] + k) : floatx4{};
#pragma unroll
    for (int i = 0; i < RT; ++i) av[0][i] = in_k ? *(const floatx4*)(ap[i] + k) : floatx4{};
    multiply(av[0], wv[0]);
  }

  float* C = (float*)a.C;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][(lane >> 4) * 4 + r][j * 16 + in] = acc[i][j][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * BN; e += 64 * kF32Waves) {
      const int m = e / BN, col = e % BN;
      const int row = row0 + i * 16 + m, n = n0 + col;
      if (row >= row_end || n >= a.N) continue;
      float v = part[0][m][col], u = 0.f;
#pragma unroll
      for (int s = 1; s < kF32Waves; ++s) v += part[s][m][col];
      if (GATED) {
        u = part[0][m][BN + col];
#pragma unroll
        for (int s = 1; s < kF32Waves; ++s) u += part[s][m][BN + col];
        if (a.bias) {
          v += a.bias[n];
          u += a.bias[a.N + n];
        }
        v = gated_output<false>(v, u, a.epilogue, a.act_limit, a.act_alpha);
      } else {
        if (a.bias) v += a.bias[n];
        v = ungated_output(v, a.epilogue == kEpilogueReluSq);
      }
      C[(int64_t)(a.c_index ? a.c_index[row] : row) * a.ldc + n] = v;
    }
  }
}

// 32-bit operands whose rows are whole 16-byte pieces. That depends on the operands' layout
// alone and not on the number of rows: a model's product takes the same kernel in every step.
bool gemm_f32_takes(const GemmArgs& a) {
  return a.in_dtype == kF32 && a.out_dtype == kF32 && a.K % 4 == 0 && a.lda % 4 == 0 &&
         a.w_group_stride % 4 == 0 && ((uintptr_t)a.A | (uintptr_t)a.W) % 16 == 0;
}

template <int RT, int CT, bool GATED>
static void launch(const GemmArgs& a, hipStream_t stream) {
  constexpr int BN = 16 * (GATED ? CT / 2 : CT);
  const int n_tiles = (a.N + BN - 1) / BN;
  const int m_tiles = (a.M + 16 * RT - 1) / (16 * RT) + (a.offsets ? a.groups : 0);
  const int grid = (n_tiles + kXcds - 1) / kXcds * kXcds * m_tiles;
  gemm_f32_kernel<RT, CT, GATED><<<grid, 64 * kF32Waves, 0, stream>>>(a, n_tiles, m_tiles);
}

template <int RT, bool GATED>
static void launch_cols(const GemmArgs& a, int ct, hipStream_t stream) {
  if (ct >= 4) return launch<RT, 4, GATED>(a, stream);
  if (GATED || ct >= 2) return launch<RT, 2, GATED>(a, stream);
  launch<RT, GATED ? 2 : 1, GATED>(a, stream);
}

int gemm_f32(const GemmArgs& a, hipStream_t stream) {
  const bool gated = epilogue_gated(a.epilogue);
  // The tile whose blocks take the least time: blocks beyond one per CU and a part of a last
  // round, times a block's time by its tiles of 16 x 16 and their operands. (Measured a round at
  // K 2,048, us: 1 x 1 11, 1 x 2 13, 2 x 2 19, 1 x 4 20, 2 x 4 29, 4 x 4 54. 173 rows x 2,048
  // features: 31 with 2 x 4 tiles, 42 with 4 x 1, 57 with 4 x 4; 1 x 6,144: 15 with 1 x 2, 19
  // with 1 x 1; 1,024 x 2,048: 109 with 4 x 4, 152 with 2 x 2.)
  const int64_t columns = (int64_t)a.N * (gated ? 2 : 1);
  const int64_t cus = device_cu_count();
  int rt = 1, ct = 1;
  int64_t least = INT64_MAX;
  for (int r = 1; r <= 4; r *= 2)
    for (int c = gated ? 2 : 1; c <= 4; c *= 2) {
      const int64_t m_tiles = (a.M + 16 * r - 1) / (16 * r) + (a.offsets ? a.groups / 2 : 0);
      const int64_t blocks = (columns + 16 * c - 1) / (16 * c) * m_tiles;
      const int64_t cost = (blocks <= cus ? cus : blocks + cus / 3) * (4 * r * c + r + c + 6);
      if (cost < least) least = cost, rt = r, ct = c;
    }
  if (gated) {
    if (rt == 1) launch_cols<1, true>(a, ct, stream);
    else if (rt == 2) launch_cols<2, true>(a, ct, stream);
    else launch_cols<4, true>(a, ct, stream);
  } else {
    if (rt == 1) launch_cols<1, false>(a, ct, stream);
    else if (rt == 2) launch_cols<2, false>(a, ct, stream);
    else launch_cols<4, false>(a, ct, stream);
  }
  NINFER_LAUNCH_CHECK();
  return 0;
}

}  // namespace ninfer
