// C = A W^T (+ bias, an activation, or gated) for a dense product of 17 to 512 rows (more than that for a router's few
// features): too many for a block that owns all of them, too few to pay for the tiles of the many-row kernel.
//
// A block owns 32 rows of A and up to 32 rows of W: two sets of up to 16 (of a gated product a set of the gate's and
// the same of the other half's), or one set. Its 8 waves (a router's 8 or 16) split K, each a contiguous part walked in
// chunks of 128;
// partial tiles meet in LDS and are summed in wave order, so a row's result depends neither on timing nor on the other
// rows. Both operands are loaded as whole 128-byte lines (8 rows an instruction) and reach the matrix instruction's
// layout through 2 KB of LDS per wave. The row parts of a feature tile lie side by side on one XCD
// (line_tile), so that the weights come from HBM once.
//
// What bounds it is the operands' way into the CU: K 2,048, 64 rows, 2,048 features, a block of 32 rows and 16
// features loads 196 KB. Loaded 64 bytes of a row at a time, as the instruction wants them, the rows of A cost most of
// the time; us in launches back to back that way and so: 2,048 features 7.8 and 6.1 (K 5,632 16.6 and 11.5), 6,144
// 14.9 and 11.1, 2 x 5,632 21.1 and 16.7. Other shapes of block, 2,048 features: 16 rows and 32 features 6.1, 64 rows
// and 8 features 7.4, 16 waves 6.2; 6,144: 64 rows and 24 features 12.0; 2 x 5,632: 64 rows and 2 x 22 18.2.
// The reference sends all products of this size to the library (src/ops/linear.hip:21-35).
#include "gemm.h"
#include <type_traits>

namespace ninfer {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRowsMax = 512;
constexpr int kRowsTiles = 2, kRowsOfBlock = 16 * kRowsTiles;

static int rows_parts(const GemmArgs& a) { return (a.M + kRowsOfBlock - 1) / kRowsOfBlock; }

struct RowsPlan {
  int sets;     // sets of W rows in a block: 1 or 2
  int rows;     // W rows of a set, up to 16
  int waves;    // 8 or 16
  int grid_x;   // feature tiles
  int grid_y;   // row parts
};

// AGAIN: another block reads the same weights (they are to stay in L2)
template <int WAVES, int SETS, bool GATED, bool AGAIN, typename TC>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_rows_kernel(GemmArgs a, RowsPlan p) {
  static_assert(!GATED || SETS == 2, "a gated product's two sets");
  constexpr int RT = kRowsTiles, GROUPS = GATED ? 1 : SETS;   // groups of features
  // partial tiles: [wave][set][row tile][token 16][feature 16]; the first bytes are the waves' 2 KB
  // each while the K range is walked
  __shared__ __attribute__((aligned(16))) float red[WAVES * SETS * RT * 256];
  unsigned char* stage = (unsigned char*)red;
  static_assert(WAVES * SETS * RT * 1024 >= WAVES * 2048, "the lines fit in the partial tiles' memory");
  const int slot = blockIdx.x / kXcds;   // line_tile: the row parts of a feature tile on one XCD
  // (few features: the feature tiles of a row part, so that the rows come from HBM once)
  const bool few = a.N <= 128;
  const int by = few ? slot / p.grid_x * kXcds + blockIdx.x % kXcds : slot % p.grid_y;
  const int bx = few ? slot % p.grid_x : slot / p.grid_y * kXcds + blockIdx.x % kXcds;
  if (bx >= p.grid_x || by >= p.grid_y) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, j = lane >> 4;
  const int n0 = bx * p.rows * GROUPS, row0 = by * kRowsOfBlock, K = a.K;
  // both operands as the loads see them: lane l reads 16 bytes of row 8 q + l / 8 at byte 16 (l % 8) of a 128-byte
  // piece. Rows that are not there are the last one again (never written); W rows beyond a set's are not loaded.
  const bf16* wline[SETS][2];
  const bf16* xline[RT][2];
  bool w_valid[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int R = 8 * q + (lane >> 3);
    w_valid[q] = R < p.rows;
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      const int n = min(n0 + (GATED ? 0 : s * p.rows) + R, a.N - 1) + (GATED && s ? a.N : 0);
      wline[s][q] = (const bf16*)a.W + (int64_t)n * K + 8 * (lane & 7);
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
      xline[t][q] = (const bf16*)a.A + (int64_t)min(row0 + 16 * t + R, a.M - 1) * a.lda + 8 * (lane & 7);
  }
  f32x4 acc[SETS][RT];
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // this wave's 2 KB of LDS: 16 rows of 128 bytes, the 16-byte units of row R in the order
  // u ^ (R % 8), so that the writes (a row per 8 lanes) and the fragment reads (lane (r, j):
  // row r, unit 4 i + j) both spread evenly over the banks
  unsigned char* my_stage = stage + wave * 2048;
  const int st_write = ((lane >> 3) * 128) + 16 * ((lane & 7) ^ ((lane >> 3) & 7));   // + 1024 q
  const int st_read = r * 128;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const int chunks = K / 128, per_wave = (chunks + WAVES - 1) / WAVES;
  const int c_end = min((wave + 1) * per_wave, chunks);
  for (int c = wave * per_wave; c < c_end; ++c) {
    bf16x8 wl[SETS][2][2], x[RT][2][2];   // [set or row tile][half of the chunk][q]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const bf16x8* at = (const bf16x8*)(wline[s][q] + c * 128 + h * 64);
          wl[s][h][q] = !w_valid[q] ? zero : AGAIN ? *at : stream_load(at);
        }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q) x[t][h][q] = *(const bf16x8*)(xline[t][q] + c * 128 + h * 64);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 xf[RT][2];
#pragma unroll
      for (int t = 0; t < RT; ++t) {
#pragma unroll
        for (int q = 0; q < 2; ++q) *(bf16x8*)(my_stage + st_write + 1024 * q) = x[t][h][q];
#pragma unroll
        for (int i = 0; i < 2; ++i) xf[t][i] = *(const bf16x8*)(my_stage + st_read + 16 * ((4 * i + j) ^ (r & 7)));
      }
#pragma unroll
      for (int s = 0; s < SETS; ++s) {
#pragma unroll
        for (int q = 0; q < 2; ++q) *(bf16x8*)(my_stage + st_write + 1024 * q) = wl[s][h][q];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const bf16x8 wf = *(const bf16x8*)(my_stage + st_read + 16 * ((4 * i + j) ^ (r & 7)));
#pragma unroll
          for (int t = 0; t < RT; ++t)
            acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[t][i], acc[s][t], 0, 0, 0);
        }
      }
    }
  }

  __syncthreads();   // every wave is done with its lines
  // the accumulator holds out[feature 4 j + v][token r]; stored as [token][feature]
#pragma unroll
  for (int s = 0; s < SETS; ++s)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[((wave * SETS + s) * RT + t) * 256 + r * 16 + 4 * j + v] = acc[s][t][v];
  __syncthreads();
  for (int idx = threadIdx.x; idx < GROUPS * RT * 256; idx += WAVES * 64) {
    const int gt = idx >> 8, g = gt / RT, t = gt % RT, m = (idx >> 4) & 15, f = idx & 15;
    const int row = row0 + 16 * t + m, col = n0 + g * p.rows + f;
    if (row >= a.M || f >= p.rows || col >= a.N) continue;
    float v = 0.f, u = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      v += red[((w * SETS + g) * RT + t) * 256 + (idx & 255)];
      if (GATED) u += red[((w * SETS + 1) * RT + t) * 256 + (idx & 255)];
    }
    if (GATED) {
      if (a.bias) {
        v += a.bias[col];
        u += a.bias[a.N + col];
      }
      v = gated_output<true>(v, u, a.epilogue, a.act_limit, a.act_alpha);
    } else {
      if (a.bias) v += a.bias[col];
      v = ungated_output(v, a.epilogue == kEpilogueReluSq);
    }
    ((TC*)a.C)[(int64_t)row * a.ldc + col] = from_f32<TC>(v);
  }
}

// Which products. The more features beside few rows, the more the rows' ways into all the blocks cost against a
// tile that keeps them (or the few-row kernel, whose blocks all read the weights again); us here and there:
// - 17 to 32 rows, against the few-row kernel: 2,048 features 5.8 and 5.7, 3,072 6.0 and 8.0, 6,144 8.7 and 11.4, 32,000
//   27 and 42; gated 2 x 1,408 7.3 and 6.8, 2 x 2,816 (K 1,024) 5.8 and 6.6, 2 x 20,480 (K 3,584) 52 and 73.
// - 33 rows and more, against the library's product: 2,048 features, 64 rows 6.0 and 8.9, 128 rows 7.0 and 8.3 (K 5,632
//   12.1 and 17.9, 14.7 and 15.9); 6,144 64 rows 12.1 and 12.7, 128 15.7 and 14.9.
//   Against tiles of 64 rows: gated 2 x 5,632 64 rows 17.7 and 20.8, 80 22.0 and 19.0; 2 x 2,816 128 rows 9.8 and
//   11.6; 2 x 1,408 256 rows 14.5 and 18; 2 x 20,480 64 rows 87 and 72; a few hundred features 5.2 and 13. Of K 512 to 896,
//   where a second round of blocks costs more than it multiplies, gated 2 x 4,096 64 rows 5.7 and 6.7, 96 7.4 and 6.5; 2 x 3,072
//   of K 768, 96 rows 8.5 and 7.6; K 1,024 9.9 and 10.8. (Below 512 a launch is a few us in either: K 384 7.3 and 5.9.)
// - beyond 128 rows, against the library's product: 2,048 features 160 rows 9.9 and 9.1; 1,024 (K 2,816) 256 rows 7.7 and
//   8.5; 768 256 rows 6.4 and 8.4, 384 9.5 and 9.1.
// - up to 128 features (a router's), against the few-row kernel, whose rows came 64 bytes at a time: 61 features, K 2,048,
//   512 rows 5.5 and 6.1 alone, but 8.6 in either beside the shared expert's products; 2,048 rows 6.3 and 13.2, 4,096 8.7
//   and 22.7.
bool gemm_skinny_rows_takes(const GemmArgs& a) {
  if (a.offsets || a.a_index || a.c_index || a.groups > 1 || a.force_kernel || a.in_dtype != kBF16 || a.M <= 16 ||
      a.K % 128 || a.lda % 8 || (uintptr_t)a.A % 16 || (uintptr_t)a.W % 16)
    return false;
  const bool gated = epilogue_gated(a.epilogue);
  const int64_t w_rows = (int64_t)a.N * (gated ? 2 : 1);
  if (a.M <= 32) return w_rows > (gated ? 4096 : 2560);
  if (a.N <= 128) return !gated && a.M > kRowsMax;
  const int most = !gated ? a.M <= 128 ? 16384 : 8192 : a.K >= 512 && a.K < 1024 ? 16384 : 24576;
  return a.M <= kRowsMax && w_rows * rows_parts(a) <= most;
}

// Features a block, so that the blocks on an XCD (the row parts of its feature tiles) fill rounds of one a CU: 6,144
// features, 64 rows 512 blocks of 24 features 11.1 us, 384 of 32 12.1, 768 of 16 12.1; 2,048 features, 80 rows 237
// blocks of 26 6.5 us, 258 of 24 9.1.
static RowsPlan plan_rows(const GemmArgs& a) {
  RowsPlan p;
  const bool gated = epilogue_gated(a.epilogue);
  const int most = gated ? 16 : 32, slots = max(1, device_cu_count() / kXcds);
  p.grid_y = rows_parts(a);
  int f = most;
  if (a.N <= 128) f = a.N <= 16 || (int64_t)p.grid_y * ((a.N + 15) / 16) <= 2 * device_cu_count() ? 16 : 32;
  else for (int rounds = 1; rounds <= 8; ++rounds) {
    const int tiles = slots * rounds / p.grid_y * kXcds;   // feature tiles on all XCDs
    if (tiles > 0 && (a.N + tiles - 1) / tiles <= most) {
      f = gated ? max(8, (a.N + tiles - 1) / tiles) : max(16, (a.N + tiles - 1) / tiles);
      break;
    }
  }
  p.sets = gated || f > 16 ? 2 : 1;
  p.rows = gated || p.sets == 1 ? f : (f + 1) / 2;
  // (up to 128 features: as many waves as the few-row kernel has of a K of 1,024 and more while its blocks are fewer than
  // eight a CU, so that a router's sums are the same in either; it has four of a shorter K or with more blocks. 16 go with one
  // set: two sets are for blocks beyond two a CU)
  const int row_tiles = (a.M + 15) / 16;
  p.waves = a.N <= 128 && (a.N + 15) / 16 * row_tiles < device_cu_count() && a.K >= 2048 ? 16 : 8;
  const int of_block = gated ? p.rows : p.sets * p.rows;
  p.grid_x = (a.N + of_block - 1) / of_block;
  return p;
}

int gemm_skinny_rows(const GemmArgs& a, hipStream_t stream) {
  NINFER_REQUIRE(gemm_skinny_rows_takes(a), "gemm: not a product for blocks of 32 rows");
  const RowsPlan p = plan_rows(a);
  const int on_xcds = a.N <= 128 ? p.grid_y : p.grid_x, beside = a.N <= 128 ? p.grid_x : p.grid_y;
  const int64_t blocks = (int64_t)((on_xcds + kXcds - 1) / kXcds) * kXcds * beside;
  NINFER_REQUIRE(blocks < (1LL << 31), "gemm: %lld blocks are too many", (long long)blocks);
  const dim3 grid((unsigned)blocks), block(p.waves * 64);
  auto launch = [&](auto again, auto tc) {
    constexpr bool AGAIN = decltype(again)::value;
    typedef decltype(tc) TC;
    if (epilogue_gated(a.epilogue)) gemm_skinny_rows_kernel<8, 2, true, AGAIN, TC><<<grid, block, 0, stream>>>(a, p);
    else if (p.waves == 16) gemm_skinny_rows_kernel<16, 1, false, AGAIN, TC><<<grid, block, 0, stream>>>(a, p);
    else if (p.sets == 2) gemm_skinny_rows_kernel<8, 2, false, AGAIN, TC><<<grid, block, 0, stream>>>(a, p);
    else gemm_skinny_rows_kernel<8, 1, false, AGAIN, TC><<<grid, block, 0, stream>>>(a, p);
  };
  auto typed = [&](auto again) {
    if (a.out_dtype == kF32) launch(again, float{});
    else launch(again, bf16{});
  };
  if (p.grid_y > 1) typed(std::true_type{});
  else typed(std::false_type{});
  NINFER_LAUNCH_CHECK();
  return 0;
}

}  // namespace ninfer
