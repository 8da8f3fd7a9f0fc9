// C = A W^T for many rows (prompt portions): which height of tile a product runs in, and the cut along K.
// The kernel is gemm_tile_direct.hip's. The reference sends these products to rocBLAS, one call per
// expert (src/models/model.hip:406-425, src/ops/linear.hip:21-35).
#include "gemm_tile.h"
#include <type_traits>

namespace ninfer {

constexpr int64_t kSplitMinBytes = 48 << 20;   // GemmArgs::split_min_bytes lowers it for tests

// What a dense product takes in tiles of 128 x 128 (two blocks a CU side by side) and of 256 x 256
// (one a CU, the last round cut into lower blocks), in us on this part. Measured
// on gated products of 128 to 2,048 rows with 2 x 2,816 and 2 x 5,632 features and K 1,024 and
// 2,048; at K 2,048, 128 rows against 256: 640 rows of 2 x 5,632 37 and 44, 800 52 and 45, 1,024 55
// and 47, 1,280 63 and 51, 2,048 94 and 82; 1,280 of 2 x 2,816 32 and 43, 1,531 50 and 43.
static float dense_us_128(int blocks, int cus, int K) {
  float rounds = blocks / (2.f * cus);
  const float last = rounds - floorf(rounds);
  if (rounds > 1.f && last > 0.f && last < 0.3f) rounds += 0.3f - last;   // a short last round is not cheap
  return 2.f + K * (0.006f + 0.014f * rounds);
}
// (Beside other products, which take the CUs that a last round leaves, it is not cut, and the part of a
// round counts as that.)
static float dense_us_256(int tiles, int cus, int K, bool beside) {
  const float round = 9.f + 0.0168f * K;                 // of up to three quarters of the CUs
  if (4 * tiles <= 3 * cus) return round;
  if (beside) return round * 1.22f * (tiles > cus ? (float)tiles / cus : 1.f);
  const int whole = tiles / cus, last = tiles % cus;
  return round * (1.22f * whole + (last == 0 ? 0.f : 4 * last <= cus ? 0.52f : 2 * last <= cus ? 0.62f : 1.22f));
}

// Tile height of a grouped product, by the number of tiles that a CU gets. A row tile's blocks run on one
// XCD (block_to_tile), so that is the number of feature tiles times that of the row tiles an XCD gets: of evenly
// filled groups, each of which has one up to three quarters of a tile's rows and a half filled one more beyond.
// - Up to 40 rows a group on average 64 rows, two blocks a CU, which stream the weights better: 60 groups of
//   2 x 1,408 x 2,048 and 2,048 x 1,408, 34 rows 122 + 63 us against 129 + 66 in tall tiles (60 rows 152 + 81 against
//   136 + 71). With choices that fall off as 1 / rank they are 2 to 10% slower instead, and up to 29% with few groups of many
//   features, where one row tile more is an XCD's second (8 groups of 2 x 14,336 x 4,096, 25 rows: 290 us against 324, so
//   432 against 336): there tall tiles.
// - 128 rows while a CU gets less than the two such tiles that it holds side by side: 16 groups of 2 x 704 x 1,024 and
//   1,024 x 704, 191 rows 23 + 14 us against 28 + 20 in tall tiles; 4 groups of 2,048 x 4,096, 256 rows 42 against 78.
//   From two on tall tiles: 10 groups of 2 x 4,096 x 4,096, 140 rows 138 us against 83; 8 of 4,096 x 14,336, 128 rows 352
//   against 229; 32 of 2 x 256 x 768, 512 rows 37 against 26.
// - The tall tile loads and multiplies only the 32-row blocks that hold rows.
static int grouped_rows_of(const GemmArgs& a, int w_rows, int cus) {
  auto per_cu = [&](int tm, int tn) {
    const float filled = (float)a.M / a.groups / tm, row_tiles = a.groups * (filled <= 0.75f ? 1.f : filled + 0.5f);
    return ceilf(row_tiles / kXcds) * ((w_rows + tn - 1) / tn) * kXcds / cus;
  };
  if (a.M / a.groups <= 40) return a.groups <= 16 && per_cu(256, 256) >= 3.f ? kGroupedTileRows : 64;
  return per_cu(128, 128) < 2.f ? 128 : kGroupedTileRows;
}

// Tile height of a dense product: 64 rows while taller tiles would leave CUs without a block, else 128 or 256 by
// an estimate of both times (dense_us_128, dense_us_256); where one output a feature is stored instead of
// one of two, as many tall tiles as CUs decide for them too, whose stores cost less (32-bit outputs, K
// 1,024: 1,531 x 12,800 56 us in tiles of 256 and 68 in those of 128, 3,000 x 6,144 53 and 66). force_kernel
// (tests) forces 64, 128 or 256 rows.
static int tile_rows_of(const GemmArgs& a) {
  if (gemm_tile_far(a)) return 128;
  if (a.force_kernel >= 1 && a.force_kernel <= 3) return 32 << a.force_kernel;
  const bool gated = epilogue_gated(a.epilogue);
  const int n_units = gated ? 2 * a.N : a.N;   // W rows
  auto blocks = [&](int tm, int tn) { return ((a.M + tm - 1) / tm) * ((n_units + tn - 1) / tn); };
  const int cus = device_cu_count(), low = blocks(128, 128), tall = blocks(256, 256);
  if (a.offsets) return grouped_rows_of(a, n_units, cus);
  if (a.M <= 64 || low < cus) return 64;   // (no taller than the rows there are)
  if (a.M <= 128) return 128;
  return (!gated && tall >= cus) || dense_us_256(tall, cus, a.K, a.beside) < dense_us_128(low, cus, a.K) ? 256 : 128;
}

int gemm_tile(const GemmArgs& a, hipStream_t stream) {
  return gemm_mid_takes(a) ? gemm_mid(a, stream) : gemm_tile_rows(a, tile_rows_of(a), stream);
}

// out[m][n] = sum over the parts, in their order, of ws[z][m][n] (+ bias[n]); four features a thread.
template <typename TC>
__global__ void sum_parts_kernel(const float* __restrict__ ws, int parts, int M, int N,
                                 const float* __restrict__ bias, TC* __restrict__ out, int ldc) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;   // quad of features
  const int quads = N / 4;
  if (q >= (int64_t)M * quads) return;
  const int m = q / quads, n = 4 * (q % quads);
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int z = 0; z < parts; ++z) {
    const float4 v = *(const float4*)(ws + ((int64_t)z * M + m) * N + n);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  if (bias) {
    s.x += bias[n]; s.y += bias[n + 1]; s.z += bias[n + 2]; s.w += bias[n + 3];
  }
  const float v[4] = {s.x, s.y, s.z, s.w};
  store_quad(out + (int64_t)m * ldc + n, v);
}

// The cut along K pays where the tiles of the output (64 x 128, or 128 x 128 beyond 128 rows)
// are fewer than the CUs, K is long, and the weights are many enough (48 MB and more) that
// their stream outweighs the second launch that adds the parts up (measured against the
// library's product at 3584 x 20480: 41 against 99 us at 64 rows, 111 against 226 at 512;
// no gain at 25 MB; at 8192 x 8192 and 384 rows the library is faster, hence K >= 2 N beyond
// 128 rows). Parts so that about two blocks per CU exist, each with at least four k tiles,
// and no part is empty.
int gemm_split_parts(const GemmArgs& a) {
  if (a.offsets || a.epilogue != kEpilogueNone || !a.workspace || !gemm_tile_takes(a)) return 1;
  if (a.M <= 32 || a.M > 512 || a.N % 4 || a.ldc % 4 || ((uintptr_t)a.C & 15)) return 1;
  if ((int64_t)a.N * a.K * 2 < (a.split_min_bytes > 0 ? a.split_min_bytes : kSplitMinBytes)) return 1;
  if (a.M > 128 && a.K < 2 * a.N) return 1;   // beyond 128 rows only where K is long against N
  const int cus = device_cu_count(), tk = 64;
  const int tm = a.M > 128 ? 128 : 64;
  const int tiles = ((a.M + tm - 1) / tm) * ((a.N + 127) / 128), nk = a.K / tk;
  if (tiles >= cus) return 1;
  const int64_t fit = a.workspace_floats / ((int64_t)a.M * a.N);
  int parts = (int)min((int64_t)min(min(16, 2 * cus / tiles), nk / 4), fit);
  if (parts < 2) return 1;
  const int per = (nk + parts - 1) / parts;
  return (nk + per - 1) / per;
}

int gemm_split(const GemmArgs& a, hipStream_t stream) {
  const int parts = gemm_split_parts(a);
  NINFER_REQUIRE(parts >= 2, "gemm: this product is not cut along K");
  GemmArgs b = a;
  b.C = a.workspace;
  b.ldc = a.N;
  b.out_dtype = kF32;
  b.bias = nullptr;
  b.k_parts = parts;
  int rc = gemm_tile_rows(b, a.M > 128 ? 128 : 64, stream);
  if (rc) return rc;
  const int64_t quads = (int64_t)a.M * (a.N / 4);
  const unsigned blocks = (unsigned)((quads + 255) / 256);
  if (a.out_dtype == kF32)
    sum_parts_kernel<float><<<blocks, 256, 0, stream>>>(a.workspace, parts, a.M, a.N, a.bias,
                                                        (float*)a.C, a.ldc);
  else
    sum_parts_kernel<bf16><<<blocks, 256, 0, stream>>>(a.workspace, parts, a.M, a.N, a.bias,
                                                       (bf16*)a.C, a.ldc);
  NINFER_LAUNCH_CHECK();
  return 0;
}

}  // namespace ninfer

// Rows of the tiles that ninfer_gemm would run a product of many rows in that is not one round of gemm_mid's.
extern "C" int ninfer_gemm_tile_rows(const ninfer::GemmArgs* args) { return ninfer::tile_rows_of(*args); }
