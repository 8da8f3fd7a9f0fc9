// C = A W^T (+ bias, an activation, or gated) for a dense bf16 product whose output is one round of tiles on the GPU: tens
// to some 2,000 rows of hundreds to thousands of features. Tiles of nine sizes, 32 x 64 to 192 x 128 and 128 x 192 (rows of A x
// rows of W), one block of eight waves to a CU; the smallest of which a round holds all is taken.
//
// Every output is one chain of sums along K, 32 numbers an instruction, as in the taller tiles and in the library's products
// that are not cut along K: the same bits, whichever of them a product's size sends it to. (Groups of waves that took k tiles
// in turn and added their sums at the end were no faster, and moved a model's logits by as much as bfloat16's rounding does.)
//
// What bounds a lone block is its way from L2 into LDS: some 80 GB/s a CU for loads straight into LDS (37 bytes a
// clock), so a tile's time goes with its rows of A and W together, whatever it multiplies, and four waves that wait for each
// other at a barrier per k tile leave even that unused (64 x 128 in four waves 18 us at K 2,048, so 12.5). A stage is
// therefore one, two or four k tiles, the more the lower the tile, with one barrier for all of them, and all eight waves share
// each. Stages lie in a ring, all of it asked for ahead: when a wave passes the barrier of stage s, stage s + 1 has landed for
// every wave and every wave holds the last fragments of stage s in registers, so its place takes stage s + NB. The fragments
// of a half k tile are read while those of the half before are multiplied.
// Against the library's product, us, with weights that come from HBM (host time 9 us a call against 24), K 2,048: 2,048
// features, 256 rows 8.4 and 9.9, 512 10.1 and 11.5, 1,280 17.4 and 18.8, 2,048 19.9 and 22.5; 4,096, 160 rows 11.7 and 16.6, 768 20.5 and
// 23.2, 1,531 27.9 and 30.7; 6,144, 256 rows 15.9 and 23.9, 512 22.0 and 24.6, 1,024 30.4 and 32.3; 1,024 features of K 1,024,
// 512 rows 6.2 and 8.6; of K 2,816 10.0 and 12.0. (With groups in turn 512 rows of 2,048 features 12.0, 256 of 6,144 15.5.)
// Against tiles of 64 and 128 rows in four waves, gated: 2 x 2,816 features, 192 rows 15.3 and 19.5, 512 21.9 and 25.1; 2 x 5,632,
// 256 rows 23.5 and 26.2, 384 27.9 and 31.3; 2 x 1,408, 1,024 rows 20.8 and 23.9.
// The reference sends these products to rocBLAS (src/ops/linear.hip:21-35).
#include "gemm_tile.h"

namespace ninfer {

template <int N> __device__ __forceinline__ void mid_wait() {   // until at most N loads of this wave are under way
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// The same for n stages' loads of NL each, n < NB (beyond: for all but NB - 1).
template <int NL, int NB> __device__ __forceinline__ void mid_wait_stages(int n) {
  if (NB > 3 && n >= 3) mid_wait<3 * NL>();
  else if (NB > 2 && n >= 2) mid_wait<2 * NL>();
  else if (n >= 1) mid_wait<NL>();
  else mid_wait<0>();
}

// TM x TN: the tile, by WM x WN waves (over rows of W and of A). A stage is KT k tiles of 64, NB of them in LDS.
template <int TM, int TN, int WM, int WN, int KT, int NB, bool GATED, typename TC>
__global__ __launch_bounds__(512, 2) void gemm_mid_kernel(GemmArgs a, int m_tiles, int n_tiles) {
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass does not know buffer resources)
  static_assert(WM * WN == 8 && NB >= 2 && NB <= 4, "eight waves");
  constexpr int FI = TN / WM / 16, FJ = TM / WN / 16;     // 16-row blocks of W and of A of a wave
  static_assert(!GATED || FI % 2 == 0, "a wave's blocks of W are gate rows, then their up rows");
  constexpr int ROW = 128;                                // bytes of a staged row: a k tile of 64
  constexpr int X_BYTES = TM * ROW, SUB = (TM + TN) * ROW, STAGE = KT * SUB;
  constexpr int PER_SUB = SUB / 1024, X_PIECES = X_BYTES / 1024;   // pieces of 1 KB, 8 rows: a wave's load
  constexpr int NL = STAGE / 1024 / 8;                    // loads of a wave and stage
  static_assert(STAGE / 1024 % 8 == 0, "whole loads");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  int bx, by;
  dense_tile(spread_over_xcds(blockIdx.x, m_tiles * n_tiles), m_tiles, n_tiles, bx, by);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int K = a.K, N = a.N;
  constexpr int OUT = GATED ? TN / 2 : TN;
  const int row0 = bx * TM, out0 = by * OUT, rows_here = min(TM, a.M - row0);

  // Load i of wave w fills piece 8 i + w of a stage: k tile (8 i + w) / PER_SUB of it, the lane at row lane / 8 of the piece.
  // Of a staged row the 16-byte chunk c lies at c ^ ((row / 2) % 8), chosen on the global side, so that the 16 rows of a
  // fragment read fall into different columns of the banks. Rows that are not there read the last one that is.
  const bf16* W = (const bf16*)a.W + (int64_t)out0 * K;
  unsigned off[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int p = (8 * i + wave) % PER_SUB;
    const int r = (p < X_PIECES ? p : p - X_PIECES) * 8 + (lane >> 3);
    unsigned row_bytes;
    if (p < X_PIECES) {
      row_bytes = (unsigned)min(r, rows_here - 1) * (unsigned)(2 * a.lda);
    } else {
      const int n = staged_w_row<TN, WM, GATED>(r, out0, N);
      row_bytes = (unsigned)((n < N ? n : n - N) - out0) * (unsigned)(2 * K);
    }
    off[i] = row_bytes + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  const auto x_res = __builtin_amdgcn_make_buffer_rsrc((void*)((const bf16*)a.A + (int64_t)row0 * a.lda), 0, 0xffffffffu, 0x00020000);
  const auto w_res = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, 0xffffffffu, 0x00020000);
  const auto up_res = __builtin_amdgcn_make_buffer_rsrc((void*)(W + (GATED ? (int64_t)N * K : 0)), 0, 0xffffffffu, 0x00020000);
  typedef __attribute__((address_space(3))) void* lptr;
  const int nk = K / 64, stages = (nk + KT - 1) / KT;
  auto issue = [&](int s, int at) {
    unsigned char* buf = smem + at + wave * 1024;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int piece = 8 * i + wave, p = piece % PER_SUB;
      const int k = min(s * KT + piece / PER_SUB, nk - 1) * ROW;   // (a last stage that K does not fill: the last k tile again)
      if (p < X_PIECES)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_res, (lptr)(buf + i * 8192), 16, off[i], k, 0, 0);
      else if (GATED && (p - X_PIECES) * 8 % (TN / WM) >= TN / WM / 2)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(up_res, (lptr)(buf + i * 8192), 16, off[i], k, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_res, (lptr)(buf + i * 8192), 16, off[i], k, 0, 0);
    }
  };

  f32x4 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int lr = lane & 15, lk = lane >> 4, sw = (lr >> 1) & 7;
  const int x_lane = (wn * (TM / WN) + lr) * ROW, w_lane = X_BYTES + (wm * (TN / WM) + lr) * ROW;
  const int chunk[2] = {16 * (lk ^ sw), 16 * ((4 + lk) ^ sw)};
  bf16x8 wf[2][FI], xf[2][FJ];
  auto read = [&](int h, int at) {   // half h of the k tile at `at`
    const unsigned char* p = smem + at + chunk[h];
#pragma unroll
    for (int i = 0; i < FI; ++i) wf[h][i] = *(const bf16x8*)(p + w_lane + i * 16 * ROW);
#pragma unroll
    for (int j = 0; j < FJ; ++j) xf[h][j] = *(const bf16x8*)(p + x_lane + j * 16 * ROW);
  };
  auto multiply = [&](int h) {
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int i = 0; i < FI; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][i], xf[h][j], acc[i][j], 0, 0, 0);
  };
  auto next = [](int at) { return at == (NB - 1) * STAGE ? 0 : at + STAGE; };
  for (int s = 0; s < NB && s < stages; ++s) issue(s, s * STAGE);
  mid_wait_stages<NL, NB>(min(NB, stages) - 1);
  __builtin_amdgcn_s_barrier();
  read(0, 0);
  int at = 0, s = 0;
  auto most_of_stage = [&]() {   // all but the last half k tile, whose fragments are in registers
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      read(1, at + u * SUB);
      multiply(0);
      if (u + 1 == KT) break;
      read(0, at + (u + 1) * SUB);
      multiply(1);
    }
  };
  for (; s + NB < stages; ++s) {
    most_of_stage();
    mid_wait<(NB - 2) * NL>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read(0, next(at));
    issue(s + NB, at);
    multiply(1);
    at = next(at);
  }
  for (; s + 1 < stages; ++s) {   // nothing left to ask for
    most_of_stage();
    mid_wait_stages<NL, NB>(stages - s - 2);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read(0, next(at));
    multiply(1);
    at = next(at);
  }
#pragma unroll
  for (int u = 0; u < KT; ++u) {
    if (s * KT + u >= nk) break;   // (a last stage that K does not fill)
    if (u) read(0, at + u * SUB);
    read(1, at + u * SUB);
    multiply(0);
    multiply(1);
  }
  __syncthreads();   // every wave has read its last fragments: the ring becomes the epilogue's place
  static_assert(WM * WN * FJ * 16 * FI * 32 <= NB * STAGE, "the epilogue's stage fits the ring");
  auto row_of = [&](int l) { return l; };
  const int tok0 = wn * (TM / WN), feat0 = out0 + wm * (OUT / WM);
  if constexpr (FI % 3 == 0)   // (rows of the epilogue's stage are powers of two)
    write_accumulators<FI, FJ, GATED, TC>(a, acc, tok0, row0, rows_here, feat0, row_of);
  else
    write_tile<FI, FJ, GATED, TC>(a, acc, smem + wave * (FJ * 16 * FI * 32), tok0, row0, rows_here, feat0, row_of);
#endif
}

// The tiles in the order of what a round of each takes (K 1,024 and 4,096, us: 6.2 and 15.4, 7.0 and 19.8, 8.5 and 23.0, 8.0 and
// 23.6, 9.2 and 28, 10.7 and 34, 11.9 and 36, 14.2 and 45, 15.2 and 46). A second round costs 0.8 of the first and more, with which no tile
// beats the taller ones or the library's: products of more than a round of the largest tile are not taken.
struct MidTile { int rows, w_rows; bool gated; };
static const MidTile kMidTiles[] = {{32, 64, false}, {64, 64, true},   {96, 64, false},  {64, 96, false}, {128, 64, true},
                                    {192, 64, true}, {128, 128, true}, {192, 128, true}, {128, 192, false}};
constexpr int kMidTileCount = sizeof(kMidTiles) / sizeof(kMidTiles[0]);

static int mid_tiles(const GemmArgs& a, const MidTile& t) {
  const int64_t w_rows = epilogue_gated(a.epilogue) ? 2ll * a.N : a.N;
  return (int)min((int64_t)(1 << 30), (int64_t)((a.M + t.rows - 1) / t.rows) * ((w_rows + t.w_rows - 1) / t.w_rows));
}
static int mid_tile(const GemmArgs& a) {
  for (int i = 0; i < kMidTileCount; ++i)
    if ((!epilogue_gated(a.epilogue) || kMidTiles[i].gated) && mid_tiles(a, kMidTiles[i]) <= device_cu_count()) return i;
  return -1;
}

// Does a product take less in the four-wave tiles of 64 x 128, of which a CU holds two, or as long? Measured on products that are gated
// or have a bias or 32-bit outputs, some 2,000 sizes (us here and there; elsewhere none of more than 2% takes longer here, but for single
// sizes whose rows of W lie badly in memory):
// - 192 x 64 leaves CUs without a block, and rows of A without a number, where those tiles are one a CU as well: 2 x 4,296 features
//   of K 1,280, 144 rows 15.3 and 13.1; 10,432 of K 1,792, 160 rows 20.0 and 17.8 (100 sizes of up to 192 rows 0.85 to 0.96 of their
//   speed). From three quarters of their number and a K beyond 2,048 on its blocks are the faster ones: 2 x 2,904 of K 4,800, 305 rows
//   36.2 and 39.0.
// - 128 x 128 for up to 64 rows: 32,000 features of K 1,024, 64 rows 20.4 and 16.0, 33 rows 16.5 and 15.4; K 2,048 34.4 and 34.8.
// - 128 x 128 and 128 x 192 of few rows more, which fill the GPU: 31,264 of K 1,024, 65 rows 20.1 and 17.3; 47,352 of K 896, 33 rows 23.8
//   and 20.0; but 28,456 of K 1,216, 66 rows 17.5 and 20.5, 36,112, 64 rows 22.0 and 26.9.
static bool low_tiles_beat(const GemmArgs& a, const MidTile& t) {
  const int cus = device_cu_count(), here = mid_tiles(a, t), low = mid_tiles(a, {64, 128, true});
  if (t.rows == 192 && t.w_rows == 64) return low <= cus && (4 * here < 3 * low || a.K <= 2048);
  if (t.rows != 128 || t.w_rows == 64) return false;
  return (a.M <= 64 && t.w_rows == 128) || (a.M <= 72 && a.K <= 1536 && 16 * here >= 15 * cus);
}

// Dense products of more than 32 rows that are one round of tiles, and no faster in lower ones. (Fewer rows go to the few-row kernel.)
bool gemm_mid_takes(const GemmArgs& a) {
  if (a.offsets || a.a_index || a.c_index || a.groups > 1 || a.k_parts > 1 || a.force_kernel || a.M <= 32 || a.N < 64 ||
      !gemm_tile_takes(a))
    return false;
  const int tile = mid_tile(a);
  return tile >= 0 && !low_tiles_beat(a, kMidTiles[tile]);
}

// Of a plain product that gemm_mid takes, which the library has otherwise: is it no slower here? Up to K 4,032 it is (2,400 sizes of
// 33 to 2,000 rows: 1.2 of the library's speed on average, 0.96 and more but for one in forty, half of them of a few hundred features, us
// in the library and here: 192 of K 832, 768 rows 5.0 and 5.8, 256 of K 2,624, 33 rows 7.4 and 8.7, 7,296 of K 3,712, 380 rows, where the
// library's time jumps, 31.4 and 35.3; against 15 us of the host's time). A longer K costs a lone block most
// where its rows of W are few for the weights there are, and the library cuts products of few blocks along K; K 4,096 to 8,192:
// - 32 x 64: 1,216 features of K 5,632, 338 rows 17.2 and 15.9; but 1,600 of K 5,120, 276 rows 19.7 and 21.1, 2,688 of K 7,168, 140
//   rows 22.3 and 25.2. From K 5,120 on it takes longer only where its tiles are at most half of the CUs: 320 of K 5,376, 768 rows
//   12.3 and 14.6, 1,344 of K 7,616, 45 rows 19.0 and 25.7; 1,024 of K 6,336, 507 rows 28.0 and 17.5.
// - 64 x 64: 2,048 of K 5,632, 335 rows 25.3 and 23.1, 512 27.8 and 27.8; but 2,176 of K 6,144, 384 rows 28.0 and 30.2.
// - 192 x 64: 1,600 of K 5,120, 1,294 rows 36.9 and 43.0, 1,920 of K 5,632, 1,482 rows 43.6 and 46.9 (and 2,560 of K 5,632, 806
//   rows, 47.7 and 40.8: the library's times jump).
// - 128 x 128: 2,048 of K 5,632, 2,048 rows 58.7 and 55.2; but 6,400 of K 4,608, 473 rows 38.8 and 44.8.
// - the others 0.93 to 1.7 of its speed.
// Beyond K 8,192 the library cuts more products along K: 1,408 features of K 14,336, 173 rows 38.9 and 43.0.
bool gemm_mid_beats_library(const GemmArgs& a) {
  if (a.K < 4096) return true;
  const int tile = mid_tile(a);
  if (a.K > 8192 || tile < 0) return false;
  const MidTile& t = kMidTiles[tile];
  if (t.w_rows == 64 && t.rows == 32)
    return a.K == 4096 || (a.N < 1536 && (a.K < 5120 || 2 * mid_tiles(a, t) > device_cu_count()));
  if (t.w_rows == 64 && t.rows == 64) return a.K < 6144;
  if (t.w_rows == 64 && t.rows == 192) return false;
  return t.w_rows != 128 || t.rows != 128 || a.M > 512;
}

template <int TM, int TN, int WM, int WN, int KT, int NB>
static int launch_mid(const GemmArgs& a, hipStream_t stream) {
  constexpr int LDS = KT * (TM + TN) * 128 * NB;
  const bool gated = epilogue_gated(a.epilogue);
  const int w_rows = gated ? 2 * a.N : a.N, m_tiles = (a.M + TM - 1) / TM, n_tiles = (w_rows + TN - 1) / TN;
  auto launch = [&](auto kernel) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return set_error(-2, "gemm: cannot get %d bytes of LDS", LDS);
    kernel<<<m_tiles * n_tiles, 512, LDS, stream>>>(a, m_tiles, n_tiles);
    return 0;
  };
  int rc;
  const bool f32 = a.out_dtype == kF32;
  if constexpr (TN / WM / 16 % 2 == 0) {
    if (gated) {
      rc = f32 ? launch(gemm_mid_kernel<TM, TN, WM, WN, KT, NB, true, float>) : launch(gemm_mid_kernel<TM, TN, WM, WN, KT, NB, true, bf16>);
      if (rc) return rc;
      NINFER_LAUNCH_CHECK();
      return 0;
    }
  }
  rc = f32 ? launch(gemm_mid_kernel<TM, TN, WM, WN, KT, NB, false, float>) : launch(gemm_mid_kernel<TM, TN, WM, WN, KT, NB, false, bf16>);
  if (rc) return rc;
  NINFER_LAUNCH_CHECK();
  return 0;
}

int gemm_mid(const GemmArgs& a, hipStream_t stream) {
  NINFER_REQUIRE(gemm_mid_takes(a), "gemm: not a product of one round of tiles");
  switch (mid_tile(a)) {
    case 0: return launch_mid<32, 64, 4, 2, 4, 3>(a, stream);
    case 1: return launch_mid<64, 64, 2, 4, 2, 4>(a, stream);
    case 2: return launch_mid<96, 64, 4, 2, 2, 3>(a, stream);
    case 3: return launch_mid<64, 96, 2, 4, 2, 3>(a, stream);
    case 4: return launch_mid<128, 64, 2, 4, 2, 3>(a, stream);
    case 5: return launch_mid<192, 64, 2, 4, 1, 4>(a, stream);
    case 6: return launch_mid<128, 128, 2, 4, 1, 4>(a, stream);
    case 7: return launch_mid<192, 128, 2, 4, 1, 3>(a, stream);
    default: return launch_mid<128, 192, 4, 2, 1, 3>(a, stream);
  }
}

}  // namespace ninfer

// The tile in which gemm_mid runs a product: 1,000 x its rows of A + its rows of W (0: it does not take it). Whether ninfer_gemm asks
// gemm_mid for it is ninfer_gemm_kernel's to say.
extern "C" int ninfer_gemm_mid_tile(const ninfer::GemmArgs* args) {
  if (!ninfer::gemm_mid_takes(*args)) return 0;
  const ninfer::MidTile& t = ninfer::kMidTiles[ninfer::mid_tile(*args)];
  return 1000 * t.rows + t.w_rows;
}
