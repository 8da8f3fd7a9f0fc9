// C = A W^T for many rows per weight matrix (bf16) on the matrix cores, dense or grouped by expert with one
// launch for all experts, with a bias or a SwiGLU epilogue: tiles of 256 x 256, 128 x 128 or 64 x 128
// (activation rows x rows of W), loaded from global memory straight into LDS (buffer_load_dwordx4 ... lds),
// so that no registers stage them, in k tiles of 64 (whole 128-byte lines of every
// row): two buffers for the rows of A, which neighbours share through L2 (three in the lowest tile), and
// three for the rows of W. The tall tile takes all 160 KB of a CU's LDS, of the others two blocks share a
// CU. The reference sends these products to rocBLAS
// (src/ops/linear.hip:21-35, src/models/model.hip:406-425).
//
// The waves of a block form a grid, 4 x 2 (two per SIMD) for the tall tile and 2 x 2 for the others; each owns
// 64 W rows x TM / 2 tokens in tiles of v_mfma_f32_16x16x32_bf16 (up to 128 accumulator registers). W rows
// are the A operand (lane l: row l % 16, k = 8 (l / 16) .. + 7), activation rows the B operand, so a
// lane's accumulator holds, for token l % 16, four consecutive output features.
// With the SwiGLU epilogue the first half of a wave's W rows are gate rows and the second half their up rows,
// so silu(g) * u is formed in registers and the block writes TN / 2 output features.
// What bounds the tall tile when full is power: the matrix cores alone reach 2.06 PFLOP/s with
// this instruction and 1.75 with 32x32x16 on random operands (2.4 both on zeros): its
// accumulators travel half as often per product. Products and fragment reads without the loads
// from global memory run at 1.75 PFLOP/s (8,192 x 8,192, K 8,192), the whole at 1.47; with
// 32x32x16, loads in one burst per k tile and k walks of their own per block it was 1.17.
// Four waves of 128 x 128 read a third less from LDS and were slower (0.98).
// The lower tiles staged their operands through registers before: 512 rows of 2 x 5,632, K 2,048, 43 -> 36 us
// in tiles of 128, 512 rows of 2 x 2,816 29 -> 20 in tiles of 64.
// A wave column multiplies only its 32-row blocks that hold rows (the tile's rows
// fill the columns' blocks one after the other, the first column's first), and in the two taller tiles
// a wave loads only the pieces of A that hold rows, so a tile with few rows costs little
// more than its share (the lowest tile loads all its pieces, so that a wait is a constant count).
//
// LDS rows are 128 bytes (64 bf16) and unpadded, because a wave's load writes
// 1 KB contiguously (lane l at 16 l); the eight 16-byte chunks of row r are
// stored in the order c ^ ((r / 2) % 8), chosen on the global side, so that the
// 16 rows which one pass of a fragment read touches fall into 16 different
// 16-byte columns of the banks.
//
// A k tile is four phases: each half of its depth against the first and the second half of the
// wave's token blocks, so that only one half's fragments of A are read ahead (64 registers of
// fragments). The fragments of every phase are read while the products of the phase before run.
// One barrier per k tile, before its last phase: when a wave passes the barrier of tile t, tile
// t + 1 has landed for every wave and every wave holds the last fragments of tile t in registers,
// so the loads of A's tile t + 2, in that last phase, may overwrite tile t; those of W's tile
// t + 2 go one by one between the products of the first three phases (into the third buffer).
// All loads in one burst behind the barrier keep the waves from issuing products while the CU
// takes them in: 0.79 against 0.75 ms at 8,192 x 8,192, K 8,192, and 90 against 85 us at 2,048 rows of
// 2 x 5,632, K 2,048. With a third buffer for the rows of A as well (the lowest tile, whose two blocks still
// fit a CU) all loads of tile t + 2 go into the first three phases and have two k tiles' time to land: 512 rows
// of 2 x 5,632 50 -> 42 us, 32 groups of 16 rows of 2 x 1,408 69 -> 60. More buffers and one block a CU gain
// nothing (64 rows of 2 x 5,632 20.7 us with three, 20.7 with six): few blocks wait for their chains of
// fragment reads and barriers.
#include "gemm_tile.h"
#include <type_traits>

namespace ninfer {

// Wait until at most N of this wave's loads are under way (and, with LDS, until its LDS
// reads have returned).
template <int N> __device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
template <int N> __device__ __forceinline__ void wait_loads_and_lds() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// A dense product's tiles run in rounds of one to a CU. The tiles of the last round, when they
// leave half of the CUs idle or more, are cut into 2 or 4 blocks of 128 or 64 rows, which take a
// half to two thirds of a whole tile's time (2 x 5,632 features, K 2,048: 2,048 rows, 352 tiles on
// 256 CUs, 96 -> 84 us; 1,531 rows, 264 tiles, 94 -> 75). Not beside other products, whose
// blocks take those CUs: a 2,048-token prompt of the headline model, whose shared expert runs beside
// the routed ones, 13.38 -> 13.56 ms with the cut.
struct DirectGrid {
  int m_tiles, n_tiles;
  int whole;   // tiles that are one block each: those before the last round
  int parts;   // blocks of each tile of the last round
};

// What the scheduler is asked for in a phase of M products: R fragment reads and L loads spread
// evenly between them.
template <int I, int M, int R, int L> __device__ __forceinline__ void spread_over_products() {
  if constexpr (I < M) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
    constexpr int r = (I + 1) * R / M - I * R / M, l = (I + 1) * L / M - I * L / M;
    if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);   // LDS reads
    if constexpr (l > 0) __builtin_amdgcn_sched_group_barrier(0x010, l, 0);   // global memory
    spread_over_products<I + 1, M, R, L>();
  }
}

// kDenseCut: the launch cuts its last round. kGroupedFar: an index gathers rows of A of which some may lie 4 GB and
// more behind its first: every lane keeps whole addresses of its rows.
enum DirectMode : int { kDense, kDenseCut, kGrouped, kGroupedFar };

template <int TM, int TN, int WGM, int WGN, int NBX, int NBW, bool SWIGLU, typename TC, DirectMode MODE>
__global__ __launch_bounds__(WGM * WGN * 64, (NBX * TM + NBW * TN) * 128 > 80 * 1024 ? 1 : 2) void gemm_tile_kernel(GemmArgs a, DirectGrid grid) {
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass does not know buffer resources)
  constexpr bool CUT = MODE == kDenseCut, FAR = MODE == kGroupedFar, GROUPED = FAR || MODE == kGrouped;
  constexpr int TK = 64;
  constexpr int WAVES = WGM * WGN;
  constexpr int COL = TM / WGN;                            // staged token rows per wave column
  constexpr int FI = TN / WGM / 16, FJ = COL / 16;         // 16-row blocks of W and of tokens per wave
  constexpr int KK = TK / 32;                // parts of a k tile: one MFMA depth each
  static_assert(KK == 2, "the phases of a k tile are written for two depths");
  constexpr int ROW_BYTES = TK * 2;
  constexpr int CPR = ROW_BYTES / 16;        // 16-byte chunks of a staged row
  constexpr int RPP = 64 / CPR;              // rows of a 1 KB piece
  constexpr int X_BYTES = TM * ROW_BYTES, W_BYTES = TN * ROW_BYTES;
  // buffers of A rows and of W rows: two and three, or three of both
  constexpr bool EVEN = NBX == NBW;
  static_assert((EVEN || NBX == 2) && NBW == 3, "buffers");
  constexpr int W_BASE = NBX * X_BYTES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int bx, by, part = 0, parts = 1;
  if constexpr (CUT) {
    const int id = blockIdx.x;
    int w = spread_over_xcds(id, grid.whole);
    if (id >= grid.whole) {   // a tile's parts follow each other on one XCD: W comes from its L2
      parts = grid.parts;
      w = spread_over_xcds(id - grid.whole, (grid.m_tiles * grid.n_tiles - grid.whole) * parts);
      part = w % parts;
      w = grid.whole + w / parts;
    }
    dense_tile(w, grid.m_tiles, grid.n_tiles, bx, by);
  } else {
    block_to_tile(GROUPED, bx, by);
  }
  int row0, row_end, group;
  // the search's three ints lie in the buffers: no load may land before every wave has them
  if (!tile_rows<TM>(a, bx, (int*)smem, row0, row_end, group)) return;
  if (CUT && parts > 1) {
    row0 += part * (TM / parts);
    row_end = min(row_end, row0 + TM / parts);
    if (row0 >= row_end) return;
  }
  __syncthreads();

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // the same in every lane: a scalar
  const int wm = wave % WGM, wn = wave / WGM;
  const int K = a.K, N = a.N;
  constexpr int OUT_PER_BLOCK = SWIGLU ? TN / 2 : TN;
  constexpr int OUT_PER_WAVE = OUT_PER_BLOCK / WGM;
  const int out0 = by * OUT_PER_BLOCK;
  const int w_first = min(out0, N - 1);
  const bf16* W = (const bf16*)a.W + (int64_t)group * a.w_group_stride + (int64_t)w_first * K;
  const int rows_here = min(TM, row_end - row0);
  // The tile's rows go to the two wave columns in whole blocks of 32, the first column
  // taking the odd one: a SIMD holds a wave of each column, so its matrix instructions are
  // those of both, and 137 rows cost it five blocks (3 + 2) where rows dealt in turn would
  // cost six (69 + 68 rows). Staged row l of column l / COL holds the tile's row
  // (l / COL) * rows0 + l % COL, or none (TM: beyond every tile's rows).
  static_assert(WGN == 2, "the rows are dealt to two wave columns");
  const int n_blocks = (rows_here + 31) / 32;
  const int rows0 = min(rows_here, 32 * ((n_blocks + 1) / 2));   // rows of the first column
  auto row_of = [&](int l) -> int {
    const int i = l % COL;
    if (l < COL) return i < rows0 ? i : TM;
    return rows0 + i < rows_here ? rows0 + i : TM;
  };

  // Loads: instruction i of wave w fills the 1 KB piece i * WAVES + w of the X (and
  // of the W) part of a buffer: RPP rows, lane l at row l / CPR, stored chunk
  // l % CPR, which holds the row's chunk (l % CPR) ^ swizzle(row), where
  // swizzle(row) = (row / (16 / CPR)) % CPR.
  constexpr int NLX = X_BYTES / 1024 / WAVES, NLW = W_BYTES / 1024 / WAVES;   // load instructions per wave and k tile
  // the row's part of the swizzle that the piece's number leaves: pieces i * WAVES + w differ
  // in multiples of WAVES * RPP rows between the loads of a wave, which the swizzle does not see
  const int chunk = (lane % CPR) ^ (((wave * RPP + lane / CPR) / (16 / CPR)) % CPR);
  static_assert((WAVES * RPP / (16 / CPR)) % CPR == 0, "the loads of a wave must share their swizzle");
  // byte offsets: of A's rows from its first one (from the tile's first, where no index gathers them), of W's
  // from the block's first gate row and its up row (gemm_tile_takes: below 4 GB)
  unsigned xoff[NLX], woff[NLW];
  const unsigned char* x_far[FAR ? NLX : 1];
  int x_row[NLX];
  unsigned x_live = 0;   // bit i: piece i of this wave's loads of A holds rows of the tile
#pragma unroll
  for (int i = 0; i < NLX; ++i) {
    const int r = row_of((i * WAVES + wave) * RPP + lane / CPR);
    // rows beyond the tile's last read its first row (one line, from L1): their results are
    // never stored
    x_row[i] = r < rows_here ? r : 0;
    // a piece none of whose rows the tile has is not loaded (what the fragments read there goes
    // into sums that are never stored); staged rows of a piece are neighbours in one column, so
    // its first row decides
    if (row_of((i * WAVES + wave) * RPP) < rows_here) x_live |= 1u << i;
  }
#pragma unroll
  for (int i = 0; i < NLW; ++i) {
    const int n = staged_w_row<TN, WGM, SWIGLU>((i * WAVES + wave) * RPP + lane / CPR, out0, N);
    woff[i] = (unsigned)((n < N ? n : n - N) - w_first) * (unsigned)(2 * K) + 16 * chunk;
  }
  if (a.a_index) {   // the index loads in flight together
    int idx[NLX];
#pragma unroll
    for (int i = 0; i < NLX; ++i) idx[i] = a.a_index[row0 + x_row[i]];
#pragma unroll
    for (int i = 0; i < NLX; ++i) x_row[i] = idx[i] / a.a_div;
  }
#pragma unroll
  for (int i = 0; i < NLX; ++i) {
    xoff[i] = (unsigned)x_row[i] * (unsigned)(2 * a.lda) + 16 * chunk;
    if constexpr (FAR) x_far[i] = (const unsigned char*)((const bf16*)a.A + (int64_t)x_row[i] * a.lda) + 16 * chunk;
  }
  const bf16* A = (const bf16*)a.A + (a.a_index ? 0 : (int64_t)row0 * a.lda);
  const auto x_res = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, 0xffffffffu, 0x00020000);
  // (a load's rows of W are all gate rows or all up rows; with eight waves that is the same for all of a wave's
  // loads, with four for every second one)
  constexpr int HALF = TN / WGM / 2 / RPP;   // loads of half a wave row's rows of W
  static_assert(!SWIGLU || WAVES % HALF == 0, "a wave's loads i and i + 2 must be alike");
  auto w_rows = [&](int i) {
    const bool up = SWIGLU && (i * WAVES + wave) / HALF % 2;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(W + (up ? (int64_t)N * K : 0)), 0, 0xffffffffu, 0x00020000);
  };
  const auto w_res0 = w_rows(0), w_res1 = w_rows(1);
  typedef const __attribute__((address_space(1))) void* gptr;
  typedef __attribute__((address_space(3))) void* lptr;
  // Every lane of every load takes part: with some lanes switched off, a load into LDS did
  // not leave the other lanes' bytes where this layout expects them (products came out wrong).
  // a product cut along K: this block's k tiles are kt_first .. kt_first + nk - 1, and its
  // sums go to part blockIdx.z of C
  int nk = K / TK, kt_first = 0;
  if (!GROUPED && a.k_parts > 1) {
    const int per = (nk + a.k_parts - 1) / a.k_parts;
    kt_first = blockIdx.z * per;
    nk = min(per, nk - kt_first);
    a.C = (TC*)a.C + (int64_t)blockIdx.z * a.M * a.ldc;
  }
  // Where the walk over the k tiles starts. Dense: at the first for every block: the 32 blocks of an
  // XCD share their rows of A and W through its L2 only while they walk in step (with starts of their own
  // 8,192 x 8,192, K 8,192 took 0.94 instead of 0.85 ms, 2,048 rows of 2 x 5,632, K 2,048, 119 instead of
  // 99 us). Grouped: in a circle from a start of the block's own, because every W panel has one reader, and
  // blocks in step read the same columns of rows that lie a power of two apart, which fall on few memory
  // channels (34 rows per expert, 60 x 2 x 1,408 x 2,048: 129 against 161 us). The start depends on the
  // expert, not on the row tile, so that a row's sum has the same order whichever tile of its expert the
  // grouping put it in.
  const int phase = GROUPED ? (int)((group * 5u + by * 3u) % (unsigned)nk) : 0;
  auto k_bytes = [&](int t) {   // of the t-th k tile of this block's walk
    const int kt = t + phase;
    return (kt_first + (GROUPED && kt >= nk ? kt - nk : kt)) * (2 * TK);
  };
  auto next_w = [](int w_off) { return w_off == (NBW - 1) * W_BYTES ? 0 : w_off + W_BYTES; };
  auto next_x = [](int x_off) { return x_off == (NBX - 1) * X_BYTES ? 0 : x_off + X_BYTES; };

  f32x4 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int jj = 0; jj < FJ; ++jj)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][jj][v] = 0.f;

  // rows dealt to this wave's column, and its 32-row blocks that hold any
  const int col_rows = wn == 0 ? rows0 : rows_here - rows0;
  const int n_jj = (col_rows + 31) / 32;
  const int tok0 = wn * COL;

  // fragment addresses: lane reads row lr of a 16-row block, k chunk 4 kk + lk, stored at
  // chunk (4 kk + lk) ^ swizzle(lr) (the block's first row is a multiple of 16)
  const int lr = lane & 15, lk = lane >> 4;
  const int sw = (lr / (16 / CPR)) % CPR;
  const int x_lane = (tok0 + lr) * ROW_BYTES;
  const int w_lane = W_BASE + (wm * (TN / WGM) + lr) * ROW_BYTES;
  int c_part[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) c_part[kk] = 16 * ((4 * kk + lk) ^ sw);

  // NJ: 16-row token blocks of the wave; ONCE: the panel of W has this block as its only reader
  auto run = [&](auto nj_tag, auto once_tag) {
    constexpr int NJ = decltype(nj_tag)::value, H0 = (NJ + 1) / 2, H1 = NJ - H0;
    // loads i0 .. i1 - 1 of A's tile t into its buffer, and of W's tile t into the one at w_off.
    // A panel of W that one block alone reads is loaded non-temporal (the last argument: 2), so that
    // it does not push the rows of A, which the expert's other feature tiles read again, out of L2 (6 to
    // 9% at 137 rows per expert; with two tiles per expert the second finds the panel in L2 and the
    // mark costs 4%).
    auto issue_x = [&](int t, int x_off, auto from, auto to) {
      unsigned char* buf = smem + x_off + wave * 1024;
      const int k = k_bytes(t);
#pragma unroll
      for (int i = decltype(from)::value; i < decltype(to)::value; ++i) {
        if (!EVEN && !(x_live & (1u << i))) continue;   // (EVEN: all, so that a wait is a constant count)
        if constexpr (FAR)
          __builtin_amdgcn_global_load_lds((gptr)(x_far[i] + k), (lptr)(buf + i * (WAVES * 1024)), 16, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(x_res, (lptr)(buf + i * (WAVES * 1024)), 16, xoff[i], k, 0, 0);
      }
    };
    auto issue_w = [&](int t, int w_off, auto from, auto to) {
      unsigned char* buf = smem + W_BASE + w_off + wave * 1024;
      const int k = k_bytes(t);
#pragma unroll
      for (int i = decltype(from)::value; i < decltype(to)::value; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(i % 2 ? w_res1 : w_res0, (lptr)(buf + i * (WAVES * 1024)), 16, woff[i], k,
                                                 0, decltype(once_tag)::value ? 2 : 0);
    };
    std::integral_constant<int, 0> i0;
    std::integral_constant<int, NLW / 2> i2;
    std::integral_constant<int, NLW * 3 / 4> i3;
    std::integral_constant<int, NLW> i4;
    std::integral_constant<int, NLX> x4;
    bf16x8 wf[KK][FI], x0[H0 > 0 ? H0 : 1], x1[H1 > 0 ? H1 : 1];
    // fragments of depth kk: W's, the first and the second half of the token blocks'
    auto read_w = [&](int kk, int w_off) {
      if constexpr (NJ == 0) return;
      const unsigned char* p = smem + w_off + c_part[kk] + w_lane;
#pragma unroll
      for (int i = 0; i < FI; ++i) wf[kk][i] = *(const bf16x8*)(p + i * 16 * ROW_BYTES);
    };
    auto read_x0 = [&](int kk, int x_off) {
      const unsigned char* p = smem + x_off + c_part[kk] + x_lane;
#pragma unroll
      for (int jj = 0; jj < H0; ++jj) x0[jj] = *(const bf16x8*)(p + jj * 16 * ROW_BYTES);
    };
    auto read_x1 = [&](int kk, int x_off) {
      const unsigned char* p = smem + x_off + c_part[kk] + x_lane;
#pragma unroll
      for (int jj = 0; jj < H1; ++jj) x1[jj] = *(const bf16x8*)(p + (H0 + jj) * 16 * ROW_BYTES);
    };
    auto multiply0 = [&](int kk) {
#pragma unroll
      for (int jj = 0; jj < H0; ++jj)
#pragma unroll
        for (int i = 0; i < FI; ++i)
          acc[i][jj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[kk][i], x0[jj], acc[i][jj], 0, 0, 0);
    };
    auto multiply1 = [&](int kk) {
#pragma unroll
      for (int jj = 0; jj < H1; ++jj)
#pragma unroll
        for (int i = 0; i < FI; ++i)
          acc[i][H0 + jj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[kk][i], x1[jj], acc[i][H0 + jj], 0, 0, 0);
    };
    int t = 0, x_cur = 0, w_cur = 0;   // w_cur, x_cur: where W's and A's tile t lie
    if constexpr (EVEN) {
      // Tile t + 2 is loaded during tile t's first three phases into the buffers that tile t - 1 has
      // left. When tile t + 1 is needed, its loads stay on their way.
      constexpr int PER = NLX + NLW;
      issue_x(0, 0, i0, x4);
      issue_w(0, 0, i0, i4);
      if (nk > 1) {
        issue_x(1, X_BYTES, i0, x4);
        issue_w(1, W_BYTES, i0, i4);
        wait_loads<PER>();
      } else {
        wait_loads<0>();
      }
      __builtin_amdgcn_s_barrier();
      read_w(0, 0);
      read_x0(0, 0);
      int x_far = 2 * X_BYTES, w_far = 2 * W_BYTES;
      for (; t + 2 < nk; ++t) {
        read_x1(0, x_cur);
        issue_w(t + 2, w_far, i0, i2);
        multiply0(0);
        spread_over_products<0, FI * H0, H1, NLW / 2>();
        read_w(1, w_cur);
        read_x0(1, x_cur);
        issue_w(t + 2, w_far, i2, i4);
        multiply1(0);
        spread_over_products<0, FI * H1, FI + H0, NLW - NLW / 2>();
        read_x1(1, x_cur);
        issue_x(t + 2, x_far, i0, x4);
        multiply0(1);
        spread_over_products<0, FI * H0, H1, NLX>();
        wait_loads_and_lds<PER>();
        __builtin_amdgcn_s_barrier();
        x_far = x_cur, w_far = w_cur;
        x_cur = next_x(x_cur), w_cur = next_w(w_cur);
        read_w(0, w_cur);
        read_x0(0, x_cur);
        multiply1(1);
        spread_over_products<0, FI * H1, FI + H0, 0>();
      }
    } else {
      // A wave's loads return in the order of their issue: A 0, W 0, A 1, W 1, then per tile t W t + 2,
      // A t + 2. When tile t + 1 is needed, the only younger loads are W's tile t + 2 (NLW loads), which
      // stay on their way. (Loads of A that are left out only make a wait longer than it has to be.)
      issue_x(0, 0, i0, x4);
      issue_w(0, 0, i0, i4);
      if (nk > 1) {
        issue_x(1, X_BYTES, i0, x4);
        issue_w(1, W_BYTES, i0, i4);
        wait_loads<NLW>();
      } else {
        wait_loads<0>();
      }
      __builtin_amdgcn_s_barrier();
      read_w(0, 0);
      read_x0(0, 0);
      // steady state, free of conditions on t: the tile t + 2 exists
      for (; t + 2 < nk; ++t) {
        const int w_nxt = next_w(w_cur), w_far = next_w(w_nxt);
        read_x1(0, x_cur);
        issue_w(t + 2, w_far, i0, i2);
        multiply0(0);
        spread_over_products<0, FI * H0, H1, NLW / 2>();
        read_w(1, w_cur);
        read_x0(1, x_cur);
        issue_w(t + 2, w_far, i2, i3);
        multiply1(0);
        spread_over_products<0, FI * H1, FI + H0, NLW * 3 / 4 - NLW / 2>();
        read_x1(1, x_cur);
        issue_w(t + 2, w_far, i3, i4);
        multiply0(1);
        spread_over_products<0, FI * H0, H1, NLW - NLW * 3 / 4>();
        // this wave's loads of tile t + 1 have landed and its last fragments of tile t are in
        // registers; after the barrier that holds for every wave, and tile t's buffers are free
        wait_loads_and_lds<NLW>();
        __builtin_amdgcn_s_barrier();
        issue_x(t + 2, x_cur, i0, x4);
        w_cur = w_nxt;
        x_cur = next_x(x_cur);
        read_w(0, w_cur);
        read_x0(0, x_cur);
        multiply1(1);
        spread_over_products<0, FI * H1, FI + H0, NLX>();
      }
    }
    // the last two tiles: nothing left to issue
    for (; t < nk; ++t) {
      read_x1(0, x_cur);
      multiply0(0);
      read_w(1, w_cur);
      read_x0(1, x_cur);
      multiply1(0);
      read_x1(1, x_cur);
      multiply0(1);
      wait_loads_and_lds<0>();
      __builtin_amdgcn_s_barrier();
      x_cur = next_x(x_cur), w_cur = next_w(w_cur);
      if (t + 1 < nk) {
        read_w(0, w_cur);
        read_x0(0, x_cur);
      }
      multiply1(1);
    }
  };
  // one straight-line instance per count of live 32-row token blocks
  auto run_rows = [&](auto once) {
    if (n_jj == 0) run(std::integral_constant<int, 0>{}, once);
    else if (FJ > 2 && n_jj == 1) run(std::integral_constant<int, 2>{}, once);
    else if (FJ > 4 && n_jj == 2) run(std::integral_constant<int, (FJ > 4 ? 4 : FJ)>{}, once);
    else if (FJ > 6 && n_jj == 3) run(std::integral_constant<int, (FJ > 6 ? 6 : FJ)>{}, once);
    else run(std::integral_constant<int, FJ>{}, once);
  };
  if constexpr (GROUPED) {   // an expert whose rows fit one tile
    if (row_end - a.offsets[group] <= TM) run_rows(std::true_type{});
    else run_rows(std::false_type{});
  } else {
    run_rows(std::false_type{});
  }
  static_assert(WAVES * FJ * 16 * FI * 32 <= NBX * X_BYTES + NBW * W_BYTES, "the epilogue's stage exceeds the buffers");
  __syncthreads();   // every wave has read its last fragments: the buffers become the epilogue's stage
  write_tile<FI, FJ, SWIGLU, TC>(a, acc, smem + wave * (FJ * 16 * FI * 32), tok0, row0, rows_here,
                                 out0 + OUT_PER_WAVE * wm, row_of);
#endif
}

// Do rows of A that an index gathers need whole addresses?
bool gemm_tile_far(const GemmArgs& a) { return a.a_index && 2ll * a.M * a.lda >= 1ll << 32; }

// K a whole number of k tiles of 64; a tile's rows below 4 GB.
bool gemm_tile_takes(const GemmArgs& a) {
  const int64_t four_gb = 1ll << 32;
  return a.in_dtype == kBF16 && a.K % 64 == 0 && a.lda % 8 == 0 && ((uintptr_t)a.A % 16 == 0) &&
         ((uintptr_t)a.W % 16 == 0) && a.w_group_stride % 8 == 0 &&
         2 * 256ll * a.lda < four_gb && 2 * 256ll * a.K < four_gb && (a.offsets || !gemm_tile_far(a));
}

int gemm_tile_row_tiles(const GemmArgs& a, int rows) {
  const int tiles = (a.M + rows - 1) / rows;
  if (!a.offsets) return tiles;
  return (tiles + a.groups + kXcds - 1) / kXcds * kXcds;   // block_to_tile's bijection
}

template <int TM, int TN, int WGM, int WGN, int NBX, int NBW>
static int launch_tiles(const GemmArgs& a, hipStream_t stream) {
  constexpr int LDS_BYTES = (NBX * TM + NBW * TN) * 64 * 2;
  const bool swiglu = epilogue_gated(a.epilogue);
  const int per_block = swiglu ? TN / 2 : TN;
  DirectGrid g = {gemm_tile_row_tiles(a, TM), (a.N + per_block - 1) / per_block, 0, 1};
  dim3 grid(g.m_tiles, g.n_tiles, a.k_parts > 1 ? a.k_parts : 1);
  if (TM == 256 && !a.offsets && a.k_parts <= 1) {
    const int tiles = g.m_tiles * g.n_tiles, cus = device_cu_count(), last = tiles % cus;
    g.parts = a.beside || last == 0 || tiles < cus ? 1 : 4 * last <= cus ? 4 : 2 * last <= cus ? 2 : 1;
    g.whole = g.parts > 1 ? tiles - last : tiles;
    if (g.parts > 1) grid = dim3(g.whole + (tiles - g.whole) * g.parts);
  }
#define NINFER_TILE_KERNEL(SW, TYPE, MODE)                                                      \
  do {                                                                                          \
    auto kern = gemm_tile_kernel<TM, TN, WGM, WGN, NBX, NBW, SW, TYPE, MODE>;                             \
    hipError_t e = hipFuncSetAttribute((const void*)kern,                                       \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);  \
    if (e != hipSuccess) return set_error(-2, "gemm: cannot get %d bytes of LDS", LDS_BYTES);   \
    kern<<<grid, WGM * WGN * 64, LDS_BYTES, stream>>>(a, g);                                    \
  } while (0)
#define NINFER_TILE_LAUNCH(SW, TYPE)                                                            \
  do {                                                                                          \
    if (TM == 128 && a.offsets && gemm_tile_far(a))                                             \
      NINFER_TILE_KERNEL(SW, TYPE, (TM == 128 ? kGroupedFar : kGrouped));                       \
    else if (a.offsets) NINFER_TILE_KERNEL(SW, TYPE, kGrouped);                                 \
    else if (TM == 256 && g.parts > 1) NINFER_TILE_KERNEL(SW, TYPE, (TM == 256 ? kDenseCut : kDense)); \
    else NINFER_TILE_KERNEL(SW, TYPE, kDense);                                                  \
  } while (0)
  if (a.out_dtype == kF32) {
    if (swiglu) NINFER_TILE_LAUNCH(true, float); else NINFER_TILE_LAUNCH(false, float);
  } else {
    if (swiglu) NINFER_TILE_LAUNCH(true, bf16); else NINFER_TILE_LAUNCH(false, bf16);
  }
#undef NINFER_TILE_KERNEL
#undef NINFER_TILE_LAUNCH
  NINFER_LAUNCH_CHECK();
  return 0;
}

// k tiles of 64 at every height: measured faster than tiles of 32 in twice the buffers (whole
// 128-byte lines per row beat the deeper queue of loads).
int gemm_tile_rows(const GemmArgs& a, int rows, hipStream_t stream) {
  static_assert(kGroupedTileRows == 256, "the grouped tile lists are made for the tall tiles");
  if (rows == 256) return launch_tiles<256, 256, 4, 2, 2, 3>(a, stream);
  if (rows == 128) return launch_tiles<128, 128, 2, 2, 2, 3>(a, stream);
  return launch_tiles<64, 128, 2, 2, 3, 3>(a, stream);
}

}  // namespace ninfer
