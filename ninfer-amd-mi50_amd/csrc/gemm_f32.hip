// C = A W^T in true 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32), dense or grouped by
// expert, with the epilogues of the product family.
//
// What every output is, whatever the batch: K is cut into 8 segments of whole chunks of 16; a
// segment is summed chunk by chunk on the matrix instruction and the 8 sums are
// added in the segments' order. Nothing of that depends on M, on the tile's size, on the waves that
// share the segments or on where a row lies in its tile, so a row's bits are the same under every cut
// of the work (which is what the 32-bit path promises), and chains of K / 8 terms round less than one
// of K.
//
// Few rows are bound by the weights' bytes, many by the matrix cores. A block owns 16 RT rows x 16 CT
// rows of W; its 4 or 8 waves take two segments or one each and walk them with operands of their own:
// stages of 32 k, whole 128-byte lines of every row, loaded straight into a ring of two stages in LDS
// (non-temporal for weights that one block alone reads; as loads of half lines into registers that mark
// cost 20%) and read back as fragments, the next stage's first half while this one's second half is
// multiplied. No barrier before the last chunk; LDS then carries the 8 partial sums, in the ring's place.
// Four waves and 48 to 80 KB a block leave room for two or three blocks on a CU, which hide each other's
// first loads and last sums; one wave a segment is for launches that do not fill the CUs.
// Measured on Qwen1.5-MoE-A2.7B's shapes, 173 rows, loads in the fragments' layout straight into registers
// before and now: the experts' gate/up (1.4 GB of weights) 297 -> 234 us, 5.9 TB/s; their down products
// 175 -> 127; 2 x 5,632 features 158 -> 95, 84 of the 155 TFLOP/s that a large matrix product reaches; 6,144
// features 85 -> 55; 2,048 features 31 -> 20. One row: 92 MB of gate/up 22 -> 18, 2,048 features 9.3 -> 7.7.
#include "gemm.h"
#include <type_traits>

namespace ninfer {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kF32Segments = 8;   // of K
constexpr int kF32Chunk = 16;     // k of a chunk: four matrix instructions

template <int N> __device__ __forceinline__ void f32_wait_loads() {   // until at most N are under way
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// FAR: an index gathers rows of A, and some may lie 4 GB and more behind its first: every lane keeps whole addresses of
// its rows (other operands' rows have 32-bit offsets from the block's own first ones).
template <int WAVES, int RT, int CT, bool GATED, bool FAR>
__global__ __launch_bounds__(64 * WAVES) void gemm_f32_kernel(GemmArgs a, int n_tiles, int m_tiles) {
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass does not know buffer resources)
  constexpr int SEGS = kF32Segments / WAVES;        // segments of a wave
  static_assert(SEGS == 1 || SEGS == 2, "a stage may hold the end of one segment and the start of the next");
  constexpr int BM = 16 * RT;                       // rows of a block
  constexpr int BN = 16 * (GATED ? CT / 2 : CT);    // output features of a block
  constexpr int COLS = 16 * CT + 4;                 // partial sums of a row in LDS (padded)
  constexpr int ROWS = 16 * (RT + CT);              // staged rows of a wave: A's, then W's
  constexpr int STAGE = ROWS * 128, NL = ROWS / 8;  // bytes and loads (1 KB, 8 rows) of a stage
  constexpr int RING = WAVES * 2 * STAGE, PARTS = kF32Segments * 16 * COLS * 4;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[RING > PARTS ? RING : PARTS];

  // The row tiles that read the same weights follow each other on one XCD.
  const int xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
  const int n_tile = slot / m_tiles * kXcds + xcd, m_tile = slot % m_tiles;
  if (n_tile >= n_tiles) return;
  int row0, row_end, group = 0;
  bool once = m_tiles == 1;   // no other block reads these weights
  if (a.offsets) {
    int* tile_info = (int*)smem;
    if (!find_tile(a.offsets, a.groups, BM, m_tile, tile_info)) return;
    row0 = tile_info[0];
    row_end = tile_info[1];
    group = tile_info[2];
    once = row_end - a.offsets[group] <= BM;
    __syncthreads();   // no load may land on the tile before every wave has it
  } else {
    row0 = m_tile * BM;
    row_end = a.M;
  }
  const int n0 = n_tile * BN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = a.K;

  // Load i of a stage: staged rows 8 i .. 8 i + 7, the lane at row lane / 8. Of a staged row (128 bytes)
  // the 16-byte chunk c lies at c ^ ((row / 2) % 8), chosen on the global side, so that the 16 rows of a
  // fragment read fall into different columns of the banks. Rows that are not there read the last one
  // that is; nothing of them is stored. Byte offsets: of A's rows from the block's first one (gathered: from
  // A's), of W's from the block's first gate row and its up row.
  unsigned off[NL];
  const char* far_row[FAR ? BM / 8 : 1];
  const int w_first = min(n0, a.N - 1);
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int r = 8 * i + (lane >> 3);
    if (r < BM) {
      const int row = min(row0 + r, row_end - 1);
      if constexpr (FAR) {
        far_row[i] = (const char*)((const float*)a.A + (int64_t)(a.a_index[row] / a.a_div) * a.lda);
        off[i] = 0;
      } else {
        off[i] = (unsigned)(a.a_index ? a.a_index[row] / a.a_div : row - row0) * (unsigned)(4 * a.lda);
      }
    } else {
      const int j = (r - BM) / 16, f = n0 + (GATED && j >= CT / 2 ? j - CT / 2 : j) * 16 + r % 16;
      off[i] = (unsigned)(min(f, a.N - 1) - w_first) * (unsigned)(4 * K);
    }
  }
  const int lane_chunk = (lane & 7) ^ (lane >> 4);   // (load i's rows add 4 i to the row / 2)
  const float* A = (const float*)a.A + (a.a_index ? 0 : (int64_t)row0 * a.lda);
  const float* W = (const float*)a.W + (int64_t)group * a.w_group_stride + (int64_t)w_first * K;
  const auto a_res = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, 0xffffffffu, 0x00020000);
  const auto w_res = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, 0xffffffffu, 0x00020000);
  const auto up_res = __builtin_amdgcn_make_buffer_rsrc((void*)(W + (GATED ? (int64_t)a.N * K : 0)), 0, 0xffffffffu, 0x00020000);
  typedef const __attribute__((address_space(1))) void* gptr;
  typedef __attribute__((address_space(3))) void* lptr;
  unsigned char* ring = smem + wave * 2 * STAGE;

  // this wave's segments: chunks b0 .. b1 - 1 and, of two, b1 .. b2 - 1; stages of two chunks from b0
  const int chunks = (K + kF32Chunk - 1) / kF32Chunk;
  const int per = (chunks + kF32Segments - 1) / kF32Segments;
  const int b0 = min(SEGS * wave * per, chunks), b1 = min(b0 + per, chunks);
  const int b2 = SEGS == 1 ? b1 : min(b1 + per, chunks);
  const int n = b2 - b0, total = (n + 1) / 2;
  auto issue = [&](int g) {
    unsigned char* buf = ring + (g & 1) * STAGE;
    const int k0 = (b0 + 2 * g) * kF32Chunk;
    // (what lies behind the row's end is never read: its last 16 bytes again)
    auto at = [&](int i) { return off[i] + 16 * min(lane_chunk ^ ((4 * i) & 7), (K - k0) / 4 - 1); };
#pragma unroll
    for (int i = 0; i < BM / 8; ++i) {
      if constexpr (FAR)
        __builtin_amdgcn_global_load_lds((gptr)(far_row[i] + at(i) + (int64_t)k0 * 4), (lptr)(buf + i * 1024), 16, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_res, (lptr)(buf + i * 1024), 16, at(i), k0 * 4, 0, 0);
    }
    auto weights = [&](auto mark) {
#pragma unroll
      for (int i = BM / 8; i < NL; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(GATED && (8 * i - BM) / 16 >= CT / 2 ? up_res : w_res,
                                                 (lptr)(buf + i * 1024), 16, at(i), k0 * 4, 0, decltype(mark)::value);
    };
    if (once) weights(std::integral_constant<int, 2>{});
    else weights(std::integral_constant<int, 0>{});
  };
  // Fragments of chunk c of stage g: the lane holds four neighbouring k of one row, so a chunk is
  // four instructions with k dealt alike to both operands.
  const int in = lane & 15, q = lane >> 4, sw = in / 2;
  floatx4 av[2][RT], wv[2][CT];
  auto read = [&](int g, int c, floatx4 (&x)[RT], floatx4 (&y)[CT]) {
    const unsigned char* p = ring + (g & 1) * STAGE + in * 128 + 16 * ((4 * c + q) ^ sw);
#pragma unroll
    for (int i = 0; i < RT; ++i) x[i] = *(const floatx4*)(p + i * 2048);
#pragma unroll
    for (int j = 0; j < CT; ++j) y[j] = *(const floatx4*)(p + (RT + j) * 2048);
    const int k = (b0 + 2 * g + c) * kF32Chunk;
    if (k + kF32Chunk > K && k + 4 * q >= K) {   // a last chunk that K does not fill (K is a multiple of 4)
#pragma unroll
      for (int i = 0; i < RT; ++i) x[i] = floatx4{};
#pragma unroll
      for (int j = 0; j < CT; ++j) y[j] = floatx4{};
    }
  };
  floatx4 acc[SEGS][RT][CT] = {};
  auto multiply = [&](floatx4 (&s)[RT][CT], const floatx4 (&x)[RT], const floatx4 (&y)[CT]) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
          s[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][k], y[j][k], s[i][j], 0, 0, 0);
  };
  if (total > 0) {
    issue(0);
    if (total > 1) {
      issue(1);
      f32_wait_loads<NL>();
    } else {
      f32_wait_loads<0>();
    }
    read(0, 0, av[0], wv[0]);
    int g = 0;
    // a stage, its first chunk's products to `s`, its second one's to `s2`
    auto stage = [&](floatx4 (&s)[RT][CT], floatx4 (&s2)[RT][CT]) {
      read(g, 1, av[1], wv[1]);
      multiply(s, av[0], wv[0]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage is read: its place is free
      if (g + 2 < total) {
        issue(g + 2);
        f32_wait_loads<NL>();
      } else {
        f32_wait_loads<0>();
      }
      if (g + 1 < total) read(g + 1, 0, av[0], wv[0]);
      if (2 * g + 1 < n) multiply(s2, av[1], wv[1]);
      ++g;
    };
    while (g < (b1 - b0) / 2) stage(acc[0], acc[0]);
    if ((b1 - b0) & 1) stage(acc[0], acc[SEGS - 1]);
    while (g < total) stage(acc[SEGS - 1], acc[SEGS - 1]);
  }

  __syncthreads();   // every ring is read: the partial sums take their place
  float (*part)[16][COLS] = (float (*)[16][COLS])smem;
  float* C = (float*)a.C;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int s = 0; s < SEGS; ++s)
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[SEGS * wave + s][q * 4 + r][j * 16 + in] = acc[s][i][j][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * BN; e += 64 * WAVES) {
      const int m = e / BN, col = e % BN;
      const int row = row0 + i * 16 + m, f = n0 + col;
      if (row >= row_end || f >= a.N) continue;
      float v = part[0][m][col], u = 0.f;
#pragma unroll
      for (int s = 1; s < kF32Segments; ++s) v += part[s][m][col];
      if (GATED) {
        u = part[0][m][BN + col];
#pragma unroll
        for (int s = 1; s < kF32Segments; ++s) u += part[s][m][BN + col];
        if (a.bias) {
          v += a.bias[f];
          u += a.bias[a.N + f];
        }
        v = gated_output<false>(v, u, a.epilogue, a.act_limit, a.act_alpha);
      } else {
        if (a.bias) v += a.bias[f];
        v = ungated_output(v, a.epilogue == kEpilogueReluSq);
      }
      C[(int64_t)(a.c_index ? a.c_index[row] : row) * a.ldc + f] = v;
    }
  }
#endif
}

// 32-bit operands whose rows are whole 16-byte pieces, a block's rows (at most 48 of A and 32 of W) below 4 GB. That
// depends on the operands' layout alone and not on the number of rows: a model's product takes the same
// kernel in every step.
bool gemm_f32_takes(const GemmArgs& a) {
  const int64_t four_gb = 1ll << 32;
  return a.in_dtype == kF32 && a.out_dtype == kF32 && a.K % 4 == 0 && a.lda % 4 == 0 &&
         a.w_group_stride % 4 == 0 && ((uintptr_t)a.A | (uintptr_t)a.W) % 16 == 0 &&
         4ll * 48 * a.lda < four_gb && 4ll * 32 * a.K < four_gb;
}

template <int WAVES, int RT, int CT, bool FAR = false>
static void launch(const GemmArgs& a, hipStream_t stream) {
  const bool gated = epilogue_gated(a.epilogue);
  const int bn = 16 * (gated ? CT / 2 : CT);
  const int n_tiles = (a.N + bn - 1) / bn;
  const int m_tiles = (a.M + 16 * RT - 1) / (16 * RT) + (a.offsets ? a.groups : 0);
  const int grid = (n_tiles + kXcds - 1) / kXcds * kXcds * m_tiles;
  if constexpr (CT > 1) {
    if (gated) {
      gemm_f32_kernel<WAVES, RT, CT, true, FAR><<<grid, 64 * WAVES, 0, stream>>>(a, n_tiles, m_tiles);
      return;
    }
  }
  gemm_f32_kernel<WAVES, RT, CT, false, FAR><<<grid, 64 * WAVES, 0, stream>>>(a, n_tiles, m_tiles);
}

// The tile whose blocks take the least time. Of each: a block alone on its CU, and what every further
// block on that CU adds, in us at K 2,048 (measured over 1 to 1,024 rows of 61 to 151,936 features, K 1,024
// to 5,632; both go with K), and of both what is left as K goes from 1,024 to nothing (starts, the 8 sums added up: 32 groups
// of 512 x 384, 4 rows each, 12.5 us with eight waves and 1 x 1 tiles, 7.3 with four and 1 x 2; 2,048 rows of 384 x 512 20.6 with
// eight and 2 x 2, 17.6 with four). Where one block fills a CU its blocks come in whole rounds; where several
// share one, a part of a round costs less. (173 rows, measured: 6,144 features 55 with four waves and 3 x 2
// tiles, 55 with 1 x 2, 60 with eight waves and 1 x 1; 2,048 features 20, 20 and 23; one row, 2,048 features: 20,
// 11 and 7.7; gated 2 x 5,632, 64 rows: 53, 43, and 41 with eight waves and 2 x 2.)
struct F32Tile { int waves, rt, ct; float alone, further, alone_short, further_short; bool shared; };
static const F32Tile kF32Tiles[] = {{8, 1, 1, 3.5f, 3.4f, 0.f, 1.5f, true},     {8, 1, 2, 5.f, 8.f, 0.f, 3.f, false},
                                    {8, 2, 2, 8.5f, 12.4f, 1.f, 6.f, false},    {4, 1, 2, 7.f, 6.2f, 0.f, 1.f, true},
                                    {4, 2, 2, 11.f, 11.9f, 1.f, 2.f, true},     {4, 3, 2, 15.5f, 16.9f, 4.5f, 6.f, true}};
static int f32_tile(const GemmArgs& a) {
  const bool gated = epilogue_gated(a.epilogue);
  const float columns = (float)a.N * (gated ? 2 : 1), cus = device_cu_count(), k = fminf(1.f, a.K / 1024.f);
  int best = -1;
  float least = 0.f;
  for (int i = 0; i < 6; ++i) {
    const F32Tile& t = kF32Tiles[i];
    if (gated && t.ct == 1) continue;
    const float rows = 16.f * t.rt;
    // (a group's last tile is half full on average)
    const float m_tiles = a.offsets ? a.M / rows + 0.5f * a.groups : ceilf(a.M / rows);
    const float per_cu = fmaxf(1.f, ceilf(columns / (16 * t.ct)) * m_tiles / cus), whole = ceilf(per_cu);
    const float alone = t.alone_short + (t.alone - t.alone_short) * k;
    const float further = t.further_short + (t.further - t.further_short) * k;
    const float us = alone + further * ((t.shared ? 0.5f * (per_cu + whole) : whole) - 1.f);
    if (best < 0 || us < least) best = i, least = us;
  }
  return best;
}

int gemm_f32(const GemmArgs& a, hipStream_t stream) {
  int best = f32_tile(a);
  // 4 GB of rows that an index gathers are many: the tallest tile. (Every tile gives the same bits.)
  if (a.a_index && 4ll * a.M * a.lda >= 1ll << 32) best = 6;
  switch (best) {
    case 0: launch<8, 1, 1>(a, stream); break;
    case 1: launch<8, 1, 2>(a, stream); break;
    case 2: launch<8, 2, 2>(a, stream); break;
    case 3: launch<4, 1, 2>(a, stream); break;
    case 4: launch<4, 2, 2>(a, stream); break;
    case 5: launch<4, 3, 2>(a, stream); break;
    default: launch<4, 3, 2, true>(a, stream); break;
  }
  NINFER_LAUNCH_CHECK();
  return 0;
}

}  // namespace ninfer

// The tile of a 32-bit product: 100 x waves + 10 x tiles of 16 rows + tiles of 16 rows of W.
extern "C" int ninfer_gemm_f32_tile(const ninfer::GemmArgs* args) {
  const ninfer::F32Tile& t = ninfer::kF32Tiles[ninfer::f32_tile(*args)];
  return 100 * t.waves + 10 * t.rt + t.ct;
}
