// Linear attention with a per-head decay ("lightning attention"), token by token:
//
//   S_t = decay_h S_(t-1) + k_t v_t^T      (S: [dim, vdim] per head, 32-bit, per-request state)
//   o_t = S_t^T q_t
//
// q, k, v are silu of the projected rows (the activation is applied here, in 32-bit, to the
// projection's stored value). One block per (request, head) walks the request's rows of the
// step in order; the state comes from and returns to the request's slot, so a request may be
// cut into steps anywhere and every row sees exactly the sums it would see in one piece.
// Thread (part, v) owns S[d][v] for d = part, part + parts, ...: it updates them and forms its
// part of o_t[v] in the same pass; the parts are added in ascending order. The order of
// every sum depends on (dim, vdim) alone.
#include "common.h"

namespace ninfer {

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }

template <typename T>
__global__ void lightning_seq_kernel(const T* __restrict__ qkv, int stride, int q_off, int k_off,
                                     int v_off, const float* __restrict__ decay,
                                     float* __restrict__ state, int64_t state_stride,
                                     float* __restrict__ out, const int* __restrict__ seq_row_start,
                                     const int* __restrict__ seq_slots, int H, int dim, int vdim,
                                     int parts) {
  extern __shared__ float smem[];
  float* S = smem;                       // [dim * vdim]
  float* qk = S + dim * vdim;            // 2 x [2 dim + vdim]: q, k, v of a row, two buffers
  float* part_s = qk + 2 * (2 * dim + vdim);   // [parts * vdim]
  const int s = blockIdx.x, h = blockIdx.y;
  const int r0 = seq_row_start[s], n = seq_row_start[s + 1] - r0;
  float* st = state + (int64_t)seq_slots[s] * state_stride + (int64_t)h * dim * vdim;
  const int tid = threadIdx.x;
  const int vv = tid % vdim, part = tid / vdim;   // blockDim.x == parts * vdim
  for (int e = tid; e < dim * vdim; e += blockDim.x) S[e] = st[e];
  const float dec = decay[h];
  const int row_floats = 2 * dim + vdim;
  for (int i = 0; i < n; ++i) {
    float* buf = qk + (i & 1) * row_floats;
    const T* row = qkv + (int64_t)(r0 + i) * stride;
    for (int e = tid; e < row_floats; e += blockDim.x) {
      int col = e < dim ? q_off + h * dim + e
                        : e < 2 * dim ? k_off + h * dim + (e - dim) : v_off + h * vdim + (e - 2 * dim);
      buf[e] = silu_f(to_f32(row[col]));
    }
    __syncthreads();   // the row is in LDS; the state of the previous row is complete
    const float* q_s = buf;
    const float* k_s = buf + dim;
    const float v_t = buf[2 * dim + vv];
    float acc = 0.f;
    for (int d = part; d < dim; d += parts) {
      const float sn = fmaf(dec, S[d * vdim + vv], k_s[d] * v_t);
      S[d * vdim + vv] = sn;
      acc = fmaf(sn, q_s[d], acc);
    }
    part_s[part * vdim + vv] = acc;
    __syncthreads();
    if (part == 0) {
      float o = 0.f;
      for (int p = 0; p < parts; ++p) o += part_s[p * vdim + vv];
      out[((int64_t)(r0 + i) * H + h) * vdim + vv] = o;
    }
    // the next row writes the other q/k/v buffer, and part_s only after its first barrier
  }
  __syncthreads();
  for (int e = tid; e < dim * vdim; e += blockDim.x) st[e] = S[e];
}

// Steps whose requests bring a row each. What a row costs there is the state's way from memory and
// back, which the kernel above takes through the LDS: 69 KB for a head of 128 x 128, two blocks a CU.
// Here the state goes memory -> registers -> memory: a block owns up to 64 value columns of a head,
// thread (part, v) the same numbers S[d][v] as above with the sums in the same order (the same
// bits), 16 of them loaded together. A thread reads back only what it wrote, so requests of more
// rows are right too, one trip per row. 64 requests of 16 heads of 128 x 128 (134 MB there and
// back): 80 -> 35 us, 3.8 TB/s, bound by memory. (64 numbers loaded together: 76 us; blocks of 32
// columns 35, of 128 41. 8 requests 12 us, one 10: four trips to memory one after the other.)
template <typename T>
__global__ void lightning_step_kernel(const T* __restrict__ qkv, int stride, int q_off, int k_off,
                                      int v_off, const float* __restrict__ decay,
                                      float* __restrict__ state, int64_t state_stride,
                                      float* __restrict__ out, const int* __restrict__ seq_row_start,
                                      const int* __restrict__ seq_slots, int H, int dim, int vdim,
                                      int parts, int cols) {
  constexpr int B = 16;
  extern __shared__ float smem[];
  float* q_s = smem;               // [dim]
  float* k_s = q_s + dim;          // [dim]
  float* part_s = k_s + dim;       // [parts * cols]
  const int s = blockIdx.x, h = blockIdx.y;
  const int r0 = seq_row_start[s], n = seq_row_start[s + 1] - r0;
  const int tid = threadIdx.x;     // blockDim.x == parts * cols
  const int part = tid / cols, vv = (int)blockIdx.z * cols + tid % cols;
  const bool mine = vv < vdim;
  const int col = mine ? vv : vdim - 1;   // (threads beyond the last column load, and write nothing)
  float* st = state + (int64_t)seq_slots[s] * state_stride + (int64_t)h * dim * vdim + col;
  const float dec = decay[h];
  for (int i = 0; i < n; ++i) {
    const T* row = qkv + (int64_t)(r0 + i) * stride;
    float S[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {   // (on their way while q and k are prepared)
      const int d = part + u * parts;
      S[u] = st[(int64_t)(d < dim ? d : dim - 1) * vdim];
    }
    const float v_t = silu_f(to_f32(row[v_off + h * vdim + col]));
#pragma unroll 4
    for (int e = tid; e < 2 * dim; e += blockDim.x)
      q_s[e] = silu_f(to_f32(row[e < dim ? q_off + h * dim + e : k_off + h * dim + (e - dim)]));
    __syncthreads();   // q and k are in LDS; the sums of the previous row have been added
    float acc = 0.f;
    for (int d0 = part; d0 < dim; d0 += B * parts) {
      if (d0 != part) {
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const int d = d0 + u * parts;
          S[u] = st[(int64_t)(d < dim ? d : dim - 1) * vdim];
        }
      }
#pragma unroll
      for (int u = 0; u < B; ++u) {
        const int d = d0 + u * parts;
        if (d < dim) {
          const float sn = fmaf(dec, S[u], k_s[d] * v_t);
          if (mine) st[(int64_t)d * vdim] = sn;
          acc = fmaf(sn, q_s[d], acc);
        }
      }
    }
    part_s[tid] = acc;
    __syncthreads();
    if (part == 0 && mine) {
      float o = 0.f;
      for (int p = 0; p < parts; ++p) o += part_s[p * cols + tid];
      out[((int64_t)(r0 + i) * H + h) * vdim + vv] = o;
    }
    // (part_s is written again only after the next row's first barrier)
  }
}

// Threads that share a value column.
static int lightning_parts(int dim, int vdim) {
  const int parts = vdim < 256 ? 256 / vdim : 1;
  return parts < dim ? parts : dim;
}

static size_t lightning_seq_lds(int dim, int vdim) {
  return ((size_t)dim * vdim + 2 * (2 * dim + vdim) + (size_t)lightning_parts(dim, vdim) * vdim) * sizeof(float);
}

}  // namespace ninfer

using namespace ninfer;

// qkv: [T, stride] rows of the activation dtype with the heads' q at column q_off, k at
// k_off (heads x dim each) and v at v_off (heads x vdim); out: [T, heads * vdim] 32-bit.
extern "C" int ninfer_lightning_attention(const void* qkv, int stride, int q_off, int k_off,
                                          int v_off, const float* decay, float* state,
                                          long long state_stride, float* out,
                                          const int* seq_row_start, const int* seq_slots, int T,
                                          int S, int H, int dim, int vdim, int dtype,
                                          hipStream_t stream) {
  NINFER_REQUIRE(T > 0 && S > 0 && H > 0 && dim > 0 && vdim > 0,
                 "lightning_attention: T=%d S=%d heads=%d dim=%d vdim=%d must be positive", T, S,
                 H, dim, vdim);
  NINFER_REQUIRE(vdim <= 1024, "lightning_attention: value size %d exceeds 1024", vdim);
  NINFER_REQUIRE(state_stride >= (long long)H * dim * vdim,
                 "lightning_attention: a request's state of %lld floats holds no %d x %d x %d",
                 state_stride, H, dim, vdim);
  NINFER_REQUIRE(dtype == kF32 || dtype == kBF16, "lightning_attention: unknown dtype %d", dtype);
  const int parts = lightning_parts(dim, vdim);
  const int block = parts * vdim;
  const size_t lds = lightning_seq_lds(dim, vdim);
  NINFER_REQUIRE(lds <= 160 * 1024, "lightning_attention: a head's state of %d x %d does not fit "
                 "the LDS", dim, vdim);
  const dim3 grid(S, H);
  // (a row per request as a rule; more rows than requests go through the LDS: one trip for all rows; so
  // do small states, many of which fit a CU's LDS: us there and in registers, heads of 16 x 16 of 256
  // requests 6.7 and 11.9, of 64 x 16 of 64 4.6 and 5.7, of 48 x 48 of 256 8.8 and 10.4, but of 100 x 40
  // of 64 7.6 and 7.0, of 64 x 64 and more less still)
  const int cols = vdim < 64 ? vdim : 64;
  const size_t bytes = (2 * (size_t)dim + (size_t)parts * cols) * sizeof(float);
  if (T <= S && dim * vdim >= 3000 && bytes <= 48 * 1024) {
    const dim3 grid(S, H, (vdim + cols - 1) / cols);
#define NINFER_LIGHTNING_STEP(TYPE)                                                             \
  lightning_step_kernel<TYPE><<<grid, parts * cols, bytes, stream>>>(                           \
      (const TYPE*)qkv, stride, q_off, k_off, v_off, decay, state, state_stride, out,           \
      seq_row_start, seq_slots, H, dim, vdim, parts, cols)
    if (dtype == kF32) NINFER_LIGHTNING_STEP(float); else NINFER_LIGHTNING_STEP(bf16);
#undef NINFER_LIGHTNING_STEP
    NINFER_LAUNCH_CHECK();
    return 0;
  }
#define NINFER_LIGHTNING_LAUNCH(TYPE)                                                          \
  do {                                                                                         \
    auto kern = lightning_seq_kernel<TYPE>;                                                    \
    if (lds > 48 * 1024) {                                                                     \
      hipError_t e = hipFuncSetAttribute((const void*)kern,                                    \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
      if (e != hipSuccess) return set_error(-2, "lightning_attention: cannot get %zu bytes of LDS", lds); \
    }                                                                                          \
    kern<<<grid, block, lds, stream>>>((const TYPE*)qkv, stride, q_off, k_off, v_off, decay,   \
                                       state, state_stride, out, seq_row_start, seq_slots, H,  \
                                       dim, vdim, parts);                                      \
  } while (0)
  if (dtype == kF32)
    NINFER_LIGHTNING_LAUNCH(float);
  else
    NINFER_LIGHTNING_LAUNCH(bf16);
#undef NINFER_LIGHTNING_LAUNCH
  NINFER_LAUNCH_CHECK();
  return 0;
}

// ---- prompt portions in chunks, on the 32-bit matrix instruction --------------------------------
//
// For the rows i = 0 .. L - 1 of a chunk (L <= 64) with the state S before it:
//
//   o_i = sum_{j <= i} d^(i - j) (q_i . k_j) v_j  +  d^(i + 1) S^T q_i
//   S' = d^L S + sum_j d^(L - 1 - j) k_j v_j^T
//
// which is the recurrence written out; all powers of the decay have exponents >= 0, so nothing
// grows. Every product runs on v_mfma_f32_32x32x2_f32: q, k, v (silu of the projections), the
// decays and the state enter in 32-bit and are never rounded to a shorter type.
//
// Two forms, and single rows apart from both:
//
//   side by side  a block per (chunk, head, 128 value columns) forms the sum of S' (lightning_chunk_sums),
//                 a thread per number of the state walks a request's chunks and leaves the state before
//                 each in the sum's place (lightning_chunk_carry), and a block per (chunk, head, 128 value
//                 columns) forms the outputs (lightning_chunk_outputs). That is 3 passes over 64 KB of state
//                 per chunk and head of 128 x 128, but 512 blocks for a prompt of 2,048 tokens with 16
//                 heads, and no chain of 32 chunks: 25 + 15 + 51 us against 903 of the walk. (Three GFLOP
//                 are 20 us at the rate of the 32-bit matrix instruction; the sums and the outputs are
//                 bound by silu of the rows and LDS before it, one and two blocks a CU.)
//   the walk      a block per (request, head, 32 value columns) takes the request's chunks one after the
//                 other with the state in registers: one launch, and the state goes to memory and back
//                 once. Better for short portions: one of 8 to 64 rows 26 to 31 us against 40 to 47.
//   single rows   requests of one row, the step's first, may go through lightning_step_kernel beside either
//                 form, which would take each for a chunk: 64 of them and a portion of 448 rows 508 us as
//                 chunks side by side, 83 apart.
//
// lightning_form chooses by an estimate of all four.
namespace ninfer {

typedef float lt_f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 lt_bf16x8 __attribute__((ext_vector_type(8)));
constexpr int kLtChunk = 64;
constexpr int kLtCols = 128;       // value columns of a block
constexpr int kLtThreads = 512;
constexpr int kLtMaxDim = 256;
constexpr int kLtStateTiles = 4;   // 32-row tiles of the state of a carrying wave (the walk): dim up to 256
constexpr int kLtTile = 32 * 33;   // a 32 x 32 tile of decayed scores in LDS

struct LightningChunks {
  const bf16* qkv;
  const float* decay;
  float* state;
  float* out;
  float* sums;   // [chunks, H, dim, vdim]: a chunk's sum, then the state before it
  const int* seq_row_start;
  const int* seq_slots;
  int64_t state_stride;
  int stride, q_off, k_off, v_off, S, H, dim, vdim;
};

__device__ __forceinline__ float decay_pow(float log2d, int n) {
  return n == 0 ? 1.f : exp2f((float)n * log2d);   // (a decay of 0 has log2 -inf: 0 * -inf is no number)
}

// Chunk `at` of the step, chunks counted request after request.
__device__ __forceinline__ bool lightning_find_chunk(const LightningChunks& a, int at, int* row0, int* rows) {
  for (int s = 0; s < a.S; ++s) {
    const int r = a.seq_row_start[s], n = a.seq_row_start[s + 1] - r;
    const int chunks = (n + kLtChunk - 1) / kLtChunk;
    if (at < chunks) {
      *row0 = r + at * kLtChunk;
      *rows = min(kLtChunk, n - at * kLtChunk);
      return true;
    }
    at -= chunks;
  }
  return false;
}

// A block walks one request's chunks, 32 value columns of a head: waves 0 and 1 form a chunk's
// outputs, waves 2 and 3 carry the state in their accumulators and hand a copy to the others through LDS.
template <bool WIDE>
__global__ __launch_bounds__(256) void lightning_walk_kernel(LightningChunks a) {
  extern __shared__ float smem[];
  const int dim = a.dim, vdim = a.vdim, H = a.H;
  const bf16* qkv = a.qkv;
  const int stride = a.stride, q_off = a.q_off, k_off = a.k_off, v_off = a.v_off;
  const int qs = dim + 1;                 // row length of q and k in LDS (odd: column reads spread)
  float* Qs = smem;                       // [64][dim + 1]
  float* Ks = Qs + kLtChunk * qs;         // [64][dim + 1]
  float* Vs = Ks + kLtChunk * qs;         // [64][33]
  float* As = Vs + kLtChunk * 33;         // [64][65]
  float* Ss = As + kLtChunk * 65;         // [dim32][33]
  float* Ws = Ss + ((dim + 31) / 32 * 32) * 33;   // [64] d^(L - 1 - j) of the chunk's rows
  const int s = blockIdx.x, h = blockIdx.y, c0 = 32 * blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 31, lk = lane >> 5;
  const int r0 = a.seq_row_start[s], n = a.seq_row_start[s + 1] - r0;
  const int dim32 = (dim + 31) / 32 * 32;
  const int d_tiles = dim32 / 32;
  float* st = a.state + (int64_t)a.seq_slots[s] * a.state_stride + (int64_t)h * dim * vdim;
  const float log2d = log2f(a.decay[h]);
  const bool col_ok = c0 + lr < vdim;
  // the state: in the accumulators of waves 2 and 3 (tiles w - 2, w, ...), a copy in LDS
  lt_f32x16 sacc[kLtStateTiles] = {};
  for (int e = tid; e < dim32 * 33; e += 256) {
    const int d = e / 33, c = e % 33;
    Ss[e] = (d < dim && c < 32 && c0 + c < vdim) ? st[(int64_t)d * vdim + c0 + c] : 0.f;
  }
  __syncthreads();
  if (w >= 2) {
#pragma unroll
    for (int x = 0; x < kLtStateTiles; ++x) {
      const int dt = (w - 2) + 2 * x;
      if (dt < d_tiles) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) sacc[x][4 * q + r] = Ss[(32 * dt + 8 * q + 4 * lk + r) * 33 + lr];
      }
    }
  }

  for (int i0 = 0; i0 < n; i0 += kLtChunk) {
    const int L = min(kLtChunk, n - i0);
    // 1. the chunk's q, k (all of the head's numbers) and this block's value columns
    if (WIDE) {   // eight neighbouring numbers per load
      const int per_row = dim / 8;
      for (int e = tid; e < kLtChunk * per_row; e += 256) {
        const int i = e / per_row, d = 8 * (e % per_row);
        float qv[8], kv[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) qv[x] = kv[x] = 0.f;
        if (i < L) {
          const bf16* row = qkv + (int64_t)(r0 + i0 + i) * stride;
          const lt_bf16x8 qx = *(const lt_bf16x8*)(row + q_off + h * dim + d);
          const lt_bf16x8 kx = *(const lt_bf16x8*)(row + k_off + h * dim + d);
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            qv[x] = silu_f((float)qx[x]);
            kv[x] = silu_f((float)kx[x]);
          }
        }
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          Qs[i * qs + d + x] = qv[x];
          Ks[i * qs + d + x] = kv[x];
        }
      }
    } else {
      for (int e = tid; e < kLtChunk * dim; e += 256) {
        const int i = e / dim, d = e % dim;
        float qv = 0.f, kv = 0.f;
        if (i < L) {
          const bf16* row = qkv + (int64_t)(r0 + i0 + i) * stride;
          qv = silu_f(to_f32(row[q_off + h * dim + d]));
          kv = silu_f(to_f32(row[k_off + h * dim + d]));
        }
        Qs[i * qs + d] = qv;
        Ks[i * qs + d] = kv;
      }
    }
    for (int e = tid; e < kLtChunk * 32; e += 256) {
      const int i = e >> 5, c = e & 31;
      float vv = 0.f;
      if (i < L && c0 + c < vdim)
        vv = silu_f(to_f32(qkv[(int64_t)(r0 + i0 + i) * stride + v_off + h * vdim + c0 + c]));
      Vs[i * 33 + c] = vv;
    }
    if (tid < kLtChunk) Ws[tid] = tid < L ? decay_pow(log2d, L - 1 - tid) : 0.f;
    __syncthreads();   // (also: the state's copy in LDS is the one before this chunk)
    // 2. A[i][j] = d^(i - j) q_i . k_j for j <= i: wave w has rows 32 (w / 2).., keys 32 (w % 2)..
    {
      const int mi = w >> 1, nj = w & 1;
      lt_f32x16 sc = {};
      if (nj <= mi) {
        const float* qrow = Qs + (32 * mi + lr) * qs + lk;
        const float* krow = Ks + (32 * nj + lr) * qs + lk;
#pragma unroll 8
        for (int d = 0; d < dim; d += 2) {
          const float qa = (d + lk < dim) ? qrow[d] : 0.f;
          const float kb = (d + lk < dim) ? krow[d] : 0.f;
          sc = __builtin_amdgcn_mfma_f32_32x32x2f32(qa, kb, sc, 0, 0, 0);
        }
      }
      const int j = 32 * nj + lr;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 32 * mi + 8 * q + 4 * lk + r;
          As[i * 65 + j] = j <= i ? sc[4 * q + r] * decay_pow(log2d, i - j) : 0.f;
        }
    }
    __syncthreads();
    // 3. waves 0, 1: the outputs of rows 32 w ..; waves 2, 3: the state after the chunk
    if (w < 2) {
      lt_f32x16 o = {};
      const int row = 32 * w + lr;
      const float* arow = As + row * 65 + lk;
#pragma unroll 8
      for (int j = 0; j < 32 * (w + 1); j += 2)
        o = __builtin_amdgcn_mfma_f32_32x32x2f32(arow[j], Vs[(j + lk) * 33 + lr], o, 0, 0, 0);
      const float carry = decay_pow(log2d, row + 1);
      const float* qrow = Qs + row * qs + lk;
#pragma unroll 8
      for (int d = 0; d < dim; d += 2) {
        const float qa = (d + lk < dim) ? qrow[d] * carry : 0.f;
        o = __builtin_amdgcn_mfma_f32_32x32x2f32(qa, Ss[(d + lk) * 33 + lr], o, 0, 0, 0);
      }
      if (col_ok) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = 32 * w + 8 * q + 4 * lk + r;
            if (i < L) a.out[((int64_t)(r0 + i0 + i) * H + h) * vdim + c0 + lr] = o[4 * q + r];
          }
      }
    } else {
      const float whole = decay_pow(log2d, L);
#pragma unroll
      for (int x = 0; x < kLtStateTiles; ++x) {
        const int dt = (w - 2) + 2 * x;
        if (dt < d_tiles) {
#pragma unroll
          for (int i = 0; i < 16; ++i) sacc[x][i] *= whole;
          const int d = 32 * dt + lr;
#pragma unroll 8
          for (int j = 0; j < kLtChunk; j += 2) {
            const int jj = j + lk;
            const float ka = (jj < L && d < dim) ? Ks[jj * qs + d] * Ws[jj] : 0.f;
            sacc[x] = __builtin_amdgcn_mfma_f32_32x32x2f32(ka, Vs[jj * 33 + lr], sacc[x], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();   // everyone has read the old copy of the state
    if (w >= 2) {
#pragma unroll
      for (int x = 0; x < kLtStateTiles; ++x) {
        const int dt = (w - 2) + 2 * x;
        if (dt < d_tiles) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) Ss[(32 * dt + 8 * q + 4 * lk + r) * 33 + lr] = sacc[x][4 * q + r];
        }
      }
    }
    // (the barrier after the next chunk's loads publishes the copy; nothing reads it before)
  }
  if (w >= 2 && col_ok) {
#pragma unroll
    for (int x = 0; x < kLtStateTiles; ++x) {
      const int dt = (w - 2) + 2 * x;
      if (dt < d_tiles) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int d = 32 * dt + 8 * q + 4 * lk + r;
            if (d < dim) st[(int64_t)d * vdim + c0 + lr] = sacc[x][4 * q + r];
          }
      }
    }
  }
}

// Columns col .. col + width - 1 of the chunk's rows, silu applied, times `scale` per row where
// given, into LDS rows of `row` floats, zeros beyond the last row and from `width` to `padded`
// (a multiple of 8). WIDE: the columns start and end at multiples of 16 bytes.
template <bool WIDE>
__device__ __forceinline__ void lightning_rows(const LightningChunks& a, int row0, int L, int col, int width,
                                               int padded, float* lds, int row, const float* scale) {
  const bf16* rows = a.qkv + (int64_t)row0 * a.stride + col;
  const int per_row = padded / 8;
  for (int e = threadIdx.x; e < kLtChunk * per_row; e += kLtThreads) {
    const int i = e / per_row, d = 8 * (e % per_row);
    float z[8];
    if (WIDE) {
      const lt_bf16x8 x = *(const lt_bf16x8*)(rows + (int64_t)min(i, L - 1) * a.stride + min(d, width - 8));
#pragma unroll
      for (int n = 0; n < 8; ++n) z[n] = (float)x[n];
    } else {
#pragma unroll
      for (int n = 0; n < 8; ++n) z[n] = to_f32(rows[(int64_t)min(i, L - 1) * a.stride + min(d + n, width - 1)]);
    }
    const float f = scale ? scale[i] : 1.f;
#pragma unroll
    for (int n = 0; n < 8; ++n) lds[i * row + d + n] = i < L && d + n < width ? silu_f(z[n]) * f : 0.f;
  }
}

// sum_j d^(L - 1 - j) k_j v_j^T of a chunk. The 32 x 32 tiles of [dim, 128 columns] go round the waves.
template <bool WIDE>
__global__ __launch_bounds__(kLtThreads) void lightning_chunk_sums_kernel(LightningChunks a) {
  extern __shared__ float smem[];
  __shared__ float w_s[kLtChunk];
  int row0, L;
  if (!lightning_find_chunk(a, blockIdx.x, &row0, &L)) return;
  const int h = blockIdx.y, c0 = kLtCols * blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, lr = lane & 31, lk = lane >> 5;
  const int dim32 = (a.dim + 31) / 32 * 32, ks = dim32 + 1, vs = kLtCols + 1;
  float* Ks = smem;                       // [64][dim32 + 1], times the decay to the chunk's end
  float* Vs = Ks + kLtChunk * ks;         // [64][129]
  if (tid < kLtChunk) w_s[tid] = tid < L ? decay_pow(log2f(a.decay[h]), L - 1 - tid) : 0.f;
  __syncthreads();
  lightning_rows<WIDE>(a, row0, L, a.k_off + h * a.dim, a.dim, dim32, Ks, ks, w_s);
  lightning_rows<WIDE>(a, row0, L, a.v_off + h * a.vdim + c0, min(kLtCols, a.vdim - c0), kLtCols, Vs, vs, nullptr);
  __syncthreads();
  float* sum = a.sums + ((int64_t)blockIdx.x * a.H + h) * a.dim * a.vdim;
  for (int t = w; t < dim32 / 32 * (kLtCols / 32); t += kLtThreads / 64) {
    const int dt = t / (kLtCols / 32), ct = t % (kLtCols / 32);
    if (c0 + 32 * ct >= a.vdim) continue;
    lt_f32x16 acc = {};
    const float* kc = Ks + lk * ks + 32 * dt + lr;
    const float* vc = Vs + lk * vs + 32 * ct + lr;
#pragma unroll 8
    for (int j = 0; j < kLtChunk; j += 2)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kc[j * ks], vc[j * vs], acc, 0, 0, 0);
    const int c = c0 + 32 * ct + lr;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 32 * dt + 8 * q + 4 * lk + r;
        if (d < a.dim && c < a.vdim) sum[(int64_t)d * a.vdim + c] = acc[4 * q + r];
      }
  }
}

// S before every chunk in place of the chunk's sum, and the state after the last.
__global__ __launch_bounds__(256) void lightning_chunk_carry_kernel(LightningChunks a) {
  const int64_t numbers = (int64_t)a.H * a.dim * a.vdim, e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= numbers) return;
  const int s = blockIdx.y;
  int first = 0;
  for (int i = 0; i < s; ++i) first += (a.seq_row_start[i + 1] - a.seq_row_start[i] + kLtChunk - 1) / kLtChunk;
  const int n = a.seq_row_start[s + 1] - a.seq_row_start[s], count = (n + kLtChunk - 1) / kLtChunk;
  const float log2d = log2f(a.decay[e / ((int64_t)a.dim * a.vdim)]);
  const float whole = decay_pow(log2d, kLtChunk);
  float* slot = a.state + (int64_t)a.seq_slots[s] * a.state_stride + e;
  float* at = a.sums + first * numbers + e;
  float S = *slot;
  for (int i0 = 0; i0 < count; i0 += 8) {
    float sum[8];   // eight loads on their way before the first is used
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] = at[min(i0 + i, count - 1) * numbers];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i0 + i < count) {
        at[(i0 + i) * numbers] = S;
        S = S * (i0 + i + 1 < count ? whole : decay_pow(log2d, n - (count - 1) * kLtChunk)) + sum[i];
      }
  }
  *slot = S;
}

// The outputs of a chunk: wave w has rows 32 (w / 4) .. and value columns 32 (w % 4) .. of the
// block's 128. The decayed scores are formed once, by three waves; values take the keys' place.
template <bool WIDE>
__global__ __launch_bounds__(kLtThreads) void lightning_chunk_outputs_kernel(LightningChunks a) {
  extern __shared__ float smem[];
  int row0, L;
  if (!lightning_find_chunk(a, blockIdx.x, &row0, &L)) return;
  const int h = blockIdx.y, c0 = kLtCols * blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, lr = lane & 31, lk = lane >> 5;
  const int dim32 = (a.dim + 31) / 32 * 32, qs = dim32 + 1, vs = kLtCols + 1;
  const float log2d = log2f(a.decay[h]);
  float* Qs = smem;                        // [64][dim32 + 1]
  float* As = Qs + kLtChunk * qs;          // scores of tiles (0, 0), (1, 0), (1, 1)
  float* Ks = As + 3 * kLtTile;            // [64][dim32 + 1], then the values [64][129]
  lightning_rows<WIDE>(a, row0, L, a.q_off + h * a.dim, a.dim, dim32, Qs, qs, nullptr);
  lightning_rows<WIDE>(a, row0, L, a.k_off + h * a.dim, a.dim, dim32, Ks, qs, nullptr);
  __syncthreads();
  if (w < 3) {
    const int mi = w > 0, nj = w > 1;
    lt_f32x16 s = {};
    const float* qrow = Qs + (32 * mi + lr) * qs + lk;
    const float* krow = Ks + (32 * nj + lr) * qs + lk;
#pragma unroll 8
    for (int d = 0; d < dim32; d += 2) s = __builtin_amdgcn_mfma_f32_32x32x2f32(qrow[d], krow[d], s, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 8 * q + 4 * lk + r, back = 32 * (mi - nj) + i - lr;
        As[w * kLtTile + i * 33 + lr] = back >= 0 ? s[4 * q + r] * decay_pow(log2d, back) : 0.f;
      }
  }
  __syncthreads();
  float* Vs = Ks;
  lightning_rows<WIDE>(a, row0, L, a.v_off + h * a.vdim + c0, min(kLtCols, a.vdim - c0), kLtCols, Vs, vs, nullptr);
  __syncthreads();
  const int mi = w >> 2, col = 32 * (w & 3);
  if (c0 + col >= a.vdim || 32 * mi >= L) return;
  const int c = min(c0 + col + lr, a.vdim - 1);
  lt_f32x16 o = {};
  for (int nj = 0; nj <= mi; ++nj) {
    const float* arow = As + (mi + nj) * kLtTile + lr * 33 + lk;
#pragma unroll 8
    for (int j = 0; j < 32; j += 2)
      o = __builtin_amdgcn_mfma_f32_32x32x2f32(arow[j], Vs[(32 * nj + j + lk) * vs + col + lr], o, 0, 0, 0);
  }
  const float carry = decay_pow(log2d, 32 * mi + lr + 1);
  const float* qrow = Qs + (32 * mi + lr) * qs + lk;
  const float* S = a.sums + ((int64_t)blockIdx.x * a.H + h) * a.dim * a.vdim + c;
#pragma unroll 16
  for (int d = 0; d < dim32; d += 2)   // (queries beyond dim are zeros)
    o = __builtin_amdgcn_mfma_f32_32x32x2f32(qrow[d] * carry, S[(int64_t)min(d + lk, a.dim - 1) * a.vdim], o, 0, 0, 0);
  if (c0 + col + lr >= a.vdim) return;
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 32 * mi + 8 * q + 4 * lk + r;
      if (i < L) a.out[((int64_t)(row0 + i) * a.H + h) * a.vdim + c] = o[4 * q + r];
    }
}

static int64_t lightning_most_chunks(int T, int S) { return T / kLtChunk + S; }   // no step has more

static size_t lightning_walk_lds(int dim) {
  const int dim32 = (dim + 31) / 32 * 32;
  return ((size_t)2 * kLtChunk * (dim + 1) + kLtChunk * 33 + kLtChunk * 65 + (size_t)dim32 * 33 + kLtChunk) * sizeof(float);
}

struct LightningForm {
  int apart;   // requests of one row that lightning_step_kernel takes
  bool side;   // the others' chunks side by side, not by the walk
};

// What a step of T rows in S requests takes each way, in us on this part (1 us more or less where one
// launch is enough; 16 heads of 128 x 128: the walk 26 for up to 8 rows, 31 for 64, 49 for two chunks and
// 23 for each more, times the rounds of its blocks, one to a CU, and part of one more; side by side 43 and
// 1.2 for every chunk, 3.2 for every request; single rows 9 and 0.4 each). `single` of the requests, the
// first, bring one row each.
static LightningForm lightning_form(int T, int S, int single, int max_qlen, int H, int dim, int vdim) {
  const float numbers = (float)H * dim * vdim / (16 * 128 * 128), longest = (max_qlen + kLtChunk - 1) / kLtChunk;
  const bool walks = lightning_walk_lds(dim) <= 160 * 1024;
  auto walk = [&](int requests) {
    const float rounds = (float)requests * H * ((vdim + 31) / 32) / device_cu_count();
    return (rounds > 1.f ? rounds + 0.4f : 1.f) * (3.f + longest * (5.f + 18.f * dim / 128));
  };
  auto side = [&](int rows, int requests) {
    return 43.f + numbers * (1.2f * (rows / kLtChunk + requests) + 3.2f * requests);
  };
  const float apart = single > 0 ? 9.f + 0.4f * single * numbers : 0.f;
  LightningForm best = {0, true};
  float least = side(T, S);
  auto look = [&](float us, int a, bool s) {
    if (us < least) least = us, best = {a, s};
  };
  if (walks) look(walk(S), 0, false);
  if (single > 0 && single < S && lightning_seq_lds(dim, vdim) <= 160 * 1024) {
    look(apart + side(T - single, S - single), single, true);
    if (walks) look(apart + walk(S - single), single, false);
  }
  return best;
}

static int lightning_lds(const void* kern, size_t lds) {
  if (lds <= 48 * 1024) return 0;
  hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return set_error(-2, "lightning_attention: cannot get %zu bytes of LDS", lds);
  return 0;
}

template <bool WIDE>
static int lightning_walk(const LightningChunks& a, hipStream_t stream) {
  const size_t lds = lightning_walk_lds(a.dim);
  if (int rc = lightning_lds((const void*)lightning_walk_kernel<WIDE>, lds)) return rc;
  lightning_walk_kernel<WIDE><<<dim3(a.S, a.H, (a.vdim + 31) / 32), 256, lds, stream>>>(a);
  NINFER_LAUNCH_CHECK();
  return 0;
}

template <bool WIDE>
static int lightning_chunks(const LightningChunks& a, int T, hipStream_t stream) {
  const int qs = (a.dim + 31) / 32 * 32 + 1, vs = kLtCols + 1;
  const size_t rows = (size_t)kLtChunk * sizeof(float);
  const size_t lds_sums = rows * (qs + vs), lds_out = rows * (qs + (qs > vs ? qs : vs)) + 3 * kLtTile * sizeof(float);
  if (int rc = lightning_lds((const void*)lightning_chunk_sums_kernel<WIDE>, lds_sums)) return rc;
  if (int rc = lightning_lds((const void*)lightning_chunk_outputs_kernel<WIDE>, lds_out)) return rc;
  const dim3 grid(lightning_most_chunks(T, a.S), a.H, (a.vdim + kLtCols - 1) / kLtCols);
  const int64_t numbers = (int64_t)a.H * a.dim * a.vdim;
  lightning_chunk_sums_kernel<WIDE><<<grid, kLtThreads, lds_sums, stream>>>(a);
  NINFER_LAUNCH_CHECK();
  lightning_chunk_carry_kernel<<<dim3((numbers + 255) / 256, a.S), 256, 0, stream>>>(a);
  NINFER_LAUNCH_CHECK();
  lightning_chunk_outputs_kernel<WIDE><<<grid, kLtThreads, lds_out, stream>>>(a);
  NINFER_LAUNCH_CHECK();
  return 0;
}

}  // namespace ninfer

// Can a step of these sizes run in chunks? (If not, the token-by-token kernel takes it. Keys too long for
// the walk come here if the kernel for single rows takes their state: a prompt that could not go on
// token by token is refused there.)
static bool lightning_chunks_take(int dim, int vdim, int dtype) {
  return dtype == kBF16 && dim <= kLtMaxDim &&
         (lightning_walk_lds(dim) <= 160 * 1024 || lightning_seq_lds(dim, vdim) <= 160 * 1024);
}

// Floats of workspace that ninfer_lightning_attention_chunks needs for a step, 0 for none; -1 when the sizes
// do not fit (the token-by-token kernel takes them).
extern "C" long long ninfer_lightning_chunk_floats(int T, int S, int single, int max_qlen, int H, int dim, int vdim,
                                                   int dtype) {
  if (!lightning_chunks_take(dim, vdim, dtype)) return -1;
  // (keys too long for the walk: side by side costs 64 us and more, token by token 7 us a row: 4 heads of
  // 256 x 64, 16 portions of 9 rows 82 and 63 us, one of 8 64 and 57, one of 30 68 and 181)
  if (max_qlen < 10 && lightning_walk_lds(dim) > 160 * 1024 && lightning_seq_lds(dim, vdim) <= 160 * 1024) return -1;
  const LightningForm f = lightning_form(T, S, single, max_qlen, H, dim, vdim);
  return f.side ? lightning_most_chunks(T - f.apart, S - f.apart) * H * dim * vdim : 0;
}

// The same as ninfer_lightning_attention for bfloat16 rows, chunk by chunk on the matrix cores: for steps that
// bring prompt portions. The first `single` requests bring one row each, the longest brings max_qlen rows.
// `work`: ninfer_lightning_chunk_floats floats.
extern "C" int ninfer_lightning_attention_chunks(const void* qkv, int stride, int q_off, int k_off,
                                                 int v_off, const float* decay, float* state,
                                                 long long state_stride, float* out,
                                                 const int* seq_row_start, const int* seq_slots,
                                                 int T, int S, int H, int dim, int vdim, int dtype,
                                                 int single, int max_qlen, float* work, hipStream_t stream) {
  NINFER_REQUIRE(T > 0 && S > 0 && H > 0 && dim > 0 && vdim > 0,
                 "lightning_attention: T=%d S=%d heads=%d dim=%d vdim=%d must be positive", T, S,
                 H, dim, vdim);
  NINFER_REQUIRE(single >= 0 && single <= S && single <= T && max_qlen > 0,
                 "lightning_attention: %d single rows of %d requests, %d rows the longest", single, S, max_qlen);
  NINFER_REQUIRE(state_stride >= (long long)H * dim * vdim,
                 "lightning_attention: a request's state of %lld floats holds no %d x %d x %d",
                 state_stride, H, dim, vdim);
  NINFER_REQUIRE(lightning_chunks_take(dim, vdim, dtype),
                 "lightning_attention: dtype %d, key size %d do not run in chunks", dtype, dim);
  const LightningForm f = lightning_form(T, S, single, max_qlen, H, dim, vdim);
  NINFER_REQUIRE(!f.side || work, "lightning_attention: no workspace");
  if (f.apart) {
    if (int rc = ninfer_lightning_attention(qkv, stride, q_off, k_off, v_off, decay, state, state_stride, out,
                                            seq_row_start, seq_slots, f.apart, f.apart, H, dim, vdim, dtype, stream))
      return rc;
  }
  // (rows are counted from the step's first whatever the first request)
  LightningChunks a = {(const bf16*)qkv, decay, state, out, work, seq_row_start + f.apart, seq_slots + f.apart,
                       state_stride, stride, q_off, k_off, v_off, S - f.apart, H, dim, vdim};
  // rows whose q and k parts, and v parts, start and end at multiples of 16 bytes
  const bool wide_qk = dim % 8 == 0 && stride % 8 == 0 && q_off % 8 == 0 && k_off % 8 == 0 && (uintptr_t)qkv % 16 == 0;
  const bool wide = wide_qk && vdim % 8 == 0 && v_off % 8 == 0;
  if (!f.side) return wide_qk ? lightning_walk<true>(a, stream) : lightning_walk<false>(a, stream);
  return wide ? lightning_chunks<true>(a, T - f.apart, stream) : lightning_chunks<false>(a, T - f.apart, stream);
}
