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
  int parts = 256 / vdim;
  if (parts < 1) parts = 1;
  if (parts > dim) parts = dim;
  const int block = parts * vdim;
  const size_t lds = ((size_t)dim * vdim + 2 * (2 * dim + vdim) + (size_t)parts * vdim) * sizeof(float);
  NINFER_REQUIRE(lds <= 160 * 1024, "lightning_attention: a head's state of %d x %d does not fit "
                 "the LDS", dim, vdim);
  const dim3 grid(S, H);
  // (a row per request as a rule; more rows than requests go through the LDS: one trip for all rows)
  if (T <= S) {
    const int cols = vdim < 64 ? vdim : 64;
    const dim3 grid(S, H, (vdim + cols - 1) / cols);
    const size_t bytes = (2 * (size_t)dim + (size_t)parts * cols) * sizeof(float);
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
// The chunks of a step lie side by side: a block per (chunk, head, 128 value columns) forms the sum
// of S' (lightning_chunk_sums), a thread per number of the state walks a request's chunks and leaves
// the state before each in the sum's place (lightning_chunk_carry), and a block per (chunk, head,
// 128 value columns) forms the outputs (lightning_chunk_outputs). That is 3 passes over 64 KB of
// state per chunk and head of 128 x 128 where one block that walks the chunks of a request keeps it
// in registers, but 512 blocks instead of 64 for a prompt of 2,048 tokens with 16 heads, and no
// chain of 32 chunks with three barriers each: 25 + 15 + 51 us against 903 for that prompt. (Three
// GFLOP are 20 us at the rate of the 32-bit matrix instruction; the sums and the outputs are bound
// by silu of the rows and LDS before it, one and two blocks a CU.)
namespace ninfer {

typedef float lt_f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 lt_bf16x8 __attribute__((ext_vector_type(8)));
constexpr int kLtChunk = 64;
constexpr int kLtCols = 128;       // value columns of a block
constexpr int kLtThreads = 512;
constexpr int kLtMaxDim = 256;
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

static int lightning_lds(const void* kern, size_t lds) {
  if (lds <= 48 * 1024) return 0;
  hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return set_error(-2, "lightning_attention: cannot get %zu bytes of LDS", lds);
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

// Floats of workspace with which a step runs in chunks; 0 when the sizes do not fit (the
// token-by-token kernel takes them).
extern "C" long long ninfer_lightning_chunk_floats(int T, int S, int H, int dim, int vdim, int dtype) {
  if (dtype != kBF16 || dim > kLtMaxDim) return 0;
  return lightning_most_chunks(T, S) * H * dim * vdim;
}

// The same as ninfer_lightning_attention for bfloat16 rows, chunk by chunk on the matrix cores:
// for steps that bring prompt portions. `work`: ninfer_lightning_chunk_floats floats.
extern "C" int ninfer_lightning_attention_chunks(const void* qkv, int stride, int q_off, int k_off,
                                                 int v_off, const float* decay, float* state,
                                                 long long state_stride, float* out,
                                                 const int* seq_row_start, const int* seq_slots,
                                                 int T, int S, int H, int dim, int vdim, int dtype,
                                                 float* work, hipStream_t stream) {
  NINFER_REQUIRE(T > 0 && S > 0 && H > 0 && dim > 0 && vdim > 0,
                 "lightning_attention: T=%d S=%d heads=%d dim=%d vdim=%d must be positive", T, S,
                 H, dim, vdim);
  NINFER_REQUIRE(state_stride >= (long long)H * dim * vdim,
                 "lightning_attention: a request's state of %lld floats holds no %d x %d x %d",
                 state_stride, H, dim, vdim);
  NINFER_REQUIRE(ninfer_lightning_chunk_floats(T, S, H, dim, vdim, dtype) > 0 && work,
                 "lightning_attention: dtype %d, key size %d do not run in chunks, or no workspace", dtype, dim);
  LightningChunks a = {(const bf16*)qkv, decay, state, out, work, seq_row_start, seq_slots, state_stride,
                       stride, q_off, k_off, v_off, S, H, dim, vdim};
  // rows whose q, k and v parts start and end at multiples of 16 bytes
  const bool wide = dim % 8 == 0 && vdim % 8 == 0 && stride % 8 == 0 && q_off % 8 == 0 && k_off % 8 == 0 &&
                    v_off % 8 == 0 && (uintptr_t)qkv % 16 == 0;
  return wide ? lightning_chunks<true>(a, T, stream) : lightning_chunks<false>(a, T, stream);
}
