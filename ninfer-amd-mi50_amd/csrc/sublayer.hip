// Row-wise kernels around a sublayer whose norm sits on its output:
//
//   short_conv     h_t + sum_j w[:, j] h_(t - taps + 1 + j): a causal convolution over the
//                  rows of each request, channel by channel, added to its input. The last
//                  taps - 1 inputs of a request are per-request state (32-bit), so a request
//                  may be cut into steps anywhere; before a request's start they are zero.
//   norm_add       x += y rsqrt(mean(y^2) + eps) g, g one number or one per channel; optionally
//                  with the row's mean taken off first (a layer norm), and with y a weighted
//                  sum of rows.
//   gated_rmsnorm  out = o rsqrt(mean(o^2) + eps) w sigmoid(g) (or w g sigmoid(g)), the norm
//                  over the whole row or over every group of columns (a head's) by itself;
//                  without a gate the last factor is 1. Or with the gate in front of the norm,
//                  o <- o act(g) first; with a divisor per group, o <- o / den first.
//   post_norm      x <- z rsqrt(mean(z^2) + eps) g with z = alpha x + y, written in 32-bit and
//                  once more in the activation dtype for whoever reads x next; y a row, a
//                  weighted sum of rows, or half-and-half of two normed rows.
//
// All sums are 32-bit and their order depends on the row alone (taps ascending; the block
// reduction's order depends on the width), never on how a request was cut or on the batch.
#include "common.h"

namespace ninfer {

// out[t, c] for all rows. Inputs before the step's first row of a request come from the
// request's state: state[slot][i * H + c] is the input at the request's position
// pos0 - (taps - 1) + i. With `update` (steps in which every request brings one row) the
// thread also shifts the state; otherwise short_conv_state_kernel does so afterwards.
template <typename T>
__global__ void short_conv_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                  float* __restrict__ state, int64_t state_stride,
                                  T* __restrict__ out, const int* __restrict__ row_seq,
                                  const int* __restrict__ seq_row_start,
                                  const int* __restrict__ seq_slots, int H, int taps, int update) {
  const int t = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= H) return;
  const int s = row_seq[t];
  const int r0 = seq_row_start[s];
  const int i = t - r0;
  float* st = state + (int64_t)seq_slots[s] * state_stride;
  const float* wc = w + (int64_t)c * taps;
  const float cur = x[(int64_t)t * H + c];
  float acc = 0.f;
  for (int j = 0; j < taps; ++j) {
    const int src = i - (taps - 1 - j);
    const float v = src >= 0 ? x[(int64_t)(r0 + src) * H + c] : st[(int64_t)(taps - 1 + src) * H + c];
    acc = fmaf(wc[j], v, acc);
  }
  out[(int64_t)t * H + c] = from_f32<T>(cur + acc);
  if (update) {   // this row is the request's only one: the state moves on by one input
    for (int k = 0; k + 2 < taps; ++k) st[(int64_t)k * H + c] = st[(int64_t)(k + 1) * H + c];
    if (taps > 1) st[(int64_t)(taps - 2) * H + c] = cur;
  }
}

// The same for 2 to 4 taps and rows of whole 16-byte pieces: a thread has four channels of ROWS
// neighbouring rows, their weights in registers, and loads the ROWS + TAPS - 1 input rows that they see
// at once. The same sums in the same order.
// SINGLE: every request brings one row, and the thread shifts its state. Else the state is the business of the
// thread whose rows hold the request's first one. It also has those of the TAPS - 2 rows behind
// that see the old state (nobody else reads it, wherever the rows fall), and writes the new state when
// they are done.
// Memory-bound. 2,048 rows of 2,048 channels with four taps (16 MB in, 8 MB out): 8.6 us from launch to launch,
// where loading each row's four inputs by themselves and the state in a launch of its own took 10.9, and a
// thread per number with its weights fetched one by one 23.
template <typename T, int TAPS, int ROWS, bool SINGLE>
__global__ __launch_bounds__(256) void short_conv_rows_kernel(
    const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ state, int64_t state_stride,
    T* __restrict__ out, const int* __restrict__ row_seq, const int* __restrict__ seq_row_start,
    const int* __restrict__ seq_slots, int rows, int H) {
  const int c = 4 * (blockIdx.y * blockDim.x + threadIdx.x);
  if (c >= H) return;
  const int base = blockIdx.x * ROWS;
  float wc[4 * TAPS];   // [channel][tap]
#pragma unroll
  for (int e = 0; e < TAPS; ++e) load_row<4>(w + (int64_t)c * TAPS + 4 * e, wc + 4 * e);
  auto finish = [&](int t, const float(*v)[4]) {   // v: the inputs of the row's taps
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < TAPS; ++j) acc = fmaf(wc[e * TAPS + j], v[j][e], acc);
      o[e] = v[TAPS - 1][e] + acc;
    }
    store_row<4>(out + (int64_t)t * H + c, o);
  };
  if constexpr (SINGLE) {
#pragma unroll
    for (int n = 0; n < ROWS; ++n) {
      const int t = base + n;
      if (t >= rows) return;
      float* st = state + (int64_t)seq_slots[row_seq[t]] * state_stride + c;
      float v[TAPS][4];
#pragma unroll
      for (int j = 0; j < TAPS; ++j)
        load_row<4>(j == TAPS - 1 ? x + (int64_t)t * H + c : st + (int64_t)j * H, v[j]);
      finish(t, v);
#pragma unroll
      for (int k = 0; k + 1 < TAPS; ++k) store_row<4>(st + (int64_t)k * H, v[k + 1]);
    }
  } else {
    float xs[ROWS + TAPS - 1][4];   // (rows that are not there: the nearest one, not used)
#pragma unroll
    for (int m = 0; m < ROWS + TAPS - 1; ++m) {
      const int t = min(max(base - (TAPS - 1) + m, 0), rows - 1);
      load_row<4>(x + (int64_t)t * H + c, xs[m]);
    }
    bool starts = false;   // a request starts in these rows
#pragma unroll
    for (int n = 0; n < ROWS; ++n) {
      const int t = base + n;
      if (t >= rows) break;
      const int s = row_seq[t], r0 = seq_row_start[s], i = t - r0;
      if (i >= TAPS - 1) {
        finish(t, xs + n);
      } else if (r0 >= base) {   // (else it is with the rows before)
        starts = true;
        const float* st = state + (int64_t)seq_slots[s] * state_stride + c;
        float v[TAPS][4];
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
          const int src = i - (TAPS - 1 - j);
          load_row<4>(src >= 0 ? x + (int64_t)(r0 + src) * H + c : st + (int64_t)(TAPS - 1 + src) * H, v[j]);
        }
        finish(t, v);
      }
    }
    if (!starts) return;
    for (int t = base + ROWS; t < min(base + ROWS + TAPS - 2, rows); ++t) {   // rows behind that see the old state
      const int s = row_seq[t], r0 = seq_row_start[s], i = t - r0;
      if (i >= TAPS - 1 || r0 >= base + ROWS) break;
      const float* st = state + (int64_t)seq_slots[s] * state_stride + c;
      float v[TAPS][4];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) {
        const int src = i - (TAPS - 1 - j);
        load_row<4>(src >= 0 ? x + (int64_t)(r0 + src) * H + c : st + (int64_t)(TAPS - 1 + src) * H, v[j]);
      }
      finish(t, v);
    }
    for (int t = base; t < min(base + ROWS, rows); ++t) {   // (as in short_conv_state_kernel)
      const int s = row_seq[t], r0 = seq_row_start[s];
      if (t != r0) continue;
      const int n = seq_row_start[s + 1] - r0;
      float* st = state + (int64_t)seq_slots[s] * state_stride + c;
#pragma unroll
      for (int k = 0; k < TAPS - 1; ++k) {
        const int p = n - (TAPS - 1) + k;
        float v[4];
        load_row<4>(p >= 0 ? x + (int64_t)(r0 + p) * H + c : st + (int64_t)(k + n) * H, v);
        store_row<4>(st + (int64_t)k * H, v);
      }
    }
  }
}

// state <- the last taps - 1 inputs of each request after this step's n rows. Entry k is the
// input at index n - (taps - 1) + k of the step's rows; a negative index is the old entry
// k + n, which lies above k, so ascending k never reads what it has written.
__global__ void short_conv_state_kernel(const float* __restrict__ x, float* __restrict__ state,
                                        int64_t state_stride,
                                        const int* __restrict__ seq_row_start,
                                        const int* __restrict__ seq_slots, int H, int taps) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= H) return;
  const int r0 = seq_row_start[s];
  const int n = seq_row_start[s + 1] - r0;
  float* st = state + (int64_t)seq_slots[s] * state_stride;
  for (int k = 0; k < taps - 1; ++k) {
    const int p = n - (taps - 1) + k;
    st[(int64_t)k * H + c] = p >= 0 ? x[(int64_t)(r0 + p) * H + c] : st[(int64_t)(k + n) * H + c];
  }
}

// x += norm(y) g with norm(y) = y rsqrt(mean(y^2) + eps), or with `center` the layer norm
// (y - mean) rsqrt(mean((y - mean)^2) + eps). y is a row of `y`, or with `w` the weighted sum of
// k rows, y_r = sum_j w[r, j] y[r k + j] (a sparse feed-forward's chosen experts), formed in
// 32-bit in the order of j. A thread keeps its (at most 8) numbers of the row in registers, in
// groups of VEC consecutive ones (VEC 4: whole 8- and 16-byte loads and stores).
// With `out2` the rows of a norm of the new x follow, norm(x) gain2 with eps2 and center2 of its own, from the registers
// that hold x (a launch and a read of x less: 64 rows of 2,048 4.4 us against 5.9 for the two, 2,048 rows 13.3 against 16.3).
constexpr int kNormAddPerThread = 8;
template <typename T, int VEC>
__global__ void norm_add_kernel(float* __restrict__ x, const T* __restrict__ y,
                                const float* __restrict__ w, int k,
                                const float* __restrict__ gain, int gain_n, int H, float eps,
                                int center, const float* __restrict__ gain2, T* __restrict__ out2, float eps2,
                                int center2) {
  constexpr int G = kNormAddPerThread / VEC;
  __shared__ float red[16];
  const int64_t r = blockIdx.x;
  float vals[G][VEC];
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
#pragma unroll
    for (int e = 0; e < VEC; ++e) vals[c][e] = 0.f;
    if (i < H) {
      if (w) {
        for (int j = 0; j < k; ++j) {
          float yv[VEC];
          load_row<VEC>(y + (r * k + j) * H + i, yv);
          const float wj = w[r * k + j];
#pragma unroll
          for (int e = 0; e < VEC; ++e) vals[c][e] = fmaf(wj, yv[e], vals[c][e]);
        }
      } else {
        load_row<VEC>(y + r * H + i, vals[c]);
      }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum += vals[c][e];
  }
  const float mean = center ? block_sum(sum, red) / (float)H : 0.f;
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const bool in = VEC * (threadIdx.x + c * blockDim.x) < H;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float d = in ? vals[c][e] - mean : 0.f;
      ss = fmaf(d, d, ss);
    }
  }
  ss = block_sum(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)H + eps);
  float* xr = x + r * H;
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
    if (i < H) {
      float xv[VEC], gv[VEC];
      load_row<VEC>(xr + i, xv);
      if (gain_n == 1) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) gv[e] = gain[0];
      } else {
        load_row<VEC>(gain + i, gv);
      }
#pragma unroll
      for (int e = 0; e < VEC; ++e) xv[e] += (vals[c][e] - mean) * inv * gv[e];
      if constexpr (VEC == 4) *(float4*)(xr + i) = make_float4(xv[0], xv[1], xv[2], xv[3]);
      else xr[i] = xv[0];
#pragma unroll
      for (int e = 0; e < VEC; ++e) vals[c][e] = xv[e];
    }
  }
  if (!out2) return;
  // (numbers beyond the row are 0 in `vals`)
  float mean2 = 0.f;
  if (center2) {
    float total = 0.f;
#pragma unroll
    for (int c = 0; c < G; ++c)
#pragma unroll
      for (int e = 0; e < VEC; ++e) total += vals[c][e];
    mean2 = block_sum(total, red) / (float)H;
  }
  float ss2 = 0.f;
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const bool in = VEC * (threadIdx.x + c * blockDim.x) < H;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float d = in ? vals[c][e] - mean2 : 0.f;
      ss2 = fmaf(d, d, ss2);
    }
  }
  ss2 = block_sum(ss2, red);
  const float inv2 = 1.f / sqrtf(ss2 / (float)H + eps2);
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
    if (i < H) {
      float gv[VEC], ov[VEC];
      load_row<VEC>(gain2 + i, gv);
#pragma unroll
      for (int e = 0; e < VEC; ++e) ov[e] = (vals[c][e] - mean2) * inv2 * gv[e];
      store_row<VEC>(out2 + r * H + i, ov);
    }
  }
}

// x <- norm(alpha x + y), norm(z) = z rsqrt(mean(z^2) + eps) gain; also as T into `out` when that
// is given. y: a row of `y`; with `w` the weighted sum of k rows (as norm_add has it); with `y2`
// factor * (rms(y) gain1 + rms(y2) gain2). The pieces of a row stay in registers throughout.
struct PostNormArgs {
  float* x;            // [T, H]
  const void* y;       // [T, H], or [T k, H] with w
  const void* y2;      // [T, H] or null
  const float* gain1;  // [H] with y2
  const float* gain2;
  const float* w;      // [T, k] or null
  const float* gain;   // [H]
  void* out;           // [T, H] or null
  int T;
  int H;
  int k;
  int dtype;
  float alpha;
  float eps;
  float factor;
};

// Two sums over a block at once; every thread gets both.
__device__ __forceinline__ void block_sum2(float& u, float& v, float (*red)[2]) {
  u = wave_sum(u);
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if (lane == 0) red[wv][0] = u, red[wv][1] = v;
  __syncthreads();
  u = v = 0.f;
  for (int i = 0; i < nw; ++i) u += red[i][0], v += red[i][1];
}

template <typename T, int VEC>
__global__ void post_norm_kernel(PostNormArgs a) {
  constexpr int G = kNormAddPerThread / VEC;
  __shared__ float red[16];
  __shared__ float red2[16][2];
  const int64_t r = blockIdx.x;
  const int H = a.H;
  const T* y = (const T*)a.y;
  float* xr = a.x + r * H;
  float z[G][VEC];
  if (a.y2) {
    const T* y2 = (const T*)a.y2;
    float b[G][VEC];
    float sa = 0.f, sb = 0.f;
#pragma unroll
    for (int c = 0; c < G; ++c) {
      const int i = VEC * (threadIdx.x + c * blockDim.x);
#pragma unroll
      for (int e = 0; e < VEC; ++e) z[c][e] = b[c][e] = 0.f;
      if (i < H) {
        load_row<VEC>(y + r * H + i, z[c]);
        load_row<VEC>(y2 + r * H + i, b[c]);
      }
#pragma unroll
      for (int e = 0; e < VEC; ++e) sa = fmaf(z[c][e], z[c][e], sa), sb = fmaf(b[c][e], b[c][e], sb);
    }
    block_sum2(sa, sb, red2);
    const float ia = a.factor / sqrtf(sa / (float)H + a.eps), ib = a.factor / sqrtf(sb / (float)H + a.eps);
#pragma unroll
    for (int c = 0; c < G; ++c) {
      const int i = VEC * (threadIdx.x + c * blockDim.x);
      if (i < H) {
        float ga[VEC], gb[VEC];
        load_row<VEC>(a.gain1 + i, ga);
        load_row<VEC>(a.gain2 + i, gb);
#pragma unroll
        for (int e = 0; e < VEC; ++e) z[c][e] = z[c][e] * ia * ga[e] + b[c][e] * ib * gb[e];
      }
    }
  } else {
#pragma unroll
    for (int c = 0; c < G; ++c) {
      const int i = VEC * (threadIdx.x + c * blockDim.x);
#pragma unroll
      for (int e = 0; e < VEC; ++e) z[c][e] = 0.f;
      if (i < H) {
        if (a.w) {
          for (int j = 0; j < a.k; ++j) {
            float yv[VEC];
            load_row<VEC>(y + (r * a.k + j) * H + i, yv);
            const float wj = a.w[r * a.k + j];
#pragma unroll
            for (int e = 0; e < VEC; ++e) z[c][e] = fmaf(wj, yv[e], z[c][e]);
          }
        } else {
          load_row<VEC>(y + r * H + i, z[c]);
        }
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
    if (i < H) {
      float xv[VEC];
      load_row<VEC>(xr + i, xv);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        z[c][e] = fmaf(a.alpha, xv[e], z[c][e]);
        ss = fmaf(z[c][e], z[c][e], ss);
      }
    }
  }
  ss = block_sum(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)H + a.eps);
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
    if (i < H) {
      float g[VEC];
      load_row<VEC>(a.gain + i, g);
#pragma unroll
      for (int e = 0; e < VEC; ++e) z[c][e] *= inv * g[e];
      if constexpr (VEC == 4) {
        *(float4*)(xr + i) = make_float4(z[c][0], z[c][1], z[c][2], z[c][3]);
      } else {
        xr[i] = z[c][0];
      }
      if (a.out) {
        T* o = (T*)a.out + r * H + i;
        if constexpr (VEC == 4 && sizeof(T) == 2) {
          union { __bf16 b[4]; uint2 u; } p;
#pragma unroll
          for (int e = 0; e < 4; ++e) p.b[e] = (__bf16)z[c][e];
          *(uint2*)o = p.u;
        } else {
#pragma unroll
          for (int e = 0; e < VEC; ++e) o[e] = from_f32<T>(z[c][e]);
        }
      }
    }
  }
}

struct GatedNormArgs {
  const float* o;       // [T, N]
  const void* gate;     // [T, gate_stride] or null
  const float* w;       // [w_n]: a number per column of the row (w_n = N) or of a group
  const float* den;     // [T, N / group] or null: what a group's numbers are divided by first
  void* out;            // [T, N]
  int gate_stride, T, N, group, w_n, silu, gate_first, dtype;
  float eps;
};

// VEC numbers of the row as the norm takes them, and the factors that follow the norm.
template <typename T, int VEC>
__device__ __forceinline__ void gated_norm_in(const GatedNormArgs& a, int64_t r, int i, float inv_den, float* v, float* after) {
  load_row<VEC>(a.o + r * a.N + i, v);
  float z[VEC];
  if (a.gate) load_row<VEC>((const T*)a.gate + r * a.gate_stride + i, z);
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    v[e] *= inv_den;
    after[e] = a.gate ? (a.silu ? z[e] : 1.f) * sigmoid_for<T>(z[e]) : 1.f;
    if (a.gate_first) v[e] *= after[e], after[e] = 1.f;
  }
}
template <typename T, int VEC>
__device__ __forceinline__ void gated_norm_out(const GatedNormArgs& a, int64_t r, int i, const float* w, float inv,
                                               const float* v, const float* after) {
  T* out = (T*)a.out + r * a.N + i;
  float g[VEC], y[VEC];
  load_row<VEC>(w, g);
#pragma unroll
  for (int e = 0; e < VEC; ++e) y[e] = v[e] * inv * g[e] * after[e];
  if constexpr (VEC == 4 && sizeof(T) == 4) {
    *(float4*)out = make_float4(y[0], y[1], y[2], y[3]);
  } else if constexpr (VEC == 4) {
    union { __bf16 b[4]; uint2 u; } p;
#pragma unroll
    for (int e = 0; e < 4; ++e) p.b[e] = (__bf16)y[e];
    *(uint2*)out = p.u;
  } else {
    out[0] = from_f32<T>(y[0]);
  }
}

// A block per (row, group); a thread keeps its (at most 16) numbers in registers, in groups of VEC
// consecutive ones.
constexpr int kGatedPerThread = 16;
template <typename T, int VEC>
__global__ void gated_rmsnorm_kernel(GatedNormArgs a) {
  constexpr int G = kGatedPerThread / VEC;
  __shared__ float red[16];
  const int64_t r = blockIdx.x;
  const int g0 = blockIdx.y * a.group;
  const float inv_den = a.den ? 1.f / a.den[r * gridDim.y + blockIdx.y] : 1.f;
  const float* w = a.w + (a.w_n == a.N ? g0 : 0);
  float v[G][VEC], sg[G][VEC];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
    if (i < a.group) {
      gated_norm_in<T, VEC>(a, r, g0 + i, inv_den, v[c], sg[c]);
#pragma unroll
      for (int e = 0; e < VEC; ++e) ss = fmaf(v[c][e], v[c][e], ss);
    }
  }
  ss = block_sum(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)a.group + a.eps);
#pragma unroll
  for (int c = 0; c < G; ++c) {
    const int i = VEC * (threadIdx.x + c * blockDim.x);
    if (i < a.group) gated_norm_out<T, VEC>(a, r, g0 + i, w + i, inv, v[c], sg[c]);
  }
}

// The same for groups of few columns (a head's values): one wave per (row, group), four groups
// to a block.
constexpr int kGatedWaveMax = 512;
template <typename T, int VEC>
__global__ __launch_bounds__(256) void gated_group_rmsnorm_kernel(GatedNormArgs a) {
  constexpr int PER = kGatedWaveMax / 64 / VEC;
  const int64_t r = blockIdx.x;
  const int g = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int g0 = g * a.group;
  if (g0 >= a.N) return;
  const float inv_den = a.den ? 1.f / a.den[r * (a.N / a.group) + g] : 1.f;
  const float* w = a.w + (a.w_n == a.N ? g0 : 0);
  float v[PER][VEC], sg[PER][VEC];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < PER; ++c) {
    const int i = VEC * (lane + 64 * c);
    if (i < a.group) {
      gated_norm_in<T, VEC>(a, r, g0 + i, inv_den, v[c], sg[c]);
#pragma unroll
      for (int e = 0; e < VEC; ++e) ss = fmaf(v[c][e], v[c][e], ss);
    }
  }
  ss = wave_sum(ss);
  const float inv = 1.f / sqrtf(ss / (float)a.group + a.eps);
#pragma unroll
  for (int c = 0; c < PER; ++c) {
    const int i = VEC * (lane + 64 * c);
    if (i < a.group) gated_norm_out<T, VEC>(a, r, g0 + i, w + i, inv, v[c], sg[c]);
  }
}

template <typename T, int VEC>
static void launch_gated_norm(const GatedNormArgs& a, hipStream_t stream) {
  const int groups = a.N / a.group;
  if (a.group <= kGatedWaveMax && groups > 1) {
    gated_group_rmsnorm_kernel<T, VEC><<<dim3(a.T, (groups + 3) / 4), 256, 0, stream>>>(a);
  } else {
    const int want = ((a.group + VEC - 1) / VEC + 63) / 64 * 64;
    gated_rmsnorm_kernel<T, VEC><<<dim3(a.T, groups), want > 1024 ? 1024 : want, 0, stream>>>(a);
  }
}

static int row_block(int H) {
  int b = (H + 63) / 64 * 64;
  return b > 256 ? 256 : b;
}

}  // namespace ninfer

using namespace ninfer;

// Whether the launch also moves the state on.
template <typename T>
static bool launch_short_conv(const float* x, const float* w, float* state, long long state_stride, T* out,
                              const int* row_seq, const int* seq_row_start, const int* seq_slots, int rows, int H,
                              int taps, bool single, hipStream_t stream) {
  const bool wide = taps >= 2 && taps <= 4 && H % 4 == 0 && state_stride % 4 == 0 && row_aligned(x) &&
                    row_aligned(w) && row_aligned(state) && row_aligned(out);
  if (!wide) {
    const int block = row_block(H);
    short_conv_kernel<T><<<dim3(rows, (H + block - 1) / block), block, 0, stream>>>(
        x, w, state, state_stride, out, row_seq, seq_row_start, seq_slots, H, taps, single ? 1 : 0);
    return single;
  }
  // four rows to a thread share its loads where that leaves the CUs enough waves, from 1.5 Mi numbers on:
  // 2,048 rows of 2,048 channels 8.7 us and 12.6 with one row to a thread, of 1,024 6.2 and 7.8. Below, a
  // prompt of 516 rows of 2,048 alone would gain (5.2 and 6.5) and lose behind seven requests of one row (8.2
  // and 6.4); 64 such requests 3.1 and 2.3, 300 rows of 64 3.4 and 3.1 (four taps)
  const int per = (int64_t)rows * H >= (3 << 19) ? 4 : 1;
  const int block = row_block(H / 4);
  const dim3 grid((rows + per - 1) / per, (H / 4 + block - 1) / block);
  auto launch = [&](auto kern) {
    kern<<<grid, block, 0, stream>>>(x, w, state, state_stride, out, row_seq, seq_row_start, seq_slots, rows, H);
  };
#define NINFER_CONV(TAPS)                                                                       \
  do {                                                                                          \
    if (per == 4)                                                                               \
      single ? launch(short_conv_rows_kernel<T, TAPS, 4, true>)                                 \
             : launch(short_conv_rows_kernel<T, TAPS, 4, false>);                               \
    else                                                                                        \
      single ? launch(short_conv_rows_kernel<T, TAPS, 1, true>)                                 \
             : launch(short_conv_rows_kernel<T, TAPS, 1, false>);                               \
  } while (0)
  if (taps == 2) NINFER_CONV(2);
  else if (taps == 3) NINFER_CONV(3);
  else NINFER_CONV(4);
#undef NINFER_CONV
  return true;
}

extern "C" int ninfer_short_conv(const float* x, const float* w, float* state,
                                 long long state_stride, void* out, const int* row_seq,
                                 const int* seq_row_start, const int* seq_slots, int T, int S,
                                 int H, int taps, int all_single, int dtype, hipStream_t stream) {
  NINFER_REQUIRE(T > 0 && S > 0 && H > 0, "short_conv: T=%d S=%d H=%d must be positive", T, S, H);
  NINFER_REQUIRE(taps >= 1, "short_conv: %d taps", taps);
  NINFER_REQUIRE(state_stride >= (long long)(taps - 1) * H,
                 "short_conv: a request's state of %lld floats holds no %d x %d inputs",
                 state_stride, taps - 1, H);
  NINFER_REQUIRE(dtype == kF32 || dtype == kBF16, "short_conv: unknown dtype %d", dtype);
  const int block = row_block(H);
  const bool moved =
      dtype == kF32 ? launch_short_conv(x, w, state, state_stride, (float*)out, row_seq, seq_row_start, seq_slots, T,
                                        H, taps, all_single != 0, stream)
                    : launch_short_conv(x, w, state, state_stride, (bf16*)out, row_seq, seq_row_start, seq_slots, T,
                                        H, taps, all_single != 0, stream);
  NINFER_LAUNCH_CHECK();
  if (!moved && taps > 1) {
    short_conv_state_kernel<<<dim3(S, (H + block - 1) / block), block, 0, stream>>>(
        x, state, state_stride, seq_row_start, seq_slots, H, taps);
    NINFER_LAUNCH_CHECK();
  }
  return 0;
}

extern "C" int ninfer_norm_add(float* x, const void* y, const float* gain, int gain_n, int T, int H,
                               float eps, int dtype, int center, const float* w, int k, const float* gain2,
                               void* out2, float eps2, int center2, hipStream_t stream) {
  NINFER_REQUIRE(T > 0 && H > 0, "norm_add: T=%d H=%d must be positive", T, H);
  NINFER_REQUIRE(gain_n == 1 || gain_n == H, "norm_add: %d gains for %d channels", gain_n, H);
  NINFER_REQUIRE(dtype == kF32 || dtype == kBF16, "norm_add: unknown dtype %d", dtype);
  NINFER_REQUIRE(H <= 1024 * kNormAddPerThread, "norm_add: width %d exceeds %d", H,
                 1024 * kNormAddPerThread);
  NINFER_REQUIRE(!w || k > 0, "norm_add: a weighted sum of %d rows", k);
  NINFER_REQUIRE(!out2 || gain2, "norm_add: a second norm without its gains");
  // groups of 4 consecutive numbers when every row stays 16-byte aligned
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const bool vec = H % 4 == 0 && aligned(x) && aligned(y) && (gain_n == 1 || aligned(gain)) && aligned(gain2) &&
                   aligned(out2);
  const int per_thread = vec ? 4 : 1;
  int block = ((H + per_thread - 1) / per_thread + 63) / 64 * 64;
  if (block > 1024) block = 1024;
  NINFER_REQUIRE((int64_t)block * kNormAddPerThread >= H, "norm_add: width %d exceeds the kernel's", H);
  if (dtype == kF32) {
    if (vec) norm_add_kernel<float, 4><<<T, block, 0, stream>>>(x, (const float*)y, w, k, gain, gain_n, H, eps, center, gain2, (float*)out2, eps2, center2);
    else norm_add_kernel<float, 1><<<T, block, 0, stream>>>(x, (const float*)y, w, k, gain, gain_n, H, eps, center, gain2, (float*)out2, eps2, center2);
  } else {
    if (vec) norm_add_kernel<bf16, 4><<<T, block, 0, stream>>>(x, (const bf16*)y, w, k, gain, gain_n, H, eps, center, gain2, (bf16*)out2, eps2, center2);
    else norm_add_kernel<bf16, 1><<<T, block, 0, stream>>>(x, (const bf16*)y, w, k, gain, gain_n, H, eps, center, gain2, (bf16*)out2, eps2, center2);
  }
  NINFER_LAUNCH_CHECK();
  return 0;
}

extern "C" int ninfer_post_norm(const PostNormArgs* args, hipStream_t stream) {
  const PostNormArgs& a = *args;
  NINFER_REQUIRE(a.T > 0 && a.H > 0 && a.x && a.y && a.gain, "post_norm: T=%d H=%d must be positive", a.T, a.H);
  NINFER_REQUIRE(a.dtype == kF32 || a.dtype == kBF16, "post_norm: unknown dtype %d", a.dtype);
  NINFER_REQUIRE(!a.w || a.k > 0, "post_norm: a weighted sum of %d rows", a.k);
  NINFER_REQUIRE(!a.y2 || (a.gain1 && a.gain2 && !a.w), "post_norm: two normed rows need their gains and no weights");
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const bool vec = a.H % 4 == 0 && aligned(a.x) && aligned(a.y) && aligned(a.gain) && aligned(a.y2) &&
                   aligned(a.gain1) && aligned(a.gain2) && aligned(a.out);
  const int per_thread = vec ? 4 : 1;
  int block = ((a.H + per_thread - 1) / per_thread + 63) / 64 * 64;
  if (block > 1024) block = 1024;
  NINFER_REQUIRE((int64_t)block * kNormAddPerThread >= a.H, "post_norm: width %d exceeds the kernel's", a.H);
  if (a.dtype == kF32) {
    if (vec) post_norm_kernel<float, 4><<<a.T, block, 0, stream>>>(a);
    else post_norm_kernel<float, 1><<<a.T, block, 0, stream>>>(a);
  } else {
    if (vec) post_norm_kernel<bf16, 4><<<a.T, block, 0, stream>>>(a);
    else post_norm_kernel<bf16, 1><<<a.T, block, 0, stream>>>(a);
  }
  NINFER_LAUNCH_CHECK();
  return 0;
}

// group 0 (or N): the norm over the whole row; else over every group of `group` columns by
// itself, with a weight of `group` numbers that the groups share or of N.
extern "C" int ninfer_gated_rmsnorm(const GatedNormArgs* args, hipStream_t stream) {
  GatedNormArgs a = *args;
  NINFER_REQUIRE(a.T > 0 && a.N > 0 && (!a.gate || a.gate_stride >= a.N), "gated_rmsnorm: T=%d N=%d gate stride %d", a.T,
                 a.N, a.gate_stride);
  NINFER_REQUIRE(a.dtype == kF32 || a.dtype == kBF16, "gated_rmsnorm: unknown dtype %d", a.dtype);
  if (a.group == 0) a.group = a.N;
  NINFER_REQUIRE(a.group > 0 && a.N % a.group == 0, "gated_rmsnorm: groups of %d columns do not fill rows of %d",
                 a.group, a.N);
  NINFER_REQUIRE(a.w_n == a.N || a.w_n == a.group, "gated_rmsnorm: %d weights for groups of %d columns", a.w_n, a.group);
  NINFER_REQUIRE(a.group <= 1024 * kGatedPerThread, "gated_rmsnorm: %d columns exceed %d", a.group, 1024 * kGatedPerThread);
  NINFER_REQUIRE(!a.gate_first || a.gate, "gated_rmsnorm: no gate to apply first");
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const bool vec = a.group % 4 == 0 && (!a.gate || a.gate_stride % 4 == 0) && aligned(a.o) && aligned(a.gate) &&
                   aligned(a.w) && aligned(a.out);
  if (a.dtype == kF32) {
    if (vec) launch_gated_norm<float, 4>(a, stream);
    else launch_gated_norm<float, 1>(a, stream);
  } else {
    if (vec) launch_gated_norm<bf16, 4>(a, stream);
    else launch_gated_norm<bf16, 1>(a, stream);
  }
  NINFER_LAUNCH_CHECK();
  return 0;
}
