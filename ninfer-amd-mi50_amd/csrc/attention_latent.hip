// Attention over a cached latent: every head reads the same cached row per key,
// [c (R numbers) | k_rot (rd numbers)], and a query that has been taken into the latent's
// space, q' = [W_uk_h^T q_unrotated (R) | q_rotated (rd)]:
//
//   score_j = (q' . row_j) * scale,  p = softmax over the visible keys,  o = sum_j p_j c_j
//
// so that neither keys nor values per head are ever formed for the cache: the head's value
// is W_uv_h o afterwards. Two kernels:
//
//   latent_kv_write  per row: c = rmsnorm(first R of the down-projection) * weight, the
//                    shared rotated key part turned by the row's position, both written to
//                    the request's page; the rotated part of every query head turned and
//                    placed behind the R absorbed numbers of q'.
//   latent_attention one wave per (row, head); keys in tiles of 64 aligned to absolute
//                    positions with an online softmax, so every sum's order depends on the
//                    row's position alone. The head's output may be multiplied by
//                    sigmoid(gate[row, head]).
//
//   latent_attention_tile (bfloat16, matrix cores): a block of eight waves owns 64 rows (or 16, in
//                    steps of few rows) of (token, head) pairs of one request, all of which read
//                    the same cached rows. Keys come in tiles of 64 through LDS as they lie in
//                    the cache ([key][numbers]), the next tile on its way in registers; the
//                    queries stay in registers, each wave with half of the numbers, so a key is
//                    read from LDS twice for 64 rows. The values' operand comes from the same
//                    tile through the transposing LDS read. S and O += P V run on the matrix
//                    cores, the softmax between them in 32-bit. The keys of long contexts are cut
//                    into chunks over several blocks whose partial sums a second kernel merges
//                    (steps of few rows would otherwise leave most of the GPU idle); a request's
//                    tiles are shared out evenly over its chunks.
//
//   latent_attention_rows  the blocks of 64 rows for latents of 256 or 512 numbers with 32 or 64 turned
//                    ones: four waves that keep 16 rows each, nothing between them but the keys.
//
// Latent 512 + 64, 16 heads, against blocks of four waves and 32 rows with the queries in LDS and the
// values gathered by two-byte reads: a 2,048-token prompt 688 -> 192 us (73 GFLOP, 380 TFLOP/s; the
// LDS traffic alone, 3,000 cycles a tile of 64 keys, is 42 us), 64 requests at 1,950 to 2,600 keys
// 188 -> 49 us (168 MB, 3.4 TB/s; at 4,000 keys, 295 MB, 71 us, 4.2 TB/s: a tile's way through LDS and
// four barriers, about 5 us a tile).
//
// The rotation turns pair (i, i + n/2), or with `interleaved` pair (2i, 2i + 1), of the first
// n = rot_n numbers of the rotated part by pos * freq[i]; cosine and sine are multiplied by `magnitude` (1 without a scaled table).
// Norm, angles, scores, softmax and the value sum are 32-bit.
#include "attention.h"

namespace ninfer {

struct LatentArgs {
  const void* dkv;          // [T, dkv_stride] down-projection rows: R latent numbers, then rd
  void* q;                  // [T, Hq * (dim + rd)] projected queries, head by head
  float* q_abs;             // [T, Hq, R + rd] 32-bit; the first R of each head are written by
                            // the caller's products, the last rd here
  void* pool;               // [pages, page_size, R + rd]
  void* out;                // [T, Hq * R] (attention) in the activation dtype
  const void* gate;         // [T, gate_stride] or null: out of head h times sigmoid(gate[t, h])
  const float* norm_w;      // [R]
  const float* freq;        // [rot_n / 2]
  const int* block_table;   // [S, bt_stride]
  const int* positions;     // [T]
  const int* row_seq;       // [T]
  const int* seq_row_start; // [S + 1] (the matrix-core kernel: rows of each request)
  const int* seq_pos0;      // [S] position of each request's first row
  float* workspace;         // partial sums of contexts cut into chunks, or null
  long long workspace_floats;
  int S;
  int max_kv_len;           // host-side bound that sizes the chunks
  int max_qlen;             // host-side: the most rows a request brings (1: a decode-only step)
  int force_plain;          // tests: the plain kernel whatever the shape
  int dkv_stride;
  int gate_stride;
  int bt_stride;
  int T;
  int Hq;
  int dim;                  // unrotated numbers per query head
  int R;                    // latent size
  int rd;                   // rotated numbers per head (and of the shared key part)
  int rot_n;                // how many of them turn (even, <= rd)
  int page_size;
  int window;               // 0: all keys
  int write_kv;
  int dtype;
  float eps;
  float magnitude;
  float scale;
  int interleaved;          // pair i of the turning numbers is (2i, 2i + 1) instead of (i, i + rot_n / 2)
  int abs_rows;             // latent_kv_write: of the rows before this one the turned parts of the queries go
                            // to q_abs, of the others they stay in q
};

// Keys and values per head for prompts (bfloat16), from the cached rows of their requests.
struct LatentHeadsArgs {
  void* latent;             // [keys, R] the requests' cached latents in order, for the product that forms kv
  void* krot;               // [keys, rd] their turned numbers
  int* key_start;           // [S] first of these rows of each request
  const void* kv;           // [keys, Hq * (dim + vdim)] keys of all heads, then values of all heads
  void* q;                  // [T, Hq * (dim + rd)], turned (latent_kv_write)
  void* out;                // [T, Hq * vdim]
  const int* seq_qlen;      // [S]
  int keys;                 // all cached positions of the S requests, this step's included
  int vdim;
};

__device__ __forceinline__ void turn_pair(float u, float v, float c, float s, float* a, float* b) {
  *a = u * c - v * s;
  *b = v * c + u * s;
}

template <typename T>
__global__ void latent_kv_write_kernel(LatentArgs a) {
  extern __shared__ float smem[];
  float* trig = smem;            // [rot_n]: cos, then sin
  __shared__ float red[16];
  const int t = blockIdx.x;
  const int pos = a.positions[t];
  const int half = a.rot_n / 2;
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    float s, c;
    sincosf((float)pos * a.freq[i], &s, &c);
    trig[i] = c * a.magnitude;
    trig[half + i] = s * a.magnitude;
  }
  const T* row = (const T*)a.dkv + (int64_t)t * a.dkv_stride;
  float ss = 0.f;
  for (int i = threadIdx.x; i < a.R; i += blockDim.x) {
    const float v = to_f32(row[i]);
    ss = fmaf(v, v, ss);
  }
  ss = block_sum(ss, red);   // (its barriers also publish trig)
  const int Dk = a.R + a.rd;
  if (a.write_kv) {
    const float inv = 1.f / sqrtf(ss / (float)a.R + a.eps);
    const int page = a.block_table[(int64_t)a.row_seq[t] * a.bt_stride + pos / a.page_size];
    T* dst = (T*)a.pool + ((int64_t)page * a.page_size + pos % a.page_size) * Dk;
    for (int i = threadIdx.x; i < a.R; i += blockDim.x)
      dst[i] = from_f32<T>(to_f32(row[i]) * inv * a.norm_w[i]);
    const T* kr = row + a.R;
    for (int i = threadIdx.x; i < a.rd; i += blockDim.x) {
      float v = to_f32(kr[i]);
      if (i < a.rot_n) {
        const int p = a.interleaved ? i >> 1 : i < half ? i : i - half;
        const int i1 = a.interleaved ? 2 * p : p, i2 = a.interleaved ? 2 * p + 1 : p + half;
        float x, y;
        turn_pair(to_f32(kr[i1]), to_f32(kr[i2]), trig[p], trig[half + p], &x, &y);
        v = i == i1 ? x : y;
      }
      dst[a.R + i] = from_f32<T>(v);
    }
  }
  const int qd = a.dim + a.rd;
  if (t >= a.abs_rows) {   // turned in place, a thread to a pair
    for (int e = threadIdx.x; e < a.Hq * half; e += blockDim.x) {
      const int h = e / half, p = e % half;
      T* qr = (T*)a.q + ((int64_t)t * a.Hq + h) * qd + a.dim;
      const int i1 = a.interleaved ? 2 * p : p, i2 = a.interleaved ? 2 * p + 1 : p + half;
      float x, y;
      turn_pair(to_f32(qr[i1]), to_f32(qr[i2]), trig[p], trig[half + p], &x, &y);
      qr[i1] = from_f32<T>(x);
      qr[i2] = from_f32<T>(y);
    }
    return;
  }
  for (int e = threadIdx.x; e < a.Hq * a.rd; e += blockDim.x) {
    const int h = e / a.rd, i = e % a.rd;
    const T* qr = (const T*)a.q + ((int64_t)t * a.Hq + h) * qd + a.dim;
    float v = to_f32(qr[i]);
    if (i < a.rot_n) {
      const int p = a.interleaved ? i >> 1 : i < half ? i : i - half;
      const int i1 = a.interleaved ? 2 * p : p, i2 = a.interleaved ? 2 * p + 1 : p + half;
      float x, y;
      turn_pair(to_f32(qr[i1]), to_f32(qr[i2]), trig[p], trig[half + p], &x, &y);
      v = i == i1 ? x : y;
    }
    a.q_abs[((int64_t)t * a.Hq + h) * Dk + a.R + i] = v;
  }
}

constexpr int kLatentMaxPerLane = 16;   // latent sizes up to 1024

template <typename T>
__global__ __launch_bounds__(64) void latent_attention_kernel(LatentArgs a) {
  extern __shared__ float smem[];
  const int Dk = a.R + a.rd;
  int64_t* off_s = (int64_t*)smem;         // [64] element offset of each key's row
  float* p_s = (float*)(off_s + 64);       // [64]
  float* q_s = p_s + 64;                   // [Dk]
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int pos = a.positions[t];
  const int* bt = a.block_table + (int64_t)a.row_seq[t] * a.bt_stride;
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const float* qr = a.q_abs + ((int64_t)t * a.Hq + h) * Dk;
  for (int d = lane; d < Dk; d += 64) q_s[d] = qr[d];
  __syncthreads();
  const T* pool = (const T*)a.pool;
  float m = -INFINITY, l = 0.f;
  float acc[kLatentMaxPerLane];
#pragma unroll
  for (int i = 0; i < kLatentMaxPerLane; ++i) acc[i] = 0.f;
  for (int tile = (lo / 64) * 64; tile <= pos; tile += 64) {
    const int j = tile + lane;
    const bool valid = j >= lo && j <= pos;
    float s = -INFINITY;
    int64_t off = 0;
    if (valid) {
      const int page = bt[j / a.page_size];
      off = ((int64_t)page * a.page_size + (j % a.page_size)) * Dk;
      const T* kr = pool + off;
      float dot = 0.f;
      for (int d = 0; d < Dk; ++d) dot = fmaf(q_s[d], to_f32(kr[d]), dot);
      s = dot * a.scale;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);   // 0 on the first tile
    l = l * alpha + wave_sum(p);
    m = m_new;
    p_s[lane] = p;
    off_s[lane] = off;
    __syncthreads();
    const int n_keys = min(64, pos - tile + 1);
    const int first = max(0, lo - tile);
#pragma unroll
    for (int i = 0; i < kLatentMaxPerLane; ++i) {
      const int d = lane + i * 64;
      if (d < a.R) {
        float v = acc[i] * alpha;
        for (int jj = first; jj < n_keys; ++jj) v = fmaf(p_s[jj], to_f32(pool[off_s[jj] + d]), v);
        acc[i] = v;
      }
    }
    __syncthreads();
  }
  float inv = 1.f / l;
  if (a.gate) {
    const float g = to_f32(((const T*)a.gate)[(int64_t)t * a.gate_stride + h]);
    inv *= 1.f / (1.f + expf(-g));
  }
  T* orow = (T*)a.out + ((int64_t)t * a.Hq + h) * a.R;
#pragma unroll
  for (int i = 0; i < kLatentMaxPerLane; ++i) {
    const int d = lane + i * 64;
    if (d < a.R) orow[d] = from_f32<T>(acc[i] * inv);
  }
}

static bool latent_tile_takes(const LatentArgs& a);
static int latent_attention_tile(const LatentArgs& a, hipStream_t stream);

static int latent_check(const LatentArgs& a, const char* who) {
  NINFER_REQUIRE(a.T > 0 && a.Hq > 0 && a.R > 0 && a.rd >= 0 && a.dim >= 0,
                 "%s: T=%d heads=%d latent=%d rotated=%d unrotated=%d", who, a.T, a.Hq, a.R, a.rd,
                 a.dim);
  NINFER_REQUIRE(a.rot_n >= 0 && a.rot_n <= a.rd && a.rot_n % 2 == 0,
                 "%s: %d turning numbers must be even and at most %d", who, a.rot_n, a.rd);
  NINFER_REQUIRE(a.rot_n == 0 || a.freq, "%s: a rotation without a table", who);
  NINFER_REQUIRE(a.page_size > 0 && a.bt_stride > 0, "%s: bad page size %d or table width %d", who,
                 a.page_size, a.bt_stride);
  NINFER_REQUIRE(a.dtype == kF32 || a.dtype == kBF16, "%s: unknown dtype %d", who, a.dtype);
  NINFER_REQUIRE(a.window >= 0, "%s: window %d must be >= 0", who, a.window);
  return 0;
}

}  // namespace ninfer

using namespace ninfer;

extern "C" int ninfer_latent_kv_write(const LatentArgs* a, hipStream_t stream) {
  if (int rc = latent_check(*a, "latent_kv_write")) return rc;
  NINFER_REQUIRE(a->dkv_stride >= a->R + a->rd, "latent_kv_write: row stride %d < %d",
                 a->dkv_stride, a->R + a->rd);
  NINFER_REQUIRE(a->eps >= 0.f, "latent_kv_write: eps must be >= 0");
  const size_t lds = (size_t)(a->rot_n > 0 ? a->rot_n : 1) * sizeof(float);
  if (a->dtype == kF32)
    latent_kv_write_kernel<float><<<a->T, 256, lds, stream>>>(*a);
  else
    latent_kv_write_kernel<bf16><<<a->T, 256, lds, stream>>>(*a);
  NINFER_LAUNCH_CHECK();
  return 0;
}

extern "C" int ninfer_latent_attention(const LatentArgs* a, hipStream_t stream) {
  if (int rc = latent_check(*a, "latent_attention")) return rc;
  NINFER_REQUIRE(a->R <= 64 * kLatentMaxPerLane, "latent_attention: latent size %d exceeds %d",
                 a->R, 64 * kLatentMaxPerLane);
  NINFER_REQUIRE(a->scale > 0.f, "latent_attention: scale %g must be positive", (double)a->scale);
  if (latent_tile_takes(*a)) return latent_attention_tile(*a, stream);
  const dim3 grid(a->T, a->Hq);
  const size_t lds = (size_t)(a->R + a->rd + 64) * sizeof(float) + 64 * sizeof(int64_t);
  NINFER_REQUIRE(lds <= 64 * 1024, "latent_attention: a query of %d numbers does not fit",
                 a->R + a->rd);
  if (a->dtype == kF32)
    latent_attention_kernel<float><<<grid, 64, lds, stream>>>(*a);
  else
    latent_attention_kernel<bf16><<<grid, 64, lds, stream>>>(*a);
  NINFER_LAUNCH_CHECK();
  return 0;
}

// ---- the matrix-core kernel ------------------------------------------------------------------
namespace ninfer {

typedef __bf16 lat_bf16x8 __attribute__((ext_vector_type(8)));
typedef float lat_f32x16 __attribute__((ext_vector_type(16)));

typedef float lat_f32x4 __attribute__((ext_vector_type(4)));
typedef short lat_short4 __attribute__((ext_vector_type(4)));
typedef short lat_short8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) lat_short4 lat_lds_short4;

constexpr int kLatKeys = 64;      // keys per tile
constexpr int kLatThreads = 512;
constexpr int kLatPRow = kLatKeys + 8;   // row length of the probabilities in LDS
// Steps of 16 numbers of half a cached row that the kernel is built for: rows of up to 160, 288, 416, 576
// and 640 numbers (what fits the registers). A row between two of them is padded up to the longer one
// with zeros, up to half as many numbers again, or as many as 80 of 160. Rows of 80 in the form of
// 288: a request of 200 keys 13.7 us, in their own 11.6; of 384 in that of 576: a 2,048-token prompt of 16 heads
// 172 us, in that of 416 160.
constexpr int kLatHalves[] = {5, 9, 13, 18, 20};
constexpr int kLatMaxHalf = 20;
constexpr float kLatLog2e = 1.44269504088896f;
// What keys whose page the table does not hold (-1) are read from. (A prompt of 2,048 tokens of 16 heads
// with 512 + 64 numbers: 188 us without the check, 192 so, 206 with such loads switched off, 228 with
// zeros written over the keys in LDS: the last two hold more registers than there are.)
__device__ const lat_bf16x8 kLatNoKey = {};

struct LatentTilePlan {
  int rows;         // (token, head) rows of a block
  int tiles;        // upper bound of row tiles over all requests
  int n_chunks;     // key chunks per row tile
  int half;         // steps of 16 numbers in half a cached row (of kLatHalves)
  int page_shift;
  size_t lds;
};

static bool latent_tile_takes(const LatentArgs& a) {
  const int Dk = a.R + a.rd;
  return a.dtype == kBF16 && !a.force_plain && Dk % 8 == 0 && a.R <= 512 && Dk <= 32 * kLatMaxHalf &&
         (a.page_size & (a.page_size - 1)) == 0 && a.seq_row_start && a.seq_pos0 && a.S > 0 &&
         ((uintptr_t)a.pool % 16 == 0) && ((uintptr_t)a.q_abs % 16 == 0);
}

// Row tiles and key chunks of a step in blocks of `rows` rows. Row tiles: in a decode-only step
// every request has the same number; otherwise a bound (a request's last tile may be partial; tiles
// that do not exist exit at once). A block counts on a CU of its own, with as long a walk over the
// keys as that allows.
static void latent_tile_split(const LatentArgs& a, int rows, int* tiles, int* n_chunks) {
  *tiles = a.max_qlen == 1 ? a.S * ((a.Hq + rows - 1) / rows)
                           : (int)(((int64_t)a.T * a.Hq + rows - 1) / rows) + a.S;
  const int key_tiles = (a.max_kv_len + kLatKeys - 1) / kLatKeys;
  int want = device_cu_count() / *tiles;
  if (want > key_tiles) want = key_tiles;
  *n_chunks = want < 1 ? 1 : want;
}

// Has the row a form of its own in the kernel whose waves keep whole rows? Latents of 256 or 512 numbers with 32
// or 64 turned ones behind them. (By the sizes alone, as the plan is, so that the workspace does not depend on
// where the output lies; an output that does not take pieces of 8 bytes runs the other kernel.)
static bool latent_rows_form(const LatentArgs& a) {
  return (a.R == 256 || a.R == 512) && (a.rd == 32 || a.rd == 64);
}

// What a step takes in blocks of 16 or 64 rows, in us on this part: rounds of blocks, each a start and
// a walk over its keys, and the merge of chunks. Low blocks start sooner (queries, first tile, output:
// 10 against 24 us at 576 numbers a row) and meet a tile of 64 keys in 0.9 us while few of them run and
// in 2.1 when they fill the GPU (every block brings the same bytes from L2), high ones in 3.6 and for
// four times the rows; in the kernel whose waves keep whole rows 0.7 of that. 512 + 64 numbers, 16 heads, us in low
// and in high blocks, of which the last in that kernel: a prompt of 64 tokens 14, 32 and 15, of 300 29, 54 and 36, of
// 2,048 389, 188 and 140; 40 heads, 64 requests at 2,500 keys 118, 84 and 60.
// A prompt of its own sees half of its keys on average, which counts once its blocks run in rounds; without that, prompts
// of 200 to 300 tokens whose few high blocks need chunks and a merge went to them (40 heads, 256 + 32 numbers, 200
// tokens: 18 us in low blocks, 29 in high ones). Taken into account for the forms of that kernel, where both were measured.
static float latent_tile_us(const LatentArgs& a, int rows, int half) {
  int tiles, n_chunks;
  latent_tile_split(a, rows, &tiles, &n_chunks);
  const int key_tiles = (a.max_kv_len + kLatKeys - 1) / kLatKeys, steps = (key_tiles + n_chunks - 1) / n_chunks;
  const float filled = (float)tiles * n_chunks / device_cu_count(), numbers = half / 18.f;
  const bool waves = latent_rows_form(a);   // (the kernel whose waves keep whole rows)
  const float high = waves ? 0.7f : 1.f;
  const float start = rows == 16 ? 10.f : 24.f * high;
  const float step = rows == 16 ? 0.9f + 1.2f * (filled < 1.f ? filled : 1.f) : 3.6f * high;
  const float seen = waves && filled > 1.f && a.max_qlen == a.max_kv_len ? 0.55f : 1.f;
  const float round = start * (0.4f + 0.6f * numbers) + steps * step * numbers * seen;
  return round * (filled > 1.f ? filled : 1.f) + (n_chunks > 1 ? 6.f : 0.f);
}

static LatentTilePlan latent_tile_plan(const LatentArgs& a) {
  LatentTilePlan p;
  const int Dk = a.R + a.rd;
  for (const int half : kLatHalves)
    if (Dk <= 32 * (p.half = half)) break;
  p.rows = latent_tile_us(a, 16, p.half) <= latent_tile_us(a, 64, p.half) ? 16 : 64;
  latent_tile_split(a, p.rows, &p.tiles, &p.n_chunks);
  p.page_shift = 0;
  while ((1 << p.page_shift) < a.page_size) ++p.page_shift;
  p.lds = (size_t)kLatKeys * (32 * p.half + 8) * 2 + (size_t)2 * p.rows * kLatKeys * 4 +
          (size_t)p.rows * kLatPRow * 2 + 3 * p.rows * 4;
  return p;
}

static int64_t latent_tile_workspace_floats(const LatentArgs& a, const LatentTilePlan& p) {
  return p.n_chunks > 1 ? (int64_t)a.T * a.Hq * p.n_chunks * (a.R + 2) : 0;
}

// Which request (s) and which of its row tiles (lt) is this block's? The tiles are dealt out from
// the last one backwards: within a request the later tiles see more keys and run longer,
// and the long ones should start first. False: there is none.
template <int ROWS>
__device__ __forceinline__ bool latent_block_tile(const LatentArgs& a, int& s, int& lt) {
  if (a.max_qlen == 1) {   // every request has one row's tiles: no walk over the requests
    const int nt = (a.Hq + ROWS - 1) / ROWS, from_last = (int)blockIdx.x;
    s = a.S - 1 - from_last / nt;
    lt = nt - 1 - from_last % nt;
    return s >= 0;
  }
  int total = 0;
  for (int i = 0; i < a.S; ++i)
    total += ((a.seq_row_start[i + 1] - a.seq_row_start[i]) * a.Hq + ROWS - 1) / ROWS;
  int left = total - 1 - (int)blockIdx.x;
  if (left < 0) return false;
  for (s = 0; s < a.S; ++s) {
    const int nt = ((a.seq_row_start[s + 1] - a.seq_row_start[s]) * a.Hq + ROWS - 1) / ROWS;
    if (left < nt) {
      lt = left;
      return true;
    }
    left -= nt;
  }
  return false;
}

// Eight waves. HALF: steps of 16 numbers of half a cached row. CT: tiles of 16 output columns of a
// wave, whose columns are 16 CT w ... In LDS lie one tile of 64 keys, the scores (two halves of
// the sum) and the probabilities; the queries stay in registers.
template <int ROWS, int HALF, int CT>
__global__ __launch_bounds__(kLatThreads, 2) void latent_attention_tile_kernel(LatentArgs a, LatentTilePlan pl) {
  extern __shared__ float smem[];
  constexpr int KROW = 32 * HALF + 8;                 // row length of a key in LDS (numbers)
  constexpr int RT = ROWS / 16;
  constexpr int PIECES = (kLatKeys * 4 * HALF + kLatThreads - 1) / kLatThreads;   // 16-byte pieces a thread fetches
  constexpr int PARTS = kLatThreads / ROWS, KEYS = kLatKeys / PARTS;   // threads of a row in the softmax, keys of each
  constexpr bool WIDE = ROWS == 64;   // scores in tiles of 32 rows x 32 keys, else 16 x 16
  constexpr int QF = WIDE ? HALF : (HALF + 1) / 2;
  const int Dk = a.R + a.rd, R = a.R, H = a.Hq;
  __bf16* Ks = (__bf16*)smem;                                   // [64][KROW]
  float* Sp = (float*)(Ks + kLatKeys * KROW);                   // [2][ROWS][64]
  __bf16* Ps = (__bf16*)(Sp + 2 * ROWS * kLatKeys);             // [ROWS][72]
  float* alpha_s = (float*)(Ps + ROWS * kLatPRow);              // [ROWS], then m and l
  float* m_s = alpha_s + ROWS;
  float* l_s = m_s + ROWS;
  __shared__ int page_s[2][kLatKeys];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;

  int s, lt;
  if (!latent_block_tile<ROWS>(a, s, lt)) return;
  const int chunk_id = blockIdx.y;
  const int row0 = a.seq_row_start[s];
  const int n_flat = (a.seq_row_start[s + 1] - row0) * H;
  const int pos0 = a.seq_pos0[s];
  const int f0 = lt * ROWS;                          // first flattened row of the tile
  const int rows_here = min(ROWS, n_flat - f0);
  if (rows_here <= 0) return;   // (a request without rows in a decode-only step)
  const int tok_first = f0 / H, tok_last = (f0 + rows_here - 1) / H;
  const int pos_last = pos0 + tok_last;
  const int lo_first = a.window > 0 ? max(0, pos0 + tok_first - a.window + 1) : 0;
  // this block's keys: its part of the tiles that its rows can see (so that the chunks of a
  // request are even, however much shorter it is than the longest)
  const int first_tile = lo_first / kLatKeys, n_tiles = pos_last / kLatKeys + 1 - first_tile;
  const int per_chunk = (n_tiles + pl.n_chunks - 1) / pl.n_chunks;
  const int k_begin = (first_tile + min(chunk_id * per_chunk, n_tiles)) * kLatKeys;
  const int k_end = min((first_tile + min((chunk_id + 1) * per_chunk, n_tiles)) * kLatKeys, pos_last + 1);
  const int* bt = a.block_table + (int64_t)s * a.bt_stride;
  const __bf16* pool = (const __bf16*)a.pool;

  // A tile's keys travel page -> registers -> LDS; the loads of the next tile are issued before
  // the products of this one. Keys outside what the rows see are fetched from the nearest that
  // they do (their probabilities are 0), so that no load waits for a condition.
  const int cpr = Dk / 8;   // 16-byte pieces of a cached row
  lat_bf16x8 next[PIECES];
  int piece[PIECES];        // key of the tile << 16 | first number of the piece
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int e = min(tid + kLatThreads * i, kLatKeys * cpr - 1);
    piece[i] = ((e / cpr) << 16) | (8 * (e % cpr));
  }
  // The pages of a tile's keys come through LDS, looked up two tiles ahead by one wave: a wave's loads
  // return in order, and an address that waits for the block table would wait for the tile before.
  auto page_of = [&](int kt) { return bt[min(max(kt + lane, lo_first), pos_last) >> pl.page_shift]; };
  auto fetch = [&](int kt, const int* pages) {
    int page[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) page[i] = pages[piece[i] >> 16];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int kp = min(max(kt + (piece[i] >> 16), lo_first), pos_last);
      const __bf16* at = pool + ((int64_t)page[i] * a.page_size + (kp & (a.page_size - 1))) * Dk + (piece[i] & 0xffff);
      next[i] = *(page[i] >= 0 ? (const lat_bf16x8*)at : &kLatNoKey);
    }
  };
  int page_next = 0;   // wave 0: the page of key `lane`, two tiles ahead
  if (w == 0 && k_begin < k_end) {
    page_s[0][lane] = page_of(k_begin);
    page_s[1][lane] = page_of(k_begin + kLatKeys);
    page_next = page_of(k_begin + 2 * kLatKeys);
  }
  __syncthreads();
  if (k_begin < k_end) fetch(k_begin, page_s[0]);

  // Q' as the products' operand, rounded to bfloat16 once; zeros beyond the row's numbers. In the
  // wide form wave w has rows 32 (w / 4) .., keys 32 (w / 2 % 2) .. and one half of the numbers;
  // in the other all 16 rows, keys 16 (w / 2) .. and one half of the numbers.
  const int kh = w & 1, kn = WIDE ? (w >> 1) & 1 : w >> 1;
  const int q_lane = WIDE ? lane & 31 : lane & 15, q_k = 8 * (WIDE ? lane >> 5 : lane >> 4);
  constexpr int STEP = WIDE ? 16 : 32;
  lat_bf16x8 qf[QF];
  {
    const int f = f0 + min((WIDE ? 32 * (w >> 2) : 0) + q_lane, rows_here - 1);
    const float* src = a.q_abs + ((int64_t)(row0 + f / H) * H + f % H) * Dk;
#pragma unroll
    for (int st = 0; st < QF; ++st) {
      const int in_half = STEP * st + q_k, d = 16 * HALF * kh + in_half;
      const bool in = d < Dk && in_half < 16 * HALF;
      const lat_f32x4 lo = *(const lat_f32x4*)(src + (in ? d : 0)), up = *(const lat_f32x4*)(src + (in ? d + 4 : 0));
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        qf[st][x] = in ? (__bf16)lo[x] : (__bf16)0.f;
        qf[st][4 + x] = in ? (__bf16)up[x] : (__bf16)0.f;
      }
    }
  }
  {   // the columns of a key's row beyond its numbers are read as zeros and never written again
    const int pad = KROW - Dk;
    for (int e = tid; e < kLatKeys * pad; e += kLatThreads) Ks[(e / pad) * KROW + Dk + e % pad] = (__bf16)0.f;
  }

  // softmax threads: row tid / PARTS, keys KEYS (tid % PARTS) .. of a tile
  const int sm_row = tid / PARTS, sm_part = tid % PARTS;
  int sm_pos = -1, sm_lo = 0;
  if (sm_row < rows_here) {
    sm_pos = pos0 + (f0 + sm_row) / H;
    sm_lo = a.window > 0 ? max(0, sm_pos - a.window + 1) : 0;
  }
  const float scale2 = a.scale * kLatLog2e;
  float m_run = -INFINITY, l_run = 0.f;   // (of the scores times log2 e)

  lat_f32x4 acc[CT][RT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[ct][rt] = lat_f32x4{0.f, 0.f, 0.f, 0.f};
  const int c = lane & 15, g = lane >> 4;

  // The loop writes a place of page_s that the fetch one tile before has read, always with a barrier
  // of that tile between the two; before the first tile this is that barrier.
  lds_barrier();
  int turn = 0;   // of the two places for pages: this tile's, where those two tiles ahead go
  for (int kt = k_begin; kt < k_end; kt += kLatKeys, turn ^= 1) {
    // 1. the tile's keys into LDS as they lie in their pages
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      *(lat_bf16x8*)(Ks + (piece[i] >> 16) * KROW + (piece[i] & 0xffff)) = next[i];
    if (w == 0) page_s[turn][lane] = page_next;
    if (kt + kLatKeys < k_end) fetch(kt + kLatKeys, page_s[turn ^ 1]);
    if (w == 0) page_next = page_of(kt + 3 * kLatKeys);
    lds_barrier();   // (orders LDS traffic only: the next tile's loads stay under way)
    // 2. scores over one half of the numbers
    float* sp = Sp + kh * ROWS * kLatKeys;
    if constexpr (WIDE) {
      lat_f32x16 sacc = {};
      const __bf16* krow = Ks + (32 * kn + q_lane) * KROW + 16 * HALF * kh + q_k;
#pragma unroll
      for (int st = 0; st < QF; ++st)
        sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[st], *(const lat_bf16x8*)(krow + 16 * st), sacc, 0, 0, 0);
      // the lane holds key 32 kn + q_lane for rows 8 q + 4 (lane / 32) + r in register 4 q + r
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sp[(32 * (w >> 2) + 8 * q + 4 * (lane >> 5) + r) * kLatKeys + 32 * kn + q_lane] = sacc[4 * q + r];
    } else {
      lat_f32x4 sacc = {};
      // (the last step of an odd HALF has 16 numbers of the half: the lanes beyond have zeros in
      // the queries, and read any number)
      const __bf16* krow = Ks + (16 * kn + c) * KROW + 16 * HALF * kh + q_k;
#pragma unroll
      for (int st = 0; st < QF; ++st) {
        const bool past = HALF % 2 && st == QF - 1 && g >= 2;
        const lat_bf16x8 kf = *(const lat_bf16x8*)(krow + (past ? 0 : 32 * st));
        sacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[st], kf, sacc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) sp[(4 * g + r) * kLatKeys + 16 * kn + c] = sacc[r];
    }
    lds_barrier();
    // 3. softmax of the tile, 32-bit
    {
      float sv[KEYS];
      float mx = -INFINITY;
#pragma unroll
      for (int x = 0; x < KEYS; ++x) {
        const int j = KEYS * sm_part + x, kp = kt + j;
        const float v = (Sp[sm_row * kLatKeys + j] + Sp[(ROWS + sm_row) * kLatKeys + j]) * scale2;
        sv[x] = kp <= sm_pos && kp >= sm_lo ? v : -INFINITY;
        mx = fmaxf(mx, sv[x]);
      }
#pragma unroll
      for (int off = 1; off < PARTS; off *= 2) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
      const float m_new = fmaxf(m_run, mx);
      const float ref = m_new == -INFINITY ? 0.f : m_new;   // nothing seen so far: all terms are 0
      const float al = __builtin_amdgcn_exp2f(m_run - ref);   // 0 while m_run is minus infinity
      float sum = 0.f;
      __bf16* prow = Ps + sm_row * kLatPRow + KEYS * sm_part;
#pragma unroll
      for (int x = 0; x < KEYS; ++x) {
        const float p = __builtin_amdgcn_exp2f(sv[x] - ref);
        prow[x] = (__bf16)p;
        sum += p;
      }
#pragma unroll
      for (int off = 1; off < PARTS; off *= 2) sum += __shfl_xor(sum, off, 64);
      l_run = l_run * al + sum;
      m_run = m_new;
      if (sm_part == 0) alpha_s[sm_row] = al;
    }
    lds_barrier();
    // 4. O = O alpha + P V on this wave's columns: V^T comes through the transposing read, a lane
    // (c, g) holds column c of a tile for keys 8 g .. + 7; P^T row c of a tile for the same keys
    {
      float al[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) al[rt] = alpha_s[16 * rt + c];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[ct][rt] *= al[rt];
#pragma unroll
      for (int k0 = 0; k0 < kLatKeys; k0 += 32) {
        lat_bf16x8 pf[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) pf[rt] = *(const lat_bf16x8*)(Ps + (16 * rt + c) * kLatPRow + k0 + 8 * g);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const int col = 16 * (CT * w + ct);
          if (col < R) {
            const __bf16* v = Ks + (k0 + 8 * g + (c >> 2)) * KROW + col + 4 * (c & 3);
            const lat_short4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lat_lds_short4*)v);
            const lat_short4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lat_lds_short4*)(v + 4 * KROW));
            const lat_short8 both = {lo.x, lo.y, lo.z, lo.w, up.x, up.y, up.z, up.w};
            const lat_bf16x8 vf = __builtin_bit_cast(lat_bf16x8, both);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
              acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[rt], acc[ct][rt], 0, 0, 0);
          }
        }
      }
    }
    lds_barrier();
  }

  if (sm_part == 0) {
    m_s[sm_row] = m_run * (1.f / kLatLog2e);   // (of the scores themselves: what the merge expects)
    l_s[sm_row] = l_run;
  }
  __syncthreads();
  // The lane holds row c of every row tile (a (token, head) pair) and columns 4 g .. of every column tile.
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int i = 16 * rt + c;
    if (i >= rows_here) continue;
    const int f = f0 + i, t = row0 + f / H, h = f % H;
    const float l = l_s[i];
    float factor = 1.f;
    float* part = nullptr;
    if (pl.n_chunks == 1) {
      factor = l > 0.f ? 1.f / l : 0.f;
      if (a.gate) {
        const float z = __bfloat162float(((const bf16*)a.gate)[(int64_t)t * a.gate_stride + h]);
        factor *= 1.f / (1.f + expf(-z));
      }
    } else {
      part = a.workspace + (((int64_t)t * H + h) * pl.n_chunks + chunk_id) * (R + 2);
      if (w == 0 && g == 0) {
        part[R] = m_s[i];
        part[R + 1] = l;
      }
    }
    __bf16* orow = (__bf16*)a.out + ((int64_t)t * H + h) * R;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * (CT * w + ct) + 4 * g + r;
        if (d >= R) continue;
        if (part) part[d] = acc[ct][rt][r];
        else orow[d] = (__bf16)(acc[ct][rt][r] * factor);
      }
  }
}

// The same in blocks of 64 rows for cached rows of 32 QF numbers whose first 16 NC are the latent: four
// waves of 16 (token, head) rows each, which keep their queries, their running maxima and sums and all
// columns of their outputs in registers, so that nothing passes between waves but the keys. Tiles
// of 32 keys come straight into LDS (global_load_lds), the next one while this one is multiplied: one barrier a
// tile, two blocks a CU. S^T = K Q^T leaves the lane (c, g) with row c and keys 4 g .. + 3 of each 16; the
// products with the values take the keys in that order (the transposing reads follow it), so the
// probabilities go from the scores to the operand without leaving the lane. A row's exponent reference
// follows its maximum only in jumps of 2^16, which the sums' and bfloat16's exponents hold, so that the 4 NC output
// registers are rescaled rarely (with jumps of 2^8 a whole 2,048-token Getodra prompt takes 0.7% longer).
// What bounds it is the LDS (68 KB of operands a wave and tile at 512 + 64 numbers, twice the matrix cores' time)
// and, with 251 registers, reads only two or three products ahead. Against the kernel above: prompts of 2,048
// tokens, 16 heads, 512 + 64 numbers 202 -> 140 us; 8 heads, 256 + 32 numbers 111 -> 74; 512 tokens behind 2,000 cached
// ones 190 -> 146; 64 requests of one row and 40 heads at 2,500 keys 83 -> 60.
// In LDS rows are unpadded (a load writes 1 KB side by side): the 16-byte piece p of key k lies at
// p ^ x(k) (lat_swizzle), chosen on the global side, so that the 16 keys of a fragment read fall into
// different columns of the banks.
constexpr int kLatRowsKeys = 32;
template <int PIECES_A_ROW> __device__ __forceinline__ int lat_swizzle(int key) {
  if constexpr (PIECES_A_ROW % 8 == 0) return (key >> 1) & 7;
  else return (key >> 2) & 3;   // (a multiple of 4: QF steps of 32 numbers)
}

template <int QF, int NC>
__global__ __launch_bounds__(256, 2) void latent_attention_rows_kernel(LatentArgs a, LatentTilePlan pl) {
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass does not know buffer resources)
  constexpr int ROWS = 64, KT = kLatRowsKeys, CPR = 4 * QF, DK = 32 * QF;
  constexpr int LOADS = (8 * CPR + 63) / 64;          // of a wave and tile: 8 keys, 1 KB a load
  constexpr int TILE = 4 * LOADS * 1024;
  static_assert(KT == 32 && 16 * DK < 65536, "a wave's keys");
  extern __shared__ float smem[];
  unsigned char* Ks = (unsigned char*)smem;           // [2][TILE]
  int (*page_s)[KT] = (int (*)[KT])(Ks + 2 * TILE);   // [2][KT]
  const int R = a.R, H = a.Hq;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;

  int s, lt;
  if (!latent_block_tile<ROWS>(a, s, lt)) return;
  const int chunk_id = blockIdx.y;
  const int row0 = a.seq_row_start[s];
  const int n_flat = (a.seq_row_start[s + 1] - row0) * H;
  const int pos0 = a.seq_pos0[s];
  const int f0 = lt * ROWS;
  const int rows_here = min(ROWS, n_flat - f0);
  if (rows_here <= 0) return;   // (a request without rows in a decode-only step)
  const int tok_first = f0 / H, tok_last = (f0 + rows_here - 1) / H;
  const int pos_last = pos0 + tok_last;
  const int lo_first = a.window > 0 ? max(0, pos0 + tok_first - a.window + 1) : 0;
  const int first_tile = lo_first / kLatKeys, n_tiles = pos_last / kLatKeys + 1 - first_tile;
  const int per_chunk = (n_tiles + pl.n_chunks - 1) / pl.n_chunks;
  const int k_begin = (first_tile + min(chunk_id * per_chunk, n_tiles)) * kLatKeys;
  const int k_end = min((first_tile + min((chunk_id + 1) * per_chunk, n_tiles)) * kLatKeys, pos_last + 1);
  const int* bt = a.block_table + (int64_t)s * a.bt_stride;
  const __bf16* pool = (const __bf16*)a.pool;

  typedef const __attribute__((address_space(1))) void* gptr;
  typedef __attribute__((address_space(3))) void* lptr;
  // Wave w fetches keys 8 w .. + 7 of a tile, CPR loads of 8 lanes' worth a key: LOADS of 64 lanes, of which the
  // last may reach into padding. Where all keys of the tile are seen by some row and pages hold 8 keys or more, the
  // wave's keys lie side by side in one page: a scalar base and the lanes' offsets, which no tile changes.
  // Elsewhere (the first and last tile, small pages, pages that the table does not hold) key by key: keys
  // outside what the rows see from the nearest that they do (their probabilities are 0).
  auto place = [&](int ln, int j, int& key, int& piece) {
    const int f = 8 * CPR % 64 ? min(64 * j + ln, 8 * CPR - 1) : 64 * j + ln;
    key = f / CPR;
    piece = (f % CPR) ^ lat_swizzle<CPR>(8 * w + key);
  };
  // Byte offsets of two loads each, where they fit the registers; with 32 tiles of output columns they are
  // formed again in every tile (kept they spill: 2,048 tokens of 16 heads, 512 + 64 numbers, 254 against 140 us; formed
  // again at 8 heads of 256 + 32 84 against 74).
  constexpr bool KEPT = NC <= 16;
  unsigned off2[KEPT ? (LOADS + 1) / 2 : 1] = {};
  if constexpr (KEPT) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      int key, piece;
      place(lane, j, key, piece);
      off2[j / 2] |= (unsigned)(key * (2 * DK) + 16 * piece) << (j % 2 ? 16 : 0);
    }
  }
  auto fetch = [&](int kt, int buf) {
    unsigned char* to = Ks + buf * TILE + w * (LOADS * 1024);
    int ln = lane;
    asm volatile("" : "+v"(ln));   // (so that nothing formed from it is kept)
    const int page = __builtin_amdgcn_readfirstlane(page_s[buf][8 * w]);
    if (kt >= lo_first && kt + KT - 1 <= pos_last && a.page_size >= 8 && page >= 0) {
      const __bf16* base = pool + ((int64_t)page * a.page_size + ((kt + 8 * w) & (a.page_size - 1))) * DK;
      const auto res = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 16 * DK, 0x00020000);   // (8 keys)
#pragma unroll
      for (int j = 0; j < LOADS; ++j) {
        unsigned at;
        if constexpr (KEPT) {
          at = j % 2 ? off2[j / 2] >> 16 : off2[j / 2] & 0xffff;
        } else {
          int key, piece;
          place(ln, j, key, piece);
          at = key * (2 * DK) + 16 * piece;
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (lptr)(to + j * 1024), 16, at, 0, 0, 0);
      }
      return;
    }
#pragma unroll 1
    for (int j = 0; j < LOADS; ++j) {
      int key, piece;
      place(ln, j, key, piece);
      const int kp = min(max(kt + 8 * w + key, lo_first), pos_last), pg = page_s[buf][8 * w + key];
      const __bf16* at = pool + ((int64_t)pg * a.page_size + (kp & (a.page_size - 1))) * DK + 8 * piece;
      __builtin_amdgcn_global_load_lds((gptr)(pg >= 0 ? (const void*)at : (const void*)&kLatNoKey), (lptr)(to + j * 1024),
                                       16, 0, 0);
    }
  };
  // pages of a tile's keys, looked up by lanes of wave 0 two tiles ahead
  auto page_of = [&](int kt) { return bt[min(max(kt + (lane & (KT - 1)), lo_first), pos_last) >> pl.page_shift]; };
  int page_next = 0;
  if (w == 0 && k_begin < k_end) {
    if (lane < KT) {
      page_s[0][lane] = page_of(k_begin);
      page_s[1][lane] = page_of(k_begin + KT);
    }
    page_next = page_of(k_begin + 2 * KT);
  }
  __syncthreads();
  if (k_begin < k_end) fetch(k_begin, 0);

  // Q' as the products' operand, rounded to bfloat16 once: lane (c, g) has row 16 w + c, numbers 8 g .. of a step
  const int my = 16 * w + c, f_row = f0 + min(my, rows_here - 1);
  lat_bf16x8 qf[QF];
  {
    const float* src = a.q_abs + ((int64_t)(row0 + f_row / H) * H + f_row % H) * DK + 8 * g;
#pragma unroll
    for (int st = 0; st < QF; ++st) {
      const lat_f32x4 lo = *(const lat_f32x4*)(src + 32 * st), up = *(const lat_f32x4*)(src + 32 * st + 4);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        qf[st][x] = (__bf16)lo[x];
        qf[st][4 + x] = (__bf16)up[x];
      }
    }
  }
  const int my_pos = pos0 + f_row / H, my_lo = a.window > 0 ? max(0, my_pos - a.window + 1) : 0;
  const float scale2 = a.scale * kLatLog2e;
  float m_ref = -INFINITY, l_run = 0.f;   // (of the scores times log2 e); l: this lane's keys alone
  lat_f32x4 acc[NC];
#pragma unroll
  for (int ct = 0; ct < NC; ++ct) acc[ct] = lat_f32x4{0.f, 0.f, 0.f, 0.f};

  // Fragment addresses in a tile. Keys 16 i + c: piece 4 st + g, at (4 st + g) ^ x; x's third bit swaps the
  // steps 2 n and 2 n + 1. (x is the same for keys 16 apart.)
  const int xk = lat_swizzle<CPR>(c), k_low = (c >> 3) * (LOADS * 1024) + (c & 7) * (16 * CPR) + 16 * (g ^ (xk & 3)), k_swap = 64 * (xk >> 2);
  // Values: transposing reads, lane at key 4 g + c / 4 (and 16 further), columns 4 (c % 4) of a tile of 16
  // (pieces 2 ct and 2 ct + 1; x moves them within a group of eight, so four tiles have addresses of their own)
  const int v_key = 4 * g + (c >> 2), xv = lat_swizzle<CPR>(v_key);
  int v_at[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v_at[j] = (v_key >> 3) * (LOADS * 1024) + (v_key & 7) * (16 * CPR) + 8 * (c & 1) + 16 * ((2 * j + ((c >> 1) & 1)) ^ xv);
  typedef __attribute__((address_space(3))) lat_short4* trptr;

  int turn = 0;
  for (int kt = k_begin; kt < k_end; kt += KT, turn ^= 1) {
    // this wave's part of the tile has landed, and after the barrier everybody's has; everybody has also
    // read the tile before, whose place the next one takes
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + KT < k_end) fetch(kt + KT, turn ^ 1);
    if (w == 0) {   // (the places of this tile's pages were read one tile ago)
      if (lane < KT) page_s[turn][lane] = page_next;
      page_next = page_of(kt + 3 * KT);
    }
    const unsigned char* tile = Ks + turn * TILE;
    // (fragments are read two steps, and values three tiles of columns, ahead of their products; the fences
    // keep the compiler from moving the reads back to them)
    lat_f32x4 sc[2] = {};
    lat_bf16x8 kf[3][2];
    auto read_keys = [&](int st) {
      const unsigned char* at = tile + k_low + 64 * st + (st % 2 ? -k_swap : k_swap);
#pragma unroll
      for (int i = 0; i < 2; ++i) kf[st % 3][i] = *(const lat_bf16x8*)(at + i * (2 * LOADS * 1024));
    };
    read_keys(0);
    read_keys(1);
#pragma unroll
    for (int st = 0; st < QF; ++st) {
      if (st + 2 < QF) read_keys(st + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        sc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[st % 3][i], qf[st], sc[i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    float sv[8], mx = -INFINITY;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int kp = kt + 16 * (x / 4) + 4 * g + x % 4;
      const float v = sc[x / 4][x % 4] * scale2;
      sv[x] = kp <= my_pos && kp >= my_lo ? v : -INFINITY;
      mx = fmaxf(mx, sv[x]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m_ref + 16.f)) {   // (also a row's first visible key: its reference is minus infinity)
      // (each row by its own maximum: rows that do not jump keep their reference, whatever their neighbours do)
      const float m_new = mx > m_ref + 16.f ? mx : m_ref;
      const float al = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_ref - m_new);
      l_run *= al;
#pragma unroll
      for (int ct = 0; ct < NC; ++ct) acc[ct] *= al;
      m_ref = m_new;
    }
    const float ref = m_ref == -INFINITY ? 0.f : m_ref;   // nothing seen so far: all terms are 0
    lat_bf16x8 pf;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const float p = __builtin_amdgcn_exp2f(sv[x] - ref);
      pf[x] = (__bf16)p;
      l_run += p;
    }
    lat_short4 vf[4][2];
    auto read_values = [&](int ct) {
      const unsigned char* v = tile + v_at[ct % 4] + 128 * (ct / 4);
      vf[ct % 4][0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr)v);
      vf[ct % 4][1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((trptr)(v + 2 * LOADS * 1024));
    };
#pragma unroll
    for (int ct = 0; ct < 3; ++ct) read_values(ct);
#pragma unroll
    for (int ct = 0; ct < NC; ++ct) {
      if (ct + 3 < NC) read_values(ct + 3);
      __builtin_amdgcn_sched_barrier(0);
      const lat_short4 lo = vf[ct % 4][0], up = vf[ct % 4][1];
      const lat_short8 both = {lo.x, lo.y, lo.z, lo.w, up.x, up.y, up.z, up.w};
      acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lat_bf16x8, both), pf, acc[ct], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (my >= rows_here) return;
  // The lane holds its row's columns 16 ct + 4 g ..
  const int t = row0 + f_row / H, h = f_row % H;
  if (pl.n_chunks > 1) {
    float* part = a.workspace + (((int64_t)t * H + h) * pl.n_chunks + chunk_id) * (R + 2);
    if (g == 0) {
      part[R] = m_ref * (1.f / kLatLog2e);   // (of the scores themselves: what the merge expects)
      part[R + 1] = l_run;
    }
#pragma unroll
    for (int ct = 0; ct < NC; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[16 * ct + 4 * g + r] = acc[ct][r];
    return;
  }
  float factor = l_run > 0.f ? 1.f / l_run : 0.f;
  if (a.gate) {
    const float z = __bfloat162float(((const bf16*)a.gate)[(int64_t)t * a.gate_stride + h]);
    factor *= 1.f / (1.f + expf(-z));
  }
  typedef __bf16 lat_bf16x4 __attribute__((ext_vector_type(4)));
  __bf16* orow = (__bf16*)a.out + ((int64_t)t * H + h) * R;
#pragma unroll
  for (int ct = 0; ct < NC; ++ct) {
    lat_bf16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (__bf16)(acc[ct][r] * factor);
    *(lat_bf16x4*)(orow + 16 * ct + 4 * g) = o;
  }
#endif
}

// out[t, h] = sum_c e^(m_c - M) O_c / sum_c e^(m_c - M) l_c over the chunks that saw keys.
__global__ void latent_attention_merge_kernel(LatentArgs a, int n_chunks) {
  extern __shared__ float smem[];   // [n_chunks] weight of each chunk: e^(m_c - M) / L (0: saw no key)
  __shared__ float red[16];
  const int64_t th = blockIdx.x;
  const int R = a.R;
  const float* part = a.workspace + th * n_chunks * (R + 2);
  float M = -INFINITY;
#pragma unroll 8
  for (int c = 0; c < n_chunks; ++c) M = fmaxf(M, part[c * (R + 2) + R]);
  float mine = 0.f;
  for (int c = threadIdx.x; c < n_chunks; c += blockDim.x) {
    const float m = part[c * (R + 2) + R];
    const float wgt = m > -INFINITY ? expf(m - M) : 0.f;
    smem[c] = wgt;
    mine += wgt * part[c * (R + 2) + R + 1];
  }
  const float L = block_sum(mine, red);   // (its barriers publish the weights)
  float inv = L > 0.f ? 1.f / L : 0.f;
  if (a.gate) {
    const int t = (int)(th / a.Hq), h = (int)(th % a.Hq);
    const float g = __bfloat162float(((const bf16*)a.gate)[(int64_t)t * a.gate_stride + h]);
    inv *= 1.f / (1.f + expf(-g));
  }
  __bf16* orow = (__bf16*)a.out + th * R;
  for (int d = threadIdx.x; d < R; d += blockDim.x) {
    // (a chunk that saw no key left zeros and has weight 0: no branch, so that the loads of
    // several chunks are under way together)
    float o = 0.f;
#pragma unroll 8
    for (int c = 0; c < n_chunks; ++c) o = fmaf(smem[c], part[c * (R + 2) + d], o);
    orow[d] = (__bf16)(o * inv);
  }
}

template <int ROWS, int HALF, int CT>
static int launch_latent_tile(const LatentArgs& a, const LatentTilePlan& p, hipStream_t stream) {
  auto kern = latent_attention_tile_kernel<ROWS, HALF, CT>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds);
  if (e != hipSuccess) return set_error(-2, "latent_attention: cannot get %zu bytes of LDS", p.lds);
  kern<<<dim3(p.tiles, p.n_chunks), kLatThreads, p.lds, stream>>>(a, p);
  NINFER_LAUNCH_CHECK();
  return 0;
}

template <int ROWS>
static int launch_latent_rows(const LatentArgs& a, const LatentTilePlan& p, hipStream_t stream) {
  const bool few = a.R <= 256;   // output columns: 8 waves of 2 or 4 tiles of 16
#define NINFER_LATENT_HALF(H) \
  if (p.half == H) return few ? launch_latent_tile<ROWS, H, 2>(a, p, stream) : launch_latent_tile<ROWS, H, 4>(a, p, stream)
  NINFER_LATENT_HALF(5);
  NINFER_LATENT_HALF(9);
  NINFER_LATENT_HALF(13);
  NINFER_LATENT_HALF(18);
#undef NINFER_LATENT_HALF
  return few ? launch_latent_tile<ROWS, 20, 2>(a, p, stream) : launch_latent_tile<ROWS, 20, 4>(a, p, stream);
}

template <int QF, int NC>
static int launch_latent_waves(const LatentArgs& a, const LatentTilePlan& p, hipStream_t stream) {
  constexpr size_t lds = 2 * 4 * ((8 * 4 * QF + 63) / 64 * 1024) + 2 * kLatRowsKeys * sizeof(int);
  auto kern = latent_attention_rows_kernel<QF, NC>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return set_error(-2, "latent_attention: cannot get %zu bytes of LDS", lds);
  kern<<<dim3(p.tiles, p.n_chunks), 256, lds, stream>>>(a, p);
  NINFER_LAUNCH_CHECK();
  return 0;
}

static int latent_attention_tile(const LatentArgs& a, hipStream_t stream) {
  const LatentTilePlan p = latent_tile_plan(a);
  const int64_t need = latent_tile_workspace_floats(a, p);
  NINFER_REQUIRE(need == 0 || (a.workspace && a.workspace_floats >= need),
                 "latent_attention: the workspace holds %lld floats, %lld are needed",
                 (long long)a.workspace_floats, (long long)need);
  int rc;
  if (p.rows == 16) rc = launch_latent_rows<16>(a, p, stream);
  else if (!latent_rows_form(a) || (uintptr_t)a.out % 8 != 0) rc = launch_latent_rows<64>(a, p, stream);
  else if (a.R == 512) rc = a.rd == 64 ? launch_latent_waves<18, 32>(a, p, stream) : launch_latent_waves<17, 32>(a, p, stream);
  else rc = a.rd == 64 ? launch_latent_waves<10, 16>(a, p, stream) : launch_latent_waves<9, 16>(a, p, stream);
  if (rc) return rc;
  if (p.n_chunks > 1) {
    const int block = a.R >= 256 ? 256 : (a.R + 63) / 64 * 64;
    latent_attention_merge_kernel<<<(unsigned)((int64_t)a.T * a.Hq), block, p.n_chunks * sizeof(float), stream>>>(a, p.n_chunks);
    NINFER_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace ninfer

// 32-bit floats of workspace that a step of this shape needs (0: none).
extern "C" long long ninfer_latent_attention_workspace_floats(const ninfer::LatentArgs* a) {
  if (!ninfer::latent_tile_takes(*a)) return 0;
  return ninfer::latent_tile_workspace_floats(*a, ninfer::latent_tile_plan(*a));
}

// (token, head) rows of a block of the matrix-core kernels for a step of this shape, 16 or 64 (0: the plain kernel).
extern "C" int ninfer_latent_attention_block_rows(const ninfer::LatentArgs* a) {
  return ninfer::latent_tile_takes(*a) ? ninfer::latent_tile_plan(*a).rows : 0;
}

// ---- keys and values per head for prompts ---------------------------------------------------------------
// A prompt's rows are many to a key: forming every head's key and value once (a product over the cached rows,
// 2 R (dim + vdim) operations a head) and attending with dim + rd and vdim numbers a head takes a quarter of the
// operations of attending in the latent's space (R + rd and R numbers). 2,048 tokens, 16 heads, 512 + 64 numbers,
// heads of 64 + 64 and 128: 61 us against 178 with the queries' and the values' products around it (attention alone 42
// against 140); against 64-bit sums 0.0027 against 0.0031 off.
// The keys' turned numbers stay one row for all heads; keys and values are rounded to bfloat16 where the other
// form rounds the query in the latent's space and the sum of latents.
namespace ninfer {

// A wave to a key: its cached row apart into the latent and the turned numbers, in the order of requests and
// positions (a page that the table does not hold: zeros).
__global__ __launch_bounds__(256) void latent_rows_kernel(LatentArgs a, LatentHeadsArgs b) {
  const int lane = threadIdx.x & 63, key = blockIdx.x * 4 + (threadIdx.x >> 6);
  int first = 0, s = -1, p = 0;   // the request that has the key, and the key's position
  for (int s0 = 0; s0 < a.S; s0 += 64) {
    const int i = s0 + lane, n = i < a.S ? a.seq_pos0[i] + b.seq_qlen[i] : 0;
    int upto = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(upto, off, 64);
      if (lane >= off) upto += v;
    }
    const int begin = first + upto - n;
    if (key == 0 && i < a.S) b.key_start[i] = begin;
    const unsigned long long mine = __ballot(key >= begin && key < begin + n);
    if (mine) {
      const int l = __ffsll(mine) - 1;
      s = s0 + l;
      p = key - __shfl(begin, l, 64);
    }
    first += __shfl(upto, 63, 64);
  }
  if (key >= b.keys || s < 0) return;
  const int page = a.block_table[(int64_t)s * a.bt_stride + p / a.page_size];
  const int Dk = a.R + a.rd;
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const bf16* row = (const bf16*)a.pool + ((int64_t)max(page, 0) * a.page_size + p % a.page_size) * Dk;
  for (int i = 8 * lane; i < Dk; i += 512) {
    const u32x4 v = page >= 0 ? *(const u32x4*)(row + i) : u32x4{0u, 0u, 0u, 0u};
    bf16* to = i < a.R ? (bf16*)b.latent + (int64_t)key * a.R + i : (bf16*)b.krot + (int64_t)key * a.rd + (i - a.R);
    *(u32x4*)to = v;
  }
}

// Which sizes the form is built for: bfloat16, heads of 128 numbers with values of 64 or 128, all keys visible,
// pieces of 16 bytes that lie wholly in one part of a row.
static bool latent_heads_takes(const LatentArgs& a, int vdim) {
  return a.dtype == kBF16 && !a.force_plain && a.dim + a.rd == 128 && a.rd > 0 && a.dim % 8 == 0 && a.R % 8 == 0 &&
         (vdim == 64 || vdim == 128) && a.window == 0 && a.seq_row_start && a.seq_pos0 && a.S > 0;
}

static int latent_heads_check(const LatentArgs& a, const LatentHeadsArgs& b, const char* who) {
  if (int rc = latent_check(a, who)) return rc;
  NINFER_REQUIRE(latent_heads_takes(a, b.vdim), "%s: heads of %d + %d and values of %d numbers, latent %d, window %d",
                 who, a.dim, a.rd, b.vdim, a.R, a.window);
  NINFER_REQUIRE(b.keys > 0 && b.krot && b.key_start && b.seq_qlen, "%s: %d keys without a place", who, b.keys);
  NINFER_REQUIRE((uintptr_t)b.krot % 16 == 0, "%s: rows that do not lie on 16 bytes", who);
  return 0;
}

}  // namespace ninfer

extern "C" int ninfer_latent_heads_takes(const LatentArgs* a, int vdim) { return latent_heads_takes(*a, vdim); }

extern "C" int ninfer_latent_rows(const LatentArgs* a, const LatentHeadsArgs* b, hipStream_t stream) {
  if (int rc = latent_heads_check(*a, *b, "latent_rows")) return rc;
  NINFER_REQUIRE(b->latent && (uintptr_t)b->latent % 16 == 0 && (uintptr_t)a->pool % 16 == 0,
                 "latent_rows: rows that do not lie on 16 bytes");
  latent_rows_kernel<<<(b->keys + 3) / 4, 256, 0, stream>>>(*a, *b);
  NINFER_LAUNCH_CHECK();
  return 0;
}

extern "C" int ninfer_latent_heads_attention(const LatentArgs* l, const LatentHeadsArgs* b, hipStream_t stream) {
  if (int rc = latent_heads_check(*l, *b, "latent_heads_attention")) return rc;
  NINFER_REQUIRE(l->scale > 0.f, "latent_heads_attention: scale %g must be positive", (double)l->scale);
  NINFER_REQUIRE((uintptr_t)b->kv % 16 == 0 && (uintptr_t)b->q % 16 == 0 && (uintptr_t)b->out % 8 == 0,
                 "latent_heads_attention: rows that do not lie on 16 bytes");
  AttnArgs a = {};
  a.q = b->q;
  a.out = b->out;
  a.kpool = b->kv;
  a.vpool = (const bf16*)b->kv + (int64_t)l->Hq * l->dim;
  a.krot = b->krot;
  a.key_start = b->key_start;
  a.kv_stride = l->Hq * (l->dim + b->vdim);
  a.kdim = l->dim;
  a.positions = l->positions;
  a.seq_row_start = l->seq_row_start;
  a.q_stride = l->Hq * 128;
  a.T = l->T;
  a.S = l->S;
  a.Hq = a.Hkv = l->Hq;
  a.D = 128;
  a.Dv = b->vdim;
  a.page_size = 64;
  a.scale = l->scale;
  a.dtype = kBF16;
  a.max_qlen = l->max_qlen;
  a.max_kv_len = l->max_kv_len;
  a.gate = l->gate;
  a.gate_stride = l->gate_stride;
  return attention_prefill(a, stream);
}
