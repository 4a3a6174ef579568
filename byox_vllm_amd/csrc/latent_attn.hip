// Latent attention over a paged cache that holds, per token, one row [latent c (kv_rank) | rotated key part (rot_dim)]
// shared by all heads.  Queries arrive in absorbed form: for head h the first kv_rank numbers are W_uk[h]^T q_unrotated
// (so that their product with c equals q_unrotated . (W_uk[h] c)), the last rot_dim are the rotated query part.  The
// kernel returns sum_j p_j c_j per head; the caller applies W_uv[h] afterwards.  Every head of a token reads the same
// key rows, so a workgroup stages a tile of them in LDS once and serves all its heads from it.
//
//   nv_latent_kv_store : RMS norm of the latent, rotation of the shared key part, store into the token's cache row;
//   nv_latent_norms      with it the query latent's RMS norm, in workgroups beside (launches of 5.7 and 5.8 us for 8 tokens)
//   nv_latent_q_rope   : rotation of the per-head query parts into the absorbed-query buffer
//   nv_latent_attn     : sliding-window softmax attention, one workgroup per (token, group of heads); single tokens of a
//                        request take latent_token.h
//   nv_latent_gather, nv_latent_expand, nv_latent_q_rows : the pieces of the EXPANDED form that long prompt portions
//                        take: the step's requests' cache rows gathered in order, keys and values of every head written
//                        out from their up-projections, whole query rows; ordinary paged attention reads the result
//
// Rotation: dimension i pairs with i + dims/2 ("rotate half"), or with `interleaved` dimension 2i with 2i + 1; the angle
// is position * inv_freq[i] in fp32, and both cosine and sine are multiplied by `mscale` (the caller folds frequency
// scaling into inv_freq and mscale).
#include "anyt.h"
#include "lds_limit.h"

namespace {

// Rows whose norm is taken beside the latent's, in workgroups of their own (blockIdx.y == 1)
struct NormRows {
  const float* x;          // or null
  int64_t rs;
  const void* w;
  void* out;
  int n, quads;
};

// out[j] = x[j] / rms(x) * w[j] by one workgroup; `store`: whether there is a place for it.  In fours (aligned rows of at most 4096) a
// row is read once and kept in registers.
template <typename T>
__device__ __forceinline__ void norm_row(const float* x, const T* w, T* out, int n, float eps, bool quads, bool store, float* red) {
  typedef typename Pack4<T>::type P;
  float ss = 0.0f;
  if (quads) {
    f32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = 4 * (threadIdx.x + 256 * k);
      v[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (j < n) v[k] = *reinterpret_cast<const f32x4*>(x + j);
#pragma unroll
      for (int r = 0; r < 4; ++r) ss += v[k][r] * v[k][r];
    }
    ss = block_sum(ss, red);
    if (!store) return;
    const float inv = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = 4 * (threadIdx.x + 256 * k);
      if (j >= n) continue;
      const f32x4 f = Pack4<T>::widen(*reinterpret_cast<const P*>(w + j));
#pragma unroll
      for (int r = 0; r < 4; ++r) v[k][r] = v[k][r] * inv * f[r];
      *reinterpret_cast<P*>(out + j) = Pack4<T>::narrow(v[k]);
    }
  } else {
    for (int j = threadIdx.x; j < n; j += blockDim.x) ss += x[j] * x[j];
    ss = block_sum(ss, red);
    if (!store) return;
    const float inv = 1.0f / sqrtf(ss / (float)n + eps);
    for (int j = threadIdx.x; j < n; j += blockDim.x) st_f32<T>(out + j, x[j] * inv * ld_f32<T>(w + j));
  }
}

// One token's latent and shared key part into the cache
struct KvRows {
  const float* kv;
  int64_t rs;
  const void* w;
  const int64_t* positions;
  const float* inv_freq;
  float mscale;
  const int32_t* slots;
  void* cache;
  int rank, rot_dim, rot_dims;
  float eps;
  int interleaved;
};

// ... a token's rotated part, by `threads` threads
template <typename T>
__device__ __forceinline__ void latent_rot_store(const KvRows& p, int64_t t, const float* row, T* dst, int thread, int threads) {
  const int rank = p.rank, rot_dims = p.rot_dims;
  const float pos = (float)p.positions[t];
  const int half = rot_dims / 2;
  for (int j = thread; j < p.rot_dim; j += threads) {
    float v = row[rank + j];
    if (j < rot_dims) {
      const bool first = p.interleaved ? (j & 1) == 0 : j < half;
      const int i = p.interleaved ? j >> 1 : (first ? j : j - half);
      const float a = pos * p.inv_freq[i];
      const float cs = cosf(a) * p.mscale, sn = sinf(a) * p.mscale;
      const float other = row[rank + (p.interleaved ? j ^ 1 : (first ? j + half : j - half))];
      v = first ? v * cs - other * sn : v * cs + other * sn;
    }
    st_f32<T>(dst + rank + j, v);
  }
}

template <typename T>
__device__ __forceinline__ void latent_kv_store(const KvRows& p, bool quads, float* red) {
  const int64_t t = blockIdx.x;
  const int32_t slot = p.slots[t];
  const float* row = p.kv + t * p.rs;
  T* dst = reinterpret_cast<T*>(p.cache) + (int64_t)(slot < 0 ? 0 : slot) * (p.rank + p.rot_dim);
  norm_row<T>(row, reinterpret_cast<const T*>(p.w), dst, p.rank, p.eps, quads, slot >= 0, red);
  if (slot >= 0) latent_rot_store<T>(p, t, row, dst, threadIdx.x, blockDim.x);
}

template <typename T, bool QUADS>
__global__ __launch_bounds__(256) void latent_kv_store_kernel(KvRows p) {
  __shared__ float red[32];
  latent_kv_store<T>(p, QUADS, red);
}

template <typename T>
__global__ __launch_bounds__(256) void latent_norms_kernel(KvRows p, int quads, NormRows q) {
  __shared__ float red[32];
  if (blockIdx.y) {
    const int64_t t = blockIdx.x;
    norm_row<T>(q.x + t * q.rs, reinterpret_cast<const T*>(q.w), reinterpret_cast<T*>(q.out) + t * q.n, q.n, p.eps, q.quads, true, red);
  } else {
    latent_kv_store<T>(p, quads, red);
  }
}

// q [tokens, H * (dim + rot_dim)] in storage type -> qa[t, h, rank .. rank + rot_dim) fp32, rotated
constexpr int TURNS = 256;
// One workgroup per token: its cosines and sines once in LDS where a thread has more than one rotated number (per head and number
// they were most of the kernel), the numbers in front in fours where rows split into them (`quads`).  53 us for 11013 tokens of 16
// heads of 96 + 32 then, 38 now (135 MB).  With one number per thread the table and its barrier only cost: 16384 tokens of 4 such
// heads 21.2 us with it, 18.7 without.
template <typename T, typename TO>
__global__ __launch_bounds__(256) void latent_q_rope_kernel(const T* __restrict__ q, int64_t q_rs,
                                                            const int64_t* __restrict__ positions,
                                                            const float* __restrict__ inv_freq, float mscale,
                                                            TO* __restrict__ qa, int H, int dim, int rot_dim,
                                                            int rot_dims, int rank, int interleaved, int copy_front,
                                                            float factor, int quads) {
  __shared__ float2 turn[TURNS];
  const int64_t t = blockIdx.x;
  const float pos = (float)positions[t];
  const int half = rot_dims / 2;
  auto angle = [&](int i) {
    const float a = pos * inv_freq[i];
    return make_float2(cosf(a) * mscale, sinf(a) * mscale);
  };
  const bool table = H * rot_dim > (int)blockDim.x;
  if (table)
    for (int i = threadIdx.x; i < min(half, TURNS); i += blockDim.x) turn[i] = angle(i);
  if (copy_front && quads) {          // the unrotated numbers in front of the rotated ones (rank == dim): a whole query row
    const int per = dim / 4;
    for (int idx = threadIdx.x; idx < H * per; idx += blockDim.x) {
      const int h = idx / per, j = 4 * (idx % per);
      f32x4 v = Pack4<T>::widen(*reinterpret_cast<const typename Pack4<T>::type*>(q + t * q_rs + (int64_t)h * (dim + rot_dim) + j));
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] *= factor;
      *reinterpret_cast<typename Pack4<TO>::type*>(qa + (t * H + h) * (rank + rot_dim) + j) = Pack4<TO>::narrow(v);
    }
  } else if (copy_front) {
    for (int idx = threadIdx.x; idx < H * dim; idx += blockDim.x) {
      const int h = idx / dim, j = idx % dim;
      st_f32<TO>(qa + (t * H + h) * (rank + rot_dim) + j, ld_f32<T>(q + t * q_rs + (int64_t)h * (dim + rot_dim) + j) * factor);
    }
  }
  if (table) __syncthreads();
  for (int idx = threadIdx.x; idx < H * rot_dim; idx += blockDim.x) {
    const int h = idx / rot_dim, j = idx % rot_dim;
    const T* src = q + t * q_rs + (int64_t)h * (dim + rot_dim) + dim;
    float v = ld_f32<T>(src + j);
    if (j < rot_dims) {
      const bool first = interleaved ? (j & 1) == 0 : j < half;
      const int i = interleaved ? j >> 1 : (first ? j : j - half);
      const float2 a = table && i < TURNS ? turn[i] : angle(i);
      const float other = ld_f32<T>(src + (interleaved ? j ^ 1 : (first ? j + half : j - half)));
      v = first ? v * a.x - other * a.y : v * a.x + other * a.y;
    }
    st_f32<TO>(qa + (t * H + h) * (rank + rot_dim) + rank + j, v * factor);
  }
}

// Both norms, a wavefront to a row of fours of at most 1024 numbers.  In latent_norms_kernel rows of less than 1024 leave wavefronts idle that
// wait at two barriers all the same: 11013 tokens of 768 and 512 + 32 numbers, bf16, 26.3 us there, 17.5 here (5.0 TB/s), of 256 and 128 + 32
// 22.4 and 8.7, 1024 tokens 4.2 and 3.8, 8 tokens 3.4 and 3.3.
template <typename T>
__global__ __launch_bounds__(256) void latent_norm_rows_kernel(KvRows p, NormRows q, int64_t tokens) {
  typedef typename Pack4<T>::type P;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= tokens) return;
  const int lane = threadIdx.x & 63, n = blockIdx.y ? q.n : p.rank, slot = blockIdx.y ? 0 : p.slots[t];
  if (slot < 0) return;
  const float* x = blockIdx.y ? q.x + t * q.rs : p.kv + t * p.rs;
  const T* w = reinterpret_cast<const T*>(blockIdx.y ? q.w : p.w);
  T* out = blockIdx.y ? reinterpret_cast<T*>(q.out) + t * n : reinterpret_cast<T*>(p.cache) + (int64_t)slot * (n + p.rot_dim);
  f32x4 v[4];
  P f[4];
  float ss;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int j = 4 * (lane + 64 * k);
    v[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (j < n) {
      v[k] = *reinterpret_cast<const f32x4*>(x + j);
      f[k] = *reinterpret_cast<const P*>(w + j);
    }
  }
  // The squares of 256 numbers at a time, as norm_row adds them: the same numbers from either.  wave_sum's pairs without the LDS crossbar,
  // through which four such sums took 0.2 - 0.5 us.
  auto squares = [&](int k) {
    float x = 0.0f, a, b;
#pragma unroll
    for (int r = 0; r < 4; ++r) x += v[k][r] * v[k][r];
    rows_pair32(x, a, b);
    rows_pair16(a + b, a, b);
    x = a + b;
    x += dpp_f32<0x128>(x);          // row_ror 8, 4, 2, 1
    x += dpp_f32<0x124>(x);
    x += dpp_f32<0x122>(x);
    x += dpp_f32<0x121>(x);
    return x;
  };
  ss = squares(0);
  if (n > 256) ss = ss + squares(1) + squares(2) + squares(3);
  const float inv = 1.0f / sqrtf(ss / (float)n + p.eps);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int j = 4 * (lane + 64 * k);
    if (j >= n) continue;
    const f32x4 g = Pack4<T>::widen(f[k]);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[k][r] = v[k][r] * inv * g[r];
    *reinterpret_cast<P*>(out + j) = Pack4<T>::narrow(v[k]);
  }
  if (!blockIdx.y) latent_rot_store<T>(p, t, x, out, lane, 64);
}

// Whole query rows in fours, up to QT tokens to a workgroup: all of their cosines and sines into LDS by as many lanes at once, then four numbers to a
// lane, whose partners of the rotation are four others half a turn on or, interleaved, among them.  Rows, heads and both halves split into fours.
// What bounded one token to a workgroup: a wavefront's cosines ahead of everybody's barrier, single numbers with two divisions each.
// 11013 tokens of 16 heads of 96 + 32, bf16 into bf16, 27.3 us there, 19.8 here (4.6 TB/s), 16384 of 4 heads 17.7 and 11.6, 100 of 16 3.7 and 3.2.
// One token to a workgroup up to 2048 (300 tokens 3.6, 4.0 with two, 5.7 with four; 2000 5.8, 6.2, 7.5), then two (3000 7.6, 7.3, 8.4; 11013 21.8,
// 19.8, 20.1), or four where a row has fours for half of the lanes at most (4 heads, 16384 tokens 16.8, 13.0, 11.6).
constexpr int QT = 4;
template <typename T, typename TO>
__global__ __launch_bounds__(256) void latent_q_rows_kernel(const T* __restrict__ q, int64_t q_rs, const int64_t* __restrict__ positions,
                                                            const float* __restrict__ inv_freq, float mscale, TO* __restrict__ out, int tokens, int per,
                                                            int H, int dim, int rot_dim, int rot_dims, int interleaved, float factor) {
  __shared__ float2 turn[QT * TURNS];
  const int t0 = blockIdx.x * per, n = min(per, tokens - t0), half = rot_dims / 2, row4 = (dim + rot_dim) / 4, step_h = 256 / row4,
            step_r = 256 % row4;
  for (int i = threadIdx.x; i < n * half; i += 256) {
    const int t = i / half;
    const float a = (float)positions[t0 + t] * inv_freq[i - t * half];
    turn[i] = make_float2(cosf(a) * mscale, sinf(a) * mscale);
  }
  __syncthreads();
  for (int t = 0; t < n; ++t) {
    const T* from = q + (int64_t)(t0 + t) * q_rs;
    TO* to = out + (int64_t)(t0 + t) * H * (4 * row4);
    const float2* by = turn + t * half;
    int h = threadIdx.x / row4, r = threadIdx.x % row4;
    for (; h < H; h += step_h, r += step_r) {
      if (r >= row4) {
        r -= row4;
        if (++h >= H) break;
      }
      const int j = 4 * r - dim;           // place in the rotated part
      const T* src = from + h * (4 * row4) + 4 * r;
      f32x4 v = Pack4<T>::widen(*reinterpret_cast<const typename Pack4<T>::type*>(src));
      if (j >= 0 && j < rot_dims) {
        if (interleaved) {
          const float2 a = by[j / 2], b = by[j / 2 + 1];
          v = f32x4{v[0] * a.x - v[1] * a.y, v[1] * a.x + v[0] * a.y, v[2] * b.x - v[3] * b.y, v[3] * b.x + v[2] * b.y};
        } else {
          const bool first = j < half;
          const f32x4 o = Pack4<T>::widen(*reinterpret_cast<const typename Pack4<T>::type*>(first ? src + half : src - half));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float2 a = by[(first ? j : j - half) + e];
            v[e] = first ? v[e] * a.x - o[e] * a.y : v[e] * a.x + o[e] * a.y;
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= factor;
      *reinterpret_cast<typename Pack4<TO>::type*>(to + h * (4 * row4) + 4 * r) = Pack4<TO>::narrow(v);
    }
  }
}

// The cache rows of every request of a step, in order of position, into one buffer: request b's row j goes to row
// cu_k[b] + j (cu_k: starts padded to whole blocks; rows past the request's end are zero).  U: what a lane moves at once, a number or 16 bytes
// (rows that split into them).  What bounded it: a row's request, looked for in one start after the other; now 64 starts at once.
// Pages of 256 and 544 numbers of bf16: 128 requests of 100 tokens (288 numbers) 78 and 8.8 us, 64 of 200 25.6 and 7.3, 8 of 1500 8.3 and 6.3.
template <typename U>
__global__ __launch_bounds__(256) void latent_gather_kernel(const U* __restrict__ cache, const int32_t* __restrict__ tables,
                                                            int table_cols, const int32_t* __restrict__ cu_k,
                                                            const int32_t* __restrict__ cu_q,
                                                            const int32_t* __restrict__ past, int B, int block_size,
                                                            int width, U* __restrict__ out) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= cu_k[B]) return;
  const int lane = threadIdx.x & 63;
  int b = 0;                     // the starts behind the first that are not past the row
  for (int i = 0; i < B - 1; i += 64) {
    const uint64_t m = __ballot(i + lane < B - 1 && row >= cu_k[min(i + lane, B - 2) + 1]);
    b += __popcll(m);
    if (~m != 0) break;
  }
  b = __builtin_amdgcn_readfirstlane(b);
  const int j = (int)(row - cu_k[b]);
  const int len = past[b] + cu_q[b + 1] - cu_q[b];
  U* dst = out + row * width;
  if (j >= len) {
    for (int e = lane; e < width; e += 64) dst[e] = U{};
    return;
  }
  const U* src = cache + ((int64_t)tables[(int64_t)b * table_cols + j / block_size] * block_size + j % block_size) * width;
  for (int e = lane; e < width; e += 64) dst[e] = src[e];
}

// Expanded key/value rows [k: H * (dim + rot_dim) | v: H * vdim] from the up-projections kv [rows, H * dim | H * vdim]
// and the gathered cache rows c [rows, rank + rot_dim]: head h's key is [W_uk[h] c | the shared rotated part].
// U: what one thread moves, a number or 16 bytes (rows and heads split into them; 59 us for 12032 rows of 16 heads of 96 + 32 and
// 128 in single numbers, 29 in 16 bytes: 185 MB)
template <typename U>
__global__ __launch_bounds__(256) void latent_expand_kernel(const U* __restrict__ kv, const U* __restrict__ c,
                                                            U* __restrict__ out, int H, int dim, int rot_dim, int vdim,
                                                            int rank) {
  const int64_t row = blockIdx.x;
  const int dk = dim + rot_dim, kw = H * dk, vw = H * vdim;
  const U* kvr = kv + row * (H * dim + vw);
  const U* rot = c + row * (rank + rot_dim) + rank;
  U* dst = out + row * (kw + vw);
  for (int i = threadIdx.x; i < kw; i += blockDim.x) {
    const int h = i / dk, e = i % dk;
    dst[i] = e < dim ? kvr[h * dim + e] : rot[e - dim];
  }
  for (int i = threadIdx.x; i < vw; i += blockDim.x) dst[kw + i] = kvr[H * dim + i];
}

struct AttnArgs {
  const float* qa;         // [tokens, H, rank + rot_dim]
  const void* cache;       // [rows, rank + rot_dim]
  const int32_t* tables;   // [B, table_cols]
  int table_cols;
  const int32_t* cu_q;     // [B + 1]
  const int32_t* past;     // [B]
  const int32_t* seq_of;   // [tokens] request index of each token
  void* out;               // [tokens, H, rank]
  int H, rank, rot_dim, block_size, window, HC, TK;
  float scale;
};

template <typename T>
__global__ __launch_bounds__(256) void latent_attn_kernel(AttnArgs p) {
  extern __shared__ float lds[];
  const int Dk = p.rank + p.rot_dim, Dp = Dk + 1;
  const int HC = p.HC, TK = p.TK;
  float* sq = lds;                    // [HC][Dk]
  float* skey = sq + HC * Dk;         // [TK][Dp]
  float* sc = skey + TK * Dp;         // [HC][TK]
  float* acc = sc + HC * TK;          // [HC][rank]
  float* sm = acc + HC * p.rank;      // [HC] running maximum
  float* sl = sm + HC;                // [HC] running sum
  float* scorr = sl + HC;             // [HC]
  const int t = blockIdx.y, h0 = blockIdx.x * HC;
  const int nh = min(HC, p.H - h0);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int b = p.seq_of[t];
  const int pos = p.past[b] + (t - p.cu_q[b]);
  const int lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  const int32_t* table = p.tables + (int64_t)b * p.table_cols;
  const T* cache = reinterpret_cast<const T*>(p.cache);

  for (int i = tid; i < nh * Dk; i += 256) sq[i] = p.qa[((int64_t)t * p.H + h0) * Dk + i];
  for (int i = tid; i < nh * p.rank; i += 256) acc[i] = 0.0f;
  if (tid < nh) {
    sm[tid] = -INFINITY;
    sl[tid] = 0.0f;
  }
  __syncthreads();
  for (int j0 = lo; j0 <= pos; j0 += TK) {
    const int nk = min(TK, pos + 1 - j0);
    for (int i = tid; i < nk * Dk; i += 256) {
      const int j = i / Dk, e = i % Dk;
      const int kp = j0 + j;
      const int64_t row = (int64_t)table[kp / p.block_size] * p.block_size + kp % p.block_size;
      skey[j * Dp + e] = ld_f32<T>(cache + row * Dk + e);
    }
    __syncthreads();
    for (int i = tid; i < nh * TK; i += 256) {
      const int h = i / TK, j = i % TK;
      float s = -INFINITY;
      if (j < nk) {
        s = 0.0f;
        const float* qv = sq + h * Dk;
        const float* kv = skey + j * Dp;
        for (int e = 0; e < Dk; ++e) s += qv[e] * kv[e];
        s *= p.scale;
      }
      sc[h * TK + j] = s;
    }
    __syncthreads();
    for (int h = wv; h < nh; h += 4) {
      float m = -INFINITY;
      for (int j = lane; j < TK; j += 64) m = fmaxf(m, sc[h * TK + j]);
      m = wave_max(m);
      const float m_old = sm[h];
      const float m_new = fmaxf(m_old, m);
      float sum = 0.0f;
      for (int j = lane; j < TK; j += 64) {
        const float e = (j < nk) ? expf(sc[h * TK + j] - m_new) : 0.0f;
        sc[h * TK + j] = e;
        sum += e;
      }
      sum = wave_sum(sum);
      if (lane == 0) {
        const float corr = expf(m_old - m_new);   // exp(-inf) = 0 at the first tile
        scorr[h] = corr;
        sm[h] = m_new;
        sl[h] = sl[h] * corr + sum;
      }
    }
    __syncthreads();
    for (int i = tid; i < nh * p.rank; i += 256) {
      const int h = i / p.rank, e = i % p.rank;
      float a = acc[i] * scorr[h];
      const float* pv = sc + h * TK;
      for (int j = 0; j < nk; ++j) a += pv[j] * skey[j * Dp + e];
      acc[i] = a;
    }
    __syncthreads();
  }
  T* out = reinterpret_cast<T*>(p.out);
  for (int i = tid; i < nh * p.rank; i += 256) {
    const int h = i / p.rank;
    st_f32<T>(out + ((int64_t)t * p.H + h0) * p.rank + i, acc[i] / sl[h]);
  }
}


// ---- the same attention on the matrix cores (bf16 cache) ----
// A workgroup owns 16 query rows: TQ consecutive tokens of one request times HQ heads (HQ * TQ = 16), which all read
// the same key rows.  Per tile of 64 keys: the rows are staged in LDS twice (row-major for S = Q K^T, transposed for
// O += P V), wavefront w computes the scores of keys 16 w .. 16 w + 15, the softmax statistics are updated by
// 16 threads per row, and every wavefront accumulates its share of the output columns.  Scores, maxima, sums and the
// rescaling are fp32.  Queries and softmax weights enter the MFMAs as the sum of two bf16 numbers (value = hi + lo,
// two MFMAs), so neither is rounded to 8 bits of mantissa; the cached rows are bf16 as stored.
// KEYS rows per tile: 64, or 32 where 64 would not fit the LDS beside wide latents (then two wavefronts compute scores)

struct MfmaAttnArgs {
  AttnArgs a;
  int B, HQ, TQ, Dkp;
  int ksplit;              // workgroups that share a tile's keys (blockIdx.z), each walking every ksplit-th key tile;
  float* partial;          // > 1: their unnormalised shares go to [tokens, H, ksplit, rank + 2] (then maximum and sum)
};

template <int NTILE, int KEYS>
__global__ __launch_bounds__(256) void latent_attn_mfma_kernel(MfmaAttnArgs q) {
  constexpr int ATT_KEYS = KEYS, ATT_PST = KEYS + 8, ATT_SST = KEYS + 4, KPT = KEYS / 16;
  extern __shared__ u32x4 lds_raw[];
  const AttnArgs& p = q.a;
  const int Dk = p.rank + p.rot_dim, R = p.rank, Dq = q.Dkp + 8;
  bf16_t* sQhi = reinterpret_cast<bf16_t*>(lds_raw);
  bf16_t* sQlo = sQhi + 16 * Dq;
  bf16_t* sK = sQlo + 16 * Dq;
  bf16_t* sVt = sK + ATT_KEYS * Dq;
  bf16_t* sPhi = sVt + R * ATT_PST;
  bf16_t* sPlo = sPhi + 16 * ATT_PST;
  float* sS = reinterpret_cast<float*>(sPlo + 16 * ATT_PST);
  float* sm = sS + 2 * 16 * ATT_SST;      // two score tiles: the second holds the other feature half (32-key tiles)
  float* sl = sm + 16;
  float* scorr = sl + 16;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c = lane & 15, g = lane >> 4;

  // which request and which of its tokens this tile covers
  int b = 0, before = 0, tstart = 0, tcount = 0;
  for (; b < q.B; ++b) {
    const int len = p.cu_q[b + 1] - p.cu_q[b];
    const int tiles = (len + q.TQ - 1) / q.TQ;
    if ((int)blockIdx.y < before + tiles) {
      tstart = p.cu_q[b] + ((int)blockIdx.y - before) * q.TQ;
      tcount = min(q.TQ, p.cu_q[b + 1] - tstart);
      break;
    }
    before += tiles;
  }
  if (b == q.B) return;
  const int h0 = blockIdx.x * q.HQ;
  const int pos0 = p.past[b] + (tstart - p.cu_q[b]);
  const int kmax = pos0 + tcount - 1;
  const int kmin = p.window > 0 ? max(0, pos0 - p.window + 1) : 0;
  const int32_t* table = p.tables + (int64_t)b * p.table_cols;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(p.cache);

  for (int i = tid; i < ATT_KEYS * Dq; i += 256) sK[i] = (bf16_t)0.0f;       // the padding columns stay zero
  for (int i = tid; i < 16 * Dq; i += 256) {
    const int r = i / Dq, f = i % Dq;
    const int tq = r / q.HQ, hh = h0 + r % q.HQ;
    float v = 0.0f;
    if (tq < tcount && hh < p.H && f < Dk) v = p.qa[((int64_t)(tstart + tq) * p.H + hh) * Dk + f];
    const bf16_t hi = (bf16_t)v;
    sQhi[i] = hi;
    sQlo[i] = (bf16_t)(v - (float)hi);
  }
  if (tid < 16) {
    sm[tid] = -INFINITY;
    sl[tid] = 0.0f;
  }
  f32x4 O[NTILE];
#pragma unroll
  for (int n = 0; n < NTILE; ++n) O[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the row this thread serves in the softmax step
  const int srow = tid >> 4, skq = tid & 15;
  const int s_tq = srow / q.HQ, s_hh = h0 + srow % q.HQ;
  const bool s_valid = s_tq < tcount && s_hh < p.H;
  const int s_pos = pos0 + s_tq;
  const int s_lo = p.window > 0 ? max(0, s_pos - p.window + 1) : 0;
  const int chunks = Dk / 8;
  __syncthreads();

  // Key rows travel memory -> registers -> LDS; the loads of the NEXT tile are issued before this tile is multiplied,
  // so their latency hides behind the MFMAs.  Consecutive threads take consecutive keys (conflict-free transposed
  // stores).  NCH bounds the 16-byte pieces per thread and tile (the launcher checks it).
  constexpr int NCH = 10;
  const int pieces = ATT_KEYS * chunks;
  u32x4 stage[NCH];
  auto fetch_tile = [&](int j0) {
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int i = tid + u * 256;
      const int key = i % ATT_KEYS, f8 = i / ATT_KEYS;
      const int kp = j0 + key;
      stage[u] = u32x4{0u, 0u, 0u, 0u};
      if (i < pieces && kp <= kmax) {
        const int64_t row = (int64_t)table[kp / p.block_size] * p.block_size + kp % p.block_size;
        stage[u] = *reinterpret_cast<const u32x4*>(cache + row * Dk + f8 * 8);
      }
    }
  };
  const int kstep = q.ksplit * ATT_KEYS;
  fetch_tile(kmin + (int)blockIdx.z * ATT_KEYS);
  for (int j0 = kmin + (int)blockIdx.z * ATT_KEYS; j0 <= kmax; j0 += kstep) {
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int i = tid + u * 256;
      const int key = i % ATT_KEYS, f8 = i / ATT_KEYS;
      if (i >= pieces) continue;
      *reinterpret_cast<u32x4*>(sK + key * Dq + f8 * 8) = stage[u];
      if (f8 * 8 < R) {
        const uint16_t* e16 = reinterpret_cast<const uint16_t*>(&stage[u]);
        uint16_t* dst = reinterpret_cast<uint16_t*>(sVt) + (f8 * 8) * ATT_PST + key;
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e * ATT_PST] = e16[e];
      }
    }
    __syncthreads();
    if (j0 + kstep <= kmax) fetch_tile(j0 + kstep);
    // S = Q K^T: with 64 keys wavefront w takes keys 16 w ..; with 32 keys the wavefront pairs (0, 1) and (2, 3) take
    // the two halves of the feature dimension and their partial scores are summed in the softmax step
    {
      constexpr int KW = ATT_KEYS / 16;             // wavefronts one pass over the keys needs
      constexpr int PARTS = 4 / KW;                 // feature ranges (1 or 2)
      const int kw = wv % KW, part = wv / KW;
      const int steps = q.Dkp / 32;
      const int f_lo = (steps * part) / PARTS * 32, f_hi = (steps * (part + 1)) / PARTS * 32;
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      const bf16_t* krow = sK + (16 * kw + c) * Dq + 8 * g;
      const bf16_t* qhi = sQhi + c * Dq + 8 * g;
      const bf16_t* qlo = sQlo + c * Dq + 8 * g;
      for (int ks = f_lo; ks < f_hi; ks += 32) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(krow + ks);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(qhi + ks), kf, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(qlo + ks), kf, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) sS[part * 16 * ATT_SST + (4 * g + r) * ATT_SST + 16 * kw + c] = acc[r] * p.scale;
    }
    __syncthreads();
    // softmax statistics: 16 threads per row, KEYS / 16 keys each
    {
      float sv[KPT], m = -INFINITY;
#pragma unroll
      for (int e = 0; e < KPT; ++e) {
        const int kp = j0 + KPT * skq + e;
        const bool ok = s_valid && kp >= s_lo && kp <= s_pos;
        sv[e] = -INFINITY;
        if (ok) {
          sv[e] = sS[srow * ATT_SST + KPT * skq + e];
          if constexpr (ATT_KEYS == 32) sv[e] += sS[16 * ATT_SST + srow * ATT_SST + KPT * skq + e];
        }
        m = fmaxf(m, sv[e]);
      }
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
      const float m_old = sm[srow];
      const float m_new = fmaxf(m_old, m);
      float sum = 0.0f;
#pragma unroll
      for (int e = 0; e < KPT; ++e) {
        const float pe = (sv[e] == -INFINITY) ? 0.0f : expf(sv[e] - m_new);
        sum += pe;
        const bf16_t hi = (bf16_t)pe;
        sPhi[srow * ATT_PST + KPT * skq + e] = hi;
        sPlo[srow * ATT_PST + KPT * skq + e] = (bf16_t)(pe - (float)hi);
      }
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      if (skq == 0) {
        const float corr = (m_new == -INFINITY) ? 1.0f : expf(m_old - m_new);
        scorr[srow] = corr;
        sm[srow] = m_new;
        sl[srow] = sl[srow] * corr + sum;
      }
    }
    __syncthreads();
    // O = O * corr + P V for this wavefront's output columns
#pragma unroll
    for (int n = 0; n < NTILE; ++n) {
      const int col0 = 16 * (wv * NTILE + n);
      if (col0 < R) {
#pragma unroll
        for (int r = 0; r < 4; ++r) O[n][r] *= scorr[4 * g + r];
#pragma unroll
        for (int ks = 0; ks < ATT_KEYS; ks += 32) {
          const bf16x8 vf = *reinterpret_cast<const bf16x8*>(sVt + (col0 + c) * ATT_PST + ks + 8 * g);
          O[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              *reinterpret_cast<const bf16x8*>(sPhi + c * ATT_PST + ks + 8 * g), vf, O[n], 0, 0, 0);
          O[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              *reinterpret_cast<const bf16x8*>(sPlo + c * ATT_PST + ks + 8 * g), vf, O[n], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  bf16_t* out = reinterpret_cast<bf16_t*>(p.out);
  if (q.ksplit > 1) {          // another launch joins the shares
    const int PW = R + 2;
#pragma unroll
    for (int n = 0; n < NTILE; ++n) {
      const int col = 16 * (wv * NTILE + n) + c;
      if (col >= R) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * g + r;
        const int tq = row / q.HQ, hh = h0 + row % q.HQ;
        if (tq < tcount && hh < p.H)
          q.partial[(((int64_t)(tstart + tq) * p.H + hh) * q.ksplit + blockIdx.z) * PW + col] = O[n][r];
      }
    }
    if (tid < 16) {
      const int tq = tid / q.HQ, hh = h0 + tid % q.HQ;
      if (tq < tcount && hh < p.H) {
        float* dst = q.partial + (((int64_t)(tstart + tq) * p.H + hh) * q.ksplit + blockIdx.z) * PW + R;
        dst[0] = sm[tid];
        dst[1] = sl[tid];
      }
    }
    return;
  }
#pragma unroll
  for (int n = 0; n < NTILE; ++n) {
    const int col = 16 * (wv * NTILE + n) + c;
    if (col >= R) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * g + r;
      const int tq = row / q.HQ, hh = h0 + row % q.HQ;
      if (tq < tcount && hh < p.H) out[((int64_t)(tstart + tq) * p.H + hh) * R + col] = (bf16_t)(O[n][r] / sl[row]);
    }
  }
}

// joins the shares of the ksplit (at most 32) workgroups that walked one (token, head)'s keys: one workgroup per row,
// the shares' weights exp(m_z - m) / l first, then every thread sums its columns over the shares
__global__ __launch_bounds__(256) void latent_attn_join_kernel(const float* __restrict__ partial, bf16_t* __restrict__ out,
                                                               int ksplit, int R) {
  __shared__ float wz[32];
  const int64_t row = blockIdx.x;
  const int PW = R + 2;
  const float* src = partial + row * ksplit * PW;
  if (threadIdx.x < 64) {
    const int z = threadIdx.x;
    const float mz = z < ksplit ? src[z * PW + R] : -INFINITY;
    const float lz = z < ksplit ? src[z * PW + R + 1] : 0.0f;
    const float m = wave_max(mz);
    const float f = mz == -INFINITY ? 0.0f : __expf(mz - m);
    const float l = wave_sum(lz * f);
    if (z < 32) wz[z] = f / l;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < R; e += 256) {
    float o = 0.0f;
#pragma unroll 8
    for (int z = 0; z < ksplit; ++z) o += src[z * PW + e] * wz[z];
    out[row * R + e] = (bf16_t)o;
  }
}

template <int NTILE, int KEYS>
hipError_t launch_mfma_attn(const MfmaAttnArgs& q, dim3 grid, size_t lds, hipStream_t s) {
  static size_t allowed = 64 * 1024;
  if (lds > allowed) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attn_mfma_kernel<NTILE, KEYS>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    allowed = lds;
  }
  latent_attn_mfma_kernel<NTILE, KEYS><<<grid, dim3(256), lds, s>>>(q);
  return hipSuccess;
}

#include "latent_token.h"

}  // namespace

extern "C" int nv_latent_kv_store(const float* kv, int64_t kv_row_stride, const void* norm_w, const int64_t* positions,
                                  const float* inv_freq, float mscale, const int32_t* slot_mapping, void* cache,
                                  int64_t tokens, int rank, int rot_dim, int rot_dims, int interleaved, float eps,
                                  int dtype, nv_stream_t stream) {
  return nv_latent_norms(kv, kv_row_stride, norm_w, positions, inv_freq, mscale, slot_mapping, cache, tokens, rank, rot_dim, rot_dims,
                         interleaved, nullptr, 0, nullptr, nullptr, 0, eps, dtype, stream);
}

extern "C" int nv_latent_norms(const float* kv, int64_t kv_row_stride, const void* norm_w, const int64_t* positions,
                               const float* inv_freq, float mscale, const int32_t* slot_mapping, void* cache, int64_t tokens,
                               int rank, int rot_dim, int rot_dims, int interleaved, const float* q, int64_t q_row_stride,
                               const void* q_norm_w, void* q_out, int q_rank, float eps, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG(kv && norm_w && positions && inv_freq && slot_mapping && cache, "nv_latent_kv_store: null pointer");
  NV_CHECK_ARG(!q || (q_norm_w && q_out && q_rank > 0), "nv_latent_norms: null pointer");
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F32, "nv_latent_kv_store: bad dtype %d", dtype);
  NV_CHECK_ARG(tokens >= 0 && rank > 0 && rot_dim >= 0 && rot_dims >= 0 && rot_dims <= rot_dim && rot_dims % 2 == 0,
               "nv_latent_kv_store: bad shape rank=%d rot_dim=%d rot_dims=%d", rank, rot_dim, rot_dims);
  if (tokens == 0) return NV_OK;
  auto quads = [](const float* x, int64_t rs, const void* w, const void* out, int n, int out_row) {
    return n <= 4096 && n % 4 == 0 && rs % 4 == 0 && out_row % 4 == 0 && ((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) % 16 == 0;
  };
  const NormRows rows{q, q_row_stride, q_norm_w, q_out, q_rank, q ? quads(q, q_row_stride, q_norm_w, q_out, q_rank, q_rank) : 0};
  const int kv_quads = quads(kv, kv_row_stride, norm_w, cache, rank, rank + rot_dim);
  const KvRows p{kv, kv_row_stride, norm_w, positions, inv_freq, mscale, slot_mapping, cache, rank, rot_dim, rot_dims, eps, interleaved};
  const dim3 grid((unsigned)tokens, q ? 2 : 1);
  hipStream_t s = (hipStream_t)stream;
  // alone, fours pay from 512 numbers on (16000 tokens of 64: 16.7 us in fours, 13.9 one at a time; of 512: 21.1 and 25.4)
  if (q && kv_quads && rows.quads && rank <= 1024 && q_rank <= 1024)
    NV_DISPATCH_T(dtype, latent_norm_rows_kernel<T><<<dim3((unsigned)((tokens + 3) / 4), 2), dim3(256), 0, s>>>(p, rows, tokens));
  else if (q) NV_DISPATCH_T(dtype, latent_norms_kernel<T><<<grid, dim3(256), 0, s>>>(p, kv_quads, rows));
  else if (kv_quads && rank >= 512) NV_DISPATCH_T(dtype, latent_kv_store_kernel<T, true><<<grid, dim3(256), 0, s>>>(p));
  else NV_DISPATCH_T(dtype, latent_kv_store_kernel<T, false><<<grid, dim3(256), 0, s>>>(p));
  NV_CHECK_LAUNCH();
  return NV_OK;
}

extern "C" int nv_latent_q_rope(const void* q, int64_t q_row_stride, const int64_t* positions, const float* inv_freq,
                                float mscale, float* qa, int64_t tokens, int heads, int dim, int rot_dim, int rot_dims,
                                int interleaved, int rank, int dtype, nv_stream_t stream) {
  return nv_latent_q_rows(q, q_row_stride, positions, inv_freq, mscale, qa, tokens, heads, dim, rot_dim, rot_dims,
                          interleaved, rank, 0, 1.0f, dtype, stream);
}

extern "C" int nv_latent_q_rows(const void* q, int64_t q_row_stride, const int64_t* positions, const float* inv_freq,
                                float mscale, float* qa, int64_t tokens, int heads, int dim, int rot_dim, int rot_dims,
                                int interleaved, int rank, int copy_front, float factor, int dtype, nv_stream_t stream) {
  return nv_latent_q_rows_as(q, q_row_stride, positions, inv_freq, mscale, qa, NV_F32, tokens, heads, dim, rot_dim, rot_dims, interleaved,
                             rank, copy_front, factor, dtype, stream);
}

extern "C" int nv_latent_q_rows_as(const void* q, int64_t q_row_stride, const int64_t* positions, const float* inv_freq,
                                   float mscale, void* qa, int qa_dtype, int64_t tokens, int heads, int dim, int rot_dim, int rot_dims,
                                   int interleaved, int rank, int copy_front, float factor, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG(qa_dtype == NV_F32 || qa_dtype == NV_BF16, "nv_latent_q_rope: bad dtype %d of the rows", qa_dtype);
  NV_CHECK_ARG(!copy_front || rank == dim, "nv_latent_q_rows: whole query rows have the unrotated numbers in front");
  NV_CHECK_ARG(q && positions && inv_freq && qa, "nv_latent_q_rope: null pointer");
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F32, "nv_latent_q_rope: bad dtype %d", dtype);
  NV_CHECK_ARG(tokens >= 0 && heads > 0 && dim >= 0 && rot_dim >= 0 && rot_dims <= rot_dim && rot_dims % 2 == 0 && rank > 0,
               "nv_latent_q_rope: bad shape");
  if (tokens == 0 || (rot_dim == 0 && !copy_front)) return NV_OK;
  const int quads = dim % 4 == 0 && rot_dim % 4 == 0 && q_row_stride % 4 == 0 && (uintptr_t)qa % 16 == 0 &&
                    (uintptr_t)q % (dtype == NV_BF16 ? 8 : 16) == 0;
  // Whole rows whose rotation is in fours as well.  Over 100 to 8000 tokens of 2 to 32 heads 141 shapes with 32 and 64 rotated numbers take 0.91 and
  // 0.80 of the time of one token to a workgroup (three 3 to 7 % more, 0.3 us at most: 400 tokens of 8 heads of 128 + 32).  Where there is
  // less to share: 16 rotated numbers 1.04 at 400 tokens, 1.00 at 1000, 0.95 at 2000, none 1.02 to 1.05 up to 3000 tokens and 0.95 at 8000.
  const bool shared = rot_dims >= 32 || tokens > (rot_dims > 0 ? 1024 : 4096);
  if (quads && copy_front && shared && rot_dims % (interleaved ? 4 : 8) == 0 && rot_dims <= 2 * TURNS && tokens < (1 << 30)) {
    const int per = tokens <= 2048 ? 1 : heads * (dim + rot_dim) <= 512 ? QT : 2;
    const dim3 g((unsigned)((tokens + per - 1) / per));
    if (qa_dtype == NV_F32)
      NV_DISPATCH_T(dtype, latent_q_rows_kernel<T, float><<<g, dim3(256), 0, (hipStream_t)stream>>>(
                               (const T*)q, q_row_stride, positions, inv_freq, mscale, (float*)qa, (int)tokens, per, heads, dim, rot_dim, rot_dims,
                               interleaved, factor));
    else
      NV_DISPATCH_T(dtype, latent_q_rows_kernel<T, bf16_t><<<g, dim3(256), 0, (hipStream_t)stream>>>(
                               (const T*)q, q_row_stride, positions, inv_freq, mscale, (bf16_t*)qa, (int)tokens, per, heads, dim, rot_dim, rot_dims,
                               interleaved, factor));
    NV_CHECK_LAUNCH();
    return NV_OK;
  }
  if (qa_dtype == NV_F32)
    NV_DISPATCH_T(dtype, latent_q_rope_kernel<T, float><<<dim3((unsigned)tokens), dim3(256), 0, (hipStream_t)stream>>>(
                             (const T*)q, q_row_stride, positions, inv_freq, mscale, (float*)qa, heads, dim, rot_dim, rot_dims, rank,
                             interleaved, copy_front, factor, quads));
  else
    NV_DISPATCH_T(dtype, latent_q_rope_kernel<T, bf16_t><<<dim3((unsigned)tokens), dim3(256), 0, (hipStream_t)stream>>>(
                             (const T*)q, q_row_stride, positions, inv_freq, mscale, (bf16_t*)qa, heads, dim, rot_dim, rot_dims, rank,
                             interleaved, copy_front, factor, quads));
  NV_CHECK_LAUNCH();
  return NV_OK;
}

// Workgroups that share one decoded token's keys: enough to put up to 512 workgroups on the chip, at most 32.  A
// function of the launch shape alone (not of the contexts), so a captured launch stays valid as contexts grow.
static int latent_attn_key_splits(int64_t tokens, int heads) {
  const int64_t groups = tokens * ((heads + 15) / 16);
  int k = 1;
  while (k < 32 && groups * k * 2 <= 512) k *= 2;
  return k;
}

extern "C" size_t nv_latent_attn_workspace_bytes(int64_t tokens, int max_q, int heads, int rank) {
  if (max_q != 1 || tokens <= 0) return 0;
  const int k = latent_attn_key_splits(tokens, heads);
  return k > 1 ? (size_t)tokens * heads * k * (rank + 2) * sizeof(float) : 0;
}

extern "C" int nv_latent_attn(const float* qa, const void* cache, const int32_t* block_tables, int table_cols,
                              const int32_t* cu_q, const int32_t* past_lens, const int32_t* seq_of_token, void* out,
                              int64_t tokens, int num_seqs, int heads, int rank, int rot_dim, int block_size, int window, float scale,
                              int dtype, nv_stream_t stream) {
  return nv_latent_attn_split(qa, cache, block_tables, table_cols, cu_q, past_lens, seq_of_token, out, tokens, num_seqs,
                              heads, rank, rot_dim, block_size, window, scale, 0, nullptr, 0, dtype, stream);
}

extern "C" int nv_latent_attn_split(const float* qa, const void* cache, const int32_t* block_tables, int table_cols,
                                    const int32_t* cu_q, const int32_t* past_lens, const int32_t* seq_of_token, void* out,
                                    int64_t tokens, int num_seqs, int heads, int rank, int rot_dim, int block_size,
                                    int window, float scale, int max_q, void* workspace, size_t workspace_bytes, int dtype,
                                    nv_stream_t stream) {
  NV_CHECK_ARG(qa && cache && block_tables && cu_q && past_lens && seq_of_token && out, "nv_latent_attn: null pointer");
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F32, "nv_latent_attn: bad dtype %d", dtype);
  NV_CHECK_ARG(tokens >= 0 && tokens <= 65535 * 1024 && heads > 0 && rank > 0 && rot_dim >= 0 && block_size > 0 && table_cols > 0,
               "nv_latent_attn: bad shape");
  if (tokens == 0) return NV_OK;
  NV_CHECK_ARG(tokens <= 65535, "nv_latent_attn: %lld tokens exceed one launch", (long long)tokens);
  const int Dk = rank + rot_dim;
  // bf16 caches whose rows split into 16-byte pieces go to the matrix cores
  if (dtype == NV_BF16 && Dk % 8 == 0 && rank % 16 == 0 && rank <= 512 && num_seqs > 0) {
    int HQ = 1;
    while (HQ < heads && HQ < 16) HQ *= 2;
    MfmaAttnArgs q{{qa, cache, block_tables, table_cols, cu_q, past_lens, seq_of_token, out, heads, rank, rot_dim,
                    block_size, window, 0, 0, scale},
                   num_seqs, HQ, 16 / HQ, ((Dk + 31) / 32) * 32, 1, reinterpret_cast<float*>(workspace)};
    // one token per request: several workgroups share its keys, when the caller brought room for their shares
    if (max_q == 1 && workspace) {
      const int k = latent_attn_key_splits(tokens, heads);
      if (k > 1 && workspace_bytes >= (size_t)tokens * heads * k * (rank + 2) * sizeof(float)) q.ksplit = k;
    }
    // single tokens whose rows split into 64-byte units: every wavefront on its own tiles of 32 keys.  Sixteen workgroups per
    // token put 2048 keys under way at once; more of them only lengthen the join where contexts are that long, and longer ones are
    // still shorter than in tiles over 32 workgroups (one token of 16 heads over 32768 rows of 512 + 32: 87 and 215 us).
    if (max_q == 1 && Dk % 32 == 0 && Dk <= 544 && (uintptr_t)cache % 16 == 0 && (uintptr_t)qa % 16 == 0 && (uintptr_t)out % 8 == 0) {
      if (q.ksplit > 16) q.ksplit = 16;
      const hipError_t e = Dk <= 160   ? launch_latent_token<5>(q, tokens, (hipStream_t)stream)
                           : Dk <= 288 ? launch_latent_token<9>(q, tokens, (hipStream_t)stream)
                                       : launch_latent_token<17>(q, tokens, (hipStream_t)stream);
      if (e != hipSuccess) {
        nv_set_error("nv_latent_attn: %s", hipGetErrorString(e));
        return NV_ERR_LAUNCH;
      }
      if (q.ksplit > 1) {
        latent_attn_join_kernel<<<dim3((unsigned)(tokens * heads)), dim3(256), 0, (hipStream_t)stream>>>(
            q.partial, reinterpret_cast<bf16_t*>(out), q.ksplit, rank);
        NV_CHECK_LAUNCH();
      }
      return NV_OK;
    }
    const int Dq = q.Dkp + 8;
    auto lds_for = [&](int keys) {
      return (size_t)(2 * 16 * Dq + keys * Dq + rank * (keys + 8) + 2 * 16 * (keys + 8)) * 2 + (size_t)(2 * 16 * (keys + 4) + 48) * 4;
    };
    const int keys = lds_for(64) <= 150 * 1024 ? 64 : 32;
    const size_t lds = lds_for(keys);
    if (lds <= 150 * 1024 && keys * (Dk / 8) <= 10 * 256) {
      const int64_t tiles = tokens / q.TQ + num_seqs;        // at most: every request may end in a partial tile
      NV_CHECK_ARG(tiles <= 65535, "nv_latent_attn: %lld tiles exceed one launch", (long long)tiles);
      dim3 grid((unsigned)((heads + HQ - 1) / HQ), (unsigned)tiles, (unsigned)q.ksplit);
      const int ntile = (rank / 16 + 3) / 4;
      hipStream_t st = (hipStream_t)stream;
      hipError_t e;
      if (keys == 64)
        e = ntile <= 2 ? launch_mfma_attn<2, 64>(q, grid, lds, st) : ntile <= 4 ? launch_mfma_attn<4, 64>(q, grid, lds, st)
                                                                                 : launch_mfma_attn<8, 64>(q, grid, lds, st);
      else
        e = launch_mfma_attn<8, 32>(q, grid, lds, st);
      if (e != hipSuccess) {
        nv_set_error("nv_latent_attn: %s", hipGetErrorString(e));
        return NV_ERR_LAUNCH;
      }
      NV_CHECK_LAUNCH();
      if (q.ksplit > 1) {
        const int64_t rows = tokens * heads;
        latent_attn_join_kernel<<<dim3((unsigned)rows), dim3(256), 0, st>>>(q.partial, reinterpret_cast<bf16_t*>(out),
                                                                            q.ksplit, rank);
        NV_CHECK_LAUNCH();
      }
      return NV_OK;
    }
  }
  // LDS plan: as many heads per workgroup as fit beside a key tile of 64 (then 32, 16, 8) rows
  const size_t budget = 64 * 1024;
  int TK = 64, HC = heads;
  auto need = [&](int hc, int tk) {
    return (size_t)(hc * Dk + tk * (Dk + 1) + hc * tk + hc * rank + 3 * hc) * sizeof(float);
  };
  while (TK > 8 && need(1, TK) > budget) TK /= 2;
  NV_CHECK_ARG(need(1, TK) <= budget, "nv_latent_attn: rows of %d numbers do not fit the LDS plan", Dk);
  while (HC > 1 && need(HC, TK) > budget) HC = (HC + 1) / 2;
  AttnArgs p{qa, cache, block_tables, table_cols, cu_q, past_lens, seq_of_token, out, heads, rank, rot_dim, block_size,
             window, HC, TK, scale};
  dim3 grid((unsigned)((heads + HC - 1) / HC), (unsigned)tokens);
  NV_DISPATCH_T(dtype, latent_attn_kernel<T><<<grid, dim3(256), need(HC, TK), (hipStream_t)stream>>>(p));
  NV_CHECK_LAUNCH();
  return NV_OK;
}

extern "C" int nv_latent_gather(const void* cache, const int32_t* block_tables, int table_cols, const int32_t* cu_k,
                                const int32_t* cu_q, const int32_t* past_lens, int num_seqs, int block_size, int row_width,
                                void* out, int64_t rows, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG(cache && block_tables && cu_k && cu_q && past_lens && out, "nv_latent_gather: null pointer");
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F32, "nv_latent_gather: bad dtype %d", dtype);
  NV_CHECK_ARG(num_seqs > 0 && block_size > 0 && row_width > 0 && rows >= 0 && table_cols > 0, "nv_latent_gather: bad shape");
  if (rows == 0) return NV_OK;
  const dim3 g((unsigned)((rows + 3) / 4));
  const int bytes = row_width * (dtype == NV_BF16 ? 2 : 4);
  if (bytes % 16 == 0 && ((uintptr_t)cache | (uintptr_t)out) % 16 == 0)
    latent_gather_kernel<u32x4><<<g, dim3(256), 0, (hipStream_t)stream>>>((const u32x4*)cache, block_tables, table_cols, cu_k, cu_q, past_lens,
                                                                          num_seqs, block_size, bytes / 16, (u32x4*)out);
  else
    NV_DISPATCH_T(dtype, latent_gather_kernel<T><<<g, dim3(256), 0, (hipStream_t)stream>>>(
                             (const T*)cache, block_tables, table_cols, cu_k, cu_q, past_lens, num_seqs, block_size,
                             row_width, (T*)out));
  NV_CHECK_LAUNCH();
  return NV_OK;
}

extern "C" int nv_latent_expand(const void* kv, const void* c, void* out, int64_t rows, int heads, int dim, int rot_dim,
                                int vdim, int rank, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG(kv && c && out, "nv_latent_expand: null pointer");
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F32, "nv_latent_expand: bad dtype %d", dtype);
  NV_CHECK_ARG(rows >= 0 && heads > 0 && dim > 0 && rot_dim >= 0 && vdim > 0 && rank > 0, "nv_latent_expand: bad shape");
  if (rows == 0) return NV_OK;
  const int per = dtype == NV_BF16 ? 8 : 4;
  if (dim % per == 0 && rot_dim % per == 0 && vdim % per == 0 && rank % per == 0 &&
      ((uintptr_t)kv | (uintptr_t)c | (uintptr_t)out) % 16 == 0) {
    latent_expand_kernel<u32x4><<<dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream>>>(
        (const u32x4*)kv, (const u32x4*)c, (u32x4*)out, heads, dim / per, rot_dim / per, vdim / per, rank / per);
  } else {
    NV_DISPATCH_T(dtype, latent_expand_kernel<T><<<dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream>>>(
                             (const T*)kv, (const T*)c, (T*)out, heads, dim, rot_dim, vdim, rank));
  }
  NV_CHECK_LAUNCH();
  return NV_OK;
}
