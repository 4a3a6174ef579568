// q/k/v of attention over its own paged rows, for prompts: the projection (and the columns behind it, gates and the like) on the tiles of
// stream_deep.h, rotated, scaled and stored on the way: queries in fp32 or bf16, cache rows [k | v] in bf16, the other columns in fp32.
//
// What bounded these steps: the projection was written in fp32 and read again.  16384 rows 2048 -> 16 + 8 + 8 heads of 128 and 16 gates: the
// product 277 us and qk_pairs_store_kernel 110; here 240, the turns' cosines and sines, once per token, among them (the layer 670 and 516).  The
// arithmetic is that of qk_pairs_store_kernel, over the same product bit for bit.  Which sizes it pays for: kernels.qkv_streams.
#include "anyt.h"
#include "stream_deep.h"

namespace {

struct QkvArgs {
  const uint16_t *x, *w;
  int64_t xs;
  const float* turns;         // [tokens, 2 * half]: cosines, then sines
  const int32_t* slots;
  uint16_t* cache;            // [rows, nkv]
  void* q;                    // [tokens, nq]
  float* rest;                // [tokens, rest_rs]
  int64_t rest_rs;
  int M, N, K, nq, nk, nkv;
  float scale;
  int q16;                    // queries in bf16
};

// HALF16: a head's rotated numbers are 2 * 16 * HALF16, i with i + 16 * HALF16; 0: none
template <int D, int HALF16>
struct QkvJob {
  typedef bf16_t T;
  typedef StreamNatural Order;
  static constexpr bool FAR_A = true, FAR_W = false, UPS = false;
  static constexpr int NSTORE_WAVE = 64, EXTRA = 0;
  QkvArgs p;
  int K, rows, cols;

  __device__ __forceinline__ int count(int) const { return rows * cols; }
  __device__ __forceinline__ StreamTile find(int tile, int) const {
    int m_tile, n_tile;
    stream_order(tile, rows, cols, m_tile, n_tile);
    return StreamTile{m_tile * STREAM_BM, p.M, n_tile * STREAM_BN, 0};
  }
  __device__ __forceinline__ const void* a_base(const StreamTile&) const { return p.x; }
  __device__ __forceinline__ uint32_t a_stride() const { return (uint32_t)p.xs * 2; }
  __device__ __forceinline__ uint32_t a_row(const StreamTile& at, int r) const { return (uint32_t)min(at.lo + r, at.hi - 1); }
  __device__ __forceinline__ const void* w_base(const StreamTile& at) const { return p.w + (int64_t)at.n0 * p.K; }
  __device__ __forceinline__ uint32_t w_stride() const { return (uint32_t)p.K * 2; }
  __device__ __forceinline__ uint32_t w_row(const StreamTile& at, int r) const { return (uint32_t)min(r, p.N - at.n0 - 1); }
  __device__ __forceinline__ uint32_t w_step() const { return 128; }
  // tiles of queries: all their stores are executed whatever the slots say
  __device__ __forceinline__ bool whole(const StreamTile& at) const { return at.lo + STREAM_BM <= at.hi && at.n0 + STREAM_BN <= p.nq; }
  __device__ __forceinline__ void fetch_extra(const StreamTile&, int, int, unsigned char*) const {}

  __device__ __forceinline__ void finish(const StreamTile& at, int wm, int wn, int lane, bool live0, bool live1, const unsigned char*) const {
    const int n0 = at.n0 + 128 * wn, fr = lane & 15, g = lane >> 4;
    if (n0 >= p.N) return;
    const bool turn = HALF16 > 0 && n0 < p.nq + p.nk, stores = n0 + 128 > p.nq && n0 < p.nq + p.nkv;
    auto token = [&](int r) { return at.lo + 128 * (r >> 2) + 64 * wm + 16 * (r & 3) + fr; };
    int slot[8];
    f32x4 cs[2][HALF16 ? 2 * HALF16 : 1];
    auto ask = [&](int r) {      // a row's turns two rows ahead, before the stores of the row between: behind them they would be waited for with them
      if (!turn) return;
      const float* from = p.turns + (int64_t)min(token(r), at.hi - 1) * (32 * HALF16) + 4 * g;
#pragma unroll
      for (int u = 0; u < 2 * HALF16; ++u) cs[r & 1][u] = *reinterpret_cast<const f32x4*>(from + 16 * u);
    };
#pragma unroll
    for (int r = 0; r < 8; ++r) slot[r] = -1;
    if (stores) {
#pragma unroll
      for (int r = 0; r < 8; ++r) slot[r] = p.slots[min(token(r), at.hi - 1)];
    }
    ask(0);
    ask(1);
    if (stores) {
#pragma unroll
      for (int r = 0; r < 8; ++r) asm volatile("" : "+v"(slot[r]));
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      __builtin_amdgcn_sched_barrier(0);
      const int t = token(r);
      f32x4 x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = deep_take(r >> 2, j, r & 3);
      if constexpr (HALF16 > 0) {
        // waited for whichever head uses them: pending, they would be waited for in the loop over blocks
#pragma unroll
        for (int u = 0; u < 2 * HALF16; ++u) asm volatile("" : "+v"(cs[r & 1][u]));
#pragma unroll
        for (int h = 0; h < 128 / D; ++h) {
          if (n0 + D * h >= p.nq + p.nk) continue;
#pragma unroll
          for (int u = 0; u < HALF16; ++u) {
            f32x4 &a = x[h * (D / 16) + u], &b = x[h * (D / 16) + u + HALF16];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float co = cs[r & 1][u][e], si = cs[r & 1][HALF16 + u][e], lo = a[e], hi = b[e];
              a[e] = lo * co - hi * si;
              b[e] = hi * co + lo * si;
            }
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (r + 2 < 8) ask(r + 2);
      __builtin_amdgcn_sched_barrier(0);
      if (t >= at.hi || !(r < 4 ? live0 : live1)) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j) {      // groups of 16 columns belong together: nq, nk and nkv are multiples of 16
        const int n = n0 + 16 * j;
        if (n < p.nq) {
          f32x4 v = x[j];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] *= p.scale;
          const int64_t to = (int64_t)t * p.nq + n + 4 * g;
          if (p.q16) *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.q) + to) = Pack4<bf16_t>::narrow(v);
          else *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.q) + to) = v;
        } else if (n < p.nq + p.nkv) {
          if (slot[r] >= 0)
            *reinterpret_cast<uint2*>(p.cache + (int64_t)slot[r] * p.nkv + (n - p.nq) + 4 * g) = Pack4<bf16_t>::narrow(x[j]);
        } else if (n < p.N) {
          float* to = p.rest + (int64_t)t * p.rest_rs + (n - p.nq - p.nkv) + 4 * g;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + 4 * g + e < p.N) to[e] = x[j][e];
        }
      }
    }
  }
};

// cosines and sines of a token's angles, times `m`: the numbers that qk_pairs_store_kernel forms
__global__ __launch_bounds__(256) void qkv_turns_kernel(const int64_t* positions, const float* inv_freq, int half, float m, float* turns,
                                                        int64_t n) {
  const int64_t i = blockIdx.x * 256ll + threadIdx.x;
  if (i >= n) return;
  const int64_t t = i / half;
  const int k = (int)(i - t * half);
  const float a = (float)positions[t] * inv_freq[k];
  turns[t * 2 * half + k] = cosf(a) * m;
  turns[t * 2 * half + half + k] = sinf(a) * m;
}

template <int D, int HALF16>
hipError_t qkv_go(const QkvArgs& p, hipStream_t s) {
  const QkvJob<D, HALF16> job{p, p.K, (p.M + STREAM_BM - 1) / STREAM_BM, (p.N + STREAM_BN - 1) / STREAM_BN};
  return launch_stream_deep(job, (int64_t)job.rows * job.cols, s);
}

}  // namespace

extern "C" int nv_qkv_stream(const void* x, int64_t x_row_stride, const void* w, int64_t tokens, int N, int K, const int64_t* positions,
                             const float* inv_freq, int rot_dims, float mscale, float scale, const int32_t* slot_mapping, void* cache,
                             float* q_out, float* rest, int64_t rest_row_stride, float* turns, int heads, int kv_heads, int dim, int vdim,
                             nv_stream_t stream) {
  return nv_qkv_stream_as(x, x_row_stride, w, tokens, N, K, positions, inv_freq, rot_dims, mscale, scale, slot_mapping, cache, q_out, NV_F32,
                          rest, rest_row_stride, turns, heads, kv_heads, dim, vdim, stream);
}

extern "C" int nv_qkv_stream_as(const void* x, int64_t x_row_stride, const void* w, int64_t tokens, int N, int K, const int64_t* positions,
                                const float* inv_freq, int rot_dims, float mscale, float scale, const int32_t* slot_mapping, void* cache,
                                void* q_out, int q_dtype, float* rest, int64_t rest_row_stride, float* turns, int heads, int kv_heads,
                                int dim, int vdim, nv_stream_t stream) {
  NV_CHECK_ARG(q_dtype == NV_F32 || q_dtype == NV_BF16, "nv_qkv_stream: bad dtype %d of the queries", q_dtype);
  NV_CHECK_ARG(x && w && slot_mapping && cache && q_out, "nv_qkv_stream: null pointer");
  NV_CHECK_ARG(dim == 64 || dim == 128, "nv_qkv_stream: head_dim %d not in {64, 128}", dim);
  NV_CHECK_ARG(heads > 0 && kv_heads > 0 && heads <= 65536 && kv_heads <= 65536 && vdim > 0 && vdim <= 65536 && kv_heads * vdim % 16 == 0,
               "nv_qkv_stream: bad shape");
  NV_CHECK_ARG(rot_dims == 0 || rot_dims == 32 || rot_dims == 64 || rot_dims == 128, "nv_qkv_stream: %d rotated numbers", rot_dims);
  NV_CHECK_ARG(rot_dims <= dim && (rot_dims == 0 || (positions && inv_freq && turns)),
               "nv_qkv_stream: a rotation over %d of %d numbers needs positions, frequencies and room for the turns", rot_dims, dim);
  const int64_t nq = (int64_t)heads * dim, nk = (int64_t)kv_heads * dim, nkv = nk + (int64_t)kv_heads * vdim;
  NV_CHECK_ARG(N >= nq + nkv && N < (1 << 20) && K >= 128 && K % 64 == 0 && K < (1 << 22), "nv_qkv_stream: N=%d K=%d", N, K);
  NV_CHECK_ARG(N == nq + nkv || (rest && rest_row_stride >= N - nq - nkv), "nv_qkv_stream: %d columns have no place", (int)(N - nq - nkv));
  NV_CHECK_ARG(tokens >= 0 && x_row_stride >= K && x_row_stride % 8 == 0 && x_row_stride < ((int64_t)1 << 30), "nv_qkv_stream: bad rows");
  NV_CHECK_ARG(((uintptr_t)x | (uintptr_t)w | (uintptr_t)q_out | (uintptr_t)turns) % 16 == 0 && (uintptr_t)cache % 8 == 0,
               "nv_qkv_stream: misaligned pointers");
  const int64_t tiles = (tokens + 255) / 256 * ((N + 255) / 256);
  NV_CHECK_ARG(tokens < ((int64_t)1 << 31) && tiles <= 256 * (STREAM_LIST - 2), "nv_qkv_stream: %lld rows exceed one launch", (long long)tokens);
  if (tokens == 0) return NV_OK;
  hipStream_t s = (hipStream_t)stream;
  if (rot_dims) {
    const int64_t n = tokens * (rot_dims / 2);
    qkv_turns_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>(positions, inv_freq, rot_dims / 2, mscale, turns, n);
    NV_CHECK_LAUNCH();
  }
  const QkvArgs p{(const uint16_t*)x, (const uint16_t*)w, x_row_stride, turns, slot_mapping, (uint16_t*)cache, q_out, rest, rest_row_stride,
                  (int)tokens, N, K, (int)nq, (int)nk, (int)nkv, scale, q_dtype == NV_BF16};
  hipError_t e;
  if (dim == 64) e = rot_dims == 0 ? qkv_go<64, 0>(p, s) : rot_dims == 32 ? qkv_go<64, 1>(p, s) : qkv_go<64, 2>(p, s);
  else e = rot_dims == 0 ? qkv_go<128, 0>(p, s) : rot_dims == 32 ? qkv_go<128, 1>(p, s) : rot_dims == 64 ? qkv_go<128, 2>(p, s) : qkv_go<128, 4>(p, s);
  if (e != hipSuccess) {
    nv_set_error("nv_qkv_stream: %s", hipGetErrorString(e));
    return NV_ERR_LAUNCH;
  }
  return NV_OK;
}
