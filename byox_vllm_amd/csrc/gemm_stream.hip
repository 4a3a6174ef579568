// The dense decoder's products of many rows (prefill) with what follows them, on the tiles of stream_deep.h: bias; SiLU(gate) * up;
// or bias, per-head norms, rotation and the KV-cache store.  16-bit weights, row-major or in nv_gemm's tiled layout, which the tiles'
// DMA reads as it lies: nothing is written out first.
//
// What bounded these steps: the vendor library's product, then a pass over its whole result that moves it twice.  14.6 k rows of 1024
// (Qwen3-0.6B): gate and up 157 us and SiluAndMul 53, q/k/v 105 and rotation with the store 61, and 5 - 7 us before each for the
// weight as rows.  Here 170 and 142 us (193 and 157 on the tiles of eight wavefronts).  What the results cost counts: with one wavefront to a
// SIMD nothing hides it.  So SiLU in 17 instructions (anyt.h; silu_f32's 27: 8 % more), roundings two at a time, and a row's cosines and sines,
// norm weights and bias on their way before they are needed.  Which sizes this pays for: kernels.gemm_many_rows and kernels.rotation_streams.
#include <type_traits>

#include "anyt.h"
#include "rope_common.h"
#include "stream_deep.h"

namespace {

struct RowsArgs {
  const void *x, *w, *bias;
  void* out;
  int64_t xs, os;
  int M, N, K, tiled;
};

enum { ROWS_PLAIN = 0, ROWS_SILU = 1, ROWS_ROPE = 2 };

template <typename TT, int WHAT, int D, bool TILED, bool FAR>     // D: head size (ROWS_ROPE); FAR: a tile's rows span 4 GiB and more
struct RowsJob {
  typedef TT T;
  typedef std::conditional_t<WHAT == ROWS_SILU, std::conditional_t<TILED, StreamQuadsTiled, StreamQuads>,
                             std::conditional_t<TILED, StreamPairedTiled, StreamPaired>> Order;
  static constexpr bool SILU = WHAT == ROWS_SILU, ROPE = WHAT == ROWS_ROPE;
  static constexpr int NOUT = SILU ? 128 : 256, NSTORE_WAVE = SILU ? 16 : 32, EXTRA = ROPE ? 3072 : 0;
  static constexpr bool FAR_A = FAR, FAR_W = FAR, UPS = false;
  RowsArgs p;
  RopeArgs ra;
  int K, rows, cols;      // row and column tiles

  __device__ __forceinline__ int count(int) const { return rows * cols; }
  __device__ __forceinline__ StreamTile find(int tile, int) const {
    int m_tile, n_tile;
    stream_order(tile, rows, cols, m_tile, n_tile);
    return StreamTile{m_tile * STREAM_BM, p.M, n_tile * NOUT, 0};
  }
  // the second half of a short tile has no rows and begins behind the last one
  __device__ __forceinline__ static int first_row(const StreamTile& at) { return min(at.lo, at.hi - 1); }
  __device__ __forceinline__ const void* a_base(const StreamTile& at) const { return reinterpret_cast<const uint16_t*>(p.x) + first_row(at) * p.xs; }
  __device__ __forceinline__ uint32_t a_stride() const { return (uint32_t)p.xs * 2; }
  __device__ __forceinline__ uint32_t a_row(const StreamTile& at, int r) const { return (uint32_t)min(r, at.hi - 1 - first_row(at)); }
  __device__ __forceinline__ const void* w_base(const StreamTile& at) const {
    return reinterpret_cast<const uint16_t*>(p.w) + (int64_t)at.n0 * (SILU ? 2 : 1) * p.K;      // a row has K numbers in either layout
  }
  __device__ __forceinline__ uint32_t w_stride() const { return (uint32_t)p.K * (TILED ? 32 : 2); }
  __device__ __forceinline__ uint32_t w_row(const StreamTile& at, int r) const {      // r: row, or 16-row tile
    const int left = p.N - at.n0 * (SILU ? 2 : 1);
    return min(r, (TILED ? left >> 4 : left) - 1);
  }
  __device__ __forceinline__ uint32_t w_step() const { return TILED ? 2048 : 128; }
  __device__ __forceinline__ bool whole(const StreamTile& at) const {
    return at.lo + STREAM_BM <= at.hi && (at.n0 + NOUT) * (SILU ? 2 : 1) <= p.N;
  }

  static __device__ __forceinline__ void widen(const u32x4& w, float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = lo_f32<T>(w[e]);
      v[2 * e + 1] = hi_f32<T>(w[e]);
    }
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[8]) {
    return u32x4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])};
  }
  static __device__ __forceinline__ void round8(float (&v)[8]) {      // two at a time: half the instructions
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const uint32_t w = pack2<T>(v[e], v[e + 1]);
      v[e] = lo_f32<T>(w);
      v[e + 1] = hi_f32<T>(w);
    }
  }

  // -------- results: 64 rows of each half of the tile by 128 rows of W to a wavefront
  __device__ __forceinline__ void fetch_extra(const StreamTile& at, int wv, int lane, unsigned char* extra) const {
    if constexpr (ROPE) {      // the rows' positions (their low halves), cache rows, bias and norm weights, a tile ahead of their use
      typedef __attribute__((address_space(1))) void global_void;
      typedef __attribute__((address_space(3))) void lds_void;
      const int t = min(at.lo + 64 * wv + lane, at.hi - 1);
      __builtin_amdgcn_global_load_lds((global_void*)(ra.positions + t), (lds_void*)(extra + 256 * wv), 4, 0, 0);
      if (ra.slots) __builtin_amdgcn_global_load_lds((global_void*)(ra.slots + t), (lds_void*)(extra + 1024 + 256 * wv), 4, 0, 0);
      const uint16_t* norm = wv & 1 ? ra.kn_w : ra.qn_w;
      const uint16_t* from = wv < 2 ? reinterpret_cast<const uint16_t*>(p.bias) : norm;      // two numbers to a lane
      const int n = wv < 2 ? min(at.n0 + 128 * wv + 2 * lane, p.N - 2) : min(2 * lane, D - 2);
      if (from) __builtin_amdgcn_global_load_lds((global_void*)(from + n), (lds_void*)(extra + 2048 + 256 * wv), 4, 0, 0);
    }
  }
  __device__ __forceinline__ void finish(const StreamTile& at, int wm, int wn, int lane, bool live0, bool live1, const unsigned char* extra) const {
    if constexpr (ROPE) {
      if (at.n0 + 128 * wn < p.N) rotate(at, wm, at.n0 + 128 * wn, lane, live0, live1, extra);
    } else {
      if (live0) store<0>(at, at.lo + 64 * wm, wn, lane);
      if (live1) store<1>(at, at.lo + 128 + 64 * wm, wn, lane);
    }
  }
  template <int HALF>
  __device__ __forceinline__ void store(const StreamTile& at, int row0, int wn, int lane) const {
    const int fr = lane & 15, g = lane >> 4;
    constexpr int PIECES = SILU ? 2 : 4;
    int n[PIECES];
    u32x4 b[PIECES];      // ahead of the first store: loads and stores are counted in one order
    const uint16_t* bias = reinterpret_cast<const uint16_t*>(p.bias);
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
      n[q] = at.n0 + (SILU ? 64 : 128) * wn + 32 * q + 8 * g;
      if (!SILU && bias) b[q] = *reinterpret_cast<const u32x4*>(bias + min(n[q], p.N - 8));
    }
    if (!SILU && bias) {
#pragma unroll
      for (int q = 0; q < PIECES; ++q) asm volatile("" : "+v"(b[q]));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int s = row0 + 16 * i + fr;
      uint16_t* row = reinterpret_cast<uint16_t*>(p.out) + s * p.os;
#pragma unroll
      for (int q = 0; q < PIECES; ++q) {
        __builtin_amdgcn_sched_barrier(0);       // a few results at a time: registers
        float v[8];
        if constexpr (SILU) {      // a lane's eight results come from 16 rows of W: N is a multiple of that
          f32x4 x[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = deep_take(HALF, 4 * q + j, i);
          float up[8];      // dtype(dtype(silu(dtype(gate))) * dtype(up)), as nv_silu_mul takes it
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            v[e] = x[e >> 2][e & 3];
            up[e] = x[2 + (e >> 2)][e & 3];
          }
          round8(v);
          round8(up);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = silu_16bit(v[e]);
          round8(v);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= up[e];
        } else {
          f32x4 x[2];
#pragma unroll
          for (int j = 0; j < 2; ++j) x[j] = deep_take(HALF, 2 * q + j, i);
          float w[8];
          if (bias) widen(b[q], w);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = x[e >> 2][e & 3] + (bias ? w[e] : -0.0f);
        }
        if (s < at.hi && n[q] * (SILU ? 2 : 1) < p.N) *reinterpret_cast<u32x4*>(row + n[q]) = pack(v);
      }
    }
  }

  // The heads of columns n0 .. n0 + 127 of the wavefront's rows: lane (fr, g) has numbers 32 q + 8 g .. + 7 of a head of row fr.  The
  // arithmetic and its roundings are those of rope_finish.  A row's cosines and sines are asked for two rows ahead, before the stores of
  // the row between: behind them they would be waited for with them.
  __device__ __forceinline__ void rotate(const StreamTile& at, int wm, int n0, int lane, bool live0, bool live1, const unsigned char* extra) const {
    constexpr int Q = D / 32, HEADS = 128 / D;
    const int fr = lane & 15, c = 8 * (lane >> 4);
    bool is_q[HEADS], is_k[HEADS];
    int hs[HEADS];
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      hs[h] = n0 / D + h;
      is_q[h] = hs[h] < ra.H;
      is_k[h] = !is_q[h] && hs[h] < ra.H + ra.Hkv;
    }
    const bool turns = n0 < (ra.H + ra.Hkv) * D;
    auto kept = [&](int r, int which) {
      return *reinterpret_cast<const uint32_t*>(extra + 1024 * which + 4 * (128 * (r >> 2) + 64 * wm + 16 * (r & 3) + fr));
    };
    f32x4 turn[2][2 * Q];      // cosines, then sines
    auto ask = [&](int r) {
      if (!turns) return;
      const float* cs = ra.cos_sin + (int64_t)kept(r, 0) * D + c;
#pragma unroll
      for (int q = 0; q < Q / 2; ++q)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          turn[r & 1][2 * q + v] = *reinterpret_cast<const f32x4*>(cs + 32 * q + 4 * v);
          turn[r & 1][Q + 2 * q + v] = *reinterpret_cast<const f32x4*>(cs + D / 2 + 32 * q + 4 * v);
        }
    };
    ask(0);
    ask(1);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      __builtin_amdgcn_sched_barrier(0);
      const int64_t t = at.lo + 128 * (r >> 2) + 64 * wm + 16 * (r & 3) + fr;
      u32x4 out[4];
#pragma unroll
      for (int h = 0; h < HEADS; ++h) {
        f32x4 a[2 * Q];
#pragma unroll
        for (int j = 0; j < 2 * Q; ++j) a[j] = deep_take(r >> 2, 2 * Q * h + j, r & 3);
        float x[Q][8];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          float w[8];
          if (p.bias) widen(*reinterpret_cast<const u32x4*>(extra + 2048 + 2 * (n0 - at.n0 + D * h + 32 * q + c)), w);
#pragma unroll
          for (int e = 0; e < 8; ++e) x[q][e] = a[2 * q + (e >> 2)][e & 3] + (p.bias ? w[e] : 0.0f);
          round8(x[q]);
        }
        if (ra.qn_w && (is_q[h] || is_k[h])) {
          float ss = 0.f;
#pragma unroll
          for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += x[q][e] * x[q][e];
          float even, odd, lower, upper;
          rows_pair16(ss, even, odd);
          rows_pair32(even + odd, lower, upper);
          const float inv = 1.0f / sqrtf((lower + upper) / (float)D + ra.eps);
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            float w[8];
            widen(*reinterpret_cast<const u32x4*>(extra + (is_q[h] ? 2560 : 2816) + 2 * (32 * q + c)), w);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[q][e] *= inv;
            round8(x[q]);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[q][e] *= w[e];
            round8(x[q]);
          }
        }
        if (is_q[h] || is_k[h]) {
#pragma unroll
          for (int q = 0; q < Q / 2; ++q)
#pragma unroll
            for (int v = 0; v < 2; ++v) {
              const f32x4 co = turn[r & 1][2 * q + v], si = turn[r & 1][Q + 2 * q + v];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float lo = x[q][4 * v + e], hi = x[q + Q / 2][4 * v + e];
                x[q][4 * v + e] = __fsub_rn(__fmul_rn(lo, co[e]), __fmul_rn(hi, si[e]));
                x[q + Q / 2][4 * v + e] = __fadd_rn(__fmul_rn(hi, co[e]), __fmul_rn(lo, si[e]));
              }
            }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) out[h * Q + q] = pack(x[q]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (r + 2 < 8) ask(r + 2);
      __builtin_amdgcn_sched_barrier(0);
      if (t >= at.hi || !(r < 4 ? live0 : live1)) continue;
      uint16_t* row = reinterpret_cast<uint16_t*>(p.out) + t * p.os + n0 + c;
#pragma unroll
      for (int h = 0; h < HEADS; ++h) {
        if (n0 + D * h >= p.N) continue;
#pragma unroll
        for (int q = 0; q < Q; ++q) *reinterpret_cast<u32x4*>(row + D * h + 32 * q) = out[h * Q + q];
        if (is_q[h] || !ra.k_cache) continue;
        const int slot = (int)kept(r, 1);
        if (slot < 0) continue;
        uint16_t* cache = (is_k[h] ? ra.k_cache : ra.v_cache) + ((int64_t)slot * ra.Hkv + (hs[h] - ra.H - (is_k[h] ? 0 : ra.Hkv))) * D + c;
#pragma unroll
        for (int q = 0; q < Q; ++q) *reinterpret_cast<u32x4*>(cache + 32 * q) = out[h * Q + q];
      }
    }
  }
};

template <typename T, int WHAT, int D, bool TILED, bool FAR>
hipError_t rows_go_as(const RowsArgs& p, const RopeArgs& ra, hipStream_t s) {
  typedef RowsJob<T, WHAT, D, TILED, FAR> Job;
  const int n = WHAT == ROWS_SILU ? p.N / 2 : p.N;
  const Job job{p, ra, p.K, (p.M + STREAM_BM - 1) / STREAM_BM, (n + Job::NOUT - 1) / Job::NOUT};
  return launch_stream_deep(job, (int64_t)job.rows * job.cols, s);
}
template <typename T, int WHAT, int D>
hipError_t rows_go(const RowsArgs& p, const RopeArgs& ra, hipStream_t s) {
  if (p.xs >= (1 << 22) || p.K >= (1 << 22))
    return p.tiled ? rows_go_as<T, WHAT, D, true, true>(p, ra, s) : rows_go_as<T, WHAT, D, false, true>(p, ra, s);
  return p.tiled ? rows_go_as<T, WHAT, D, true, false>(p, ra, s) : rows_go_as<T, WHAT, D, false, false>(p, ra, s);
}

template <typename T>
hipError_t rows_pick(const RowsArgs& p, const RopeArgs& ra, int what, hipStream_t s) {
  if (what == ROWS_SILU) return rows_go<T, ROWS_SILU, 0>(p, ra, s);
  if (what == ROWS_PLAIN) return rows_go<T, ROWS_PLAIN, 0>(p, ra, s);
  return ra.D == 128 ? rows_go<T, ROWS_ROPE, 128>(p, ra, s) : rows_go<T, ROWS_ROPE, 64>(p, ra, s);
}

int rows_launch(const char* name, const RowsArgs& p, const RopeArgs& ra, int what, int wfmt, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG(p.x && p.w && p.out, "%s: null pointer", name);
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F16, "%s: bad dtype %d", name, dtype);
  NV_CHECK_ARG(wfmt == NV_W_DENSE || wfmt == NV_W_DENSE_TILED, "%s: weight format %d is not a 16-bit one", name, wfmt);
  NV_CHECK_ARG(p.M >= 0 && p.N > 0 && p.K >= 128 && p.K % 64 == 0 && p.N % 16 == 0 && (!p.tiled || p.K % 128 == 0),
               "%s: M=%d N=%d K=%d", name, p.M, p.N, p.K);
  NV_CHECK_ARG(p.xs >= p.K && p.xs % 8 == 0 && p.xs < ((int64_t)1 << 31) && p.os % 8 == 0 && p.os >= (what == ROWS_SILU ? p.N / 2 : p.N) &&
                   p.K < (1 << 26), "%s: bad row strides", name);
  NV_CHECK_ARG(((uintptr_t)p.x | (uintptr_t)p.w | (uintptr_t)p.out | (uintptr_t)p.bias) % 16 == 0, "%s: pointers must be 16-byte aligned",
               name);
  const int64_t tiles = (int64_t)((p.M + 255) / 256) * ((p.N + 255) / 256);
  NV_CHECK_ARG(tiles <= 256 * (STREAM_LIST - 2), "%s: M=%d N=%d exceed one launch", name, p.M, p.N);
  if (p.M == 0) return NV_OK;
  const hipError_t e = dtype == NV_BF16 ? rows_pick<bf16_t>(p, ra, what, (hipStream_t)stream)
                                        : rows_pick<f16_t>(p, ra, what, (hipStream_t)stream);
  if (e != hipSuccess) {
    nv_set_error("%s: %s", name, hipGetErrorString(e));
    return NV_ERR_LAUNCH;
  }
  return NV_OK;
}

}  // namespace

extern "C" int nv_gemm_stream(const void* x, int64_t x_row_stride, const void* w, const void* bias, void* out, int64_t out_row_stride,
                              int M, int N, int K, int wfmt, int silu_mul, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG(!silu_mul || !bias, "nv_gemm_stream: the silu*up epilogue takes no bias");
  const RowsArgs p{x, w, bias, out, x_row_stride, out_row_stride, M, N, K, wfmt == NV_W_DENSE_TILED};
  return rows_launch("nv_gemm_stream", p, RopeArgs{}, silu_mul ? ROWS_SILU : ROWS_PLAIN, wfmt, dtype, stream);
}

extern "C" int nv_gemm_stream_rope_kv_store(const void* x, int64_t x_row_stride, const void* w, const void* bias, void* qkv,
                                            int64_t qkv_row_stride, int M, int K, int wfmt, const int64_t* positions,
                                            const float* cos_sin, const int32_t* slot_mapping, void* k_cache, void* v_cache,
                                            const void* q_norm_w, const void* k_norm_w, float eps, int H, int Hkv, int D, int dtype,
                                            nv_stream_t stream) {
  NV_CHECK_ARG(positions && cos_sin, "nv_gemm_stream_rope_kv_store: null pointer");
  NV_CHECK_ARG(D == 64 || D == 128, "nv_gemm_stream_rope_kv_store: head_dim %d not in {64, 128}", D);
  NV_CHECK_ARG(H >= 0 && Hkv >= 0 && H + Hkv > 0, "nv_gemm_stream_rope_kv_store: bad head counts");
  NV_CHECK_ARG((k_cache == nullptr) == (v_cache == nullptr) && (!k_cache || slot_mapping),
               "nv_gemm_stream_rope_kv_store: k_cache, v_cache and slot_mapping go together");
  NV_CHECK_ARG((q_norm_w == nullptr) == (k_norm_w == nullptr), "nv_gemm_stream_rope_kv_store: q_norm_w and k_norm_w go together");
  NV_CHECK_ARG(((uintptr_t)cos_sin | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w) % 16 == 0,
               "nv_gemm_stream_rope_kv_store: pointers must be 16-byte aligned");
  RopeArgs ra;
  ra.positions = positions; ra.cos_sin = cos_sin; ra.slots = slot_mapping;
  ra.k_cache = (uint16_t*)k_cache; ra.v_cache = (uint16_t*)v_cache;
  ra.qn_w = (const uint16_t*)q_norm_w; ra.kn_w = (const uint16_t*)k_norm_w;
  ra.eps = eps; ra.H = H; ra.Hkv = Hkv; ra.D = D;
  const RowsArgs p{x, w, bias, qkv, x_row_stride, qkv_row_stride, M, (H + 2 * Hkv) * D, K, wfmt == NV_W_DENSE_TILED};
  return rows_launch("nv_gemm_stream_rope_kv_store", p, ra, ROWS_ROPE, wfmt, dtype, stream);
}
