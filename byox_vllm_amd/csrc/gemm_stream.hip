// The dense decoder's products of many rows (prefill) with what follows them, on the tiles of stream_tiles.h: bias; SiLU(gate) * up;
// or bias, per-head norms, rotation and the KV-cache store.  16-bit weights, row-major or in nv_gemm's tiled layout, which the tiles'
// DMA reads as it lies: nothing is written out first.
//
// What bounded these steps: the vendor library's product, then a pass over its whole result that moves it twice.  14.6 k rows of 1024
// (Qwen3-0.6B): gate and up 157 us and SiluAndMul 53, q/k/v 105 and rotation with the store 61, and 5 - 7 us before each for the
// weight as rows.  Here 190 and 151 us; SiLU by exp and quotient, as in the pass, is 20 of the first.  Which sizes this pays for:
// kernels.gemm_many_rows and kernels.rotation_streams.
#include <type_traits>

#include "rope_common.h"
#include "stream_tiles.h"

namespace {

struct RowsArgs {
  const void *x, *w, *bias;
  void* out;
  int64_t xs, os;
  int M, N, K, tiled;
};

enum { ROWS_PLAIN = 0, ROWS_SILU = 1, ROWS_ROPE = 2 };

template <typename TT, int WHAT, int D, bool TILED>     // D: head size (ROWS_ROPE)
struct RowsJob {
  typedef TT T;
  typedef std::conditional_t<WHAT == ROWS_SILU, std::conditional_t<TILED, StreamQuadsTiled, StreamQuads>,
                             std::conditional_t<TILED, StreamPairedTiled, StreamPaired>> Order;
  static constexpr bool SILU = WHAT == ROWS_SILU, ROPE = WHAT == ROWS_ROPE;
  // a wavefront has whole heads, 128 columns, where their halves meet; else 64 columns and more rows
  static constexpr int WN = ROPE ? 2 : 4, MT = 2 * WN, NT = 32 / WN / 2, NOUT = SILU ? 128 : 256;
  static constexpr int NSTORE = MT * (SILU ? 1 : NT / 2);
  RowsArgs p;
  RopeArgs ra;
  int K, rows, cols;      // row and column tiles

  __device__ __forceinline__ int count(int) const { return rows * cols; }
  __device__ __forceinline__ StreamTile find(int tile, int) const {
    int m_tile, n_tile;
    stream_order(tile, rows, cols, m_tile, n_tile);
    return StreamTile{m_tile * STREAM_BM, p.M, n_tile * NOUT, 0};
  }
  __device__ __forceinline__ const void* a_base(const StreamTile&) const { return p.x; }
  __device__ __forceinline__ uint32_t a_stride() const { return (uint32_t)p.xs * 2; }
  __device__ __forceinline__ uint32_t a_row(const StreamTile& at, int r) const { return (uint32_t)min(at.lo + r, at.hi - 1); }
  __device__ __forceinline__ const void* w_base(const StreamTile&) const { return p.w; }
  __device__ __forceinline__ uint32_t w_stride() const { return (uint32_t)p.K * (TILED ? 32 : 2); }
  __device__ __forceinline__ uint32_t w_row(const StreamTile& at, int r) const {      // r: row, or 16-row tile
    const int n = at.n0 * (SILU ? 2 : 1);
    return TILED ? min((n >> 4) + r, (p.N >> 4) - 1) : min(n + r, p.N - 1);
  }
  __device__ __forceinline__ uint32_t w_step() const { return TILED ? 2048 : 128; }
  __device__ __forceinline__ bool whole(const StreamTile& at) const {
    return at.lo + STREAM_BM <= at.hi && (at.n0 + NOUT) * (SILU ? 2 : 1) <= p.N;
  }

  static __device__ __forceinline__ void widen(const uint16_t* at, float (&v)[8]) {
    const u32x4 w = *reinterpret_cast<const u32x4*>(at);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = lo_f32<T>(w[e]);
      v[2 * e + 1] = hi_f32<T>(w[e]);
    }
  }
  static __device__ __forceinline__ u32x4 pack(const float (&v)[8]) {
    return u32x4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])};
  }
  static __device__ __forceinline__ float rounded(float v) { return bits_to_f32<T>(f32_to_bits<T>(v)); }

  __device__ __forceinline__ void store(const StreamTile& at, int row0, int wn, int lane, const f32x4 (&acc)[NT][MT]) const {
    const int fr = lane & 15, g = lane >> 4;
    const uint16_t* bias = reinterpret_cast<const uint16_t*>(p.bias);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      __builtin_amdgcn_sched_barrier(0);       // one row's results at a time: registers
      const int s = row0 + 16 * i + fr;
      if constexpr (SILU) {
        const int n = at.n0 + 32 * wn + 8 * g;        // a lane's eight results come from 16 rows of W: N is a multiple of that
        if (s >= at.hi || 2 * n >= p.N) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          // dtype(dtype(silu(dtype(gate))) * dtype(up)), as nv_silu_mul takes it
          const float gt = rounded(acc[e >> 2][i][e & 3]), up = rounded(acc[2 + (e >> 2)][i][e & 3]);
          v[e] = rounded(gt / (1.0f + expf(-gt))) * up;
        }
        *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(p.out) + s * p.os + n) = pack(v);
      } else {
        const int n0 = at.n0 + 16 * NT * wn;
        uint16_t* row = reinterpret_cast<uint16_t*>(p.out) + s * p.os;
        if constexpr (!ROPE) {
          if (s >= at.hi) continue;
#pragma unroll
          for (int q = 0; q < NT / 2; ++q) {
            const int n = n0 + 32 * q + 8 * g;
            if (n >= p.N) continue;
            float v[8], b[8] = {};
            if (bias) widen(bias + n, b);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = acc[2 * q + (e >> 2)][i][e & 3] + b[e];
            *reinterpret_cast<u32x4*>(row + n) = pack(v);
          }
        } else {
#pragma unroll
          for (int h = 0; h < 128 / D; ++h) rope_row(s, s < at.hi, n0 + D * h, 8 * g, bias, row, acc, i, 2 * (D / 32) * h);
        }
      }
    }
  }

  // One head of one token, spread over the four lanes g: `c` = 8 g, numbers 32 q + c .. + 7 from products j0 + 2 q and j0 + 2 q + 1.
  // The arithmetic and its roundings are those of rope_finish.
  __device__ __forceinline__ void rope_row(int64_t t, bool live, int n, int c, const uint16_t* bias, uint16_t* row,
                                           const f32x4 (&acc)[NT][MT], int i, int j0) const {
    constexpr int Q = D / 32;
    if (n >= p.N) return;
    const int hs = n / D;
    const bool is_q = hs < ra.H, is_k = !is_q && hs < ra.H + ra.Hkv;
    float x[Q][8];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      float b[8] = {};
      if (bias) widen(bias + n + 32 * q + c, b);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[q][e] = rounded(acc[j0 + 2 * q + (e >> 2)][i][e & 3] + b[e]);
    }
    const int slot = ra.slots && live ? ra.slots[t] : -1;
    const uint16_t* nw = is_q ? ra.qn_w : is_k ? ra.kn_w : nullptr;
    if (nw) {
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
        widen(nw + 32 * q + c, w);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[q][e] = rounded(rounded(x[q][e] * inv) * w[e]);
      }
    }
    if (!live) return;
    if (is_q || is_k) {
      const float* cs = ra.cos_sin + ra.positions[t] * D + c;
#pragma unroll
      for (int q = 0; q < Q / 2; ++q) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const f32x4 co = *reinterpret_cast<const f32x4*>(cs + 32 * q + 4 * v), si = *reinterpret_cast<const f32x4*>(cs + D / 2 + 32 * q + 4 * v);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = x[q][4 * v + e], b = x[q + Q / 2][4 * v + e];
            x[q][4 * v + e] = __fsub_rn(__fmul_rn(a, co[e]), __fmul_rn(b, si[e]));
            x[q + Q / 2][4 * v + e] = __fadd_rn(__fmul_rn(b, co[e]), __fmul_rn(a, si[e]));
          }
        }
      }
    }
    uint16_t* cache = nullptr;
    if (!is_q && slot >= 0 && ra.k_cache)
      cache = (is_k ? ra.k_cache : ra.v_cache) + ((int64_t)slot * ra.Hkv + (hs - ra.H - (is_k ? 0 : ra.Hkv))) * D;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const u32x4 v = pack(x[q]);
      *reinterpret_cast<u32x4*>(row + n + 32 * q + c) = v;
      if (cache) *reinterpret_cast<u32x4*>(cache + 32 * q + c) = v;
    }
  }
};

template <typename T, int WHAT, int D, bool TILED>
hipError_t rows_go_as(const RowsArgs& p, const RopeArgs& ra, hipStream_t s) {
  typedef RowsJob<T, WHAT, D, TILED> Job;
  const int n = WHAT == ROWS_SILU ? p.N / 2 : p.N;
  const Job job{p, ra, p.K, (p.M + STREAM_BM - 1) / STREAM_BM, (n + Job::NOUT - 1) / Job::NOUT};
  return launch_stream_tiles<Job::WN>(job, (int64_t)job.rows * job.cols, s);
}
template <typename T, int WHAT, int D>
hipError_t rows_go(const RowsArgs& p, const RopeArgs& ra, hipStream_t s) {
  return p.tiled ? rows_go_as<T, WHAT, D, true>(p, ra, s) : rows_go_as<T, WHAT, D, false>(p, ra, s);
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
