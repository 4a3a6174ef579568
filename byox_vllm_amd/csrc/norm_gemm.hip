// A decode step's residual add + RMSNorm inside the product that reads it, for a few rows: q/k/v (with bias, head norms, rotation and
// the KV-cache store behind it) and gate/up (with SiLU(gate) * up behind it).  16-bit weights in nv_gemm's tiled layout.
//
// What bounds a step of one row: launches.  Each of 8 per layer is one trip to memory and back, 3 - 5 us whatever it computes, and the
// norm and the rotation are two of them around a product whose weights do not depend on them.  Here every workgroup forms the norm of
// all rows itself (a few KB), four numbers to a thread, while its weights are already on their way: 16 rows by 32 of K
// per wavefront and register set, the whole K of a tile of 16 outputs dealt to PARTS wavefronts.  Only the first workgroup writes the
// new residual, to another buffer than the one the others may still be reading.  Qwen2-0.5B, one row, under the profiler: norm 3.7 +
// product 8.3 us and 3.7 + 4.6 + rotation 4.5, here 8.5 and 8.3; the step in a captured graph 867 and 774.  The norm is repeated by every
// workgroup, in passes over the rows that its wavefronts hold at once: which sizes that pays for is kernels.norm_gemm_pays.
#include "rope_common.h"
#include "splitk.h"

namespace {

struct NormGemmArgs {
  const uint16_t* x;          // [M, K], or null: the rows are `nparts` fp32 slabs
  const float* part;
  int nparts;
  const uint16_t* res;        // [M, K] or null (no add)
  uint16_t* res_out;
  const uint16_t* nw;
  float eps;
  const u32x4* w;
  const uint16_t* bias;
  uint16_t* out;
  int64_t os;
  int M, N, K;
};

enum { NG_SILU = 0, NG_ROPE = 1 };

template <typename T, int TILES, int PARTS, int WHAT>
__global__ __launch_bounds__(64 * TILES * PARTS) void norm_gemm_kernel(NormGemmArgs p, RopeArgs ra) {
  typedef typename VecOf<T>::x8 vec_t;
  constexpr int WAVES = TILES * PARTS, PRE = PARTS < 4 ? 16 : 8, D = 16 * TILES;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  f32x4* red = reinterpret_cast<f32x4*>(lds_raw);                                       // [PARTS][TILES][64]
  unsigned char* rows = lds_raw + WAVES * 1024;                                         // [M][2 K + 16 bytes]
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = wv % TILES, part = wv / TILES, c = lane & 15, g = lane >> 4;
  const int nk = p.K >> 5, ks0 = part * nk / PARTS, ks1 = (part + 1) * nk / PARTS;
  const int nt = blockIdx.x * TILES + tile;
  const bool has = 16 * nt < p.N;
  const u32x4* wp = p.w + ((int64_t)(has ? nt : 0) * nk + ks0) * 64 + lane;
  u32x4 pre[PRE];
#pragma unroll
  for (int u = 0; u < PRE; ++u) pre[u] = wp[min(u, ks1 - ks0 - 1) * 64];

  // what a head's end needs of memory is asked for now, two dependent trips ahead of its use: then the CU's cache has it
  float warm = 0.f;
  if constexpr (WHAT == NG_ROPE) {
    constexpr int LPH = D / 8;
    const int t = tid / LPH, sub = tid % LPH;
    if (t < p.M) {
      const float* cs = ra.cos_sin + ra.positions[t] * D + 4 * sub;
      warm = cs[0] + cs[D / 2];
      if (ra.slots) warm += (float)ra.slots[t];
      if (p.bias) warm += (float)p.bias[blockIdx.x * D + 8 * sub];
      if (ra.qn_w) warm += (float)ra.qn_w[8 * sub] + (float)ra.kn_w[8 * sub];
    }
  }

  // the norm: four numbers per thread, a row to as many wavefronts as that takes
  const int nvec = p.K >> 2, stride = 2 * p.K + 16, wide = (nvec + 63) >> 6, at_once = WAVES / wide;      // wide <= 8
  const int i = (wv % wide) * 64 + lane, mine = wv / wide;
  float* sums = reinterpret_cast<float*>(red);
  for (int m0 = 0; m0 < p.M; m0 += at_once) {
    const int m = m0 + mine;
    const bool live = i < nvec && mine < at_once && m < p.M;
    const int64_t at = (int64_t)(live ? m : 0) * p.K + 4 * (live ? i : 0);
    const u32x2 ww = *reinterpret_cast<const u32x2*>(p.nw + 4 * (live ? i : 0));
    u32x2 b = {0, 0};
    if (p.res) b = *reinterpret_cast<const u32x2*>(p.res + at);
    f32x4 a;
    if (p.x) {
      a = unpack4<T>(*reinterpret_cast<const u32x2*>(p.x + at));
    } else {     // the rows as the product before would have stored them
      f32x4 s[1];
      slab_sum<1>(p.part + at, (int64_t)p.M * p.K, p.nparts, s);
      a = round4<T>(s[0]);
    }
    if (p.res) {
      a += unpack4<T>(b);
      if (blockIdx.x == 0 && live) *reinterpret_cast<u32x2*>(p.res_out + at) = pack4<T>(a);
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(a[e], a[e], ss);
    ss = wave_sum(live ? ss : 0.f);
    if (m0) __syncthreads();
    if (lane == 0) sums[wv] = ss;
    __syncthreads();
    ss = 0.f;
    for (int k = 0; k < wide; ++k) ss += sums[min(mine * wide + k, WAVES - 1)];
    const float inv = 1.0f / sqrtf(ss / (float)p.K + p.eps);
    if (live) *reinterpret_cast<u32x2*>(rows + m * stride + 8 * i) = pack4<T>(round4<T>(a * inv) * unpack4<T>(ww));
  }
  __syncthreads();

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto product = [&](const u32x4& wf, int ks) {
    u32x4 xf = {0, 0, 0, 0};
    if (c < p.M) xf = *reinterpret_cast<const u32x4*>(rows + c * stride + 64 * ks + 16 * g);
    acc = mfma16(__builtin_bit_cast(vec_t, wf), __builtin_bit_cast(vec_t, xf), acc);      // row n = 4 g + r, column m = c
  };
#pragma unroll
  for (int u = 0; u < PRE; ++u)
    if (ks0 + u < ks1) product(pre[u], ks0 + u);
  for (int k = PRE; ks0 + k < ks1; k += PRE) {
#pragma unroll
    for (int u = 0; u < PRE; ++u) pre[u] = wp[min(k + u, ks1 - ks0 - 1) * 64];
#pragma unroll
    for (int u = 0; u < PRE; ++u)
      if (ks0 + k + u < ks1) product(pre[u], ks0 + k + u);
  }
  red[wv * 64 + lane] = acc;
  asm volatile("" ::"v"(warm));
  __syncthreads();
  if constexpr (WHAT == NG_SILU) {
    if (part != 0 || !has || c >= p.M) return;
#pragma unroll
    for (int q = 1; q < PARTS; ++q) acc += red[(q * TILES + tile) * 64 + lane];
    // rows (gate j, gate j + 1, up j, up j + 1): dtype(dtype(silu(dtype(gate))) * dtype(up))
    float r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float gt = bits_to_f32<T>(f32_to_bits<T>(acc[e])), up = bits_to_f32<T>(f32_to_bits<T>(acc[2 + e]));
      r[e] = bits_to_f32<T>(f32_to_bits<T>(gt * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * gt)))) * up;
    }
    *reinterpret_cast<uint32_t*>(p.out + c * p.os + 8 * nt + 2 * g) = pack2<T>(r[0], r[1]);
  } else {
    // a workgroup has one head: D / 8 lanes per token take it from the partial sums and finish it
    constexpr int LPH = D / 8;
    const int t = tid / LPH, sub = tid % LPH;
    if (tid - lane >= LPH * p.M) return;             // whole wavefronts: the others exchange values
    const bool live = t < p.M;
    f32x4 x[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int col = h * (D / 2) + 4 * sub, at = (col >> 4) * 64 + 16 * ((col & 15) >> 2) + (live ? t : 0);
      x[h] = red[at];
#pragma unroll
      for (int q = 1; q < PARTS; ++q) x[h] += red[q * TILES * 64 + at];
      if (p.bias) x[h] += unpack4<T>(*reinterpret_cast<const u32x2*>(p.bias + blockIdx.x * D + col));
      x[h] = round4<T>(x[h]);
    }
    rope_finish<T>(x[0], x[1], ra, blockIdx.x, live ? t : 0, sub, p.out + (live ? t : 0) * p.os + (int64_t)blockIdx.x * D, true, live);
  }
}

template <typename T, int TILES, int PARTS, int WHAT>
int norm_gemm_go(const NormGemmArgs& p, const RopeArgs& ra, hipStream_t s) {
  const int tiles = (p.N + 15) / 16;
  const size_t lds = TILES * PARTS * 1024 + (size_t)p.M * (2 * p.K + 16);
  norm_gemm_kernel<T, TILES, PARTS, WHAT><<<dim3((tiles + TILES - 1) / TILES), dim3(64 * TILES * PARTS), lds, s>>>(p, ra);
  NV_CHECK_LAUNCH();
  return NV_OK;
}

int norm_gemm_launch(const char* name, const NormGemmArgs& p, const RopeArgs& ra, int what, int dtype, nv_stream_t stream) {
  NV_CHECK_ARG((p.x || (p.part && p.nparts >= 1)) && p.nw && p.w && p.out, "%s: null pointer", name);
  NV_CHECK_ARG(dtype == NV_BF16 || dtype == NV_F16, "%s: bad dtype %d", name, dtype);
  NV_CHECK_ARG(p.M >= 0 && p.M <= 16 && p.K >= 128 && p.K <= 2048 && p.K % 128 == 0 && p.N > 0 && p.N % 16 == 0, "%s: M=%d N=%d K=%d", name,
               p.M, p.N, p.K);
  NV_CHECK_ARG((int64_t)p.M * (2 * p.K + 16) <= 48 * 1024, "%s: M=%d rows of K=%d do not fit a workgroup", name, p.M, p.K);
  NV_CHECK_ARG((p.res == nullptr) == (p.res_out == nullptr) && (!p.res || p.res != p.res_out),
               "%s: the residual goes with another buffer for the new one", name);
  NV_CHECK_ARG(((uintptr_t)p.x | (uintptr_t)p.part | (uintptr_t)p.res | (uintptr_t)p.res_out | (uintptr_t)p.nw | (uintptr_t)p.w) % 16 == 0 &&
                   ((uintptr_t)p.out | (uintptr_t)p.bias) % 8 == 0 && p.os % 4 == 0 && p.os >= (what == NG_SILU ? p.N / 2 : p.N),
               "%s: misaligned pointers or row strides", name);
  if (p.M == 0) return NV_OK;
  hipStream_t s = (hipStream_t)stream;
  if (what == NG_SILU)
    return dtype == NV_BF16 ? norm_gemm_go<bf16_t, 2, 4, NG_SILU>(p, ra, s) : norm_gemm_go<f16_t, 2, 4, NG_SILU>(p, ra, s);
  if (ra.D == 64)
    return dtype == NV_BF16 ? norm_gemm_go<bf16_t, 4, 2, NG_ROPE>(p, ra, s) : norm_gemm_go<f16_t, 4, 2, NG_ROPE>(p, ra, s);
  return dtype == NV_BF16 ? norm_gemm_go<bf16_t, 8, 1, NG_ROPE>(p, ra, s) : norm_gemm_go<f16_t, 8, 1, NG_ROPE>(p, ra, s);
}

}  // namespace

extern "C" int nv_norm_gemm_silu(const void* x, const float* partials, int num_partials, const void* residual, void* residual_out,
                                 const void* norm_w, float eps, const void* w_tiled, void* out, int64_t out_row_stride, int M, int N,
                                 int K, int dtype, nv_stream_t stream) {
  const NormGemmArgs p{(const uint16_t*)x, partials, num_partials, (const uint16_t*)residual, (uint16_t*)residual_out,
                       (const uint16_t*)norm_w, eps, (const u32x4*)w_tiled, nullptr, (uint16_t*)out, out_row_stride, M, N, K};
  return norm_gemm_launch("nv_norm_gemm_silu", p, RopeArgs{}, NG_SILU, dtype, stream);
}

extern "C" int nv_norm_gemm_rope_kv_store(const void* x, const float* partials, int num_partials, const void* residual,
                                          void* residual_out, const void* norm_w, float eps, const void* w_tiled, const void* bias,
                                          void* qkv, int64_t qkv_row_stride, int M, int K, const int64_t* positions,
                                          const float* cos_sin, const int32_t* slot_mapping, void* k_cache, void* v_cache,
                                          const void* q_norm_w, const void* k_norm_w, float head_eps, int H, int Hkv, int D, int dtype,
                                          nv_stream_t stream) {
  NV_CHECK_ARG(positions && cos_sin, "nv_norm_gemm_rope_kv_store: null pointer");
  NV_CHECK_ARG(D == 64 || D == 128, "nv_norm_gemm_rope_kv_store: head_dim %d not in {64, 128}", D);
  NV_CHECK_ARG(H >= 0 && Hkv >= 0 && H + Hkv > 0, "nv_norm_gemm_rope_kv_store: bad head counts");
  NV_CHECK_ARG((k_cache == nullptr) == (v_cache == nullptr) && (!k_cache || slot_mapping),
               "nv_norm_gemm_rope_kv_store: k_cache, v_cache and slot_mapping go together");
  NV_CHECK_ARG((q_norm_w == nullptr) == (k_norm_w == nullptr), "nv_norm_gemm_rope_kv_store: q_norm_w and k_norm_w go together");
  NV_CHECK_ARG((uintptr_t)cos_sin % 16 == 0 && ((uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)q_norm_w | (uintptr_t)k_norm_w) % 8 == 0,
               "nv_norm_gemm_rope_kv_store: misaligned pointer");
  RopeArgs ra;
  ra.positions = positions; ra.cos_sin = cos_sin; ra.slots = slot_mapping;
  ra.k_cache = (uint16_t*)k_cache; ra.v_cache = (uint16_t*)v_cache;
  ra.qn_w = (const uint16_t*)q_norm_w; ra.kn_w = (const uint16_t*)k_norm_w;
  ra.eps = head_eps; ra.H = H; ra.Hkv = Hkv; ra.D = D;
  const NormGemmArgs p{(const uint16_t*)x, partials, num_partials, (const uint16_t*)residual, (uint16_t*)residual_out,
                       (const uint16_t*)norm_w, eps, (const u32x4*)w_tiled, (const uint16_t*)bias, (uint16_t*)qkv, qkv_row_stride, M,
                       (H + 2 * Hkv) * D, K};
  return norm_gemm_launch("nv_norm_gemm_rope_kv_store", p, ra, NG_ROPE, dtype, stream);
}
