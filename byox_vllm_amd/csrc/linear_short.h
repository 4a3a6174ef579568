// nv_linear, many rows by a K of at most 128 bytes; included by linear.hip.
//
// Such a product (the up-projection of a low-rank pair) is bound by writing its result.  All of K is one or two fragments, so there
// is nothing to stage: a wavefront reads the fragments of 64 rows and 64 columns from memory at once and stores sixteen tiles,
// four numbers of a row per lane; four wavefronts stand side by side, so a workgroup writes 1 KB (fp32) of each of its 64 rows.
// 16384 rows by 1024 columns of K = 32 in bf16, fp32 result: 42 us on the LDS tiles with
// operands in the caches, 14 here (67 MB: 4.9 TB/s); 200 rows by the same 14.4 and 5.2.
#pragma once

template <typename T, typename TO, int EPI, int KF>      // KF fragments of K
__global__ __launch_bounds__(256) void linear_short_kernel(LinArgs p) {
  typedef typename Frag<T>::type F;
  constexpr int KS = Frag<T>::KS, PER = Frag<T>::PER;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const int z = blockIdx.z, n0 = blockIdx.x * 256 + wv * 64;
  const int64_t m0 = (int64_t)blockIdx.y * 64;
  if (n0 >= p.N) return;
  const T* A = reinterpret_cast<const T*>(p.a) + z * p.a_bs;
  const T* W = reinterpret_cast<const T*>(p.w) + z * p.w_bs;
  const F none = {};
  F w[4][KF], x[4][KF];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int f = 0; f < KF; ++f) {
      // rows and columns that are not there repeat the first (never stored), pieces past K are zeros
      const int k = f * KS + PER * g, n = n0 + 16 * i + c < p.N ? n0 + 16 * i + c : n0;
      const int64_t s = m0 + 16 * i + c < p.M ? m0 + 16 * i + c : m0;
      const bool in = k < p.K;
      const F a = *reinterpret_cast<const F*>(W + (int64_t)n * p.w_rs + (in ? k : 0));
      const F b = *reinterpret_cast<const F*>(A + (int64_t)(p.a_rows ? p.a_rows[s] : s) * p.a_rs + (in ? k : 0));
      w[i][f] = in ? a : none;
      x[i][f] = in ? b : none;
    }
  TO* O = reinterpret_cast<TO*>(p.out) + z * p.out_bs;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + z * p.bias_bs : nullptr;
  const bool whole = p.out_rs % 4 == 0 && p.out_bs % 4 == 0 && (uintptr_t)p.out % 16 == 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + 16 * i + 4 * g;
    f32x4 b4 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (bias)
#pragma unroll
      for (int r = 0; r < 4; ++r) b4[r] = n + r < p.N ? ld_f32<T>(bias + n + r) : 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int f = 0; f < KF; ++f) acc = mma(w[i][f], x[j][f], acc);
      const int64_t s = m0 + 16 * j + c;
      if (s >= p.M) continue;
      const float rsc = p.row_scale ? p.row_scale[s] : 1.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[r] = acc[r] * rsc + b4[r];
        if constexpr (EPI == EPI_SOFTCAP) acc[r] = p.epi_c * tanhf(acc[r] / p.epi_c);
        if constexpr (EPI == EPI_ACT) acc[r] = unary_act(acc[r], p.act, p.epi_ptr, p.epi_c);
        if constexpr (EPI == EPI_ROW_GATE)
          acc[r] *= sigmoid_f32(p.epi_ptr[s * p.epi_rs + (p.act ? (int64_t)z * p.N + (n + r < p.N ? n + r : n0) : z)]);
      }
      TO* o = O + s * p.out_rs + n;
      if (whole && n + 3 < p.N) {
        if constexpr (sizeof(TO) == 4) *reinterpret_cast<f32x4*>(o) = acc;
        else *reinterpret_cast<uint2*>(o) = Pack4<TO>::narrow(acc);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < p.N) st_f32<TO>(o + r, acc[r]);
      }
    }
  }
}

template <typename T, typename TO, int KF>
void launch_short_as(const LinArgs& p, int epi, int batch, hipStream_t s) {
  const dim3 grid((unsigned)((p.N + 255) / 256), (unsigned)((p.M + 63) / 64), (unsigned)batch);
  switch (epi) {
    case EPI_NONE: linear_short_kernel<T, TO, EPI_NONE, KF><<<grid, dim3(256), 0, s>>>(p); break;
    case EPI_SOFTCAP: linear_short_kernel<T, TO, EPI_SOFTCAP, KF><<<grid, dim3(256), 0, s>>>(p); break;
    case EPI_ACT: linear_short_kernel<T, TO, EPI_ACT, KF><<<grid, dim3(256), 0, s>>>(p); break;
    default: linear_short_kernel<T, TO, EPI_ROW_GATE, KF><<<grid, dim3(256), 0, s>>>(p); break;
  }
}

template <typename T, typename TO>
void launch_short(const LinArgs& p, int epi, int batch, hipStream_t s) {
  if (p.K <= Frag<T>::KS) launch_short_as<T, TO, 1>(p, epi, batch, s);
  else launch_short_as<T, TO, 2>(p, epi, batch, s);
}
