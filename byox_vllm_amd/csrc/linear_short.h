// nv_linear, many rows by a K of at most 128 bytes; included by linear.hip.
//
// Such a product (the up-projection of a low-rank pair) is bound by writing its result.  All of K is one or two fragments, so there
// is nothing to stage: a wavefront reads the fragments of 64 rows and CT tiles of 16 columns from memory at once and stores the
// results, four numbers of a row per lane; four wavefronts stand side by side.
// One tile per wavefront, as a rule: more of them are a longer chain of matrix instructions and epilogues in fewer workgroups (fp32,
// 300 rows by 256 columns of K = 16 with a soft cap: 13.8 us with four tiles, 5.5 with one, 8.6 in the kernel for any K).  Four,
// 256 columns per workgroup, where every CU has a workgroup all the same and the rows' fragments are two: they are read once for all
// the columns then (bf16, 16384 rows by 2048 columns of K = 64: 43.6 us with one tile, 34.3 with four; K = 32: 25.0 and 28.7).
// 16384 rows by 1000 columns of K = 32 in bf16, fp32 result, alone (21 us inside a layer, where the result finds other rows in the
// caches): 54.9 us on the LDS tiles, 20.5 with four tiles per wavefront, 16.3
// with one (67 MB: 4.1 TB/s).
#pragma once

template <typename T, typename TO, int EPI, int KF, int CT>      // KF fragments of K; CT tiles of 16 columns per wavefront
__global__ __launch_bounds__(256) void linear_short_kernel(LinArgs p) {
  typedef typename Frag<T>::type F;
  constexpr int KS = Frag<T>::KS, PER = Frag<T>::PER;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const int z = blockIdx.z, n0 = (blockIdx.x * 4 + wv) * (16 * CT);
  const int64_t m0 = (int64_t)blockIdx.y * 64;
  if (n0 >= p.N) return;
  const T* A = reinterpret_cast<const T*>(p.a) + z * p.a_bs;
  const T* W = reinterpret_cast<const T*>(p.w) + z * p.w_bs;
  const F none = {};
  F w[CT][KF], x[4][KF];
  // rows and columns that are not there repeat the first (never stored), pieces past K are zeros
#pragma unroll
  for (int f = 0; f < KF; ++f) {
    const int k = f * KS + PER * g;
    const bool in = k < p.K;
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      const int n = n0 + 16 * i + c < p.N ? n0 + 16 * i + c : n0;
      const F a = *reinterpret_cast<const F*>(W + (int64_t)n * p.w_rs + (in ? k : 0));
      w[i][f] = in ? a : none;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t s = m0 + 16 * j + c < p.M ? m0 + 16 * j + c : m0;
      const F b = *reinterpret_cast<const F*>(A + (int64_t)(p.a_rows ? p.a_rows[s] : s) * p.a_rs + (in ? k : 0));
      x[j][f] = in ? b : none;
    }
  }
  TO* O = reinterpret_cast<TO*>(p.out) + z * p.out_bs;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + z * p.bias_bs : nullptr;
  const bool whole = p.out_rs % 4 == 0 && p.out_bs % 4 == 0 && (uintptr_t)p.out % 16 == 0;
#pragma unroll
  for (int i = 0; i < CT; ++i) {
    const int n = n0 + 16 * i + 4 * g;
    if (n0 + 16 * i >= p.N) break;
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
      const float gate = EPI == EPI_ROW_GATE && !p.act ? sigmoid_f32(p.epi_ptr[s * p.epi_rs + z]) : 1.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[r] = acc[r] * rsc + b4[r];
        if constexpr (EPI == EPI_SOFTCAP || EPI == EPI_ACT) {
          if (n + r >= p.N) break;
          acc[r] = EPI == EPI_SOFTCAP ? p.epi_c * tanhf(acc[r] / p.epi_c) : unary_act(acc[r], p.act, p.epi_ptr, p.epi_c);
        }
        if constexpr (EPI == EPI_ROW_GATE)
          acc[r] *= p.act ? sigmoid_f32(p.epi_ptr[s * p.epi_rs + (int64_t)z * p.N + (n + r < p.N ? n + r : n0)]) : gate;
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
  const dim3 grid((unsigned)((p.N + 63) / 64), (unsigned)((p.M + 63) / 64), (unsigned)batch);
  switch (epi) {
    case EPI_NONE: linear_short_kernel<T, TO, EPI_NONE, KF, 1><<<grid, dim3(256), 0, s>>>(p); break;
    case EPI_SOFTCAP: linear_short_kernel<T, TO, EPI_SOFTCAP, KF, 1><<<grid, dim3(256), 0, s>>>(p); break;
    case EPI_ACT: linear_short_kernel<T, TO, EPI_ACT, KF, 1><<<grid, dim3(256), 0, s>>>(p); break;
    default: linear_short_kernel<T, TO, EPI_ROW_GATE, KF, 1><<<grid, dim3(256), 0, s>>>(p); break;
  }
}

template <typename T, typename TO>
void launch_short(const LinArgs& p, int epi, int batch, hipStream_t s) {
  if (p.K <= Frag<T>::KS) {
    launch_short_as<T, TO, 1>(p, epi, batch, s);
  } else if ((epi == EPI_NONE || epi == EPI_ROW_GATE) && p.N > 128 && ((p.M + 63) / 64) * ((p.N + 255) / 256) * batch >= 256) {
    const dim3 grid((unsigned)((p.N + 255) / 256), (unsigned)((p.M + 63) / 64), (unsigned)batch);
    if (epi == EPI_NONE) linear_short_kernel<T, TO, EPI_NONE, 2, 4><<<grid, dim3(256), 0, s>>>(p);
    else linear_short_kernel<T, TO, EPI_ROW_GATE, 2, 4><<<grid, dim3(256), 0, s>>>(p);
  } else {
    launch_short_as<T, TO, 2>(p, epi, batch, s);
  }
}
