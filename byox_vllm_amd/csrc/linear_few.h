// nv_linear, up to 64 rows per (group of) product; included by linear.hip.
//
// Such a launch is bound by how many weight loads are in flight.  A workgroup owns ONE 16-column tile and its NW wavefronts split K
// between them; the partial sums meet in LDS and wavefront i finishes the i-th sixteen rows.  Rows and columns that are not there read the first one's
// numbers instead (their products are never stored), so the loop carries no branch and the loads of a round are all under way
// together.  Tested per lane and piece, every load was waited for by itself (K 1024 and 2048, bf16 but for the second): 64 rows by
// 16 columns 11.4 us then, 4.2 now; by 1024 columns in fp32 24.3 and 7.1; by 2 x 8192 gated columns 65.6 and 29.5; 8 rows by the
// same 21.1 and 17.1 (67 MB: 3.9 TB/s).
//
// NSUB = 16-row sub-tiles of a workgroup; rows past them go to another one (blockIdx.y).
#pragma once

// one round of operands: 4 fragments of every row
template <typename T, bool GLU, int NS> struct FewRound {
  typename Frag<T>::type w[4], u[GLU ? 4 : 1], x[NS][4];
};

// K pieces from k on; `tail`: K ends inside the round, pieces past it are zeros
template <typename T, bool GLU, int NS>
__device__ __forceinline__ void few_load(FewRound<T, GLU, NS>& r, const T* wrow, const T* urow, const T* const (&arow)[NS], int k, int K,
                                         bool tail) {
  typedef typename Frag<T>::type F;
  constexpr int KS = Frag<T>::KS;
  if (!tail) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r.w[i] = *reinterpret_cast<const F*>(wrow + k + i * KS);
      if constexpr (GLU) r.u[i] = *reinterpret_cast<const F*>(urow + k + i * KS);
#pragma unroll
      for (int j = 0; j < NS; ++j) r.x[j][i] = *reinterpret_cast<const F*>(arow[j] + k + i * KS);
    }
    return;
  }
  const F none = {};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool in = k + i * KS < K;
    const int at = in ? k + i * KS : 0;
    const F w = *reinterpret_cast<const F*>(wrow + at);
    r.w[i] = in ? w : none;
    if constexpr (GLU) {
      const F u = *reinterpret_cast<const F*>(urow + at);
      r.u[i] = in ? u : none;
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const F x = *reinterpret_cast<const F*>(arow[j] + at);
      r.x[j][i] = in ? x : none;
    }
  }
}

template <typename T, bool GLU, int NS>
__device__ __forceinline__ void few_mma(const FewRound<T, GLU, NS>& r, f32x4* acc, f32x4* accu) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      acc[j] = mma(r.w[i], r.x[j][i], acc[j]);
      if constexpr (GLU) accu[j] = mma(r.u[i], r.x[j][i], accu[j]);
    }
}

// a wavefront's share [k_lo, k_hi) of K, both whole rounds but for the end of K; rows point at the lane's piece of k = 0
template <typename T, bool GLU, bool AHEAD, int NS>
__device__ __forceinline__ void few_sum(const T* wrow, const T* urow, const T* const (&arow)[NS], int k_lo, int k_hi, int K, int piece,
                                        f32x4* acc, f32x4* accu) {
  constexpr int ROUND = 4 * Frag<T>::KS;
  if (k_lo >= k_hi) return;
  const int lim = K - piece;        // this lane's pieces below here are inside K
  // AHEAD: a second round in flight.  Gate and up rows fill half again as many registers: there it costs more in wavefronts per SIMD
  // than it brings (64 rows over 16 experts of 6.3 MB: 30 us with it, 26 without; their down rows, of one kind: 16.4 with it, 18
  // without)
  if constexpr (!AHEAD) {
    for (int k = k_lo; k < k_hi; k += ROUND) {
      FewRound<T, GLU, NS> r;
      few_load<T, GLU, NS>(r, wrow, urow, arow, k, lim, k + ROUND > K);
      few_mma<T, GLU, NS>(r, acc, accu);
    }
    return;
  }
  FewRound<T, GLU, NS> a, b;
  few_load<T, GLU, NS>(a, wrow, urow, arow, k_lo, lim, k_lo + ROUND > K);
  for (int k = k_lo; k < k_hi; k += 2 * ROUND) {
    if (k + ROUND < k_hi) few_load<T, GLU, NS>(b, wrow, urow, arow, k + ROUND, lim, k + 2 * ROUND > K);
    few_mma<T, GLU, NS>(a, acc, accu);
    if (k + ROUND >= k_hi) break;
    if (k + 2 * ROUND < k_hi) few_load<T, GLU, NS>(a, wrow, urow, arow, k + 2 * ROUND, lim, k + 3 * ROUND > K);
    few_mma<T, GLU, NS>(b, acc, accu);
  }
}

// VEC: rows are 16-byte aligned and K a multiple of 16 bytes
template <typename T, typename TO, int EPI, int NSUB, int NW, bool VEC, bool AHEAD>
__global__ __launch_bounds__(64 * NW) void linear_few_kernel(LinArgs p) {
  typedef typename Frag<T>::type F;
  constexpr int KS = Frag<T>::KS, PER = Frag<T>::PER, ROUND = 4 * KS;
  constexpr bool GLU = EPI == EPI_GLU;
  __shared__ f32x4 part[GLU ? 2 : 1][NW][NSUB][64];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int z = blockIdx.z;
  int64_t lo = 0, hi = p.M;
  if (p.group_off) {
    lo = p.group_off[z];
    hi = p.group_off[z + 1];
  }
  lo += (int64_t)blockIdx.y * (16 * NSUB);
  if (lo >= hi) return;
  const int nsub = (int)((hi - lo + 15) / 16 < NSUB ? (hi - lo + 15) / 16 : NSUB);
  const int n0 = blockIdx.x * 16;
  const T* A = reinterpret_cast<const T*>(p.a) + z * p.a_bs;
  const T* W = reinterpret_cast<const T*>(p.w) + z * p.w_bs;
  const int n_here = n0 + c < p.N ? n0 + c : n0;
  const T* wrow = W + (int64_t)n_here * p.w_rs;
  const T* urow = GLU ? W + (int64_t)(p.N + n_here) * p.w_rs : nullptr;
  const T* arow[NSUB];
#pragma unroll
  for (int i = 0; i < NSUB; ++i) {
    const int64_t s = lo + 16 * i + c < hi ? lo + 16 * i + c : lo;
    arow[i] = A + (int64_t)(p.a_rows ? p.a_rows[s] : s) * p.a_rs;
  }
  // this wavefront's share of K, in whole rounds
  const int rounds = (p.K + ROUND - 1) / ROUND;
  const int k_lo = (rounds * wv) / NW * ROUND, k_hi = (rounds * (wv + 1)) / NW * ROUND;
  f32x4 acc[NSUB], accu[NSUB];
#pragma unroll
  for (int i = 0; i < NSUB; ++i) acc[i] = accu[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
    wrow += PER * g;
    if constexpr (GLU) urow += PER * g;
#pragma unroll
    for (int i = 0; i < NSUB; ++i) arow[i] += PER * g;
    if (NSUB > 1 && nsub == 1) {
      const T* const one[1] = {arow[0]};
      few_sum<T, GLU, AHEAD, 1>(wrow, urow, one, k_lo, k_hi, p.K, PER * g, acc, accu);
    } else {
      few_sum<T, GLU, AHEAD, NSUB>(wrow, urow, arow, k_lo, k_hi, p.K, PER * g, acc, accu);
    }
  } else if constexpr (NSUB == 1 && sizeof(T) == 4) {
    // numbers one by one: rows that are not there are not read, and a round's loads precede its products (one row by 777 columns of
    // K = 1030: 11.1 us so, 12.2 step by step with every lane reading; 64 rows 40.2 and 32.9, bf16 12.9 and 12.3: below)
    for (int k0 = k_lo; k0 < k_hi; k0 += ROUND) {
      F w[4], u[GLU ? 4 : 1], x[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int k = k0 + f * KS + PER * g;
        w[f] = load_frag<T>(wrow, k, p.K, p.vec_w);
        if constexpr (GLU) u[f] = load_frag<T>(urow, k, p.K, p.vec_w);
        x[f] = load_frag<T>(lo + c < hi ? arow[0] : nullptr, k, p.K, p.vec_a);
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        acc[0] = mma(w[f], x[f], acc[0]);
        if constexpr (GLU) accu[0] = mma(u[f], x[f], accu[0]);
      }
    }
  } else {
    for (int k0 = k_lo; k0 < k_hi; k0 += KS) {
      const int k = k0 + PER * g;
      const F w = load_frag<T>(wrow, k, p.K, p.vec_w);
      F u;
      if constexpr (GLU) u = load_frag<T>(urow, k, p.K, p.vec_w);
#pragma unroll
      for (int i = 0; i < NSUB; ++i) {
        if (i < nsub) {
          const F x = load_frag<T>(arow[i], k, p.K, p.vec_a);
          acc[i] = mma(w, x, acc[i]);
          if constexpr (GLU) accu[i] = mma(u, x, accu[i]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NSUB; ++i) {
    part[0][wv][i][lane] = acc[i];
    if constexpr (GLU) part[1][wv][i][lane] = accu[i];
  }
  __syncthreads();
  if (wv >= nsub) return;                 // wavefront i finishes sub-tile i
  TO* O = reinterpret_cast<TO*>(p.out) + z * p.out_bs;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + z * p.bias_bs : nullptr;
  const int64_t s = lo + 16 * wv + c;
  if (s >= hi) return;
  const float rsc = p.row_scale ? p.row_scale[s] : 1.0f;
  f32x4 sum = part[0][0][wv][lane], sumu = part[GLU ? 1 : 0][0][wv][lane];
#pragma unroll
  for (int w = 1; w < NW; ++w) {
    sum += part[0][w][wv][lane];
    if constexpr (GLU) sumu += part[1][w][wv][lane];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + 4 * g + r;
    if (n >= p.N) continue;
    float v = sum[r] * rsc;
    if (bias) v += ld_f32<T>(bias + n);
    if constexpr (GLU) {
      float u = sumu[r] * rsc;
      if (bias) u += ld_f32<T>(bias + p.N + n);
      v = glu_act(v, u, p.act, p.epi_c);
    } else if constexpr (EPI == EPI_SOFTCAP) {
      v = p.epi_c * tanhf(v / p.epi_c);
    } else if constexpr (EPI == EPI_ROW_GATE) {
      v *= sigmoid_f32(p.epi_ptr[s * p.epi_rs + (p.act ? (int64_t)z * p.N + n : z)]);
    } else if constexpr (EPI == EPI_ACT) {
      v = unary_act(v, p.act, p.epi_ptr, p.epi_c);
    }
    st_f32<TO>(O + s * p.out_rs + n, v);
  }
}

template <typename T, typename TO, int NSUB, int NW, bool VEC, bool AHEAD = VEC>
void launch_few_as(const LinArgs& p, int epi, dim3 grid, hipStream_t s) {
  grid.y = (unsigned)((p.M + 16 * NSUB - 1) / (16 * NSUB));
  switch (epi) {
    case EPI_NONE: linear_few_kernel<T, TO, EPI_NONE, NSUB, NW, VEC, AHEAD><<<grid, dim3(64 * NW), 0, s>>>(p); break;
    case EPI_GLU: linear_few_kernel<T, TO, EPI_GLU, NSUB, NW, VEC, false><<<grid, dim3(64 * NW), 0, s>>>(p); break;
    case EPI_SOFTCAP: linear_few_kernel<T, TO, EPI_SOFTCAP, NSUB, NW, VEC, AHEAD><<<grid, dim3(64 * NW), 0, s>>>(p); break;
    case EPI_ACT: linear_few_kernel<T, TO, EPI_ACT, NSUB, NW, VEC, AHEAD><<<grid, dim3(64 * NW), 0, s>>>(p); break;
    default: linear_few_kernel<T, TO, EPI_ROW_GATE, NSUB, NW, VEC, AHEAD><<<grid, dim3(64 * NW), 0, s>>>(p); break;
  }
}

// At most 64 rows.  As many sub-tiles per workgroup as leave the chip a workgroup per CU (each further workgroup reads the weights
// again): 64 rows by 1024 columns of K = 1024 take 24 us in 64 workgroups of four sub-tiles, 7 in 256 of one.  A group of rows
// seldom has more than 32 (two sub-tiles for up to 32 rows also where they leave a quarter of the CUs idle: 20 rows over 4 experts of
// 2 x 768 x 1024 7.4 us in single ones, 5.8; in 128 workgroups 6.3 and 8.0).  Sixteen wavefronts share K where even single
// sub-tiles leave CUs idle and every wavefront still gets a round (8 rows by 1024 columns of K = 1024 in fp32: 9.0 us on four, 6.3 on sixteen).  Of groups, few may have rows, and then the
// registers of a second round in flight cost more than it brings, unless K is long: with at most 8 rows in all (mean over routings of
// 1 to 8 rows, 16 experts of 2048 x 3072: 13.4 us with it, 11.7 without, 32 of 1024 x 1536 6.7 and 6.1), up to 16 rows per group below
// K = 3072 (16 rows over 64 experts of 512 x 2048: 12.4 and 10.2 us; 10 to 39 rows over 16 of 2048 x 3072 2 to 4 % longer without),
// of more rows below K = 1024, or 1536 from 32 groups on (64 over 64 experts of 2048 x 768: 32.5 and 26.5 us; 16 experts of 768 x 1024
// 3 to 12 % longer without, 32 of them 6 % shorter).
template <typename T, typename TO>
void launch_few(const LinArgs& p, int epi, int64_t total_rows, int batch, hipStream_t s) {
  const dim3 grid((unsigned)((p.N + 15) / 16), 1, (unsigned)batch);
  if (!p.vec_a || !p.vec_w || p.K % Frag<T>::PER) {
    if (p.M <= 16) launch_few_as<T, TO, 1, 4, false>(p, epi, grid, s);
    else launch_few_as<T, TO, 4, 4, false>(p, epi, grid, s);
    return;
  }
  constexpr int ROUND = 4 * Frag<T>::KS;
  const int64_t tiles = (int64_t)grid.x * batch;
  auto groups = [&](int nsub) { return tiles * ((p.M + 16 * nsub - 1) / (16 * nsub)); };
  if (p.M > 32 && !p.group_off && groups(4) >= 256) launch_few_as<T, TO, 4, 4, true>(p, epi, grid, s);
  else if (p.M > 16 && groups(2) >= (p.group_off && p.M <= 32 ? 192 : 256)) {
    if (p.group_off && p.K < (batch < 32 ? 8 : 12) * ROUND) launch_few_as<T, TO, 2, 4, true, false>(p, epi, grid, s);
    else launch_few_as<T, TO, 2, 4, true>(p, epi, grid, s);
  }
  else if (groups(1) <= 256 && p.K >= 16 * ROUND) launch_few_as<T, TO, 1, 16, true>(p, epi, grid, s);
  else if (p.group_off && (total_rows <= 8 || p.K < 24 * ROUND)) launch_few_as<T, TO, 1, 4, true, false>(p, epi, grid, s);
  else launch_few_as<T, TO, 1, 4, true>(p, epi, grid, s);
}
