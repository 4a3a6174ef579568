// Recurrences with a matrix state per head and one decay per head and token over prompts (the matrix memory of xLSTM, Mamba-2), thirty-two
// tokens at a time, their fp32 products on the 16-bit matrix instructions.  Included by chunk_scan.h, whose equations these are and whose
// kernel keeps steps of few tokens to a request (in_parts) and the decays per channel.
//
// What bounded these there: the fp32 matrix instructions, 37 % of the time, under which no vector instruction runs (those were half of it).  A
// number of fp32 is the sum of three of bf16, and a product the sum of six: a sixteen-by-sixteen tile of 32 numbers costs 96 cycles of the
// matrix cores for 256, under which the vector instructions of the SIMD's other wavefronts run, and chunks twice as long halve what a
// chunk costs whatever its length (decays of the state, its split, barriers).
//   * q and k are split once, by the lanes that stage them, and lie in LDS as parts; a value's weight in the state is on v, so that k
//     serves the scores and the state alike, read by rows for the one and through transposing reads for the other.
//   * The state stays in accumulators and is split where q meets it.  Channels lie in LDS in the order in which two of its tiles hold them,
//     which makes them the operand as they are.
//   * The three tiles of scores on and below the diagonal are three wavefronts', who form k q^T: a lane then holds four keys of one query.
// Measured: whole fp32 layers of 4 requests of about 1000 tokens, 32 heads of 128 x 64 433 and 380 us, 8 requests of 2048 tokens in bf16 1250 and
// 1040; exponential gates, 3 requests of 1500 tokens, 8 heads of 128 x 128 458 and 318, 64 of about 256 tokens, 64 x 128 229 and 210.  What
// bounds it now: waiting, 60 % of the wavefronts' time with two or three to a SIMD, at the chunk's two barriers and for its rows.
// Channel decays in this form (exponents taken from the chunk's middle, per-channel factors around the products) were 5 % slower than there:
// their second form for chunks that decay far takes the registers that keep two workgroups on a CU.
#pragma once

namespace chunk_scan {

constexpr int PTOK = 32;      // tokens of a chunk

// the last lane's x of each sixteen, in all of them
__device__ __forceinline__ uint32_t row_last(uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x15f, 0xf, 0xf, false); }
__device__ __forceinline__ float row_last(float x) { return __uint_as_float(row_last(__float_as_uint(x))); }
// running sums and maxima over the 32 lanes of each half
__device__ __forceinline__ double running_sum32(double x) {
  x = running_sum(x);
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  uint32_t lo, hi, none;
  rows_pair16(row_last((uint32_t)u), lo, none);
  rows_pair16(row_last((uint32_t)(u >> 32)), hi, none);
  const double first = __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
  return threadIdx.x & 16 ? x + first : x;
}
__device__ __forceinline__ float running_max32(float x) {
  x = running_max(x);
  float first, none;
  rows_pair16(row_last(x), first, none);
  return threadIdx.x & 16 ? fmaxf(x, first) : x;
}
__device__ __forceinline__ double from_lane31(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, 31), hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), 31);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// ---- fp32 products on the 16-bit matrix instructions: a number is the sum of three of bf16, and the six largest of the nine products of two
// such sums are added up in fp32 (off by less than 2^-25 of the product).
// The third part of a number below 2^-110 is below the least number of bf16, so q, k and the values enter times SCALE, which brings the last
// bit of every number of fp32 above that; the state and the scores are kept times SCALE^2 and what they form times SCALE^3.  Rows and states of
// 97 tokens, 128 x 64, positive numbers whose parts are as large as can be: 0.6 to 2.7e-7 of the norm off float64, wherever in fp32's range.
// Infinities and numbers too large for that have no parts.  They leave a result that is not finite, and then the workgroup walks its tokens
// again as chunk_scan_kernel does: its rows and states are that kernel's, and cost twice.
constexpr float SCALE = 16777216.0f, SCALE2 = SCALE * SCALE, SCALE3 = SCALE2 * SCALE;      // 2^24
struct Parts { u32x4 p[3]; };      // eight numbers
__device__ __forceinline__ void split2(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l) {
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(h) : "v"(x), "v"(y));
  x -= __uint_as_float(h << 16);
  y -= __uint_as_float(h & 0xffff0000u);
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(m) : "v"(x), "v"(y));
  x -= __uint_as_float(m << 16);
  y -= __uint_as_float(m & 0xffff0000u);
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(l) : "v"(x), "v"(y));
}
__device__ __forceinline__ Parts split8(const f32x4& a, const f32x4& b) {
  Parts r;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    uint32_t h, m, l;
    split2(a[2 * e], a[2 * e + 1], h, m, l);
    r.p[0][e] = h, r.p[1][e] = m, r.p[2][e] = l;
    split2(b[2 * e], b[2 * e + 1], h, m, l);
    r.p[0][2 + e] = h, r.p[1][2 + e] = m, r.p[2][2 + e] = l;
  }
  return r;
}
__device__ __forceinline__ f32x4 mma6(const Parts& a, const Parts& b, f32x4 acc) {
  constexpr int of_a[6] = {2, 0, 1, 1, 0, 0}, of_b[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int q = 0; q < 6; ++q) acc = mfma16(__builtin_bit_cast(bf16x8, a.p[of_a[q]]), __builtin_bit_cast(bf16x8, b.p[of_b[q]]), acc);
  return acc;
}

template <int MODE, int D, int NW>
struct PartsPlan {
  static constexpr int RB = 2 * D + 16, PLANE = PTOK * RB, PRB = 2 * PTOK + 16, PPLANE = PTOK * PRB;      // bytes
  static constexpr int Q = 0, K = 3 * PLANE, P = 6 * PLANE, F = P + 3 * PPLANE;                         // parts of q, of k, of the scores; doubles
  static constexpr int E = F + 2 * PTOK * 8;                                                             // floats from here on
  static constexpr int NQ = E + 3 * PTOK * 4, PN = NQ + (MODE == EXPGATE ? NW * PTOK * 4 : 0), END = PN + (MODE == EXPGATE ? 3 * PTOK * 4 : 0);
  static constexpr int WALK = (int)(lds_floats<D, NW>() * sizeof(float)), BYTES = END > WALK ? END : WALK;
};

template <int MODE, typename T, int D, int NW>
__global__ __launch_bounds__(64 * NW, D > 64 ? 2 : NW == 8 ? 4 : 3) void chunk_parts_kernel(Args p) {
  typedef PartsPlan<MODE, D, NW> L;
  constexpr int DT = D / 16, KT = D / 32, CPL = D / (2 * NW), U = CPL < 4 ? CPL : 4;
  constexpr bool EARLY = NW == 4 || D > 64;      // registers for values and gates asked for a chunk and a phase ahead of their use
  static_assert(CPL >= 2 && CPL <= 16 && NW % 4 == 0, "every lane stages whole pieces of channels");
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  extern __shared__ float4 lds4[];
  char* lds = reinterpret_cast<char*>(lds4);
  float* sf = reinterpret_cast<float*>(lds + L::E);      // [3][32] factor of q . S; EXPGATE exp(-m), SSD step size; a value's weight in the state
  double* sF = reinterpret_cast<double*>(lds + L::F);    // [32] log factor of a query's scores, [32] of a key's
  float* snq = reinterpret_cast<float*>(lds + L::NQ);    // [NW][32] EXPGATE: shares of n . q
  float* spn = reinterpret_cast<float*>(lds + L::PN);    // [3][32] EXPGATE: a score tile's sums over its keys
  const int h = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lc = lane & 15, lg = lane >> 4;
  const int tl = lane & 31, half = lane >> 5;
  int t0 = p.cu_q[b], t1 = p.cu_q[b + 1];
  const int t_end = t1, j = MODE != EXPGATE ? (int)blockIdx.z + (p.pass == 2 ? 1 : 0) : 0;
  if constexpr (MODE != EXPGATE) {
    if (p.runs > 1) {
      t0 += j * p.run_len;
      if (j + 1 < p.runs) t1 = min(t1, t0 + p.run_len);
    }
  }
  if (t1 <= t0) return;
  const bool emit = MODE == EXPGATE || j == 0 || p.pass == 2;      // else: the first pass of a later run, its end state alone
  if (!emit && t1 == t_end) return;      // which nobody needs behind the last run
  const int64_t run0 = ((int64_t)b * p.H + h) * p.runs;
  const int d = p.dim, vd = p.vdim, ch0 = (2 * wv + half) * CPL, col = 16 * wv + lc;
  const bool own = col < vd;             // a column of the state
  float* S_g = p.state + ((int64_t)p.slots[b] * p.H + h) * p.per_head;
  const bool fresh = p.past[b] == 0;
  const int hq = MODE == SSD ? h / p.heads_per_group : h;
  const f32x4 zero = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // per-head constants
  float bias_i = 0.0f, bias_f = 0.0f, rate = 0.0f, skip = 0.0f;
  const T* w0 = reinterpret_cast<const T*>(p.w0);
  const T* w1 = reinterpret_cast<const T*>(p.w1);
  if constexpr (MODE == EXPGATE) {
    if (w0) bias_i = ld_f32<T>(w0 + h);
    if (w1) bias_f = ld_f32<T>(w1 + h);
  }
  if constexpr (MODE == SSD) {
    bias_i = ld_f32<T>(w0 + h);
    rate = expf(ld_f32<T>(w1 + h));
    skip = ld_f32<T>(reinterpret_cast<const T*>(p.w2) + h);
  }

  f32x4 S[DT];
  const int s_at = own ? (4 * lg * vd + col) * 4 : ABSENT;       // rows from d on lie past the end
  {
    const auto r_s = rows_of(S_g, (MODE == EXPGATE || j == 0) && !fresh ? d * vd * 4 : 0);
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = SCALE2 * load_1(r_s, s_at + (16 * i + r) * vd * 4);
  }
  if (MODE != EXPGATE && p.pass == 2) {       // what the runs ahead left: S <- D_i S + E_i in turn
    for (int64_t run = run0; run < run0 + j; ++run) {
      const auto r_s = rows_of(p.ws_state + run * d * vd, d * vd * 4);
      const float f = p.ws_decay[run];
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = f * S[i][r] + SCALE2 * load_1(r_s, s_at + (16 * i + r) * vd * 4);
    }
  }
  double run_lf = 0.0;                   // SSD: the run's log decay
  float n0[CPL], m_run = 0.0f;           // EXPGATE: normaliser of this lane's channels, running maximum (every lane)
  if constexpr (MODE == EXPGATE) {
    const float* n_g = S_g + (int64_t)d * vd;
#pragma unroll
    for (int i = 0; i < CPL; ++i) n0[i] = (!fresh && ch0 + i < d) ? n_g[ch0 + i] : 0.0f;
    if (!fresh) m_run = n_g[d];
  }

  // byte offsets of this lane's numbers from a chunk's first row
  const int left = d - ch0, qk_at[2] = {(int)(tl * p.q_rs + ch0) * 4, (int)(tl * p.k_rs + ch0) * 4};
  // tokens 16 a + 4 lg + m: number 4 a + m of eight
  const uint32_t v_at = own ? (uint32_t)(4 * lg * p.v_rs + col) * 4 : ABSENT, g_at = own ? (uint32_t)(4 * lg * p.g_rs + col) * 4 : ABSENT,
                 o_at = own ? (uint32_t)(4 * lg * p.out_rs + col) * 4 : ABSENT;
  const uint32_t o_step = (uint32_t)p.out_rs * 4;
  auto row8 = [](int e) { return 16 * (e >> 2) + (e & 3); };
  float q[CPL], k[CPL];
#pragma unroll
  for (int i = 0; i < CPL; ++i) q[i] = 0.0f;
  // the next chunk's rows; the pointers advance with it
  const float *q_p = p.q + t0 * p.q_rs + hq * d, *k_p = p.k + t0 * p.k_rs + hq * d, *v_p = p.v + t0 * p.v_rs + h * vd;
  const float* g_p = MODE != EXPGATE ? p.g + t0 * p.g_rs + h * vd : nullptr;
  auto fetch = [&](int c0) {
    const int last = min(PTOK, t1 - c0) - 1;      // 64 rows lie within 2 GB (serves): 32 bits hold every size
    if (emit) load_n(q, rows_of(q_p, (last * (int)p.q_rs + d) * 4), qk_at[0], left);
    load_n(k, rows_of(k_p, (last * (int)p.k_rs + d) * 4), qk_at[1], left);
    q_p += PTOK * p.q_rs;
    k_p += PTOK * p.k_rs;
  };
  auto column8 = [&](f32x4 (&x)[2], const float* from, int last, int64_t rs, uint32_t at) {
    const auto r = rows_of(from, (last * (int)rs + vd) * 4);
    asm volatile("" : "+v"(at));         // its sums are formed here each time: kept, they take eight registers
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e >> 2][e & 3] = load_1(r, (int)(at + row8(e) * ((uint32_t)rs * 4)));
  };
  char* out_p = reinterpret_cast<char*>(p.out) + (t0 * p.out_rs + h * vd) * 4;
  // the gates of 64 tokens, one per lane, for two chunks in turn
  float s_in = 0.0f, f_in = 0.0f, s_gate = 0.0f, s_lf = 0.0f;
  auto fetch_gates = [&](int c0) {
    const int64_t last = min(64, t1 - c0) - 1;
    s_in = load_1(rows_of(p.s0 + (int64_t)c0 * p.s_rs + h, (last * p.s_rs + 1) * 4), (int)(lane * p.s_rs) * 4);
    if constexpr (MODE == EXPGATE)
      f_in = load_1(rows_of(p.s1 + (int64_t)c0 * p.s_rs + h, (last * p.s_rs + 1) * 4), (int)(lane * p.s_rs) * 4);
  };
  auto gates = [&]() {
    if constexpr (MODE == EXPGATE) {
      s_gate = p.c0 * tanhf((s_in + bias_i) / p.c0);
      s_lf = log_sigmoid_f32(p.c0 * tanhf((f_in + bias_f) / p.c0));
    } else {
      s_gate = softplus(s_in + bias_i);
      s_lf = -rate * s_gate;
    }
    s_lf = s_lf < LEAST ? LEAST : s_lf;
  };

  // A row of parts holds channel c at place 32 (c / 32) + 8 (c / 4 % 4) + 4 (c / 16 % 2) + c % 4: with that, two accumulator tiles of S ARE
  // the operand of q . S.
  auto place = [](int c) { return 32 * (c >> 5) + 8 * ((c >> 2) & 3) + 4 * ((c >> 4) & 1) + (c & 3); };
  auto put = [&](int at, const float (&x)[CPL]) {      // this lane's channels of token tl
#pragma unroll
    for (int u = 0; u < CPL; u += U) {
      char* to = lds + at + tl * L::RB + 2 * place(ch0 + u);
      uint32_t a[3], c[3];
      split2(x[u], x[u + 1], a[0], a[1], a[2]);
      if constexpr (U == 4) {
        split2(x[u + 2], x[u + 3], c[0], c[1], c[2]);
#pragma unroll
        for (int t = 0; t < 3; ++t) *reinterpret_cast<uint2*>(to + t * L::PLANE) = make_uint2(a[t], c[t]);
      } else {
#pragma unroll
        for (int t = 0; t < 3; ++t) *reinterpret_cast<uint32_t*>(to + t * L::PLANE) = a[t];
      }
    }
  };
  auto rows16 = [&](int at, int first, int kk) {      // 16 tokens from `first` on by channels 32 kk .. + 31
    Parts r;
    const char* from = lds + at + (first + lc) * L::RB + 64 * kk + 16 * lg;
#pragma unroll
    for (int t = 0; t < 3; ++t) r.p[t] = *reinterpret_cast<const u32x4*>(from + t * L::PLANE);
    return r;
  };
  auto columns16 = [&](int i) {      // k's channels 16 i .. + 15 by all tokens: those of a lane are 4 lg .. + 3 and 16 further
    Parts r;
    const char* from = lds + L::K + (4 * lg + (lc >> 2)) * L::RB + 64 * (i >> 1) + 16 * (lc & 3) + 8 * (i & 1);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(from + t * L::PLANE)));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(from + t * L::PLANE + 16 * L::RB)));
      r.p[t] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    return r;
  };
  auto score_place = [](int s) { return 8 * ((s >> 2) & 3) + 4 * (s >> 4) + (s & 3); };

  if (emit && tid < PTOK * 3) {       // queries of the first half see no key of the second: these places stay zeros
    if (tid % PTOK < 16) {
      char* row = lds + L::P + tid / PTOK * L::PPLANE + tid % PTOK * L::PRB;
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<uint2*>(row + 16 * g + 8) = make_uint2(0, 0);
    }
  }
  fetch_gates(t0);
  fetch(t0);
  f32x4 v[2];
  auto fetch_v = [&](int c0) {
    if (c0 < t1) column8(v, v_p, min(PTOK, t1 - c0) - 1, p.v_rs, v_at);
    v_p += PTOK * p.v_rs;
  };
  if constexpr (EARLY) fetch_v(t0);
  float finite = 0.0f;                   // NaN once a result was not
  int second = 0;
  for (int c0 = t0; c0 < t1; c0 += PTOK, second ^= 1) {
    const int n = min(PTOK, t1 - c0);
    f32x4 gate[2] = {zero, zero};
    if constexpr (!EARLY) fetch_v(c0);
    // -------- stage: lane = token, two lane groups and the wavefronts share the channels
    float whole = 1.0f, m_end = 0.0f;    // scalar decays: the state's factor over the chunk
    if (second == 0) {
      gates();
      if (c0 + 64 < t1) fetch_gates(c0 + 64);
    }
    const float lf = __shfl(s_lf, 32 * second + tl, 64);            // log decay
    const float in_gate = __shfl(s_gate, 32 * second + tl, 64);     // log input gate, or the step size
    const double Fd = running_sum32(tl < n ? (double)lf : 0.0);
    const double end = from_lane31(Fd);
    float w, rowf, m_t = 0.0f;
    if constexpr (MODE == EXPGATE) {
      // m_t = F_t + max(m ahead, max_(s <= t) (i_s - F_s))
      const double u = (double)in_gate - Fd;
      const float top = running_max32(tl < n ? (float)u : -INFINITY);
      m_t = (float)(Fd + (double)fmaxf(m_run, top));
      m_end = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(m_t), 31));
      w = tl < n ? expf((float)(end + u - (double)m_end)) : 0.0f;
      rowf = expf((float)(Fd + (double)m_run - (double)m_t));
      whole = expf((float)(end + (double)m_run - (double)m_end));
    } else {
      run_lf += end;
      w = in_gate * expf((float)(end - Fd));
      rowf = expf((float)Fd);
      whole = expf((float)end);
    }
    float nq = 0.0f;
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      q[i] *= SCALE * p.q_scale;
      k[i] *= SCALE * p.k_scale;
      if constexpr (MODE == EXPGATE) {
        nq += q[i] * n0[i];
        float a, c;
        rows_pair16(lanes_sum<16>(k[i] * w), a, c);
        n0[i] = whole * n0[i] + (a + c) * (1.0f / SCALE);
      }
    }
    if (emit) put(L::Q, q);
    put(L::K, k);
    if constexpr (MODE == EXPGATE) {
      float a, c;
      rows_pair32(nq, a, c);
      if (half == 0) snq[wv * PTOK + tl] = a + c;
    }
    if (tid < PTOK) {
      // the score of t and s takes exp(sF[t] + sF[32 + s]); in double, because the running sums cancel
      if constexpr (MODE == EXPGATE) {
        sF[tl] = Fd - (double)m_t;
        sF[PTOK + tl] = tl < n ? (double)in_gate - Fd : 0.0;
        sf[PTOK + tl] = expf(-m_t);
      } else {
        sF[tl] = Fd;
        sF[PTOK + tl] = -Fd;
        sf[PTOK + tl] = in_gate;
      }
      sf[tl] = rowf;
      sf[2 * PTOK + tl] = SCALE * w;
    }
    m_run = m_end;
    __syncthreads();
    // -------- scores k_s . q_t of the chunk: three tiles of 16 by 16, one to a wavefront
    if (emit && wv < 3) {
      const int sb = wv == 1 ? 16 : 0, ta = wv == 0 ? 0 : 16;
      f32x4 acc = zero;
#pragma unroll
      for (int kk = 0; kk < KT; ++kk) acc = mma6(rows16(L::K, sb, kk), rows16(L::Q, ta, kk), acc);
      const int t = ta + lc;
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int s = sb + 4 * lg + r;
        if (s > t) {
          acc[r] = 0.0f;
        } else {
          acc[r] *= expf((float)(sF[t] + sF[PTOK + s]));
          if constexpr (MODE == SSD) acc[r] *= sf[PTOK + s];
        }
        sum += acc[r];
      }
      uint32_t a[3], c[3];
      split2(acc[0], acc[1], a[0], a[1], a[2]);
      split2(acc[2], acc[3], c[0], c[1], c[2]);
#pragma unroll
      for (int i = 0; i < 3; ++i)
        *reinterpret_cast<uint2*>(lds + L::P + i * L::PPLANE + t * L::PRB + 2 * score_place(sb + 4 * lg)) = make_uint2(a[i], c[i]);
      if constexpr (MODE == EXPGATE) {
        float x, y;
        rows_pair16(sum, x, y);
        rows_pair32(x + y, x, y);
        if (lg == 0) spn[wv * PTOK + t] = x + y;
      }
    }
    // what the results need of this chunk's staging: the next one's overwrites it
    float ahead = 0.0f, row_ahead = 0.0f, floor_t = 0.0f;
    if constexpr (MODE == EXPGATE) {
#pragma unroll
      for (int w = 0; w < NW; ++w) ahead += snq[w * PTOK + tl];
      row_ahead = sf[tl];
      floor_t = sf[PTOK + tl];
    }
    if (c0 + PTOK < t1) fetch(c0 + PTOK);
    if constexpr (MODE != EXPGATE && EARLY) {
      if (emit) column8(gate, g_p, n - 1, p.g_rs, g_at);
      g_p += PTOK * p.g_rs;
    }
    // -------- what the state ahead of the chunk contributes
    f32x4 o[2] = {zero, zero};
    if (emit) {
#pragma unroll
      for (int kk = 0; kk < KT; ++kk) {
        const Parts s = split8(S[2 * kk], S[2 * kk + 1]);
#pragma unroll
        for (int a = 0; a < 2; ++a) o[a] = mma6(rows16(L::Q, 16 * a, kk), s, o[a]);
        __builtin_amdgcn_sched_barrier(0);       // a step's operands at a time: registers
      }
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const f32x4 f = at4(sf + 16 * a + 4 * lg);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[a][r] *= f[r];
      }
    }
    // -------- the state behind the chunk
    Parts vp;
    {
      f32x4 x[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const f32x4 w = at4(sf + 2 * PTOK + 16 * a + 4 * lg);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[a][r] = v[a][r] * w[r];
      }
      const Parts vw = split8(x[0], x[1]);
#pragma unroll
      for (int i = 0; i < DT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] *= whole;
        S[i] = mma6(columns16(i), vw, S[i]);
        if (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
      vp = split8(v[0] * SCALE, v[1] * SCALE);
    }
    if constexpr (MODE != EXPGATE && !EARLY) {
      if (emit) column8(gate, g_p, n - 1, p.g_rs, g_at);
      g_p += PTOK * p.g_rs;
    }
    if (EARLY && (MODE != SSD || !emit)) fetch_v(c0 + PTOK);
    __syncthreads();                     // the scores are there; the parts of q and k may be overwritten
    if (!emit) continue;
    // -------- what the chunk's own tokens contribute
    // A score of a later token is 0, but 0 times an infinity or a NaN is not: with such a value in the chunk the tokens are walked again.
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      Parts P;
#pragma unroll
      for (int t = 0; t < 3; ++t) P.p[t] = *reinterpret_cast<const u32x4*>(lds + L::P + t * L::PPLANE + (16 * a + lc) * L::PRB + 16 * lg);
      o[a] = mma6(P, vp, o[a]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        finite = fmaf(o[a][r], 0.0f, finite);
        o[a][r] *= 1.0f / SCALE3;
      }
    }
    const auto ro = rows_of(out_p, ((n - 1) * (int)p.out_rs + vd) * 4);
    uint32_t out_at = o_at;
    asm volatile("" : "+v"(out_at));
    out_p += PTOK * p.out_rs * 4;
    if constexpr (MODE == EXPGATE) {
      // n_t . q_t of token tl: its scores and the normaliser ahead of the chunk
      const float nq = (tl < 16 ? spn[tl] : spn[PTOK + tl] + spn[2 * PTOK + tl]) * (1.0f / SCALE2) + ahead * (1.0f / SCALE) * row_ahead;
      finite = fmaf(nq, 0.0f, finite);
      const float under = 1.0f / (fmaxf(fabsf(nq), floor_t) + 1e-6f);
#pragma unroll
      for (int e = 0; e < 8; ++e) store_1<float>(ro, (int)(out_at + row8(e) * o_step), o[e >> 2][e & 3] * __shfl(under, 4 * lg + row8(e), 64));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        store_1<float>(ro, (int)(out_at + row8(e) * o_step), (o[e >> 2][e & 3] + skip * v[e >> 2][e & 3]) * silu(gate[e >> 2][e & 3]));
      if constexpr (EARLY) fetch_v(c0 + PTOK);
    }
  }
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) finite = fmaf(S[i][r], 0.0f, finite);
  if constexpr (MODE == EXPGATE) {
#pragma unroll
    for (int i = 0; i < CPL; ++i) finite = fmaf(n0[i], 0.0f, finite);
  }
  int* again = reinterpret_cast<int*>(lds);
  __syncthreads();                       // everybody is through with the last chunk
  if (lane == 0) again[wv] = 0;
  if (finite != 0.0f) again[wv] = 1;
  __syncthreads();
  int any = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) any |= again[w];
  if (__builtin_expect(any, 0)) {
    __syncthreads();
    uint64_t args = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    int thread = threadIdx.x;
    asm volatile("" : "+s"(args), "+v"(thread));       // formed anew from here on: kept until here, 10 to 20 registers in the loop above
    chunk_walk<MODE, T, D, NW>(*reinterpret_cast<const Args*>(args), thread);
    return;
  }
  if (own) {
    const bool to_slot = emit && t1 == t_end, to_ws = MODE != EXPGATE && p.runs > 1 && p.pass == 1 && t1 < t_end;
    float* E = p.ws_state + (run0 + j) * d * vd;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + 4 * lg + r;
        if (row < d) {
          const float x = S[i][r] * (1.0f / SCALE2);
          if (to_slot) S_g[(int64_t)row * vd + col] = x;
          if (to_ws) E[(int64_t)row * vd + col] = x;
        }
      }
    if (MODE == SSD && to_ws && tid == 0) p.ws_decay[run0 + j] = expf((float)run_lf);
  }
  if constexpr (MODE == EXPGATE) {
    for (int c = 0; c < (vd + 63) / 64; ++c) {
      float* n_g = S_g + (int64_t)d * vd + (int64_t)c * (d + 1);
#pragma unroll
      for (int i = 0; i < CPL; ++i)
        if (tl == 0 && ch0 + i < d) n_g[ch0 + i] = n0[i];
      if (tid == 0) n_g[d] = m_run;
    }
  }
}

}  // namespace chunk_scan
