// Recurrences with a matrix state per head over prompts, sixteen tokens at a time on the fp32 matrix cores:
//
//   S_t = decay_t S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t        S [dim, vdim]
//
// with a decay per key channel (gated linear attention) or per head and token (Mamba-2, the matrix memory of xLSTM).  For
// the tokens t, s of a chunk, F the running sum of log decays inside it and S the state ahead of it:
//
//   o_t = exp(F_t) q_t . S + sum_(s <= t) (q_t . k_s exp(F_t - F_s)) v_s,    S <- exp(F_end) S + sum_s exp(F_end - F_s) k_s v_s^T
//
// Every exponent is at most 0, so nothing leaves the range of fp32, whatever the decays.  (Channel decays reach the scores
// as two factors, exp(F_t) on q and exp(-F_s) on k, while the chunk's decays stay above 2^-SCORE_RANGE; chunks that decay
// further take them term by term, exp(F_t - F_s) on each product.)
//
// A workgroup owns one (head, request); wavefront w owns the 16 state columns from 16 w on and keeps their S in MFMA
// accumulators for the whole prompt.  Sixteen tokens per chunk because the state then never leaves the registers: with step
// m of a four-number sum taking the numbers {16 kk + 4 g + m}, an accumulator of S (rows 4 g + m of tile kk, column c) IS
// the operand fragment of the next chunk's q . S.  The serial chain of a prompt is one chunk of about 40 matrix
// instructions per wavefront; the walk it replaces is bound by the issue of 2 dim FMAs per column and token.
// Prompts with a decay per head and token take chunk_parts.h instead, but for steps of few tokens to a request.
//
// Measured against that walk: channel decays, 8 x 2048 tokens, 16 heads of 64 x 128: 2560 us then, 316 now (542 MB of operands:
// 1.7 TB/s); exponential gates, 64 requests of about 256 tokens, 8 heads of 64 x 128: 477 and 82; one decay per token, 4 requests
// of about 1000 tokens, 32 heads of 128 x 64: 645 and 136.  What bounds it now, with two workgroups on a CU: matrix
// instructions 37 % of the time and the vector instructions around them half, next to no overlap of the two (32768 tokens: 400 us;
// a third fewer vector instructions gained 4 %).  Registers are held to 128 up to 64 channels, and for wide
// state-space heads, for the sake of the second workgroup.
#pragma once
#include "anyt.h"
#include "lds_limit.h"

namespace chunk_scan {

enum Mode { GLA = 0, EXPGATE = 1, SSD = 2 };

struct Args {
  const float* q;        // token 0's rows; head h at h * q_hs (SSD: the head's group)
  const float* k;
  int64_t q_rs, k_rs;
  const float* v;        // [tokens, v_rs], head h at h * vdim
  int64_t v_rs;
  const float* g;        // GLA, SSD: gate logits, head h at h * vdim
  int64_t g_rs;
  const float* s0;       // GLA: decay logits per channel [tokens, s_rs]; EXPGATE: input-gate logits; SSD: raw step sizes
  const float* s1;       // EXPGATE: forget-gate logits
  int64_t s_rs;
  const void* w0;        // GLA: norm weight [vdim]; EXPGATE: input-gate bias [H] or null; SSD: dt_bias [H]
  const void* w1;        // EXPGATE: forget-gate bias [H] or null; SSD: A_log [H]
  const void* w2;        // SSD: D [H]
  float* state;          // [slots, H, per_head]
  int64_t per_head;
  const int32_t* cu_q;
  const int32_t* past;
  const int32_t* slots;
  void* out;             // GLA: storage type; else fp32
  int64_t out_rs;
  int H, heads_per_group, dim, vdim;
  float q_scale, k_scale, c0, eps;      // c0: GLA 1 / tau, EXPGATE the gate cap
  // GLA, SSD: long prompts of few requests as runs of run_len tokens side by side, in two passes (see launch_runs)
  float* ws_state;       // [B * H * runs][dim * vdim] state at the end of each run
  float* ws_decay;       // SSD [B * H * runs], GLA [B * H * runs][dim]: product of the run's decays
  int runs, run_len, pass;
  int in_parts;          // EXPGATE, SSD: the kernel of chunk_parts.h
};

constexpr int TOK = 16, CP = 20;
constexpr float SCORE_RANGE = 24.0f;     // log2; a running sum of this size still leaves its exponential 1e-6 exact
constexpr float LEAST = -1e4f;           // a log decay below this is a decay of 0 all the same; keeps differences finite

template <int D, int NW>
constexpr size_t lds_floats() {
  return 2 * (2 * TOK * (D + 4) + (size_t)D * CP + D + 6 * TOK) + (size_t)(D / 16 < 2 ? 2 : D / 16) * TOK * CP + 3 * NW * TOK +
         2 * NW;
}

// Rows are read and written through buffer descriptors over the chunk's tokens: tokens and channels that are not there lie
// past the end and read as zeros (writes are dropped), so no access needs a branch or a clamped address.
constexpr int ABSENT = 0x7ff00000;       // an offset past every end, with room for what is added to it
static_assert((int64_t)ABSENT + 128 * 128 * 4 <= INT32_MAX, "an absent state column's rows stay within an int");
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ float load_1(__amdgpu_buffer_rsrc_t r, int at) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
}
template <int N> __device__ __forceinline__ void load_n(float (&x)[N], __amdgpu_buffer_rsrc_t r, int at, int left) {
  // `left`: channels from here to the head's end, a multiple of 4
  if constexpr (N == 1) {
    x[0] = load_1(r, left > 0 ? at : ABSENT);
  } else if constexpr (N == 2) {
    const u32x2 u = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, left > 0 ? at : ABSENT, 0, 0));
    x[0] = __uint_as_float(u[0]);
    x[1] = __uint_as_float(u[1]);
  } else {
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const u32x4 u = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, left > i ? at + 4 * i : ABSENT, 0, 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) x[i + e] = __uint_as_float(u[e]);
    }
  }
}
template <typename T> __device__ __forceinline__ void store_1(__amdgpu_buffer_rsrc_t r, int at, float v) {
  if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, (T)v), r, at, 0, 0);
  else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, at, 0, 0);
}

template <int N> __device__ __forceinline__ void store_n(float* p, const float (&r)[N]) {
  constexpr int U = N < 4 ? N : 4;
#pragma unroll
  for (int i = 0; i < N; i += U) {
    if constexpr (U == 4) *reinterpret_cast<f32x4*>(p + i) = f32x4{r[i], r[i + 1], r[i + 2], r[i + 3]};
    else if constexpr (U == 2) *reinterpret_cast<float2*>(p + i) = make_float2(r[i], r[i + 1]);
    else p[i] = r[i];
  }
}

// lane l of each sixteen takes x of lane l - N, lanes below N take `none`
template <int N> __device__ __forceinline__ float from_below(float x, float none) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(none), (int)__float_as_uint(x), 0x110 + N,
                                                              0xf, 0xf, false));
}
template <int N> __device__ __forceinline__ double from_below(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x110 + N, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x110 + N, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ float running_sum(float x) {
  x += from_below<1>(x, 0.0f);
  x += from_below<2>(x, 0.0f);
  x += from_below<4>(x, 0.0f);
  return x + from_below<8>(x, 0.0f);
}
__device__ __forceinline__ double running_sum(double x) {
  x += from_below<1>(x);
  x += from_below<2>(x);
  x += from_below<4>(x);
  return x + from_below<8>(x);
}
__device__ __forceinline__ float running_max(float x) {
  x = fmaxf(x, from_below<1>(x, -INFINITY));
  x = fmaxf(x, from_below<2>(x, -INFINITY));
  x = fmaxf(x, from_below<4>(x, -INFINITY));
  return fmaxf(x, from_below<8>(x, -INFINITY));
}
__device__ __forceinline__ f32x4 at4(const float* q) { return *reinterpret_cast<const f32x4*>(q); }
__device__ __forceinline__ f32x4 step4(const f32x4& a, const f32x4& x, f32x4 acc) {
#pragma unroll
  for (int m = 0; m < 4; ++m) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], x[m], acc, 0, 0, 0);
  return acc;
}
__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))); }
// The channel decays' two transcendentals per key number, as library calls, took more instructions than everything else.
// log2(sigmoid(z)) = min(z, 0) log2(e) - log2(1 + e), e = exp(-|z|), by ln(1 + e) = 2 artanh(e / (2 + e)): the argument is at
// most 1/3, seven terms of the series leave 2e-8 relative, also where the decay is close to 1.
__device__ __forceinline__ float log2_sigmoid(float z) {
  constexpr float L2E = 1.4426950408889634f;
  const float e = __builtin_amdgcn_exp2f(-fabsf(z) * L2E), s = e * __builtin_amdgcn_rcpf(2.0f + e), y = s * s;
  float r = fmaf(y, 1.0f / 13.0f, 1.0f / 11.0f);
  r = fmaf(y, r, 1.0f / 9.0f);
  r = fmaf(y, r, 1.0f / 7.0f);
  r = fmaf(y, r, 1.0f / 5.0f);
  r = fmaf(y, r, 1.0f / 3.0f);
  r = fmaf(y * s, r, s);
  return fminf(z, 0.0f) * L2E - 2.0f * L2E * r;
}
// 1 / x to within a rounding: the hardware's estimate and one Newton step (x is finite and not tiny here)
__device__ __forceinline__ float inverse(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ float silu(float z) {
  const float e = __builtin_amdgcn_exp2f(fminf(-z * 1.4426950408889634f, 126.0f));
  return z * inverse(1.0f + e);
}

template <int MODE, typename T, int D, int NW>
__device__ __forceinline__ void chunk_walk(const Args& p, int tid) {
  constexpr int DP = D + 4, DT = D / 16, CPL = D / (4 * NW), NP = DT < 2 ? 2 : DT;
  static_assert(CPL >= 1 && CPL <= 8 && NW % 4 == 0 && D * CP >= TOK * DP, "every lane stages whole channels");
  constexpr int BUF = 2 * TOK * DP + D * CP + D + 6 * TOK;
  extern __shared__ float4 lds4[];
  float* lds = reinterpret_cast<float*>(lds4);
  float* sp = lds + 2 * BUF;             // [NP][16][CP] score partials by 16 channels
  float* sred = sp + NP * TOK * CP;      // [NW][16] sums across wavefronts
  float* snq = sred + NW * TOK;          // [2][NW][16] EXPGATE: shares of n . q
  float* sflag = snq + 2 * NW * TOK;     // [2][NW] GLA: this wavefront's channels decay out of the scores' range
  const int h = blockIdx.x, b = blockIdx.y;
  const int lane = tid & 63, wv = tid >> 6, lc = lane & 15, lg = lane >> 4;
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
  const int d = p.dim, vd = p.vdim, ch0 = (4 * wv + lg) * CPL, col = 16 * wv + lc;
  const bool own = col < vd;             // a column of the state
  float* S_g = p.state + ((int64_t)p.slots[b] * p.H + h) * p.per_head;
  const bool fresh = p.past[b] == 0;
  const int hq = MODE == SSD ? h / p.heads_per_group : h;
  const f32x4 zero = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // per-head constants
  float nw = 0.0f, bias_i = 0.0f, bias_f = 0.0f, rate = 0.0f, skip = 0.0f;
  const T* w0 = reinterpret_cast<const T*>(p.w0);
  const T* w1 = reinterpret_cast<const T*>(p.w1);
  if constexpr (MODE == GLA) nw = own ? ld_f32<T>(w0 + col) : 0.0f;
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
      for (int r = 0; r < 4; ++r) S[i][r] = load_1(r_s, s_at + (16 * i + r) * vd * 4);
  }
  if (MODE != EXPGATE && p.pass == 2) {       // what the runs ahead left: S <- D_i S + E_i in turn
    for (int64_t run = run0; run < run0 + j; ++run) {
      const auto r_s = rows_of(p.ws_state + run * d * vd, d * vd * 4);
      const auto r_d = rows_of(p.ws_decay + (MODE == GLA ? run * d : run), MODE == GLA ? d * 4 : 4);
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        float f[4];
        if constexpr (MODE == GLA) load_n(f, r_d, (16 * i + 4 * lg) * 4, d - 16 * i - 4 * lg);
        else f[0] = f[1] = f[2] = f[3] = load_1(r_d, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = f[r] * S[i][r] + load_1(r_s, s_at + (16 * i + r) * vd * 4);
      }
    }
  }
  double run_lf = 0.0;                   // SSD: the run's log decay
  float run_e[MODE == GLA ? CPL : 1];    // GLA: the run's decays of this lane's channels
#pragma unroll
  for (int i = 0; i < (MODE == GLA ? CPL : 1); ++i) run_e[i] = 1.0f;
  float n0[CPL], m_run = 0.0f;           // EXPGATE: normaliser of this lane's channels, running maximum (every lane)
  if constexpr (MODE == EXPGATE) {
    const float* n_g = S_g + (int64_t)d * vd;
#pragma unroll
    for (int i = 0; i < CPL; ++i) n0[i] = (!fresh && ch0 + i < d) ? n_g[ch0 + i] : 0.0f;
    if (!fresh) m_run = n_g[d];
  }

  // byte offsets of this lane's numbers from a chunk's first row
  const int left = d - ch0, qk_at[3] = {(int)(lc * p.q_rs + ch0) * 4, (int)(lc * p.k_rs + ch0) * 4, (int)(lc * p.s_rs + ch0) * 4};
  int v_at[4], g_at[4], o_at[4];
  constexpr int OUT = MODE == GLA ? (int)sizeof(T) : 4;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    v_at[m] = own ? (int)((4 * lg + m) * p.v_rs + col) * 4 : ABSENT;
    g_at[m] = own ? (int)((4 * lg + m) * p.g_rs + col) * 4 : ABSENT;
    o_at[m] = own ? (int)((4 * lg + m) * p.out_rs + col) * OUT : ABSENT;
  }
  float q[CPL], k[CPL], z[MODE == GLA ? CPL : 1], vn[4], gn[4];
#pragma unroll
  for (int i = 0; i < CPL; ++i) q[i] = 0.0f;
#pragma unroll
  for (int m = 0; m < 4; ++m) gn[m] = 0.0f;
  // the next chunk's rows; the pointers advance with it
  const float *q_p = p.q + t0 * p.q_rs + hq * d, *k_p = p.k + t0 * p.k_rs + hq * d, *v_p = p.v + t0 * p.v_rs + h * vd;
  const float* g_p = MODE != EXPGATE ? p.g + t0 * p.g_rs + h * vd : nullptr;
  const float* z_p = MODE == GLA ? p.s0 + t0 * p.s_rs + h * d : nullptr;
  auto fetch = [&](int c0) {
    const int last = min(TOK, t1 - c0) - 1;      // 64 rows within 2 GB: 32 bits hold every size
    if (emit) load_n(q, rows_of(q_p, (last * (int)p.q_rs + d) * 4), qk_at[0], left);
    load_n(k, rows_of(k_p, (last * (int)p.k_rs + d) * 4), qk_at[1], left);
    if constexpr (MODE == GLA) load_n(z, rows_of(z_p, (last * (int)p.s_rs + d) * 4), qk_at[2], left);
    const auto rv = rows_of(v_p, (last * (int)p.v_rs + vd) * 4);
#pragma unroll
    for (int m = 0; m < 4; ++m) vn[m] = load_1(rv, v_at[m]);
    if (MODE != EXPGATE && emit) {
      const auto rg = rows_of(g_p, (last * (int)p.g_rs + vd) * 4);
#pragma unroll
      for (int m = 0; m < 4; ++m) gn[m] = load_1(rg, g_at[m]);
    }
    q_p += TOK * p.q_rs;
    k_p += TOK * p.k_rs;
    v_p += TOK * p.v_rs;
    if constexpr (MODE != EXPGATE) g_p += TOK * p.g_rs;
    if constexpr (MODE == GLA) z_p += TOK * p.s_rs;
  };
  char* out_p = reinterpret_cast<char*>(p.out) + (t0 * p.out_rs + h * vd) * OUT;
  const float inv_vd = 1.0f / (float)vd;
  // the gates of 64 tokens, one per lane, for four chunks in turn
  float s_in = 0.0f, f_in = 0.0f, s_gate = 0.0f, s_lf = 0.0f;
  auto fetch_gates = [&](int c0) {
    if constexpr (MODE != GLA) {
      const int64_t last = min(64, t1 - c0) - 1;
      s_in = load_1(rows_of(p.s0 + (int64_t)c0 * p.s_rs + h, (last * p.s_rs + 1) * 4), (int)(lane * p.s_rs) * 4);
      if constexpr (MODE == EXPGATE)
        f_in = load_1(rows_of(p.s1 + (int64_t)c0 * p.s_rs + h, (last * p.s_rs + 1) * 4), (int)(lane * p.s_rs) * 4);
    }
  };
  auto gates = [&]() {
    if constexpr (MODE == EXPGATE) {
      s_gate = p.c0 * tanhf((s_in + bias_i) / p.c0);
      s_lf = log_sigmoid_f32(p.c0 * tanhf((f_in + bias_f) / p.c0));
    } else if constexpr (MODE == SSD) {
      s_gate = softplus(s_in + bias_i);
      s_lf = -rate * s_gate;
    }
    s_lf = s_lf < LEAST ? LEAST : s_lf;
  };

  fetch_gates(t0);
  fetch(t0);
  int cur = 0, quarter = 0;
  for (int c0 = t0; c0 < t1; c0 += TOK, cur ^= 1, quarter = (quarter + 1) & 3) {
    const int n = min(TOK, t1 - c0);
    float* sq = lds + cur * BUF;         // [16][DP]
    float* sk = sq + TOK * DP;           // [16][DP]
    float* skT = sk + TOK * DP;          // [D][CP] k times its decay to the chunk's end
    float* se = skT + D * CP;            // [D] GLA: the chunk's decay per channel
    double* sF = reinterpret_cast<double*>(se + D);   // [16] log factor of a query's scores, [16] of a key's
    float* sf = se + D + 4 * TOK;        // [16] factor of q . S; [16] EXPGATE: exp(-m), SSD: the step size
    // -------- stage: lane = token, four lane groups and the wavefronts share the channels
    float raw_f[MODE == GLA ? CPL : 1], rest_f[MODE == GLA ? CPL : 1];       // F and what rounding it left out
    float whole = 1.0f, m_end = 0.0f;    // scalar decays: the state's factor over the chunk
    if constexpr (MODE == GLA) {       // F in units of log2
      float qs[CPL], ks[CPL], la[CPL], end[CPL], back[CPL];
      bool far = false;
#pragma unroll
      for (int i = 0; i < CPL; ++i) {
        la[i] = log2_sigmoid(z[i]) * p.c0;
        la[i] = lc < n && ch0 + i < d ? (la[i] < LEAST ? LEAST : la[i]) : 0.0f;
        raw_f[i] = running_sum(la[i]);
        end[i] = __shfl(raw_f[i], (lane & 48) | 15, 64);
        back[i] = end[i] - raw_f[i];
        rest_f[i] = 0.0f;
        far |= !(end[i] > -SCORE_RANGE);
      }
      const bool any = __any(far);
      if (any) {       // long sums cancel in their differences: in double
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
          const double f = running_sum((double)la[i]), e = __shfl(f, (lane & 48) | 15, 64);
          raw_f[i] = (float)f;
          rest_f[i] = (float)(f - (double)raw_f[i]);
          end[i] = (float)e;
          back[i] = (float)(e - f);
        }
      }
#pragma unroll
      for (int i = 0; i < CPL; ++i) {
        q[i] *= p.q_scale;
        k[i] *= p.k_scale;
        skT[(ch0 + i) * CP + lc] = k[i] * __builtin_amdgcn_exp2f(back[i]);
        const float e = __builtin_amdgcn_exp2f(end[i]);
        run_e[i] *= e;
        if (lc == 15) se[ch0 + i] = e;
      }
      if (emit) {
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
          qs[i] = q[i] * __builtin_amdgcn_exp2f(raw_f[i]);
          ks[i] = k[i] * __builtin_amdgcn_exp2f(-raw_f[i]);
        }
        store_n(sq + lc * DP + ch0, qs);
        store_n(sk + lc * DP + ch0, ks);
        if (lane == 0) sflag[cur * NW + wv] = any ? 1.0f : 0.0f;
      }
    } else {
      if (quarter == 0) {
        gates();
        if (c0 + 64 < t1) fetch_gates(c0 + 64);
      }
      const float lf = __shfl(s_lf, 16 * quarter + lc, 64);            // log decay
      const float in_gate = __shfl(s_gate, 16 * quarter + lc, 64);     // log input gate, or the step size
      const double Fd = running_sum(lc < n ? (double)lf : 0.0);
      const double end = __shfl(Fd, (lane & 48) | 15, 64);
      float w, rowf, m_t = 0.0f;
      if constexpr (MODE == EXPGATE) {
        // m_t = F_t + max(m ahead, max_(s <= t) (i_s - F_s))
        const double u = (double)in_gate - Fd;
        const float top = running_max(lc < n ? (float)u : -INFINITY);
        m_t = (float)(Fd + (double)fmaxf(m_run, top));
        m_end = __shfl(m_t, (lane & 48) | 15, 64);
        w = lc < n ? expf((float)(end + u - (double)m_end)) : 0.0f;
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
        q[i] *= p.q_scale;
        k[i] *= p.k_scale;
        skT[(ch0 + i) * CP + lc] = k[i] * w;
        if constexpr (MODE == EXPGATE) {
          nq += q[i] * n0[i];
          n0[i] = whole * n0[i] + lanes_sum<16>(k[i] * w);
        }
      }
      store_n(sq + lc * DP + ch0, q);
      store_n(sk + lc * DP + ch0, k);
      if constexpr (MODE == EXPGATE) {
        float a, bb;
        rows_pair16(nq, a, bb);
        rows_pair32(a + bb, a, bb);
        if (lg == 0) snq[(cur * NW + wv) * TOK + lc] = a + bb;
      }
      if (tid < TOK) {
        // the score of t and s takes exp(sF[t] + sF[16 + s]); in double, because the running sums cancel
        if constexpr (MODE == EXPGATE) {
          sF[lc] = Fd - (double)m_t;
          sF[16 + lc] = lc < n ? (double)in_gate - Fd : 0.0;
          sf[16 + lc] = expf(-m_t);
        } else {
          sF[lc] = Fd;
          sF[16 + lc] = -Fd;
          sf[16 + lc] = in_gate;
        }
        sf[lc] = rowf;
      }
      m_run = m_end;
    }
    float v[4], gate[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      v[m] = vn[m];
      gate[m] = MODE == EXPGATE ? 0.0f : gn[m];
    }
    bool odd = false;                    // of this wavefront's values, is one not finite?
#pragma unroll
    for (int m = 0; m < 4; ++m) odd |= __builtin_amdgcn_classf(v[m], 0x207);         // NaNs and infinities
    odd = __any(odd);
    __syncthreads();
    // -------- scores q_t . k_s of the chunk, shares of sixteen channels dealt to the wavefronts
    bool slow = false;
    if (MODE == GLA && emit) {
#pragma unroll
      for (int w = 0; w < NW; ++w) slow |= sflag[cur * NW + w] != 0.0f;
    }
    if (!emit) {
    } else if (!slow) {
      for (int kk = wv; kk < NP; kk += NW) {
        f32x4 acc = zero;
        if (kk < DT) acc = step4(at4(sq + lc * DP + 16 * kk + 4 * lg), at4(sk + lc * DP + 16 * kk + 4 * lg), acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 4 * lg + r, s = lc;
          float x = acc[r];
          if (s > t) {
            x = 0.0f;
          } else {
            if constexpr (MODE != GLA) x *= expf((float)(sF[t] + sF[16 + s]));
            if constexpr (MODE == SSD) x *= sf[16 + s];
          }
          sp[(kk * TOK + t) * CP + s] = x;
        }
      }
    } else if constexpr (MODE == GLA) {
      // the other buffer is free until the next chunk is staged: q, k and F as they are
      float* rq = lds + (cur ^ 1) * BUF;
      float* rf = rq + TOK * DP;
      float* rr = rf + TOK * DP;
      store_n(rq + lc * DP + ch0, q);
      store_n(rf + lc * DP + ch0, raw_f);
      store_n(rr + lc * DP + ch0, rest_f);
      store_n(sk + lc * DP + ch0, k);
      __syncthreads();
      constexpr int PARTS = NW / 4, CH = D / PARTS;
      const int pair = tid & 255, part = tid >> 8, t = pair >> 4, s = pair & 15;
      float x = 0.0f;
      if (s <= t) {
#pragma unroll 2
        for (int c = part * CH; c < (part + 1) * CH; ++c)
          x += rq[t * DP + c] * sk[s * DP + c] * __builtin_amdgcn_exp2f((rf[t * DP + c] - rf[s * DP + c]) + (rr[t * DP + c] - rr[s * DP + c]));
      }
#pragma unroll
      for (int w = 0; w < NP; ++w)
        if (w % PARTS == part) sp[(w * TOK + t) * CP + s] = w == part ? x : 0.0f;
    }
    if (c0 + TOK < t1) fetch(c0 + TOK);
    // -------- what the state ahead of the chunk contributes
    f32x4 o0 = zero, o1 = zero;
#pragma unroll
    for (int kk = 0; kk < DT && emit; kk += 2) {
      o0 = step4(at4(sq + lc * DP + 16 * kk + 4 * lg), S[kk], o0);
      if (kk + 1 < DT) o1 = step4(at4(sq + lc * DP + 16 * kk + 16 + 4 * lg), S[kk + 1], o1);
    }
    f32x4 o;
    if constexpr (MODE == GLA) {
      o = o0 + o1;
    } else {
      const f32x4 f = at4(sf + 4 * lg);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (o0[r] + o1[r]) * f[r];
    }
    // -------- the state behind the chunk
    const f32x4 vv = f32x4{v[0], v[1], v[2], v[3]};
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      if constexpr (MODE == GLA) {
        const f32x4 e = at4(se + 16 * i + 4 * lg);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] *= e[r];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] *= whole;
      }
      S[i] = step4(at4(skT + (16 * i + lc) * CP + 4 * lg), vv, S[i]);
    }
    if (!emit) continue;                 // the next chunk goes to the other buffer: one barrier a chunk
    __syncthreads();
    // -------- what the chunk's own tokens contribute
    f32x4 P = at4(sp + lc * CP + 4 * lg);
#pragma unroll
    for (int w = 1; w < NP; ++w) {
      const f32x4 x = at4(sp + (w * TOK + lc) * CP + 4 * lg);
#pragma unroll
      for (int r = 0; r < 4; ++r) P[r] += x[r];
    }
    // A score of a later token is 0, but 0 times an infinity or a NaN is not: with such a value in the chunk its terms are summed one
    // by one, so that a token's row depends on the tokens up to it alone.
    if (!odd) {
      o = step4(P, vv, o);
    } else {
#pragma unroll 1
      for (int s = 0; s < TOK; ++s) {
        const float vs = __shfl(s & 2 ? (s & 1 ? vv[3] : vv[2]) : (s & 1 ? vv[1] : vv[0]), 16 * (s >> 2) + lc, 64);
        const float ps = s & 2 ? (s & 1 ? P[3] : P[2]) : (s & 1 ? P[1] : P[0]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = __shfl(ps, 16 * (s >> 2) + 4 * lg + r, 64);
          if (s <= 4 * lg + r) o[r] = fmaf(x, vs, o[r]);
        }
      }
    }
    const auto ro = rows_of(out_p, ((n - 1) * (int)p.out_rs + vd) * OUT);
    out_p += TOK * p.out_rs * OUT;
    if constexpr (MODE == GLA) {
      f32x4 share;                       // columns that are not there hold zeros
#pragma unroll
      for (int r = 0; r < 4; ++r) share[r] = lanes_sum<16>(o[r] * o[r]);
      if (lc == 0) *reinterpret_cast<f32x4*>(sred + wv * TOK + 4 * lg) = share;
      __syncthreads();
      // token lc's norm, then those of this lane's four rows
      float ss = sred[lc];
#pragma unroll
      for (int w = 1; w < NW; ++w) ss += sred[w * TOK + lc];
      const float var = ss * inv_vd + p.eps;
      float inv = __builtin_amdgcn_rsqf(var);                          // and one Newton step
      inv *= fmaf(-0.5f * var * inv, inv, 1.5f);
#pragma unroll
      for (int r = 0; r < 4; ++r) store_1<T>(ro, o_at[r], o[r] * __shfl(inv, 4 * lg + r, 64) * nw * silu(gate[r]));
    } else if constexpr (MODE == EXPGATE) {
      // n_t . q_t of token lc: the scores' row and the normaliser ahead of the chunk
      float a, bb, nq = (P[0] + P[1]) + (P[2] + P[3]);
      rows_pair16(nq, a, bb);
      rows_pair32(a + bb, a, bb);
      nq = a + bb;
      float ahead = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) ahead += snq[(cur * NW + w) * TOK + lc];
      nq += ahead * sf[lc];
      const float under = 1.0f / (fmaxf(fabsf(nq), sf[16 + lc]) + 1e-6f);
#pragma unroll
      for (int r = 0; r < 4; ++r) store_1<float>(ro, o_at[r], o[r] * __shfl(under, 4 * lg + r, 64));
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) store_1<float>(ro, o_at[r], (o[r] + skip * v[r]) * silu(gate[r]));
    }
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
          if (to_slot) S_g[(int64_t)row * vd + col] = S[i][r];
          if (to_ws) E[(int64_t)row * vd + col] = S[i][r];
        }
      }
    if (MODE == SSD && to_ws && tid == 0) p.ws_decay[run0 + j] = expf((float)run_lf);
  }
  if constexpr (MODE == GLA) {
    if (p.runs > 1 && p.pass == 1 && t1 < t_end && lc == 0) {
#pragma unroll
      for (int i = 0; i < CPL; ++i)
        if (ch0 + i < d) p.ws_decay[(run0 + j) * d + ch0 + i] = run_e[i];
    }
  }
  if constexpr (MODE == EXPGATE) {
    for (int c = 0; c < (vd + 63) / 64; ++c) {
      float* n_g = S_g + (int64_t)d * vd + (int64_t)c * (d + 1);
#pragma unroll
      for (int i = 0; i < CPL; ++i)
        if (lc == 0 && ch0 + i < d) n_g[ch0 + i] = n0[i];
      if (tid == 0) n_g[d] = m_run;
    }
  }
}

template <int MODE, typename T, int D, int NW>
__global__ __launch_bounds__(64 * NW, D <= 64 || (MODE == SSD && NW == 8) ? 4 : 1) void chunk_scan_kernel(Args p) {
  chunk_walk<MODE, T, D, NW>(p, threadIdx.x);
}

}  // namespace chunk_scan

#include "chunk_parts.h"

namespace chunk_scan {

// Scalar decays in chunks of thirty-two from twenty tokens to a request of the step on: below, most of its chunks would be empty places (us,
// both, state-space layers of 16 heads of 128 x 64 and exponential gates of 64 x 128: 24 requests of 33 tokens 22.8 and 20.4, 21.7 and
// 21.8, of 16 12.5 and 13.7, 12.6 and 15.1; 64 single tokens beside a piece of 40 37.4 and 35.2, 29.3 and 33.5).
inline bool in_parts(int64_t tokens, int num_seqs) { return tokens >= 20 * (int64_t)num_seqs; }

template <int MODE, typename T, int D, int NW>
hipError_t launch_one(const Args& p, int num_seqs, int runs, hipStream_t s) {
  void (*kernel)(Args) = chunk_scan_kernel<MODE, T, D, NW>;
  size_t lds = lds_floats<D, NW>() * sizeof(float);
  static std::atomic<uint64_t> devices[2] = {{0}, {0}};
  int form = 0;
  if constexpr (MODE != GLA) {
    if (p.in_parts) {
      kernel = chunk_parts_kernel<MODE, T, D, NW>;
      lds = PartsPlan<MODE, D, NW>::BYTES;
      form = 1;
    }
  }
  static_assert(lds_floats<D, NW>() * sizeof(float) <= 160 * 1024, "the chunk fits the LDS");
  if (lds > 64 * 1024) {
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(kernel), lds, devices[form]);
    if (e != hipSuccess) return e;
  }
  kernel<<<dim3(p.H, num_seqs, runs), dim3(64 * NW), lds, s>>>(p);
  return hipGetLastError();
}

// Sizes and alignments that the kernel serves: rows that split into 16-byte pieces, keys and values up to 128 numbers per
// head, 64 rows within the 2 GB of a buffer descriptor's offsets.  Key rows must not overlap: those past a request's end are zeros
// because they start past the last row's end (a row expanded over the tokens, with a stride of 0, goes to the walk).
constexpr int64_t FAR = 1 << 22;
inline bool serves(const Args& p) {
  auto al16 = [](const void* q) { return (uintptr_t)q % 16 == 0; };
  return p.dim % 4 == 0 && p.dim <= 128 && p.vdim <= 128 && p.q_rs % 4 == 0 && p.k_rs % 4 == 0 && al16(p.q) && al16(p.k) &&
         p.k_rs >= p.dim && p.q_rs < FAR && p.k_rs < FAR && p.v_rs < FAR && p.g_rs < FAR && p.s_rs < FAR && p.out_rs < FAR;
}

template <int MODE, typename T>
hipError_t launch(const Args& p, int num_seqs, hipStream_t s, int runs = 1) {
  if (p.vdim <= 64) {
    if (p.dim <= 32) return launch_one<MODE, T, 32, 4>(p, num_seqs, runs, s);
    if (p.dim <= 64) return launch_one<MODE, T, 64, 4>(p, num_seqs, runs, s);
    return launch_one<MODE, T, 128, 4>(p, num_seqs, runs, s);
  }
  if (p.dim <= 32) return launch_one<MODE, T, 32, 8>(p, num_seqs, runs, s);
  if (p.dim <= 64) return launch_one<MODE, T, 64, 8>(p, num_seqs, runs, s);
  return launch_one<MODE, T, 128, 8>(p, num_seqs, runs, s);
}

// Decays per token (SSD) or per token and channel (GLA) make a run of tokens an affine map of the state, S -> D S + E, so the
// long prompts of few requests are cut into runs that are walked side by side.  First pass: run 0 starts from the slot and is
// final; the runs between it and the last start from zero and leave their end state E and the product D of their decays.  Second
// pass: run j >= 1 folds those of the runs ahead of it into its start and walks its tokens, writing their rows; the run with the
// step's last token leaves the state in the slot (which nobody reads in the second pass).
template <int MODE, typename T>
hipError_t launch_runs(Args& p, int num_seqs, hipStream_t s) {
  p.pass = 1;
  const hipError_t e = launch<MODE, T>(p, num_seqs, s, p.runs);
  if (e != hipSuccess || p.runs == 1) return e;
  p.pass = 2;
  return launch<MODE, T>(p, num_seqs, s, p.runs - 1);
}

}  // namespace chunk_scan
