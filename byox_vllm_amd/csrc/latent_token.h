// Latent attention of single tokens (steps that bring one token per request), included by latent_attn.hip.
//
// What bounded the tile kernel here (60 us for 8 tokens over 2048 rows of 1.1 KB, 15 MB): every load touched 64 cache lines,
// rows were written into LDS twice (once transposed, two bytes at a time) and three workgroup barriers stood in each tile of
// 32 keys.  Here a wavefront works alone on 32 keys at a time: their rows go into its own part of LDS by LDS-DMA, are read
// back as K fragments and, through transposing reads, as V^T fragments, and its softmax state is private; wavefronts and
// workgroups (blockIdx.z) take every 4 * ksplit-th tile and meet once at the end.  22 us for the same rows (each wavefront has
// one tile there: what is left is the chain of look-ups, the rows' latency and the merge).  A layer's whole step of 128 tokens over up
// to 2000 rows of 320, 576 and 1088 bytes went from 194, 310 and 515 us to 84, 106 and 176.
//
// In LDS a tile is [64-byte unit of a row][32 keys][64 bytes]: a DMA instruction moves one unit of sixteen keys, a K fragment
// is 1 KB in sequence, and the 16-byte pieces of a unit are dealt by XOR with bits 2 and 3 of the key, so that neither the
// fragment nor the transposing reads meet bank conflicts.  S^T = K q^T with the heads as columns: a lane owns eight scores of
// one head.  Queries and probabilities enter the products as the sum of two bf16 numbers, as in the tile kernel.
#pragma once

template <int KS>      // 64-byte units of a row, at most
__global__ __launch_bounds__(256, KS > 9 ? 1 : 2) void latent_token_kernel(MfmaAttnArgs a, int bs_shift) {
  constexpr int NT = 2 * KS;             // 16-number tiles of a row's latent, at most
  constexpr float L2E = 1.4426950408889634f;
  extern __shared__ u32x4 lds_raw[];
  __shared__ float s_m[4][16], s_l[4][16];
  typedef __attribute__((address_space(1))) const void global_void;
  typedef __attribute__((address_space(3))) void lds_void;
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  const AttnArgs& p = a.a;
  const int Dk = p.rank + p.rot_dim, R = p.rank, units = Dk / 32, nt = R / 16;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int t = blockIdx.y, h0 = blockIdx.x * 16;
  const int b = p.seq_of[t];
  const int pos = p.past[b] + (t - p.cu_q[b]);
  const int kmin = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  const int32_t* table = p.tables + (int64_t)b * p.table_cols;
  constexpr int area = KS * 2048;
  unsigned char* mine = reinterpret_cast<unsigned char*>(lds_raw) + wv * area;

  auto swz = [](int key) { return 2 * ((key >> 2) & 1) + ((key >> 3) & 1); };
  // this lane's part of the DMA: keys lane / 4 and 16 + lane / 4, one piece of every unit
  const int piece = ((lane & 3) ^ swz(lane >> 2)) << 4;      // swz(key + 16) = swz(key)
  int page[2], in_page[2];
  auto look_up = [&](int j0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int kp = min(j0 + 16 * i + (lane >> 2), pos);      // keys past the token repeat it (they are masked)
      const int n = bs_shift >= 0 ? kp >> bs_shift : kp / p.block_size;
      in_page[i] = kp - n * p.block_size;
      page[i] = table[n];
    }
  };
  f32x4 o[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) o[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY, l_run = 0.0f;
  const int step = 4 * a.ksplit * 32;
  int j0 = kmin + ((int)blockIdx.z * 4 + wv) * 32;
  if (j0 <= pos) look_up(j0);
  // queries: lane holds numbers 32 u + 8 g .. + 7 of head c, as hi + lo.  Units past the row's are zeros here and in LDS
  // (nothing writes them), so that the loops below carry no branch: with one around each unit the 17 loads of a query and the
  // fragment reads waited one by one (33 us instead of 22 for 8 tokens over 2048 rows).
  bf16x8 qh[KS], ql[KS];
  {
    const bool on = h0 + c < p.H;
    const float* row = p.qa + ((int64_t)t * p.H + (on ? h0 + c : h0)) * Dk + 8 * g;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const int at = 32 * min(u, units - 1);
      const f32x4 x = *reinterpret_cast<const f32x4*>(row + at), y = *reinterpret_cast<const f32x4*>(row + at + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = on && u < units ? (e < 4 ? x[e & 3] : y[e & 3]) : 0.0f;
        qh[u][e] = (bf16_t)v;
        ql[u][e] = (bf16_t)(v - (float)qh[u][e]);
      }
    }
  }
  for (int i = units * 2048 + lane * 16; i < area; i += 1024) *reinterpret_cast<u32x4*>(mine + i) = u32x4{0, 0, 0, 0};
  const int k_at = c * 64 + ((g ^ swz(c)) << 4);
  // V^T: four tokens by sixteen numbers per sixteen lanes: tokens 4 g + (lane & 15) / 4 (and 16 further), numbers 4 (lane & 3) ..
  const int vt = 4 * g + (c >> 2), v_sw = swz(vt), v_lo = (lane & 1) * 8, v_p = (lane & 3) >> 1;
  for (; j0 <= pos; j0 += step) {
    {
      const char* base[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        base[i] = reinterpret_cast<const char*>(p.cache) + ((int64_t)page[i] * p.block_size + in_page[i]) * (2 * Dk) + piece;
      for (int u = 0; u < units; ++u) {
        __builtin_amdgcn_global_load_lds((global_void*)(base[0] + 64 * u), (lds_void*)(mine + 2048 * u), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((global_void*)(base[1] + 64 * u), (lds_void*)(mine + 2048 * u + 1024), 16, 0, 0);
      }
    }
    if (j0 + step <= pos) look_up(j0 + step);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wavefront's own rows: no barrier
    f32x4 s[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) s[i][0] = s[i][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < KS; ++u) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(mine + 2048 * u + 1024 * i + k_at);
        s[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qh[u], s[i][0], 0, 0, 0);
        s[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, ql[u], s[i][1], 0, 0, 0);
      }
    }
    float x[8], mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int key = j0 + 16 * (e >> 2) + 4 * g + (e & 3);
      x[e] = key <= pos ? (s[e >> 2][0][e & 3] + s[e >> 2][1][e & 3]) * p.scale : -INFINITY;
      mx = fmaxf(mx, x[e]);
    }
    float u0, u1;
    rows_pair16(mx, u0, u1);
    rows_pair32(fmaxf(u0, u1), u0, u1);
    const float m_new = fmaxf(m_run, fmaxf(u0, u1));       // finite: the tile has a key of the token's
    if (__any(m_new != m_run)) {
      const float corr = __builtin_amdgcn_exp2f((m_run - m_new) * L2E);
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][r] *= corr;
      l_run *= corr;
      m_run = m_new;
    }
    bf16x8 ph, pl;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float w = __builtin_amdgcn_exp2f((x[e] - m_run) * L2E);
      l_run += w;
      ph[e] = (bf16_t)w;
      pl[e] = (bf16_t)(w - (float)ph[e]);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const unsigned char* v = mine + 2048 * (n >> 1) + vt * 64 + (((2 * (n & 1) + v_p) ^ v_sw) << 4) + v_lo;
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)v));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(v + 1024)));
      const bf16x8 vf = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph, o[n], 0, 0, 0);
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, o[n], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the next tile's rows may overwrite these
  }
  // the wavefronts' shares: lane holds numbers 16 n + 4 g + r of head c
  {
    float u0, u1;
    rows_pair16(l_run, u0, u1);
    rows_pair32(u0 + u1, u0, u1);
    if (g == 0) {
      s_m[wv][c] = m_run;
      s_l[wv][c] = u0 + u1;
    }
  }
  __syncthreads();
  float m = s_m[0][c];
#pragma unroll
  for (int w = 1; w < 4; ++w) m = fmaxf(m, s_m[w][c]);
  float l = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) l += s_m[w][c] == -INFINITY ? 0.0f : s_l[w][c] * __builtin_amdgcn_exp2f((s_m[w][c] - m) * L2E);
  const float f = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m_run - m) * L2E);
  float* share = reinterpret_cast<float*>(mine);              // [16 heads][R], 64 R bytes of 64 (R + rot)
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    if (n < nt) {
    f32x4 v = o[n];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] *= f;
    *reinterpret_cast<f32x4*>(share + c * R + 16 * n + 4 * g) = v;
    }
  }
  __syncthreads();
  const int heads = min(16, p.H - h0);
  for (int i = tid; i < heads * (R / 4); i += 256) {
    const int h = i / (R / 4), e = i % (R / 4) * 4;
    f32x4 v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 4; ++w)
      v += *reinterpret_cast<const f32x4*>(reinterpret_cast<const unsigned char*>(lds_raw) + w * area + (h * R + e) * 4);
    float ml = s_m[0][h];
#pragma unroll
    for (int w = 1; w < 4; ++w) ml = fmaxf(ml, s_m[w][h]);
    float ll = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) ll += s_m[w][h] == -INFINITY ? 0.0f : s_l[w][h] * __builtin_amdgcn_exp2f((s_m[w][h] - ml) * L2E);
    if (a.ksplit > 1) {       // another launch joins the workgroups' shares
      float* dst = a.partial + (((int64_t)t * p.H + h0 + h) * a.ksplit + blockIdx.z) * (R + 2);
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[e + r] = v[r];
      if (e == 0) {
        dst[R] = ml;
        dst[R + 1] = ll;
      }
    } else {
      const float inv = 1.0f / ll;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] *= inv;
      *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.out) + ((int64_t)t * p.H + h0 + h) * R + e) = Pack4<bf16_t>::narrow(v);
    }
  }
}

template <int KS>
hipError_t launch_latent_token(const MfmaAttnArgs& q, int64_t tokens, hipStream_t s) {
  constexpr size_t lds = (size_t)4 * KS * 2048;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> devices{0};
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(&latent_token_kernel<KS>), lds, devices);
    if (e != hipSuccess) return e;
  }
  int shift = -1;
  if ((q.a.block_size & (q.a.block_size - 1)) == 0)
    for (shift = 0; (1 << shift) < q.a.block_size;) ++shift;
  latent_token_kernel<KS><<<dim3((q.a.H + 15) / 16, (unsigned)tokens, q.ksplit), dim3(256), lds, s>>>(q, shift);
  return hipGetLastError();
}
