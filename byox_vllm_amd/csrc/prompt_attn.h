// Prompt attention over paged bf16 rows, included by window_attn.hip (WAttnArgs, close_softmax): the walk of
// window_attn_mfma_kernel for heads of 64 or 128 numbers, arranged for many query rows per key.
//
// What bounded the older kernel at 0.1 PFLOP/s: 64 query rows per staged tile of 64 keys, V written transposed into LDS two
// bytes at a time, three workgroup barriers per tile and no load under the arithmetic.  Here
//   * a workgroup holds 128 query rows (128 / R tokens times the R heads of a key head), 32 per wavefront;
//   * keys and values travel as whole rows into LDS by LDS-DMA, the next tile under the current one's arithmetic, with one
//     barrier per tile; their 16-byte pieces are dealt by XOR with the row so that fragment reads meet no bank conflicts;
//   * S^T = K Q^T: a lane owns one query row and sixteen keys of a 32 x 32 product, so maxima and sums are lane-local but for
//     one exchange between the wavefront's halves, and P^T is the operand of O^T = V^T P^T as it lies in the registers;
//     V^T fragments come from transposing LDS reads (ds_read_b64_tr_b16);
//   * tiles that every row of the wavefront sees whole take no mask, and the outputs are rescaled only when some row's
//     maximum grew.
// A tile holds tokens of one request: steps bring prompt pieces and decoding requests together, and a tile over up to 128 / R of the
// latter walked their contexts one after the other.  The grid has room for a part tile per request, and a workgroup finds its own
// with one prefix sum over the requests.  A layer of 16 heads of 128 over 64 requests of 2048 cached tokens, one new token each, and
// a prompt of 512: 8900 us in the older kernel, 4430 with tiles over several requests, 302 now; two heads per key head and a window
// of 512: 1495, 1515, 109; prompts alone as before (8 x 2048 ragged: 589 and 577).
// Scores, maxima, sums and outputs are fp32; q and P enter the products as bf16, so queries may come in bf16 as well (half the bytes of the
// rows that a workgroup begins with).  Of what held the walk up besides its softmax:
//   * the compiler put every fragment's read right before its product, and ahead of the first transposing read waited for the next tile's
//     DMA: both are placed by hand, fragments four products ahead, weights of sixteen keys under the products of the sixteen before;
//   * page numbers and addresses were a lane's own, 200 of a tile's 500 vector instructions: tiles begin at multiples of 64, so that blocks
//     of a multiple of 64 hold whole tiles at a place that one scalar gives.  In one kernel with the lanes' own the registers did not suffice;
//   * a tile's request and first position were looked up in turn, ahead of its queries.
// Measured, 8 prompts of 2048 tokens, 16 heads of 128: window 512 beside 16 kept keys, two heads per key head, 554 us in the older kernel,
// 179, now 145; 16 key heads, ragged, every earlier key, 549, 181, now 155.  Heads of 64 have three wavefronts to a SIMD; with two, kept keys
// and a window of 700 took 3 % more of a layer.  What is left: the queries' and results' bytes, which nothing overlaps at a workgroup's
// beginning and end (40 us), and 330 vector instructions per 32 products.
#pragma once

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int PA_ROWS = 128, PA_KEYS = 64;

// A weight of 0 times an infinity or a NaN is NaN: a value row that is not finite reaches the rows that meet it in a tile without
// seeing it, those ahead of it among them.  Rows that came out so (bit i of `rest`: row row0 + i of the tile's tokens from ts on) are
// formed again by one wavefront from the keys that they see, one by one.
template <int D, bool EXT>
__device__ __forceinline__ void prompt_rows_again(const WAttnArgs& a, uint32_t rest, int row0, int64_t ts, int b, int g, int bs_shift) {
  constexpr float LOG2E = 1.4426950408889634f;
  const int lane = threadIdx.x & 63, heads = a.H / a.G, first_pos = a.past[b] + (int)(ts - a.cu_q[b]);
  const int32_t* table = a.tables + (int64_t)b * a.table_cols;
  const char* k_base = reinterpret_cast<const char*>(a.cache) + (int64_t)g * (2 * D);
  const char* v_base = reinterpret_cast<const char*>(a.cache) + ((int64_t)a.v_col + (int64_t)g * D) * 2;
#pragma unroll 1
  for (; rest != 0; rest &= rest - 1) {
    const int row = row0 + __ffs(rest) - 1, row_tok = row / heads, row_head = g * heads + row % heads, row_pos = first_pos + row_tok;
    const int first = max(a.window > 0 ? row_pos - a.window + 1 : 0, EXT && a.chunk > 0 ? row_pos / a.chunk * a.chunk : 0);
    const int from = max(first, 0), kept = EXT ? min(a.keep, from) : 0, count = kept + row_pos + 1 - from;
    const int64_t q_at = ((ts + row_tok) * a.H + row_head) * D;
    auto query = [&](int e) {
      return a.q16 ? (float)reinterpret_cast<const bf16_t*>(a.q)[q_at + e] : (float)(bf16_t)reinterpret_cast<const float*>(a.q)[q_at + e];
    };
    auto row_at = [&](int c) {             // byte offset of the row's c-th visible key
      const int key = c < kept ? c : from + c - kept, n = bs_shift >= 0 ? key >> bs_shift : key / a.block_size;
      return ((int64_t)table[n] * a.block_size + (key - n * a.block_size)) * (2 * (int64_t)a.cw);
    };
    auto score = [&](int c) {
      const char* k = k_base + row_at(c);
      float sum = 0.0f;
#pragma unroll 1
      for (int e = 0; e < D; e += 8) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(k + 2 * e);
#pragma unroll
        for (int j = 0; j < 8; ++j) sum = fmaf(query(e + j), (float)x[j], sum);
      }
      return sum;
    };
    float m = -INFINITY;
    bool undefined = false;
#pragma unroll 1
    for (int c0 = 0; c0 < count; c0 += 64) {
      const float x = score(min(c0 + lane, count - 1));
      m = fmaxf(m, x);
      undefined |= x != x || x == INFINITY;
    }
    if (__any(undefined)) continue;        // all of the row is NaN, as stored
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    const float m_use = m == -INFINITY ? 0.0f : m * LOG2E;
    float l = 0.0f, acc[D / 64];
#pragma unroll
    for (int i = 0; i < D / 64; ++i) acc[i] = 0.0f;
#pragma unroll 1
    for (int c0 = 0; c0 < count; c0 += 64) {
      const float e = c0 + lane < count ? __builtin_amdgcn_exp2f(fmaf(score(min(c0 + lane, count - 1)), LOG2E, -m_use)) : 0.0f;
      l += e;
#pragma unroll 1
      for (int c = c0; c < min(c0 + 64, count); ++c) {
        const float w = (float)(bf16_t)__shfl(e, c - c0, 64);
        const bf16_t* v = reinterpret_cast<const bf16_t*>(v_base + row_at(c)) + lane;
#pragma unroll
        for (int i = 0; i < D / 64; ++i) acc[i] += w * (float)v[64 * i];
      }
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) l += __shfl_xor(l, d, 64);
    float fs, den;
    close_softmax(m, l, a.sink != nullptr, a.sink ? ld_f32<bf16_t>(reinterpret_cast<const bf16_t*>(a.sink) + row_head) : 0.0f, fs, den);
    const float f = a.out_scale * fs / den;
    const float* gates = a.gate ? a.gate + (ts + row_tok) * a.gate_rs : nullptr;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
      const int n = row_head * D + lane + 64 * i;
      const float on = !gates ? 1.0f : sigmoid_f32(gates[EXT && a.gate_head ? row_head : n]);
      reinterpret_cast<bf16_t*>(a.out)[(ts + row_tok) * a.out_rs + n] = (bf16_t)(acc[i] * f * on);
    }
  }
}

// 16 bytes to a lane into LDS at `dst` + 16 * lane.  Not the builtin: the compiler waits for every DMA under way ahead of a transposing
// read, for the next tile's too; what has to be waited for is said at the tile's beginning.
__device__ __forceinline__ void pa_dma(const void* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ void pa_dma(const void* base, uint32_t off, uint32_t dst) {      // one base for the wavefront
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}

// WHOLE: blocks of a multiple of 64 hold whole tiles (and rows of less than 32 MB, so that a place in a tile is 32 bits)
template <int D, bool EXT, bool WHOLE>
__global__ __launch_bounds__(256, D == 64 && EXT ? 3 : 2) void prompt_attn_kernel(WAttnArgs p, int tiles, int num_seqs, int bs_shift) {
  constexpr int KS = D / 16, DT = D / 32, ROWB = 2 * D, TILE = PA_KEYS * ROWB;      // bytes of one operand's tile
  constexpr int RPI = 1024 / ROWB, NI = PA_KEYS / RPI / 4;                          // rows per DMA instruction; instructions per wavefront
  constexpr float L2E = 1.4426950408889634f;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2 * TILE];
  typedef __attribute__((address_space(3))) unsigned char lds_byte;
  const uint32_t lds_at = (uint32_t)(uintptr_t)(lds_byte*)&lds[0][0];
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  // tiles that share keys run on one XCD; late tiles of a request, which see the most keys, first
  int g, tile;
  {
    const int total = tiles * p.G, share = (total + 7) / 8, slot = blockIdx.x >> 3, id = (blockIdx.x & 7) * share + slot;
    if (slot >= share || id >= total) return;
    g = id / tiles;
    tile = tiles - 1 - id % tiles;
  }
  const int R = p.H / p.G;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  // the tile's tokens: of one request where their number is known, else of as many as have tokens there
  int64_t t_begin = (int64_t)tile * p.TQ, t_end = min(p.tokens, t_begin + p.TQ);
  int owner = -1, owner_pos = 0;       // the request and the position of the tile's first token
  if (num_seqs > 1) {
    for (int base = 0, before = 0; base < num_seqs && owner < 0; base += 64) {
      const int i = min(base + lane, num_seqs - 1);
      const int first = (int)min((int64_t)p.cu_q[i], p.tokens), end = (int)min((int64_t)p.cu_q[i + 1], p.tokens), ahead = p.past[i];
      const int mine = base + lane < num_seqs ? (end - first + p.TQ - 1) / p.TQ : 0;
      int upto = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(upto, o, 64);
        if (lane >= o) upto += x;
      }
      const uint64_t hit = __ballot(tile < before + upto);
      if (hit) {
        const int l = __ffsll((unsigned long long)hit) - 1;
        const int local = tile - before - __builtin_amdgcn_readlane(upto, l) + __builtin_amdgcn_readlane(mine, l);
        owner = base + l;
        t_begin = __builtin_amdgcn_readlane(first, l) + (int64_t)local * p.TQ;
        t_end = min((int64_t)__builtin_amdgcn_readlane(end, l), t_begin + p.TQ);
        owner_pos = __builtin_amdgcn_readlane(ahead, l) + local * p.TQ;
      }
      before += __builtin_amdgcn_readlane(upto, 63);
    }
    if (owner < 0) return;               // the grid covers the largest possible number of tiles
  }
  const char* k_base = reinterpret_cast<const char*>(p.cache) + (int64_t)g * ROWB;
  const char* v_base = reinterpret_cast<const char*>(p.cache) + ((int64_t)p.v_col + (int64_t)g * D) * 2;
  const int64_t row_bytes = (int64_t)p.cw * 2;
  const bf16_t* sink = reinterpret_cast<const bf16_t*>(p.sink);
  auto k_swz = [](int r) { return D == 128 ? r & 15 : (r >> 1) & 7; };
  auto v_swz = [](int r) { return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); };

  // this lane's part of the DMA: row RPI * (wv * NI + i) + lane / (64 / RPI) of the tile, piece lane % (64 / RPI)
  constexpr int PIECES = 64 / RPI;                 // 16-byte pieces of a row
  const int dma_r = lane / PIECES, dma_p = lane % PIECES;
  uint32_t k_off[NI], v_off[NI];      // WHOLE: from the tile's first row, else from its own
  auto row_of = [&](int i) { return RPI * (wv * NI + i) + dma_r; };
  auto k_piece = [&](int i) { return (uint32_t)(dma_p ^ k_swz(row_of(i))) << 4; };
  auto v_piece = [&](int i) { return (uint32_t)(dma_p ^ v_swz(row_of(i))) << 4; };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const uint32_t row = WHOLE ? (uint32_t)row_of(i) * (uint32_t)row_bytes : 0;
    k_off[i] = row + k_piece(i);
    v_off[i] = row + v_piece(i);
  }
  // fragment addresses inside a tile: K row lr of a 32-row tile, piece 2 ks + lh; V^T: four tokens by sixteen numbers per
  // sixteen lanes, rows 4 lh + (lane & 15) / 4 (and 8 further), numbers 16 (lr >> 4) + 4 (lane & 3)
  const int ksw = k_swz(lr);
  const int vq = (lane & 15) >> 2, vr = 4 * lh + vq, vsw = v_swz(vr);
  auto v_at = [&](int dt) { return vr * ROWB + (((4 * dt + 2 * (lr >> 4) + ((lane & 3) >> 1)) ^ vsw) << 4) + (lane & 1) * 8; };

  for (int64_t ts = t_begin; ts < t_end;) {
    const int b = owner >= 0 ? owner : p.seq_of[ts];
    const int64_t te = owner >= 0 ? t_end : min(t_end, (int64_t)p.cu_q[b + 1]);
    const int nq = (int)(te - ts), rows = nq * R;
    const int p0 = owner >= 0 ? owner_pos : p.past[b] + (int)(ts - p.cu_q[b]);
    const int32_t* table = p.tables + (int64_t)b * p.table_cols;
    const int row0 = 32 * wv, rr = row0 + lr;
    const bool valid = rr < rows, wave_on = row0 < rows;
    const int tok = valid ? rr / R : 0, head = g * R + (valid ? rr % R : 0);
    const int pos = p0 + tok;
    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    const int wpos_lo = p0 + row0 / R, wpos_hi = p0 + min(rows - 1, row0 + 31) / R;

    // The walk is over tiles of 64 keys from multiples of 64 on: those with kept keys, then those from the first key of the tile's first row
    // to the last key of its last.  Kept keys that fit the places ahead of that first key lie there instead of in a tile of their own.
    auto first_of = [&](int at) { return max(p.window > 0 ? at - p.window + 1 : 0, EXT && p.chunk > 0 ? at / p.chunk * p.chunk : 0); };
    const int low = first_of(pos), hi = p0 + nq - 1, wlow_lo = first_of(wpos_lo), wlow_hi = first_of(wpos_hi);
    const int first_key = first_of(p0), kept_keys = EXT ? min(p.keep, first_key) : 0;
    const int merged = EXT && first_key >= PA_KEYS && kept_keys <= first_key % PA_KEYS ? kept_keys : 0;
    const int kept_tiles = merged > 0 ? 0 : (kept_keys + PA_KEYS - 1) / PA_KEYS;
    const int skipped = max(first_key / PA_KEYS - kept_tiles, 0), count = hi / PA_KEYS + 1 - skipped;
    auto tile_key = [&](int it) { return PA_KEYS * (it < kept_tiles ? it : it + skipped); };
    // Where its rows are.  Blocks of a multiple of 64 hold whole tiles: one page number for all lanes, asked for a tile ahead (as a vector
    // load: what waits for a scalar one waits for all reads of LDS too), and every lane's place in a tile is the same each time.  Else every
    // lane looks its rows up.  Places past the last key repeat it: they are masked, and what nobody has written there may be a NaN.  Places
    // between the kept keys and the first key of the tile's first row, masked as well, repeat that key: their blocks may be anybody's by now,
    // and their entries of the table are not read (with whole tiles in a block, the entry is that of a key that is seen).
    int page[NI], in_page[NI], no_lane;
    asm volatile("v_mov_b32 %0, 0" : "=v"(no_lane));
    auto look_up = [&](int it) {
      const int j0 = tile_key(min(it, count - 1));
      if constexpr (WHOLE) {
        page[0] = table[(bs_shift >= 0 ? j0 >> bs_shift : j0 / p.block_size) + no_lane];
        if (EXT && merged > 0 && it == 0) page[1] = table[no_lane];
      } else {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int r = row_of(i), key = min(j0 + r, hi), kp = EXT && it == 0 && r < merged ? r : key < kept_keys ? key : max(key, first_key);
          const int n = bs_shift >= 0 ? kp >> bs_shift : kp / p.block_size;
          in_page[i] = kp - n * p.block_size;
          page[i] = table[n];
        }
      }
    };
    auto fill = [&](int buf, int it) {
      const uint32_t dst = lds_at + buf * 2 * TILE + wv * NI * 1024;
      if constexpr (WHOLE) {
        const int j0 = tile_key(it), n = bs_shift >= 0 ? j0 >> bs_shift : j0 / p.block_size;
        const int64_t at = ((int64_t)__builtin_amdgcn_readfirstlane(page[0]) * p.block_size + (j0 - n * p.block_size)) * row_bytes;
        const bool ends = hi - j0 < PA_KEYS - 1;
        if (EXT && merged > 0 && it == 0) {
          const int64_t at_kept = (int64_t)__builtin_amdgcn_readfirstlane(page[1]) * p.block_size * row_bytes;
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            const int r = row_of(i);
            const int64_t row = r < merged ? at_kept + r * row_bytes : at + min(r, hi - j0) * row_bytes;
            pa_dma(k_base + row + k_piece(i), dst + i * 1024);
            pa_dma(v_base + row + v_piece(i), dst + i * 1024 + TILE);
          }
          return;
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          uint32_t k = k_off[i], v = v_off[i];
          if (ends) {
            const uint32_t row = (uint32_t)min(row_of(i), hi - j0) * (uint32_t)row_bytes;
            k = row + k_piece(i);
            v = row + v_piece(i);
          }
          pa_dma(k_base + at, k, dst + i * 1024);
          pa_dma(v_base + at, v, dst + i * 1024 + TILE);
        }
      } else {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int64_t at = ((int64_t)page[i] * p.block_size + in_page[i]) * row_bytes;
          pa_dma(k_base + at + k_off[i], dst + i * 1024);
          pa_dma(v_base + at + v_off[i], dst + i * 1024 + TILE);
        }
      }
    };
    __builtin_amdgcn_s_barrier();            // an earlier request's walk through this tile has read its last buffer
    look_up(0);
    const float head_gate = EXT && p.gate_head && p.gate ? p.gate[(ts + tok) * p.gate_rs + head] : 0.0f;      // waited for at the end
    fill(0, 0);
    look_up(1);
    // queries: lane holds numbers 16 ks + 8 lh .. + 7 of its row
    bf16x8 qf[KS];
    {
      const int64_t at = ((ts + tok) * p.H + head) * D + 8 * lh;
      if (p.q16) {
        const bf16_t* qrow = reinterpret_cast<const bf16_t*>(p.q) + at;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(qrow + 16 * ks);
        if (!valid) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) qf[ks] = __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0});
        }
      } else {
        const float* qrow = reinterpret_cast<const float*>(p.q) + at;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(qrow + 16 * ks), c = *reinterpret_cast<const f32x4*>(qrow + 16 * ks + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            qf[ks][e] = (bf16_t)(valid ? a[e] : 0.0f);
            qf[ks][4 + e] = (bf16_t)(valid ? c[e] : 0.0f);
          }
        }
      }
    }
    int buf = 0;
    for (int it = 0; it < count; ++it, buf ^= 1) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (it + 1 < count) {
        fill(buf ^ 1, it + 1);
        look_up(it + 2);
      }
      // keys that this wavefront's rows can see at all, and whether some row sees none of the first or none of the last of them
      const int j0 = tile_key(it), j1 = j0 + PA_KEYS - 1;
      const bool with_kept = EXT && merged > 0 && it == 0;
      if (!wave_on || j0 > wpos_hi || (j1 < wlow_lo && (!EXT || (j0 >= p.keep && !with_kept)))) continue;
      const bool cut_low = wlow_hi > j0 && (!EXT || j1 >= p.keep), cut_high = j1 > wpos_lo;
      const unsigned char* kt = lds[buf];
      f32x16 s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
      // every product has its fragment read AHEAD products before it, in the order written here: left alone, the compiler reads each
      // right before its product and waits for it
      constexpr int AHEAD = D == 64 ? 3 : 4, QK = 2 * KS, PV = 4 * DT;
      bf16x8 kf[QK], vf[PV];
      auto k_read = [&](int f) { kf[f] = *reinterpret_cast<const bf16x8*>(kt + (32 * (f & 1) + lr) * ROWB + (((f & ~1) + lh) ^ ksw) * 16); };
      auto v_read = [&](int f) {
        const unsigned char* a = kt + TILE + 16 * (f / DT) * ROWB + v_at(f % DT);
        const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)a));
        const u32x2 y = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(a + 8 * ROWB)));
        vf[f] = __builtin_bit_cast(bf16x8, u32x4{x[0], x[1], y[0], y[1]});
      };
#pragma unroll
      for (int f = 0; f < AHEAD; ++f) k_read(f);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < QK; ++f) {
        s[f & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[f], qf[f >> 1], s[f & 1], 0, 0, 0);
        if (f + AHEAD < QK) k_read(f + AHEAD);
        else v_read(f + AHEAD - QK);
        __builtin_amdgcn_sched_barrier(0);
      }
      // place k of the lane's keys is key c0 + k
      const int c0 = j0 + 4 * lh, last = pos - c0, first = low - c0, kept = with_kept ? merged - 4 * lh : p.keep - c0;
      if (cut_low) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int k = 32 * t + 8 * (r >> 2) + (r & 3);
            bool vis = k >= first;
            if constexpr (EXT) vis = vis || k < kept;
            s[t][r] = vis && k <= last ? s[t][r] : -INFINITY;
          }
      } else if (cut_high) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[t][r] = 32 * t + 8 * (r >> 2) + (r & 3) <= last ? s[t][r] : -INFINITY;
      }
      float mx[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        mx[e] = fmaxf(s[0][e], s[1][e]);
#pragma unroll
        for (int r = 4; r < 16; r += 4) mx[e] = fmaxf(mx[e], fmaxf(s[0][r + e], s[1][r + e]));
      }
      float m_lo, m_hi;
      rows_pair32(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])), m_lo, m_hi);
      const float m_new = fmaxf(m_run, fmaxf(m_lo, m_hi));
      const float m_use = m_new == -INFINITY ? 0.0f : m_new * L2E;
      if (__any(m_new != m_run)) {
        const float corr = __builtin_amdgcn_exp2f(fmaf(m_run, L2E, -m_use));       // exp2(-inf) = 0 at the first tile
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= corr;
        l_run *= corr;
        m_run = m_new;
      }
      // weights of sixteen keys at a time, under the products of the sixteen before
      float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      bf16x8 pf[4];
      auto weights = [&](int ss, int from, int to) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (i < from || i >= to) continue;
          const int t = ss >> 1, r = 8 * (ss & 1) + i;
          const float e = __builtin_amdgcn_exp2f(fmaf(s[t][r], L2E, -m_use));
          sum[r & 3] += e;
          pf[ss][i] = (bf16_t)e;
        }
      };
      weights(0, 0, 8);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < PV; ++f) {
        const int ss = f / DT, dt = f % DT;
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[f], pf[ss], o[dt], 0, 0, 0);
        if (f + AHEAD < PV) v_read(f + AHEAD);
        if (ss < 3) weights(ss + 1, 8 / DT * dt, 8 / DT * (dt + 1));
        __builtin_amdgcn_sched_barrier(0);
      }
      l_run += (sum[0] + sum[1]) + (sum[2] + sum[3]);
    }
    if (wave_on) {
      float none[4] = {0.0f, 0.0f, 0.0f, 0.0f};       // 0 times every number: NaN where one is not finite
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) none[r & 3] = fmaf(o[dt][r], 0.0f, none[r & 3]);
      const bool odd = !((none[0] + none[1]) + (none[2] + none[3]) == 0.0f);
      const uint64_t odd_lanes = __ballot(odd && valid);
      float l_lo, l_hi;
      rows_pair32(l_run, l_lo, l_hi);
      int again = rr;                           // what the walk does not need is formed anew: registers
      asm volatile("" : "+v"(again));
      if (again < rows) {
        const int tok = again / R, head = g * R + again % R;
        const float* gates = p.gate ? p.gate + (ts + tok) * p.gate_rs : nullptr;
        float fs, den;
        close_softmax(m_run, l_lo + l_hi, sink != nullptr, sink ? ld_f32<bf16_t>(sink + head) : 0.0f, fs, den);
        float f = p.out_scale * fs / den;
        const float* grow = gates;
        if (EXT && p.gate_head) {
          if (grow) f *= sigmoid_f32(head_gate);
          grow = nullptr;
        }
        bf16_t* orow = reinterpret_cast<bf16_t*>(p.out) + (ts + tok) * p.out_rs + (int64_t)head * D + 4 * lh;
        if (grow) grow += (int64_t)head * D + 4 * lh;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {           // register 4 q + r produced number 32 dt + 8 q + 4 lh + r
            f32x4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              v[r] = o[dt][4 * q + r] * f * (grow ? sigmoid_f32(grow[32 * dt + 8 * q + r]) : 1.0f);
            *reinterpret_cast<uint2*>(orow + 32 * dt + 8 * q) = Pack4<bf16_t>::narrow(v);
          }
      }
      if (odd_lanes != 0) {
        uint64_t args = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(args));         // read again: kept in registers, the arguments slow the walk
        prompt_rows_again<D, EXT>(*reinterpret_cast<const WAttnArgs*>(args), (uint32_t)(odd_lanes | odd_lanes >> 32), row0, ts, b, g,
                                  bs_shift);
      }
    }
    ts = te;
  }
}

template <int D>
hipError_t launch_prompt_attn(WAttnArgs p, int num_seqs, hipStream_t s) {
  p.TQ = PA_ROWS / (p.H / p.G);
  const int64_t seqs = min((int64_t)num_seqs, p.tokens);       // requests that bring a token: each may end inside a tile
  const int64_t tiles = num_seqs > 1 ? (p.tokens - seqs) / p.TQ + seqs : (p.tokens + p.TQ - 1) / p.TQ;
  int shift = -1;
  if ((p.block_size & (p.block_size - 1)) == 0)
    for (shift = 0; (1 << shift) < p.block_size;) ++shift;
  const dim3 grid((unsigned)((tiles * p.G + 7) / 8 * 8));
  const bool whole = p.block_size % PA_KEYS == 0 && p.cw < (1 << 24);
  if (p.chunk > 0 || p.keep > 0 || (p.gate && p.gate_head)) {
    if (whole) prompt_attn_kernel<D, true, true><<<grid, dim3(256), 0, s>>>(p, (int)tiles, num_seqs, shift);
    else prompt_attn_kernel<D, true, false><<<grid, dim3(256), 0, s>>>(p, (int)tiles, num_seqs, shift);
  } else {
    if (whole) prompt_attn_kernel<D, false, true><<<grid, dim3(256), 0, s>>>(p, (int)tiles, num_seqs, shift);
    else prompt_attn_kernel<D, false, false><<<grid, dim3(256), 0, s>>>(p, (int)tiles, num_seqs, shift);
  }
  return hipGetLastError();
}
