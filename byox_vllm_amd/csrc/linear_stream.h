// nv_linear for many rows: the products, groups and epilogues of LinArgs in 16 bits on the tiles of stream_tiles.h (linear_eight.hip)
// and stream_deep.h (linear_deep.hip).  Groups (experts) of unknown size: every workgroup counts the tiles from the offsets with one
// wavefront-wide prefix sum; a group that ends in the upper half of a tile's rows costs the half.
#pragma once
#include <type_traits>

#include "linear_args.h"
#include "stream_deep.h"

// value(s) of one output, bias and scale included -> what the epilogue makes of it; `gate`: the row's
template <int EPI, int ACT = -1>
__device__ __forceinline__ float lin_epilogue(const LinArgs& p, float v, float u, float gate) {
  if constexpr (EPI == EPI_GLU) return glu_act(v, u, ACT < 0 ? p.act : ACT, p.epi_c);
  else if constexpr (EPI == EPI_SOFTCAP) return p.epi_c * tanhf(v / p.epi_c);
  else if constexpr (EPI == EPI_ROW_GATE) return v * gate;
  else if constexpr (EPI == EPI_ACT) return unary_act(v, ACT < 0 ? p.act : ACT, p.epi_ptr, p.epi_c);
  else return v;
}
// the same with scale, bias and gate taken from memory here
template <typename T, int EPI, int ACT = -1>
__device__ __forceinline__ float lin_finish(const LinArgs& p, const T* bias, float v, float u, float rsc, float gate, int64_t s, int n,
                                            int z) {
  v *= rsc;
  if (bias) v += ld_f32<T>(bias + n);
  if constexpr (EPI == EPI_GLU) {
    u *= rsc;
    if (bias) u += ld_f32<T>(bias + p.N + n);
  }
  if constexpr (EPI == EPI_ROW_GATE)
    if (p.act) gate = sigmoid_f32(p.epi_ptr[s * p.epi_rs + (int64_t)z * p.N + n]);
  return lin_epilogue<EPI, ACT>(p, v, u, gate);
}

// eight consecutive results of one row -> 16 bytes
__device__ __forceinline__ u32x4 pack8(const float* v) {
  return u32x4{pack2<bf16_t>(v[0], v[1]), pack2<bf16_t>(v[2], v[3]), pack2<bf16_t>(v[4], v[5]), pack2<bf16_t>(v[6], v[7])};
}

template <typename TO, int EPI, bool FAR_UPS = false>     // FAR_UPS: a gated product's ups lie 4 GiB and more from their gates
struct LinearJob {
  typedef bf16_t T;
  static constexpr int BM = STREAM_BM, MT = 8, NT = 4;              // four wavefronts along the columns
  static constexpr bool GLU = EPI == EPI_GLU, PAIRED = sizeof(TO) == 2;
  typedef std::conditional_t<PAIRED, StreamPaired, StreamNatural> Order;
  static constexpr int NOUT = GLU ? 128 : 256;                      // columns of results per tile
  static constexpr int NSTORE = BM / 32 * (PAIRED ? 2 : 4) / (GLU ? 2 : 1);
  LinArgs p;
  int K, groups, batch, nt, vec;      // groups: 0, or the number of them

  __device__ __forceinline__ static int row_tiles(int rows) { return (rows + BM - 1) / BM; }
  __device__ __forceinline__ int group_tiles(int g) const { return g < groups ? row_tiles(p.group_off[g + 1] - p.group_off[g]) : 0; }
  __device__ __forceinline__ int count(int lane) const {
    if (!groups) return row_tiles((int)p.M) * nt * batch;
    int all = 0;
    for (int base = 0; base < groups; base += 64) {
      int n = group_tiles(base + lane);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
      all += n;
    }
    return __builtin_amdgcn_readfirstlane(all) * nt;
  }
  __device__ __forceinline__ StreamTile find(int tile, int lane) const {
    StreamTile at{0, (int)p.M, 0, 0};
    int rows = row_tiles((int)p.M), in = tile, m_tile, n_tile;
    if (!groups) {
      at.z = tile / (rows * nt);
      in = tile - at.z * rows * nt;
    } else {
      int before = 0;
      bool found = false;
      for (int base = 0; base < groups; base += 64) {
        const int mine = group_tiles(base + lane);
        for (int l = 0; l < 64 && base + l < groups; ++l) {
          const int here = __builtin_amdgcn_readlane(mine, l);
          if (!found && tile < (before + here) * nt) {
            found = true;
            at.z = base + l;
            rows = here;
            in = tile - before * nt;
          }
          before += here;
        }
      }
      at.lo = p.group_off[at.z];
      at.hi = p.group_off[at.z + 1];
    }
    stream_order(in, rows, nt, m_tile, n_tile);
    at.lo += m_tile * BM;
    at.n0 = n_tile * NOUT;
    return at;
  }
  __device__ __forceinline__ const void* a_base(const StreamTile& at) const { return reinterpret_cast<const T*>(p.a) + at.z * p.a_bs; }
  __device__ __forceinline__ uint32_t a_stride() const { return (uint32_t)p.a_rs * sizeof(T); }
  __device__ __forceinline__ uint32_t a_row(const StreamTile& at, int r) const {
    const int s = min(at.lo + r, at.hi - 1);
    return (uint32_t)(p.a_rows ? p.a_rows[s] : s);
  }
  // W's rows from the tile's first on; gates and ups within 4 GiB from the matrix's first
  static constexpr bool MOVES = !GLU || FAR_UPS;
  __device__ __forceinline__ const void* w_base(const StreamTile& at) const {
    return reinterpret_cast<const T*>(p.w) + at.z * p.w_bs + (MOVES ? at.n0 * p.w_rs : 0);
  }
  __device__ __forceinline__ uint32_t w_stride() const { return (uint32_t)p.w_rs * sizeof(T); }
  __device__ __forceinline__ uint64_t w_ups() const { return (uint64_t)p.N * p.w_rs * sizeof(T); }
  __device__ __forceinline__ uint32_t w_row(const StreamTile& at, int r) const {
    const int n0 = MOVES ? 0 : at.n0, last = MOVES ? p.N - at.n0 - 1 : p.N - 1;
    // a wavefront's 64 rows: 64 columns, or 32 columns' gates and the same columns' ups
    if constexpr (GLU) return min(n0 + 32 * (r >> 6) + (r & 31), last) + (!UPS && (r & 32) ? p.N : 0);
    else return min(r, last);
  }
  __device__ __forceinline__ uint32_t w_step() const { return 128; }
  __device__ __forceinline__ bool whole(const StreamTile& at) const {
    return vec && at.lo + BM <= at.hi && at.n0 + NOUT <= p.N;
  }
  static constexpr int NSTORE_WAVE = 2 * NSTORE, EXTRA = 0;
  static constexpr bool FAR_A = true, FAR_W = false, UPS = FAR_UPS;      // A's rows may lie anywhere; W's: stream_takes
  __device__ __forceinline__ void fetch_extra(const StreamTile&, int, int, unsigned char*) const {}
  __device__ __forceinline__ void finish(const StreamTile& at, int wm, int wn, int lane, bool live0, bool live1, const unsigned char*) const {
    if (live0) store_wave<0>(at, at.lo + 64 * wm, wn, lane);
    if (live1) store_wave<1>(at, at.lo + 128 + 64 * wm, wn, lane);
  }
  // 64 rows by 128 rows of W of stream_deep.h.  What the results need of memory is fetched ahead of the first store: loads and stores
  // are counted in one order, so a load behind a store is waited for behind it too.
  template <int HALF>
  __device__ __forceinline__ void store_wave(const StreamTile& at, int row0, int wn, int lane) const {
    if (!vec || (EPI == EPI_ROW_GATE && p.act)) {
      store<4>(at, row0, 2 * wn, lane, [](int j, int i) { return deep_take(HALF, j, i); });
      store<4>(at, row0, 2 * wn + 1, lane, [](int j, int i) { return deep_take(HALF, 4 + j, i); });
      return;
    }
    if constexpr (EPI == EPI_NONE) {
      if (!p.bias && !p.row_scale) return store_ahead<HALF, -1, false>(at, row0, wn, lane);
    }
    if constexpr (EPI == EPI_GLU) {
      switch (p.act) {      // as glu_act: what is neither GELU nor the clamped unit is SiLU
        case 1: return store_ahead<HALF, 1, true>(at, row0, wn, lane);
        case 2: return store_ahead<HALF, 2, true>(at, row0, wn, lane);
        default: return store_ahead<HALF, 0, true>(at, row0, wn, lane);
      }
    } else if constexpr (EPI == EPI_ACT) {
      switch (p.act) {
        case 0: return store_ahead<HALF, 0, true>(at, row0, wn, lane);
        case 1: return store_ahead<HALF, 1, true>(at, row0, wn, lane);
        case 2: return store_ahead<HALF, 2, true>(at, row0, wn, lane);
        case 4: return store_ahead<HALF, 4, true>(at, row0, wn, lane);
        default: return store_ahead<HALF, 3, true>(at, row0, wn, lane);
      }
    } else {
      store_ahead<HALF, -1, true>(at, row0, wn, lane);
    }
  }
  template <int HALF, int ACT, bool MORE>      // MORE: scale, bias or gate; 1 and -0, which change nothing, where there is none
  __device__ __forceinline__ void store_ahead(const StreamTile& at, int row0, int wn, int lane) const {
    constexpr int LEN = PAIRED ? 8 : 4, PIECES = (GLU ? 2 : 4) * 4 / LEN, UP = 2;
    const int fr = lane & 15, g = lane >> 4;
    float rsc[4], gate[4], bias[2][PIECES * LEN], up[GLU ? 2 : 1][GLU ? PIECES * LEN : 1];
    int n[2][PIECES];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < PIECES; ++q) n[h][q] = at.n0 + (GLU ? 32 : 64) * (2 * wn + h) + 4 * LEN * q + LEN * g;
    if constexpr (MORE) {
#pragma unroll
      for (int i = 0; i < 4; ++i) rsc[i] = gate[i] = 1.0f;
      if (p.row_scale) {
#pragma unroll
        for (int i = 0; i < 4; ++i) rsc[i] = p.row_scale[min(row0 + 16 * i + fr, at.hi - 1)];
      }
      if constexpr (EPI == EPI_ROW_GATE) {
#pragma unroll
        for (int i = 0; i < 4; ++i) gate[i] = p.epi_ptr[min(row0 + 16 * i + fr, at.hi - 1) * p.epi_rs + at.z];
#pragma unroll
        for (int i = 0; i < 4; ++i) gate[i] = sigmoid_f32(gate[i]);
      }
      // one branch for all of them, or each is waited for by itself
      if (p.bias) {
        const T* from = reinterpret_cast<const T*>(p.bias) + at.z * p.bias_bs;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < PIECES; ++q)
#pragma unroll
            for (int e = 0; e < LEN; ++e) {
              const int at_n = min(n[h][q], p.N - LEN) + e;
              bias[h][q * LEN + e] = ld_f32<T>(from + at_n);
              if constexpr (GLU) up[h][q * LEN + e] = ld_f32<T>(from + p.N + at_n);
            }
      } else {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < PIECES * LEN; ++e) {
            bias[h][e] = -0.0f;
            if constexpr (GLU) up[h][e] = -0.0f;
          }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(rsc[i]), "+v"(gate[i]));      // all of them waited for here
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < PIECES * LEN; ++e) {
          asm volatile("" : "+v"(bias[h][e]));
          if constexpr (GLU) asm volatile("" : "+v"(up[h][e]));
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t s = row0 + 16 * i + fr;
      TO* o = reinterpret_cast<TO*>(p.out) + at.z * p.out_bs + s * p.out_rs;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        __builtin_amdgcn_sched_barrier(0);       // one row's results at a time: registers
        f32x4 x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = deep_take(HALF, 4 * h + j, i);
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
          float v[LEN];
#pragma unroll
          for (int e = 0; e < LEN; ++e) {
            const int j = q * (LEN / 4) + e / 4;
            float a = x[j][e & 3], u = GLU ? x[(j + UP) % NT][e & 3] : 0.0f;
            if constexpr (MORE) {
              a = a * rsc[i] + bias[h][q * LEN + e];
              if constexpr (GLU) u = u * rsc[i] + up[h][q * LEN + e];
            }
            if constexpr (GLU && ACT == 0 && PAIRED) v[e] = silu_16bit(a) * u;
            else v[e] = lin_epilogue<EPI, ACT>(p, a, u, MORE ? gate[i] : 1.0f);
          }
          if (s < at.hi && n[h][q] < p.N) {
            if constexpr (PAIRED) *reinterpret_cast<u32x4*>(o + n[h][q]) = pack8(v);
            else *reinterpret_cast<f32x4*>(o + n[h][q]) = f32x4{v[0], v[1], v[2], v[3]};
          }
        }
      }
    }
  }
  template <int ROWS, typename Take>
  __device__ __forceinline__ void store(const StreamTile& at, int64_t row0, int wn, int lane, Take take) const {
    if constexpr (EPI == EPI_ACT) {      // one function per copy: with the choice inside, the loops would not unroll
      switch (p.act) {
        case 0: return store_as<0, ROWS>(at, row0, wn, lane, take);
        case 1: return store_as<1, ROWS>(at, row0, wn, lane, take);
        case 2: return store_as<2, ROWS>(at, row0, wn, lane, take);
        case 4: return store_as<4, ROWS>(at, row0, wn, lane, take);
        default: return store_as<3, ROWS>(at, row0, wn, lane, take);
      }
    } else {
      store_as<-1, ROWS>(at, row0, wn, lane, take);
    }
  }
  template <int ACT, int ROWS, typename Take>
  __device__ __forceinline__ void store_as(const StreamTile& at, int64_t row0, int wn, int lane, Take take) const {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      __builtin_amdgcn_sched_barrier(0);       // one row's results at a time: registers
      f32x4 x[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) x[j] = take(j, i);
      const int64_t s = row0 + 16 * i + (lane & 15);
      if (s < at.hi) store_row<ACT>(at, s, wn, lane, x);
    }
  }
  template <int ACT>
  __device__ __forceinline__ void store_row(const StreamTile& at, int64_t s, int wn, int lane, const f32x4 (&x)[NT]) const {
    const int g = lane >> 4;
    const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + at.z * p.bias_bs : nullptr;
    constexpr int LEN = PAIRED ? 8 : 4, PIECES = (GLU ? 2 : 4) * 4 / LEN, UP = 2;
    float rsc = 1.0f;
    if (p.row_scale) {
      rsc = p.row_scale[s];
      asm volatile("" : "+v"(rsc));       // waited for here: pending on a path without its use, it would be waited for in the loop over blocks
    }
    const float gate = EPI == EPI_ROW_GATE && !p.act ? sigmoid_f32(p.epi_ptr[s * p.epi_rs + at.z]) : 1.0f;
    auto result = [&](int q, int e, int n) {
      const int j = q * (LEN / 4) + e / 4;
      return lin_finish<T, EPI, ACT>(p, bias, x[j][e & 3], GLU ? x[(j + UP) % NT][e & 3] : 0.0f, rsc, gate, s, n + e, at.z);
    };
    TO* o = reinterpret_cast<TO*>(p.out) + at.z * p.out_bs + s * p.out_rs;
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
      const int n = at.n0 + (GLU ? 32 : 64) * wn + 4 * LEN * q + LEN * g;
      if (vec) {
        if (n >= p.N) continue;
        float v[LEN];
#pragma unroll
        for (int e = 0; e < LEN; ++e) v[e] = result(q, e, n);
        if constexpr (PAIRED) *reinterpret_cast<u32x4*>(o + n) = pack8(v);
        else *reinterpret_cast<f32x4*>(o + n) = f32x4{v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int e = 0; e < LEN; ++e)
          if (n + e < p.N) st_f32<TO>(o + n + e, result(q, e, n));
      }
    }
  }
};

// two K blocks at least, row strides whose bytes are 32-bit numbers, tiles that fit the workgroups' lists
inline bool stream_takes(const LinArgs& p, int esz, int64_t total_rows, int batch, int cols) {
  const int64_t rows = p.group_off ? total_rows / 256 + batch : (p.M + 255) / 256 * batch;
  if (total_rows >= ((int64_t)1 << 31) || rows * ((cols + 255) / 256) > 256 * (STREAM_LIST - 2)) return false;
  return p.K * esz >= 256 && p.K * esz % 128 == 0 && p.a_rs >= 0 && p.w_rs >= 0 && p.a_rs < ((int64_t)1 << 30) && p.w_rs < ((int64_t)1 << 30);
}

inline bool stream_vec(const LinArgs& p, bool out_16bit) {      // whether a row's results are stored 16 bytes at a time
  const int64_t unit = out_16bit ? 8 : 4;
  return p.N % unit == 0 && p.out_rs % unit == 0 && p.out_bs % unit == 0 && (uintptr_t)p.out % 16 == 0;
}

// stream_deep.h has a tile's 256 rows of W within 4 GiB, stream_tiles.h anywhere
inline bool stream_deep_takes(const LinArgs& p) { return p.w_rs < ((int64_t)1 << 23); }

// Whether a 16-bit product's 256 x 256 tiles are four wavefronts' (stream_deep.h) or eight's (stream_tiles.h).  Four are faster over K (0.8 - 0.9 of
// the time at long K), but alone on their SIMDs: nothing runs under the chains of instructions of a result's function, its gate or bias fetched for it
// alone, stores of single numbers.  Results that eight take longer for, because they fetch a bias where it is added, are four's from the first
// K on.  Four against eight, 16384 rows by 2048, bf16: plain K 192 0.97, 256 0.89 (6000 by 1536 1.09, 0.97); with a bias 0.61; SiLU 512 1.07, 1024
// 1.01; GELU 2048 1.08, 4096 0.99, with a bias 512 1.05, 1024 1.01, gated 192 1.08, 512 0.95; xIELU 4096 1.07, 8192 0.91; soft cap 2048 1.05,
// 4096 0.97; a gate for every number 4096 1.13, 8192 0.97; 2044 columns and a bias 4096 1.04, 8192 0.92, gated 2048 1.24, 8192 0.90.
inline bool linear_four_wavefronts(const LinArgs& p, int epi, bool out_16bit) {
  static const int from[11][4] = {      // K from which four are faster: 16 bytes at a time, and a bias; numbers one by one, and a bias
      {256, 0, 512, 8192},              // plain
      {0, 0, 8192, 8192},               // gated
      {3072, 0, 1024, 8192},            // soft cap
      {0, 0, 4096, 8192},               // a gate for a row
      {8192, 8192, 8192, 8192},         // a gate for a number
      {1024, 0, 1024, 8192},            // SiLU
      {4096, 1024, 4096, 8192},         // GELU, tanh form
      {8192, 4608, 8192, 8192},         // xIELU
      {384, 0, 512, 8192},              // multiplication
      {3072, 0, 4096, 8192},            // GELU, erf form
      {512, 0, 8192, 8192}};            // gated by GELU
  const int what = epi == EPI_ACT ? 5 + p.act : epi == EPI_ROW_GATE ? (p.act ? 4 : 3) : epi == EPI_GLU && p.act == 1 ? 10 : epi;
  return p.K >= from[what][(stream_vec(p, out_16bit) ? 0 : 2) + (p.bias ? 1 : 0)];
}

template <typename TO, int EPI, bool FAR_UPS = false>
LinearJob<TO, EPI, FAR_UPS> linear_job(const LinArgs& p, int batch) {
  typedef LinearJob<TO, EPI, FAR_UPS> Job;
  const int nt = (p.N + Job::NOUT - 1) / Job::NOUT;
  return Job{p, p.K, p.group_off ? batch : 0, batch, nt, stream_vec(p, sizeof(TO) == 2)};
}
inline int64_t linear_job_tiles(const LinArgs& p, int nt, int64_t total_rows, int batch) {      // at most
  return (p.group_off ? total_rows / STREAM_BM + batch : (p.M + STREAM_BM - 1) / STREAM_BM * batch) * nt;
}
