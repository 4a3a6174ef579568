// nv_linear for many rows: the products, groups and epilogues of LinArgs on the tiles of stream_tiles.h.  Included by
// linear.hip.  Groups (experts) of unknown size: every workgroup counts the tiles from the offsets with one wavefront-wide prefix
// sum; a group that ends in the upper half of a tile's rows costs the half.
#pragma once
#include <type_traits>

#include "stream_tiles.h"

// value(s) of one output -> what is stored (bias, activation, gate); `gate`: the row's, where there is one for all of it
template <typename T, int EPI, int ACT = -1>
__device__ __forceinline__ float lin_finish(const LinArgs& p, const T* bias, float v, float u, float rsc, float gate, int64_t s, int n,
                                            int z) {
  v *= rsc;
  if (bias) v += ld_f32<T>(bias + n);
  if constexpr (EPI == EPI_GLU) {
    u *= rsc;
    if (bias) u += ld_f32<T>(bias + p.N + n);
    v = glu_act(v, u, p.act, p.epi_c);
  } else if constexpr (EPI == EPI_SOFTCAP) {
    v = p.epi_c * tanhf(v / p.epi_c);
  } else if constexpr (EPI == EPI_ROW_GATE) {
    v *= p.act ? sigmoid_f32(p.epi_ptr[s * p.epi_rs + (int64_t)z * p.N + n]) : gate;
  } else if constexpr (EPI == EPI_ACT) {
    v = unary_act(v, ACT < 0 ? p.act : ACT, p.epi_ptr, p.epi_c);
  }
  return v;
}

// eight consecutive results of one row -> 16 bytes
__device__ __forceinline__ u32x4 pack8(const float* v) {
  return u32x4{pack2<bf16_t>(v[0], v[1]), pack2<bf16_t>(v[2], v[3]), pack2<bf16_t>(v[4], v[5]), pack2<bf16_t>(v[6], v[7])};
}

template <typename TT, typename TO, int EPI>
struct LinearJob {
  typedef TT T;
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
  __device__ __forceinline__ const void* w_base(const StreamTile& at) const { return reinterpret_cast<const T*>(p.w) + at.z * p.w_bs; }
  __device__ __forceinline__ uint32_t w_stride() const { return (uint32_t)p.w_rs * sizeof(T); }
  __device__ __forceinline__ uint32_t w_row(const StreamTile& at, int r) const {
    // a wavefront's 64 rows: 64 columns, or 32 columns' gates and the same columns' ups
    if constexpr (GLU) return min(at.n0 + 32 * (r >> 6) + (r & 31), p.N - 1) + ((r & 32) ? p.N : 0);
    else return min(at.n0 + r, p.N - 1);
  }
  __device__ __forceinline__ uint32_t w_step() const { return 128; }
  __device__ __forceinline__ bool whole(const StreamTile& at) const {
    return vec && at.lo + BM <= at.hi && at.n0 + NOUT <= p.N;
  }
  __device__ __forceinline__ void store(const StreamTile& at, int64_t row0, int wn, int lane, const f32x4 (&acc)[NT][MT]) const {
    if constexpr (EPI == EPI_ACT) {      // one function per copy: with the choice inside, the loops would not unroll
      switch (p.act) {
        case 0: return store_as<0>(at, row0, wn, lane, acc);
        case 1: return store_as<1>(at, row0, wn, lane, acc);
        case 2: return store_as<2>(at, row0, wn, lane, acc);
        case 4: return store_as<4>(at, row0, wn, lane, acc);
        default: return store_as<3>(at, row0, wn, lane, acc);
      }
    } else {
      store_as<-1>(at, row0, wn, lane, acc);
    }
  }
  template <int ACT>
  __device__ __forceinline__ void store_as(const StreamTile& at, int64_t row0, int wn, int lane, const f32x4 (&acc)[NT][MT]) const {
    const int fr = lane & 15, g = lane >> 4;
    TO* O = reinterpret_cast<TO*>(p.out) + at.z * p.out_bs;
    const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + at.z * p.bias_bs : nullptr;
    constexpr int LEN = PAIRED ? 8 : 4, PIECES = (GLU ? 2 : 4) * 4 / LEN, UP = 2;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      __builtin_amdgcn_sched_barrier(0);       // one row's results at a time: registers
      const int64_t s = row0 + 16 * i + fr;
      if (s >= at.hi) continue;
      const float rsc = p.row_scale ? p.row_scale[s] : 1.0f;
      const float gate = EPI == EPI_ROW_GATE && !p.act ? sigmoid_f32(p.epi_ptr[s * p.epi_rs + at.z]) : 1.0f;
      auto result = [&](int q, int e, int n) {
        const int j = q * (LEN / 4) + e / 4;
        return lin_finish<T, EPI, ACT>(p, bias, acc[j][i][e & 3], GLU ? acc[(j + UP) % NT][i][e & 3] : 0.0f, rsc, gate, s, n + e, at.z);
      };
      TO* o = O + s * p.out_rs;
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
  }
};

// two K blocks at least, row strides whose bytes are 32-bit numbers, tiles that fit the workgroups' lists
inline bool stream_takes(const LinArgs& p, int esz, int64_t total_rows, int batch, int cols) {
  const int64_t rows = p.group_off ? total_rows / 256 + batch : (p.M + 255) / 256 * batch;
  if (total_rows >= ((int64_t)1 << 31) || rows * ((cols + 255) / 256) > 256 * (STREAM_LIST - 2)) return false;
  return p.K * esz >= 256 && p.K * esz % 128 == 0 && p.a_rs >= 0 && p.w_rs >= 0 && p.a_rs < ((int64_t)1 << 30) && p.w_rs < ((int64_t)1 << 30);
}

template <typename T, typename TO, int EPI>
hipError_t launch_stream_epi(const LinArgs& p, int64_t total_rows, int batch, hipStream_t s) {
  typedef LinearJob<T, TO, EPI> Job;
  constexpr int64_t unit = sizeof(TO) == 2 ? 8 : 4;
  const int nt = (p.N + Job::NOUT - 1) / Job::NOUT;
  const int vec = p.N % unit == 0 && p.out_rs % unit == 0 && p.out_bs % unit == 0 && (uintptr_t)p.out % 16 == 0;
  const Job job{p, p.K, p.group_off ? batch : 0, batch, nt, vec};
  return launch_stream_tiles<4>(job, (p.group_off ? total_rows / Job::BM + batch : (p.M + Job::BM - 1) / Job::BM * batch) * nt, s);
}
