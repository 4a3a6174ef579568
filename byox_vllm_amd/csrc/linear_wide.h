// nv_linear in 16 bits for many rows: tiles of BM x BN outputs with both operands in LDS, filled by LDS-DMA.  Included by linear.hip.  These
// serve what tiles of 256 x 256 (linear_stream.h) would leave much of the chip idle for.
//
// What bounds it: the matrix cores, and for small products the latency of one round of tiles.
//   * a K block is 128 bytes of every row;
//   * the following blocks' rows go from L2 straight into the other LDS buffers (global_load_lds, 16 bytes per lane) while a
//     block is multiplied; no staging registers, no LDS store instructions.  Tiles of 128 x 128 share a CU in pairs with two buffers
//     each; tiles of 64 x 128 have three, because there a block is multiplied faster than one arrives;
//   * LDS rows are 128 bytes apart and their 16-byte pieces are dealt by XOR with half the row number, through the DMA's
//     source addresses, so the 16 rows that one read phase touches lie in 16 different bank groups;
//   * fragments of the next step of K are read while the current step's matrix instructions run (two register sets);
//   * workgroups that share operands run on one XCD: tile numbers are dealt to the XCDs in contiguous eighths.
// Groups (experts) of unknown size: the grid covers the largest possible number of tiles, every workgroup finds its group
// from the offsets with one wavefront-wide prefix sum, and the surplus leaves at once.
//
// Measured alone: 1000 rows 2048 -> 1024 27 us on tiles of 128 x 128, 19 on 64 x 128.
#pragma once
#include "linear_stream.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mma32(const u32x4& a, const u32x4& b, f32x16 c, bf16_t) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// fp32 numbers as they are (what linear_split.hip cannot split)
__device__ __forceinline__ f32x16 mma32(const u32x4& a, const u32x4& b, f32x16 c, float) {
  // step m takes number 4 half + m of the eight that the two half-wavefronts hold
#pragma unroll
  for (int m = 0; m < 4; ++m) c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[m]), __uint_as_float(b[m]), c, 0, 0, 0);
  return c;
}

// The workgroup's tile of BM rows: false where there is none left for it
struct WidePlace {
  int z, m_tile, n_tile;
  int64_t lo, hi;
};
template <int BM>
__device__ __forceinline__ bool wide_place(const LinArgs& p, int mt_max, int nt_all, int lane, WidePlace& at) {
  at = WidePlace{(int)blockIdx.z, 0, 0, 0, p.M};
  int tile = blockIdx.x;
  if (p.group_off) {
    const int groups = mt_max;       // grouped: the number of groups
    int real = 0;
    for (int base = 0; base < groups; base += 64) {
      const int g = base + lane;
      int mt = g < groups ? (p.group_off[g + 1] - p.group_off[g] + BM - 1) / BM : 0;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) mt += __shfl_xor(mt, o, 64);
      real += mt;
    }
    real = __builtin_amdgcn_readfirstlane(real) * nt_all;
    const int share = (real + 7) / 8, slot = tile >> 3;
    tile = (tile & 7) * share + slot;
    if (slot >= share || tile >= real) return false;
    int before = 0;
    at.z = -1;
    for (int base = 0; base < groups && at.z < 0; base += 64) {
      const int g = base + lane;
      const int mine = g < groups ? (p.group_off[g + 1] - p.group_off[g] + BM - 1) / BM : 0;
      int upto = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(upto, o, 64);
        if (lane >= o) upto += x;
      }
      const uint64_t hit = __ballot(tile < (before + upto) * nt_all);
      if (hit) {
        const int l = __ffsll((unsigned long long)hit) - 1;
        at.z = base + l;
        const int count = __builtin_amdgcn_readlane(mine, l);
        const int local = tile - (before + __builtin_amdgcn_readlane(upto, l) - count) * nt_all;
        at.m_tile = local % count;
        at.n_tile = local / count;
      } else {
        before += __builtin_amdgcn_readlane(upto, 63);
      }
    }
    at.lo = p.group_off[at.z];
    at.hi = p.group_off[at.z + 1];
  } else {
    const int real = mt_max * nt_all, share = (real + 7) / 8, slot = tile >> 3;
    tile = (tile & 7) * share + slot;
    if (slot >= share || tile >= real) return false;
    at.m_tile = tile % mt_max;
    at.n_tile = tile / mt_max;
  }
  return true;
}

// Results of MT x 2 tiles of 32 x 32, the wavefront's first row `row0`: the lane holds row fr of each row tile, columns 8 g + 4 fh + r of
// each column tile
template <typename T, typename TO, int EPI, int MT>
__device__ __forceinline__ void wide_results(const LinArgs& p, const f32x16 (&acc)[2][MT], int z, int64_t row0, int64_t hi, int n0, int wn,
                                             int fr, int fh) {
  constexpr bool GLU = EPI == EPI_GLU;
  TO* O = reinterpret_cast<TO*>(p.out) + z * p.out_bs;
  const T* bias = p.bias ? reinterpret_cast<const T*>(p.bias) + z * p.bias_bs : nullptr;
  typedef typename Pack4<TO>::type P4;
  const bool vec = p.N % 4 == 0 && p.out_rs % 4 == 0 && p.out_bs % 4 == 0 && (uintptr_t)p.out % 16 == 0;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int64_t s = row0 + 32 * i + fr;
    if (s >= hi) continue;
    const float rsc = p.row_scale ? p.row_scale[s] : 1.0f;
    const float gate = EPI == EPI_ROW_GATE && !p.act ? sigmoid_f32(p.epi_ptr[s * p.epi_rs + z]) : 1.0f;
#pragma unroll
    for (int j = 0; j < (GLU ? 1 : 2); ++j) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = n0 + (GLU ? 32 * wn : 64 * wn + 32 * j) + 8 * g + 4 * fh;
        if (n >= p.N) continue;
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = n + r < p.N ? lin_finish<T, EPI>(p, bias, acc[j][i][4 * g + r], GLU ? acc[1][i][4 * g + r] : 0.0f, rsc, gate, s, n + r,
                                                z)
                             : 0.0f;
        TO* o = O + s * p.out_rs + n;
        if (vec) {
          *reinterpret_cast<P4*>(o) = Pack4<TO>::narrow(v);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < p.N) st_f32<TO>(o + r, v[r]);
        }
      }
    }
  }
}

// MT x 2 tiles of 32 x 32 per wavefront, WM wavefronts along the rows, WN along the columns
template <typename TO, int EPI, int MT, int WM, int WN, int STAGES>
__global__ __launch_bounds__(64 * WM * WN, 2) void linear_wide_kernel(LinArgs p, int mt_max, int nt_all) {
  typedef bf16_t T;
  constexpr bool GLU = EPI == EPI_GLU;
  constexpr int NW = WM * WN, BM = 32 * MT * WM, BN = 64 * WN, NOUT = GLU ? BN / 2 : BN;
  constexpr int PER = 8, BK = 8 * PER;                              // numbers per 16-byte piece; per K block
  constexpr int AG = BM / 8 / NW, WG = BN / 8 / NW;                 // DMA instructions (8 rows each) per wavefront
  static_assert(AG >= 1 && WG >= 1 && AG * 8 * NW == BM && WG * 8 * NW == BN, "the tile splits into whole DMA instructions");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv % WM, wn = wv / WM;

  WidePlace at;
  if (!wide_place<BM>(p, mt_max, nt_all, lane, at)) return;
  const int z = at.z;
  const int64_t mbase = at.lo + (int64_t)at.m_tile * BM, hi = at.hi;
  const int n0 = at.n_tile * NOUT;
  const T* A = reinterpret_cast<const T*>(p.a) + z * p.a_bs;
  const T* W = reinterpret_cast<const T*>(p.w) + z * p.w_bs;

  // -------- DMA: instruction i of this wavefront fills rows 8 (wv + NW i) .. + 7; lane l the piece l & 7 of row l >> 3
  const int dr = lane >> 3, dp = lane & 7;
  const T* ap[AG];
  const T* wp[WG];
#pragma unroll
  for (int i = 0; i < AG; ++i) {
    const int r = 8 * (wv + NW * i) + dr;
    int64_t s = mbase + r;
    if (s >= hi) s = hi - 1;                                        // rows past the end repeat the last one
    ap[i] = A + (int64_t)(p.a_rows ? p.a_rows[s] : s) * p.a_rs + PER * (dp ^ ((r >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < WG; ++i) {
    const int r = 8 * (wv + NW * i) + dr;
    int row;
    if constexpr (GLU) row = r < BN / 2 ? min(n0 + r, p.N - 1) : p.N + min(n0 + r - BN / 2, p.N - 1);
    else row = min(n0 + r, p.N - 1);
    wp[i] = W + (int64_t)row * p.w_rs + PER * (dp ^ ((r >> 1) & 7));
  }
  typedef __attribute__((address_space(1))) void global_void;
  typedef __attribute__((address_space(3))) void lds_void;
  auto fill = [&](int buf) {
    unsigned char* b = lds_raw + buf * (BM + BN) * 128;
#pragma unroll
    for (int i = 0; i < AG; ++i) {
      __builtin_amdgcn_global_load_lds((global_void*)ap[i], (lds_void*)(b + (wv + NW * i) * 1024), 16, 0, 0);
      ap[i] += BK;
    }
#pragma unroll
    for (int i = 0; i < WG; ++i) {
      __builtin_amdgcn_global_load_lds((global_void*)wp[i], (lds_void*)(b + BM * 128 + (wv + NW * i) * 1024), 16, 0, 0);
      wp[i] += BK;
    }
  };

  const int fr = lane & 31, fh = lane >> 5;
  int a_row[MT], w_row[2];
#pragma unroll
  for (int i = 0; i < MT; ++i) a_row[i] = 32 * (MT * wm + i) + fr;
#pragma unroll
  for (int j = 0; j < 2; ++j) w_row[j] = BM + (GLU ? (BN / 2) * j + 32 * wn : 64 * wn + 32 * j) + fr;
  const int sw = (fr >> 1) & 7;                                     // every tile starts at a multiple of 32 rows
  auto piece = [&](const unsigned char* b, int row, int step) {
    return *reinterpret_cast<const u32x4*>(b + row * 128 + (((2 * step + fh) ^ sw) << 4));
  };

  f32x16 acc[2][MT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;

  const int blocks = p.K / BK;
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i)
    if (i < blocks) fill(i);
  int buf = 0;
  for (int t = 0; t < blocks; ++t) {
    // this wavefront's part of block t has arrived (later blocks may still be on their way), then everybody's has; the
    // barrier also says that block t - 1 is no longer read
    if (STAGES > 2 && t + 1 < blocks) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * (AG + WG)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + STAGES - 1 < blocks) fill(buf == 0 ? STAGES - 1 : buf - 1);
    const unsigned char* b = lds_raw + buf * (BM + BN) * 128;
    buf = buf + 1 == STAGES ? 0 : buf + 1;
    u32x4 wf[2][2], af[2][MT];
#pragma unroll
    for (int j = 0; j < 2; ++j) wf[0][j] = piece(b, w_row[j], 0);
#pragma unroll
    for (int i = 0; i < MT; ++i) af[0][i] = piece(b, a_row[i], 0);
#pragma unroll
    for (int step = 0; step < 4; ++step) {
      const int cur = step & 1, nxt = cur ^ 1;
      if (step < 3) {
#pragma unroll
        for (int j = 0; j < 2; ++j) wf[nxt][j] = piece(b, w_row[j], step + 1);
#pragma unroll
        for (int i = 0; i < MT; ++i) af[nxt][i] = piece(b, a_row[i], step + 1);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j][i] = mma32(wf[cur][j], af[cur][i], acc[j][i], T{});
      // one fragment of the next step is requested behind each of this step's first products; left alone, the compiler
      // puts the reads right before their use
#pragma unroll
      for (int i = 0; i < 2 * MT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (step < 3 && i < MT + 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
  }

  wide_results<T, TO, EPI, MT>(p, acc, z, mbase + 32 * MT * wm, hi, n0, wn, fr, fh);
}

template <typename TO, int EPI, int MT, int WM, int WN, int STAGES>
hipError_t launch_wide_one(const LinArgs& p, int64_t total_rows, int batch, hipStream_t s) {
  constexpr int BM = 32 * MT * WM, BN = 64 * WN, NOUT = EPI == EPI_GLU ? BN / 2 : BN;
  constexpr size_t lds = STAGES * (size_t)(BM + BN) * 128;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> devices{0};
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(&linear_wide_kernel<TO, EPI, MT, WM, WN, STAGES>), lds, devices);
    if (e != hipSuccess) return e;
  }
  const int64_t nt = (p.N + NOUT - 1) / NOUT;
  const int64_t mt = p.group_off ? total_rows / BM + batch : (p.M + BM - 1) / BM;      // at most this many row tiles
  const dim3 grid((unsigned)((mt * nt + 7) / 8 * 8), 1, p.group_off ? 1 : batch);
  linear_wide_kernel<TO, EPI, MT, WM, WN, STAGES><<<grid, dim3(64 * WM * WN), lds, s>>>(p, p.group_off ? batch : (int)mt, (int)nt);
  return hipGetLastError();
}

// Which tile: the one whose launch takes the fewest chip-wide rounds of tile area, each by what it reaches when the chip is
// full (bf16, 32768 rows by 6144 columns of K 2048: 742 and 608 TFLOP/s in the tiles of 128 x 128 and 64 x 128, of which two share a CU; the
// streams of 256 x 256, which have one to themselves, reach 1150 at the K of the smallest products that they are taken for and 1550 at the largest:
// of 629 shapes of 256 to 8192 rows this picks the fastest within 0.5 % on average, 26 of them more than 5 % off).  A last round of 256 x 256
// that half of the chip would have is dealt in halves and costs 0.85 of a round, in 16 bits on four wavefronts less (12000 rows by 2048, K 1024, 1.5 rounds: 65 us, 128 x 128 93, 64 x 128 88; 4096 by 2048, half a round:
// 29.4, 29.3, 33; 5000 by 1536, K 1536: 38, 34, 43).
enum { TILE_256 = 2, TILE_128 = 1, TILE_64 = 0, TILE_256_EIGHT = 3, TILE_256_FOUR = 4 };      // the last two: in 16 bits by so many wavefronts
inline int64_t wide_tiles(int bm, int bn, int64_t m, int64_t total_rows, int cols, int batch, bool grouped) {
  // groups end inside a tile: half a tile each on average
  return (grouped ? (total_rows + bm - 1) / bm + batch / 2 : (m + bm - 1) / bm * batch) * ((cols + bn - 1) / bn);
}
inline int pick_wide_tile(int64_t m, int64_t total_rows, int cols, int batch, bool grouped, bool has_256) {
  auto tiles = [&](int bm, int bn) { return wide_tiles(bm, bn, m, total_rows, cols, batch, grouped); };
  auto rounds = [&](int bm, int bn, int64_t slots, double half) {
    const int64_t n = tiles(bm, bn), over = n % slots;
    return (double)(n / slots) + (over == 0 ? 0.0 : bm == 256 && 2 * over <= slots ? half : 1.0);
  };
  const double c64 = rounds(64, 128, 512, 1.0) * 2 * 64 * 128 / 608, c128 = rounds(128, 128, 512, 1.0) * 2 * 128 * 128 / 742;
  const double c256 = rounds(256, 256, 256, 0.85) * 256 * 256 / 1150;
  if (has_256 && c256 < c128 && c256 < c64) return TILE_256;
  return c128 < c64 ? TILE_128 : TILE_64;
}

// Tiles of the split products, 64 x 128 (two to a CU), 128 x 128 and 256 x 128 (one each): what a chip-wide round of them takes for its K, in
// units of two tiles of 64 x 128 on a CU.  Of 230 shapes (64 to 6000 rows, 32 to 6000 columns, K 64 to 2048, some gated) this picks the
// fastest within 0.5 % on average, five of them 8 to 14 % off, and none is slower than the fp32 instructions' tiles were.  us of 64 x 128, 128 x 128,
// 256 x 128: 256 by 1024, K 1024 27, 38, 65; 3135 by 1024, K 2048 85, 77, 119; 3135 by 4416, K 1024 170, 177, 159.
inline int pick_split_tile(int64_t m, int64_t total_rows, int cols, int K, int batch, bool grouped) {
  const int64_t n64 = wide_tiles(64, 128, m, total_rows, cols, batch, grouped), n128 = wide_tiles(128, 128, m, total_rows, cols, batch, grouped),
                n256 = wide_tiles(256, 128, m, total_rows, cols, batch, grouped);
  const double c64 = n64 <= 256 ? 0.6 : 1.1 * (n64 <= 512 ? 1.0 : n64 / 512.0);
  const double c128 = 1.1 * ((n128 + 255) / 256) - (K >= 512 ? 0.05 : 0.0), c256 = 1.75 * ((n256 + 255) / 256);
  return c64 <= c128 && c64 <= c256 ? SPLIT_64 : c128 <= c256 ? SPLIT_128 : SPLIT_256;
}

template <typename TO, int EPI>
hipError_t launch_wide_epi(const LinArgs& p, int64_t total_rows, int batch, int tile, hipStream_t s) {
  if (tile >= TILE_256) {
    const bool four = stream_deep_takes(p) && (tile == TILE_256 ? linear_four_wavefronts(p, EPI, sizeof(TO) == 2) : tile == TILE_256_FOUR);
    return (four ? linear_deep_launch : linear_eight_launch)(p, EPI, sizeof(TO) == 2, total_rows, batch, s);
  }
  if (tile == TILE_128) return launch_wide_one<TO, EPI, 2, 2, 2, 2>(p, total_rows, batch, s);
  return launch_wide_one<TO, EPI, 1, 2, 2, 3>(p, total_rows, batch, s);
}

template <typename TO>
hipError_t launch_wide(const LinArgs& p, int epi, int64_t total_rows, int batch, int tile, hipStream_t s) {
  switch (epi) {
    case EPI_NONE: return launch_wide_epi<TO, EPI_NONE>(p, total_rows, batch, tile, s);
    case EPI_GLU: return launch_wide_epi<TO, EPI_GLU>(p, total_rows, batch, tile, s);
    case EPI_SOFTCAP: return launch_wide_epi<TO, EPI_SOFTCAP>(p, total_rows, batch, tile, s);
    case EPI_ACT: return launch_wide_epi<TO, EPI_ACT>(p, total_rows, batch, tile, s);
    default: return launch_wide_epi<TO, EPI_ROW_GATE>(p, total_rows, batch, tile, s);
  }
}
