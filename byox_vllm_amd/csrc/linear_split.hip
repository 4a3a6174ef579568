// nv_linear in fp32 for many rows: fp32 products by the 16-bit matrix instructions, which are 16 times as fast.
//
// A number of fp32 is the sum of three of bf16, exactly: x = h + m + l with h = bf16(x), m = bf16(x - h), l = x - h - m.  Of the nine products
// of two such sums the six largest are added up in fp32; the three left out are below 2^-25 of the product of the two numbers.  Off float64,
// normal values, K 96, 1024, 2048: 1.4e-7, 4.9e-7, 7.0e-7 of the norm (the fp32 instructions' sums 1.8e-7, 5.7e-7, 8.1e-7, which add K one by
// one).
//
// What bounds it: the matrix cores, 16-bit products at up to 1.3 PFLOP/s while a chip-wide round is full, and in smaller launches the issue of
// one wavefront to a SIMD, which has five other instructions to a product in tiles of 128 x 128 and four in 256 x 128.
//   * A block's rows go through registers once to be split, eight numbers to a lane, and lie in LDS as parts; the sixteen numbers of K that a
//     product takes come in any order, the same for both operands, so a lane's eight are two pieces of 16 bytes that are 64 bytes apart.
//   * The instructions of the split stand between the products, one step behind each, in an order without waits (sched_barrier; left alone
//     the compiler puts them in lumps that the products wait for: 3135 rows 1024 -> 4416 in 128 x 128 189 us, 177).
//   * The barrier stands before a block's second step, whose fragments are in registers by then.
// Measured against the fp32 instructions' tiles: 3135 rows 1024 -> 4416 303 and 160 us, 2048 -> 1024 143 and 77, 512 rows 512 -> 1536 23.5 and
// 16.8; of 230 shapes of K 64 to 2048 none slower, 0.97 of the time at K 64, 0.78 at 256, 0.63 at 2048.
#include <utility>

#include "lds_limit.h"
#include "linear_args.h"

namespace {

#include "linear_wide.h"

// f(0), f(1) .. f(N - 1) with numbers that are constants
template <int... I, typename F> __device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, const F& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void each(const F& f) { each_of(std::make_integer_sequence<int, N>{}, f); }

// The third part of a number below 2^-110 is below the least number of bf16.  So both operands are multiplied by SCALE, which brings all
// numbers of fp32 above that, and the sums by its inverse square; what this makes too large is formed without parts, as are infinities.
constexpr float SCALE = 1099511627776.0f;      // 2^40

// MT x 2 tiles of 32 x 32 per wavefront, WM wavefronts along the rows, WN along the columns
template <typename TO, int EPI, int MT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void linear_split_kernel(LinArgs p, int mt_max, int nt_all) {
  constexpr bool GLU = EPI == EPI_GLU;
  constexpr int NT = 64 * WM * WN, BM = 32 * MT * WM, BN = 64 * WN, NOUT = GLU ? BN / 2 : BN, ROWS = BM + BN;
  constexpr int RP = 4 * ROWS / NT, BUF = ROWS * 192;      // rows that a thread splits; bytes of a block's parts
  constexpr int R0 = (RP + 1) / 2;
  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, R0> IR{};
  constexpr std::integral_constant<int, RP> IP{};
  static_assert(RP * NT == 4 * ROWS && NT / 4 % 16 == 0 && BM % (NT / 4) == 0, "whole rows to a thread, W's behind A's");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv % WM, wn = wv / WM;
  WidePlace at;
  if (!wide_place<BM>(p, mt_max, nt_all, lane, at)) return;
  const int64_t mbase = at.lo + (int64_t)at.m_tile * BM, hi = at.hi;
  const int n0 = at.n_tile * NOUT;
  const float* A = reinterpret_cast<const float*>(p.a) + at.z * p.a_bs;
  const float* W = reinterpret_cast<const float*>(p.w) + at.z * p.w_bs;
  auto a_row = [&](int r) {                                         // rows past the end repeat the last one
    int64_t s = mbase + r;
    if (s >= hi) s = hi - 1;
    return A + (int64_t)(p.a_rows ? p.a_rows[s] : s) * p.a_rs;
  };
  auto w_row = [&](int r) {
    int row;
    if constexpr (GLU) row = r < BN / 2 ? min(n0 + r, p.N - 1) : p.N + min(n0 + r - BN / 2, p.N - 1);
    else row = min(n0 + r, p.N - 1);
    return W + (int64_t)row * p.w_rs;
  };

  // -------- a thread splits eight numbers of every NT / 4th row: from memory through registers into LDS
  const int sr = tid >> 2, sk = tid & 3;
  const float* from[RP];
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    const int r = sr + NT / 4 * i;
    from[i] = (NT / 4 * i < BM ? a_row(r) : w_row(r - BM)) + 4 * sk;
  }
  f32x4 raw[RP][2];
  auto fetch = [&](int i, int k) {
    raw[i][0] = *reinterpret_cast<const f32x4*>(from[i] + k);
    raw[i][1] = *reinterpret_cast<const f32x4*>(from[i] + k + 16);
  };
  // Row r of a block: 192 bytes, 64 of each part, in pieces of 16 that are dealt by XOR with (r >> 2) & 3, so that the 16 rows that a read
  // touches lie in 16 bank groups.
  const int put_at = sr * 192 + ((sk ^ ((sr >> 2) & 3)) << 4);
  // The split of rows i0 .. i1 - 1 in steps whose instructions do not wait for each other: step n rounds a pair of numbers to its part,
  // widens the pair of the step before and takes that of the one before that off its numbers.  Twelve to a row: four pairs, three parts.
  u32x4 part[RP][3];
  float wide[RP][2][8];
  auto split = [&](auto i0, auto i1, auto step, int bo, int k_next) {
    constexpr int n = step, last = 12 * (i1 - i0);
    each<2>([&](auto behind) {      // the pairs of a row's first four steps times SCALE, a step ahead
      constexpr int m = n + behind;
      if constexpr (m < last && m % 12 < 4 && (behind == 1 || n == 0)) {
        constexpr int i = i0 + m / 12, e = m % 4;
#pragma unroll
        for (int h = 0; h < 2; ++h) raw[i][e >> 1][2 * (e & 1) + h] *= SCALE;
      }
    });
    if constexpr (n >= 2 && n - 2 < last && (n - 2) % 12 < 8) {
      constexpr int i = i0 + (n - 2) / 12, t = (n - 2) % 12 / 4, e = (n - 2) % 4;
#pragma unroll
      for (int h = 0; h < 2; ++h) raw[i][e >> 1][2 * (e & 1) + h] -= wide[i][t][2 * e + h];
    }
    if constexpr (n >= 1 && n - 1 < last && (n - 1) % 12 < 8) {
      constexpr int i = i0 + (n - 1) / 12, t = (n - 1) % 12 / 4, e = (n - 1) % 4;
      wide[i][t][2 * e] = __uint_as_float(part[i][t][e] << 16);
      wide[i][t][2 * e + 1] = __uint_as_float(part[i][t][e] & 0xffff0000u);
    }
    if constexpr (n < last) {
      constexpr int i = i0 + n / 12, t = n % 12 / 4, e = n % 4;
      uint32_t u;
      asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(u) : "v"(raw[i][e >> 1][2 * (e & 1)]), "v"(raw[i][e >> 1][2 * (e & 1) + 1]));
      part[i][t][e] = u;
      if constexpr (e == 3) *reinterpret_cast<u32x4*>(lds_raw + bo + put_at + NT / 4 * 192 * i + 64 * t) = part[i][t];
      if constexpr (n % 12 == 11) fetch(i, k_next);
    }
  };
  const int fr = lane & 31, fh = lane >> 5;
  auto w_tile = [&](int j) { return GLU ? (BN / 2) * j + 32 * wn : 64 * wn + 32 * j; };
  int wat[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) wat[s] = fr * 192 + (((2 * s + fh) ^ ((fr >> 2) & 3)) << 4);
  u32x4 wf[2][2][3], af[2][MT][3];
  constexpr int READS = 3 * (MT + 2), PRODUCTS = 12 * MT;
  auto read = [&](int bo, int s, int m) {      // fragment m of a step
    const int t = m / (MT + 2), f = m % (MT + 2);
    if (f < 2) wf[s][f & 1][t] = *reinterpret_cast<const u32x4*>(lds_raw + bo + wat[s] + (BM + w_tile(f)) * 192 + 64 * t);
    else af[s][f < 2 ? 0 : f - 2][t] = *reinterpret_cast<const u32x4*>(lds_raw + bo + wat[s] + 32 * (MT * wm + f - 2) * 192 + 64 * t);
  };
  f32x16 acc[2][MT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;
  // The products of step s; behind each a fragment of the next step (of the block at `rbo`) and a share of the split of rows i0 .. i1 - 1
  auto multiply = [&](auto s, int rbo, auto i0, auto i1, int bo, int k_next) {
    constexpr int steps = 12 * (i1 - i0) + 2;
    each<PRODUCTS>([&](auto at) {
      constexpr int of_w[6] = {0, 2, 1, 0, 1, 0}, of_a[6] = {2, 0, 1, 1, 0, 0};
      constexpr int m = at, q = m / (2 * MT), i = m / 2 % MT, j = m % 2, first = m * steps / PRODUCTS, behind = (m + 1) * steps / PRODUCTS;
      acc[j][i] = mma32(wf[s][j][of_w[q]], af[s][i][of_a[q]], acc[j][i], bf16_t{});
      if constexpr (m == 0) __builtin_amdgcn_sched_barrier(0);
      if constexpr (m < READS) read(rbo, 1 - s, m);
      each<behind - first>([&](auto n) { split(i0, i1, std::integral_constant<int, first + n>{}, bo, k_next); });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto meet = [&]() {      // what this wavefront has written is there and what it has asked for has arrived; then everybody's
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // -------- K in blocks of 32, two steps of 16.  Under the products of step 0 of a block the second part of the next block is split and
  // step 1 is read; behind the barrier, under those of step 1, the first part of the block after it, into the buffer just left.
  const int blocks = p.K / 32;
  auto at_k = [&](int t) { return 32 * min(t, blocks - 1); };      // blocks past the end: the last one again, unused
#pragma unroll
  for (int i = 0; i < RP; ++i) fetch(i, 0);
  each<12 * RP + 2>([&](auto n) { split(I0, IP, n, 0, at_k(1)); });
  each<12 * R0 + 2>([&](auto n) { split(I0, IR, n, BUF, at_k(2)); });
  meet();
#pragma unroll
  for (int m = 0; m < READS; ++m) read(0, 0, m);
  int bo = 0;
  for (int t = 0; t < blocks; ++t) {
    multiply(I0, bo, IR, IP, BUF - bo, at_k(t + 2));
    meet();
    multiply(I1, BUF - bo, I0, IR, bo, at_k(t + 3));
    bo = BUF - bo;
  }

  // -------- An infinity, a NaN and a number of 2^88 and more have no such parts and leave a result that is not finite, as a sum of 2^48 and
  // more does: these results, and only these, are formed again from the numbers as they are, so that no result depends on other rows and columns.
  // 3135 rows 1024 -> 4416: 178 us, 233 with an infinity in one row, 695 where no result can be kept; 2048 -> 1024 80, 211, 354.
  constexpr float BACK = 1.0f / (SCALE * SCALE);
  auto odd = [&](int j, int i) {
    float finite = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) finite = fmaf(acc[j][i][r], 0.0f, finite);
    return finite != 0.0f;
  };
  bool any = false;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) any |= odd(j, i);
  if (__builtin_expect(__any(any), 0)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        f32x16 again = acc[j][i];
        if (__any(odd(j, i))) {
          const float *ap = a_row(32 * (MT * wm + i) + fr) + 4 * fh, *wp = w_row(w_tile(j) + fr) + 4 * fh;
#pragma unroll
          for (int r = 0; r < 16; ++r) again[r] = 0.0f;
#pragma unroll 1
          for (int k = 0; k < p.K; k += 8)
            again = mma32(*reinterpret_cast<const u32x4*>(wp + k), *reinterpret_cast<const u32x4*>(ap + k), again, 0.0f);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][i][r] = __builtin_isfinite(acc[j][i][r]) ? acc[j][i][r] * BACK : again[r];
      }
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][i][r] *= BACK;
  }
  wide_results<float, TO, EPI, MT>(p, acc, at.z, mbase + 32 * MT * wm, hi, n0, wn, fr, fh);
}

template <typename TO, int EPI, int MT, int WM, int WN>
hipError_t launch_split_one(const LinArgs& p, int64_t total_rows, int batch, hipStream_t s) {
  constexpr int BM = 32 * MT * WM, BN = 64 * WN, NOUT = EPI == EPI_GLU ? BN / 2 : BN;
  constexpr size_t lds = 2 * (size_t)(BM + BN) * 192;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> devices{0};
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(&linear_split_kernel<TO, EPI, MT, WM, WN>), lds, devices);
    if (e != hipSuccess) return e;
  }
  const int64_t nt = (p.N + NOUT - 1) / NOUT;
  const int64_t mt = p.group_off ? total_rows / BM + batch : (p.M + BM - 1) / BM;      // at most this many row tiles
  const dim3 grid((unsigned)((mt * nt + 7) / 8 * 8), 1, p.group_off ? 1 : batch);
  linear_split_kernel<TO, EPI, MT, WM, WN><<<grid, dim3(64 * WM * WN), lds, s>>>(p, p.group_off ? batch : (int)mt, (int)nt);
  return hipGetLastError();
}

template <typename TO, int EPI>
hipError_t launch_split(const LinArgs& p, int64_t total_rows, int batch, int tile, hipStream_t s) {
  if (tile >= SPLIT_256) return launch_split_one<TO, EPI, 4, 2, 2>(p, total_rows, batch, s);
  if (tile == SPLIT_128) return launch_split_one<TO, EPI, 2, 2, 2>(p, total_rows, batch, s);
  return launch_split_one<TO, EPI, 1, 2, 2>(p, total_rows, batch, s);
}

template <typename TO>
hipError_t launch_split_epi(const LinArgs& p, int epi, int64_t total_rows, int batch, int tile, hipStream_t s) {
  switch (epi) {
    case EPI_NONE: return launch_split<TO, EPI_NONE>(p, total_rows, batch, tile, s);
    case EPI_GLU: return launch_split<TO, EPI_GLU>(p, total_rows, batch, tile, s);
    case EPI_SOFTCAP: return launch_split<TO, EPI_SOFTCAP>(p, total_rows, batch, tile, s);
    case EPI_ACT: return launch_split<TO, EPI_ACT>(p, total_rows, batch, tile, s);
    default: return launch_split<TO, EPI_ROW_GATE>(p, total_rows, batch, tile, s);
  }
}

}  // namespace

hipError_t linear_split_launch(const LinArgs& p, int epilogue, bool out_16bit, int64_t total_rows, int batch, int tile, hipStream_t s) {
  return out_16bit ? launch_split_epi<bf16_t>(p, epilogue, total_rows, batch, tile, s)
                   : launch_split_epi<float>(p, epilogue, total_rows, batch, tile, s);
}
