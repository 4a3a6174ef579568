// Products of many rows in 16 bits: tiles of 256 x 256 outputs by four wavefronts of 128 x 128 each, their K blocks one stream (the tiles
// and their order are those of stream_tiles.h, which keeps the products whose results take long to form).
//
// What bounds it: the matrix cores and their power.  The eight wavefronts of 128 x 64 that this form replaced read 192 KB of LDS per K
// block of 64 for 128 KB here, asked for a block about half a block's products before it was waited for, and took 852 us at 8192 x 8192
// x 8192; this one takes 710 (1550 TFLOP/s; the vendor library 685).  What it rests on:
//   * a wavefront has a SIMD to itself: 256 accumulation registers hold its results, 128 vector registers the fragments of a whole K block;
//   * a K block is multiplied in quarters (64 rows by 64 columns of a wavefront), so a quarter of a block is all that lies between the last
//     read of a piece of LDS and its refill: with two barriers to a block, what is fetched has two and a half blocks' halves to arrive in
//     (2816 cycles of products; the form before had 1000 - 2000).  The order of products, LDS reads and DMA is fixed in the source;
//   * DMA a few at a time: eight products between two instructions; eight of them two apart queue up (8192^3: 756 against 730 us);
//   * no branch between products in the loop for whole tiles (8192^3: 756 with one per half block, 710 without), and no vector address that
//     moves with K: the tile's rows are offsets, K is in the scalar base.  A tile's first pair of blocks, whose products are
//     added to nothing (256 registers less to clear) while stores are still on their way, the last pair of an odd number of blocks, and tiles
//     with wavefronts that have no rows take the other loop (8192 rows 3008 -> 6144, 47 blocks: 205 us, all of them there 257);
//   * a wavefront has rows 64 of each half of the tile, so a half of 128 rows, or a ragged tile, is half the work for each of them, in a
//     loop of its own: half of W's columns to a barrier, products above all reads and DMA (3000 rows 2048 -> 2048, 192 halves: 0.67 of the
//     time in the loop with branches, where they were 1.07 of eight wavefronts' time; 8192 -> 2048 0.59 and 1.15).
// The sums are those of stream_tiles.h, bit for bit: K in the same order.  Measured, eight wavefronts and these (us): the experts' layer of 16384
// rows, 2048 -> 2 x 3072 -> 2048, 1401 and 1143; 16384 rows 2048 -> 2 x 6144 with SiLU 734 and 607; 2048 -> 6144 into fp32 349 and 329; 14600 rows
// 1024 -> 4096 114 and 105; gate/up of 1024 -> 2 x 3072 193 and 170, q/k/v with rotation 157 and 142.
// Job: as for stream_tiles.h, and
//   bool FAR_A, FAR_W                     whether a tile's rows of A (W) may lie 4 GiB and more from its base
//   bool UPS, w_ups()                     whether W's rows 32 - 63 of every 64 lie another w_ups() bytes on (which may be 4 GiB and more)
//   NSTORE_WAVE                           stores of a wavefront of a whole tile, at least
//   EXTRA, fetch_extra(tile, wv, lane, lds)   bytes of LDS a tile's results need of memory (3 KB fit), and the DMA for them, a tile ahead
//   finish(tile, wm, wn, lane, live0, live1, lds)   the results: rows 128 h + 64 wm .. of the tile, h = 0 and 1 as far as live, by rows 128 wn ..
//                                         of W's tile; deep_take(h, j, i) has row 16 i + lane % 16, fragment row 4 (lane / 16) + r of product j of eight
#pragma once
#include "stream_tiles.h"

// The accumulators: all 256 accumulation registers, by number.  Four from 4 (32 h + 4 j + i) on hold the product of W fragment j (of eight)
// and A fragment i (of four) of half h of the rows.  The compiler, told of them as variables, copies them about (and does not know of the
// wait states between these instructions and its own); it is only told, at each barrier, that they are not its to use.
#define DEEP_REGISTERS \
      "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
      "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
      "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
      "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", \
      "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
      "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", \
      "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
      "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", \
      "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
      "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
      "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
      "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", \
      "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", \
      "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", \
      "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", \
      "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
__device__ __forceinline__ constexpr int deep_at(int h, int j, int i) { return 4 * (32 * h + 4 * j + i); }
template <bool NEW = false>      // NEW: the accumulators' first product, added to nothing
__device__ __forceinline__ void deep_mma(int at, const u32x4& w, const u32x4& a, bf16_t) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (NEW) asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, 0" ::"v"(w), "v"(a), "i"(at), "i"(at + 3));
  else asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(w), "v"(a), "i"(at), "i"(at + 3));
#endif
}
template <bool NEW = false>      // NEW: the accumulators' first product, added to nothing
__device__ __forceinline__ void deep_mma(int at, const u32x4& w, const u32x4& a, f16_t) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (NEW) asm volatile("v_mfma_f32_16x16x32_f16 a[%2:%3], %0, %1, 0" ::"v"(w), "v"(a), "i"(at), "i"(at + 3));
  else asm volatile("v_mfma_f32_16x16x32_f16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(w), "v"(a), "i"(at), "i"(at + 3));
#endif
}
__device__ __forceinline__ f32x4 deep_take(int h, int j, int i) {
  float a = 0.f, b = 0.f, c = 0.f, d = 0.f;
#if defined(__HIP_DEVICE_COMPILE__)
  const int at = deep_at(h, j, i);
  asm volatile("v_accvgpr_read_b32 %0, a[%4]\n\tv_accvgpr_read_b32 %1, a[%5]\n\tv_accvgpr_read_b32 %2, a[%6]\n\tv_accvgpr_read_b32 %3, a[%7]"
               : "=v"(a), "=v"(b), "=v"(c), "=v"(d)
               : "i"(at), "i"(at + 1), "i"(at + 2), "i"(at + 3));
#endif
  return f32x4{a, b, c, d};
}

constexpr int DEEP_PA = 128 * 128, DEEP_PW = 128 * 128 + 1024;      // one half of the rows of A or W, one K block
constexpr int DEEP_BUFFER = 2 * (DEEP_PA + DEEP_PW);
template <typename Job>
__global__ __launch_bounds__(256, 1) void stream_deep_kernel(Job job) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef typename Job::T T;
  typedef typename Job::Order Order;
  constexpr int BM = STREAM_BM;
  typedef __attribute__((address_space(1))) void global_void;
  typedef __attribute__((address_space(3))) void lds_void;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv >> 1, wn = wv & 1, fr = lane & 15, g = lane >> 4;

  StreamTile* const list = reinterpret_cast<StreamTile*>(lds_raw + 2 * DEEP_BUFFER);
  int tiles;
  {
    const int per = gridDim.x >> 3, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int64_t all = job.count(lane);
    const int first = (int)(all * xcd >> 3), mine_all = (int)(all * (xcd + 1) >> 3) - first, over = mine_all % per;
    const int halves = 2 * over <= per ? 2 * over : 0, rounds = halves ? mine_all - over : mine_all, end = rounds + halves;
    tiles = slot < end ? (end - slot + per - 1) / per : 0;
    if (tiles == 0) return;
    for (int base = 0; base < tiles; base += 256) {
      const int n = base + (int)threadIdx.x, t = min(slot + n * per, end - 1), h = t - rounds;
      StreamTile mine = job.find(first + (h < 0 ? t : rounds + (h >> 1)), lane);
      if (h >= 0) {
        mine.lo += (h & 1) * (BM / 2);
        mine.hi = min(mine.hi, mine.lo + BM / 2);
      }
      if (n < STREAM_LIST) list[n] = mine;
    }
    __syncthreads();
  }
  auto listed = [&](int n) {
    const StreamTile at = list[n];
    return StreamTile{__builtin_amdgcn_readfirstlane(at.lo), __builtin_amdgcn_readfirstlane(at.hi),
                      __builtin_amdgcn_readfirstlane(at.n0), __builtin_amdgcn_readfirstlane(at.z)};
  };

  const uint32_t a_stride = job.a_stride(), w_stride = job.w_stride(), w_step = job.w_step();
  // Where this lane's pieces lie, in bytes from the tile's bases; and the bases, at the K block that is fetched next.  (Addresses that move
  // with K would be 32 registers, moved about wherever the ways through the loop below meet.)
  std::conditional_t<Job::FAR_A, uint64_t, uint32_t> ap[2][4];
  std::conditional_t<Job::FAR_W, uint64_t, uint32_t> wp[2][4];
  uint64_t abase, wbase, ubase = 0;
  auto point = [&](const StreamTile& at) {
    const int l = lane, r8 = 8 * wv + (l >> 3);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ap[h][q] = (uint64_t)job.a_row(at, 128 * h + r8 + 32 * q) * a_stride + 16 * ((l & 7) ^ ((r8 >> 1) & 7));
        if constexpr (Order::TILED) {
          const int t = (wv >> 1) + 2 * q;
          wp[h][q] = (uint64_t)job.w_row(at, 8 * (t >> 2) + 4 * h + (t & 3)) * w_stride + 1024 * (wv & 1) + 16 * l;
        } else {
          const int r = r8 + 32 * q;
          wp[h][q] = (uint64_t)job.w_row(at, 128 * (r >> 6) + 64 * h + (r & 63)) * w_stride + 16 * ((l & 7) ^ Order::key(r));
        }
      }
    abase = reinterpret_cast<uint64_t>(job.a_base(at));
    wbase = reinterpret_cast<uint64_t>(job.w_base(at));
    if constexpr (Job::UPS) ubase = wbase + job.w_ups();
  };
  auto fill_a = [&](int bo, int h, int q) {
    __builtin_amdgcn_global_load_lds((global_void*)(abase + ap[h][q]), (lds_void*)(lds_raw + bo + h * DEEP_PA + (wv + 4 * q) * 1024), 16, 0, 0);
  };
  auto fill_w = [&](int bo, int h, int q) {
    int place;
    if constexpr (Order::TILED) place = Order::place((wv >> 1) + 2 * q) + 1024 * (wv & 1);
    else place = (wv + 4 * q) * 1024;
    const uint64_t base = Job::UPS && (q & 1) ? ubase : wbase;
    __builtin_amdgcn_global_load_lds((global_void*)(base + wp[h][q]), (lds_void*)(lds_raw + bo + 2 * DEEP_PA + h * DEEP_PW + place), 16, 0, 0);
  };
  auto next_block = [&]() {
    abase += 128;
    wbase += w_step;
    ubase += w_step;
  };
  u32x4 fa[2][4][2], fw[2][4][2];
  int aat[2], wat[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int in = 16 * (((4 * s + g) ^ (fr >> 1)) & 7);
    aat[s] = in + (64 * wm + fr) * 128;
    if constexpr (Order::TILED) wat[s] = Order::place(4 * wn) + Order::frag(fr) + 1024 * s + 256 * g;
    else wat[s] = in + 64 * wn * 128 + Order::frag(fr);
  }
  auto read_a = [&](int bo, int h, int r, int set) {      // r: which of the eight
    const int s = r >> 2, i = r & 3;
    fa[set][i][s] = *reinterpret_cast<const u32x4*>(lds_raw + bo + h * DEEP_PA + aat[s] + 2048 * i);
  };
  auto read_w = [&](int bo, int h, int r) {
    const int s = r >> 2, j = r & 3;
    fw[h][j][s] = *reinterpret_cast<const u32x4*>(lds_raw + bo + 2 * DEEP_PA + h * DEEP_PW + wat[s] + Order::off(j));
  };
  // What tile n's results need lies in one of four places.  Where a tile has one pair of blocks, no barrier stands between a wavefront's finish
  // of tile n - 1 and another's DMA for n + 1, so three are in use at once.
  auto extra = [&](int n) { return lds_raw + 2 * DEEP_BUFFER + STREAM_LIST * sizeof(StreamTile) + (n & 3) * Job::EXTRA; };
  const int blocks = job.K / 64, pairs = (blocks + 1) / 2;
  const bool odd = blocks & 1;
  StreamTile at = listed(0);
  point(at);
  job.fetch_extra(at, wv, lane, extra(0));
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int q = 0; q < 4; ++q) fill_a(b * DEEP_BUFFER, 0, q);
#pragma unroll
    for (int q = 0; q < 4; ++q) fill_w(b * DEEP_BUFFER, b, q);
#pragma unroll
    for (int q = 0; q < 4; ++q) fill_w(b * DEEP_BUFFER, 1 - b, q);
#pragma unroll
    for (int q = 0; q < 4; ++q) fill_a(b * DEEP_BUFFER, 1, q);
    next_block();
  }
  asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // Half a block: the products of half of A's rows with all of W's.  Their first fragments are in registers; under them the next ones are
  // read and the pieces of LDS that were read before the barrier are filled again, in this order.  What is waited for was asked for
  // three halves before: sixteen operations are younger, and a tile's stores where they came between (`behind`).
  constexpr int BEHIND = 16 + Job::NSTORE_WAVE < 63 ? 16 + Job::NSTORE_WAVE : 63;
  auto arrive = [&](bool behind) {
    if (behind) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND) : "memory");
    else asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory", DEEP_REGISTERS);
  };
  auto refill = [&](auto bb, auto ss, int k) {
    constexpr int B = decltype(bb)::value, S = decltype(ss)::value, here = B * DEEP_BUFFER;
    if constexpr (S == 0) {
      if (k < 4) fill_a(here, 0, k);
      else fill_w(here, B, k - 4);
    } else {
      if (k < 4) fill_w(here, 1 - B, k);
      else fill_a(here, 1, k - 4);
    }
  };
  auto half = [&](auto plain, auto bb, auto ss, bool live, bool fresh, bool behind) {
    constexpr bool PLAIN = decltype(plain)::value;
    constexpr int B = decltype(bb)::value, S = decltype(ss)::value, X = B, Y = 1 - B;
    constexpr int here = B * DEEP_BUFFER, there = (1 - B) * DEEP_BUFFER;
    arrive(!PLAIN && behind);
    auto reads = [&](int m) {
      if constexpr (S == 0) {
        if (m < 8) read_w(here, Y, m);
        else if (m < 16) read_a(here, 1, m - 8, 1);
      } else {
        if (m < 8) read_a(there, 0, m, 0);
        else if (m >= 32 && m < 40) read_w(there, Y, m - 32);
      }
    };
    auto fills = [&](int k) { refill(bb, ss, k); };
    auto product = [&](int m, auto is_new) {
      const int hw = (m < 32) == (S == 0) ? X : Y, s = (m >> 4) & 1, j = (m >> 2) & 3, i = m & 3;
      deep_mma<decltype(is_new)::value>(deep_at(S, 4 * hw + j, i), fw[hw][j][s], fa[S][i][s], T{});
    };
    if constexpr (PLAIN) {
#pragma unroll
      for (int m = 0; m < 64; ++m) {
        product(m, std::false_type{});
        __builtin_amdgcn_sched_barrier(0);
        reads(m);
        if (m % 8 == 3) fills(m / 8);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {      // what is not for all wavefronts has no results but in the accumulators: nothing to be merged behind it
      auto quarter = [&](int from) {
        if (!live) return;
        if (B == 0 && fresh) {
#pragma unroll
          for (int m = 0; m < 16; ++m) product(from + m, std::true_type{});
        } else {
#pragma unroll
          for (int m = 0; m < 16; ++m) product(from + m, std::false_type{});
        }
#pragma unroll
        for (int m = 16; m < 32; ++m) product(from + m, std::false_type{});
      };
#pragma unroll
      for (int m = 0; m < 32; ++m) reads(m);
#pragma unroll
      for (int k = 0; k < 8; ++k) fills(k);
      quarter(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 32; m < 64; ++m) reads(m);
      quarter(32);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // The same for a wavefront that has rows in the tile's first half alone: half of W's columns in each half, so that reads and refills have
  // products above them; A's fragments in either set by turns, W's behind the last of their products.
  auto narrow = [&](auto bb, auto ss) {
    constexpr int B = decltype(bb)::value, S = decltype(ss)::value, Y = 1 - B, hw = S == 0 ? B : Y;
    constexpr int here = B * DEEP_BUFFER, there = (1 - B) * DEEP_BUFFER;
    arrive(false);
#pragma unroll
    for (int m = 0; m < 32; ++m) {
      const int s = m >> 4, j = (m >> 2) & 3, i = m & 3;
      deep_mma(deep_at(0, 4 * hw + j, i), fw[hw][j][s], fa[B][i][s], T{});
      __builtin_amdgcn_sched_barrier(0);
      if (S == 0 && m < 8) read_w(here, Y, m);
      if (S == 1 && m < 8) read_a(there, 0, m, 1 - B);
      if (S == 1 && i == 3) read_w(there, Y, m >> 2);      // in place of the fragment that has been multiplied
      if (m % 4 == 1) refill(bb, ss, m / 4);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const std::integral_constant<int, 0> I0;
  const std::integral_constant<int, 1> I1;
  int left = pairs, tile = 0;
  bool stored = false, live0 = at.lo + 64 * wm < at.hi, live1 = at.lo + 128 + 64 * wm < at.hi;
  auto first = [&]() {
#pragma unroll
    for (int r = 0; r < 8; ++r) read_a(0, 0, r, 0);
#pragma unroll
    for (int r = 0; r < 8; ++r) read_w(0, 0, r);
  };
  auto ask_ahead = [&]() {      // with a tile's last pair the next one's first is fetched; behind the last tile that one's again, unused
    if (left > 1) return;
    const StreamTile ahead = listed(min(tile + 1, tiles - 1));
    point(ahead);
    job.fetch_extra(ahead, wv, lane, extra(tile + 1));
  };
  for (;;) {
    // Each way reads its first fragments itself: handed from one to the other they would be moved between registers.
    if (live0 && live1 && left < pairs && left > odd) {
      const std::true_type plain;
      first();
      for (; left > odd; --left) {
        ask_ahead();
        half(plain, I0, I0, true, false, false);
        half(plain, I0, I1, true, false, false);
        if (!(odd && left == 2)) next_block();
        half(plain, I1, I0, true, false, false);
        half(plain, I1, I1, true, false, false);
        next_block();
      }
    } else if (live0 && !live1 && left < pairs && left > odd) {
      asm volatile("; half" ::: "memory");
      first();
      for (; left > odd; --left) {
        ask_ahead();
        narrow(I0, I0);
        narrow(I0, I1);
        if (!(odd && left == 2)) next_block();
        narrow(I1, I0);
        narrow(I1, I1);
        next_block();
      }
    } else {
      const std::false_type plain;
      asm volatile("; not all" ::: "memory");      // or the reads of all ways become one, ahead of them
      first();
      ask_ahead();
      half(plain, I0, I0, live0, left == pairs, stored);
      half(plain, I0, I1, live1, left == pairs, stored);
      if (!(odd && left == 2)) next_block();      // the last pair has no second block: the first one again, unused
      const bool full = !odd || left > 1;
      half(plain, I1, I0, live0 && full, false, stored);
      half(plain, I1, I1, live1 && full, false, false);
      next_block();
      stored = false;
      --left;
    }
    if (left > 0) continue;
    left = pairs;
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory", DEEP_REGISTERS);      // the last products are through the matrix cores
    job.finish(at, wm, wn, stream_lane(), live0, live1, extra(tile));
    stored = job.whole(at);
    if (++tile == tiles) break;
    at = listed(tile);
    live0 = at.lo + 64 * wm < at.hi;
    live1 = at.lo + 128 + 64 * wm < at.hi;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#endif
}

template <typename Job>
hipError_t launch_stream_deep(const Job& job, int64_t max_tiles, hipStream_t s) {
  constexpr size_t lds = 2 * DEEP_BUFFER + STREAM_LIST * sizeof(StreamTile) + 4 * Job::EXTRA;
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static std::atomic<uint64_t> devices{0};
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(&stream_deep_kernel<Job>), lds, devices);
  if (e != hipSuccess) return e;
  const unsigned grid = (unsigned)(max_tiles < 128 ? (2 * max_tiles + 7) / 8 * 8 : 256);
  stream_deep_kernel<Job><<<dim3(grid), dim3(256), lds, s>>>(job);
  return hipGetLastError();
}
