// Products of many rows: a workgroup per CU walks tiles of 256 x 256 outputs whose K blocks form one stream.
//
// Here: eight wavefronts of 128 x 64 each, for 16-bit products whose results take long to form (linear_four_wavefronts); the others:
// stream_deep.h, whose tiles, their order and W's rows in LDS are those of this file.
//
// What bounds it: the matrix cores (852 us at 8192 x 8192 x 8192, stream_deep.h 705), two wavefronts to a SIMD, of which one forms results
// while the other has products.
//   * 16-row products: a lane's results lie where whole 64-byte pieces of rows can be stored;
//   * the barrier stands before the block's last step of K, whose fragments are in registers: behind it the first fragments of the
//     next block are read under that step's products, and the buffer just left is refilled, one DMA instruction behind every few
//     products;
//   * the order of products, LDS reads and DMA is fixed in the source (sched_barrier); left alone, the compiler puts the reads
//     behind two thirds of the products and waits for them at once;
//   * workgroups stay: the first two blocks of the next tile are on their way while the results of a tile are stored, and nothing
//     waits for those stores but the second block after them.  Their tiles are found once, by a thread each, and kept in LDS.
// LDS rows are 128 bytes, their 16-byte pieces dealt by XOR (through the DMA's source addresses) so that the 16 rows a read touches lie
// in 16 bank groups.  Tiles go to the XCDs in contiguous eighths, within them in bands of eight row
// tiles, so the 32 workgroups of an XCD share 8 row and 4 column panels in its L2.  A group's short last row tile stays in its band
// (at the end of everything, its column panels come from memory again: sixteen experts in bf16 1450 us against 1418).
//
// Job (what is multiplied and what becomes of it) provides:
//   T (stream_deep.h: what is multiplied), Order (how W lies, below; here in rows), NSTORE, K (elements, two blocks of 128 bytes at least)
//   int count(lane)                       how many tiles there are
//   StreamTile find(tile, lane)           which rows and columns the thread's tile has (every thread of a wavefront calls it)
//   const void* a_base(tile); uint32_t a_row(tile, r); uint32_t a_stride()      row r of the tile's A rows (those past the end
//                                         repeat a real one) lies at base + row * stride bytes, its K in 16-byte pieces
//   w_base, w_row, w_stride, w_step()     the same of row r of the W tile in LDS (stream_deep.h: or of its 16-row tile r); bytes to the next K block
//   bool whole(tile)                      NSTORE stores of a wavefront at least are executed for this tile
//   void store<MT>(tile, first row, wn, lane, take)   take(j, i): row 16 i + lane % 16 of the wavefront's, fragment row 4 (lane / 16) + r of product j
// Four wavefronts lie along the columns, two along the rows.
#pragma once
#include "anyt.h"
#include "lds_limit.h"

struct alignas(16) StreamTile {
  int lo, hi;       // first row of the tile; end of the rows it may touch
  int n0, z;        // first column; which product of a batch or which group
};
constexpr int STREAM_LIST = 512;      // tiles of one workgroup at most
constexpr int STREAM_BM = 256, STREAM_BN = 256;
constexpr int STREAM_BUFFER = (STREAM_BM + STREAM_BN) * 128;      // a K block of both

__device__ __forceinline__ f32x4 stream_mma(const u32x4& a, const u32x4& b, f32x4 c) {
  return mfma16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c);
}

// Where W lies in LDS and which of its rows a fragment has.  W stays in the order it has in memory, so that neighbouring lanes of a
// DMA instruction fetch whole lines of it; the fragments choose which results a lane gets (frag and off, in bytes).  In rows: row r is
// 128 bytes, its pieces XORed with key(r); of the 16 rows that a fragment reads no two of the same parity share a key, and row
// frag / 128 + off / 128 has key (fr >> 1) & 7.  In tiles (TILED; nv_gemm's layout): 16 rows by 32 of K are 1 KB, row c's K piece g at
// 16 (16 g + c); tile t lies at place(t), 2 KB apart and a little more, so that the parts of tiles which one fragment reads meet in
// different banks.
struct StreamNatural {      // four consecutive columns to a lane and product: 16 bytes of fp32
  static constexpr bool TILED = false;
  static __device__ __forceinline__ int frag(int fr) { return 128 * fr; }
  static __host__ __device__ constexpr int off(int j) { return 2048 * j; }
  static __device__ __forceinline__ int key(int r) { return (r >> 1) & 7; }
};
struct StreamPaired {       // eight consecutive columns to a lane and pair of products: 16 bytes of 16-bit results
  static constexpr bool TILED = false;
  static __device__ __forceinline__ int frag(int fr) { return 128 * (8 * (fr >> 2) + (fr & 3)); }
  static __host__ __device__ constexpr int off(int j) { return 128 * (32 * (j >> 1) + 4 * (j & 1)); }
  static __device__ __forceinline__ int key(int r) { return ((r >> 1) & 1) | (((r >> 3) & 3) << 1); }
};
struct StreamQuads {        // rows (gate 2 i, gate 2 i + 1, up 2 i, up 2 i + 1): gates in products 0 and 1, ups in 2 and 3, as pairs
  static constexpr bool TILED = false;
  static __device__ __forceinline__ int frag(int fr) { return 128 * (16 * (fr >> 2) + 4 * ((fr >> 1) & 1) + (fr & 1)); }
  static __host__ __device__ constexpr int off(int j) { return 128 * (8 * (j & 1) + 2 * (j >> 1)); }
  static __device__ __forceinline__ int key(int r) { return ((r >> 2) & 1) | (((r >> 4) & 3) << 1); }
};
struct StreamPairedTiled {
  static constexpr bool TILED = true;
  static __host__ __device__ constexpr int place(int t) { return 2112 * t; }
  static __device__ __forceinline__ int frag(int fr) { return place(fr >> 3) + 16 * (8 * ((fr >> 2) & 1) + (fr & 3)); }
  static __host__ __device__ constexpr int off(int j) { return place(2 * (j >> 1)) + 64 * (j & 1); }
};
struct StreamQuadsTiled {
  static constexpr bool TILED = true;
  static __host__ __device__ constexpr int place(int t) { return 2048 * t + 32 * (t & 1) + 128 * ((t >> 1) & 1) + 256 * (t >> 2); }
  static __device__ __forceinline__ int frag(int fr) { return place(fr >> 2) + 16 * (4 * ((fr >> 1) & 1) + (fr & 1)); }
  static __host__ __device__ constexpr int off(int j) { return 128 * (j & 1) + 32 * (j >> 1); }
};

// place `in` of a group of `rows` row tiles by `cols` column tiles: bands of eight row tiles (the last of up to fifteen), rows first
__device__ __forceinline__ void stream_order(int in, int rows, int cols, int& m_tile, int& n_tile) {
  const int bands = max(1, rows >> 3), band = min(in / (8 * cols), bands - 1), first = 8 * band;
  const int wide = band == bands - 1 ? rows - first : 8;
  in -= first * cols;
  m_tile = first + in % wide;
  n_tile = in / wide;
}

// the lane's number, formed where it is used: what depends on it alone is not kept in registers through the loop over blocks
__device__ __forceinline__ int stream_lane() {
  uint32_t all = ~0u;
  asm volatile("" : "+s"(all));
  return (int)__builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
}

template <typename Job>
__global__ __launch_bounds__(512, 2) void stream_tiles_kernel(Job job) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int WN = 4, WM = 8 / WN, MT = STREAM_BM / 16 / WM, NT = STREAM_BN / 16 / WN;
  typedef typename Job::Order Order;
  constexpr int BM = STREAM_BM, BN = STREAM_BN, BO = STREAM_BUFFER;     // BO: bytes of one buffer
  constexpr int AG = BM / 64, WG = BN / 64, D = AG + WG;                // DMA instructions (8 rows each) of a wavefront per block
  constexpr int P = MT * NT, R = MT + NT;                               // products and fragment reads of a step
  typedef __attribute__((address_space(1))) void global_void;
  typedef __attribute__((address_space(3))) void lds_void;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const int lane = stream_lane(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wv / WN, wn = wv % WN;                                 // a SIMD has one wavefront of each half of the rows

  // -------- this workgroup's tiles: every per-th of its XCD's.  A last round that at most half of the workgroups would have is dealt
  // as tiles of half the rows.  One thread finds one tile; the list is in LDS.
  StreamTile* const list = reinterpret_cast<StreamTile*>(lds_raw + 2 * BO);
  int tiles;
  {
    const int per = gridDim.x >> 3, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int64_t all = job.count(lane);
    const int first = (int)(all * xcd >> 3), mine_all = (int)(all * (xcd + 1) >> 3) - first, over = mine_all % per;
    const int halves = 2 * over <= per ? 2 * over : 0, rounds = halves ? mine_all - over : mine_all, end = rounds + halves;
    tiles = slot < end ? (end - slot + per - 1) / per : 0;
    if (tiles == 0) return;
    const int t = min(slot + (int)threadIdx.x * per, end - 1), h = t - rounds;
    StreamTile mine = job.find(first + (h < 0 ? t : rounds + (h >> 1)), lane);
    if (h >= 0) {
      mine.lo += (h & 1) * (BM / 2);
      mine.hi = min(mine.hi, mine.lo + BM / 2);      // the second half of a short tile has no rows
    }
    list[threadIdx.x] = mine;
    __syncthreads();
  }
  auto listed = [&](int n) {
    const StreamTile at = list[n];
    return StreamTile{__builtin_amdgcn_readfirstlane(at.lo), __builtin_amdgcn_readfirstlane(at.hi),
                      __builtin_amdgcn_readfirstlane(at.n0), __builtin_amdgcn_readfirstlane(at.z)};
  };

  // -------- the stream of blocks
  const uint32_t a_stride = job.a_stride(), w_stride = job.w_stride(), w_step = job.w_step();
  uint32_t arow[AG], wrow[WG];
  uint64_t apos, wpos;            // where the next K block begins, less what depends on the lane
  auto point = [&](const StreamTile& at) {
    const int r0 = 8 * wv + (stream_lane() >> 3);
#pragma unroll
    for (int i = 0; i < AG; ++i) arow[i] = job.a_row(at, r0 + 64 * i);
#pragma unroll
    for (int i = 0; i < AG; ++i) asm volatile("" : "+v"(arow[i]));      // a gathered row's number is waited for here, not at each fetch
#pragma unroll
    for (int i = 0; i < WG; ++i) wrow[i] = job.w_row(at, r0 + 64 * i);
    apos = reinterpret_cast<uint64_t>(job.a_base(at));
    wpos = reinterpret_cast<uint64_t>(job.w_base(at));
  };
  // DMA instruction i fills LDS rows 8 (wv + 8 i) + l / 8, whose place among the XORs is the same for every i
  uint32_t alane, wlane;
  auto lanes = [&]() {
    const int l = stream_lane(), r0 = 8 * wv + (l >> 3);
    alane = 16 * ((l & 7) ^ ((r0 >> 1) & 7));
    wlane = 16 * ((l & 7) ^ Order::key(r0));
  };
  auto fill = [&](int bo, int i) {
    if (i < AG) {
      const int q = i < AG ? i : 0;
      __builtin_amdgcn_global_load_lds((global_void*)(apos + (uint64_t)arow[q] * a_stride + alane), (lds_void*)(lds_raw + bo + (wv + 8 * q) * 1024),
                                       16, 0, 0);
    } else {
      const int q = i < AG ? 0 : i - AG;
      __builtin_amdgcn_global_load_lds((global_void*)(wpos + (uint64_t)wrow[q] * w_stride + wlane),
                                       (lds_void*)(lds_raw + bo + (BM + 8 * (wv + 8 * q)) * 128), 16, 0, 0);
    }
    if (i == AG - 1) apos += 128;
    if (i == D - 1) wpos += w_step;
  };
  // where this lane's first fragments of W and A lie in the buffer at `bo`; formed for every step anew (registers).  Every fragment
  // starts at a multiple of 16 rows.
  auto fragments = [&](int bo, int step, int& wat, int& aat) {
    const int l = stream_lane(), fr = l & 15, in = bo + 16 * (((4 * step + (l >> 4)) ^ (fr >> 1)) & 7);
    wat = in + (BM + 16 * NT * wn) * 128 + Order::frag(fr);
    aat = in + (16 * MT * wm + fr) * 128;
  };
  u32x4 wf[2][NT], af[2][MT];
  auto read = [&](int wat, int aat, int r, int set) {
    if (r < NT) wf[set][r < NT ? r : 0] = *reinterpret_cast<const u32x4*>(lds_raw + wat + Order::off(r < NT ? r : 0));
    else af[set][r < NT ? 0 : r - NT] = *reinterpret_cast<const u32x4*>(lds_raw + aat + 2048 * (r - NT));
  };

  f32x4 acc[NT][MT];
  auto clear = [&]() {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();

  const int blocks = job.K / 64;
  StreamTile at = listed(0), ahead = at;
  point(at);
  lanes();
#pragma unroll
  for (int i = 0; i < D; ++i) fill(0, i);
#pragma unroll
  for (int i = 0; i < D; ++i) fill(BO, i);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int wat, aat;
  fragments(0, 0, wat, aat);
#pragma unroll
  for (int r = 0; r < R; ++r) read(wat, aat, r, 0);
  int fetched = 2, left = blocks, tile = 0, next = 0, bo = 0;
  bool stored = false, live = at.lo + 16 * MT * wm < at.hi;

  for (;;) {
    if (fetched == blocks) {        // the stream goes on with the next tile; behind the last one with that one again, unused
      fetched = 0;
      if (next + 1 < tiles) ahead = listed(++next);
      point(ahead);
    }
    if (live) {
      fragments(bo, 1, wat, aat);
#pragma unroll
      for (int m = 0; m < P; ++m) {
        acc[m % NT][m / NT] = stream_mma(wf[0][m % NT], af[0][m / NT], acc[m % NT][m / NT]);
        if (m == 0) __builtin_amdgcn_sched_barrier(0);       // or the first product waits for the first of these reads
        if (m < R) read(wat, aat, m, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {       // the second set holds nothing then: said so, or its registers stay taken around the loop
#pragma unroll
      for (int j = 0; j < NT; ++j) asm volatile("" : "=v"(wf[1][j]));
#pragma unroll
      for (int i = 0; i < MT; ++i) asm volatile("" : "=v"(af[1][i]));
    }
    // this wavefront's part of the next block has arrived and it has read the last of this one; then everybody has.  Behind a
    // whole tile's stores only what came before them is waited for: loads and stores are counted in the order of their issue.
    if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(Job::NSTORE) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fragments(BO - bo, 0, wat, aat);
    lanes();
    if (live) {
      constexpr int EVERY = P / D;
#pragma unroll
      for (int m = 0; m < P; ++m) {
        acc[m % NT][m / NT] = stream_mma(wf[1][m % NT], af[1][m / NT], acc[m % NT][m / NT]);
        if (m == 0) __builtin_amdgcn_sched_barrier(0);       // or the first product waits for the first of these reads
        if (m < R) read(wat, aat, m, 0);
        if (m % EVERY == 0 && m / EVERY < D) fill(bo, m / EVERY);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) read(wat, aat, r, 0);
#pragma unroll
      for (int i = 0; i < D; ++i) fill(bo, i);
    }
    ++fetched;
    bo = BO - bo;
    stored = false;
    if (--left > 0) continue;

    left = blocks;
    if (live) {
      job.template store<MT>(at, at.lo + 16 * MT * wm, wn, stream_lane(), [&](int j, int i) { return acc[j][i]; });
      stored = job.whole(at);
      clear();
    }
    if (++tile == tiles) break;
    fragments(bo, 0, wat, aat);
#pragma unroll
    for (int r = 0; r < R; ++r) read(wat, aat, r, 0);       // again: their registers were the epilogue's
    at = ahead;       // with at least two blocks to a tile the stream is there already
    live = at.lo + 16 * MT * wm < at.hi;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");     // no DMA outlives the workgroup's LDS
#endif
}

template <typename Job>
hipError_t launch_stream_tiles(const Job& job, int64_t max_tiles, hipStream_t s) {
  constexpr size_t lds = 2 * STREAM_BUFFER + STREAM_LIST * sizeof(StreamTile);
  static std::atomic<uint64_t> devices{0};
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(&stream_tiles_kernel<Job>), lds, devices);
  if (e != hipSuccess) return e;
  // with few tiles there is a workgroup for each half of one
  const unsigned grid = (unsigned)(max_tiles < 128 ? (2 * max_tiles + 7) / 8 * 8 : 256);
  stream_tiles_kernel<Job><<<dim3(grid), dim3(512), lds, s>>>(job);
  return hipGetLastError();
}
