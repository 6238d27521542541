// Triangle contraction on bf16 MFMA:  T[c][i][j] = sum_k A[c][i][k] * B[c][j][k]
// for a batch of channels c, bf16 in and out, fp32 accumulation.  The same
// kernel, with a per-column or SwiGLU epilogue, takes the large dense
// projections (x W^T with thousands of rows and columns) of the diffusion
// transformer and the outer-product mean.
//
// Both operands are k-contiguous (the natural fragment order of
// v_mfma_f32_32x32x16_bf16).  The tile is as large as the register file
// allows: one workgroup of four waves per CU, a 256x256 block, each wave a
// 128x128 quadrant = 4x4 MFMA tiles = 256 fp32 accumulators (the unified
// 512-entry register file of a lone wave per SIMD), half a 16-byte fragment
// read per MFMA and 128 FLOPs per byte fetched from L2.
//
// What paces the kernel is the CU's vector memory path: it takes in about one cache line every two
// cycles, whole or in part, and a wave that issues a load into a full queue stalls with its MFMAs behind it.
// A lone wave per SIMD has nobody to cover for it.  So:
//   * slabs are 64 k deep, a slab row is one whole 128-byte line: 115 bytes/ns into a CU where 64-byte
//     pieces bring 62 (32-deep slabs, in four buffers).  Two buffers of 64 KB are what LDS holds;
//   * slabs go from global memory straight into LDS (buffer_load_dwordx4 .. lds: no staging
//     registers, no LDS stores in the instruction stream), range-checked, so that a ragged K end
//     arrives as zeros and needs no other code;
//   * the loads are dealt between the fragment reads of two of a slab's four k-steps, which keeps
//     the memory path evenly busy instead of saturated in bursts;
//   * the one barrier per slab sits in front of its last k-step, after the wave has
//     read all its fragments of the slab: the MFMAs of that k-step cover
//     the barrier and the first fragment reads of the next slab, and the
//     buffer is free for refill the moment the barrier is passed;
//   * the workgroups are persistent, one per CU, and the slab pipeline never drains: the
//     loads that run ahead of a tile's last slabs fetch the first slabs of the
//     workgroup's next tile, the epilogue stages through an LDS area of its own and does
//     not wait for its stores, so a tile's first slab is in LDS when the previous tile's
//     last store has been issued.
// A load puts lane l's 16 bytes at LDS base + 16 l, so rows cannot be padded;
// instead the eight 16-byte chunks of a row are permuted, chunk c of row
// r living at position c ^ ((r >> 1) & 7), which makes the fragment reads (32
// rows x one chunk per half-wave) conflict-free over the 64 banks.  The
// permutation is applied on the global side, where a lane is free to fetch
// any chunk.
//
// 32-deep -> 64-deep slabs, us: contraction of 128 channels at N = 187 9.9 -> 8.9, 300 25.4 -> 22.0, 387 40.3 -> 35.5,
// 500 46.2 -> 44.0, 1536 881 -> 860; 4096 x 24576 x 1024 regrouped 224 -> 206; 3840 x 3072 x 768 with column epilogue
// 29.1 -> 26.0, with SwiGLU 23.6 -> 20.2; 8192^3 852 -> 805 (1366 TFLOP/s).  At N = 768 (140 both) memory decides: 450 MB
// pass in and out.  In large products the matrix cores are busy 77 % of the time and power sets the clock (1.66 GHz).
//
// The accumulators hold T^T tiles (B fragments as the MFMA's A operand), so a
// lane owns one output row i and four consecutive columns j per register quad:
// the epilogue packs those to 8 bytes, stages 32 rows x 64 columns at a time per wave
// through LDS and writes 128-byte row segments.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace {

// The block is 64 IT x 256: IT = 4 MFMA tiles per wave along i (256 x 256), or IT = 3 (192 x 256) where
// that saves enough rounds of workgroups (N = 384: tiles of 256 would be half empty).
constexpr int CN = 256, CK = 64;
constexpr int ROWB = CK * 2;            // bytes of a slab row in LDS (unpadded): one cache line
constexpr uint32_t SLAB = (256 + CN) * ROWB;  // 64 KB at IT = 4: A rows first, then B rows
constexpr int LDE = 64 + 8;             // LDS row stride of a wave's output staging area (bf16)
constexpr int EPI_BYTES = 32 * LDE * 2;  // 32 rows x 64 columns per wave at a time
constexpr int RSRC_RAW = 0x00020000;     // last word of a raw (unstructured, range-checked) buffer descriptor

// 64 lanes x 16 bytes from a range-checked buffer (descriptor, wave-uniform byte offset, per-lane byte offset) to
// the KB of LDS at the wave-uniform address lds + BYTES.  An offset past the descriptor's size writes zeros.  Issued
// as inline assembly on purpose:
// the compiler keeps a scoreboard of the loads into LDS that it can see and, where paths with
// different waits meet, makes a later fragment read wait for ALL of them (vmcnt(0)), the ones
// issued a moment ago for slabs far ahead included.  Here every buffer is read only after an
// explicit wait and barrier that follow the load's issue.
template <int BYTES>
__device__ __forceinline__ void load_to_lds(const u32x4 rsrc, uint32_t soff, uint32_t off, uint32_t lds) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(off), "s"(rsrc),
               "s"(soff), "n"(BYTES)
               : "m0", "scc");
}
__device__ __forceinline__ u32x4 buffer_of(const void* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return u32x4{lo, hi & 0xffffu, 0x7fffffffu, RSRC_RAW};
}

template <int N>
using I = std::integral_constant<int, N>;
// f(I<0>{}), .., f(I<N - 1>{})
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (N > 0) {
    each<N - 1>(f);
    f(I<N - 1>{});
  }
}

// a pointer the compiler cannot prove wave-uniform, moved to scalar registers
template <typename T>
__device__ __forceinline__ T* uniform_ptr(T* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<T*>(((uint64_t)hi << 32) | lo);
}

// One accumulator value, read where the source says: left to itself the register allocator,
// faced with an epilogue of many basic blocks, copies most of the 256 accumulators out of their
// accumulation registers up front, which costs as many vector registers (and spills).
__device__ __forceinline__ float acc_read(float a) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}

// s_waitcnt vmcnt(N) lgkmcnt(0): all but the N youngest vector memory operations done, and every LDS read: behind a
// barrier that follows, the buffers that the waves have read are free.  (vmcnt in bits 0-3 and 14-15, expcnt in bits 4-6,
// all ones for no wait, lgkmcnt in bits 8-11.)
template <int N>
__device__ __forceinline__ void wait_loads_but() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70);
}

// MODE 0: plain bf16 product (the triangle contraction).
// MODE 1: per-column epilogue of the dense projections, (acc + bias) * alpha
//         and / or a sigmoid, uniform over the tile or chosen per segment of
//         seg_len columns, and optionally the 32x32-regrouped output order.
// MODE 2: SwiGLU, weight rows packed in blocks of 64 (32 "a" rows, then the 32
//         matching "b" rows): output column 32 p + x = silu(a) * b of block p.
// MODE 3: outer-product mean. Rows and columns are (token, 32 channels); the tile, 8 x 8 token pairs' outer
//         products, never leaves the workgroup: it goes to LDS in bf16, [pair][1024], and is multiplied there with
//         the output weights [128][1024] (outer_tile).
enum { BIG_PLAIN = 0, BIG_COLUMN_OPS = 1, BIG_SWIGLU = 2, BIG_OUTER_MEAN = 3 };

template <int MODE, int IT = 4>
__global__ __launch_bounds__(256, 1) void contract_kernel(GemmArgs g) {
  args_at_once<GemmArgs>();
  constexpr int CM = 64 * IT, WM = 32 * IT;  // block and wave extent along i
  constexpr int SLAB_A = CM * ROWB;
  constexpr int LA = 2 * IT, NLOAD = LA + 8;  // loads per wave and slab, of which A
  constexpr int NSTORE = (MODE == BIG_SWIGLU ? 4 : 8) * IT;  // stores per wave and full tile
  // A slab's loads go out in two halves, the first into a buffer the moment it is free, the second over the next
  // k-step: they have two to three and a half k-steps (1000 to 1800 cycles) to land.
  constexpr int EARLY = NLOAD / 2;
  static_assert(NLOAD < 64 && NSTORE < 64, "vmcnt has six bits");
  // two slab buffers and the waves' output staging areas
  __shared__ __attribute__((aligned(1024))) char smem[2 * SLAB];
  __shared__ __attribute__((aligned(16))) char sOut[MODE == BIG_OUTER_MEAN ? 16 : 4 * EPI_BYTES];
  // (a wave's) 128 bias values
  __shared__ __attribute__((aligned(16))) float sColBias[MODE == BIG_COLUMN_OPS ? 4 * 128 : MODE == BIG_OUTER_MEAN ? 128 : 4];

  const int tid = threadIdx.x, lane = tid & 63;
  if (MODE == BIG_OUTER_MEAN && tid < 128) sColBias[tid] = g.bias[tid];  // (read behind many barriers)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, l31 = lane & 31;
  const int wm = (wave >> 1) * WM, wn = (wave & 1) * 128;

  // The workgroups are persistent (one per CU) and walk their tiles in a fixed order.
  // Workgroup ids are dealt round-robin to the 8 XCDs: id -> (xcd, slot) -> tile (XcdWalk), so that the tiles that
  // share a panel of A or B run on one XCD at about the same time and find it in its L2.
  const int tiles_m = (g.M + CM - 1) / CM, tiles_n = (g.N + CN - 1) / CN;
  const int total = tiles_m * tiles_n * g.batch;
  const int per_xcd = (total + 7) / 8;
  const int xcd = blockIdx.x & 7, slot_step = gridDim.x >> 3;
  struct Tile { int m0, n0, bz; };
  auto tile_at = [&](int& slot, Tile& t) -> bool {
    if constexpr (MODE == BIG_OUTER_MEAN) {
      // Both operands are much larger than an L2: an XCD's 32 CUs take 4 x 8 tiles at a time, 12 panels for 32 tiles.
      const int gm = (tiles_m + 3) / 4, groups = gm * ((tiles_n + 7) / 8);
      for (;; slot += slot_step) {
        const int group = (slot >> 5) * 8 + xcd;
        if (group >= groups) return false;
        const int tm = group % gm * 4 + (slot & 3), tn = group / gm * 8 + (slot >> 2 & 7);
        t.m0 = __builtin_amdgcn_readfirstlane(tm * CM);
        t.n0 = __builtin_amdgcn_readfirstlane(tn * CN);
        t.bz = 0;
        if (tm < tiles_m && tn < tiles_n) return true;
      }
    }
    int tm, tn;
    t.bz = 0;
    if (g.xcd_m) {
      if (!xcd_rect_tile(g.xcd_m, xcd, slot, tiles_m, tiles_n, &tm, &tn)) return false;
    } else {
      const int logical = xcd * per_xcd + slot;
      if (slot >= per_xcd || logical >= total) return false;
      tm = logical % tiles_m;
      tn = (logical / tiles_m) % tiles_n;
      t.bz = logical / (tiles_m * tiles_n);
    }
    // (the divisions above go through the vector unit; say again that the results are uniform)
    t.m0 = __builtin_amdgcn_readfirstlane(tm * CM);
    t.n0 = __builtin_amdgcn_readfirstlane(tn * CN);
    t.bz = __builtin_amdgcn_readfirstlane(t.bz);
    return true;
  };
  int slot = blockIdx.x >> 3, load_slot = slot;
  Tile cur_t, load_t;
  if (!tile_at(slot, cur_t)) return;
  load_t = cur_t;

  // Per slab a wave issues LA loads for A and eight for B: load i covers rows 16 IT wave + 8 i .. + 8 of A, 64 wave +
  // 8 i .. + 8 of B (one 128-byte row per 8 lanes).  The lane at position pc of row r fetches chunk pc ^ ((r >> 1) & 7).
  // Rows past the end repeat the last one (what they produce lands in output rows that
  // are never stored or in columns N..ldc-1 of T, which no consumer reads); a
  // chunk past K gets an offset past the buffer's end and arrives as zeros.
  const int ld_r = lane >> 3;
  const int ld_c[2] = {(lane & 7) ^ (lane >> 4), (lane & 7) ^ (4 + (lane >> 4))};  // even and odd i
  u32x4 A, B;
  uint32_t offa[LA], offb[8];
  auto point = [&](const Tile& t) {
    if constexpr (MODE == BIG_OUTER_MEAN) {  // operands of any size: offsets from the tile's first rows
      A = buffer_of(g.A + t.m0 * g.lda);
      B = buffer_of(g.B + t.n0 * g.ldb);
#pragma unroll
      for (int i = 0; i < LA; ++i)
        offa[i] = ((uint32_t)min(16 * IT * wave + 8 * i + ld_r, g.M - 1 - t.m0) * (uint32_t)g.lda + ld_c[i & 1] * 8) * 2u;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        offb[i] = ((uint32_t)min(64 * wave + 8 * i + ld_r, g.N - 1 - t.n0) * (uint32_t)g.ldb + ld_c[i & 1] * 8) * 2u;
      return;
    }
    A = buffer_of(g.A + (int64_t)t.bz * g.sA);
    B = buffer_of(g.B + (int64_t)t.bz * g.sB);
#pragma unroll
    for (int i = 0; i < LA; ++i)
      offa[i] = ((uint32_t)min(t.m0 + 16 * IT * wave + 8 * i + ld_r, g.M - 1) * (uint32_t)g.lda + ld_c[i & 1] * 8) * 2u;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      offb[i] = ((uint32_t)min(t.n0 + 64 * wave + 8 * i + ld_r, g.N - 1) * (uint32_t)g.ldb + ld_c[i & 1] * 8) * 2u;
  };
  const int nk = (g.K + CK - 1) / CK;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)smem;
  // The slab being loaded: slab load_k of load_t, to the buffer at load_a (its A part, this wave's share) / load_b.
  // It runs on across tiles: behind a tile's last slab come the workgroup's next tile's (behind the last tile's,
  // its own first ones again, unused), so a tile's first slabs arrive while the previous tile finishes and is stored.
  int load_k = 0;
  uint32_t load_a = __builtin_amdgcn_readfirstlane(lds0 + 16 * IT * wave * ROWB);
  uint32_t load_b = __builtin_amdgcn_readfirstlane(lds0 + SLAB_A + 64 * wave * ROWB);
  uint32_t kb = 0;
  bool in_k[2];
  auto begin_slab = [&]() {
    kb = __builtin_amdgcn_readfirstlane((uint32_t)load_k * (CK * 2));
    in_k[0] = load_k * CK + ld_c[0] * 8 < g.K;
    in_k[1] = load_k * CK + ld_c[1] * 8 < g.K;
  };
  auto next_slab = [&]() {
    load_a ^= SLAB;
    load_b ^= SLAB;
    if (++load_k == nk && MODE != BIG_OUTER_MEAN) {  // (there the loads past the end are zeros without a fetch)
      load_k = 0;
      load_slot += slot_step;
      if (!tile_at(load_slot, load_t)) load_t = cur_t;
      point(load_t);
    }
    begin_slab();
  };
  auto load = [&](auto i_c) {
    constexpr int i = decltype(i_c)::value;
    if constexpr (i < LA) load_to_lds<i * 8 * ROWB>(A, kb, in_k[i & 1] ? offa[i] : 0x80000000u, load_a);
    else load_to_lds<(i - LA) * 8 * ROWB>(B, kb, in_k[(i - LA) & 1] ? offb[i - LA] : 0x80000000u, load_b);
  };
  auto loads = [&](auto from_c, auto to_c) {  // loads from .. to - 1 of the slab
    constexpr int from = decltype(from_c)::value;
    each<decltype(to_c)::value - from>([&](auto i_c) { load(I<from + decltype(i_c)::value>{}); });
  };

  // Fragment (row R = base + 32 t + l31, k-step ks, half hh) is chunk 2 ks + hh
  // of row R, at position (2 ks + hh) ^ ((R >> 1) & 7); the bases are multiples
  // of 32, so the permutation depends on l31 only.
  uint32_t fra[4], frb[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const uint32_t fo = (uint32_t)(l31 * ROWB + (((2 * ks + hh) ^ ((l31 >> 1) & 7)) << 4));
    fra[ks] = wm * ROWB + fo;
    frb[ks] = SLAB_A + wn * ROWB + fo;
  }

  // acc[jt][it] = (T^T) tile: rows j = wn + 32 jt + .., columns i = wm + 32 it + ..
  f32x16 acc[4][IT];

  bf16x8 fa[2][IT], fb[2][4];
  auto frag = [&](int set, int ks, int j) {
    if (j < IT) fa[set][j] = as_frag(*reinterpret_cast<const u32x4*>(smem + fra[ks] + j * (32 * ROWB)));
    else fb[set][j - IT] = as_frag(*reinterpret_cast<const u32x4*>(smem + frb[ks] + (j - IT) * (32 * ROWB)));
  };
  // The IT + 4 fragment reads of a k-step with loads FROM .. TO - 1 dealt evenly between them, in
  // this order in the source: the loads are opaque to the scheduler, which keeps memory
  // operations on their side of one, so this is what spreads the loads over the k-step.
  auto frags_and_loads = [&](int set, int ks, auto from_c, auto to_c) {
    constexpr int from = decltype(from_c)::value, n = decltype(to_c)::value - from, J = IT + 4;
    each<J>([&](auto j_c) {
      constexpr int j = decltype(j_c)::value;
      frag(set, ks, j);
      loads(I<from + j * n / J>{}, I<from + (j + 1) * n / J>{});
    });
  };
  // `fresh`: the first k-step of a tile starts its accumulators from the constant zero
  auto mfmas = [&](int set, auto fresh_c) {
    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int jt = 0; jt < 4; ++jt)
#pragma unroll
      for (int it = 0; it < IT; ++it)
        acc[jt][it] = mfma32(fb[set][jt], fa[set][it], decltype(fresh_c)::value ? zero : acc[jt][it]);
  };
  // 4 IT MFMAs with the IT + 4 fragment reads (and the loads that sit between them) spread over them
  auto interleave = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, IT - 2, 0);  // two MFMAs (one when there are twelve)
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  auto issue_first = [&]() {  // the first two slabs of cur_t
    point(cur_t);
    load_k = 0;
    begin_slab();
    loads(I<0>{}, I<NLOAD>{});
    next_slab();
    loads(I<0>{}, I<NLOAD>{});
  };
  auto await_first = [&]() {  // its first slab has landed, the first fragments are read
    wait_loads_but<NLOAD>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < IT + 4; ++j) frag(0, 0, j);
  };
  issue_first();
  await_first();

  // One slab, its first fragments already in set 0.  FRESH: a tile's first (all of the next slab's loads are under way,
  // and the previous tile's NSTORE stores, if any, behind them).
  const I<0> none{};
  auto stage = [&](auto fresh_c, bool stores_behind) {
    constexpr bool fresh = decltype(fresh_c)::value;
    frags_and_loads(1, 1, I<fresh ? NLOAD : EARLY>{}, I<NLOAD>{});
    mfmas(0, fresh_c);
    interleave();
    frags_and_loads(0, 2, none, none);
    mfmas(1, std::false_type{});
    interleave();
    frags_and_loads(1, 3, none, none);
    mfmas(0, std::false_type{});
    interleave();
    // This wave has read all it needs of the slab, and its share of the next one has landed.  Past the barrier
    // that holds for every wave: the next slab is complete, this one's buffer is free.
    if (fresh && stores_behind) wait_loads_but<NSTORE>();
    else wait_loads_but<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      fra[ks] ^= SLAB;
      frb[ks] ^= SLAB;
    }
    next_slab();
    frags_and_loads(0, 0, I<0>{}, I<EARLY>{});
    mfmas(1, std::false_type{});
    interleave();
  };

  // Epilogue of one tile, per wave and without a barrier: the wave stages 32 rows i x 64 columns j
  // of its quadrant at a time in its own corner of sOut and reads them back itself (a wave's
  // LDS operations execute in order), then writes 128-byte row segments.  It touches neither the
  // slab buffers nor the loads in flight into them.
  // Lane (l31, hh), register quad q of tile (jt, it): row i = 32 it + l31,
  // columns j = 32 jt + 8 q + 4 hh + 0..3.  Values are finished four at a time on their way from
  // the accumulators to LDS, so that few of them are live at once.
  bf16_t* sE = reinterpret_cast<bf16_t*>(sOut + wave * EPI_BYTES);
  auto store_tile = [&](const Tile& t) {
    bf16_t* C = reinterpret_cast<bf16_t*>(g.C) + (int64_t)t.bz * g.sC;
    // SwiGLU: accumulator tiles (0,1) and (2,3) give 32 output columns each, one pass per 32 rows;
    // otherwise two passes of 64 output columns
    constexpr int PASSES = MODE == BIG_SWIGLU ? 1 : 2;
    const int c8 = lane & 7, rsub = lane >> 3;  // 8 chunks of 8 output columns per row, 8 rows per instruction
    const uint32_t lane_off = (uint32_t)(rsub * g.ldc + c8 * 8) * 2u;
    const int col_end = MODE == BIG_SWIGLU ? g.N / 2 : MODE == BIG_PLAIN ? g.ldc : g.N;
    const __amdgpu_buffer_rsrc_t whole =
        __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(C), 0, MODE == BIG_COLUMN_OPS && g.regroup32 ? g.M * g.N * 2 : 0, RSRC_RAW);
    // Pass n = (it, p): 32 rows x 64 output columns.  convert: accumulators -> eight packed 8-byte
    // pieces per lane; write: those into the staging area; read_store: 16 bytes per lane back out
    // of it and to memory.  The passes are software-pipelined in the source (write n, convert
    // n + 1, read_store n): the conversions of the next pass fill the LDS round trip of this one.
    constexpr int NP = IT * PASSES;
    // The bias of the wave's 128 columns goes through LDS once per tile, requested before the
    // tile's first store: a load from memory issued between the stores would wait for them all
    // (vector memory operations retire in order).
    float* sBiasW = sColBias + (MODE == BIG_COLUMN_OPS ? wave * 128 : 0);
    if constexpr (MODE == BIG_COLUMN_OPS) {
      // the bias array only covers the segments that use it
      int first;
      const bool uses_bias = big_tile_bias_quad(g, t.n0 + wn + 4 * lane, &first) && lane < 32;
      f32x4 b4 = {0.f, 0.f, 0.f, 0.f};
      if (uses_bias) b4 = *reinterpret_cast<const f32x4*>(g.bias + first);
      if (lane < 32) *reinterpret_cast<f32x4*>(sBiasW + 4 * lane) = b4;
    }
    auto convert = [&](int n, u32x2* out) {
      const int it = n / PASSES, p = n % PASSES;
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int jt = MODE == BIG_SWIGLU ? 2 * jj : 2 * p + jj;
        // column ops: a 32-column block never straddles segments (seg_len % 32 == 0)
        bool affine = false, sig = false;
        float alpha = 1.f;
        const int nb = t.n0 + wn + 32 * jt;
        if constexpr (MODE == BIG_COLUMN_OPS) {
          int op = SEG_BIAS_SCALE;
          sig = g.act_sigmoid != 0;
          if (g.epi == EPI_SEGMENTED) {
            op = (g.seg_ops >> (4 * (min(nb, g.N - 1) / g.seg_len))) & 15;
            sig = op == SEG_SIGMOID;
          }
          affine = op == SEG_BIAS_SCALE;
          if (affine) alpha = g.alpha;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float o[4];
          f32x4 bb = {0.f, 0.f, 0.f, 0.f};
          if constexpr (MODE == BIG_COLUMN_OPS) {
            if (affine && g.bias) bb = *reinterpret_cast<const f32x4*>(sBiasW + 32 * jt + 8 * q + 4 * hh);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = acc_read(acc[jt][it][4 * q + e]);
            if constexpr (MODE == BIG_COLUMN_OPS) {
              v = (v + bb[e]) * alpha;
              if (sig) v = sigmoidf_(v);
            }
            if constexpr (MODE == BIG_SWIGLU) v = v * sigmoidf_(v) * acc_read(acc[jt + 1][it][4 * q + e]);
            o[e] = v;
          }
          out[4 * jj + q].x = pack2bf(o[0], o[1]);
          out[4 * jj + q].y = pack2bf(o[2], o[3]);
        }
      }
    };
    auto write = [&](const u32x2* in) {
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<u32x2*>(sE + l31 * LDE + 32 * jj + 8 * q + 4 * hh) = in[4 * jj + q];
    };
    // Bounds are enforced by the memory pipeline, not by branches (which would cut the
    // epilogue into many basic blocks): a buffer descriptor that ends with the last valid row
    // of this 32-row block drops rows past M, and lanes whose columns lie past the end
    // get an offset beyond any descriptor.  Every wave issues all its stores.
    auto read_store = [&](int n) {
      const int it = n / PASSES, p = n % PASSES;
      const int row0 = t.m0 + wm + 32 * it;
      const __amdgpu_buffer_rsrc_t rows32 = __builtin_amdgcn_make_buffer_rsrc(
          uniform_ptr(C + (int64_t)row0 * g.ldc), 0,
          __builtin_amdgcn_readfirstlane(max(0, min(32, g.M - row0)) * g.ldc * 2), RSRC_RAW);
      const int col0 = MODE == BIG_SWIGLU ? (t.n0 + wn) / 2 : t.n0 + wn + 64 * p;
      const uint32_t voff = c8 * 8 < col_end - col0 ? lane_off + (uint32_t)col0 * 2u : 0x80000000u;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int r = 8 * s + rsub;
        const u32x4 v = *reinterpret_cast<const u32x4*>(sE + r * LDE + c8 * 8);
        if (MODE == BIG_COLUMN_OPS && g.regroup32) {
          const int row = row0 + r, col = col0 + c8 * 8;
          const uint32_t off = ((((uint32_t)(row >> 5) * (uint32_t)(g.N >> 5) + (col >> 5)) * 32 + (row & 31)) * 32 + (col & 31)) * 2u;
          __builtin_amdgcn_raw_buffer_store_b128(v, whole, row < g.M && col < g.N ? off : 0x80000000u, 0, 0);
        } else {
          __builtin_amdgcn_raw_buffer_store_b128(v, rows32, voff + (uint32_t)(8 * s * g.ldc) * 2u, 0, 0);
        }
      }
    };
    u32x2 vals[2][8];
    convert(0, vals[0]);
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      write(vals[n & 1]);
      if (n + 1 < NP) convert(n + 1, vals[(n + 1) & 1]);
      read_store(n);
    }
  };

  // Outer-product mean of the tile's 2 IT x 8 token pairs (b, d): pair = (res ? pair : 0) + (W vec(outer) + bias) * gate.
  // The outer products go to the slab buffers (which hold nothing by now) as 16 IT rows of 1024 bf16, chunk c of row r at
  // position c ^ (c >> 4 & 3) ^ (r & 15): both the 8-byte writes and the fragment reads spread over the banks.  Wave w
  // takes outputs 32 w .. 32 w + 31 of all pairs; its share of the weights, packed in the order of its loads, comes
  // from L2, 64 KB per tile (W's rows in the order swap23: eight consecutive outputs per lane).
  // 768 tokens, 1024 MSA rows: 1080 us, of which a tile's K loop is two thirds.  As two products with the outer products
  // in memory between them (six times 205 + 66 us) the same bits took 1630; 187 tokens, 301 rows 47 (75; with
  // tiles of 192 rows 41), 160 tokens, 128 rows 25 (55).
  constexpr int PH = IT == 2 ? 1 : 2;  // a tile's 2 IT x 8 token pairs, 32 at a time
  f32x16 outer[PH];                    // 32 outputs x 32 pairs each
  float outer_gate[PH];
  u32x4 outer_res[PH][2][2];
  auto outer_pixel = [&](const Tile& t, int p, bool* ok) {
    const int n = g.N >> 5, b = (t.m0 >> 5) + 4 * p + (l31 >> 3), d = (t.n0 >> 5) + (l31 & 7);
    *ok = b < n && d < n && 4 * p + (l31 >> 3) < 2 * IT;
    return (int64_t)min(b, n - 1) * n + min(d, n - 1);
  };
  auto outer_tile = [&](const Tile& t) {
    constexpr int KSTEPS = 64, RW = 8, RX = 6;  // fragments under way: weights from L2, outer products from LDS
    const bf16_t* wp = uniform_ptr(g.w2 + wave * KSTEPS * 512) + lane * 8;
    u32x4 wf[RW], xf[RX][PH];
    auto load_w = [&](int ks) {
      if (ks < KSTEPS) wf[ks % RW] = *reinterpret_cast<const u32x4*>(wp + ks * 512);
    };
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) load_w(ks);
    // (a lane number that the compiler cannot know to be the same for every tile: it would keep the 128 addresses below
    // in registers for the kernel's lifetime)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int hh = ln >> 5, l31 = ln & 31;
    const uint32_t st = (uint32_t)((8 * (wm >> 5) + (wn >> 5)) * 2048 + 8 * hh);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t chunk = (uint32_t)(4 * l31 + (q ^ (l31 >> 2 & 3))) ^ (uint32_t)((wn >> 5) + 8 * (wm >> 5 & 1));
#pragma unroll
      for (int it = 0; it < IT; ++it)
#pragma unroll
        for (int jt = 0; jt < 4; ++jt) {
          u32x2 v;
          v.x = pack2bf(acc_read(acc[jt][it][4 * q]), acc_read(acc[jt][it][4 * q + 1]));
          v.y = pack2bf(acc_read(acc[jt][it][4 * q + 2]), acc_read(acc[jt][it][4 * q + 3]));
          *reinterpret_cast<u32x2*>(smem + st + ((chunk ^ (8 * (it & 1) + jt)) << 4) + (8 * it + jt) * 2048) = v;
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const uint32_t rd = (uint32_t)(l31 * 2048 + ((hh ^ (l31 & 15)) << 4));
    auto read_x = [&](int ks) {
      if (ks < KSTEPS) {
        const uint32_t at = rd ^ (uint32_t)((2 * ks ^ (ks >> 3 & 3)) << 4);
#pragma unroll
        for (int p = 0; p < PH; ++p) xf[ks % RX][p] = *reinterpret_cast<const u32x4*>(smem + at + p * 65536);
      }
    };
#pragma unroll
    for (int p = 0; p < PH; ++p)
#pragma unroll
      for (int r = 0; r < 16; ++r) outer[p][r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < RX - 1; ++ks) read_x(ks);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      if (ks == 0) {
#pragma unroll
        for (int i = 4; i < RW - 1; ++i) load_w(i);
      }
      if (ks == KSTEPS / 2) {  // what the results are joined with
#pragma unroll
        for (int p = 0; p < PH; ++p) {
          bool ok;
          const int64_t pix = outer_pixel(t, p, &ok);
          outer_gate[p] = g.gate[pix];
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const int64_t o = pix * 128 + 32 * wave + 16 * s + 8 * hh;
            outer_res[p][s][0] = outer_res[p][s][1] = u32x4{0, 0, 0, 0};
            if (g.res_f32) {
              outer_res[p][s][0] = *reinterpret_cast<const u32x4*>(g.res_f32 + o);
              outer_res[p][s][1] = *reinterpret_cast<const u32x4*>(g.res_f32 + o + 4);
            }
            if (g.res_bf16) outer_res[p][s][0] = *reinterpret_cast<const u32x4*>(g.res_bf16 + o);
          }
        }
      }
      load_w(ks + RW - 1);
      read_x(ks + RX - 1);
#pragma unroll
      for (int p = 0; p < PH; ++p) outer[p] = mfma32(as_frag(wf[ks % RW]), as_frag(xf[ks % RX][p]), outer[p]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto outer_store = [&](const Tile& t) {
#pragma unroll
    for (int p = 0; p < PH; ++p) {
      bool ok;
      const int64_t pix = outer_pixel(t, p, &ok);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int64_t o = 32 * wave + 16 * s + 8 * hh;
        float v[8], bias[8], res[8];
        Elem<float>::load8(sColBias + o, bias);
        if (g.res_f32)
          for (int e = 0; e < 8; ++e) res[e] = __uint_as_float(outer_res[p][s][e >> 2][e & 3]);
        else unpack8(outer_res[p][s][0], res);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (outer[p][8 * s + e] + bias[e]) * outer_gate[p] + res[e];
        if (!ok) continue;
        if (g.out_f32) Elem<float>::store8(reinterpret_cast<float*>(g.C) + pix * 128 + o, v);
        else Elem<bf16_t>::store8(reinterpret_cast<bf16_t*>(g.C) + pix * 128 + o, v);
      }
    }
  };

  bool stored = false;  // a tile's epilogue (NSTORE stores per wave, whatever the bounds) lies behind
  while (true) {
    stage(std::true_type{}, stored);
    for (int kt = 1; kt < nk; ++kt) stage(std::false_type{}, false);
    if constexpr (MODE == BIG_OUTER_MEAN) {
      wait_loads_but<0>();
      __builtin_amdgcn_s_barrier();  // every wave has read its last fragments, and no load into the buffers is under way
      asm volatile("" ::: "memory");
      outer_tile(cur_t);
      // every wave has read its outer products: the next tile's slabs may come, while this one's results go
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const Tile done = cur_t;
      slot += slot_step;
      const bool more = tile_at(slot, cur_t);
      if (more) {
        load_a ^= SLAB;  // back to the buffer that the fragments are read from next
        load_b ^= SLAB;
        issue_first();
      }
      outer_store(done);
      if (!more) break;
      await_first();
    } else {
      loads(I<EARLY>{}, I<NLOAD>{});
      store_tile(cur_t);
      __builtin_amdgcn_sched_barrier(0);
      slot += slot_step;
      if (!tile_at(slot, cur_t)) break;
      stored = true;
    }
  }
  wait_loads_but<0>();  // nothing may be in flight into LDS when the workgroup ends
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// Layout assumptions the large tile shares over its modes.
static bool big_tile_layout_ok(const GemmArgs& g) {
  return !g.out_f32 && g.M > 0 && g.N > 0 && g.K > 0 && g.batch > 0 && (g.lda & 7) == 0 && (g.ldb & 7) == 0 &&
         (g.ldc & 7) == 0 && (g.K & 7) == 0 && g.K <= g.lda && g.K <= g.ldb && (g.sA & 7) == 0 && (g.sB & 7) == 0 &&
         (g.sC & 7) == 0 && al16(g.A) && al16(g.B) && al16(g.C) &&
         (int64_t)g.M * g.lda < (1ll << 30) && (int64_t)g.N * g.ldb < (1ll << 30) && g.ldc < (1 << 24);
}

// Plain bf16 batched NT product with the large tile; false if the operands do
// not meet its layout assumptions (the caller then takes the general GEMM).
bool contract_supported(const GemmArgs& g) {
  return g.epi == EPI_PLAIN && !g.bias && !g.act_sigmoid && g.alpha == 1.f && !g.regroup32 && !g.gate &&
         big_tile_layout_ok(g) && g.ldc >= ((g.N + 7) & ~7);
}

// Which large-tile instance can take this product with its epilogue: -1 = none.
int big_tile_mode(const GemmArgs& g) {
  if (!big_tile_layout_ok(g) || g.gate || g.res_f32 || g.res_bf16) return -1;
  if (g.epi == EPI_SWIGLU) return (g.N & 63) == 0 && g.ldc >= g.N / 2 && !g.regroup32 ? BIG_SWIGLU : -1;
  if (g.N & 7) return -1;
  if (!g.regroup32 && g.ldc < g.N) return -1;
  if (g.bias && !al16(g.bias)) return -1;
  if (g.epi == EPI_SEGMENTED) return g.seg_len > 0 && (g.seg_len & 31) == 0 && !g.regroup32 ? BIG_COLUMN_OPS : -1;
  if (g.epi != EPI_PLAIN) return -1;
  if (g.regroup32)
    return g.batch == 1 && (g.M & 31) == 0 && (g.N & 31) == 0 && (int64_t)g.M * g.N < (1ll << 30) ? BIG_COLUMN_OPS : -1;
  return (g.bias || g.act_sigmoid || g.alpha != 1.f) ? BIG_COLUMN_OPS : BIG_PLAIN;
}

void gemm_bias_span(const GemmArgs& g, bool big, int64_t* first, int64_t* last) {
  int64_t lo = INT64_MAX, hi = 0;
  if (g.bias && g.N > 0 && (g.epi != EPI_SEGMENTED || g.seg_len > 0)) {
    if (big) {
      // every (tile column, wave column, lane) of the epilogue's bias fetch
      for (int n0 = 0; n0 < g.N; n0 += CN)
        for (int wn = 0; wn < CN; wn += 128)
          for (int lane = 0; lane < 32; ++lane) {
            int f;
            if (!big_tile_bias_quad(g, n0 + wn + 4 * lane, &f)) continue;
            lo = std::min<int64_t>(lo, f);
            hi = std::max<int64_t>(hi, (int64_t)f + 4);
          }
    } else {
      // gemm_nt_kernel: chunk of up to 8 columns from every multiple of 8 below N
      for (int n = 0; n < g.N; n += 8) {
        if (!gemm_col_uses_bias(g, n)) continue;
        lo = std::min<int64_t>(lo, n);
        hi = std::max<int64_t>(hi, std::min<int64_t>(n + 8, g.N));
      }
    }
  }
  *first = hi > 0 ? lo : 0;
  *last = hi;
}

// the device's CUs, at least 8
static int cu_count() {
  static int cus = 0;
  if (cus == 0) {
    int dev_id = 0;
    hipDeviceProp_t prop;
    cus = hipGetDevice(&dev_id) == hipSuccess && hipGetDeviceProperties(&prop, dev_id) == hipSuccess &&
                  prop.multiProcessorCount > 0
              ? std::max(prop.multiProcessorCount, 8)
              : 256;
  }
  return cus;
}

int launch_big_tile(const GemmArgs& g_in, int mode, hipStream_t stream) {
  GemmArgs g = g_in;
  if (!g.A || !g.B || !g.C) return AF3_ERR_BAD_ARG;
  if (mode != big_tile_mode(g) && !(mode == BIG_PLAIN && contract_supported(g))) return AF3_ERR_BAD_ARG;
  if (mode < BIG_PLAIN || mode > BIG_SWIGLU) return AF3_ERR_BAD_ARG;
  if (mode == BIG_COLUMN_OPS && g.bias) {
    // the epilogue fetches the bias in groups of four per lane: nothing it touches may lie outside the array
    int64_t first, last;
    gemm_bias_span(g, true, &first, &last);
    if (first < 0 || last > g.bias_len) return AF3_ERR_BAD_ARG;
  }
  const int64_t tiles_n = (g.N + CN - 1) / CN;
  const int64_t total4 = (int64_t)((g.M + 255) / 256) * tiles_n * g.batch;
  const int64_t total3 = (int64_t)((g.M + 191) / 192) * tiles_n * g.batch;
  // Rounds of workgroups on the device's CUs (one workgroup per CU) times the cost of one.  A 192 x 256
  // block costs 0.83 - 0.86 of a 256 x 256 one, not 0.75 (measured: pipeline fill and the epilogue do not
  // shrink with it), so it is taken for the plain product only when it saves more rounds than that:
  // N = 256 .. 576, not 768 (six rounds against five) or beyond.
  const int cus = cu_count();
  const bool flat = ((total3 + cus - 1) / cus) * 7 < ((total4 + cus - 1) / cus) * 8;
  const XcdWalk walk = xcd_walk((g.M + (flat ? 191 : 255)) / (flat ? 192 : 256), tiles_n, g.batch, flat ? 192 : 256, CN, cus / 8);
  if (walk.slots * 8 > 0x3fffffff) return AF3_ERR_BAD_ARG;
  g.xcd_m = walk.rows;
  // persistent workgroups, one per CU (a multiple of 8: ids are dealt round-robin to the 8 XCDs)
  const int64_t blocks = std::min<int64_t>(walk.slots * 8, cus / 8 * 8);
  const dim3 grid((unsigned)blocks), block(256);
  if (flat && mode == BIG_PLAIN) hipLaunchKernelGGL((contract_kernel<BIG_PLAIN, 3>), grid, block, 0, stream, g);
  else if (flat && mode == BIG_COLUMN_OPS) hipLaunchKernelGGL((contract_kernel<BIG_COLUMN_OPS, 3>), grid, block, 0, stream, g);
  else if (flat) hipLaunchKernelGGL((contract_kernel<BIG_SWIGLU, 3>), grid, block, 0, stream, g);
  else if (mode == BIG_PLAIN) hipLaunchKernelGGL(contract_kernel<BIG_PLAIN>, grid, block, 0, stream, g);
  else if (mode == BIG_COLUMN_OPS) hipLaunchKernelGGL(contract_kernel<BIG_COLUMN_OPS>, grid, block, 0, stream, g);
  else hipLaunchKernelGGL(contract_kernel<BIG_SWIGLU>, grid, block, 0, stream, g);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

// A = left [(b, c)][lda], B = right [(d, e)][ldb] with c, e < 32 and M = N = 32 n, w2 the packed output weights
// (outer_mean_weight), bias [128], gate [n][n], C (and residual) [n][n][128].
int launch_outer_mean(const GemmArgs& g, hipStream_t stream) {
  if (!g.A || !g.B || !g.C || !g.w2 || !g.bias || !g.gate || g.M <= 0 || g.M != g.N || (g.M & 31) || g.K <= 0 || g.batch != 1)
    return AF3_ERR_BAD_ARG;
  if ((g.K & 7) || (g.lda & 7) || (g.ldb & 7) || g.K > g.lda || g.K > g.ldb || g.lda >= (1 << 21) || g.ldb >= (1 << 21))
    return AF3_ERR_BAD_ARG;
  if (!al16(g.A) || !al16(g.B) || !al16(g.C) || !al16(g.w2) || !al16(g.bias) || !al16(g.res_f32) || !al16(g.res_bf16))
    return AF3_ERR_BAD_ARG;
  // Tiles of 256, 192 or 128 rows, by what their rounds cost (an XCD's CUs take 4 x 8 tiles at a time): a slab of 64 MSA
  // rows 0.31 us for every 64 tile rows, the epilogue 10 us, of 32 token pairs 6.  The whole operator, tokens x MSA rows, us
  // with 256 / 192 / 128 rows: 64 x 512 44.3 / 41.3 / 36.4, 96 x 512 46.6 / 42.5 / 49.1, 128 x 512 47.1 / 60.1 / 52.3,
  // 160 x 128 47.2 / 53.8 / 52.0, 187 x 301 79.0 / 73.2 / 77.6, 187 x 1024 132 / 116 / 133, 260 x 1024 216 / 217 / 250.
  const int64_t tn = (g.M + 255) / 256, nk = (g.K + CK - 1) / CK;
  auto slots_of = [&](int it) { return ((g.M + 64 * it - 1) / (64 * it) + 3) / 4 * ((tn + 7) / 8); };
  auto cost = [&](int it) { return (slots_of(it) + 7) / 8 * (it * nk + (it == 2 ? 20 : 32)); };
  int it = 4;
  if (cost(3) * 20 < cost(it) * 19) it = 3;
  if (cost(2) * 20 < cost(it) * 19) it = 2;
  const int64_t slots = (slots_of(it) + 7) / 8 * 256;
  if (slots > 0x3fffffff) return AF3_ERR_BAD_ARG;
  const dim3 grid((unsigned)std::min<int64_t>(slots, cu_count() / 8 * 8)), block(256);
  if (it == 2) hipLaunchKernelGGL((contract_kernel<BIG_OUTER_MEAN, 2>), grid, block, 0, stream, g);
  else if (it == 3) hipLaunchKernelGGL((contract_kernel<BIG_OUTER_MEAN, 3>), grid, block, 0, stream, g);
  else hipLaunchKernelGGL((contract_kernel<BIG_OUTER_MEAN, 4>), grid, block, 0, stream, g);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

int launch_contract(const GemmArgs& g, hipStream_t stream) {
  if (!g.A || !g.B || !g.C || !contract_supported(g)) return AF3_ERR_BAD_ARG;
  return launch_big_tile(g, BIG_PLAIN, stream);
}
