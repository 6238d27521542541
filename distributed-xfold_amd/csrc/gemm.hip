// Batched "NT" GEMM on bf16 MFMA:  C[b][m][n] = epi( sum_k A[b][m][k] * B[b][n][k] )
//
// Both operands are k-contiguous, which is the natural fragment order of
// v_mfma_f32_32x32x16_bf16, so a 16-byte read feeds one fragment.  This file
// carries the dense projections outside the 128-channel pair path (single /
// diffusion / atom attention and transitions) and the triangle contraction of
// small token counts; large products whose epilogue the 256x256-tile kernel
// (contract.hip) knows are handed to it by launch_gemm_nt.
//
// Most of these products are short: 64 to 4000 rows, K = 128 ... 1536, 0.1 to
// 10 GFLOP, so that what they cost is not matrix time but the number of CUs
// that have a tile and the length of one workgroup's chain (first miss, K loop,
// hand-over, store).  Hence:
//   * the tile shrinks with the product (128x128 down to 32x32) until about every CU has one, and
//     where that is not enough and the caller does not mind the order of summation (GemmArgs::split_k)
//     the waves of a workgroup share the K range of one tile instead of its area (WK groups; their fp32
//     partial tiles are added in LDS): K = 1536 is then a chain of three slabs, not of 24;
//   * slabs are 64 deep, so a slab row is one whole 128-byte cache line.  From L2 a CU takes
//     in 115 bytes/ns that way; in 64-byte row pieces it is 62 (measured, LDS-direct loads);
//   * slabs go from global memory straight into LDS, all of a workgroup's first ones
//     before anything is waited for.  A group of one wave (ALONE) shares its slabs with
//     nobody: its K loop has no barrier, only waits for its own loads;
//   * the accumulators hold C^T tiles (weight fragments as the MFMA's A operand): a
//     lane owns one row and four consecutive columns per register quad, so a partial
//     tile goes to LDS in 16-byte stores.
//
// Without split_k every tile sums K in the same order, one 16-deep MFMA step after the other
// from k = 0, as the 256x256 tile does: a row gives the same bits alone and in a batch, whatever
// tile it lands in.
//
// Measured against the register-staged 128x128-tile kernel this replaces (weights not in L2): 500x768x768 5.6 us
// (was 14.3), 500x768x1536 7.5 (21.4), 500x3072x768 8.7 (16.2), 1920x3072x768 16.7 (22.6), 3840x768x768 13.8 (15.3),
// 768x73728x384 to fp32 112 (125), 12000x256x128 6.4 (11.3); with split_k 64x384x384 3.4 (8.9), 64x384x1536 4.9 (19.6).
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace {

constexpr int KS = 64;        // slab depth
constexpr int ROWB = KS * 2;  // bytes of a slab row in LDS (unpadded, 16-byte chunks permuted)
constexpr uint32_t BUFFER_END = 0x7fffffffu;  // size of a buffer descriptor that covers every offset of a tile

// 64 lanes x 16 bytes from a range-checked buffer (descriptor, wave-uniform byte offset, per-lane byte offset) to
// the ith KB of LDS behind the wave-uniform address lds.  An offset past the descriptor's size writes zeros and fetches
// nothing, but the load counts like any other: the waits of a loop can be constants, and K needs no tail.  Inline assembly, because the
// compiler's own form makes later LDS reads wait for every such load in flight; here a buffer is read only behind
// an explicit wait.
__device__ __forceinline__ void load_to_lds(const u32x4 rsrc, uint32_t soff, uint32_t off, uint32_t lds, int i) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(off), "s"(rsrc),
               "s"(soff), "n"(i * 1024)
               : "m0", "scc", "memory");
}
// raw buffer descriptor of a uniform pointer (word 3: untyped 32-bit data)
__device__ __forceinline__ u32x4 buffer_of(const void* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return u32x4{lo, hi & 0xffffu, BUFFER_END, 0x00020000u};
}
template <int N>
__device__ __forceinline__ void wait_loads_but() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A workgroup of WM x WN x WK waves computes BM = 32 MT WM rows x BN = 32 NT WN columns; ST slab buffers per group.
// CLEAN: K is a multiple of the slab depth.  KIND: the epilogue.  VEC: all of its loads and stores are 16-byte ones (without:
// element by element, for odd column counts and unaligned operands).  WPS: waves per SIMD the tile's LDS leaves room for; the
// registers have to as well (a wave more or less per SIMD is up to a factor of two in the short products).
enum { KIND_COLUMNS = 0, KIND_GATE_RES = 1, KIND_SWIGLU = 2 };
template <int MT, int NT, int WM, int WN, int WK, int ST, int WPS, bool CLEAN, int KIND, bool VEC, bool OUT_F32>
__global__ __launch_bounds__(64 * WM * WN * WK, WPS) void gemm_nt_kernel(GemmArgs g) {
  args_at_once<GemmArgs>();
  constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN, NTHR = 64 * WM * WN * WK, GW = WM * WN;
  constexpr int SLAB = (BM + BN) * ROWB;     // A rows first, then B rows
  constexpr int NLOAD = (BM + BN) / 8 / GW;  // 1 KB loads per wave and slab
  constexpr int LA = BM / 8 / GW;            // of which A
  static_assert(WK == 1 || WK == 2 || WK == 4 || WK == 8, "");
  static_assert((BM / 8) % GW == 0 && (BN / 8) % GW == 0, "loads of a slab are dealt evenly");
  constexpr bool ALONE = GW == 1;
  static_assert(ST >= 2 && (ST - 1) * NLOAD < 64, "vmcnt has six bits");
  constexpr int LDS_C = BN + 4;              // row stride (fp32) of a partial tile
  constexpr int BYTES = WK * ST * SLAB > WK * BM * LDS_C * 4 ? WK * ST * SLAB : WK * BM * LDS_C * 4;
  __shared__ __attribute__((aligned(1024))) char smem[BYTES];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, l31 = lane & 31;
  const int grp = wave / GW, gw = wave % GW;
  const int wm = (gw / WN) * 32 * MT, wn = (gw % WN) * 32 * NT;

  // Workgroup ids are dealt round-robin to the 8 XCDs: id -> (xcd, slot) -> tile (XcdWalk).
  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  int tm, tn, bz = 0;
  if (g.xcd_m) {
    if (!xcd_rect_tile(g.xcd_m, blockIdx.x & 7, blockIdx.x >> 3, tiles_m, tiles_n, &tm, &tn)) return;
  } else {
    const int total = tiles_m * tiles_n * g.batch, per_xcd = (total + 7) / 8;
    const int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || logical >= total) return;
    tm = logical % tiles_m;
    tn = (logical / tiles_m) % tiles_n;
    bz = __builtin_amdgcn_readfirstlane(logical / (tiles_m * tiles_n));
  }
  const int m0 = __builtin_amdgcn_readfirstlane(tm) * BM, n0 = __builtin_amdgcn_readfirstlane(tn) * BN;

  // the tile's first rows: what a lane adds to these fits 32 bits whatever the operands' size
  const u32x4 A = buffer_of(g.A + (int64_t)bz * g.sA + (int64_t)m0 * g.lda);
  const u32x4 B = buffer_of(g.B + (int64_t)bz * g.sB + (int64_t)n0 * g.ldb);

  // Load i of a wave covers eight rows of A (i < LA) or B, one 128-byte row per 8 lanes.  Chunk c of row r lives at
  // position c ^ ((r >> 1) & 7) of the row (a load cannot pad rows): 16 consecutive rows' reads of one chunk then
  // cover all 64 banks.  Rows past the end repeat the last one; what they produce is not stored.
  const int lr = lane >> 3;
  auto row_of = [&](int i) { return i < LA ? 8 * (LA * gw + i) + lr : 8 * ((NLOAD - LA) * gw + i - LA) + lr; };
  auto chunk_of = [&](int i) { return (lane & 7) ^ ((row_of(i) >> 1) & 7); };
  uint32_t off[NLOAD];
#pragma unroll
  for (int i = 0; i < NLOAD; ++i)
    off[i] = i < LA ? ((uint32_t)min(row_of(i), g.M - 1 - m0) * (uint32_t)g.lda + chunk_of(i) * 8) * 2u
                    : ((uint32_t)min(row_of(i), g.N - 1 - n0) * (uint32_t)g.ldb + chunk_of(i) * 8) * 2u;
  const int ns = (g.K + KS - 1) / KS;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)smem;
  const int s0 = grp * ns / WK, cnt = (grp + 1) * ns / WK - s0;
  const uint32_t mine = (uint32_t)(grp * (ST * SLAB));  // this group's buffers in smem
  auto issue = [&](int s, uint32_t dst) {  // slab s of this wave's share; past its end: zeros
    const uint32_t da = __builtin_amdgcn_readfirstlane(lds0 + dst + LA * gw * 1024);
    const uint32_t db = __builtin_amdgcn_readfirstlane(lds0 + dst + BM * ROWB + (NLOAD - LA) * gw * 1024);
    const int k0 = (s0 + s) * KS;
    const uint32_t kb = __builtin_amdgcn_readfirstlane((uint32_t)k0 * 2u);
    u32x4 ra = A, rb = B;
    ra.z = rb.z = __builtin_amdgcn_readfirstlane(s < cnt ? BUFFER_END : 0u);
#pragma unroll
    for (int i = 0; i < NLOAD; ++i) {
      const uint32_t o = CLEAN || k0 + chunk_of(i) * 8 < g.K ? off[i] : 0x80000000u;
      if (i < LA) load_to_lds(ra, kb, o, da, i);
      else load_to_lds(rb, kb, o, db, i - LA);
    }
  };

  // ------------------------------------------------------------- epilogue operands
  // After the K loop a thread finishes chunks of 8 consecutive columns.  Gate and residual of PRE chunks are
  // requested at a time, ahead of the stores (which may alias the residual, so no load moves above one); where a
  // thread has no more chunks than that and registers to spare, ahead of the K loop (500 rows, gate and residual in HBM:
  // a token transformer of 24 blocks 1 % faster; the tiles of four waves, of which others are there to cover, no faster).
  constexpr int CPR = BN / 8;                        // chunks per row
  constexpr int NCH = (BM * CPR + NTHR - 1) / NTHR;  // chunks per thread
  constexpr int PRE = NCH < 2 ? NCH : 2;
  constexpr bool EARLY = NCH <= PRE && (NCH == 1 || WPS == 1);
  struct Pre { float gate[8]; u32x4 r0, r1; };
  Pre pre[PRE];
  auto fetch = [&](int k, Pre& p) {
    const int idx = tid + k * NTHR, m = min(m0 + idx / CPR, g.M - 1), n = n0 + (idx % CPR) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) p.gate[e] = 1.f;
    p.r0 = p.r1 = u32x4{0, 0, 0, 0};
    if ((BM * CPR < NTHR && idx >= BM * CPR) || n >= g.N) return;
    const int64_t roff = (int64_t)bz * g.sRes + (int64_t)m * g.ld_res + n;
    const float* gp = g.gate && !g.gate_per_row ? g.gate + (int64_t)(m % g.gate_rows) * g.ld_gate + n : nullptr;
    if (g.gate && g.gate_per_row) {
      const float f = g.gate[m % g.gate_rows];
#pragma unroll
      for (int e = 0; e < 8; ++e) p.gate[e] = f;
    }
    if constexpr (VEC) {
      if (gp) Elem<float>::load8(gp, p.gate);
      if (g.res_f32) {
        p.r0 = *reinterpret_cast<const u32x4*>(g.res_f32 + roff);
        p.r1 = *reinterpret_cast<const u32x4*>(g.res_f32 + roff + 4);
      } else if (g.res_bf16) {
        p.r0 = *reinterpret_cast<const u32x4*>(g.res_bf16 + roff);
      }
    } else {
      for (int e = 0; e < min(8, g.N - n); ++e) {
        if (gp) p.gate[e] = gp[e];
        if (g.res_f32) (e < 4 ? p.r0 : p.r1)[e & 3] = __float_as_uint(g.res_f32[roff + e]);
        else if (g.res_bf16) p.r0[e >> 1] |= (uint32_t)g.res_bf16[roff + e] << (16 * (e & 1));
      }
    }
  };

  f32x16 acc[MT][NT];
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = zero;

  uint32_t fo[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) fo[ks] = (uint32_t)(l31 * ROWB + (((2 * ks + hh) ^ ((l31 >> 1) & 7)) << 4));

#pragma unroll
  for (int p = 0; p < ST; ++p) issue(p, mine + p * SLAB);
  if constexpr (KIND == KIND_GATE_RES && EARLY)
#pragma unroll
    for (int k = 0; k < PRE; ++k) fetch(k, pre[k]);

  struct Frags { bf16x8 a[4][MT], b[4][NT]; };
  auto read_frags = [&](Frags& f, uint32_t bo) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int t = 0; t < MT; ++t) f.a[ks][t] = as_frag(*reinterpret_cast<const u32x4*>(smem + bo + (wm + t * 32) * ROWB + fo[ks]));
#pragma unroll
      for (int t = 0; t < NT; ++t) f.b[ks][t] = as_frag(*reinterpret_cast<const u32x4*>(smem + bo + (BM + wn + t * 32) * ROWB + fo[ks]));
    }
  };
  auto products = [&](const Frags& f) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int x = 0; x < MT; ++x)
#pragma unroll
        for (int y = 0; y < NT; ++y) acc[x][y] = mfma32(f.b[ks][y], f.a[ks][x], acc[x][y]);
  };
  // the waves that share slabs meet; a lone wave waits for its own LDS reads
  auto meet = [&]() {
    if constexpr (ALONE) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else lds_barrier();
  };
  // Step i: slab i + 1 has landed (for every wave that shares it), slab i's fragments are in registers, so its buffer
  // takes slab i + ST; the fragments of slab i + 1 are read while the products of slab i run.  A 32x32 accumulator is
  // one chain of dependent MFMAs, and nothing else should lengthen it.  (Groups of waves with a slab less than the
  // next take part in all steps: their last slab is zeros.)
  const int trips = (ns + WK - 1) / WK;
  Frags f0, f1;
  uint32_t cur = 0;  // byte offset of slab i's buffer
  auto step = [&](int i, const Frags& now, Frags& then) {
    const uint32_t nxt = cur + SLAB == ST * SLAB ? 0 : cur + SLAB;
    // (towards the end nothing younger than slab i + 1 may be in flight any more)
    if (ST > 2 && i + ST - 1 < trips) wait_loads_but<(ST - 2) * NLOAD>();
    else wait_loads_but<0>();
    meet();
    if (i + ST < trips) issue(i + ST, mine + cur);
    read_frags(then, mine + nxt);
    products(now);
    cur = nxt;
  };
  wait_loads_but<(ST - 1) * NLOAD>();
  meet();
  read_frags(f0, mine);
  int i = 0;
  for (; i + 1 < trips; i += 2) {
    step(i, f0, f1);
    step(i + 1, f1, f0);
  }
  if (i < trips) products(f0);

  if constexpr (KIND == KIND_GATE_RES && !EARLY)
#pragma unroll
    for (int k = 0; k < PRE; ++k) fetch(k, pre[k]);
  // partial tiles -> LDS, over the slab buffers: every wave must have finished its slabs (and the loads past their
  // end must have written their zeros)
  wait_loads_but<0>();
  float* sC = reinterpret_cast<float*>(smem);
  lds_barrier();
#pragma unroll
  for (int x = 0; x < MT; ++x)
#pragma unroll
    for (int y = 0; y < NT; ++y)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = {acc[x][y][4 * q], acc[x][y][4 * q + 1], acc[x][y][4 * q + 2], acc[x][y][4 * q + 3]};
        *reinterpret_cast<f32x4*>(sC + (grp * BM + wm + 32 * x + l31) * LDS_C + wn + 32 * y + 8 * q + 4 * hh) = v;
      }
  lds_barrier();
  auto gather8 = [&](int row, int c, float* v) {
    auto part = [&](int w, int at) { return *reinterpret_cast<const f32x4*>(sC + (w * BM + row) * LDS_C + at); };
    f32x4 lo = part(0, c), hi = part(0, c + 4);
    if constexpr (WK >= 2) { lo += part(1, c); hi += part(1, c + 4); }
    if constexpr (WK >= 4) { lo += part(2, c) + part(3, c); hi += part(2, c + 4) + part(3, c + 4); }
    if constexpr (WK == 8) {
      lo += (part(4, c) + part(5, c)) + (part(6, c) + part(7, c));
      hi += (part(4, c + 4) + part(5, c + 4)) + (part(6, c + 4) + part(7, c + 4));
    }
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  };
  using OutT = std::conditional_t<OUT_F32, float, bf16_t>;
  OutT* C = reinterpret_cast<OutT*>(g.C);
  auto put = [&](int64_t o, const float* v, int nv) {
    if constexpr (VEC) Elem<OutT>::store8(C + o, v);
    else
      for (int e = 0; e < nv; ++e) Elem<OutT>::store(C + o + e, v[e]);
  };

  if constexpr (KIND == KIND_SWIGLU) {
    static_assert(KIND != KIND_SWIGLU || BN >= 64, "");
    // weight rows are packed in blocks of 64: 32 "a" rows then the 32 matching "b" rows; N / 2 output columns
    constexpr int OPR = BN >= 64 ? BN / 16 : 1;  // chunks of 8 output columns per row
#pragma unroll
    for (int k = 0; k < (BM * OPR + NTHR - 1) / NTHR; ++k) {
      const int idx = tid + k * NTHR;
      const int row = idx / OPR, oc = (idx % OPR) * 8, m = m0 + row;
      if (idx >= BM * OPR || m >= g.M || n0 + 2 * oc >= g.N) continue;
      const int c = (oc >> 5) * 64 + (oc & 31);
      float a[8], b[8], o[8];
      gather8(row, c, a);
      gather8(row, BN >= 64 ? c + 32 : c, b);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = a[e] * sigmoidf_(a[e]) * b[e];
      put((int64_t)bz * g.sC + (int64_t)m * g.ldc + n0 / 2 + oc, o, 8);
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < NCH; ++k) {
    if (KIND == KIND_GATE_RES && k > 0 && k % PRE == 0)
#pragma unroll
      for (int j = 0; j < PRE; ++j) fetch(k + j, pre[j]);
    const int idx = tid + k * NTHR;
    const int row = idx / CPR, c = (idx % CPR) * 8;
    const int m = m0 + row, n = n0 + c;
    if (idx >= BM * CPR || m >= g.M || n >= g.N) continue;
    const int nv = min(8, g.N - n);  // valid columns of this chunk
    const Pre& p = pre[k % PRE];
    float v[8], bias[8];
    gather8(row, c, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) bias[e] = 0.f;
    if (gemm_col_uses_bias(g, n))  // seg_len % 8 == 0: a chunk never straddles segments
    {
      if constexpr (VEC) Elem<float>::load8(g.bias + n, bias);
      else
        for (int e = 0; e < nv; ++e) bias[e] = g.bias[n + e];
    }
    if (KIND == KIND_COLUMNS && g.epi == EPI_SEGMENTED) {
      const int op = (g.seg_ops >> (4 * (n / g.seg_len))) & 15;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (op == SEG_BIAS_SCALE) v[e] = (v[e] + bias[e]) * g.alpha;
        else if (op == SEG_SIGMOID) v[e] = sigmoidf_(v[e]);
      }
    } else if (KIND == KIND_GATE_RES) {
      float rs[8];
      if (g.res_f32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) rs[e] = __uint_as_float(e < 4 ? p.r0[e & 3] : p.r1[e & 3]);
      } else {
        unpack8(p.r0, rs);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (v[e] + bias[e]) * p.gate[e] + rs[e];
    } else {  // EPI_PLAIN
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[e] = (v[e] + bias[e]) * g.alpha;
        if (g.act_sigmoid) v[e] = sigmoidf_(v[e]);
      }
    }
    put(g.regroup32 ? ((((int64_t)(m >> 5) * (g.N >> 5) + (n >> 5)) * 32 + (m & 31)) * 32 + (n & 31))
                    : (int64_t)bz * g.sC + (int64_t)m * g.ldc + n, v, nv);
  }
}

template <int MT, int NT, int WM, int WN, int WK, int ST, int WPS, bool CLEAN = true, bool VEC = true>
int launch_tile(GemmArgs g, hipStream_t stream) {
  constexpr int BM = 32 * MT * WM, BN = 32 * NT * WN;
  constexpr int PER_CU = WPS * 4 / (WM * WN * WK);  // workgroups that a CU holds
  static_assert(PER_CU >= 1, "WPS is in waves per SIMD");
  const XcdWalk walk = xcd_walk((g.M + BM - 1) / BM, (g.N + BN - 1) / BN, g.batch, BM, BN, XCD_CUS * PER_CU);
  const int64_t blocks = walk.slots * 8;
  if (blocks > 0x3fffffff) return AF3_ERR_BAD_ARG;
  g.xcd_m = walk.rows;
  const dim3 grid((unsigned)blocks), block(64 * WM * WN * WK);
#define LAUNCH(KIND, OUT_F32) hipLaunchKernelGGL((gemm_nt_kernel<MT, NT, WM, WN, WK, ST, WPS, CLEAN, KIND, VEC, OUT_F32>), grid, block, 0, stream, g)
  if (g.epi == EPI_SWIGLU) {
    if constexpr (BN >= 64) LAUNCH(KIND_SWIGLU, false);
    else return AF3_ERR_BAD_ARG;
  } else if (g.epi == EPI_GATE_RES) {
    if (g.out_f32) LAUNCH(KIND_GATE_RES, true);
    else LAUNCH(KIND_GATE_RES, false);
  } else {
    if (g.out_f32) LAUNCH(KIND_COLUMNS, true);
    else LAUNCH(KIND_COLUMNS, false);
  }
#undef LAUNCH
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

}  // namespace

// Wide products whose tiles come out just below a whole number per CU (256 CUs), which is worth more than the tile's
// bytes per FLOP: one product's tiles all run at once, and a few tiles more than that cost another round.  Eight waves.
// T: 128x128 tiles; us, the tile that the rules of launch_gemm_nt give otherwise behind it.
//   128x128, one per CU, four slab buffers   200 < T <= 256 and K >= 512: 4600x768x768 11.2 (12.8), 1150x3072x768 11.0
//                                            (12.6), 9000x384x768 11.2 (12.7), 1150x3072x512 9.7 (9.9).  SwiGLU from 190:
//                                            1000x3072x768 9.6 (9.9), 1060 rows 9.7 (11.6), 1250 rows 10.0 (12.4).  With
//                                            gate and residual from K = 1024, 4600x768x1024 16.0 (17.6): at K = 768 it is
//                                            4600 rows 14.3 (15.3), but 4992 rows 15.6 (15.6) and 1280x3072 16.6 (16.0)
//   128x192, one per CU                      where that many hold the product: 1700x3072x768 17.6 (18.6), SwiGLU 12.5 (14.3),
//                                            1900 rows 13.0 (15.2); 7000x768x768 14.7 (15.6); 5400x768x1536 25.1 (30.5)
//   128x128, two per CU                      352 < T <= 512: 2300x3072x768 20.7 (26.4), SwiGLU 15.3 (19.9);
//                                            9000x768x1536 31.2 (47.0)
enum { MID_NONE = 0, MID_128_ONE, MID_192, MID_128_TWO };
static int mid_tile_choice(const GemmArgs& g) {
  if (g.batch != 1 || (g.K % KS) || g.M <= 128 || g.N <= 128) return MID_NONE;
  const int64_t rows = (g.M + 127) / 128, t128 = rows * ((g.N + 127) / 128), t192 = rows * ((g.N + 191) / 192);
  const bool swiglu = g.epi == EPI_SWIGLU, gated = g.epi == EPI_GATE_RES;
  if (g.K >= 512 && t128 > (swiglu ? 190 : 200) && t128 <= 256 && (!gated || g.K >= 1024)) return MID_128_ONE;
  if (g.K >= 512 && g.N >= 768 && t128 > 256 && t192 <= 256) return MID_192;
  return t128 > 352 && t128 <= 512 ? MID_128_TWO : MID_NONE;
}

// Products of at least 120 tiles of 256x256 go to the large-tile kernel where one of its epilogues fits: a
// 128x128 tile of the kernel above needs twice the fragment reads per MFMA and is bound by them from there on
// (3840x3072x768: 34 us against 26).
int gemm_big_tile_choice(const GemmArgs& g) {
  constexpr int64_t BIG_TILE_MIN_TILES = 120;
  const int64_t tiles = (int64_t)((g.M + 255) / 256) * ((g.N + 255) / 256) * g.batch;
  if (g.small_tiles || mid_tile_choice(g) != MID_NONE) return -1;
  return g.M > 128 && g.N > 128 && tiles >= BIG_TILE_MIN_TILES ? big_tile_mode(g) : -1;
}

int launch_gemm_nt(const GemmArgs& g_in, hipStream_t stream) {
  GemmArgs g = g_in;
  if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.batch <= 0) return AF3_ERR_BAD_ARG;
  {
    const int big = gemm_big_tile_choice(g);
    if (big >= 0) return launch_big_tile(g, big, stream);
  }
  if ((g.K & 7) || (g.lda & 7) || (g.ldb & 7) || (g.sA & 7) || (g.sB & 7)) return AF3_ERR_BAD_ARG;
  if (((uintptr_t)g.A & 15) || ((uintptr_t)g.B & 15)) return AF3_ERR_BAD_ARG;
  if (g.K > g.lda || g.K > g.ldb) return AF3_ERR_BAD_ARG;
  if (g.lda >= (1ll << 22) || g.ldb >= (1ll << 22)) return AF3_ERR_BAD_ARG;  // 31-bit byte offsets inside a tile
  if (g.epi == EPI_SWIGLU && ((g.N & 63) || g.out_f32)) return AF3_ERR_BAD_ARG;
  if (g.epi == EPI_SEGMENTED && (g.seg_len <= 0 || (g.seg_len & 7))) return AF3_ERR_BAD_ARG;
  if (g.gate && g.gate_rows <= 0) return AF3_ERR_BAD_ARG;
  if (g.bias) {
    int64_t first, last;
    gemm_bias_span(g, false, &first, &last);
    if (first < 0 || last > g.bias_len) return AF3_ERR_BAD_ARG;
  }
  if (g.regroup32 && (g.epi != EPI_PLAIN || g.batch != 1 || (g.M & 31) || (g.N & 31))) return AF3_ERR_BAD_ARG;
  // 16-byte stores and loads need aligned rows and whole chunks of 8 columns (a plain bf16 result may have the rest
  // of its last chunk in row padding, which nobody reads)
  const int esz = g.out_f32 ? 4 : 2;
  auto al = [](const void* p, int64_t bytes0, int64_t bytes1) { return !p || ((uintptr_t)p % 16 == 0 && bytes0 % 16 == 0 && bytes1 % 16 == 0); };
  const bool whole = (g.N & 7) == 0;
  const bool padded = g.epi == EPI_PLAIN && !g.bias && !g.out_f32 && g.ldc >= ((g.N + 7) & ~7);
  const bool vec = (whole || padded) && al(g.C, g.ldc * esz, g.sC * esz) && al(g.bias, 0, 0) &&
                   (g.gate_per_row || al(g.gate, g.ld_gate * 4, 0)) && al(g.res_f32, g.ld_res * 4, g.sRes * 4) &&
                   al(g.res_bf16, g.ld_res * 2, g.sRes * 2);

  // The tile, by the number T of 64x64 tiles, on 256 CUs.  The lines up to 512 lie where a CU gets its second and third
  // tile; each with both sides at the line, us.  (Measured over M = 64 ... 92160, N = 128 ... 73728, K = 64 ... 1536.)
  //   T <= 128   32x32, the 64x64 tiles would leave half of the CUs without one (500x768x768 6.2, 64x64 6.7); with split_k
  //              the K range goes to four waves, or eight where it is long.  (SwiGLU pairs 32-column blocks: 64 columns or
  //              more)
  //   T <= 384   with split_k: 64x64, K split two ways (eight waves per tile); long ones are faster unsplit
  //   T <= 256   64x64 with four slab buffers, a workgroup to a CU
  //   T <= 512   64x64 with three, two to a CU: 2555x768x768 gated 9.8, with two buffers 10.2; K = 1536 14.5, 16.1; past
  //              the line 2811x768x768 11.9, 10.9; K = 1536 18.5, 16.8.  A SwiGLU of K >= 384 whose 128x64 tiles are at
  //              most one to a CU, but not many fewer: 500x3072x768 7.4, 64x64 7.7; 635 rows 7.5, 8.0; 571x3072x1536 11.1,
  //              11.8; past the line 699x3072x768 9.5, 9.2 (two buffers), 763x3072x384 7.2, 6.5; K = 128 6400x256 4.0, 4.0
  //   T <= 1000  64x64 with two, four to a CU
  //   T <= 2600  64x128, else 128x128: bytes per FLOP count once every CU has several tiles (and never wider than N)
  const int64_t T = (int64_t)((g.M + 63) / 64) * ((g.N + 63) / 64) * g.batch;
  const bool wide = g.epi == EPI_SWIGLU;
  if (!vec) return launch_tile<1, 1, 2, 2, 1, 2, 4, false, false>(g, stream);
  if (wide_product_applies(g)) return launch_wide_product(g, stream);  // (K = 384, many fp32 results)
  if (g.K % KS) return launch_tile<1, 1, 2, 2, 1, 2, 4, false>(g, stream);
  if (g.split_k && g.K > 256) {
    if (T <= 128 && !wide) return g.K >= 1024 ? launch_tile<1, 1, 1, 1, 8, 2, 2>(g, stream) : launch_tile<1, 1, 1, 1, 4, 2, 2>(g, stream);
    if (T <= 384 && g.K < 1024) return launch_tile<1, 1, 2, 2, 2, 2, 4>(g, stream);
  }
  switch (mid_tile_choice(g)) {
    case MID_128_ONE: return launch_tile<1, 2, 4, 2, 1, 4, 2>(g, stream);
    case MID_192: return launch_tile<1, 3, 4, 2, 1, 3, 2>(g, stream);
    case MID_128_TWO: return launch_tile<1, 2, 4, 2, 1, 2, 4>(g, stream);
  }
  if (T <= 128 && !wide) return launch_tile<1, 1, 1, 1, 1, 4, 1>(g, stream);
  if (T <= 256) return launch_tile<1, 1, 2, 2, 1, 4, 2>(g, stream);
  const int64_t T128x64 = (int64_t)((g.M + 127) / 128) * ((g.N + 63) / 64) * g.batch;
  if (wide && T > 352 && T128x64 <= 256 && g.K >= 384) return launch_tile<2, 1, 2, 2, 1, 3, 2>(g, stream);
  if (T <= 512) return launch_tile<1, 1, 2, 2, 1, 3, 3>(g, stream);
  if (T <= 1000 || g.N <= 64) return launch_tile<1, 1, 2, 2, 1, 2, 4>(g, stream);
  if (T <= 2600 || g.N <= 128) return launch_tile<1, 2, 2, 2, 1, 2, 3>(g, stream);
  return launch_tile<2, 2, 2, 2, 1, 2, 2>(g, stream);
}
