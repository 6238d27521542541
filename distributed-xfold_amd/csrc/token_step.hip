// The token transformer's adaptive LayerNorm and the product behind it (queries, keys, values and gate; or the SwiGLU
// transition's first layer) in one kernel, for rows of 768 channels on a bf16 stream.
//
// At a few hundred rows the two are launches of 5 and 8 to 10 us, of which the norm is a trip to memory and two reductions, and
// the product waits for the norm's last row before its first.  Here a workgroup keeps up to 32 normalised rows in LDS (48 KB)
// and multiplies them with 256 rows of the weights; its eight waves own 32 of those each and stream their fragments (frags of
// af3_diffusion_block) from L2 into registers, the first ones on their way while the rows are normalised.  Every row is
// normalised by each of the twelve workgroups that need it: what that costs is the conditioning, 6 KB of fp32 a token, so a
// tile holds all samples of its tokens, which share it.  With the weights' rows in the order of the accumulators a lane ends
// with runs of eight result columns (or with both factors of eight hidden units) and stores them as they are.
// Values are rounded where the separate kernels store them and every sum has their order: the same bits.
//
// What bounds it: 0.45 MB of weights, rows and conditioning through the CU's vector memory path (64 bytes a cycle: 3.3 us at
// 2.1 GHz) and the norms' vector instructions, which overlap but for their ends.  100 tokens of 5 samples: 9.2 us either, and
// of a wave's 15000 cycles 3700 until the rows are there, 5000 norms, 3000 product, 1000 result, the rest at the barrier between.
// (The norms with eight channels to a lane in two chunks, a quarter of the second without any, and the division by 768 as it
// stands: 9.5 and 9.7 us.)  An evaluation of the diffusion head, us, norm and rows_product_kernel / this: 1 x 100 tokens 1143 / 1024,
// 1 x 256 1286 / 1209, 3 x 120 1220 / 1141, 4 x 128 1265 / 1194, 5 x 60 1158 / 1033, 5 x 100 1267 / 1167, 5 x 120 1302 / 1251.  At one
// workgroup to a CU the twelvefold norms cost what they save (3 x 200 1350 / 1363); past it, more.
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int K = TOKEN_STEP_CHANNELS, ROWS = 32, NW = 8, BN = 32 * NW;
constexpr int NKS = K / 16, PIECES = NKS / 8, NB = 5;  // k-steps; pieces of eight; pieces in flight
constexpr int PANEL = K / 64 * ROWS * 128;             // slabs of 64 channels, [slab][row][128 bytes]
constexpr int WARM_LINES = 4;  // per thread
constexpr int CUS = 256, WARM_CUS = 24;  // of which some for the workgroups that warm

// TPW: tokens of a wave, SMAX: samples at most
template <int TPW, int SMAX, bool SWIGLU>
__global__ __launch_bounds__(64 * NW, 2) void norm_product_kernel(NormProductArgs a) {
  args_at_once<NormProductArgs>();
  __shared__ __attribute__((aligned(1024))) char sP[PANEL];
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (blockIdx.x >= a.work_blocks) {
    // workgroups on the idle CUs bring what the next kernels read into the last-level cache (see ln_rows_kernel)
    bring_lines<WARM_LINES>(a.warm, a.warm_lines, (blockIdx.x - a.work_blocks) * (WARM_LINES * 64u * NW) + tid, 64u * NW);
    return;
  }
  // A range of the weights' rows for every XCD, each with the tiles of all rows one after the other
  const int idx = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= a.per_xcd || idx >= a.total) return;
  const int tn = a.tiles == 1 ? idx : (int)__umulhi((uint32_t)idx, a.magic_tiles), tt_n = a.tile_tokens;  // idx / tiles
  const int t0 = (idx - tn * a.tiles) * tt_n, n0 = tn * BN;

  // ---- the rows this wave normalises: all samples of tokens wave, wave + 8, .. of the tile; six tokens of five samples: the
  // last two tokens by two waves each, so that every SIMD has seven or eight rows ----
  // (What is too many is a copy of the last and is not kept: the rows' chains run beside each other in one block, or two.)
  const bool split = SMAX == 5 && tt_n == 6 && wave >= 4;
  const int tt_0 = split ? 4 + ((wave - 4) >> 1) : wave, s_0 = split && (wave & 1) ? 3 : 0;
  const int count = split ? 3 - (wave & 1) : a.samples;
  auto each_row = [&](auto f) {
#pragma unroll
    for (int k = 0; k < TPW; ++k)
#pragma unroll
      for (int s = 0; s < min(SMAX, 3); ++s) f(k, s);
    if constexpr (SMAX > 3) {
      if (count > 3) {
        f(0, 3);
        f(0, 4);
      }
    }
  };
  u32x4 raw[TPW][SMAX];
  u32x2 raw4[TPW][SMAX];
  f32x4 sc[TPW][3], sh[TPW][3];
  const int c0 = lane * 8, c1 = 512 + lane * 4;
#pragma unroll
  for (int k = 0; k < TPW; ++k) {
    const int token = min(t0 + min(tt_0 + NW * k, tt_n - 1), a.tokens - 1);
    const bf16_t* x = a.x + (s_0 * a.tokens + token) * K;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      raw[k][s] = *reinterpret_cast<const u32x4*>(x + c0);
      raw4[k][s] = *reinterpret_cast<const u32x2*>(x + c1);
      x += s + 1 < count ? a.tokens * K : 0;
    }
    const float* p = a.scale + (int64_t)token * a.ld_cond;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int c = i < 2 ? c0 + 4 * i : c1;
      sc[k][i] = *reinterpret_cast<const f32x4*>(p + c);
      sh[k][i] = *reinterpret_cast<const f32x4*>(p + K + c);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 w[NB][8];
  auto fetch = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (n < PIECES) load_frags<8>(a.w, n0 / 32 + wave, NKS, 8 * n, lane, w[n % NB]);
    __builtin_amdgcn_sched_barrier(0);
  };
#define PIECE(n) std::integral_constant<int, (n)>{}
  // A wave cannot go on before the CU's vector memory path has taken its loads, 16 cycles each: the rows first, and when they
  // are there one piece in front of each part of the normalisation, as far as there are registers.
  constexpr int AHEAD = TPW == 1 ? 3 : 2;
  const bool busy = tt_0 < tt_n;  // (waves without a token)
  if (busy)
#pragma unroll
    for (int k = 0; k < TPW; ++k)
#pragma unroll
      for (int s = 0; s < SMAX; ++s) asm volatile("" ::"v"(raw[k][s].x), "v"(raw4[k][s].x));
  fetch(PIECE(0));

  // adaptive LayerNorm, ln_rows_768_kernel's sums
  float v[TPW][SMAX][12], rstd[TPW][SMAX];
  if (busy)
    each_row([&](int k, int s) {
      float* x = v[k][s];
      float sum = 0.f;
      unpack12(raw[k][s], raw4[k][s], x);
#pragma unroll
      for (int e = 0; e < 12; ++e) sum += x[e];
      const float mean = over_768(wave_sum(sum));
#pragma unroll
      for (int e = 0; e < 12; ++e) x[e] -= mean;
    });
  fetch(PIECE(1));
  if (busy)
    each_row([&](int k, int s) {
      const float* d = v[k][s];
      rstd[k][s] = rsqrtf(over_768(wave_sum(add_squares4(d + 8, add_squares8(d, 0.f, true)))) + LN_EPS);
    });
  if constexpr (AHEAD > 2) fetch(PIECE(2));
  if (busy) {
    float gain[TPW][12];
#pragma unroll
    for (int k = 0; k < TPW; ++k)
#pragma unroll
      for (int e = 0; e < 12; ++e) gain[k][e] = sigmoidf_(sc[k][e >> 2][e & 3]);
    // 16 bytes of slab lane / 8 and 8 of slab 8 + lane / 16; chunk c of a slab's row lies at position c ^ (row / 2 % 8)
    char *const at0 = sP + (lane >> 3) * (ROWS * 128), *const at1 = sP + (8 + (lane >> 4)) * (ROWS * 128) + (lane & 1) * 8;
    each_row([&](int k, int s) {
      const int tt = tt_0 + NW * k, row = tt * a.samples + s_0 + s, x = (row >> 1) & 7;
      const bool keep = tt < tt_n && s < count;
      float o[12];
#pragma unroll
      for (int e = 0; e < 12; ++e) {
        const float t = v[k][s][e] * rstd[k][s];
        o[e] = gain[k][e] * t + sh[k][e >> 2][e & 3];
      }
      if (keep) {
        *reinterpret_cast<u32x4*>(at0 + row * 128 + (((lane & 7) ^ x) << 4)) = pack8(o);
        *reinterpret_cast<u32x2*>(at1 + row * 128 + ((((lane >> 1) & 7) ^ x) << 4)) = u32x2{pack2bf(o[8], o[9]), pack2bf(o[10], o[11])};
      }
    });
  }
  if constexpr (AHEAD < 3) fetch(PIECE(2));
  fetch(PIECE(3));
  fetch(PIECE(4));
  // a lane's registers 8 u .. are result columns 32 wave + 16 u + 8 hh .. of row j (with swiglu 8 u: first and second factor of
  // hidden units 16 wave + 8 hh ..)
  const int col = n0 + 32 * wave + 8 * hh;
  const bool queries = !SWIGLU && tn < K / BN;
  float bias[16];
  if constexpr (!SWIGLU) {
#pragma unroll
    for (int u = 0; u < 2; ++u) load_param8(queries && a.q_bias ? a.q_bias + col + 16 * u : nullptr, 0.f, bias + 8 * u);
  }
  lds_barrier();

  // ---- the product, a lane owns a row ----
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  bf16x8 xf[2][8];
  auto rows = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < PIECES)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int ks = 8 * n + i, c = 2 * (ks & 3) + hh;
        xf[n & 1][i] = as_frag(*reinterpret_cast<const u32x4*>(sP + (ks >> 2) * (ROWS * 128) + j * 128 + ((c ^ ((j >> 1) & 7)) << 4)));
      }
  };
  auto piece = [&](auto n_c) {  // (the next one's rows are read meanwhile)
    constexpr int n = decltype(n_c)::value;
    rows(PIECE(n + 1));
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = mfma32(w[n % NB][i], xf[n & 1][i], acc);
    fetch(PIECE(n + NB));
  };
  rows(PIECE(0));
  piece(PIECE(0));
  piece(PIECE(1));
  piece(PIECE(2));
  piece(PIECE(3));
  piece(PIECE(4));
  piece(PIECE(5));
  static_assert(PIECES == 6, "all of them");
#undef PIECE

  // ---- column operations, 64 bytes of a row to a wave (SwiGLU 32) ----
  const int tt = (j * a.magic_samples) >> 16, token = t0 + tt;  // j / samples
  if (tt >= tt_n || token >= a.tokens) return;
  bf16_t* const out = a.out + ((int64_t)(j - tt * a.samples) * a.tokens + token) * a.ldc;
  float o[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) o[r] = acc[r];
  if constexpr (SWIGLU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = o[e] * sigmoidf_(o[e]) * o[8 + e];
    *reinterpret_cast<u32x4*>(out + n0 / 2 + 16 * wave + 8 * hh) = pack8(o);
  } else {
    if (queries) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = (o[r] + bias[r]) * a.q_scale;
    } else if (tn >= 3 * (K / BN)) {  // the gate
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = sigmoidf_(o[r]);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4*>(out + col + 16 * u) = pack8(o + 8 * u);
  }
}

// The products that lead back into the stream: act = (y w^T) gate + act, 768 result columns, K = 128 KP.  A workgroup takes 32
// rows and 32 columns per wave; the rows go to LDS as a panel, all of them at once, the weights' fragments straight to registers,
// gate and stream asked for behind them: one trip to memory, a chain of 48 or 96 matrix instructions (some 36 cycles each), and
// the result back from the registers.  The general kernel's 32x32 tile, a slab at a time, takes 7.5 us on average of the two at
// 500 rows.  Two waves share a panel where that keeps to one workgroup a CU, one has it alone at up to 320 rows.
// A token transformer of 24 blocks with the norms in its other products, us, without this / with it: 5 x 40 tokens 981 / 867,
// 5 x 100 1132 / 1044, 5 x 126 1335 / 1185, 1 x 100 1024 / 905, 3 x 100 1080 / 961, 2 x 300 1423 / 1330.
template <int KP, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 1) void gated_product_kernel(GatedProductArgs a) {
  args_at_once<GatedProductArgs>();
  constexpr int KK = 128 * KP, SLABS = KK / 64, RING = 5;
  __shared__ __attribute__((aligned(1024))) char sP[SLABS * ROWS * 128];
  const int lane = threadIdx.x & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int idx = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= a.per_xcd || idx >= a.total) return;
  const int tn = a.tiles == 1 ? idx : (int)__umulhi((uint32_t)idx, a.magic_tiles);
  const int m0 = (idx - tn * a.tiles) * ROWS, n0 = (tn * WAVES + wave) * 32;

  // the panel, slab by slab; a wave brings every WAVES-th group of eight rows
  const bf16_t* const y = a.y + (int64_t)m0 * KK;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)sP;
  uint32_t off[4 / WAVES];
#pragma unroll
  for (int i = 0; i < 4 / WAVES; ++i) {
    const int row = 8 * (WAVES * i + wave) + (lane >> 3);
    off[i] = (uint32_t)(min(row, a.rows - 1 - m0) * KK + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2u;
  }
#pragma unroll
  for (int s = 0; s < SLABS; ++s)
#pragma unroll
    for (int i = 0; i < 4 / WAVES; ++i)
      load_to_lds(y + 64 * s, off[i], __builtin_amdgcn_readfirstlane(lds0 + s * (ROWS * 128) + (WAVES * i + wave) * 1024));
  bf16x8 w[RING][8];
  auto fetch = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (n < KP) load_frags<8>(a.w, tn * WAVES + wave, KK / 16, 8 * n, lane, w[n % RING]);
    __builtin_amdgcn_sched_barrier(0);
  };
#define PIECE(n) std::integral_constant<int, (n)>{}
  fetch(PIECE(0));
  fetch(PIECE(1));
  fetch(PIECE(2));
  // a lane's registers 8 u .. are columns 16 u + 8 hh .. of row j
  const int row = min(m0 + j, a.rows - 1), col = n0 + 8 * hh;
  const int cond = row - (a.cond_rows == 1 ? row : (int)__umulhi((uint32_t)row, a.magic_cond)) * a.cond_rows;
  bf16_t* const act = a.act + (int64_t)row * K + col;
  const float* const gp = a.gate + (int64_t)cond * a.ld_gate + col;
  f32x4 gate[2][2];
  u32x4 res[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    gate[u][0] = *reinterpret_cast<const f32x4*>(gp + 16 * u);
    gate[u][1] = *reinterpret_cast<const f32x4*>(gp + 16 * u + 4);
    res[u] = *reinterpret_cast<const u32x4*>(act + 16 * u);
  }
  fetch(PIECE(3));
  fetch(PIECE(4));
  // The fragments asked for behind the panel may be on their way still.  Loads issued behind it that are not counted only make the
  // wait longer, ones counted and not issued would end it too soon: so the fragments alone, which sched_barrier keeps where they
  // are, and not gate and stream (the first matrix instruction waits for more than the six loads that this costs).
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * RING) : "memory");
  lds_barrier();

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  bf16x8 xf[2][8];
  auto rows = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < KP)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int ks = 8 * n + i, c = 2 * (ks & 3) + hh;
        xf[n & 1][i] = as_frag(*reinterpret_cast<const u32x4*>(sP + (ks >> 2) * (ROWS * 128) + j * 128 + ((c ^ ((j >> 1) & 7)) << 4)));
      }
  };
  auto piece = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < KP) {
      rows(PIECE(n + 1));
#pragma unroll
      for (int i = 0; i < 8; ++i) acc = mfma32(w[n % RING][i], xf[n & 1][i], acc);
      fetch(PIECE(n + RING));
    }
  };
  rows(PIECE(0));
  piece(PIECE(0)); piece(PIECE(1)); piece(PIECE(2)); piece(PIECE(3)); piece(PIECE(4)); piece(PIECE(5));
  piece(PIECE(6)); piece(PIECE(7)); piece(PIECE(8)); piece(PIECE(9)); piece(PIECE(10)); piece(PIECE(11));
  static_assert(KP <= 12, "all of them");
#undef PIECE
  if (m0 + j >= a.rows) return;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    float o[8], x[8];
    unpack8(res[u], x);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (acc[8 * u + e] + 0.f) * gate[u][e >> 2][e & 3] + x[e];
    *reinterpret_cast<u32x4*>(act + 16 * u) = pack8(o);
  }
}

// The same products over more rows: x w^T with the weights' fragments straight from memory to registers and the rows through LDS.
// A workgroup takes 32 RB rows (two to four blocks: rows_product_blocks) x 128 columns, a wave all rows of 32 columns; slabs of 64
// channels of the rows go straight into a ring of LDS buffers that the four waves share, with one barrier a slab; a wave's
// fragments are RP_RING slabs ahead; the result goes out through LDS, in whole lines.  Cycles of a workgroup of 96 x 128, all of 3840
// rows: first slab there 3700, loop 8400 (4600 of it the matrix unit's), result 2700.  What bounds it is the CU's vector memory path,
// 16 KB of weights and 4 RB KB of rows a slab, and in large tiles that the chip's results leave all at once.  Results stored from the
// accumulators, 32 bytes of a row at a time, were slower where there is a gate and a stream to read the same way: 768 columns at
// 3840 rows 11.7 / 15.7 us (K = 768 / 1536) against 8.6 / 14.1, at 1920 (two blocks) 6.6 / 9.8 against 6.0 / 8.9.  Two column blocks a
// wave (192 x 256 at 3840 rows, queries to gate 23.1 us): the chip's only round ends in 8500 cycles of results.
enum { ROWS_QKVG, ROWS_SWIGLU, ROWS_GATED };
constexpr int RP_BN = 128, RP_BUFFERS = 4, RP_RING = 4;
static_assert(RP_RING == RP_BUFFERS);  // (rows_product_younger counts on it)
// loads of a wave issued behind its own for slab s of the rows, when it waits for these (in step s - 1 of the loop): statements and
// loads that sched_barrier keeps in this order; any others issued between them only make the wait longer
constexpr int rows_product_younger(int s, int slabs, int rows) {
  int n = 0;
  bool behind = false;
  auto issue = [&](int slab) {  // rows, then fragments: in front of the loop, and in each of its steps before the wait
    if (behind && slab < slabs) n += rows;
    if (slab == s) behind = true;
    if (behind && slab < slabs) n += 4;
  };
  for (int i = 0; i < RP_BUFFERS; ++i) issue(i);
  for (int i = 0; i + 1 < s; ++i) issue(i + RP_BUFFERS);
  return n < 63 ? n : 63;
}
template <typename F, int... I>
__device__ __forceinline__ void each(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <int SLABS, int KIND, int RB>
__global__ __launch_bounds__(256, RB == 2 ? 3 : 2) void rows_product_kernel(RowsProductArgs a) {
  args_at_once<RowsProductArgs>();
  constexpr int KK = 64 * SLABS, BM = 32 * RB, BN = RP_BN, BUF = BM * 128;
  __shared__ __attribute__((aligned(1024))) char sA[RP_BUFFERS * BUF];
  const int lane = threadIdx.x & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // XCD (i, k) of a grid of xcd_m x 8 / xcd_m takes a rectangle of m_chunk x n_chunk tiles, row tiles fastest
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int sn = a.m_chunk == 1 ? slot : (int)__umulhi((uint32_t)slot, a.magic_chunk);
  const int tm = (xcd & (a.xcd_m - 1)) * a.m_chunk + slot - sn * a.m_chunk, tn = (xcd >> a.xcd_shift) * a.n_chunk + sn;
  if (tm * BM >= a.rows || tn * BN >= a.N) return;
  const int m0 = tm * BM, blk = tn * 4 + wave;

  // a wave brings RB of a slab's 4 RB groups of eight rows
  const bf16_t* const x = a.x + (int64_t)m0 * KK;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)sA + 1024 * RB * wave;
  uint32_t off[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int row = 8 * (RB * wave + i) + (lane >> 3);
    off[i] = (uint32_t)(min(row, a.rows - 1 - m0) * KK + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2u;
  }
  auto bring = [&](auto s_c) {
    constexpr int s = decltype(s_c)::value;
    if constexpr (s < SLABS) {
#pragma unroll
      for (int i = 0; i < RB; ++i)
        load_to_lds(x + 64 * s, off[i], __builtin_amdgcn_readfirstlane(lds0 + (s % RP_BUFFERS) * BUF + 1024 * i));
    }
  };
  bf16x8 w[RP_RING][4];
  auto fetch = [&](auto s_c) {
    constexpr int s = decltype(s_c)::value;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (s < SLABS) load_frags<4>(a.w, blk, KK / 16, 4 * s, lane, w[s % RP_RING]);
    __builtin_amdgcn_sched_barrier(0);
  };
#define SLAB(n) std::integral_constant<int, (n)>{}
  each([&](auto s_c) {
    constexpr int s = decltype(s_c)::value;
    if constexpr (s < RP_BUFFERS) bring(s_c);
    fetch(s_c);
  }, std::make_integer_sequence<int, RP_RING>{});

  f32x16 acc[RB];
#pragma unroll
  for (int t = 0; t < RB; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  bf16x8 xf[2][RB];
  auto rows = [&](auto s_c, int ks) {  // k-step ks of slab s
    constexpr int s = decltype(s_c)::value;
#pragma unroll
    for (int t = 0; t < RB; ++t)
      xf[ks & 1][t] = as_frag(*reinterpret_cast<const u32x4*>(sA + (s % RP_BUFFERS) * BUF + (32 * t + j) * 128 +
                                                              (((2 * ks + hh) ^ ((j >> 1) & 7)) << 4)));
  };
  auto landed = [&](auto s_c) {  // slab s is in LDS, for every wave
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(rows_product_younger(decltype(s_c)::value, SLABS, RB)) : "memory");
    lds_barrier();
  };
  // gated: gate and stream for eight columns of rows tid / 16, ..
  const int tid = threadIdx.x;
  constexpr int EACH = KIND == ROWS_GATED ? BM / 16 : 1;
  float g[EACH][8];
  u32x4 res[EACH];
  auto load_gates = [&]() {
    if constexpr (KIND == ROWS_GATED) {
#pragma unroll
      for (int e = 0; e < EACH; ++e) {
        const int row = min(m0 + (tid >> 4) + 16 * e, a.rows - 1), col = tn * BN + (tid & 15) * 8;
        const int cond = row - (a.cond_rows == 1 ? row : (int)__umulhi((uint32_t)row, a.magic_cond)) * a.cond_rows;
        Elem<float>::load8(a.gate + (int64_t)cond * a.ld_gate + col, g[e]);
        res[e] = *reinterpret_cast<const u32x4*>(a.out + (int64_t)row * a.ldc + col);
      }
    }
  };
  landed(SLAB(0));
  rows(SLAB(0), 0);
  each([&](auto i_c) {
    constexpr int i = decltype(i_c)::value;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) {
        rows(i_c, ks + 1);
      } else if constexpr (i + 1 < SLABS) {
        landed(SLAB(i + 1));  // (and every wave has slab i's fragments: its buffer is free)
        bring(SLAB(i + RP_BUFFERS));
        rows(SLAB(i + 1), 0);
        if constexpr (i + 2 == SLABS) load_gates();  // (no counted wait behind it)
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < RB; ++t) acc[t] = mfma32(w[i % RP_RING][ks], xf[ks & 1][t], acc[t]);
    }
    fetch(SLAB(i + RP_RING));
  }, std::make_integer_sequence<int, SLABS>{});
#undef SLAB

  // A lane's registers 8 u .. are columns 32 c + 16 u + 8 hh .. of row 32 t + j for column block c of the wave (SwiGLU: both factors of
  // hidden units 16 c + 8 hh ..): 32 bytes of a row to a store.  So the tile goes through LDS, where the slabs were, and out in
  // whole lines; pieces of 16 bytes at piece ^ (row % 16).
  lds_barrier();
  if constexpr (KIND == ROWS_GATED) {
#pragma unroll
    for (int t = 0; t < RB; ++t)
#pragma unroll
      for (int p = 0; p < 4; ++p)
        *reinterpret_cast<f32x4*>(sA + (32 * t + j) * 512 + (((8 * wave + 4 * (p >> 1) + 2 * hh + (p & 1)) ^ (j & 15)) << 4)) =
            f32x4{acc[t][4 * p], acc[t][4 * p + 1], acc[t][4 * p + 2], acc[t][4 * p + 3]};
    lds_barrier();
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
      const int r = (tid >> 4) + 16 * e, row = m0 + r;
      float o[8], x[8];
      unpack8(res[e], x);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(sA + r * 512 + (((2 * (tid & 15) + q) ^ (r & 15)) << 4));
#pragma unroll
        for (int k = 0; k < 4; ++k) o[4 * q + k] = (v[k] + 0.f) * g[e][4 * q + k] + x[4 * q + k];
      }
      if (row < a.rows) *reinterpret_cast<u32x4*>(a.out + (int64_t)row * a.ldc + tn * BN + (tid & 15) * 8) = pack8(o);
    }
  } else {
    constexpr int COLS = KIND == ROWS_SWIGLU ? BN / 2 : BN, PIECES = COLS / 8;
    const int seg = tn / (K / BN);
    float bias[16];
    if constexpr (KIND == ROWS_QKVG)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        load_param8(seg == 0 && a.q_bias ? a.q_bias + 32 * blk + 16 * u + 8 * hh : nullptr, 0.f, bias + 8 * u);
#pragma unroll
    for (int t = 0; t < RB; ++t) {
      char* const at = sA + (32 * t + j) * (2 * COLS);
      float o[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = acc[t][r];
      if constexpr (KIND == ROWS_SWIGLU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = o[e] * sigmoidf_(o[e]) * o[8 + e];
        *reinterpret_cast<u32x4*>(at + (((2 * wave + hh) ^ (j & (PIECES - 1))) << 4)) = pack8(o);
      } else {
        if (seg == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) o[r] = (o[r] + bias[r]) * a.q_scale;
        } else if (seg == 3) {
#pragma unroll
          for (int r = 0; r < 16; ++r) o[r] = sigmoidf_(o[r]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4*>(at + (((4 * wave + 2 * u + hh) ^ (j & (PIECES - 1))) << 4)) = pack8(o + 8 * u);
      }
    }
    lds_barrier();
#pragma unroll
    for (int e = 0; e < BM * PIECES / 256; ++e) {
      const int i = tid + 256 * e, r = i / PIECES, p = i % PIECES;
      const u32x4 v = *reinterpret_cast<const u32x4*>(sA + r * (2 * COLS) + ((p ^ (r & (PIECES - 1))) << 4));
      if (m0 + r < a.rows) *reinterpret_cast<u32x4*>(a.out + (int64_t)(m0 + r) * a.ldc + tn * COLS + p * 8) = v;
    }
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// Tokens of a tile, by the number of samples.  One of fewer leaves rows of the matrix instruction empty, but its norms are done
// sooner: taken while every tile has a CU of its own (24 blocks, us: 1 x 100 tokens by 32 1174, by 8 1024; 3 x 152 by 8 1203, 3 x 160
// by 10 1284; 5 x 76 by 4 1110, 5 x 80 by 6 1097).  Five samples are the most: a wave keeps all rows of its token in registers
// while it normalises them (222 and 233 of 256 with five); six take norm and product in kernels of their own.
static int tile_tokens(const NormProductArgs& a) {
  static constexpr int sizes[5][2] = {{8, 16}, {8, 16}, {8, 10}, {4, 8}, {4, 6}};
  const int* const of = sizes[a.samples - 1];
  return (int64_t)((a.tokens - 1) / of[0] + 1) * (a.N / BN) <= CUS - WARM_CUS ? of[0] : of[1];
}

bool norm_product_applies(const NormProductArgs& a) {
  return a.x && a.w && a.out && a.scale && a.samples > 0 && a.samples <= 5 && a.tokens > 0 && a.N > 0 && a.N % BN == 0 &&
         (a.swiglu || a.N == 4 * K) && (int64_t)((a.tokens - 1) / tile_tokens(a) + 1) * (a.N / BN) <= CUS && a.ld_cond >= 2 * K &&
         a.ld_cond % 4 == 0 && a.ldc % 8 == 0 && al16(a.x) && al16(a.w) && al16(a.out) && al16(a.scale) && al16(a.q_bias);
}

int launch_norm_product(const NormProductArgs& args, hipStream_t s) {
  if (!norm_product_applies(args)) return AF3_ERR_BAD_ARG;
  NormProductArgs a = args;
  a.tile_tokens = tile_tokens(a);
  a.tiles = (a.tokens + a.tile_tokens - 1) / a.tile_tokens;
  a.total = a.tiles * (a.N / BN);
  a.per_xcd = (a.total + 7) / 8;
  a.work_blocks = 8u * a.per_xcd;
  a.magic_tiles = a.tiles == 1 ? 0u : 0xffffffffu / (uint32_t)a.tiles + 1u;  // idx / tiles = umulhi(idx, magic): idx tiles < 2^32
  a.magic_samples = 65536 / a.samples + 1;                                   // row / samples, row < 32
  // (no more workgroups that warm than there are CUs left: one that waits for a CU makes the kernel longer)
  const int64_t lines = (int64_t)a.warm_lines[0] + a.warm_lines[1] + a.warm_lines[2];
  const int64_t warm = (lines + 64 * NW * WARM_LINES - 1) / (64 * NW * WARM_LINES), idle = CUS - (int64_t)a.work_blocks;
  const dim3 grid(a.work_blocks + (unsigned)(warm < idle ? warm : idle > 0 ? idle : 0)), block(64 * NW);
#define LAUNCH(TPW, SMAX)                                                                           \
  do {                                                                                              \
    if (a.swiglu) hipLaunchKernelGGL((norm_product_kernel<TPW, SMAX, true>), grid, block, 0, s, a); \
    else hipLaunchKernelGGL((norm_product_kernel<TPW, SMAX, false>), grid, block, 0, s, a);         \
  } while (0)
  if (a.samples > 3) LAUNCH(1, 5);
  else if (a.samples > 1 && a.tile_tokens > 8) LAUNCH(2, 3);
  else if (a.samples > 1) LAUNCH(1, 3);
  else if (a.tile_tokens > 8) LAUNCH(2, 1);
  else LAUNCH(1, 1);
#undef LAUNCH
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

bool gated_product_applies(const GatedProductArgs& a) {
  return a.y && a.w && a.act && a.gate && a.rows > 0 && (a.K == 768 || a.K == 1536) && a.cond_rows > 0 && a.ld_gate >= K &&
         a.ld_gate % 4 == 0 && al16(a.y) && al16(a.w) && al16(a.act) && al16(a.gate) && (int64_t)((a.rows - 1) / ROWS + 1) * (K / 64) <= CUS;
}

int launch_gated_product(const GatedProductArgs& args, hipStream_t s) {
  if (!gated_product_applies(args)) return AF3_ERR_BAD_ARG;
  GatedProductArgs a = args;
  a.tiles = (a.rows + ROWS - 1) / ROWS;
  const int waves = a.tiles * (K / 32) <= CUS ? 1 : 2;
  a.total = a.tiles * (K / 32 / waves);
  a.per_xcd = (a.total + 7) / 8;
  a.magic_tiles = a.tiles == 1 ? 0u : 0xffffffffu / (uint32_t)a.tiles + 1u;
  a.magic_cond = a.cond_rows == 1 ? 0u : 0xffffffffu / (uint32_t)a.cond_rows + 1u;
  const dim3 grid(8u * a.per_xcd), block(64 * waves);
#define LAUNCH(KP)                                                                                  \
  do {                                                                                              \
    if (waves == 1) hipLaunchKernelGGL((gated_product_kernel<KP, 1>), grid, block, 0, s, a);        \
    else hipLaunchKernelGGL((gated_product_kernel<KP, 2>), grid, block, 0, s, a);                   \
  } while (0)
  if (a.K == 768) LAUNCH(6);
  else LAUNCH(12);
#undef LAUNCH
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

bool rows_product_applies(const RowsProductArgs& a) {
  return a.x && a.w && a.out && a.rows > 0 && a.rows < (1 << 20) && a.N > 0 && a.N % RP_BN == 0 && (a.K == 768 || a.K == 1536) &&
         a.ldc % 8 == 0 && al16(a.x) && al16(a.w) && al16(a.out) && al16(a.q_bias) &&
         (a.gate ? a.N == K && a.ldc == K && a.cond_rows > 0 && (int64_t)a.rows * a.cond_rows <= 0xffffffffll && a.ld_gate >= K && a.ld_gate % 4 == 0 && al16(a.gate)
                 : a.K == K && (a.swiglu || a.N == 4 * K));
}

// Row blocks of a workgroup's tile.  A CU's time goes by the tiles that it gets, one after the other or at once, and a tile's by its
// rows, less for a row the more there are, as they share the weights (us a tile, queries to gate: 3.25, 4.6 and 6.0): the blocks
// with which the CU that gets most is done first.  us at these rows, two / three / four blocks / af3_linear_forward's kernels:
//   queries to gate  700: 8.7 7.1 8.4 9.6   1280: 9.9 12.1 9.6 11.8   1920: 13.5 12.6 14.5 15.7  2560: 16.1 16.9 15.8 18.7
//                    3200: 20.0 20.5 20.3 -   3840: 22.8 21.8 22.5 -   5600: 33.3 30.1 31.1 -     7680: 44.7 40.3 39.7 -
//   SwiGLU           700: 7.7 6.4 7.6 8.9   1280: 9.2 10.8 8.7 9.9    1920: 12.3 11.6 13.3 13.2  2560: 15.3 14.8 14.5 16.9
//                    3840: 21.4 19.7 21.2 20.6  5000: 27.2 26.8 25.1 25.5  5600: 30.7 28.3 30.0 35.6  7680: 40.7 36.8 36.6 36.8
//   768 gated        700: 5.8 7.0 8.2 6.7   1920: 6.2 7.4 8.6 8.1     2560: 6.6 7.7 8.9 8.9      2730: 9.3 7.9 9.2 10.2
//                    3840: 10.2 8.5 9.8 12.1  4600: 10.6 15.6 11.7 15.5  5600: 15.5 13.9 17.1 18.1  7680: 16.5 16.2 17.7 20.0
//   1536 gated       700: 8.4 9.9 11.8 9.0  1920: 8.9 10.4 12.3 12.2  2560: 9.7 11.4 13.0 14.1   2730: 14.7 12.0 13.6 16.4
//                    3840: 16.2 14.6 15.6 19.1  4600: 17.0 21.0 17.1 20.1  5600: 24.3 20.7 25.5 25.1  7680: 26.3 24.1 26.2 28.0
static int rows_product_blocks(const RowsProductArgs& a) {
  static constexpr int weight[3] = {65, 90, 120};
  int best = 0, rb = 2;
  for (int i = 0; i < 3; ++i) {
    const int64_t tiles = (int64_t)((a.rows + 32 * (i + 2) - 1) / (32 * (i + 2))) * (a.N / RP_BN);
    const int64_t cost = (tiles + CUS - 1) / CUS * weight[i];
    if (i == 0 || cost < best) { best = (int)cost; rb = i + 2; }
  }
  return rb;
}

template <int RB>
static int launch_rows(const RowsProductArgs& args, hipStream_t s) {
  RowsProductArgs a = args;
  const int tiles_m = (a.rows + 32 * RB - 1) / (32 * RB), tiles_n = a.N / RP_BN, per_round = CUS / 8 * (RB == 2 ? 3 : 2);
  // the grid of XCDs with the fewest rounds of workgroups, and of those the one that fetches least
  int64_t best = -1;
  for (int m = 1, shift = 0; m <= 8; m *= 2, ++shift) {
    const int mc = (tiles_m + m - 1) / m, nc = (tiles_n + 8 / m - 1) / (8 / m);
    const int64_t cost = ((int64_t)(mc * nc + per_round - 1) / per_round << 32) + mc * 32 * RB + nc * RP_BN;
    if (best >= 0 && cost >= best) continue;
    best = cost;
    a.xcd_m = m; a.xcd_shift = shift; a.m_chunk = mc; a.n_chunk = nc;
  }
  a.magic_chunk = a.m_chunk == 1 ? 0u : 0xffffffffu / (uint32_t)a.m_chunk + 1u;
  a.magic_cond = a.cond_rows <= 1 ? 0u : 0xffffffffu / (uint32_t)a.cond_rows + 1u;
  const dim3 grid(8u * a.m_chunk * a.n_chunk), block(256);
  if (a.gate) {
    if (a.K == 768) hipLaunchKernelGGL((rows_product_kernel<12, ROWS_GATED, RB>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((rows_product_kernel<24, ROWS_GATED, RB>), grid, block, 0, s, a);
  } else if (a.swiglu) {
    hipLaunchKernelGGL((rows_product_kernel<12, ROWS_SWIGLU, RB>), grid, block, 0, s, a);
  } else {
    hipLaunchKernelGGL((rows_product_kernel<12, ROWS_QKVG, RB>), grid, block, 0, s, a);
  }
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

int launch_rows_product(const RowsProductArgs& a, hipStream_t s) {
  if (!rows_product_applies(a)) return AF3_ERR_BAD_ARG;
  switch (rows_product_blocks(a)) {
    case 2: return launch_rows<2>(a, s);
    case 3: return launch_rows<3>(a, s);
    default: return launch_rows<4>(a, s);
  }
}
