// Triangle attention, the flash-attention core (4 heads of 32 channels, or of 16).
//
// Operands (all produced by triattn_proj_kernel, see kernels.h):
//   Q, K    : bf16 [b][h][s][D]  (Q pre-multiplied by log2(e)/sqrt(D))
//   Vt      : bf16 [b][h][D][ldn], V transposed, ldn = N rounded up to 16, columns
//             permuted inside every aligned group of 16 (tri_vt_pos) so that the 8 keys one
//             lane feeds to a P.V MFMA are 16 contiguous bytes
//   bias    : fp16, pair bias * log2(e) in MFMA-fragment order (tri_bias_offset)
//   mask    : fp32 [N][N] 0/1 or null
//
// What sets the pace on this machine (measured): a wave64 exp2 occupies the SIMD's issue port
// for 8 cycles, any other vector instruction for 4-5, a 32x32x16 MFMA for 9 to 16 of the 32
// cycles it takes in the matrix unit, whichever wave it comes from; what is left of them another
// wave's vector instructions fill.  From some 700 tokens on the clock gives way as well (1.95 to
// 2.07 GHz in this kernel, 2.35 in arithmetic alone), to the loads more than to the arithmetic.
// The other cost is what a workgroup pulls in from L2 per key
// tile: with every load taken out of the key-tile loop (operands reused, results wrong) the
// kernel runs 30 % faster, 17 % of which remain when the same loads all hit the CU's own
// cache, i.e. are the loads into LDS as such, the rest is the L2 traffic (8 KB of K / V^T per
// row and 4 KB of bias per wave and key tile: 28 GB per launch at 1536 tokens).  The kernel
// is built around both:
//   * one wave = 32 queries of R rows b; lane = one query; S^T = K Q^T so that the softmax
//     reductions are per lane.  The pair bias enters on the matrix unit as well, S^T += I *
//     bias^T with an fp16 identity; its fragments do not depend on the row, so the R rows of a
//     wave share one load of them, straight into registers.  (With the fp32 bias as the
//     accumulators' initial value the kernel ran 35 % slower than without any bias: the bytes
//     the bias brings in from L2 are half of all it loads; hence fp16 and two rows per wave.)
//   * the key mask rides in the product as a third k-step (K side 0 / -1e9 / -inf, Q side 1.0),
//     and so does the softmax's running base: the Q side of the next slot holds -base, so the
//     accumulator comes out as s - base and exp2 takes it as it is.  `base` only moves when a
//     tile's scores leave [-64, 16] relative to it (a wave-uniform, rare branch that rescales
//     O and l by an exact-in-fp32 factor and repeats the tile's score product); for ordinary
//     logits it never moves and the softmax is computed without a single subtraction.
//     The third k-step is left out (wave-uniformly) for a tile of 64 unmasked keys while no
//     lane of the row has moved its base: eight MFMAs per key tile and row (the algorithm's
//     own count) plus the four of the bias.
//   * the probabilities of tile v go into O while the exponentials of tile v+1 are computed:
//     each of those four MFMAs is issued in front of eight exponentials of the same wave, its
//     V^T fragment read from LDS one group ahead.  Row sums are taken from the bf16
//     probabilities by v_dot2c_f32_bf16 against a pair of ones (per lane, i.e. per half of the
//     keys; the halves are added once at the end).  Heads of 16 leave half of the P.V product's
//     rows to spare: a row of ones behind V^T makes the sum there (768 tokens 3 % of a block).
//   * K and V^T tiles go from global memory straight into LDS (global_load_lds_dwordx4: no
//     staging registers, no LDS store instructions), double-buffered per row with one barrier
//     per key tile; unpadded rows with XOR-permuted 16-byte chunks keep the fragment reads
//     conflict-free.
// Key tiles whose 64 keys are masked in every row of the wave are left out (their
// probabilities are exactly zero); a row whose keys are ALL masked gets the reference's exact
// answer, the mean of V, directly.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace {

constexpr int H = 4;
constexpr int KT = 64;    // keys per tile
constexpr int QW = 128;   // queries per workgroup (32 per wave)
constexpr int tile_bytes(int d) { return KT * d * 2; }  // a K tile [64 keys][d] or a V^T tile [d][64 keys], bf16
constexpr int RSRC_RAW = 0x00020000;  // last word of a raw (unstructured, range-checked) buffer descriptor
constexpr uint32_t BF16_ONE = 0x3F80u, BF16_NEG_INF = 0xFF80u, BF16_NEG_1E9 = 0xCE6Eu;
// A tile's scores, relative to the base, may rise to 2^T_HI before the base is moved (fp32 and
// bf16 share their exponent range, so nothing is lost up there); the first tile with an unmasked
// key moves it if its maximum lies below 2^T_LO.  Scores of masked keys sit near -1e9.
constexpr float T_HI = 16.f, T_LO = -64.f, LIVE_MIN = -1e8f;

// 64 lanes x 16 bytes from global memory (wave-uniform base + per-lane byte offset + OFF) to
// 1 KB of LDS at the wave-uniform `dst` + OFF (lane l's bytes land at 16 l).  Issued as inline
// assembly on purpose: the compiler tracks loads into LDS that it can see and, unable to tell
// the buffers apart, makes every later fragment read wait for ALL loads in flight (vmcnt(0)),
// the ones issued a moment ago for the next tile included.  Here each buffer is read only
// after a dma_barrier() that follows the load's issue, which is what makes this safe.
template <int OFF>
__device__ __forceinline__ void dma16(const char* gbase, uint32_t voff, const char* dst) {
  const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3"
               :: "s"(lds), "v"(voff), "s"(gbase), "n"(OFF) : "memory", "m0");
}
__device__ __forceinline__ bf16x8 lds16(const char* p) { return as_frag(*reinterpret_cast<const u32x4*>(p)); }

// Workgroup barrier that also waits for this wave's loads, those into LDS and the ordinary ones
// (the bias registers).  The wait is a builtin so that the compiler sees it: it then knows the
// registers have landed and puts no wait of its own in front of their use, where it would also
// wait for the loads into LDS issued since.
__device__ __forceinline__ void dma_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ float max32(const f32x16& a, const f32x16& b) {
  // maximum of the lane's 32 scores as a tree of three-input maxima
  float t3[11];
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    const int e = 3 * i;
    const float x = e < 16 ? a[e & 15] : b[e & 15];
    const float y = e + 1 < 16 ? a[(e + 1) & 15] : b[(e + 1) & 15];
    const float z = e + 2 < 16 ? a[(e + 2) & 15] : b[(e + 2) & 15];
    t3[i] = fmaxf(fmaxf(x, y), z);
  }
  t3[10] = fmaxf(b[14], b[15]);
  const float t9a = fmaxf(fmaxf(t3[0], t3[1]), t3[2]), t9b = fmaxf(fmaxf(t3[3], t3[4]), t3[5]);
  const float t9c = fmaxf(fmaxf(t3[6], t3[7]), t3[8]), t9d = fmaxf(t3[9], t3[10]);
  return fmaxf(fmaxf(fmaxf(t9a, t9b), t9c), t9d);
}

// o *= f with every register multiplied in place.  Written as plain C++ inside a rarely taken
// branch, the compiler keeps the accumulator in two register tuples and copies all sixteen
// registers on the path that does NOT multiply, every iteration.
__device__ __forceinline__ void scale_in_place(f32x16& o, float f) {
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    float t = o[e];
    asm volatile("v_mul_f32 %0, %1, %0" : "+v"(t) : "v"(f));
    o[e] = t;
  }
}

template <int R, bool HAS_BIAS, int D, bool SPARE>
__global__ __launch_bounds__(256, R == 1 ? 3 : 2) void triattn_flash_kernel(TriAttnArgs a) {
  args_at_once<TriAttnArgs>();
  constexpr int TILE_BYTES = tile_bytes(D);
  constexpr int KS = D / 16;  // k-steps of the score product
  // [buffer][row] as separate arrays: a load in flight to one of them provably does not alias
  // a fragment read from another
  __shared__ __attribute__((aligned(1024))) char sK00[TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) char sK01[R > 1 ? TILE_BYTES : 16];
  __shared__ __attribute__((aligned(1024))) char sK10[TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) char sK11[R > 1 ? TILE_BYTES : 16];
  // Heads of 16: a V^T tile has one row more, of ones.  The sixteen rows of the P.V product that no channel needs read it,
  // so that O's register 8 is the row's sum of probabilities.
  constexpr int V_BYTES = TILE_BYTES + (D == 16 ? KT * 2 : 0);
  __shared__ __attribute__((aligned(1024))) char sV00[V_BYTES];
  __shared__ __attribute__((aligned(1024))) char sV01[R > 1 ? V_BYTES : 16];
  __shared__ __attribute__((aligned(1024))) char sV10[V_BYTES];
  __shared__ __attribute__((aligned(1024))) char sV11[R > 1 ? V_BYTES : 16];
  __shared__ __attribute__((aligned(16))) uint64_t sBits[4][R][2];  // per wave and row, a bit per key tile: see the mask pass
  __shared__ float sMean[D];
  __shared__ uint32_t sRedo;  // a wave's unmasked-tile shortcut went wrong: the workgroup repeats its rows without it
  extern __shared__ __attribute__((aligned(16))) uint16_t sCode[];  // [R][nkt * 64] mask code per key of the tiles that need one
#define KBUF(ph, r) ((ph) == 0 ? ((r) == 0 ? sK00 : sK01) : ((r) == 0 ? sK10 : sK11))
#define VBUF(ph, r) ((ph) == 0 ? ((r) == 0 ? sV00 : sV01) : ((r) == 0 ? sV10 : sV11))

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, j = lane & 31;
  const int xaddr = half_swap_addr();
  const int N = a.N;
  const int ldn = (int)a.ldn;
  const int NG = (N + R - 1) / R;  // groups of R rows
  // Workgroup ids are dealt round-robin to the 8 XCDs (the x dimension of the grid).  The query tiles of one (row group,
  // head) share its K / V and run back to back on one XCD (y); the (row group, head) pairs are
  // dealt to the XCDs in turn (z), so every XCD works on one head at a time (pair % 4 follows
  // from xcd % 4) and finds that head's bias in its L2.
  const int qt = blockIdx.y, slot = blockIdx.z * gridDim.y + qt;
  const int pair_idx = blockIdx.z * 8 + blockIdx.x;
  if (pair_idx >= H * NG) return;
  const int rg = pair_idx / H;
  const int h = pair_idx % H;
  // SPARE: the blocks of 32 queries leave some wave of a tile without one.  They are shared out evenly between the tiles
  // of a (row group, head); a wave without a block takes part in the loads and the barriers only and leaves its SIMD to
  // the other workgroup on the CU (which wave that is changes from workgroup to workgroup).  Computing on clamped queries
  // instead, as the other form does where no wave is without: 387 tokens 106 us against 99, 450 131 against 129, 600
  // 253 against 245; with a block for every wave the even form is the slower one, 768 tokens 434 against 430.
  const int first = SPARE ? qt * a.tile_blocks + min(qt, a.tile_extra) : qt * 4;
  const int turn = SPARE ? (wave + slot + (slot >> 5)) & 3 : wave;
  const bool active = !SPARE || turn < a.tile_blocks + (qt < a.tile_extra ? 1 : 0);
  const int qblk = active ? first + turn : first;
  const int nq = active ? min(32, N - qblk * 32) : 0;  // queries of this wave (past the end it works on clamped ones)
  const uint64_t query_lanes = nq == 32 ? ~0ull : ((1ull << max(nq, 0)) - 1ull) * 0x100000001ull;
  const int qi = min(qblk * 32 + j, N - 1);
  const int nkt = (N + KT - 1) / KT;
  const int nk64 = nkt * KT;

  int brow[R];
  bool bvalid[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    bvalid[r] = rg * R + r < N;
    brow[r] = min(rg * R + r, N - 1);
  }

  // ---- per-lane constants ----
  u32x4 qm[R];  // Q side of the mask k-step: slot 0 = 1.0 (times the key's code), slot 1 = -base
  const char* kglob[R];
  const char* vglob[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t bh = (int64_t)brow[r] * H + h;
    qm[r] = u32x4{hh == 0 ? (BF16_ONE | 0x80000000u) : 0u, 0u, 0u, 0u};  // -0.0 in slot 1
    kglob[r] = reinterpret_cast<const char*>(a.k + bh * N * D);
    vglob[r] = reinterpret_cast<const char*>(a.vt + bh * D * a.ldn);
  }
  // fragment reads: K row (32 u + j), chunk (2 ks + hh) ^ ((j >> 2) & 3); V^T row j, chunk (2 s + hh) ^ ((j >> 1) & 7)
  // heads of 16: K in blocks of 32 rows, the rows' first chunks and then their second ones; V^T row min(j, 16)
  const int ksw = (j >> 2) & 3;
  const int ka0 = D == 16 ? j * 16 + hh * 512 : j * 64 + ((hh ^ ksw) << 4), ka1 = j * 64 + (((2 + hh) ^ ksw) << 4);
  const int vrow = min(j, D), vsw = (vrow >> 1) & 7;
  int va[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) va[s] = vrow * 128 + (((2 * s + hh) ^ vsw) << 4);
  // loads into LDS: K keys 16 w + lane / 4, position lane % 4; V^T rows 8 w + lane / 8, position lane % 8
  // heads of 16: K by the first two waves, V^T by the other two
  const int part = D == 16 ? wave & 1 : wave;
  const bool loads_k = D == 32 || wave < 2, loads_v = D == 32 || wave >= 2;
  const int dk_key = D == 16 ? 32 * part + j : 16 * part + (lane >> 2);
  const uint32_t dk_chunk = D == 16 ? (uint32_t)(hh << 4) : (uint32_t)(((lane & 3) ^ ((dk_key >> 2) & 3)) << 4);
  const int dv_row = 8 * part + (lane >> 3);
  const int dv_col = ((lane & 7) ^ ((dv_row >> 1) & 7)) * 8;
  auto dma_k = [&](int tile, int r, char* buf) {  // a tile past the end re-reads the last one (never used)
    if (!loads_k) return;
    const int key = min(min(tile, nkt - 1) * KT + dk_key, N - 1);
    dma16<0>(kglob[r], (uint32_t)key * (D * 2u) + dk_chunk, buf + part * 1024);
  };
  auto dma_v = [&](int tile, int r, char* buf) {
    if (!loads_v) return;
    const int col = min(tile, nkt - 1) * KT + dv_col;  // columns past ldn: any finite data will do (P is zero there)
    dma16<0>(vglob[r], (uint32_t)(dv_row * ldn + (col < ldn ? col : 0)) * 2u, buf + part * 1024);
  };
  // bias tiles of this wave's 32-query block: 4 KB per key tile
  const char* bbase =
      HAS_BIAS ? reinterpret_cast<const char*>(a.bias + tri_bias_offset(N, h, qblk * 32, 0)) : nullptr;
  // The bias tile of key tile t + 1 (four 1 KB fp16 fragments; fragment i = 2 u + st: keys
  // 32 u + 16 st + 8 hh .. + 8 of this lane's query, bytes 32 j + 16 hh of run i) is only ever
  // read by this wave, so it goes from memory straight into registers, requested when tile t
  // begins.  The wait that the barrier in the middle of tile t needs anyway covers it.  While
  // the last row of tile t computes its exponentials the fragments are turned into fp32 on
  // the matrix unit, bt = I * bias^T with an fp16 identity: the initial value of the score
  // accumulators of every row of tile t + 1 (four MFMAs per key tile, each issued between
  // two groups of exponentials).  With one row per wave (LATE) there is nothing to share: the fragments start the tile's
  // own score product, requested behind that of the tile before, and without bt's registers a third wave fits the SIMD
  // (201 -> 168; 160 tokens 16.5 -> 13.8 us, 208 25.6 -> 22.2).  (Staged through LDS like K and V^T, by loads into LDS two
  // tiles ahead, the same kernel ran 3.5 % slower: a load into LDS costs the wave more than
  // a load into registers, and the fragments cost an LDS read each on top.)
  constexpr bool LATE = R == 1 && HAS_BIAS;
  f32x16 bt[2];
  u32x4 bnext[4];
  auto load_bias = [&](int tile) {
    if (!HAS_BIAS) return;
    const char* p = bbase + (size_t)min(tile, nkt - 1) * 4096u + (j * 32 + hh * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) bnext[i] = *reinterpret_cast<const u32x4*>(p + 1024 * i);
  };
  auto first_loads = [&](int cur, int next) {
    dma_k(cur, 0, KBUF(0, 0));
    if (R == 2) {
      dma_k(cur, R - 1, KBUF(0, R - 1));
      dma_k(next, 0, KBUF(1, 0));
      dma_v(cur, 0, VBUF(0, 0));
      dma_v(cur, R - 1, VBUF(0, R - 1));
    }
  };

  // ---- mask pass: per-key codes for the mask k-step, live key tiles, dead rows ----
  // A wave takes every fourth key tile; the mask values of four of its tiles and all rows are requested together.  Behind the
  // first batch go Q, the first bias tile and the loads into LDS for the first key tile, as if that were tile 0 (and the one
  // after it tile 1; they are unless a sequence begins with 64 masked keys, and then these are loaded again below): a
  // workgroup begins with one trip to memory.  What costs here are not the trips but the instructions: up to some 400 tokens
  // a workgroup has few key tiles to spread them over, so the mask comes through range-checked loads off one address (what
  // lies past the row reads as masked), a wholly unmasked tile costs a comparison and two scalar instructions (no codes: its
  // few readers on the careful route know it), and what the waves found out meets in LDS as bit masks.  Of a workgroup's 17000
  // cycles at 301 tokens 3600 went by before the end of this pass and 2100 more before the loop (us, two trips and a byte per
  // tile before / now: 100 tokens 6.58 / 6.30, 187 15.55 / 14.77, 256 24.9 / 23.8, 320 50.9 / 49.5, from 400 on +-1 %).
  bf16x8 qf[R][KS];
  // (a key tile's bit: the first 63 tiles one each, the others share the last one; `all_bits` knows the first 64 only)
  uint64_t any_bits[R], all_bits[R];
  __amdgpu_buffer_rsrc_t mrow[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    any_bits[r] = all_bits[r] = 0ull;
    mrow[r] = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.mask ? a.mask + (int64_t)brow[r] * N : nullptr), 0, a.mask ? N * 4 : 0,
                                                RSRC_RAW);
  }
  for (int t0 = wave; t0 < nkt || t0 == wave; t0 += 16) {
    float mv[R][4];
    if (a.mask) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          mv[r][u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mrow[r], (t0 * KT + lane) * 4 + u * 4 * KT * 4, 0, 0));
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int u = 0; u < 4; ++u) mv[r][u] = (t0 + 4 * u) * KT + lane < N ? 1.f : 0.f;
    }
    if (t0 == wave) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int64_t row = ((int64_t)brow[r] * H + h) * N + qi;
        const bf16_t* qp = a.q + row * D + 8 * hh;
        qf[r][0] = as_frag(*reinterpret_cast<const u32x4*>(qp));
        if constexpr (KS == 2) qf[r][1] = as_frag(*reinterpret_cast<const u32x4*>(qp + 16));
      }
      load_bias(0);
      __builtin_amdgcn_sched_barrier(0);
      first_loads(0, 1);
      if (tid == 0) sRedo = 0u;
      if (D == 16 && tid < KT / 8) {
        const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
        const int at = TILE_BYTES + tid % (KT / 8) * 16;
        *reinterpret_cast<u32x4*>(sV00 + at) = ones;
        *reinterpret_cast<u32x4*>(sV10 + at) = ones;
        if constexpr (R > 1) {
          *reinterpret_cast<u32x4*>(sV01 + at) = ones;
          *reinterpret_cast<u32x4*>(sV11 + at) = ones;
        }
      }
      // the buffer the first virtual tile reads its "previous" V^T from must hold finite data
      if (tid * 16 < TILE_BYTES) *reinterpret_cast<u32x4*>(VBUF(1, R - 1) + tid * 16) = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int tile = t0 + 4 * u;
      if (tile >= nkt) break;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint64_t on_lanes = __ballot(mv[r][u] != 0.f);
        const uint64_t bit = 1ull << min(tile, 63);
        if (on_lanes != 0ull) any_bits[r] |= bit;
        if (on_lanes == ~0ull && tile < 64) {
          all_bits[r] |= bit;
        } else {
          const int key = tile * KT + lane;
          sCode[r * nk64 + key] = (uint16_t)(key >= N ? BF16_NEG_INF : (mv[r][u] == 0.f ? BF16_NEG_1E9 : 0u));
        }
      }
    }
  }
  if (lane < R) {
    sBits[wave][lane][0] = R == 2 && lane == 1 ? any_bits[R - 1] : any_bits[0];
    sBits[wave][lane][1] = R == 2 && lane == 1 ? all_bits[R - 1] : all_bits[0];
  }
  dma_barrier();  // (a workgroup without a live key has its loads into LDS behind it, too)
  bool dead[R];
  uint64_t live = 0ull;
  uint64_t plain[R];  // tiles of 64 unmasked keys below N (none beyond the 64th tile): they need no mask k-step
  bool all_dead = true;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    u32x4 w = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 4; ++i) w |= *reinterpret_cast<const u32x4*>(&sBits[i][r][0]);
    const uint64_t any = (uint64_t)__builtin_amdgcn_readfirstlane(w.y) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane(w.x);
    plain[r] = (uint64_t)__builtin_amdgcn_readfirstlane(w.w) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane(w.z);
    dead[r] = any == 0ull;
    all_dead = all_dead && dead[r];
    live |= any;
  }
  // next live tile, or nkt when none is left; more than 64 tiles are simply taken in order
  uint64_t rest = 0ull;
  int seq = 0;
  auto pop = [&]() {
    const bool found = rest != 0ull;
    const int tile = found ? __builtin_ctzll(rest) : seq;
    rest &= rest - 1;
    seq = min(seq + (found ? 0 : 1), nkt);
    return tile;
  };

  // mask code of a key (a tile of unmasked keys has none in LDS)
  auto code = [&](int r, int tile, int key) -> uint32_t {
    return tile < 64 && ((plain[r] >> tile) & 1ull) != 0ull ? 0u : sCode[r * nk64 + tile * KT + key];
  };
  f32x16 o[R];
  float lrun[R], base[R], mrel[R];  // lrun: sum of the probabilities of THIS lane's keys (half of each tile)
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int e = 0; e < 16; ++e) o[r][e] = 0.f;
    lrun[r] = 0.f;
    base[r] = 0.f;
    mrel[r] = -__builtin_huge_valf();
  }

  if (!all_dead) {
    // Identity fragments (fp16): A-fragment of k-step st: lane (row i = j, half hh) holds
    // I[i][16 st + 8 hh + e], e = 0..7: a single 1.0 where 16 st + 8 hh + e == i.
    f16x8 idf[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int e1 = j - 16 * st - 8 * hh;
      const uint32_t one = (j & 1) ? (0x3C00u << 16) : 0x3C00u;
      const int at = e1 >> 1;  // negative, or 4 and more, where this lane has none
      idf[st] = as_frag_f16(u32x4{at == 0 ? one : 0u, at == 1 ? one : 0u, at == 2 ? one : 0u, at == 3 ? one : 0u});
    }
    f32x16 zero16;
#pragma unroll
    for (int e = 0; e < 16; ++e) zero16[e] = 0.f;
    // K fragments of 64 keys [k-step][half of the keys], and one row's scores on top of the bias
    auto load_k_frags = [&](const char* kb, bf16x8 (&k)[KS][2]) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        k[0][u] = lds16(kb + u * (TILE_BYTES / 2) + ka0);
        if constexpr (KS == 2) k[1][u] = lds16(kb + u * (TILE_BYTES / 2) + ka1);
      }
    };
    auto scores = [&](const bf16x8 (&k)[KS][2], const bf16x8* q, f32x16& s0, f32x16& s1) {
      if constexpr (LATE) {
        s0 = mfma32_f16(idf[0], as_frag_f16(bnext[0]), zero16);
        s1 = mfma32_f16(idf[0], as_frag_f16(bnext[2]), zero16);
        s0 = mfma32_f16(idf[1], as_frag_f16(bnext[1]), s0);
        s1 = mfma32_f16(idf[1], as_frag_f16(bnext[3]), s1);
        s0 = mfma32(k[0][0], q[0], s0);
        s1 = mfma32(k[0][1], q[0], s1);
      } else {
        s0 = mfma32(k[0][0], q[0], bt[0]);
        s1 = mfma32(k[0][1], q[0], bt[1]);
      }
      if constexpr (KS == 2) {
        s0 = mfma32(k[1][0], q[1], s0);
        s1 = mfma32(k[1][1], q[1], s1);
      }
    };
#pragma unroll
    for (int e = 0; e < 16; ++e) bt[0][e] = bt[1][e] = 0.f;
    bool based[R];  // some lane of the wave has moved this row's base off zero
    float pend_alpha = 1.f;  // R == 1: a rescaling of O and l that waits for the tile in flight
    bool pend = false;
    // Tiles of 64 unmasked keys take their exponentials without looking at the tile's maximum
    // first ("fast").  Every lane of such a tile has 32 live keys, so the sums of what it got say
    // afterwards where the scores lay: a tile sum that is not below 2^60 (an overflow included)
    // means scores far above the base, a row total below 2^-30 scores far below it.  Per tile
    // only the largest tile sum is kept (one instruction); both conditions are looked at once,
    // when the row is through.  Either is rare and makes the whole workgroup repeat its rows
    // with every tile on the careful route.
    bool allow_fast = true;
    uint64_t bad = 0ull;
    float lmax[R];      // largest sum of one fast tile (heads of 16: of all tiles, whenever O was rescaled)
    bool used_fast[R];  // this wave took some tile of the row the fast way
    bf16x8 kpre[KS][2];  // R == 2: row 0's K fragments of the next key tile
    u32x4 pp[4];  // probabilities of the previous virtual tile (bf16 B fragments), zero before the first

    int t_cur = 0, t_n1 = 0, t_n2 = 0;  // this key tile and the next two
    // One virtual tile = (key tile, row RR): scores, softmax, and meanwhile the previous
    // virtual tile's probabilities go into its row sums and its O.
    auto iter = [&](auto PHc, auto RRc, int tile) {
      constexpr int PH = decltype(PHc)::value, RR = decltype(RRc)::value;
      constexpr int PR = (RR + R - 1) % R, VPH = RR == 0 ? PH ^ 1 : PH;
      const char* kb = KBUF(PH, RR);
      const char* vb = VBUF(VPH, PR);
      if (R == 1 && pend) {
        if constexpr (D == 16) lmax[0] = fmaxf(lmax[0], o[0][8]);
        scale_in_place(o[0], pend_alpha);
        pend = false;
      }
      // The third k-step carries the key mask and the base.  A tile of 64 unmasked keys whose row
      // still has base 0 in every lane needs neither (wave-uniform).
      const bool fast = allow_fast && tile < 64 && ((plain[RR] >> tile) & 1ull) != 0ull;
      const bool step3 = based[RR] || !fast;
      // Two rows per wave: row 0's K tile has been in LDS since the barrier before the previous
      // virtual tile, whose last group of exponentials fetched these fragments (kpre).
      bf16x8 kf[KS][2];
      if constexpr (R == 2 && RR == 0) {
#pragma unroll
        for (int i = 0; i < 2 * KS; ++i) kf[i >> 1][i & 1] = kpre[i >> 1][i & 1];
      } else {
        load_k_frags(kb, kf);
      }
      bf16x8 af0, af1;
      f32x16 s0, s1;
      scores(kf, qf[RR], s0, s1);
      if (step3) {
        const uint32_t c0 = code(RR, tile, j), c1 = code(RR, tile, 32 + j);
        af0 = as_frag(u32x4{hh == 0 ? (c0 | (BF16_ONE << 16)) : 0u, 0u, 0u, 0u});
        af1 = as_frag(u32x4{hh == 0 ? (c1 | (BF16_ONE << 16)) : 0u, 0u, 0u, 0u});
        s0 = mfma32(af0, as_frag(qm[RR]), s0);
        s1 = mfma32(af1, as_frag(qm[RR]), s1);
      }

      if (!fast) {
      float mx = max32(s0, s1);
      mx = fmaxf(mx, half_swap(xaddr, mx));
      const float mnew = fmaxf(mrel[RR], mx);
      // (lanes of queries past the end have no say: in a partly filled block they see bias values nobody wrote)
      const bool want = mx > T_HI || (mnew < T_LO && mnew > LIVE_MIN);
      if ((__ballot(want) & query_lanes) != 0ull) {
        // Move the base of every query of the wave to its running maximum (rounded to bf16, the
        // form the matrix unit takes it in), rescale what the row has accumulated, and repeat the
        // score product.  Lanes that have seen no unmasked key yet keep their base: their O and l
        // are still exactly zero.
        const bool has_live = mnew > LIVE_MIN;
        const float nb = has_live ? bf2f(f2bf(base[RR] + mnew)) : base[RR];
        const float delta = nb - base[RR];
        const float alpha = mrel[RR] > LIVE_MIN ? __builtin_amdgcn_exp2f(-delta) : 1.f;
        base[RR] = nb;
        mrel[RR] = mnew - delta;
        qm[RR].x = hh == 0 ? (BF16_ONE | ((uint32_t)f2bf(-nb) << 16)) : 0u;
        based[RR] = true;
        if (!step3) {
          const uint32_t c0 = code(RR, tile, j), c1 = code(RR, tile, 32 + j);
          af0 = as_frag(u32x4{hh == 0 ? (c0 | (BF16_ONE << 16)) : 0u, 0u, 0u, 0u});
          af1 = as_frag(u32x4{hh == 0 ? (c1 | (BF16_ONE << 16)) : 0u, 0u, 0u, 0u});
        }
        lrun[RR] *= alpha;  // the row sums are up to date (taken when the probabilities are made)
        if (R == 1) {
          // the previous virtual tile belongs to the same row and its probabilities, relative to the
          // old base, are not in O yet: O gets the factor once they are (top of the next iteration)
          pend_alpha = alpha;
          pend = true;
        } else {
          if constexpr (D == 16) lmax[RR] = fmaxf(lmax[RR], o[RR][8]);  // (an infinity may become a NaN here)
          scale_in_place(o[RR], alpha);
        }
        scores(kf, qf[RR], s0, s1);
        s0 = mfma32(af0, as_frag(qm[RR]), s0);
        s1 = mfma32(af1, as_frag(qm[RR]), s1);
      } else {
        mrel[RR] = mnew;
      }
      }
      float linc = 0.f;
      // From here to the end: one basic block in a fixed order.  Each of the four P.V MFMAs of the
      // previous virtual tile is issued in front of eight exponentials of this one (the matrix
      // unit works while the wave goes on issuing vector instructions), with its V^T fragment read from LDS one group ahead.
      if constexpr (LATE) load_bias(t_n1);
      bf16x8 vf = lds16(vb + va[0]);
      u32x4 bfr[4];  // the next key tile's bias fragments (the last row of this one fetches them)
      if (HAS_BIAS && !LATE && RR == R - 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) bfr[i] = bnext[i];  // (the registers are free for the next request)
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bf16x8 vcur = vf;
        if (s < 3) {
          vf = lds16(vb + va[s + 1]);
          __builtin_amdgcn_sched_barrier(0);
        } else if (R == 2 && RR == 1) {
          load_k_frags(KBUF(PH ^ 1, 0), kpre);
          __builtin_amdgcn_sched_barrier(0);
        }
        o[PR] = mfma32(vcur, as_frag(pp[s]), o[PR]);
        float p8[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) p8[e] = __builtin_amdgcn_exp2f(s < 2 ? s0[8 * (s & 1) + e] : s1[8 * (s & 1) + e]);
        if (HAS_BIAS && !LATE && RR == R - 1) {
          // fragments 2 u + st: bt[u] = I(st = 0) * f(2 u) + I(st = 1) * f(2 u + 1); group s does (u, st) = (s / 2, s % 2)
          asm volatile("" : "+v"(p8[0]), "+v"(p8[1]), "+v"(p8[2]), "+v"(p8[3]));
          bt[s >> 1] = mfma32_f16(idf[s & 1], as_frag_f16(bfr[s]), (s & 1) ? bt[s >> 1] : zero16);
        }
#pragma unroll
        for (int e = 4; e < 8; ++e) p8[e] = __builtin_amdgcn_exp2f(s < 2 ? s0[8 * (s & 1) + e] : s1[8 * (s & 1) + e]);
        // this tile's probabilities take the place of the previous tile's, whose last reader (the
        // MFMA above) has been issued
        pp[s] = pack8(p8);
        // pins the exponentials to this group (without it they sink to where their values are used,
        // the next iteration's MFMAs)
        asm volatile("" : "+v"(pp[s].x), "+v"(pp[s].y), "+v"(pp[s].z), "+v"(pp[s].w));
        if constexpr (D == 32) linc = dot2_ones(pp[s].w, dot2_ones(pp[s].z, dot2_ones(pp[s].y, dot2_ones(pp[s].x, linc))));
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (D == 32) lrun[RR] += linc;
      if (fast) {
        if constexpr (D == 32) lmax[RR] = fmaxf(lmax[RR], linc);
        // If the row passes its check at the end, its total is at least 2^-30 over at most 4096
        // keys: a lower bound of the running maximum, all the careful route's lower guard needs
        // (if it does not, the rows are repeated and what a careful tile decided meanwhile is void).
        mrel[RR] = fmaxf(mrel[RR], -42.f);
        used_fast[RR] = true;
      }
    };
    // the tail of the pipeline: the last virtual tile's probabilities
    auto drain = [&](const char* vb) {
      constexpr int PR = R - 1;
      if (D == 16 && R == 1 && pend) lmax[0] = fmaxf(lmax[0], o[0][8]);
      if (R == 1 && pend) scale_in_place(o[0], pend_alpha);  // what was accumulated before the last tile moved the base
#pragma unroll
      for (int s = 0; s < 4; ++s) o[PR] = mfma32(lds16(vb + va[s]), as_frag(pp[s]), o[PR]);
    };

#pragma nounroll
    for (int pass = 0; pass < 2; ++pass) {
    allow_fast = pass == 0;
    bad = 0ull;
    rest = nkt > 64 ? 0ull : live;
    seq = nkt > 64 ? 0 : nkt;
    pend = false;
#pragma unroll
    for (int s = 0; s < 4; ++s) pp[s] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // A zero that the compiler cannot see: of a known one it makes sixteen scalar registers, since this is a template over the
      // head dimension, spills others to lanes for them (two rows: 84 lane moves) and copies them from there.  Four blocks at
      // 768 tokens 9337 -> 9319 us, 387 2465 -> 2459: what the template had cost, no more.
      float zero = 0.f;
      asm("" : "+v"(zero));
#pragma unroll
      for (int e = 0; e < 16; ++e) o[r][e] = zero;
      lrun[r] = 0.f;
      base[r] = 0.f;
      mrel[r] = -__builtin_huge_valf();
      qm[r].x = hh == 0 ? (BF16_ONE | 0x80000000u) : 0u;
      based[r] = false;
      lmax[r] = 0.f;
      used_fast[r] = false;
    }
    t_cur = pop(); t_n1 = pop(); t_n2 = pop();
    if (pass == 1 || t_cur != 0 || (R == 2 && t_n1 != 1 && t_n1 < nkt)) {
      load_bias(t_cur);
      first_loads(t_cur, t_n1);
      if (tid * 16 < TILE_BYTES) *reinterpret_cast<u32x4*>(VBUF(1, R - 1) + tid * 16) = u32x4{0u, 0u, 0u, 0u};
      dma_barrier();
    }
    if (HAS_BIAS && !LATE) {
      bt[0] = mfma32_f16(idf[1], as_frag_f16(bnext[1]), mfma32_f16(idf[0], as_frag_f16(bnext[0]), zero16));
      bt[1] = mfma32_f16(idf[1], as_frag_f16(bnext[3]), mfma32_f16(idf[0], as_frag_f16(bnext[2]), zero16));
    }
    if (R == 2) load_k_frags(KBUF(0, 0), kpre);
    // Every ordinary load issued so far (Q, the first bias tile) is waited for HERE, with a wait
    // the compiler can see: otherwise it keeps a vmcnt(0) for them at the top of the loop, where
    // it would also wait, every iteration, for the loads into LDS issued just before.
    __builtin_amdgcn_s_waitcnt(0x0F70);
    // One key tile per step.  R = 2: row 0's virtual tile, barrier, loads for what is read
    // after the NEXT barrier (K of row 1 of the next tile, K of row 0 of the tile after it,
    // V^T of the next tile), row 1's virtual tile.  R = 1: barrier, loads (next K, this V^T),
    // the virtual tile.
    auto step = [&](auto PHc) {
      constexpr int PH = decltype(PHc)::value;
      using P0 = std::integral_constant<int, PH>;
      if (R == 2) {
        load_bias(t_n1);
        iter(P0{}, std::integral_constant<int, 0>{}, t_cur);
        dma_barrier();
        dma_k(t_n1, 1, KBUF(PH ^ 1, 1));
        dma_k(t_n2, 0, KBUF(PH, 0));
        dma_v(t_n1, 0, VBUF(PH ^ 1, 0));
        dma_v(t_n1, 1, VBUF(PH ^ 1, 1));
        iter(P0{}, std::integral_constant<int, R - 1>{}, t_cur);
      } else {
        dma_barrier();
        dma_k(t_n1, 0, KBUF(PH ^ 1, 0));
        dma_v(t_cur, 0, VBUF(PH, 0));
        iter(P0{}, std::integral_constant<int, 0>{}, t_cur);
      }
      t_cur = t_n1;
      t_n1 = t_n2;
      t_n2 = pop();
    };
    int last_ph = 0;
    if (SPARE && !active) {
      // the loads and barriers of the steps
      for (int ph = 0; t_cur < nkt; ph ^= 1) {
        dma_barrier();
        if (R == 2) {
          dma_k(t_n1, R - 1, ph == 0 ? KBUF(1, R - 1) : KBUF(0, R - 1));
          dma_k(t_n2, 0, ph == 0 ? KBUF(0, 0) : KBUF(1, 0));
          dma_v(t_n1, 0, ph == 0 ? VBUF(1, 0) : VBUF(0, 0));
          dma_v(t_n1, R - 1, ph == 0 ? VBUF(1, R - 1) : VBUF(0, R - 1));
        } else {
          dma_k(t_n1, 0, ph == 0 ? KBUF(1, 0) : KBUF(0, 0));
          dma_v(t_cur, 0, ph == 0 ? VBUF(0, 0) : VBUF(1, 0));
        }
        t_cur = t_n1;
        t_n1 = t_n2;
        t_n2 = pop();
      }
    } else {
      while (true) {
        step(std::integral_constant<int, 0>{});
        last_ph = 0;
        if (t_cur >= nkt) break;
        step(std::integral_constant<int, 1>{});
        last_ph = 1;
        if (t_cur >= nkt) break;
      }
    }
    dma_barrier();  // every load into LDS has landed (none is in flight when the workgroup ends)
    if (active) drain(last_ph == 0 ? VBUF(0, R - 1) : VBUF(1, R - 1));
    if (pass == 1) break;
    // (lanes of queries past the end work on clamped operands and, in a partly filled bias block, on
    // bias values nobody wrote: they have no say)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!used_fast[r] || dead[r]) continue;
      const float lt = D == 16 ? o[r][8] : lrun[r] + half_swap(xaddr, lrun[r]);
      bad |= query_lanes & __ballot((!((D == 16 ? fmaxf(lt, lmax[r]) : lmax[r]) < 0x1p60f) || lt < 0x1p-30f));
    }
    if (bad != 0ull && lane == 0) sRedo = 1u;
    lds_barrier();  // also: every wave is done with the K / V^T tiles before a second pass loads over them
    if (__builtin_amdgcn_readfirstlane(sRedo) == 0u) break;
    }
  }

  // (what follows takes the lane's numbers anew: kept over the loops they would cost registers there)
  int tid_end = threadIdx.x;
  asm volatile("" : "+v"(tid_end));
  const int hh_end = (tid_end >> 5) & 1, j_end = tid_end & 31;
  // a query's keys are split over the two half-waves
#pragma unroll
  for (int r = 0; r < R; ++r) lrun[r] = D == 16 ? o[r][8] : lrun[r] + half_swap(xaddr, lrun[r]);

  // ---- rows whose keys are all masked: the reference replaces every logit by the same -1e9,
  // the softmax is exactly uniform and each query's output is the mean of V over the N keys ----
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (!dead[r]) continue;
    lds_barrier();
    const int v_d = (tid >> 3) & (D - 1), c8 = (tid & 7) * 8;
    const bf16_t* vrow = a.vt + (((int64_t)brow[r] * H + h) * D + v_d) * a.ldn;
    float acc = 0.f;
    // columns N..ldn-1 are zero; eight loads in flight at a time (one at a time, each waits out a
    // trip to memory, and a row of padding costs as much as a row of attention)
    for (int kb = c8; kb < ldn; kb += 512) {
      u32x4 raw[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k0 = kb + 64 * i;
        raw[i] = *reinterpret_cast<const u32x4*>(vrow + (k0 < ldn ? k0 : c8));
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float f[8];
        unpack8(raw[i], f);
        if (kb + 64 * i < ldn) {
#pragma unroll
          for (int e = 0; e < 8; ++e) acc += f[e];
        }
      }
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    acc += __shfl_xor(acc, 4);
    if ((tid & 7) == 0) sMean[v_d] = acc;
    lds_barrier();
#pragma unroll
    for (int e = 0; e < 16; ++e) o[r][e] = sMean[8 * ((e >> 2) & (D / 8 - 1)) + 4 * hh_end + (e & 3)];
    lrun[r] = (float)N;
  }

  if (j_end >= nq) return;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (!bvalid[r]) continue;
    const float inv = 1.f / lrun[r];  // the sum over both half-waves' keys
    bf16_t* op = a.og + ((int64_t)brow[r] * N + qblk * 32 + j_end) * (H * D) + h * D + 4 * hh_end;
#pragma unroll
    for (int g = 0; g < D / 8; ++g) {
      u32x2 w;
      w.x = pack2bf(o[r][4 * g] * inv, o[r][4 * g + 1] * inv);
      w.y = pack2bf(o[r][4 * g + 2] * inv, o[r][4 * g + 3] * inv);
      *reinterpret_cast<u32x2*>(op + 8 * g) = w;
    }
  }
#undef KBUF
#undef VBUF
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int launch_triattn_flash(const TriAttnArgs& a, hipStream_t stream) {
  if (!a.q || !a.k || !a.vt || !a.og || a.N <= 0 || a.N > 8192) return AF3_ERR_BAD_ARG;
  if (a.ldn < a.N || (a.ldn & 15) || (a.head_dim != 32 && a.head_dim != 16)) return AF3_ERR_BAD_ARG;
  if (!al16(a.q) || !al16(a.k) || !al16(a.vt) || !al16(a.og) || !al16(a.bias)) return AF3_ERR_BAD_ARG;
  const int QT = (a.N + QW - 1) / QW;
  const int nkt = (a.N + KT - 1) / KT;
  // One row per wave leaves room for three waves to a SIMD, two rows share one load of the bias.  The line lies where the
  // workgroups are enough rounds for the traffic to count more than the waves that hide each other's waits; us, one row
  // against two: 64 tokens 4.3 (5.8), 160 13.8 (17.0), 208 22.2 (24.5), 256 25.5 (26.4), 310 52.9 (54.0), but 320 53.5
  // (52.9), 384 74.6 (71.8), 512 150 (143), 768 452 (429).  Heads of 16, whose row is less to load, a pair block: 187 tokens
  // 111 (113), 301 199 (205), 420 381 (384), but 512 491 (480), 768 1484 (1409).
  // (One row, too, when the per-key mask codes of two would not fit the LDS share of a workgroup.)
  int R = (int64_t)((a.N + 1) / 2) * H * QT >= (a.head_dim == 16 ? 3500 : 1920) ? 2 : 1;
  // static LDS: K / V buffers, small arrays; dynamic: the mask codes.  Two workgroups must fit a
  // CU's 160 KB.
  const int tile = tile_bytes(a.head_dim);
  const size_t stat2 = 8 * (size_t)tile + 1024;
  if (R == 2 && stat2 + 2 * (size_t)nkt * KT * sizeof(uint16_t) > 80 * 1024) R = 1;
  const int NG = (a.N + R - 1) / R;
  const size_t dyn = (size_t)R * nkt * KT * sizeof(uint16_t);
  const dim3 grid(8, QT, (H * NG + 7) / 8), block(256);
  TriAttnArgs args = a;
  args.tile_blocks = (a.N + 31) / 32 / QT;
  args.tile_extra = (a.N + 31) / 32 % QT;
  const size_t stat = (R == 2 ? 8 : 4) * (size_t)tile + 1024;
  auto launch = [&](void (*kernel)(TriAttnArgs)) {
    // more than 64 KB of LDS per workgroup in all (static + dynamic) has to be asked for
    // (a per-function, per-device setting of the runtime: no allocation, no synchronisation; always for the most tokens, since
    // another thread may be launching with another size)
    if (stat + dyn > 65536) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(2 * 8192 * sizeof(uint16_t)));
      (void)hipGetLastError();
    }
    hipLaunchKernelGGL(kernel, grid, block, dyn, stream, args);
  };
  const bool spare = (a.N + 31) / 32 % 4 != 0;
  if (a.head_dim == 16) {
    if (!a.bias) return AF3_ERR_BAD_ARG;  // (nobody asks for it)
    if (R == 2) launch(spare ? triattn_flash_kernel<2, true, 16, true> : triattn_flash_kernel<2, true, 16, false>);
    else launch(spare ? triattn_flash_kernel<1, true, 16, true> : triattn_flash_kernel<1, true, 16, false>);
  } else if (!a.bias) {
    launch(R == 2 ? triattn_flash_kernel<2, false, 32, false> : triattn_flash_kernel<1, false, 32, false>);
  } else if (R == 2) {
    launch(spare ? triattn_flash_kernel<2, true, 32, true> : triattn_flash_kernel<2, true, 32, false>);
  } else {
    launch(spare ? triattn_flash_kernel<1, true, 32, true> : triattn_flash_kernel<1, true, 32, false>);
  }
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
