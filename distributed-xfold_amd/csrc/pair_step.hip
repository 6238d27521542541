// Steps of the pair path: the operators between two long products, one kernel (128 channels up to the sizes that sequence.hip
// sets, 64 channels throughout).
//
// Up to some two hundred tokens the pair tensor is a few hundred tiles of 128 positions, and a kernel of pair_tile.hip is
// one tile's chain of loads, LayerNorm, products and stores, run by a part of the CUs while the rest idles: at 64 tokens
// thirteen dependent launches of 4 to 16 us a block.  Beyond, each of them is a pass over the tensor.  All but the contraction
// and the attention core work on a pixel at a time, so here each run of them between two of those is one kernel, on tiles of 32
// or 64 positions:
//
//   outgoing epilogue  + incoming prologue           (patches of 4 x 8 pixels: the one reads rows, the other writes columns)
//   incoming epilogue  + starting-node projections   (rows)
//   starting-node gate and output projection + ending-node projections   (columns)
//   ending-node gate and output projection + transition [+ pair logits] [+ outgoing prologue of the next block]  (rows)
//
// A workgroup is one tile; its four waves share the rows of every weight matrix, 32 output channels each, so a weight is
// read once per tile.  The fragments come from L2 straight into registers, in the order the MFMAs take them (pair_frags
// of af3_pairformer_block: 1 KB per wave and load), requested a stage ahead; a row-major matrix would put every lane of
// such a load on a cache line of its own.  The tile's residual stream stays in registers from the first LayerNorm on and
// is rounded where the operators of pair_tile.hip store it, so the values are the same.
//
// What bounds it: at 64 tokens (128 tiles, one to a CU) the tile's chain, in which a weight that is not in L2 yet costs a
// trip to memory; with more tiles, and with a transition about equally, what a tile fetches of the weights (0.6 MB from L2 at
// 140 B/ns and CU, 4.3 us), vector issue (3.2 us a tile of 32 positions) and the matrix unit (2.3), which overlap as far as
// the waves of a SIMD do: 9.5 us a tile with two of them.  So the registers go to a third wave or to twice the positions for a
// weight, and not to weights in flight: one or two pieces of 32 rows, where four (three with a transition) were no faster at 64
// tokens and kept the third wave out.  Kernel alone, us, at 64 / 128 / 160 / 200 / 301 tokens, bf16 stream (128: fp32):
//   outgoing epilogue + incoming prologue 10.4 / 17.8 / 21.1 / 33 / -, in patches of 4 x 8 / 8 x 8 pixels
//   incoming epilogue + projections 7.9 / 15.5 / 19.1 / 24.5 / 42, output + projections 8.0 / 14.5 / 18.8 / 23.8 / 41
//     (three and four pieces: 8.4 / 16.1 / 19.9 / 27.1 / 43, 8.2 / 14.9 / 19.2 / 25.9 / 41)
//   output + transition + logits + prologue 13.9 / 22.7 / 31.6 / 47 / - (three pieces, tiles of 32: 14.1 / 22.9 / 36.4 / 53.4 / -)
//
// 64 channels (the template embedding): workgroups of two waves, otherwise the same code.  A quarter of the weights to a
// position and half of the rest, so that here the steps are the faster form whatever the number of tokens, and the tensor
// need not be padded to 128 channels and back (bf16, 301 tokens, us a block: 345 -> 221, 768: 1940 -> 1460; kernel alone
// at 301, bound by what it moves, 25 to 40 MB, and vector issue, four waves to a SIMD / three with twice the weights in flight:
// outgoing prologue 13.1 / 13.9, outgoing epilogue + incoming prologue 32.5 / 32.9 (8 x 8 patches 36), incoming epilogue +
// projections 20.5 / 21.9, output + projections 20.1 / 20.6, output + transition 20.2 / 22.0).
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int H = 4;
// hidden units of the transition: a chunk, and how many of them there are room for
constexpr int hidden_chunk_of(int channels) { return 2 * channels; }
constexpr int hidden_chunks(int channels) { return channels == 128 ? 2 : 1; }
enum { IN_NONE, IN_EPILOGUE, IN_ATTENTION };
enum { MAP_ROWS, MAP_COLUMNS, MAP_PATCH };
enum { NEXT_NONE, NEXT_PROLOGUE, NEXT_PROJECT };

// Row p of 32 in LDS (p = 8 g + 4 hh + e: accumulator register 4 g + e of lane half hh) is position 16 hh + 4 g + e,
// so that a lane's sixteen registers are sixteen consecutive positions.
__device__ __forceinline__ int step_pos(int p) { return ((p & 4) << 2) | ((p & 24) >> 1) | (p & 3); }

struct Pixel {
  int o, r;       // row and place in the row, in the frame the tile walks (rows or columns of the pair tensor)
  bool ok;
};

template <int PB, int MAP>
struct StepTile {
  int N, W;         // W: row length, N rounded up to 16
  int o0, r0;       // rows, columns: row and place of the first position;  patch: first pixel (i, j), 4 PB x 8 of them
  uint32_t magic;
  __device__ __forceinline__ Pixel at(int pos) const {  // position (not LDS row) of the tile
    Pixel x;
    if constexpr (MAP == MAP_PATCH) {
      x.o = o0 + (pos >> 3);
      x.r = r0 + (pos & 7);
    } else {
      const int v = r0 + pos, q = (int)__umulhi((uint32_t)v, magic);  // v < W + 64
      x.o = o0 + q;
      x.r = v - q * W;
    }
    x.ok = x.o < N && x.r < N;
    return x;
  }
  __device__ __forceinline__ int position(int p) const { return MAP == MAP_PATCH ? p : (p & 32) + step_pos(p & 31); }
  __device__ __forceinline__ Pixel row(int p) const { return at(position(p)); }
  // pixel of the pair tensor; of one outside it, the first
  __device__ __forceinline__ uint32_t pix(const Pixel& x) const {
    const uint32_t v = MAP == MAP_COLUMNS ? (uint32_t)x.r * N + x.o : (uint32_t)x.o * N + x.r;
    return x.ok ? v : 0u;
  }
};

// Pieces of the weights (32 rows) in flight: what the registers leave beside the waves of a SIMD.
constexpr int pieces_in_flight(int ch, int pb, int waves, bool transition) {
  return ch == 128 && (waves == 4 || (transition && (pb == 2 || waves == 3))) ? 1 : 2;
}

template <typename TIO, int CH, int PB, int IN, int MAP, bool TRANSITION, int NEXT, int PER_SIMD>
__global__ __launch_bounds__(2 * CH, PER_SIMD) void pair_step_kernel(PairStepArgs a) {
  args_at_once<PairStepArgs>();
  using E = Elem<TIO>;
  constexpr int TS = 32 * PB;           // positions per tile, in blocks of an MFMA's 32
  constexpr int C = CH, D = C / H, LDX = C + 8, LDS_F = C + 4;
  constexpr int WAVES = C / 32, NT = 2 * C, CHUNKS = C / 8, KS = C / 16;
  constexpr int HIDDEN_CHUNK = hidden_chunk_of(C), MAX_HIDDEN = HIDDEN_CHUNK * hidden_chunks(C);
  constexpr int NB = pieces_in_flight(C, PB, PER_SIMD, TRANSITION);
  // LDS row stride (bf16) of a channel's positions: the 16 lanes of a pixel, 8 channels apart, on 8 banks
  constexpr int LDT = TS + 2;
  constexpr int LDH = HIDDEN_CHUNK + 8;
  constexpr int U_BYTES = TS * LDS_F * 4;
  static_assert(U_BYTES >= C * LDT * 2 && U_BYTES >= TS * LDH * 2, "what takes turns in the staging tile fits");
  __shared__ __attribute__((aligned(16))) bf16_t sA[TS * LDX];
  __shared__ __attribute__((aligned(16))) bf16_t sB[TS * LDX];
  __shared__ __attribute__((aligned(16))) char sU[U_BYTES];
  __shared__ __attribute__((aligned(16))) float sMask[TS];
  __shared__ __attribute__((aligned(16))) float sP[8 * C];  // LayerNorm weights and biases: input, second, last, logits
  bf16_t* const sT = reinterpret_cast<bf16_t*>(sU);  // the contraction's tile, [channel][position]
  float* const sS = reinterpret_cast<float*>(sU);    // staged fp32 results, [LDS row][channel]
  bf16_t* const sH = reinterpret_cast<bf16_t*>(sU);  // a chunk of the transition's hidden layer, [LDS row][unit]
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chunk = tid % CHUNKS, prow = tid / CHUNKS;  // as in load_ln_tile: eight channels of rows prow, prow + 16, ..

  StepTile<PB, MAP> t;
  t.N = a.N;
  t.W = a.ldn;
  if constexpr (MAP == MAP_PATCH) {
    // an XCD takes a run of patches, those of one column block first: its L2 then puts together the cache lines of the
    // transposed operands, to which a patch contributes a few bytes each
    const int ib = a.Np / (4 * PB), total = ib * (a.Np >> 3), per = (total + 7) >> 3;
    const int idx = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || idx >= total) return;
    t.o0 = idx % ib * (4 * PB);
    t.r0 = idx / ib * 8;
  } else {
    const int l0 = (int)blockIdx.x * TS;
    t.o0 = __builtin_amdgcn_readfirstlane((uint32_t)l0 / (uint32_t)t.W);
    t.r0 = l0 - t.o0 * t.W;
    t.magic = __builtin_amdgcn_readfirstlane(0xffffffffu / (uint32_t)t.W) + 1u;
  }
  TIO* const pair = reinterpret_cast<TIO*>(a.pair);
  const int plane = (int)a.plane;
  Pixel mine[2 * PB], own[PB];  // of the thread's shares of pixels; of the lane's accumulator columns
#pragma unroll
  for (int u = 0; u < 2 * PB; ++u) mine[u] = t.row(prow + 16 * u);
#pragma unroll
  for (int b = 0; b < PB; ++b) own[b] = t.row(32 * b + j);

  // Everything the first stage needs is requested up front, in the order in which it is needed.  (Caches are cold: the
  // kernel before ran elsewhere, so every request of a stage's own would be a trip to memory in the tile's chain.)
  typename E::Raw raw[2 * PB];
#pragma unroll
  for (int u = 0; u < 2 * PB; ++u) raw[u] = E::load_raw(at32(pair, t.pix(mine[u]) * C + chunk * 8));
  f32x4 param = {0.f, 0.f, 0.f, 0.f};
  {
    // arrays 0, 1: input norm; 2, 3: contraction's or transition's; 4, 5: last stage's; 6, 7: logits'
    const int n = tid / (C / 4);
    const float* const w = n < 2 ? a.ln1_w : n < 4 ? (IN == IN_EPILOGUE ? a.ln_c_w : a.ln2_w) : n < 6 ? a.ln3_w : a.sl_ln_w;
    const float* const b = n < 2 ? a.ln1_b : n < 4 ? (IN == IN_EPILOGUE ? a.ln_c_b : a.ln2_b) : n < 6 ? a.ln3_b : a.sl_ln_b;
    const float* const src = (n & 1) ? b : w;
    if (src) param = *reinterpret_cast<const f32x4*>(src + tid % (C / 4) * 4);
  }
  u32x4 tt[2 * PB];
  u32x4 og[PB][2];
  if constexpr (IN == IN_EPILOGUE) {
#pragma unroll
    for (int u = 0; u < 2 * PB; ++u) {
      const int idx = tid + NT * u, c = idx / (4 * PB);
      const Pixel x = t.at(idx % (4 * PB) * 8);
      const bool ok = x.o < a.N && x.r < a.Np && c < a.valid_c;  // (positions past N in the row: zeroed with their pixel)
      tt[u] = *reinterpret_cast<const u32x4*>(at32(a.t_buf, ok ? (uint32_t)(c * plane + x.o * a.Np + x.r) : 0u));
      if (!ok) tt[u] = u32x4{0u, 0u, 0u, 0u};
    }
  } else if constexpr (IN == IN_ATTENTION) {
    // the attention output lies in the frame of the operator that made it: starting node (rows) before a step over
    // columns, ending node (columns) before a step over rows
#pragma unroll
    for (int b = 0; b < PB; ++b) {
      const uint32_t at = own[b].ok ? (uint32_t)(own[b].r * a.N + own[b].o) : 0u;
#pragma unroll
      for (int u = 0; u < 2; ++u) og[b][u] = *reinterpret_cast<const u32x4*>(at32(a.og, at * C + wave * 32 + 16 * u + 8 * hh));
    }
  }
  float mk = 0.f;
  if constexpr (NEXT == NEXT_PROLOGUE) {
    if (tid < TS) {
      const Pixel x = t.row(tid);
      mk = x.ok ? (a.mask ? *at32(a.mask, t.pix(x)) : 1.f) : 0.f;
    }
  }

  // The wave's weights, 32 rows of all k-steps (eight fragments or four) at a time, in the order of their use; piece n + NB
  // is asked for as soon as piece n has been multiplied.
  constexpr int OCT_HIDDEN = IN == IN_NONE ? 0 : 2, OCT_LOGITS = OCT_HIDDEN + (TRANSITION ? 6 * hidden_chunks(C) : 0);
  constexpr int OCT_NEXT = OCT_LOGITS + (TRANSITION && C == 128 ? 1 : 0);
  constexpr int OCTETS = OCT_NEXT + (NEXT == NEXT_NONE ? 0 : 4);
  const int pg = (wave >> 1) * 4 + (wave & 1);  // 32 projection rows; the gate rows that go with them are two blocks on
  const int n_hidden = a.hidden >> 5, nks = a.hidden >> 4;
  bf16x8 w[NB][KS];
  auto fetch = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < OCTETS) {
      bf16x8* const d = w[n % NB];
      if constexpr (n < OCT_HIDDEN) load_frags<KS>(n == 0 ? a.f_gate : a.f_out, wave, KS, 0, lane, d);
      else if constexpr (n < OCT_LOGITS) {
        constexpr int c = (n - OCT_HIDDEN) / 6, r = (n - OCT_HIDDEN) % 6;
        if constexpr (r < 4) {
          // hidden block hb of 32 units: rows 32 (hb & 1) of the 64 "a" rows of chunk hb / 2, then of its 64 "b" rows
          const int hb = min(c * (HIDDEN_CHUNK / 32) + wave + WAVES * (r >> 1), n_hidden - 1);
          load_frags<KS>(a.f_w1, (hb >> 1) * 4 + (hb & 1) + 2 * (r & 1), KS, 0, lane, d);
        } else {
          constexpr int k0 = c * (HIDDEN_CHUNK / 16) + (r - 4) * KS;  // (k-steps come in fours)
#pragma unroll
          for (int q = 0; q < KS; q += 4) load_frags<4>(a.f_w2, wave, nks, min(k0 + q, nks - 4), lane, d + q);
        }
      } else if constexpr (n < OCT_NEXT) {
        if (a.logits && wave * 32 < a.logit_heads) load_frags<KS>(a.f_logits, wave, KS, 0, lane, d);
      } else if constexpr (NEXT == NEXT_PROLOGUE) {
        constexpr int r = n - OCT_NEXT;
        load_frags<KS>(a.f_next, pg + (r & 1) * 2 + (r >> 1) * (C / 16), KS, 0, lane, d);
      } else {
        constexpr int r = n - OCT_NEXT;
        if constexpr (r < 2) load_frags<KS>(a.f_next, WAVES * r + wave, KS, 0, lane, d);
        else if (r == 2 || wave == 0) load_frags<KS>(a.f_v, r == 2 ? wave : WAVES, KS, 0, lane, d);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#define OCTET(n) std::integral_constant<int, (n)>{}
  fetch(OCTET(0));
  if constexpr (NB > 1) fetch(OCTET(1));
  // Weights further down the chain: the workgroups of an XCD between them touch every cache line once, so that the tiles,
  // which reach each stage at about the same time, find it in L2.
  uint32_t warm = 0u;
  {
    constexpr uint32_t LINES = C / 64;  // a row of C
    const uint32_t line = (blockIdx.x >> 3) * (uint32_t)NT + (uint32_t)tid;
    const uint32_t n0 = TRANSITION ? (uint32_t)a.hidden * 2u * LINES : 0u, n1 = TRANSITION ? (uint32_t)a.hidden * LINES : 0u;
    constexpr uint32_t n2 = NEXT == NEXT_PROLOGUE ? 4 * C * LINES : NEXT == NEXT_PROJECT ? 2 * C * LINES : 0u;
    constexpr uint32_t n3 = NEXT == NEXT_PROJECT ? (C + 32) * LINES : 0u;
    const bf16_t* const from = line < n0 ? a.f_w1 : line < n0 + n1 ? a.f_w2 - n0 * 64 : line < n0 + n1 + n2 ? a.f_next - (n0 + n1) * 64
                                                                                             : a.f_v - (n0 + n1 + n2) * 64;
    if (line < n0 + n1 + n2 + n3) warm = *reinterpret_cast<const uint32_t*>(from + line * 64u);
  }
  __builtin_amdgcn_sched_barrier(0);

  bf16x8 xf[PB][KS];
  auto frags_of = [&](const bf16_t* s) {
#pragma unroll
    for (int b = 0; b < PB; ++b)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) xf[b][ks] = lds_frag(s, LDX, 32 * b, ks * 16, lane);
  };
  // octet n (32 rows) x the tile: T form (a lane owns a position), D form (a lane owns a channel)
  auto product = [&](auto n_c, auto d_form, f32x16* acc) {
    constexpr int n = decltype(n_c)::value;
    const bf16x8* const wn = w[n % NB];
#pragma unroll
    for (int b = 0; b < PB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int b = 0; b < PB; ++b)
        acc[b] = decltype(d_form)::value ? mfma32(xf[b][ks], wn[ks], acc[b]) : mfma32(wn[ks], xf[b][ks], acc[b]);
    fetch(OCTET(n + NB));
  };
  auto sum_channels = [](float v) {
    if constexpr (CHUNKS == 16) return sum_chunks(v);
    else return group8_sum(v);
  };
  using T_form = std::false_type;
  using D_form = std::true_type;
  auto norm = [&](int which, bf16_t* dst) {
    float lw[8], lb[8];
    load_param8(sP + 2 * which * C + chunk * 8, 1.f, lw);
    load_param8(sP + (2 * which + 1) * C + chunk * 8, 0.f, lb);
#pragma unroll
    for (int u = 0; u < 2 * PB; ++u) {
      u32x4 pk = ln_pixel8<TIO, CHUNKS>(raw[u], lw, lb, false, a.lw.inv_c, a.lw.pad);
      if (!mine[u].ok) pk = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(dst + (prow + 16 * u) * LDX + chunk * 8) = pk;
    }
  };
  // T-form results -> residual stream: raw (and the tensor) become raw + results, rounded to the stream's type
  auto add_to_stream = [&](const f32x16* acc) {
#pragma unroll
    for (int b = 0; b < PB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(sS + (32 * b + j) * LDS_F + wave * 32 + 8 * g + 4 * hh) =
            f32x4{acc[b][4 * g], acc[b][4 * g + 1], acc[b][4 * g + 2], acc[b][4 * g + 3]};
    lds_barrier();
#pragma unroll
    for (int u = 0; u < 2 * PB; ++u) {
      float v[8], x[8];
      const float* s = sS + (prow + 16 * u) * LDS_F + chunk * 8;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(s), hi = *reinterpret_cast<const f32x4*>(s + 4);
      v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
      E::unpack_raw(raw[u], x);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += x[e];
      raw[u] = pack_raw<TIO>(v);
    }
  };

  *reinterpret_cast<f32x4*>(sP + tid * 4) = param;
  if (NEXT == NEXT_PROLOGUE && tid < TS) sMask[tid] = mk;
  lds_barrier();
  f32x16 acc[PB];
  // ---- gate and output projection of the operator before ----
  if constexpr (IN != IN_NONE) {
    norm(0, sA);
    if constexpr (IN == IN_EPILOGUE) {
#pragma unroll
      for (int u = 0; u < 2 * PB; ++u) {
        const int idx = tid + NT * u;
        uint32_t* const d = reinterpret_cast<uint32_t*>(sT + idx / (4 * PB) * LDT + idx % (4 * PB) * 8);
        d[0] = tt[u].x; d[1] = tt[u].y; d[2] = tt[u].z; d[3] = tt[u].w;
      }
    }
    lds_barrier();
    frags_of(sA);
    f32x16 gate[PB];
    product(OCTET(0), T_form{}, gate);
    if constexpr (IN == IN_EPILOGUE) {
      // LayerNorm of the contraction's result over its channels
      float lw[8], lb[8];
      load_param8(sP + 2 * C + chunk * 8, 1.f, lw);
      load_param8(sP + 3 * C + chunk * 8, 0.f, lb);
#pragma unroll
      for (int u = 0; u < 2 * PB; ++u) {
        const int p = prow + 16 * u, pos = t.position(p);
        float v[8], o[8], s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] = bf2f(sT[(chunk * 8 + e) * LDT + pos]);
          s1 += v[e];
        }
        const float mean = sum_channels(s1) * a.lw.inv_c;
#pragma unroll
        for (int e = 0; e < 8; ++e) { const float d = v[e] - mean; s2 = fmaf(d, d, s2); }
        const float rstd = rsqrtf((sum_channels(s2) - a.lw.pad * mean * mean) * a.lw.inv_c + LN_EPS);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = mine[u].ok ? (v[e] - mean) * rstd * lw[e] + lb[e] : 0.f;
        *reinterpret_cast<u32x4*>(sB + p * LDX + chunk * 8) = pack8(o);
      }
#pragma unroll
      for (int b = 0; b < PB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) gate[b][r] = sigmoidf_(gate[b][r]);
    } else {
      // gated attention output: the lane's registers 8 u .. are channels 32 wave + 16 u + 8 hh .. of its position
#pragma unroll
      for (int b = 0; b < PB; ++b)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          float f[8];
          unpack8(og[b][u], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] *= sigmoidf_(gate[b][8 * u + e]);
          *reinterpret_cast<u32x4*>(sB + (32 * b + j) * LDX + wave * 32 + 16 * u + 8 * hh) = own[b].ok ? pack8(f) : u32x4{0u, 0u, 0u, 0u};
        }
    }
    lds_barrier();
    frags_of(sB);
    product(OCTET(1), T_form{}, acc);
    if constexpr (IN == IN_EPILOGUE) {
#pragma unroll
      for (int b = 0; b < PB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] *= gate[b][r];
    }
    add_to_stream(acc);  // (sT was last read in front of the barrier above)
  }

  // ---- transition, a chunk of the hidden layer at a time ----
  if constexpr (TRANSITION) {
    norm(1, sA);
    lds_barrier();  // (also: the staged results have been read, the hidden layer may take their place)
    frags_of(sA);
    f32x16 sum[PB];
#pragma unroll
    for (int b = 0; b < PB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[b][r] = 0.f;
    auto hidden_chunk = [&](auto c_c) {
      constexpr int c = decltype(c_c)::value, n0 = OCT_HIDDEN + 6 * c;
      if (c > 0) lds_barrier();  // the chunk before has been multiplied
      auto block = [&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        f32x16 y[PB];
        product(OCTET(n0 + 2 * i), T_form{}, acc);
        product(OCTET(n0 + 2 * i + 1), T_form{}, y);
        if (c * (HIDDEN_CHUNK / 32) + wave + WAVES * i < n_hidden) {
#pragma unroll
          for (int b = 0; b < PB; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              float h[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) h[e] = acc[b][4 * g + e] * sigmoidf_(acc[b][4 * g + e]) * y[b][4 * g + e];
              u32x2 v;
              v.x = pack2bf(h[0], h[1]);
              v.y = pack2bf(h[2], h[3]);
              *reinterpret_cast<u32x2*>(sH + (32 * b + j) * LDH + (wave + WAVES * i) * 32 + 8 * g + 4 * hh) = v;
            }
        }
      };
      block(std::integral_constant<int, 0>{});
      block(std::integral_constant<int, 1>{});
      lds_barrier();
      // this wave's 32 channels, all units of the chunk
      auto second = [&](auto h_c) {
        constexpr int h = decltype(h_c)::value, n = n0 + 4 + h;
#pragma unroll
        for (int k = 0; k < KS; ++k)
          if (c * (HIDDEN_CHUNK / 16) + KS * h + k < nks)
#pragma unroll
            for (int b = 0; b < PB; ++b) sum[b] = mfma32(w[n % NB][k], lds_frag(sH, LDH, 32 * b, (KS * h + k) * 16, lane), sum[b]);
        fetch(OCTET(n + NB));
      };
      second(std::integral_constant<int, 0>{});
      second(std::integral_constant<int, 1>{});
    };
    hidden_chunk(std::integral_constant<int, 0>{});
    if constexpr (hidden_chunks(C) > 1) hidden_chunk(std::integral_constant<int, 1>{});
    lds_barrier();  // every wave is done with the hidden layer
    add_to_stream(sum);
  }
  if constexpr (IN != IN_NONE)
#pragma unroll
    for (int u = 0; u < 2 * PB; ++u)
      if (mine[u].ok) store_raw<TIO>(at32(pair, t.pix(mine[u]) * C + chunk * 8), raw[u]);
  asm volatile("" ::"v"(warm));
  if constexpr (NEXT == NEXT_NONE)
    if (C != 128 || !a.logits) return;

  // ---- what the next long product takes ----
  if constexpr (NEXT != NEXT_NONE) norm(2, sA);
  if constexpr (TRANSITION && C == 128)
    if (a.logits) norm(3, sB);
  lds_barrier();
  if constexpr (TRANSITION && C == 128) {
    // pair logits with quads of keys outermost, [head][key / 4][query][key % 4], keys past the end of the last quad zero
    const int quads = (a.N + 3) >> 2;
    for (int blk = wave; a.logits && blk * 32 < a.logit_heads; blk += WAVES) {
      if (blk >= WAVES) load_frags<KS>(a.f_logits, blk, KS, 0, lane, w[OCT_LOGITS % NB]);
      frags_of(sB);
#pragma unroll
      for (int b = 0; b < PB; ++b) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc[b] = mfma32(w[OCT_LOGITS % NB][ks], xf[b][ks], acc[b]);
        if (own[b].o < a.N && own[b].r < quads * 4) {
          float* const d = at32(a.logits, (uint32_t)((own[b].r >> 2) * a.N * 4 + own[b].o * 4 + (own[b].r & 3)));
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int h = blk * 32 + acc_row(r, lane);
            if (h < a.logit_heads) *at32(d, (uint32_t)(h * quads * a.N * 4)) = own[b].ok ? acc[b][r] : 0.f;
          }
        }
      }
    }
    fetch(OCTET(OCT_LOGITS + NB));
  }
  if constexpr (NEXT == NEXT_PROLOGUE) {
    frags_of(sA);
    // 32 channels (32 projection and 32 gate rows) of operand a and the same of operand b
    auto half = [&](auto h_c) {
      constexpr int h = decltype(h_c)::value;
      f32x16 g[PB];
      product(OCTET(OCT_NEXT + 2 * h), D_form{}, acc);
      product(OCTET(OCT_NEXT + 2 * h + 1), D_form{}, g);
      bf16_t* const out = at32(h ? a.b_buf : a.a_buf, (uint32_t)((wave * 32 + j) * plane));
#pragma unroll
      for (int b = 0; b < PB; ++b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 m4 = *reinterpret_cast<const f32x4*>(sMask + 32 * b + 8 * q + 4 * hh);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[b][4 * q + e] = m4[e] != 0.f ? acc[b][4 * q + e] * m4[e] * sigmoidf_(g[b][4 * q + e]) : 0.f;
        }
        if constexpr (MAP != MAP_PATCH) {
          const Pixel x = t.at(32 * b + 16 * hh);  // (a group of sixteen positions lies in one row)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = acc[b][8 * u + e];
            if (x.o < a.N && x.r + 8 * u < a.Np) *reinterpret_cast<u32x4*>(at32(out, (uint32_t)(x.o * a.Np + x.r + 8 * u))) = pack8(f);
          }
        }
      }
      if constexpr (MAP == MAP_PATCH) {
        // transposed: rows o0 .. of the pixels (., r0 + 4 hh + e)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = t.r0 + 4 * hh + e;
          uint32_t v[2 * PB];
#pragma unroll
          for (int b = 0; b < PB; ++b) {
            v[2 * b] = pack2bf(acc[b][e], acc[b][4 + e]);
            v[2 * b + 1] = pack2bf(acc[b][8 + e], acc[b][12 + e]);
          }
          if (col < a.N) {
            bf16_t* const d = at32(out, (uint32_t)(col * a.Np + t.o0));
            if constexpr (PB == 2) *reinterpret_cast<u32x4*>(d) = u32x4{v[0], v[1], v[2 * PB - 2], v[2 * PB - 1]};
            else *reinterpret_cast<u32x2*>(d) = u32x2{v[0], v[1]};
          }
        }
      }
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
  }
  if constexpr (NEXT == NEXT_PROJECT) {
    frags_of(sA);
    // a wave is one head of 32 or two of 16: q, k in T form, v in D form
    auto qk = [&](auto c_c) {
      constexpr int c = decltype(c_c)::value;
      product(OCTET(OCT_NEXT + c), T_form{}, acc);
#pragma unroll
      for (int b = 0; b < PB; ++b)
        if (own[b].ok) {
          bf16_t* const dst = at32(c == 0 ? a.q : a.k, (uint32_t)((own[b].o * H + wave * (32 / D)) * a.N + own[b].r) * D + 8 * hh);
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float f[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = c == 0 ? acc[b][8 * u + e] * a.q_scale : acc[b][8 * u + e];
            *reinterpret_cast<u32x4*>(dst + (D == 32 ? 16 * u : u * a.N * D)) = pack8(f);
          }
        }
    };
    qk(std::integral_constant<int, 0>{});
    qk(std::integral_constant<int, 1>{});
    product(OCTET(OCT_NEXT + 2), D_form{}, acc);
#pragma unroll
    for (int b = 0; b < PB; ++b) {
      // channel j of the wave's 32, positions 16 hh ..; the middle quads of a group of 16 keys change places (tri_vt_pos)
      const Pixel x = t.at(32 * b + 16 * hh);
      if (x.o < a.N) {
        bf16_t* const dst = at32(a.vt, (uint32_t)((x.o * C + wave * 32 + j) * a.ldn + x.r));
        const float lo[8] = {acc[b][0], acc[b][1], acc[b][2], acc[b][3], acc[b][8], acc[b][9], acc[b][10], acc[b][11]};
        const float hi[8] = {acc[b][4], acc[b][5], acc[b][6], acc[b][7], acc[b][12], acc[b][13], acc[b][14], acc[b][15]};
        *reinterpret_cast<u32x4*>(dst) = pack8(lo);
        *reinterpret_cast<u32x4*>(dst + 8) = pack8(hi);
      }
    }
    if (wave == 0) {
      product(OCTET(OCT_NEXT + 3), T_form{}, acc);
#pragma unroll
      for (int b = 0; b < PB; ++b)
        if (hh == 0 && own[b].ok) {
          const int q = MAP == MAP_COLUMNS ? own[b].r : own[b].o, k = MAP == MAP_COLUMNS ? own[b].o : own[b].r;
#pragma unroll
          for (int h = 0; h < H; ++h) *at32(a.bias, (uint32_t)tri_bias_offset(a.N, h, q, k)) = f2h_sat(acc[b][h] * a.bias_scale);
          // keys past N in the last key tile read as zero bias: the tile's real keys share them out
          const int k_last = (a.N - 1) & ~63, real = a.N - k_last;
          if (k >= k_last)
            for (int kp = a.N + k - k_last; kp < k_last + 64; kp += real)
#pragma unroll
              for (int h = 0; h < H; ++h) *at32(a.bias, (uint32_t)tri_bias_offset(a.N, h, q, kp)) = 0;
        }
    }
  }
#undef OCTET
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Patches of 8 x 8 pixels from one workgroup per CU on: what a patch writes of a transposed operand is then whole 16-byte
// pieces.
constexpr int64_t WIDE_PATCHES = 256 * 64;
// Projections behind an epilogue or an output in tiles of 64 positions: half of the weights' traffic, where there are rounds of
// workgroups enough (two a CU against three); us, 32 / 64 positions, 160 tokens 19.1 / 19.5 (epilogue), 18.8 / 18.3 (output), 208
// 24.6 / 27.0, 23.9 / 25.3, 240 30.5 / 29.3, 29.2 / 28.8, 301 44.0 / 41.8, 42.4 / 40.7, 400 68.6 / 64.3, 66.9 / 63.6.
constexpr int64_t WIDE_ROWS = 208 * 208 + 1;
// ... and between three tiles of 32 to a CU and three and a half a fourth workgroup instead of a second round of a few: three / four,
// 157 tokens (785 tiles) 19.3 / 17.7 (epilogue), 18.0 / 17.4 (output), 160 (800) 18.7 / 17.0, 17.3 / 16.7, 176 (968) 20.2 / 20.5, 17.8 /
// 18.5.  Its 128 registers leave one piece of the weights in flight, which costs where it saves no round: 64 tokens 7.6 / 7.9, 7.8 /
// 8.0, 130 15.8 / 15.5, 15.4 / 16.6, 200 (1300) 23.2 / 23.7, 23.0 / 23.4.
bool four_a_simd(int64_t positions) { return positions > 32 * 3 * 256 && positions <= 32 * 7 * 128; }
// The steps with a transition: tiles of 32 positions, two or three workgroups to a CU, or tiles of 64 (half of the weights'
// traffic), two to a CU, by the rounds that they make on 256 CUs; us, with the next prologue, two / three / wide: 128 tokens (512
// tiles of 32) 22.8 / 23.2 / 25.0, 152 (760) 31.2 / 29.1 / 31.2, 160 (800) 36.4 / 36.0 / 31.6, 181 (1086, wide ones 543) 45.1 / 43.1 /
// 46.7, 192 (1152) 45.8 / 42.8 / 46.6, 208 (1352) 52.7 / 49.3 / 48.2.
enum TransitionForm { TWO_A_SIMD, THREE_A_SIMD, WIDE };
TransitionForm transition_form(int64_t positions) {
  const int64_t tiles = (positions + 31) / 32;
  if (tiles <= 2 * 256) return TWO_A_SIMD;
  return tiles <= 3 * 256 || (tiles > 4 * 256 && tiles <= 5 * 256) ? THREE_A_SIMD : WIDE;
}

template <int CH, int PB, int IN, int MAP, bool TRANSITION, int NEXT, int PER_SIMD = CH == 64 ? 4 : PB == 2 ? 2 : 3>
int launch_tiles(const PairStepArgs& a, hipStream_t s) {
  const int64_t blocks = MAP == MAP_PATCH ? ((int64_t)(a.Np / (4 * PB)) * (a.Np / 8) + 7) / 8 * 8
                                          : ((int64_t)a.N * a.ldn + 32 * PB - 1) / (32 * PB);
  if (blocks <= 0 || blocks > 0x7fffffff) return AF3_ERR_BAD_ARG;
  const dim3 grid((unsigned)blocks), block(2 * CH);
  if (a.io_f32) hipLaunchKernelGGL((pair_step_kernel<float, CH, PB, IN, MAP, TRANSITION, NEXT, PER_SIMD>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((pair_step_kernel<bf16_t, CH, PB, IN, MAP, TRANSITION, NEXT, PER_SIMD>), grid, block, 0, s, a);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
}  // namespace

int launch_pair_step(const PairStepArgs& a, int step, hipStream_t s) {
  if (a.N <= 0 || a.N > 8192 || a.Np < a.N || (a.Np & 7) || a.ldn != tri_ldn(a.N) || !a.pair || !al16(a.pair) ||
      (a.channels != 128 && a.channels != 64) || a.valid_c < 1 || a.valid_c > a.channels)
    return AF3_ERR_BAD_ARG;
  // every array is addressed with 32 bits
  if (a.plane * a.channels * 2 >= (1ll << 32) || (int64_t)a.N * a.ldn * a.channels * (a.io_f32 ? 4 : 2) >= (1ll << 32))
    return AF3_ERR_BAD_ARG;
  const bool first = step == PAIR_STEP_FIRST, epilogue = step == PAIR_STEP_INCOMING || step == PAIR_STEP_PROJECT_START;
  const bool prologue = first || step == PAIR_STEP_INCOMING || step == PAIR_STEP_NEXT;
  const bool project = step == PAIR_STEP_PROJECT_START || step == PAIR_STEP_PROJECT_END, transition = step >= PAIR_STEP_LAST;
  if (!first && (!a.f_gate || !a.f_out || !a.ln1_w || !a.ln1_b || !al16(a.f_gate) || !al16(a.f_out))) return AF3_ERR_BAD_ARG;
  if (epilogue && (!a.t_buf || !a.ln_c_w || !a.ln_c_b || a.plane < tri_plane(a.N))) return AF3_ERR_BAD_ARG;
  if (!epilogue && !first && !a.og) return AF3_ERR_BAD_ARG;
  if (prologue && (!a.a_buf || !a.b_buf || !a.f_next || !a.ln3_w || !a.ln3_b || a.plane < tri_plane(a.N))) return AF3_ERR_BAD_ARG;
  if (project && (!a.q || !a.k || !a.vt || !a.bias || !a.f_next || !a.f_v || !a.ln3_w || !a.ln3_b)) return AF3_ERR_BAD_ARG;
  if (transition && (!a.f_w1 || !a.f_w2 || !a.ln2_w || !a.ln2_b || a.hidden <= 0 || (a.hidden & 63) ||
                     a.hidden > pair_step_max_hidden(a.channels)))
    return AF3_ERR_BAD_ARG;
  if (a.logits && (a.channels != 128 || !transition || !a.f_logits || !a.sl_ln_w || !a.sl_ln_b || a.logit_heads <= 0))
    return AF3_ERR_BAD_ARG;
  const int64_t positions = (int64_t)a.N * a.ldn;
  const TransitionForm form = transition_form(positions);
  if (a.channels == 64) switch (step) {
    case PAIR_STEP_FIRST: return launch_tiles<64, 1, IN_NONE, MAP_ROWS, false, NEXT_PROLOGUE>(a, s);
    case PAIR_STEP_INCOMING: return launch_tiles<64, 1, IN_EPILOGUE, MAP_PATCH, false, NEXT_PROLOGUE>(a, s);
    case PAIR_STEP_PROJECT_START: return launch_tiles<64, 1, IN_EPILOGUE, MAP_ROWS, false, NEXT_PROJECT>(a, s);
    case PAIR_STEP_PROJECT_END: return launch_tiles<64, 1, IN_ATTENTION, MAP_COLUMNS, false, NEXT_PROJECT>(a, s);
    case PAIR_STEP_LAST: return launch_tiles<64, 1, IN_ATTENTION, MAP_ROWS, true, NEXT_NONE>(a, s);
    case PAIR_STEP_NEXT: return launch_tiles<64, 1, IN_ATTENTION, MAP_ROWS, true, NEXT_PROLOGUE>(a, s);
  }
  else switch (step) {
    case PAIR_STEP_INCOMING:
      if ((int64_t)a.N * a.ldn >= WIDE_PATCHES) return launch_tiles<128, 2, IN_EPILOGUE, MAP_PATCH, false, NEXT_PROLOGUE>(a, s);
      return launch_tiles<128, 1, IN_EPILOGUE, MAP_PATCH, false, NEXT_PROLOGUE>(a, s);
    case PAIR_STEP_PROJECT_START:
      if (positions >= WIDE_ROWS) return launch_tiles<128, 2, IN_EPILOGUE, MAP_ROWS, false, NEXT_PROJECT>(a, s);
      if (four_a_simd(positions)) return launch_tiles<128, 1, IN_EPILOGUE, MAP_ROWS, false, NEXT_PROJECT, 4>(a, s);
      return launch_tiles<128, 1, IN_EPILOGUE, MAP_ROWS, false, NEXT_PROJECT>(a, s);
    case PAIR_STEP_PROJECT_END:
      if (positions >= WIDE_ROWS) return launch_tiles<128, 2, IN_ATTENTION, MAP_COLUMNS, false, NEXT_PROJECT>(a, s);
      if (four_a_simd(positions)) return launch_tiles<128, 1, IN_ATTENTION, MAP_COLUMNS, false, NEXT_PROJECT, 4>(a, s);
      return launch_tiles<128, 1, IN_ATTENTION, MAP_COLUMNS, false, NEXT_PROJECT>(a, s);
    case PAIR_STEP_LAST:
      if (form == TWO_A_SIMD) return launch_tiles<128, 1, IN_ATTENTION, MAP_ROWS, true, NEXT_NONE, 2>(a, s);
      if (form == THREE_A_SIMD) return launch_tiles<128, 1, IN_ATTENTION, MAP_ROWS, true, NEXT_NONE>(a, s);
      return launch_tiles<128, 2, IN_ATTENTION, MAP_ROWS, true, NEXT_NONE>(a, s);
    case PAIR_STEP_NEXT:
      if (form == TWO_A_SIMD) return launch_tiles<128, 1, IN_ATTENTION, MAP_ROWS, true, NEXT_PROLOGUE, 2>(a, s);
      if (form == THREE_A_SIMD) return launch_tiles<128, 1, IN_ATTENTION, MAP_ROWS, true, NEXT_PROLOGUE>(a, s);
      return launch_tiles<128, 2, IN_ATTENTION, MAP_ROWS, true, NEXT_PROLOGUE>(a, s);
  }
  return AF3_ERR_BAD_ARG;
}
