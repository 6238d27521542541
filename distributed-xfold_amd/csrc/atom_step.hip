// What an atom transformer block (128 channels) does row by row, between one window attention and the next, in one kernel:
//
//   tail: output projection, AdaLN-Zero gate, residual;  adaptive LayerNorm, SwiGLU transition (at most 256 hidden units),
//         gate, residual; in place on the activations
//   head: the adaptive LayerNorms of the row as a query and as a key;  q and gate, k and v
//
// As seven kernels (two norms, four products, two of them with a gate and a residual, and the SwiGLU product) every row
// went to memory and back five times and the hidden layer once, and at few atoms each was a launch of a few us in a chain.
// Here a workgroup keeps 32 rows; its four waves own 32 output channels each and stream the weights' fragments (frags of
// af3_diffusion_block) from L2, a stage ahead.  Values are rounded where the separate kernels store them and every sum
// has their order, so the results are the same bits.
//
// What bounds it: with many rows memory (92160 rows: 117 MB in and out of the tail with its conditioning, 133 MB more of
// the head) and the weights, 0.36 MB a tile; with few, the tile's chain.  us, as one kernel and as those
// before it, 92160 rows / 12000: tail 49 (24 + 20 + 28 + 26) / 10.7 (6.8 + 6.3 + 6.6 + 8.0), head 53 (24 + 28 + 17) / 12.1
// (6.3 + 6.8 + 6.6), both 91 / 18.5.  (Operands stored from the accumulators, 32 bytes of a row at a time: both 95.)
// Tiles of 64 rows, which halve the weights, do not fit the registers (tail: 89 us against 49).
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int HIDDEN = ATOM_STEP_MAX_HIDDEN;

// sum over 16 lanes, neighbours first (ln_rows_small_kernel's order)
__device__ __forceinline__ float sum16(float v) {
  v = group8_sum(v);
  return v + dpp_mov<0x128>(v);  // row_ror:8
}

template <typename TIO, bool TAIL, bool HEAD>
__global__ __launch_bounds__(256, 2) void atom_step_kernel(AtomStepArgs a) {
  using E = Elem<TIO>;
  constexpr int TS = 32, NB = 3, LDH = HIDDEN + 8;
  constexpr int U_BYTES = TS * LDS_F * 4;
  static_assert(U_BYTES >= TS * LDH * 2, "the hidden layer fits the staging tile");
  __shared__ __attribute__((aligned(16))) bf16_t sA[TS * LDX];
  __shared__ __attribute__((aligned(16))) bf16_t sB[HEAD ? TS * LDX : 8];
  __shared__ __attribute__((aligned(16))) char sU[U_BYTES];
  float* const sS = reinterpret_cast<float*>(sU);    // staged fp32 results, [row][channel]
  bf16_t* const sH = reinterpret_cast<bf16_t*>(sU);  // the hidden layer, [row][unit]
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chunk = tid & 15, prow = tid >> 4;

  // The samples' rows of the same atoms, which share their conditioning, run back to back on one XCD.
  const int all = (a.atoms + TS - 1) / TS, tiles = a.tiles ? min(a.tiles[0], all) : all, total = tiles * a.samples, per = (total + 7) >> 3;
  const int idx = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || idx >= total) return;
  const int place = __builtin_amdgcn_readfirstlane(idx / a.samples), sample = __builtin_amdgcn_readfirstlane(idx % a.samples);
  const int tile = a.tiles ? a.tiles[1 + place] : place;
  if ((unsigned)tile >= (unsigned)all) return;
  const int a0 = tile * TS;
  TIO* const act = reinterpret_cast<TIO*>(a.act) + (int64_t)sample * a.atoms * C;
  const bf16_t* const y = a.y + (int64_t)sample * a.atoms * C;
  int atom[2];
  bool ok[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    ok[u] = a0 + prow + 16 * u < a.atoms;
    atom[u] = min(a0 + prow + 16 * u, a.atoms - 1);
  }

  u32x4 yv[2];
  typename E::Raw raw[2];
  f32x4 gate[2][2];
  auto load_gate = [&](const float* g) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float* p = g + (int64_t)atom[u] * C + chunk * 8;
      gate[u][0] = *reinterpret_cast<const f32x4*>(p);
      gate[u][1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
  };
  if constexpr (TAIL)
#pragma unroll
    for (int u = 0; u < 2; ++u) yv[u] = *reinterpret_cast<const u32x4*>(y + (int64_t)atom[u] * C + chunk * 8);
#pragma unroll
  for (int u = 0; u < 2; ++u) raw[u] = E::load_raw(act + (int64_t)atom[u] * C + chunk * 8);

  // The wave's weights, 32 rows x 8 k-steps at a time, in the order of their use: output projection; two hidden blocks of
  // 32 units, "a" rows and "b" rows; its 32 channels of the second layer in two halves of K; of q, the gate, k and v
  constexpr int HEAD0 = TAIL ? 7 : 0, PIECES = HEAD0 + (HEAD ? 4 : 0);
  const int n_hidden = a.hidden >> 5, nks = a.hidden >> 4;
  bf16x8 w[NB][8];
  auto fetch = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < PIECES) {
      bf16x8* const d = w[n % NB];
      if constexpr (n >= HEAD0) load_frags<8>(a.f_head, 4 * (n - HEAD0) + wave, 8, 0, lane, d);
      else if constexpr (n == 0) load_frags<8>(a.f_out, wave, 8, 0, lane, d);
      else if constexpr (n < 5) load_frags<8>(a.f_w1, 2 * min(wave + 4 * ((n - 1) >> 1), n_hidden - 1) + ((n - 1) & 1), 8, 0, lane, d);
      else {
        constexpr int k0 = (n - 5) * 8;  // (k-steps come in fours)
        load_frags<4>(a.f_w2, wave, nks, min(k0, nks - 4), lane, d);
        load_frags<4>(a.f_w2, wave, nks, min(k0 + 4, nks - 4), lane, d + 4);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#define PIECE(n) std::integral_constant<int, (n)>{}
  fetch(PIECE(0));
  if constexpr (TAIL) load_gate(a.gate1);
  fetch(PIECE(1));
  fetch(PIECE(2));

  bf16x8 xf[8];
  auto frags_of = [&](const bf16_t* s) {
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) xf[ks] = lds_frag(s, LDX, 0, ks * 16, lane);
  };
  auto product = [&](auto n_c, f32x16& acc) {  // a lane owns a row
    constexpr int n = decltype(n_c)::value;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) acc = mfma32(w[n % NB][ks], xf[ks], acc);
    fetch(PIECE(n + NB));
  };
  // raw = gate * results + raw, rounded to the stream's type
  auto add_to_stream = [&](const f32x16& acc) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(sS + j * LDS_F + wave * 32 + 8 * g + 4 * hh) = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    lds_barrier();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float v[8], x[8];
      const float* s = sS + (prow + 16 * u) * LDS_F + chunk * 8;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(s), hi = *reinterpret_cast<const f32x4*>(s + 4);
      E::unpack_raw(raw[u], x);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (e < 4 ? lo[e & 3] : hi[e & 3]) * gate[u][e >> 2][e & 3] + x[e];
      raw[u] = pack_raw<TIO>(v);
    }
  };

  f32x4 cond[2][4];  // of this thread's rows: scale, shift
  auto load_cond = [&](const float* from, int64_t ld, f32x4 (&to)[2][4]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float* p = from + (int64_t)atom[u] * ld + chunk * 8;
      to[u][0] = *reinterpret_cast<const f32x4*>(p);
      to[u][1] = *reinterpret_cast<const f32x4*>(p + 4);
      to[u][2] = *reinterpret_cast<const f32x4*>(p + C);
      to[u][3] = *reinterpret_cast<const f32x4*>(p + C + 4);
    }
  };
  // adaptive LayerNorm of raw into `to`, and with a second conditioning into `to2`
  auto norm = [&](const f32x4 (&c1)[2][4], bf16_t* to, const f32x4 (*c2)[4], bf16_t* to2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float v[8], o[8], s = 0.f, q = 0.f;
      E::unpack_raw(raw[u], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[e];
      const float mean = sum16(s) / (float)C;
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = v[e] - mean; q += d * d; }
      const float rstd = rsqrtf(sum16(q) / (float)C + LN_EPS);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float t = (v[e] - mean) * rstd;
        o[e] = sigmoidf_(c1[u][e >> 2][e & 3]) * t + c1[u][2 + (e >> 2)][e & 3];
      }
      *reinterpret_cast<u32x4*>(to + (prow + 16 * u) * LDX + chunk * 8) = pack8(o);
      if (!to2) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float t = (v[e] - mean) * rstd;
        o[e] = sigmoidf_(c2[u][e >> 2][e & 3]) * t + c2[u][2 + (e >> 2)][e & 3];
      }
      *reinterpret_cast<u32x4*>(to2 + (prow + 16 * u) * LDX + chunk * 8) = pack8(o);
    }
  };
  f32x16 acc;
  f32x4 cond_k[2][4];

  if constexpr (TAIL) {
    // ---- output projection ----
#pragma unroll
    for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4*>(sA + (prow + 16 * u) * LDX + chunk * 8) = yv[u];
    lds_barrier();
    frags_of(sA);
    f32x16 second;
    product(PIECE(0), acc);
    load_cond(a.scale, a.ld_cond, cond);
    add_to_stream(acc);  // (its barrier: every wave has read the attention's tile)

    // ---- transition ----
    norm(cond, sA, nullptr, nullptr);
    load_gate(a.gate2);
    lds_barrier();  // (also: the staged results have been read, the hidden layer may take their place)

    frags_of(sA);
    auto block = [&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      product(PIECE(1 + 2 * i), acc);
      product(PIECE(2 + 2 * i), second);
      if (wave + 4 * i < n_hidden) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float h[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = acc[4 * g + e] * sigmoidf_(acc[4 * g + e]) * second[4 * g + e];
          u32x2 v;
          v.x = pack2bf(h[0], h[1]);
          v.y = pack2bf(h[2], h[3]);
          *reinterpret_cast<u32x2*>(sH + j * LDH + (wave + 4 * i) * 32 + 8 * g + 4 * hh) = v;
        }
      }
    };
    block(std::integral_constant<int, 0>{});
    block(std::integral_constant<int, 1>{});
    lds_barrier();
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    auto half = [&](auto h_c) {
      constexpr int h = decltype(h_c)::value;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (8 * h + k < nks) acc = mfma32(w[(5 + h) % NB][k], lds_frag(sH, LDH, 0, (8 * h + k) * 16, lane), acc);
      fetch(PIECE(5 + h + NB));
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
    if constexpr (HEAD) {
      load_cond(a.scale_q, a.ld_cond, cond);
      load_cond(a.scale_k, a.ld_cond_k, cond_k);
    }
    lds_barrier();  // every wave is done with the hidden layer
    add_to_stream(acc);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (ok[u]) store_raw<TIO>(act + (int64_t)atom[u] * C + chunk * 8, raw[u]);
  }

  // ---- the next attention's operands ----
  if constexpr (HEAD) {
    if constexpr (!TAIL) {
      load_cond(a.scale_q, a.ld_cond, cond);
      load_cond(a.scale_k, a.ld_cond_k, cond_k);
    }
    // the lane's registers 8 u .. are channels 32 wave + 16 u + 8 hh .. of row j
    const int c0 = wave * 32 + 8 * hh;
    float bias[16];
#pragma unroll
    for (int u = 0; u < 2; ++u) load_param8(a.q_bias ? a.q_bias + c0 + 16 * u : nullptr, 0.f, bias + 8 * u);
    norm(cond, sA, cond_k, sB);
    lds_barrier();
    // q and gate, then k and v, go out through LDS: 512 bytes of a row at a time
    constexpr int LDO = 2 * C + 8;
    static_assert(U_BYTES >= TS * LDO * 2, "two operands fit the staging tile");
    bf16_t* const sO = reinterpret_cast<bf16_t*>(sU);
    auto store_rows = [&](bf16_t* out) {
      lds_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = (tid >> 5) + 8 * i, at = (tid & 31) * 8;
        const u32x4 v = *reinterpret_cast<const u32x4*>(sO + r * LDO + at);
        if (a0 + r < a.atoms) *reinterpret_cast<u32x4*>(out + ((int64_t)sample * a.atoms + a0 + r) * (2 * C) + at) = v;
      }
    };
    auto operand = [&](auto n_c) {
      constexpr int n = decltype(n_c)::value;
      product(PIECE(HEAD0 + n), acc);
      if (n == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = (acc[r] + bias[r]) * a.q_scale;
      } else if (n == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = sigmoidf_(acc[r]);
      }
      if (n == 2) lds_barrier();  // q and gate have been read
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = acc[8 * u + e];
        *reinterpret_cast<u32x4*>(sO + j * LDO + (n & 1) * C + c0 + 16 * u) = pack8(f);
      }
    };
    frags_of(sA);
    operand(std::integral_constant<int, 0>{});
    operand(std::integral_constant<int, 1>{});
    store_rows(a.qg);
    frags_of(sB);
    operand(std::integral_constant<int, 2>{});
    operand(std::integral_constant<int, 3>{});
    store_rows(a.kv);
  }
#undef PIECE
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

bool atom_steps_apply(const AtomStepArgs& a) {
  return a.act && a.y && a.f_out && a.f_w1 && a.f_w2 && a.gate1 && a.gate2 && a.scale && a.scale_q && a.scale_k && a.f_head &&
         a.qg && a.kv && a.atoms > 0 && a.samples > 0 && a.hidden > 0 && a.hidden <= HIDDEN && a.hidden % 64 == 0 &&
         a.ld_cond >= 2 * C && a.ld_cond % 4 == 0 && a.ld_cond_k >= 2 * C && a.ld_cond_k % 4 == 0 && al16(a.act) && al16(a.y) &&
         al16(a.f_out) && al16(a.f_head) && al16(a.gate1) && al16(a.gate2) && al16(a.scale) && al16(a.scale_q) && al16(a.scale_k) &&
         al16(a.qg) && al16(a.kv) && al16(a.q_bias);
}

int launch_atom_step(const AtomStepArgs& a, bool tail, bool head, hipStream_t s) {
  if (!atom_steps_apply(a) || !(tail || head)) return AF3_ERR_BAD_ARG;
  const int64_t blocks = (((int64_t)a.atoms + 31) / 32 * a.samples + 7) / 8 * 8;
  if (blocks > 0x7fffffff) return AF3_ERR_BAD_ARG;
  const dim3 grid((unsigned)blocks), block(256);
#define LAUNCH(TAIL, HEAD)                                                                            \
  do {                                                                                                \
    if (a.io_f32) hipLaunchKernelGGL((atom_step_kernel<float, TAIL, HEAD>), grid, block, 0, s, a);    \
    else hipLaunchKernelGGL((atom_step_kernel<bf16_t, TAIL, HEAD>), grid, block, 0, s, a);            \
  } while (0)
  if (!tail) LAUNCH(false, true);
  else if (head) LAUNCH(true, true);
  else LAUNCH(true, false);
#undef LAUNCH
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
