// The per-row tail of an atom transformer block (128 channels), one kernel, in place on the activations:
//
//   output projection, AdaLN-Zero gate, residual;  adaptive LayerNorm, SwiGLU transition (at most 256 hidden units), gate, residual
//
// As four kernels (two products with a gate and a residual, the norm, the SwiGLU product) every row went to memory and back
// three times and the hidden layer once, and at few atoms each was a launch of a few us in a chain.  Here a workgroup
// keeps 32 rows; its four waves own 32 output channels each and stream the weights' fragments (frags of
// af3_diffusion_block) from L2, a stage ahead.  Values are rounded where the separate kernels store them and every sum
// has their order, so the results are the same bits.
//
// What bounds it: with many rows memory (92160 rows: 117 MB in and out with the conditioning) and the weights, 0.23 MB a
// tile; with few, the tile's chain.  92160 rows 49 us (24 + 20 + 28 + 26 before), 12000 rows 13 (6.8 + 6.3 + 6.6 + 8.0).
// Tiles of 64 rows, which halve the weights, do not fit the registers: 89 us.
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

template <typename TIO>
__global__ __launch_bounds__(256, 2) void atom_tail_kernel(AtomStepArgs a) {
  using E = Elem<TIO>;
  constexpr int TS = 32, NB = 3, LDH = HIDDEN + 8;
  constexpr int U_BYTES = TS * LDS_F * 4;
  static_assert(U_BYTES >= TS * LDH * 2, "the hidden layer fits the staging tile");
  __shared__ __attribute__((aligned(16))) bf16_t sA[TS * LDX];
  __shared__ __attribute__((aligned(16))) char sU[U_BYTES];
  float* const sS = reinterpret_cast<float*>(sU);    // staged fp32 results, [row][channel]
  bf16_t* const sH = reinterpret_cast<bf16_t*>(sU);  // the hidden layer, [row][unit]
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chunk = tid & 15, prow = tid >> 4;

  // The samples' rows of the same atoms, which share their conditioning, run back to back on one XCD.
  const int tiles = (a.atoms + TS - 1) / TS, total = tiles * a.samples, per = (total + 7) >> 3;
  const int idx = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || idx >= total) return;
  const int a0 = __builtin_amdgcn_readfirstlane(idx / a.samples) * TS, sample = __builtin_amdgcn_readfirstlane(idx % a.samples);
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
#pragma unroll
  for (int u = 0; u < 2; ++u) yv[u] = *reinterpret_cast<const u32x4*>(y + (int64_t)atom[u] * C + chunk * 8);
#pragma unroll
  for (int u = 0; u < 2; ++u) raw[u] = E::load_raw(act + (int64_t)atom[u] * C + chunk * 8);

  // The wave's weights, 32 rows x 8 k-steps at a time, in the order of their use: output projection; two hidden blocks of
  // 32 units, "a" rows and "b" rows; its 32 channels of the second layer in two halves of K
  constexpr int PIECES = 7;
  const int n_hidden = a.hidden >> 5, nks = a.hidden >> 4;
  bf16x8 w[NB][8];
  auto fetch = [&](auto n_c) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n < PIECES) {
      bf16x8* const d = w[n % NB];
      if constexpr (n == 0) load_frags<8>(a.f_out, wave, 8, 0, lane, d);
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
  load_gate(a.gate1);
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

  // ---- output projection ----
#pragma unroll
  for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4*>(sA + (prow + 16 * u) * LDX + chunk * 8) = yv[u];
  lds_barrier();
  frags_of(sA);
  f32x16 acc, second;
  product(PIECE(0), acc);
  f32x4 cond[2][4];  // scale, shift
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float* p = a.scale + (int64_t)atom[u] * a.ld_cond + chunk * 8;
    cond[u][0] = *reinterpret_cast<const f32x4*>(p);
    cond[u][1] = *reinterpret_cast<const f32x4*>(p + 4);
    cond[u][2] = *reinterpret_cast<const f32x4*>(p + C);
    cond[u][3] = *reinterpret_cast<const f32x4*>(p + C + 4);
  }
  add_to_stream(acc);  // (its barrier: every wave has read the attention's tile)

  // ---- adaptive LayerNorm ----
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
      o[e] = sigmoidf_(cond[u][e >> 2][e & 3]) * t + cond[u][2 + (e >> 2)][e & 3];
    }
    *reinterpret_cast<u32x4*>(sA + (prow + 16 * u) * LDX + chunk * 8) = pack8(o);
  }
  load_gate(a.gate2);
  lds_barrier();  // (also: the staged results have been read, the hidden layer may take their place)

  // ---- transition ----
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
  };
  half(std::integral_constant<int, 0>{});
  half(std::integral_constant<int, 1>{});
  lds_barrier();  // every wave is done with the hidden layer
  add_to_stream(acc);
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (ok[u]) store_raw<TIO>(act + (int64_t)atom[u] * C + chunk * 8, raw[u]);
#undef PIECE
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

bool atom_tail_applies(const AtomStepArgs& a) {
  return a.act && a.y && a.f_out && a.f_w1 && a.f_w2 && a.gate1 && a.gate2 && a.scale && a.atoms > 0 && a.samples > 0 &&
         a.hidden > 0 && a.hidden <= HIDDEN && a.hidden % 64 == 0 && a.ld_cond >= 2 * C && a.ld_cond % 4 == 0 && al16(a.act) &&
         al16(a.y) && al16(a.f_out) && al16(a.gate1) && al16(a.gate2) && al16(a.scale);
}

int launch_atom_tail(const AtomStepArgs& a, hipStream_t s) {
  if (!atom_tail_applies(a)) return AF3_ERR_BAD_ARG;
  const int64_t blocks = (((int64_t)a.atoms + 31) / 32 * a.samples + 7) / 8 * 8;
  if (blocks > 0x7fffffff) return AF3_ERR_BAD_ARG;
  const dim3 grid((unsigned)blocks), block(256);
  if (a.io_f32) hipLaunchKernelGGL((atom_tail_kernel<float>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((atom_tail_kernel<bf16_t>), grid, block, 0, s, a);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
