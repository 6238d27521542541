// The SwiGLU transition of rows of 384 channels on an fp32 stream (the diffusion head's single conditionings, a row per token and
// noise level), in place: LayerNorm, both products and the residual in one pass over the rows.
//
// As a norm and two products the rows' normalised copy and the hidden layer, twice as wide, go to memory and come back: 76800 rows
// 0.6 GB in 260 us.  Here a workgroup takes 64 rows: normalised, they stay in LDS (48 KB); 128 hidden units at a time are multiplied,
// gated, put into LDS (16 KB) and multiplied with their part of the second matrix, whose sums stay in registers.  A wave takes 32 of
// the units and 96 of the channels, for all rows, so that a weight passes once through the CU; the fragments (16 rows of 4 k-steps of
// either factor, or 2 k-steps of the 96 channels: 8 KB) come from L2 straight into registers, a piece ahead of the one that is
// multiplied.  Values are rounded where the separate kernels store them.
//
// 250 registers, two workgroups to a CU.  What bounds it: 1.8 MB of weights a tile through the CU's vector memory path and, about
// equally, the matrix unit at the clock that it leaves (76800 rows 0.84 PFLOP/s; 134 us without matrix instructions, 137 without
// weights and LDS reads, in the run in which all was 177), and the ends of a tile, which at 2.3 rounds of workgroups coincide.  us, norm
// and two products / this: 8192 rows 36 / 33, 16384 58 / 39, 30000 101 / 70, 76800 258 / 163, 307200 1078 / 640.  (Matrix phases at a
// higher priority, or every second workgroup begun later: the same.)
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int CH = ROW_TRANSITION_CHANNELS, TS = 64, SLABS = CH / 64, KS = CH / 16;
constexpr int CHUNK = 128, PIECES = KS / 4 + CHUNK / 32;  // of the weights, in a chunk
constexpr int SLAB = TS * 128, LDF = CH + 4;               // a slab of 64 channels, [row][128 bytes]; fp32 results of 32 rows

__global__ __launch_bounds__(256, 2) void row_transition_kernel(RowTransitionArgs a) {
  // chunk c (16 bytes) of a slab's row lies at position c ^ (row / 2 % 8)
  __shared__ __attribute__((aligned(1024))) char sX[SLABS * SLAB + CHUNK / 64 * SLAB];
  char* const sH = sX + SLABS * SLAB;
  float* const sF = reinterpret_cast<float*>(sX);
  static_assert(sizeof(sX) >= 32 * LDF * 4, "the results of 32 rows fit");
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = (int)blockIdx.x * TS, last = a.rows - 1 - m0;  // (of the tile's rows; what lies behind it is a copy of it)
  float* const act = a.act + (int64_t)m0 * CH;

  // the rows: lane s of a group of sixteen takes chunks s, s + 16 and s + 32 of rows g, g + 16, ..
  const int sub = tid & 15, grp = tid >> 4;
  Elem<float>::Raw raw[4][3];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int i = 0; i < 3; ++i) raw[u][i] = Elem<float>::load_raw(act + min(grp + 16 * u, last) * CH + (sub + 16 * i) * 8);
  const int chunks = a.hidden / CHUNK, nks = a.hidden / 16;
  bf16x8 w[2][8];
  auto fetch = [&](auto n_c, int c) {
    constexpr int n = decltype(n_c)::value % PIECES;
    c = min(c + decltype(n_c)::value / PIECES, chunks - 1);
    bf16x8* const d = w[n & 1];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (n < KS / 4) {
#pragma unroll
      for (int f = 0; f < 2; ++f) load_frags<4>(a.w1, (c * (CHUNK / 32) + wave) * 2 + f, KS, 4 * n, lane, d + 4 * f);
    } else {
#pragma unroll
      for (int q = 0; q < 3; ++q) load_frags<2>(a.w2, 3 * wave + q, nks, c * (CHUNK / 16) + 2 * (n - KS / 4), lane, d + 2 * q);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#define PIECE(n) std::integral_constant<int, (n)>{}
  static_assert(PIECES % 2 == 0, "the ring starts anew with every chunk");
  fetch(PIECE(0), 0);
  {
    float lw[3][8], lb[3][8];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      Elem<float>::load8(a.ln_w + (sub + 16 * i) * 8, lw[i]);
      Elem<float>::load8(a.ln_b + (sub + 16 * i) * 8, lb[i]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float v[3][8], s = 0.f, q = 0.f;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        Elem<float>::unpack_raw(raw[u][i], v[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[i][e];
      }
      const float mean = group16_sum(s) * (1.f / CH);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] -= mean;
        q = add_squares8(v[i], q, i == 0);
      }
      const float rstd = rsqrtf(group16_sum(q) * (1.f / CH) + LN_EPS);
      const int row = grp + 16 * u;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = v[i][e] * rstd * lw[i][e] + lb[i][e];
        const int chunk = sub + 16 * i;
        *reinterpret_cast<u32x4*>(sX + (chunk >> 3) * SLAB + row * 128 + (((chunk & 7) ^ ((row >> 1) & 7)) << 4)) = pack8(o);
      }
    }
  }
  fetch(PIECE(1), 0);
  lds_barrier();

  auto frag = [&](const char* slabs, int b, int ks) {
    return as_frag(*reinterpret_cast<const u32x4*>(slabs + (ks >> 2) * SLAB + (32 * b + j) * 128 + (((2 * (ks & 3) + hh) ^ ((j >> 1) & 7)) << 4)));
  };
  f32x16 sum[3][2];
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[q][b][r] = 0.f;
  for (int c = 0; c < chunks; ++c) {
    f32x16 acc[2][2];  // [factor][32 rows]
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[f][b][r] = 0.f;
    auto first = [&](auto n_c) {
      constexpr int n = decltype(n_c)::value;
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const bf16x8 x = frag(sX, b, 4 * n + k);
#pragma unroll
          for (int f = 0; f < 2; ++f) acc[f][b] = mfma32(w[n & 1][4 * f + k], x, acc[f][b]);
        }
      fetch(PIECE(n + 2), c);
    };
    first(PIECE(0)); first(PIECE(1)); first(PIECE(2)); first(PIECE(3)); first(PIECE(4)); first(PIECE(5));
    lds_barrier();  // the chunk before has been multiplied
    // registers 8 u .. of row 32 b + j are units 32 wave + 16 u + 8 hh ..
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = acc[0][b][8 * u + e] * sigmoidf_(acc[0][b][8 * u + e]) * acc[1][b][8 * u + e];
        *reinterpret_cast<u32x4*>(sH + (wave >> 1) * SLAB + (32 * b + j) * 128 + (((4 * (wave & 1) + 2 * u + hh) ^ ((j >> 1) & 7)) << 4)) = pack8(h);
      }
    lds_barrier();
    auto second = [&](auto n_c) {
      constexpr int n = decltype(n_c)::value, r = n - KS / 4;
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const bf16x8 h = frag(sH, b, 2 * r + k);
#pragma unroll
          for (int q = 0; q < 3; ++q) sum[q][b] = mfma32(w[n & 1][2 * q + k], h, sum[q][b]);
        }
      fetch(PIECE(n + 2), c);
    };
    second(PIECE(6)); second(PIECE(7)); second(PIECE(8)); second(PIECE(9));
  }
#undef PIECE

  // back into the stream by way of LDS, 32 rows at a time, in whole lines
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int row = 32 * b + (tid >> 3);
    float* const p = act + min(row, last) * CH + (tid & 7) * 4;
    f32x4 x[CH / 32];
#pragma unroll
    for (int i = 0; i < CH / 32; ++i) x[i] = *reinterpret_cast<const f32x4*>(p + 32 * i);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();  // what lies there has been read
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(sF + j * LDF + 32 * (3 * wave + q) + 16 * (g >> 1) + 8 * hh + 4 * (g & 1)) =
            f32x4{sum[q][b][4 * g], sum[q][b][4 * g + 1], sum[q][b][4 * g + 2], sum[q][b][4 * g + 3]};
    lds_barrier();
    if (row <= last)
#pragma unroll
      for (int i = 0; i < CH / 32; ++i) *reinterpret_cast<f32x4*>(p + 32 * i) = x[i] + *reinterpret_cast<const f32x4*>(sF + (tid >> 3) * LDF + (tid & 7) * 4 + 32 * i);
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int launch_row_transition(const RowTransitionArgs& a, hipStream_t s) {
  if (!a.act || !a.ln_w || !a.ln_b || !a.w1 || !a.w2 || a.rows <= 0 || a.hidden <= 0 || a.hidden % CHUNK || a.hidden > 8192 ||
      !al16(a.act) || !al16(a.ln_w) || !al16(a.ln_b) || !al16(a.w1) || !al16(a.w2))
    return AF3_ERR_BAD_ARG;
  hipLaunchKernelGGL(row_transition_kernel, dim3((unsigned)((a.rows - 1) / TS + 1)), dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
