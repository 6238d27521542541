// The single track's LayerNorm and the product behind it (queries, keys, values and gate; or the SwiGLU transition's first layer) in
// one kernel, for rows of 384 channels.
//
// A few hundred rows make launches of 4 to 6 us of which next to nothing is arithmetic: the launch, a trip to memory, a chain of 24
// matrix instructions, the stores; and at some 64 tokens the host, 3 us a launch, sets the pace of the whole stack.  Here both
// operands come in one trip: a workgroup asks for its 32 rows and, straight into LDS, for its 64 rows of the weights (48 KB),
// normalises the rows, sixteen lanes to each, and multiplies, two waves sharing the channels of 32 columns.  Every row is normalised
// by each of the 24 or 48 workgroups that need it, which costs less than a launch.  72 KB of LDS, so that a workgroup finds room
// beside those of the pair operators, which run at the same time: with 128 rows of the weights (120 KB) it waits for an empty CU
// (128 tokens 8.7 -> 11.5 us, the stack 460 -> 463).
// Bound by launch, trip and chain: 64 tokens 5.4 and 5.8 us against 4.6 + 4.4 and 4.6 + 5.3 as two kernels each.  A stack of four
// blocks, us, two kernels / this, bf16 stream (128: fp32): 40 tokens 370 / 337, 64 357 / 337, 100 420 / 415, 128 468 / 460, 160 602 / 599,
// 200 840 / 835, 260 1368 / 1361, 387 2630 / 2625, 500 4038 / 4050: up to SINGLE_STEP_ROWS.
#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int K = SINGLE_STEP_CHANNELS, SLABS = K / 64, ROWS = 32, BN = 64;
constexpr int KSTEPS = K / 16 / 2, GROUP = 6;  // of a wave; of these, whose fragments are read while the group before is multiplied

template <typename TIO, bool SWIGLU>
__global__ __launch_bounds__(256, 2) void single_step_kernel(SingleStepArgs a) {
  args_at_once<SingleStepArgs>();
  using E = Elem<TIO>;
  constexpr int EACH = ROWS / 16;  // rows of a group of sixteen lanes
  // slabs of 64 channels, [slab][row][128 bytes], chunk c (16 bytes) of a row at position c ^ (row / 2 % 8)
  __shared__ __attribute__((aligned(1024))) char sW[SLABS * BN * 128];
  __shared__ __attribute__((aligned(1024))) char sX[SLABS * ROWS * 128];
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (int)blockIdx.x * BN, m0 = (int)blockIdx.y * ROWS;

  // the rows: lane s of a group takes chunks s, s + 16 and s + 32 of rows g, g + 16, ..
  const int sub = tid & 15, grp = tid >> 4;
  const TIO* const x = reinterpret_cast<const TIO*>(a.x);
  typename E::Raw raw[EACH][3];
#pragma unroll
  for (int u = 0; u < EACH; ++u)
#pragma unroll
    for (int i = 0; i < 3; ++i) raw[u][i] = E::load_raw(x + (int64_t)min(m0 + grp + 16 * u, a.rows - 1) * K + (sub + 16 * i) * 8);
  float lw[3][8], lb[3][8], bias[16];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    Elem<float>::load8(a.ln_w + (sub + 16 * i) * 8, lw[i]);
    Elem<float>::load8(a.ln_b + (sub + 16 * i) * 8, lb[i]);
  }
  const int block = wave & 1, half = wave >> 1, col = n0 + 32 * block + 8 * hh;
  const bool queries = !SWIGLU && n0 < K, biased = queries && a.q_bias;
  if constexpr (!SWIGLU) {
    const float* const p = biased ? a.q_bias + col : a.ln_b;
#pragma unroll
    for (int u = 0; u < 2; ++u) Elem<float>::load8(p + 16 * u, bias + 8 * u);
  }
  __builtin_amdgcn_sched_barrier(0);
  // The weights' rows, 1 KB (eight rows of a slab) at a time, in the order in which a lane's sixteen accumulators become runs of
  // result columns: LDS row 32 q + r is column 32 q + r with bits 2 and 3 exchanged; with SwiGLU rows 0..15 of 32 are the first
  // factor of hidden units 16 q .. (bits 2 and 3 exchanged), the others the second (w in blocks of 32 + 32 rows).
#pragma unroll
  for (int i = 0; i < BN / 32; ++i) {
    const int p = 8 * (4 * i + wave) + (lane >> 3), r = p & 31;
    const int s = (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1);
    const int unit = n0 / 2 + 16 * (p >> 5) + (s & 15);
    const int row = SWIGLU ? (unit >> 5) * 64 + (unit & 31) + (r & 16 ? 32 : 0) : n0 + 32 * (p >> 5) + s;
    const bf16_t* const w = a.w + (int64_t)row * K + ((lane & 7) ^ ((p >> 1) & 7)) * 8;
#pragma unroll
    for (int sl = 0; sl < SLABS; ++sl)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(w + 64 * sl),
                                       (__attribute__((address_space(3))) void*)(sW + sl * (BN * 128) + 1024 * (4 * i + wave)), 16, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int u = 0; u < EACH; ++u) {
    float v[3][8], s = 0.f, q = 0.f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      E::unpack_raw(raw[u][i], v[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[i][e];
    }
    const float mean = group16_sum(s) * (1.f / K);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] -= mean;
      q = add_squares8(v[i], q, i == 0);
    }
    const float rstd = rsqrtf(group16_sum(q) * (1.f / K) + LN_EPS);
    const int row = grp + 16 * u;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = v[i][e] * rstd * lw[i][e] + lb[i][e];
      const int chunk = sub + 16 * i;
      *reinterpret_cast<u32x4*>(sX + (chunk >> 3) * (ROWS * 128) + row * 128 + (((chunk & 7) ^ ((row >> 1) & 7)) << 4)) = pack8(o);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the weights' rows
  lds_barrier();

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  auto frag = [&](const char* slabs, int rows, int first, int ks) {
    return as_frag(*reinterpret_cast<const u32x4*>(slabs + (ks >> 2) * (rows * 128) + (first + j) * 128 +
                                                   (((2 * (ks & 3) + hh) ^ ((j >> 1) & 7)) << 4)));
  };
  bf16x8 wf[2][GROUP], xf[2][GROUP];
  auto read = [&](int g) {
#pragma unroll
    for (int i = 0; i < GROUP; ++i) {
      wf[g & 1][i] = frag(sW, BN, 32 * block, half * KSTEPS + GROUP * g + i);
      xf[g & 1][i] = frag(sX, ROWS, 0, half * KSTEPS + GROUP * g + i);
    }
  };
  read(0);
#pragma unroll
  for (int g = 0; g < KSTEPS / GROUP; ++g) {
    if (g + 1 < KSTEPS / GROUP) read(g + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < GROUP; ++i) acc = mfma32(wf[g & 1][i], xf[g & 1][i], acc);
  }
  lds_barrier();  // (the operands have been read)
  f32x4* const sum = reinterpret_cast<f32x4*>(sX) + block * 256 + lane;
  if (half)
#pragma unroll
    for (int g = 0; g < 4; ++g) sum[g * 64] = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  lds_barrier();
  if (half) return;

  // a lane's registers 8 u .. are columns 32 block + 16 u + 8 hh .. of row j (SwiGLU: both factors of hidden units 16 block + 8 hh ..)
  const int row = m0 + j;
  if (row >= a.rows) return;
  bf16_t* const out = a.out + (int64_t)row * a.ldc;
  float o[16];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 v = sum[g * 64];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[4 * g + e] = acc[4 * g + e] + v[e];
  }
  if constexpr (SWIGLU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = o[e] * sigmoidf_(o[e]) * o[8 + e];
    *reinterpret_cast<u32x4*>(out + n0 / 2 + 16 * block + 8 * hh) = pack8(o);
  } else {
    if (queries) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = (o[r] + (biased ? bias[r] : 0.f)) * a.q_scale;
    } else if (n0 >= 3 * K) {  // the gate
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = sigmoidf_(o[r]);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) *reinterpret_cast<u32x4*>(out + col + 16 * u) = pack8(o + 8 * u);
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

bool single_step_applies(const SingleStepArgs& a) {
  return a.x && a.w && a.out && a.ln_w && a.ln_b && a.rows > 0 && a.rows <= SINGLE_STEP_ROWS && a.N > 0 && a.N % BN == 0 &&
         (a.swiglu || a.N == 4 * K) && a.ldc % 8 == 0 && al16(a.x) && al16(a.w) && al16(a.out) && al16(a.ln_w) && al16(a.ln_b) && al16(a.q_bias);
}

int launch_single_step(const SingleStepArgs& a, hipStream_t s) {
  if (!single_step_applies(a)) return AF3_ERR_BAD_ARG;
  const dim3 grid((unsigned)(a.N / BN), (unsigned)((a.rows + ROWS - 1) / ROWS)), block(256);
  if (a.io_f32 && a.swiglu) hipLaunchKernelGGL((single_step_kernel<float, true>), grid, block, 0, s, a);
  else if (a.io_f32) hipLaunchKernelGGL((single_step_kernel<float, false>), grid, block, 0, s, a);
  else if (a.swiglu) hipLaunchKernelGGL((single_step_kernel<bf16_t, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((single_step_kernel<bf16_t, false>), grid, block, 0, s, a);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
