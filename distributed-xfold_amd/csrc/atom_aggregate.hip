// Atoms to tokens: out[b][t] = the mean over a token's atoms of relu(x w^T), 128 channels to 768.
//
// As a product and a gather the projected atoms, empty slots and those of padding among them, are written and read back: at 5 x 768
// tokens of 24 slots 141 MB each way, 42 + 29 us.  Here a wave keeps 96 rows of w in registers (96 of them) and the token's
// atoms come to it: a workgroup gathers the atoms of four tokens into LDS, eight slots of each to a block of 32 rows (an
// empty one is zero, a block without an atom is left out), four waves multiply them with 384 rows of w, and since a lane owns a
// channel and a group of its registers a token, the mean is a sum of registers and one exchange between the halves of a wave.  The
// next four tokens' atoms are on their way meanwhile.  The product is rounded to bf16, as where it was stored.
// us, product and gather / this, tokens of 24 slots: 5 x 100 10.4 + 11.5 / 6.6, 5 x 384 21.8 + 15.6 / 15.5, 5 x 768 40 + 29 / 27.  What
// bounds it: a unit's vector instructions (relu, rounding, sums, the gather's addresses) and its products, which two
// workgroups to a CU overlap in part (5 x 768: 21 without the matrix instructions, 25 without the stores, 27 without the gather).
#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int IN = 128, KSTEPS = IN / 16, OUT = 768, HALF = OUT / 2, TOKENS = 4, COLS = HALF / 4 / 32;
constexpr int BLOCK = 32 * IN * 2;  // 32 atoms in LDS, two slabs of 64 channels, chunk c (16 bytes) of a row at position c ^ (row / 2 % 8)

template <int OCTETS>
__global__ __launch_bounds__(256, 2) void atom_aggregate_kernel(AtomAggregateArgs a) {
  __shared__ __attribute__((aligned(1024))) char sX[2][OCTETS * BLOCK];
  __shared__ int sLive[2][OCTETS];  // the unit (plus one) in which a block has an atom
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (int)blockIdx.y * HALF + wave * 32 * COLS;
  const int groups = (a.tokens + TOKENS - 1) / TOKENS, units = groups * a.batch;

  // thread: chunk tid % 16 of rows tid / 16 and 16 more of every block; row 8 t + s of block o is slot 8 o + s of token t
  const int chunk = tid & 15, row = tid >> 4;
  int at[OCTETS][2], at_next[OCTETS][2];  // of the unit that is gathered, and of the one behind it
  u32x4 x[OCTETS][2];
  auto first_token = [&](int unit) { return (unit - (int)((uint32_t)unit / (uint32_t)groups) * groups) * TOKENS; };
  auto slots = [&](int unit) {  // (asked for; what lies past the last token or slot is another one's)
    const int t0 = first_token(unit);
#pragma unroll
    for (int o = 0; o < OCTETS; ++o)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        at_next[o][h] = a.idx[min(t0 + 2 * h + (row >> 3), a.tokens - 1) * a.slots + min(8 * o + (row & 7), a.slots - 1)];
  };
  auto take = [&](int unit) {
    const int t0 = first_token(unit);
#pragma unroll
    for (int o = 0; o < OCTETS; ++o)
#pragma unroll
      for (int h = 0; h < 2; ++h) at[o][h] = t0 + 2 * h + (row >> 3) < a.tokens && 8 * o + (row & 7) < a.slots ? at_next[o][h] : -1;
  };
  auto gather = [&](int unit) {
    const bf16_t* const src = a.x + (int64_t)min((uint32_t)unit / (uint32_t)groups, (uint32_t)a.batch - 1u) * a.n_src * IN;
#pragma unroll
    for (int o = 0; o < OCTETS; ++o)
#pragma unroll
      for (int h = 0; h < 2; ++h) x[o][h] = *reinterpret_cast<const u32x4*>(src + (int64_t)max(at[o][h], 0) * IN + chunk * 8);
  };
  auto put = [&](int unit, int buf) {
#pragma unroll
    for (int o = 0; o < OCTETS; ++o)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = row + 16 * h;
        if (at[o][h] >= 0) sLive[buf][o] = unit + 1;
        *reinterpret_cast<u32x4*>(sX[buf] + o * BLOCK + (chunk >> 3) * (32 * 128) + r * 128 + (((chunk & 7) ^ ((r >> 1) & 7)) << 4)) =
            at[o][h] >= 0 ? x[o][h] : u32x4{0u, 0u, 0u, 0u};
      }
  };
  int unit = (int)blockIdx.x;
  slots(unit);
  if (tid < 2 * OCTETS) sLive[tid / OCTETS][tid % OCTETS] = 0;
  bf16x8 w[COLS][KSTEPS];
#pragma unroll
  for (int c = 0; c < COLS; ++c) load_frags<KSTEPS>(a.w, n0 / 32 + c, KSTEPS, 0, lane, w[c]);
  take(unit);
  gather(unit);
  slots(unit + (int)gridDim.x);
  lds_barrier();
  put(unit, 0);
  // (a wait for the weights that the compiler sees: it would put one into the loop, where it waits for the rows on their way as well)
  __builtin_amdgcn_s_waitcnt(0x0F70);
  lds_barrier();

  for (int buf = 0; unit < units; unit += (int)gridDim.x, buf ^= 1) {
    const int next = unit + (int)gridDim.x;
    const bool more = next < units;
    const int b = (int)((uint32_t)unit / (uint32_t)groups), t0 = (unit - b * groups) * TOKENS;
    float count[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) count[g] = a.count[min(t0 + g + 2 * hh, a.tokens - 1)];
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      take(next);
      gather(next);
      slots(next + (int)gridDim.x);
    }
    __builtin_amdgcn_sched_barrier(0);
    float sum[COLS][TOKENS];
#pragma unroll
    for (int c = 0; c < COLS; ++c)
#pragma unroll
      for (int g = 0; g < TOKENS; ++g) sum[c][g] = 0.f;
#pragma unroll
    for (int o = 0; o < OCTETS; ++o) {
      if (__builtin_amdgcn_readfirstlane(sLive[buf][o]) != unit + 1) continue;
      f32x16 acc[COLS];
#pragma unroll
      for (int c = 0; c < COLS; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[c][r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const bf16x8 f = as_frag(*reinterpret_cast<const u32x4*>(sX[buf] + o * BLOCK + (ks >> 2) * (32 * 128) + j * 128 +
                                                                 (((2 * (ks & 3) + hh) ^ ((j >> 1) & 7)) << 4)));
#pragma unroll
        for (int c = 0; c < COLS; ++c) acc[c] = mfma32(f, w[c][ks], acc[c]);
      }
      // registers 4 g + e: slot 8 o + 4 hh + e of token g
#pragma unroll
      for (int c = 0; c < COLS; ++c)
#pragma unroll
        for (int g = 0; g < TOKENS; ++g) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = fmaxf(acc[c][4 * g + e], 0.f);  // (the rounding keeps the sign)
          sum[c][g] = dot2_ones(pack2bf(v[2], v[3]), dot2_ones(pack2bf(v[0], v[1]), sum[c][g]));
        }
    }
    // both halves' slots; the lower half of the wave writes tokens 0 and 1, the upper one 2 and 3
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int token = t0 + g + 2 * hh;
      asm volatile("" : "+v"(count[g]));  // (waited for here on every path: a load left open makes the next unit's products wait)
      float* const out = a.out + ((int64_t)b * a.tokens + token) * OUT + n0 + j;
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum[c][g]), __float_as_uint(sum[c][g + 2]), false, false);
        if (token < a.tokens) out[32 * c] = (__uint_as_float(s[0]) + __uint_as_float(s[1])) / count[g];
      }
    }
    if (!more) break;
    put(next, buf ^ 1);  // (that buffer was last read in front of the barrier before)
    lds_barrier();
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int launch_atom_aggregate(const AtomAggregateArgs& a, hipStream_t s) {
  if (!a.x || !a.idx || !a.count || !a.w || !a.out || a.batch <= 0 || a.tokens <= 0 || a.n_src <= 0 || a.slots <= 0 || a.slots > 32 ||
      (int64_t)a.tokens * a.slots > 0x7fffffff || !al16(a.x) || !al16(a.w))
    return AF3_ERR_BAD_ARG;
  const int64_t units = (int64_t)((a.tokens + TOKENS - 1) / TOKENS) * a.batch;
  if (units > 0x3fffffff) return AF3_ERR_BAD_ARG;
  // of a workgroup; two to a CU, one for either half of the channels (5 x 768 with one / two / four / eight units to a workgroup 29.1 / 27.4 /
  // 27.3 / 30.8, 5 x 100 with two 9.7 against 6.4)
  const int64_t each = (units + 255) / 256;
  const dim3 grid((unsigned)((units + each - 1) / each), 2), block(256);
  switch ((a.slots + 7) / 8) {
    case 1: hipLaunchKernelGGL(atom_aggregate_kernel<1>, grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL(atom_aggregate_kernel<2>, grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL(atom_aggregate_kernel<3>, grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL(atom_aggregate_kernel<4>, grid, block, 0, s, a); break;
  }
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
