// C = A B^T of K = 384 with an fp32 result of very many columns (the conditioning of all blocks of a token transformer: some hundred
// rows, 73728 and 36864 columns): what it writes is most of what it moves, and the chip's memory sets the pace.
//
// In the tiles of gemm.hip a workgroup loads, multiplies and stores, and since all begin at once the chip does one after the other:
// 768 x 73728 121 us, 56 of it without the stores, for 226 MB of results and 57 of weights (58 us at the rate of a copy).  Here a
// wave keeps 32 rows of B, all of K, in registers (96 of them) and the rows of A come past, 32 at a time by DMA into one of two
// panels in LDS (24 KB) that the workgroup's four waves share; each step's results, whole lines of 32 columns, are on their way while
// the next ones are multiplied.  Three workgroups to a CU; the sums have gemm.hip's order (the same bits).
// us, gemm.hip / this: 384 x 73728 59 / 48, 768 x 73728 118 / 76, 1536 x 73728 238 / 143, 768 x 36864 59 / 47, 3840 x 18432 129 / 86.
// What bounds it: with the weights' trip (14 us until the first results, each lane of a load on a line of its own) 45 us of 768 x 73728
// are matrix instructions and LDS reads, which the stores lengthen; 59 without them, 74 without matrix instructions, and the same
// with the results side by side in memory, the LDS reads a group ahead, or without the wait for the stores but one.
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "tile_common.h"

namespace {

constexpr int WK = 384, KSTEPS = WK / 16, SLABS = WK / 64, ROWS = 32, BN = 128;
// From so many results on; us, gemm.hip / this: 200 x 73728 (14.7 M) 41.1 / 35.6, 500 x 36864 43.2 / 36.5, 1000 x 18432 34.9 / 31.3,
// 1536 x 12288 35.2 / 30.4, 3840 x 6144 45.0 / 36.2, 10000 x 3072 55.0 / 51.2; below 768 x 18432 28.1 / 27.0, 384 x 36864 (13.5 M) 32.3 / 31.0, 768
// x 12288 20.3 / 22.5, 100 x 73728 22.3 / 24.0; narrower 10000 x 1536 28.8 / 33.6, 40000 x 384 32.4 / 34.7.
constexpr int64_t WIDE_RESULTS = (int64_t)14 << 20;
constexpr int WIDE_COLUMNS = 3072;
constexpr int PANEL = SLABS * ROWS * 128;  // [slab of 64 of K][row][128 bytes], chunk c (16 bytes) at position c ^ (row / 2 % 8)

__global__ __launch_bounds__(256, 3) void wide_product_kernel(GemmArgs g, WideWalk walk) {
  __shared__ __attribute__((aligned(1024))) char sA[2][PANEL];
  const int lane = threadIdx.x & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // every XCD takes a run of strips of 128 columns, the parts of a strip's rows one after the other
  const int idx = (int)(blockIdx.x & 7) * walk.per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= walk.per_xcd || idx >= walk.total) return;
  const int strip = walk.parts == 1 ? idx : (int)__umulhi((uint32_t)idx, walk.magic_parts), part = idx - strip * walk.parts;
  const int m0 = part * walk.panels * ROWS, m1 = min(m0 + walk.panels * ROWS, g.M), n0 = strip * BN + 32 * wave;
  if (m0 >= g.M) return;

  const bf16_t* const x = g.A + (int64_t)m0 * g.lda;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)sA + 1024 * wave;
  const int mine = 8 * wave + (lane >> 3);  // row of a panel
  auto bring = [&](int p) {
    const bf16_t* const rows = x + (int64_t)p * ROWS * g.lda;
    const uint32_t off = ((uint32_t)min(mine, m1 - 1 - m0 - p * ROWS) * (uint32_t)g.lda + ((lane & 7) ^ ((mine >> 1) & 7)) * 8) * 2u;
#pragma unroll
    for (int s = 0; s < SLABS; ++s)
      load_to_lds(rows + 64 * s, off, __builtin_amdgcn_readfirstlane(lds0 + (p & 1) * PANEL + s * (ROWS * 128)));
  };
  const int panels = (m1 - m0 + ROWS - 1) / ROWS;
  bring(0);
  if (panels > 1) bring(1);
  bf16x8 w[KSTEPS];
  const bf16_t* const b = g.B + (int64_t)n0 * g.ldb;
  const uint32_t row_off = (uint32_t)j * (uint32_t)g.ldb + 8 * hh;
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) w[ks] = as_frag(*reinterpret_cast<const u32x4*>(at32(b + 16 * ks, row_off)));
  const float bias = g.bias ? g.bias[n0 + j] : 0.f;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();

  float* const out = reinterpret_cast<float*>(g.C) + (int64_t)m0 * g.ldc + n0;
  const uint32_t lane_off = (uint32_t)(4 * hh) * (uint32_t)g.ldc + j;
  for (int p = 0; p < panels; ++p) {
    const char* const panel = sA[p & 1];
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const bf16x8 a = as_frag(*reinterpret_cast<const u32x4*>(panel + (ks >> 2) * (ROWS * 128) + j * 128 + (((2 * (ks & 3) + hh) ^ ((j >> 1) & 7)) << 4)));
      acc = mfma32(a, w[ks], acc);
    }
    float o[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      o[r] = (acc[r] + bias) * g.alpha;
      if (g.act_sigmoid) o[r] = sigmoidf_(o[r]);
    }
    // The next panel is there: behind its loads were issued the last step's sixteen stores and nothing else (loads and stores are
    // counted off in the order of their issue).  The first step's follows the weights' wait, the last one's has no next panel.
    if (p > 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(16) : "memory");
    lds_barrier();  // (and this one has been read)
    if (p + 2 < panels) bring(p + 2);
    // registers 4 q + e: row 8 q + 4 hh + e of the panel; lane j: column j
    float* const d = out + (int64_t)p * ROWS * g.ldc;
    const int left = m1 - m0 - p * ROWS;
    if (left >= ROWS) {
#pragma unroll
      for (int r = 0; r < 16; ++r) *at32(d + (int64_t)(8 * (r >> 2) + (r & 3)) * g.ldc, lane_off) = o[r];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + (r & 3) + 4 * hh < left) *at32(d + (int64_t)(8 * (r >> 2) + (r & 3)) * g.ldc, lane_off) = o[r];
    }
  }
}

}  // namespace

bool wide_product_applies(const GemmArgs& g) {
  return g.batch == 1 && g.K == WK && g.out_f32 && g.epi == EPI_PLAIN && !g.regroup32 && g.N % BN == 0 && g.M > 0 && g.lda < (1 << 20) &&
         g.ldb < (1 << 20) && g.ldc < (1 << 26) && g.M <= (1 << 20) && g.N <= (1 << 26) &&
         g.N >= WIDE_COLUMNS && (int64_t)g.M * g.N >= WIDE_RESULTS;
}

int launch_wide_product(const GemmArgs& g, hipStream_t s) {
  if (!wide_product_applies(g)) return AF3_ERR_BAD_ARG;
  const int strips = g.N / BN, panels = (g.M + ROWS - 1) / ROWS;
  WideWalk w;
  // four to five workgroups' work for a CU, as long as a part has four panels for its weights (768 x 73728 in one / two / three / four
  // parts 86 / 81 / 82 / 88 us, 384 x 73728 55 / 50 / 53 / 55, 768 x 36864 52 / 42 / 41 / 41)
  w.parts = std::max(1, std::min((1023 + strips) / strips, panels / 4));
  w.panels = (panels + w.parts - 1) / w.parts;
  w.total = strips * w.parts;
  w.per_xcd = (w.total + 7) / 8;
  w.magic_parts = w.parts == 1 ? 0u : 0xffffffffu / (uint32_t)w.parts + 1u;
  hipLaunchKernelGGL(wide_product_kernel, dim3(8u * w.per_xcd), dim3(256), 0, s, g, w);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
