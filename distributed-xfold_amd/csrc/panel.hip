// Products of a few hundred rows a channel, T[c] = A[c] B[c]^T in bf16: the triangle contraction at few tokens.
//
// At 160 tokens a channel is 160 x 160 x 160, half a microsecond of a CU's matrix units, and the general kernel's tiles fetch their
// panels in slabs of K, one trip to memory after the other: what bounds it is those trips.  Here a workgroup brings all of K at once,
// some row blocks of A and some of B, straight into LDS (86 KB at 160 tokens), waits once and multiplies, with eight waves to a CU.
// Rows lie an odd number of 16-byte chunks apart, so that fragment reads of eight rows spread over the banks; what lies past a row or
// past the last row is read past the buffer's end, which writes zeros.  B's rows are taken in the order that leaves a lane with eight
// consecutive columns of its row, which it stores as they are.  K in ascending steps of 16, as the other kernels have it: the same
// bits.  us before / here, 128 channels: 40 tokens 4.0 / 3.2, 64 3.9 / 3.3, 90 5.3 / 3.8, 128 5.6 / 4.8, 144 9.1 / 5.8, 160 9.1 / 6.2,
// 187 9.6 / 7.6, 208 12.0 / 8.8, 224 12.3 / 10.0; 64 channels: 100 tokens 4.7 / 3.8, 160 7.3 / 5.8, 224 10.1 / 8.1, 256 9.8 / 9.2,
// 301 15.8 / 13.9.
#include "common.h"
#include "kernels.h"

namespace {

constexpr int WAVES = 8, ROW_WAVES = 2, COLUMN_WAVES = 4;  // a wave takes every second row block and every fourth column block

struct PanelArgs {
  const bf16_t *A, *B;
  bf16_t* C;
  int64_t plane;
  int n, K, ld, batch;
  int blocks;                      // of 32 rows (columns)
  int parts, part_blocks;          // parts of a channel's rows; row blocks in one
  int column_parts, column_blocks;
  int stride;                      // of a row in LDS, in chunks
  uint32_t magic;                  // of the division by it
  int a_loads, b_loads;            // of 1 KB
};

__device__ __forceinline__ u32x4 buffer_of(const void* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return u32x4{lo, hi & 0xffffu, 0x7fffffffu, 0x00020000u};
}

// NR x NC blocks of a wave: row blocks r0, r0 + ROW_WAVES, column blocks c0, c0 + COLUMN_WAVES
template <int NR, int NC>
__device__ __forceinline__ void multiply(const PanelArgs& a, const char* sA, const char* sB, int r0, int c0, int m0, int n0, bf16_t* out) {
  const int lane = threadIdx.x & 63, hh = lane >> 5, j = lane & 31, swap = (j & ~12) | ((j & 4) << 1) | ((j & 8) >> 1);
  const int row_bytes = a.stride * 16;
  const char *pa[NR], *pb[NC];
  f32x16 acc[NR][NC];
#pragma unroll
  for (int r = 0; r < NR; ++r) pa[r] = sA + ((r0 + ROW_WAVES * r) * 32 + j) * row_bytes + hh * 16;
#pragma unroll
  for (int c = 0; c < NC; ++c) pb[c] = sB + ((c0 + COLUMN_WAVES * c) * 32 + swap) * row_bytes + hh * 16;
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[r][c][e] = 0.f;
  const int steps = a.stride >> 1;  // (the stride is one more than the chunks of a row, two to a step)
  for (int k = 0; k < steps; ++k) {
    bf16x8 fa[NR], fb[NC];
#pragma unroll
    for (int r = 0; r < NR; ++r) fa[r] = as_frag(*reinterpret_cast<const u32x4*>(pa[r] + k * 32));
#pragma unroll
    for (int c = 0; c < NC; ++c) fb[c] = as_frag(*reinterpret_cast<const u32x4*>(pb[c] + k * 32));
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[r][c] = mfma32(fb[c], fa[r], acc[r][c]);
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int row = m0 + (r0 + ROW_WAVES * r) * 32 + j;
    if (row >= a.n) continue;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int col = n0 + (c0 + COLUMN_WAVES * c) * 32 + 16 * u + 8 * hh;
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = acc[r][c][8 * u + e];
        if (col < a.ld) *reinterpret_cast<u32x4*>(out + (int64_t)row * a.ld + col) = pack8(f);
      }
  }
}

__global__ __launch_bounds__(64 * WAVES) void panel_product_kernel(PanelArgs a) {
  args_at_once<PanelArgs>();
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the parts of a channel follow each other on one XCD, which has its B in L2
  const int slot = blockIdx.x >> 3, each = a.parts * a.column_parts, turn = slot / each, tile = slot - turn * each;
  const int ch = turn * 8 + (blockIdx.x & 7), column_part = tile / a.parts, part = tile - column_part * a.parts;
  const int first = part * a.part_blocks, count = min(a.part_blocks, a.blocks - first);
  const int first_column = column_part * a.column_blocks, columns = min(a.column_blocks, a.blocks - first_column);
  if (ch >= a.batch || count <= 0 || columns <= 0) return;
  const int m0 = first * 32, n0 = first_column * 32, chunks = a.K >> 3;
  const u32x4 ra = buffer_of(a.A + ch * a.plane), rb = buffer_of(a.B + ch * a.plane);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  for (int i = wave; i < a.a_loads + a.b_loads; i += WAVES) {
    const bool is_b = i >= a.a_loads;
    const uint32_t e = (uint32_t)((is_b ? i - a.a_loads : i) * 64 + lane);
    const int row = (int)__umulhi(e, a.magic), pos = (int)e - row * a.stride, at = (is_b ? n0 : m0) + row;
    const uint32_t off = pos < chunks && at < a.n ? (uint32_t)(at * a.ld + pos * 8) * 2u : 0x80000000u;
    const uint32_t lds = __builtin_amdgcn_readfirstlane(lds0 + i * 1024);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(off), "s"(is_b ? rb : ra)
                 : "m0", "memory");
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  const int r0 = wave / COLUMN_WAVES, c0 = wave % COLUMN_WAVES;
  if (r0 >= count || c0 >= columns) return;
  const char *sA = smem, *sB = smem + a.a_loads * 1024;
  bf16_t* const out = a.C + ch * a.plane;
  const bool two_rows = r0 + ROW_WAVES < count, two_columns = c0 + COLUMN_WAVES < columns;
  if (two_rows && two_columns) multiply<2, 2>(a, sA, sB, r0, c0, m0, n0, out);
  else if (two_rows) multiply<2, 1>(a, sA, sB, r0, c0, m0, n0, out);
  else if (two_columns) multiply<1, 2>(a, sA, sB, r0, c0, m0, n0, out);
  else multiply<1, 1>(a, sA, sB, r0, c0, m0, n0, out);
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

constexpr int PANEL_LDS = 160 * 1024, CUS = 256;

// Past these a channel takes several rounds of workgroups, each with a trip of its own, and the slabs that overlap their loads with
// the product are ahead.  us, those / here, 128 channels: 224 tokens 12.3 / 10.0, 240 13.2 / 13.4, 256 12.9 / 15.0; 64 channels:
// 304 15.7 / 14.0, 312 16.6 / 17.1, 320 16.0 / 17.2.
constexpr int PANEL_TOKENS = 224, PANEL_TOKENS_64 = 304;

static bool panel_args(const GemmArgs& g, PanelArgs* a, int* lds) {
  if (!g.A || !g.B || !g.C || g.M <= 0 || g.M != g.N || g.M > (g.batch > 64 ? PANEL_TOKENS : PANEL_TOKENS_64) || g.K <= 0 || (g.K & 7) || g.K > g.lda || g.lda != g.ldb ||
      g.lda != g.ldc || g.lda > 4096 || (g.lda & 7) || g.sA != g.sB || g.sA != g.sC || (g.sA & 7) || g.batch <= 0 || g.out_f32 ||
      g.epi != EPI_PLAIN || g.bias || g.alpha != 1.f || g.act_sigmoid || g.regroup32 || !al16(g.A) || !al16(g.B) || !al16(g.C))
    return false;
  a->A = g.A; a->B = g.B; a->C = static_cast<bf16_t*>(g.C);
  a->plane = g.sA; a->n = g.M; a->K = g.K; a->ld = (int)g.lda; a->batch = g.batch;
  a->blocks = (g.M + 31) / 32;
  a->stride = 2 * ((g.K + 15) / 16) + 1;
  a->magic = 0xffffffffu / (uint32_t)a->stride + 1u;
  // the tiling that fits (two row blocks and two column blocks to a wave) with the least rounds times KB, and as much as 40 KB for
  // what a round takes whatever its size
  auto loads = [&](int blocks) { return (blocks * 32 * a->stride + 63) / 64; };
  int64_t best = -1;
  for (int rows = 1; rows <= 2 * ROW_WAVES && rows <= a->blocks; ++rows)
    for (int columns = 1; columns <= 2 * COLUMN_WAVES && columns <= a->blocks; ++columns) {
      const int parts = (a->blocks + rows - 1) / rows, column_parts = (a->blocks + columns - 1) / columns, kb = loads(rows) + loads(columns);
      const int64_t cost = ((int64_t)g.batch * parts * column_parts + CUS - 1) / CUS * (kb + 40);
      if (kb * 1024 > PANEL_LDS || (best >= 0 && cost >= best)) continue;
      best = cost;
      a->parts = parts; a->part_blocks = rows; a->column_parts = column_parts; a->column_blocks = columns;
    }
  if (best < 0) return false;
  a->a_loads = loads(a->part_blocks);
  a->b_loads = loads(a->column_blocks);
  *lds = (a->a_loads + a->b_loads) * 1024;
  return true;
}

int launch_panel_product(const GemmArgs& g, hipStream_t s) {
  PanelArgs a;
  int lds;
  if (!panel_args(g, &a, &lds)) return AF3_ERR_UNSUPPORTED;
  // (more than 64 KB have to be asked for; always for as much as there is, since another thread may be launching with another size)
  if (lds > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(panel_product_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         PANEL_LDS) != hipSuccess) {
    (void)hipGetLastError();
    return AF3_ERR_LAUNCH;
  }
  hipLaunchKernelGGL(panel_product_kernel, dim3((unsigned)((g.batch + 7) / 8 * 8 * a.parts * a.column_parts)), dim3(64 * WAVES), lds, s, a);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
