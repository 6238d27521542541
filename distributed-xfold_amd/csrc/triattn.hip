// Triangle attention, the fast path: the projection kernel.  It produces, in one
// pass over the pair tensor, everything the attention core (triattn_core.hip)
// reads, in the layouts it wants (described in kernels.h): head-major q (scaled)
// and k, V transposed with the key order the core's MFMA fragments use, and the
// fp16 pair bias in the order of the core's MFMA fragments.  (The output gate is
// computed where it is used, by attn_out_kernel.)
#include "common.h"
#include "kernels.h"
#include <type_traits>

#include "tile_common.h"

namespace {

constexpr int H = 4, D = 32;

// ============================================================================
// projections: LN -> q (scaled), k (position-major) and v (channel-major),
// + pair-bias heads
// ============================================================================
// SPLIT: a workgroup takes one of q (with the pair bias), k and v (blockIdx.y), where tiles are few.
template <typename TIO, bool CROSS, bool SPLIT>
__global__ __launch_bounds__(256, 3) void triattn_proj_kernel(TriAttnProjArgs a) {
  // 34.8 KB + 17.4 KB of LDS and at most 168 registers: three workgroups per CU.  The kernel is a chain of
  // short dependent phases (load, LayerNorm, MFMA, stage, store), so what it needs is company.
  __shared__ __attribute__((aligned(16))) bf16_t sX[TM * LDX];  // LN tile, then staging
  __shared__ __attribute__((aligned(16))) bf16_t sW[64 * LDX];  // 64 weight rows at a time
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // (b, s) = (o, r), flat over rows of ldn positions (the row length of V transposed, a multiple of 16: a tile starts on
  // a group of 16 keys); for the transposed operator the rows are columns of the pair tensor.
  // last tile first: the pair tensor was written front to back by the operator
  // before this one, and the attention core that follows starts with row 0,
  // which is then the freshest part of q / k / v (measured: 1.4 % of the block)
  const auto t = make_tile<CROSS>(a.N, (int)a.ldn, a.transpose != 0, true);
  const TIO* x = reinterpret_cast<const TIO*>(a.pair);
  // Step s = 2 * chunk + half: weight rows 64 half .. + 63 of chunk s / 2 (chunks q, k, v of w_qkvg),
  // four 16-byte pieces per thread; the 32 (padded) pair-bias rows ride in the same registers.
  u32x4 wr[4];
  auto wload = [&](int s) {
    const bf16_t* base = a.w_qkvg + (int64_t)s * 64 * C;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i;
      wr[i] = *reinterpret_cast<const u32x4*>(base + (idx >> 4) * C + (idx & 15) * 8);
    }
  };
  auto wload_bias = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + 256 * i;
      wr[i] = *reinterpret_cast<const u32x4*>(a.w_bias + (idx >> 4) * C + (idx & 15) * 8);
    }
  };
  auto wstore = [&](int n) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i;
      if (i < n) *reinterpret_cast<u32x4*>(sW + (idx >> 4) * LDX + (idx & 15) * 8) = wr[i];
    }
  };
  const int part = SPLIT ? (int)blockIdx.y : 0;
  const bool bias = a.n_bias > 0 && part == 0;
  wload(2 * part);
  load_ln_tile<TIO>(x, t, a.ln_w, a.ln_b, sX, tid, a.skip_ln != 0, a.lw.inv_c, a.lw.pad);
  wstore(4);
  lds_barrier();
  bf16x8 xf[8];
  load_x_frags(sX, wave, lane, xf);
  lds_barrier();  // sX is free from here on: it becomes the staging tile

  // v takes the channel-major route.  The step index is a compile-time constant of the body: with a
  // run-time index the compiler evaluates the sigmoid for every chunk and selects.
  auto do_step = [&](auto step_c) {
    constexpr int step = decltype(step_c)::value, chunk = step >> 1, pairt = step & 1;
    // The next weights are requested BEFORE this chunk's results are stored:
    // vector memory operations retire in order, so a load issued behind the
    // stores would make its consumer wait for the stores' round trip to HBM.
    constexpr bool last = SPLIT ? pairt == 1 : step == 5;
    if (!last) wload(step + 1);
    else if (bias) wload_bias();
    {
      f32x16 acc[2];
      if (chunk == 2) {
        // v: D form, lane owns channel (lane & 31) of a tile, registers walk pixels
        mfma_chunk<false, 2>(xf, sW, lane, acc);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int ch = (pairt * 2 + nt) * 32 + (lane & 31);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int p0 = wave * 32 + 8 * g + 4 * (lane >> 5);
            u32x2 pk;
            pk.x = pack2bf(acc[nt][4 * g], acc[nt][4 * g + 1]);
            pk.y = pack2bf(acc[nt][4 * g + 2], acc[nt][4 * g + 3]);
            *reinterpret_cast<u32x2*>(sX + ch * LDX + tri_vt_pos(p0)) = pk;
          }
        }
      } else {
        mfma_chunk<true, 2>(xf, sW, lane, acc);
        const int px = wave * 32 + (lane & 31);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float y = acc[nt][4 * g + e];
              v[e] = chunk == 0 ? y * a.q_scale : y;
            }
            const int ch = (pairt * 2 + nt) * 32 + 8 * g + 4 * (lane >> 5);
            u32x2 pk;
            pk.x = pack2bf(v[0], v[1]);
            pk.y = pack2bf(v[2], v[3]);
            *reinterpret_cast<u32x2*>(sX + px * LDX + ch) = pk;
          }
      }
    }
    lds_barrier();  // staging visible; every wave is done with sW
    if (!last) wstore(4);
    else if (bias) wstore(2);
    if (pairt == 1) {
      // both halves of the chunk are staged: 128 channels per position go out
      if (chunk == 2) {
        // Vt[(b*H + h)*32 + d][tri_vt_pos(s)]: per channel 128 consecutive columns (the quads of
        // a 16-key group were swapped on their way into the staging tile)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int idx = tid + 256 * i, ch = idx >> 4, pc = idx & 15;
          int o, r;
          t.at(pc * 8, &o, &r);
          if (o < a.N)
            *reinterpret_cast<u32x4*>(a.vt + ((int64_t)o * H * D + ch) * a.ldn + r) =
                *reinterpret_cast<const u32x4*>(sX + ch * LDX + pc * 8);
        }
      } else {
        bf16_t* plane = chunk == 0 ? a.q : a.k;
        const int ck = tid & 15, prow = tid >> 4;
        const int h = ck >> 2, part = ck & 3;
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const int p = it * 16 + prow;
          int o, r;
          t.at(p, &o, &r);
          if (r < a.N && o < a.N)
            *reinterpret_cast<u32x4*>(plane + (((int64_t)o * H + h) * a.N + r) * D + part * 8) =
                *reinterpret_cast<const u32x4*>(sX + p * LDX + ck * 8);
        }
      }
    }
    lds_barrier();
  };
  if (!SPLIT || part == 0) {
    do_step(std::integral_constant<int, 0>{});
    do_step(std::integral_constant<int, 1>{});
  }
  if (!SPLIT || part == 1) {
    do_step(std::integral_constant<int, 2>{});
    do_step(std::integral_constant<int, 3>{});
  }
  if (!SPLIT || part == 2) {
    do_step(std::integral_constant<int, 4>{});
    do_step(std::integral_constant<int, 5>{});
  }

  // pair-bias heads (T form: lane = pixel, rows = heads): bias[h][q][k] with
  // (q, k) the pixel's own (row, col) in the un-transposed pair tensor
  if (bias) {
    f32x16 acc[1];
    mfma_chunk<true, 1>(xf, sW, lane, acc);
    if ((lane >> 5) == 0) {  // heads 0..3 are accumulator rows 0..3: registers 0..3 of the low half
      const int p = wave * 32 + lane;
      int o, r;
      t.at(p, &o, &r);
      if (r < a.N && o < a.N) {
        const int q = a.transpose ? r : o, k = a.transpose ? o : r;
#pragma unroll
        for (int h = 0; h < H; ++h) a.bias[tri_bias_offset(a.N, h, q, k)] = f2h_sat(acc[0][h] * a.bias_scale);
        // keys N .. of the last key tile are padding and read as zero bias: the tile's real keys share them out
        const int k_last = (a.N - 1) & ~63, real = a.N - k_last;
        if (k >= k_last)
          for (int kp = a.N + k - k_last; kp < k_last + 64; kp += real)
#pragma unroll
            for (int h = 0; h < H; ++h) a.bias[tri_bias_offset(a.N, h, q, kp)] = 0;
      }
    }
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Tiles up to which q, k and v are three workgroups' work: all of them are on the chip at once (three fit a CU), and the
// kernel takes two steps of a tile and its LayerNorm instead of six.  Kernel alone, N = 64, 128, 176: 10.6 -> 7.6 us,
// 15.3 -> 13.3 us, 15.9 -> 13.7 us; past the line, N = 212, 17.9 instead of 16.3 us.
constexpr int64_t SPLIT_TILES = 256;

}  // namespace

int launch_triattn_proj(const TriAttnProjArgs& a, hipStream_t stream) {
  if (a.N <= 0 || !a.pair || !a.w_qkvg || !a.q || !a.k || !a.vt) return AF3_ERR_BAD_ARG;
  if (a.ldn < a.N || (a.ldn & 15)) return AF3_ERR_BAD_ARG;
  if (a.n_bias != 0 && (a.n_bias != H || !a.w_bias || !a.bias)) return AF3_ERR_BAD_ARG;
  if (!al16(a.pair) || !al16(a.w_qkvg) || !al16(a.w_bias) || !al16(a.q) || !al16(a.k) || !al16(a.vt) ||
      !al16(a.bias))
    return AF3_ERR_BAD_ARG;
  const int64_t tiles = ((int64_t)a.N * a.ldn + TM - 1) / TM;
  if (tiles > 0x7fffffff) return AF3_ERR_BAD_ARG;
  const bool cross = tile_crosses(a.ldn), split = tiles <= SPLIT_TILES;
  const dim3 grid((unsigned)tiles, split ? 3 : 1), block(256);
  auto launch = [&](auto split_c) {
    constexpr bool S = decltype(split_c)::value;
    if (a.io_f32 && cross) hipLaunchKernelGGL((triattn_proj_kernel<float, true, S>), grid, block, 0, stream, a);
    else if (a.io_f32) hipLaunchKernelGGL((triattn_proj_kernel<float, false, S>), grid, block, 0, stream, a);
    else if (cross) hipLaunchKernelGGL((triattn_proj_kernel<bf16_t, true, S>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((triattn_proj_kernel<bf16_t, false, S>), grid, block, 0, stream, a);
  };
  if (split) launch(std::true_type{});
  else launch(std::false_type{});
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}
