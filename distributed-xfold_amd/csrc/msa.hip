// Kernels of the Evoformer's MSA track (64 channels): what surrounds the two long products, the outer-product mean and
// the pair-weighted average, each of which wants an operand with the summation index (MSA rows, tokens) innermost.
//
// All of them move a [rows][n][64] tensor once or twice and do little to it, so what counts is passes over memory.
// A lane owns one position (32 channels of it: chunks 16 ks + 8 hh), LayerNorm is a sum over its registers and one
// exchange with the other half of the wave, and the normalised chunks are MFMA fragments as they stand: nothing of the
// activations goes through LDS.  Where a product's result has to be the next one's operand, or is to be stored in
// 16-byte pieces, the rows of its left operand are taken in the order swap23 (bits 2 and 3 exchanged): registers
// 8 s .. 8 s + 7 of a lane are then eight consecutive rows of the result.
//
// bf16, 1024 rows x 768 tokens (100 MB), in place of LayerNorm, projections, mask product, gating and transposes as
// launches of their own and of a transition on a copy padded to 128 channels: operands of the outer-product mean 67 us
// (were 226), values 60 (were 155, with the gate), update 160 (output projection 140, transition 330).
#include "common.h"
#include "kernels.h"

namespace {

constexpr int MC = 64;          // MSA channels
constexpr int WLD = MC + 8;     // LDS row stride of a [.][64] weight (bf16)
constexpr int MAX_HIDDEN = 256;

__device__ __forceinline__ int swap23(int r) { return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1); }

// a lane's 32 channels of one position, as loaded
template <typename TIO>
struct Position {
  typename Elem<TIO>::Raw r[4];
  __device__ __forceinline__ void load(const TIO* p, int hh) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) r[ks] = Elem<TIO>::load_raw(p + 16 * ks + 8 * hh);
  }
  __device__ __forceinline__ void unpack(float* v) const {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) Elem<TIO>::unpack_raw(r[ks], v + 8 * ks);
  }
};

// Sum over a position's eight chunks (a lane's four and those of the other half of the wave), as a tree over the chunks
// in their order.
__device__ __forceinline__ float chunk_sum(const float* c, int xaddr) {
  float t[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) t[ks] = c[ks] + half_swap(xaddr, c[ks]);
  return (t[0] + t[1]) + (t[2] + t[3]);
}

// a * b + c, rounded twice: as the row norms of rowops.hip compute weight and bias
__device__ __forceinline__ float mul_add(float a, float b, float c) {
#pragma clang fp contract(off)
  const float t = a * b;
  return t + c;
}

// LayerNorm of a position -> the four k-step fragments.  sLn: weight [64], bias [64].  ONE_PASS: sum and sum of squares
// together, as the pair's tile kernels take a bf16 stream.
template <bool ONE_PASS>
__device__ __forceinline__ void layer_norm_frags(const float* v, const float* sLn, int hh, int xaddr, bf16x8* f) {
  float cs[4], cq[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    cs[ks] = cq[ks] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      cs[ks] += v[8 * ks + e];
      if (ONE_PASS) cq[ks] = fmaf(v[8 * ks + e], v[8 * ks + e], cq[ks]);
    }
  }
  const float mean = chunk_sum(cs, xaddr) * (1.f / MC);
  if (!ONE_PASS) {
#pragma unroll
    for (int i = 0; i < 32; ++i) { const float d = v[i] - mean; cq[i >> 3] += d * d; }
  }
  const float q = chunk_sum(cq, xaddr);
  const float rstd = rsqrtf(ONE_PASS ? fmaxf(fmaf(q, 1.f / MC, -mean * mean), 0.f) + LN_EPS : q * (1.f / MC) + LN_EPS);
  const float shift = -mean * rstd;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    float w[8], b[8], o[8];
    Elem<float>::load8(sLn + 16 * ks + 8 * hh, w);
    Elem<float>::load8(sLn + MC + 16 * ks + 8 * hh, b);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      o[e] = ONE_PASS ? fmaf(fmaf(v[8 * ks + e], rstd, shift), w[e], b[e])
                      : mul_add((v[8 * ks + e] - mean) * rstd, w[e], b[e]);
    f[ks] = as_frag(pack8(o));
  }
}

// Zero, as far as the compiler knows a new value each time: an LDS address with it added is not loop-invariant, and
// what is read there (weights, LayerNorm parameters) is not kept in registers that the loop has better use for.
__device__ __forceinline__ int fresh_zero() {
  int z = 0;
  asm volatile("" : "+s"(z));
  return z;
}

__device__ __forceinline__ f32x16 zero16() { return f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}; }

// ------------------------------------------------------------------ projections, transposed
// y = LayerNorm(msa) W^T (64 outputs) with the outputs as rows and a run of positions innermost:
//   VALUES = false: positions are MSA rows of one token b; outputs 0..31 (left) and 32..63 (right) times mask[row][b]
//                   to out[0 / 1][(b, c)][ld], ld = rows rounded up to 8;
//   VALUES = true:  positions are tokens k of one MSA row a; output c = (head, d) to out[0][(head, a, d)][ld],
//                   ld = n rounded up to 8.
// Entries past the count are zero.  A wave takes 64 positions (a 128-byte line of every output row) at a time; the
// weights stay in its registers.
template <typename TIO, bool VALUES>
__global__ __launch_bounds__(256) void msa_project_kernel(MsaProjectArgs a) {
  __shared__ __attribute__((aligned(16))) float sLn[2 * MC];
  __shared__ __attribute__((aligned(16))) float sMask[4][64];
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, l31 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < MC) {
    sLn[tid] = a.ln_w[tid];
    sLn[MC + tid] = a.ln_b[tid];
  }
  __syncthreads();
  const int xaddr = half_swap_addr();
  bf16x8 wf[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      wf[t][ks] = as_frag(*reinterpret_cast<const u32x4*>(a.w + (32 * t + l31) * MC + 16 * ks + 8 * hh));
  const int lines = VALUES ? a.rows : a.n, count = VALUES ? a.n : a.rows;
  const int per_line = ((int)a.ld + 63) / 64, tiles = lines * per_line;
  const TIO* msa = reinterpret_cast<const TIO*>(a.msa);
  for (int tile = blockIdx.x * 4 + wave; tile < tiles; tile += gridDim.x * 4) {
    // neighbours in memory side by side: tokens of an MSA row
    const int line = __builtin_amdgcn_readfirstlane(VALUES ? tile / per_line : tile % lines);
    const int first = __builtin_amdgcn_readfirstlane(64 * (VALUES ? tile % per_line : tile / lines));
    Position<TIO> pos[2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int p = first + 32 * sub + swap23(l31), pc = min(p, count - 1);
      const int64_t pix = VALUES ? (int64_t)line * a.n + pc : (int64_t)pc * a.n + line;
      pos[sub].load(msa + pix * MC, hh);
      if constexpr (!VALUES) sMask[wave][32 * sub + swap23(l31)] = p < count ? bf2f(f2bf(a.mask[pix])) : 0.f;
    }
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int z = fresh_zero();
      float v[32];
      bf16x8 xf[4];
      pos[sub].unpack(v);
      layer_norm_frags<false>(v, sLn + z, hh, xaddr, xf);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x16 acc = zero16();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc = mfma32(xf[ks], wf[t][ks], acc);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int at = first + 32 * sub + 16 * s + 8 * hh;
          float o[8];
          if constexpr (!VALUES) Elem<float>::load8(&sMask[wave][32 * sub + 16 * s + 8 * hh], o);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float y = acc[8 * s + e];
            if constexpr (VALUES) o[e] = at + e < count ? y : 0.f;
            else o[e] *= bf2f(f2bf(y));
          }
          const int c = 32 * t + l31;
          bf16_t* row = VALUES ? a.out[0] + (((int64_t)(c >> 3) * a.rows + line) * 8 + (c & 7)) * a.ld
                               : a.out[t] + ((int64_t)line * 32 + l31) * a.ld;
          if (at < a.ld) *reinterpret_cast<u32x4*>(row + at) = pack8(o);
        }
      }
    }
  }
}

// ------------------------------------------------------------------ the MSA's own update
// ATT:   x += W_o (avg * sigmoid(W_g LayerNorm(x)))      (avg: the weighted average, [head][token][row][8])
// TRANS: x += W_2 (silu(W_a LayerNorm(x)) * W_b LayerNorm(x))
// in one pass: a position needs nothing of any other.  The stream is rounded to its type between the two.  (Without
// `residual` the update alone is written.)
// Vector arithmetic decides: the SiLU gates of 256 hidden units cost a SIMD about twice the time of the MFMAs.  All
// weights (126 KB) sit in LDS for a workgroup's lifetime, one workgroup of eight waves per CU.  The MFMAs of a slab of
// 32 hidden units are issued with the gating of the previous one between them.
template <typename TIO, bool ATT, bool TRANS>
__global__ __launch_bounds__(512, 2) void msa_update_kernel(MsaUpdateArgs a) {
  __shared__ __attribute__((aligned(16))) bf16_t sG[ATT ? MC * WLD : 8], sO[ATT ? MC * WLD : 8];
  __shared__ __attribute__((aligned(16))) bf16_t sW1[TRANS ? 2 * MAX_HIDDEN * WLD : 8], sW2[TRANS ? MC * (MAX_HIDDEN + 8) : 8];
  __shared__ __attribute__((aligned(16))) float sLn[4 * MC];
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, l31 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ld2 = a.hidden + 8;
  auto copy = [&](bf16_t* dst, int ld, const bf16_t* src, int rows, int cols) {
    for (int i = tid; i < rows * (cols / 8); i += 512) {
      const int r = i / (cols / 8), c = (i % (cols / 8)) * 8;
      *reinterpret_cast<u32x4*>(dst + r * ld + c) = *reinterpret_cast<const u32x4*>(src + r * cols + c);
    }
  };
  if constexpr (ATT) {
    copy(sG, WLD, a.w_g, MC, MC);
    copy(sO, WLD, a.w_o, MC, MC);
    if (tid < MC) { sLn[tid] = a.att_ln_w[tid]; sLn[MC + tid] = a.att_ln_b[tid]; }
  }
  if constexpr (TRANS) {
    copy(sW1, WLD, a.w1, 2 * a.hidden, MC);
    copy(sW2, ld2, a.w2, MC, a.hidden);
    if (tid < MC) { sLn[2 * MC + tid] = a.tr_ln_w[tid]; sLn[3 * MC + tid] = a.tr_ln_b[tid]; }
  }
  __syncthreads();
  const int xaddr = half_swap_addr(), sw = swap23(l31);
  const int tiles = a.n * ((a.rows + 31) / 32);
  const TIO* msa = reinterpret_cast<const TIO*>(a.msa);
  TIO* out = reinterpret_cast<TIO*>(a.out);
  int z = 0;
  auto weight = [&](const bf16_t* w, int ld, int row, int k) {
    return as_frag(*reinterpret_cast<const u32x4*>(w + z + (row + sw) * ld + k + 8 * hh));
  };
  auto product64 = [&](const bf16_t* w, int row, const bf16x8* x) {  // 32 outputs from 64 channels
    f32x16 acc = zero16();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) acc = mfma32(weight(w, WLD, row, 16 * ks), x[ks], acc);
    return acc;
  };
  // v (32 channels of the lane) = res ? v + y : y, rounded to the stream's type
  auto add = [&](float* v, const f32x16* y) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      v[i] = y[i >> 4][i & 15] + (a.residual ? v[i] : 0.f);
      if constexpr (ATT && TRANS && sizeof(TIO) == 2) v[i] = bf2f(f2bf(v[i]));
    }
  };
  for (int tile = blockIdx.x * 8 + wave; tile < tiles; tile += gridDim.x * 8) {
    z = fresh_zero();
    const int q = __builtin_amdgcn_readfirstlane(tile % a.n), first = __builtin_amdgcn_readfirstlane(tile / a.n * 32);
    const int p = first + l31, pc = min(p, a.rows - 1);
    const int64_t pix = (int64_t)pc * a.n + q;
    Position<TIO> pos;
    pos.load(msa + pix * MC, hh);
    u32x4 avg[4];
    if constexpr (ATT) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)  // channels 16 ks + 8 hh ..: head 2 ks + hh
        avg[ks] = *reinterpret_cast<const u32x4*>(a.avg + (((int64_t)(2 * ks + hh) * a.n + q) * a.rows + pc) * 8);
    }
    float v[32];
    bf16x8 xf[4];
    pos.unpack(v);
    if constexpr (ATT) {
      layer_norm_frags<false>(v, sLn + z, hh, xaddr, xf);
      bf16x8 gated[4];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const f32x16 g = product64(sG, 32 * t, xf);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          float o[8];
          unpack8(avg[2 * t + s], o);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] *= bf2f(f2bf(sigmoidf_(g[8 * s + e])));
          gated[2 * t + s] = as_frag(pack8(o));
        }
      }
      const f32x16 y[2] = {product64(sO, 0, gated), product64(sO, 32, gated)};
      add(v, y);
    }
    if constexpr (TRANS) {
      layer_norm_frags<sizeof(TIO) == 2>(v, sLn + 2 * MC + z, hh, xaddr, xf);
      f32x16 y[2] = {zero16(), zero16()};
      f32x16 ga = product64(sW1, 0, xf), gb = product64(sW1, a.hidden, xf);
      for (int h = 0; h < a.hidden; h += 32) {
        const int nx = h + 32 < a.hidden ? h + 32 : 0;  // (behind the last slab: the first again, unused)
        const f32x16 na = product64(sW1, nx, xf), nb = product64(sW1, a.hidden + nx, xf);
        bf16x8 hf[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          float o[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float g = ga[8 * s + e];
            o[e] = g * sigmoidf_(g) * gb[8 * s + e];
          }
          hf[s] = as_frag(pack8(o));
#pragma unroll
          for (int t = 0; t < 2; ++t) y[t] = mfma32(weight(sW2, ld2, 32 * t, h + 16 * s), hf[s], y[t]);
        }
        ga = na;
        gb = nb;
      }
      add(v, y);
    }
    if (p < a.rows) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) Elem<TIO>::store8(out + pix * MC + 16 * ks + 8 * hh, v + 8 * ks);
    }
  }
}

// ------------------------------------------------------------------ what the MSA mask decides
// inv[b][d] = 1 / (eps + sum over rows of m[row][b] m[row][d]),  live[b] = max over rows of m[row][b].
// A 32 x 32 block per workgroup on the fp32 matrix instruction, whose operands are rows of the mask as they lie; the
// eight waves share the MSA rows and meet in LDS.  What it costs is the chain of loads and MFMAs over rows / 8.
__global__ __launch_bounds__(512) void msa_coverage_kernel(const float* m, int rows, int n, float eps, float* inv, float* live) {
  __shared__ float part[8][32 * 33];
  __shared__ float top[8][64];
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, l31 = lane & 31, wave = tid >> 6;
  const int b0 = blockIdx.x * 32, d0 = blockIdx.y * 32;
  const int b = min(b0 + l31, n - 1), d = min(d0 + l31, n - 1);
  const int share = (rows + 15) / 16 * 2, end = min(rows, (wave + 1) * share);
  f32x16 acc = zero16();
  float mx = -__builtin_huge_valf();
  constexpr int U = 16;
  for (int k = wave * share; k < end; k += 2 * U) {
    float x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = min(k + 2 * u + hh, rows - 1);
      x[u] = m[(int64_t)r * n + b];
      y[u] = m[(int64_t)r * n + d];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool ok = k + 2 * u + hh < end;
      mx = fmaxf(mx, x[u]);  // (a repeated row changes no maximum)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ok ? x[u] : 0.f, ok ? y[u] : 0.f, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) part[wave][acc_row(r, lane) * 33 + l31] = acc[r];
  top[wave][lane] = mx;
  __syncthreads();
  for (int i = tid; i < 1024; i += 512) {
    const int r = i >> 5, c = i & 31, o = r * 33 + c;
    float sum = 0.f;
    for (int w = 0; w < 8; ++w) sum += part[w][o];
    if (b0 + r < n && d0 + c < n)
      inv[(int64_t)(b0 + r) * n + d0 + c] = 1.f / (eps + sum);
  }
  if (blockIdx.y == 0 && tid < 32 && b0 + tid < n) {
    float t = top[0][tid];
    for (int w = 0; w < 8; ++w) t = fmaxf(t, fmaxf(top[w][tid], top[w][tid + 32]));
    live[b0 + tid] = t;
  }
}

__global__ __launch_bounds__(256) void transpose_f32_kernel(const float* in, float* out, int n) {
  __shared__ float tile[32][33];
  const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5, i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  for (int r = r0; r < 32; r += 8)
    if (i0 + r < n && j0 + c < n) tile[r][c] = in[(int64_t)(i0 + r) * n + j0 + c];
  __syncthreads();
  for (int r = r0; r < 32; r += 8)
    if (j0 + r < n && i0 + c < n) out[(int64_t)(j0 + r) * n + i0 + c] = tile[c][r];
}

int status() { return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH; }
bool bad_size(int rows, int n) { return rows <= 0 || n <= 0 || (int64_t)rows * n > (1ll << 30); }
bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int launch_msa_project(const MsaProjectArgs& a, bool values, hipStream_t s) {
  if (bad_size(a.rows, a.n) || !a.msa || !a.ln_w || !a.ln_b || !a.w || !a.out[0] || (!values && (!a.out[1] || !a.mask)))
    return AF3_ERR_BAD_ARG;
  if (!al16(a.msa) || !al16(a.w) || !al16(a.out[0]) || !al16(a.out[1]) || a.ld != ((values ? a.n : a.rows) + 7) / 8 * 8)
    return AF3_ERR_BAD_ARG;
  // up to eight workgroups per CU; a wave of a long product takes several tiles, its weights stay
  const int64_t tiles = (int64_t)(values ? a.rows : a.n) * ((a.ld + 63) / 64);
  const dim3 grid((unsigned)((tiles + 3) / 4 < 2048 ? (tiles + 3) / 4 : 2048)), block(256);
  if (a.io_f32) {
    if (values) hipLaunchKernelGGL((msa_project_kernel<float, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((msa_project_kernel<float, false>), grid, block, 0, s, a);
  } else {
    if (values) hipLaunchKernelGGL((msa_project_kernel<bf16_t, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((msa_project_kernel<bf16_t, false>), grid, block, 0, s, a);
  }
  return status();
}

int launch_msa_update(const MsaUpdateArgs& a, hipStream_t s) {
  const bool att = a.avg != nullptr, trans = a.w1 != nullptr;
  if (bad_size(a.rows, a.n) || !a.msa || !a.out || (!att && !trans) || !al16(a.msa) || !al16(a.out)) return AF3_ERR_BAD_ARG;
  if (att && (!a.att_ln_w || !a.att_ln_b || !a.w_g || !a.w_o || !al16(a.avg) || !al16(a.w_g) || !al16(a.w_o))) return AF3_ERR_BAD_ARG;
  if (trans && (!a.tr_ln_w || !a.tr_ln_b || !a.w2 || !al16(a.w1) || !al16(a.w2) || a.hidden <= 0 || (a.hidden & 31) || a.hidden > MAX_HIDDEN))
    return AF3_ERR_BAD_ARG;
  if (att && trans && !a.residual) return AF3_ERR_BAD_ARG;  // the transition reads the updated stream
  const int64_t tiles = (int64_t)a.n * ((a.rows + 31) / 32);
  const dim3 grid((unsigned)((tiles + 7) / 8 < 256 ? (tiles + 7) / 8 : 256)), block(512);
#define MSA_UPDATE(A, T)                                                                              \
  do {                                                                                                \
    if (a.io_f32) hipLaunchKernelGGL((msa_update_kernel<float, A, T>), grid, block, 0, s, a);         \
    else hipLaunchKernelGGL((msa_update_kernel<bf16_t, A, T>), grid, block, 0, s, a);                 \
  } while (0)
  if (att && trans) MSA_UPDATE(true, true);
  else if (att) MSA_UPDATE(true, false);
  else MSA_UPDATE(false, true);
#undef MSA_UPDATE
  return status();
}

int launch_msa_coverage(const float* mask, int rows, int n, float eps, float* inv, float* live, hipStream_t s) {
  if (bad_size(rows, n) || !mask || !inv || !live) return AF3_ERR_BAD_ARG;
  const unsigned t = (unsigned)(n + 31) / 32;
  hipLaunchKernelGGL(msa_coverage_kernel, dim3(t, t), dim3(512), 0, s, mask, rows, n, eps, inv, live);
  return status();
}

int launch_transpose_f32(const float* in, float* out, int n, hipStream_t s) {
  if (!in || !out || n <= 0) return AF3_ERR_BAD_ARG;
  const unsigned t = (unsigned)(n + 31) / 32;
  hipLaunchKernelGGL(transpose_f32_kernel, dim3(t, t), dim3(256), 0, s, in, out, n);
  return status();
}
