// Device helpers shared by the row-tile kernels of the 128-channel pair path:
// tile geometry, LayerNorm of a 128-pixel tile into LDS, weight staging, MFMA
// chunk products in "D form" (out[px][ch], lane owns a channel) or "T form"
// (out^T[ch][px], lane owns a pixel), and staged stores.
#pragma once
#include "common.h"

namespace {

constexpr int C = 128;    // pair channels
constexpr int TM = 128;   // positions per tile
constexpr int LDX = 136;  // LDS row stride (bf16) for [row][128] tiles: 272 B
constexpr int LDS_F = 132;  // LDS row stride (fp32) for staged output tiles

// A tile is TM consecutive positions of the operator's frame laid out flat, rows o of W positions each: W = N, or N
// rounded up to what the kernel's channel-major planes are padded to (positions N .. W - 1 of a row are padding).
// A tile runs on from one row into the next, so that a row length that is no multiple of TM costs no partly filled
// tile per row (at 387 tokens a quarter, at 160 three eighths of the positions computed).  Position (o, r) is pixel
// o * so + r * sr of the pair tensor.
// CROSS: false where W is a multiple of TM (or there is one row): the row is the workgroup's, and the indexing costs
// nothing.
template <bool CROSS>
struct TileT {
  int l0;          // flat index of the first position
  int o0, r0;      // its row and place in the row
  int N, W;
  uint32_t magic;  // CROSS: ceil(2^32 / W); v / W = umulhi(v, magic) for v < W + TM, as W (W + TM) < 2^32
  int64_t so, sr;
  __device__ __forceinline__ void at(int p, int* o, int* r) const {
    *o = o0;
    *r = r0 + p;
    if constexpr (CROSS) {
      const int q = (int)__umulhi((uint32_t)*r, magic);
      *o += q;
      *r -= q * W;
    }
  }
  __device__ __forceinline__ bool valid(int p) const {
    int o, r;
    at(p, &o, &r);
    return r < N && (!CROSS || o < N);
  }
  // pixel of position p; of one that is not valid, that of some valid position
  __device__ __forceinline__ int64_t pix(int p) const {
    int o, r;
    at(p, &o, &r);
    if constexpr (CROSS) return r < N && o < N ? (uint32_t)o * (uint32_t)so + (uint32_t)r * (uint32_t)sr : 0u;
    return (int64_t)o * so + (int64_t)(r < N ? r : r0) * sr;
  }
  // every position is valid (uniform over the workgroup; rows that are crossed are left to the per-position test)
  __device__ __forceinline__ bool full() const { return r0 + TM <= N; }
};

// `reverse`: walk the tiles from the last to the first.  A kernel that reads
// what the previous kernel has just written (and whose output the next kernel
// starts reading from the other end) finds the most recently written part
// still in the last-level cache when it starts there.
template <bool CROSS>
__device__ __forceinline__ TileT<CROSS> make_tile(int N, int W, bool column_mode, bool reverse = false) {
  TileT<CROSS> t;
  const unsigned bid = reverse ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
  t.N = N;
  t.W = W;
  // (the divisions go through the vector unit; say again that the results are uniform)
  const uint32_t o0 = __builtin_amdgcn_readfirstlane(bid * TM / (uint32_t)W);
  t.l0 = (int)(bid * TM);
  t.o0 = (int)o0;
  t.r0 = t.l0 - (int)o0 * W;
  t.magic = W == 1 ? 1u : __builtin_amdgcn_readfirstlane(0xffffffffu / (uint32_t)W) + 1u;  // (W = 1: one pixel, position 0)
  t.so = column_mode ? 1 : N;
  t.sr = column_mode ? N : 1;
  return t;
}
inline bool tile_crosses(int64_t W) { return W % TM != 0; }
// One row of n positions (any count).
__device__ __forceinline__ TileT<false> make_tile_1d(int n) {
  TileT<false> t;
  t.N = t.W = n;
  t.l0 = t.r0 = (int)blockIdx.x * TM;
  t.o0 = 0;
  t.so = 0;
  t.sr = 1;
  return t;
}
// A piece of one row: tiles do not cross rows (the kernel takes per-row values from o0).
__device__ __forceinline__ TileT<false> make_tile_in_row(int N) {
  const int tiles_r = (N + TM - 1) / TM;
  TileT<false> t;
  t.N = t.W = N;
  t.o0 = blockIdx.x / tiles_r;
  t.r0 = (blockIdx.x % tiles_r) * TM;
  t.l0 = t.o0 * N + t.r0;
  t.so = N;
  t.sr = 1;
  return t;
}

// 32 queries x 4 keys of the pair: position p is query q0 + p / 4, key 4 quad + p % 4; a wave's 32 positions are 8 quads.
struct TileQuads {
  int N, q0, quad, quads;
  __device__ __forceinline__ int query(int p) const { return q0 + (p >> 2); }
  __device__ __forceinline__ bool valid(int p) const { return query(p) < N && 4 * quad + (p & 3) < N; }
  __device__ __forceinline__ int64_t pix(int p) const {
    return (int64_t)min(query(p), N - 1) * N + min(4 * quad + (p & 3), N - 1);
  }
  __device__ __forceinline__ bool full() const { return q0 + 32 <= N && 4 * quad + 4 <= N; }
};
__device__ __forceinline__ TileQuads make_tile_quads(int N) {
  TileQuads t;
  t.N = N;
  t.quads = (N + 3) / 4;
  t.quad = blockIdx.x % t.quads;
  t.q0 = blockIdx.x / t.quads * 32;
  return t;
}

// Eight consecutive fp32 parameters (LayerNorm weight / bias slice of a thread),
// or a constant when the pointer is null.
__device__ __forceinline__ void load_param8(const float* p, float fill, float* out) {
  if (p) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p);
    const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
    out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
    out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = fill;
  }
}

// LayerNorm of one pixel's eight channels (the thread's share: LANES lanes cooperate on the
// pixel's statistics) -> packed bf16.
//
// This phase is vector arithmetic per element and a large share of every tile
// kernel's instructions, so the bf16 stream takes the short form: sum and sum of
// squares in one pass (variance = E[x^2] - mean^2 in fp32: the error relative to
// the variance is 1e-7 (1 + mean^2 / variance), and a bf16 tensor cannot hold a
// mean of more than ~2^8 standard deviations to begin with), normalisation as two
// FMAs per element (x * rstd - mean * rstd, then * w + b), and no per-element
// select when every pixel of the tile is in range.  The fp32 stream keeps the
// two-pass form.  Zero-padded channels (fewer than 128 real ones) add nothing to
// either sum; the two-pass form takes their pad * mean^2 out again.
// ROUNDED (fp32 rows): rowops.hip's row LayerNorm to the last bit, with its order of the sums and the product with the weight
// rounded before the bias is added.
template <typename TIO, int LANES = 16, bool ROUNDED = false>
__device__ __forceinline__ u32x4 ln_pixel8(const typename Elem<TIO>::Raw& raw, const float* w, const float* b,
                                           bool skip_ln, float inv_c, float pad) {
  using E = Elem<TIO>;
  constexpr bool ONE_PASS = sizeof(TIO) == 2;
  float v[8], o[8];
  E::unpack_raw(raw, v);
  if (ONE_PASS) {
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { s += v[e]; q = fmaf(v[e], v[e], q); }
    const float mean = group_sum<LANES>(s) * inv_c;
    const float var = fmaxf(fmaf(group_sum<LANES>(q), inv_c, -mean * mean), 0.f);
    // (an already normalised input comes with w = 1, b = 0: scale 1 and shift 0 pass it through unchanged)
    const float rstd = skip_ln ? 1.f : rsqrtf(var + LN_EPS);
    const float shift = skip_ln ? 0.f : -mean * rstd;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = fmaf(fmaf(v[e], rstd, shift), w[e], b[e]);
  } else {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += v[e];
    auto sum = [](float x) { return ROUNDED ? group16_sum_halving(x) : group_sum<LANES>(x); };
    const float mean = sum(s) * inv_c;
    float q = 0.f;
    if constexpr (ROUNDED) {
      float d[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] = v[e] - mean;
      q = add_squares8(d, 0.f, true);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = v[e] - mean; q += d * d; }
    }
    // (zero-padded channels, if any, each put mean^2 into the sum)
    const float rstd = rsqrtf((sum(q) - pad * mean * mean) * inv_c + LN_EPS);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (ROUNDED) {
#pragma clang fp contract(off)
        const float t = (v[e] - mean) * rstd * w[e];
        o[e] = t + b[e];
      } else {
        o[e] = skip_ln ? v[e] : (v[e] - mean) * rstd * w[e] + b[e];
      }
    }
  }
  return pack8(o);
}

// LayerNorm of a tile of pixels from global memory into sX[p][c] (bf16).
// Thread (prow = tid / 16, chunk = tid % 16) handles channels 8*chunk..+7 of
// pixels prow, prow + 16, ...; 16 lanes cooperate on one pixel's statistics.
// Out-of-range pixels become zero rows.  The loads of a batch of pixels are
// unconditional (an out-of-range position re-reads some valid pixel) and all
// issued before any value is converted: a load under a lane mask, or one whose
// value is touched at once, costs a full memory round trip per pixel.
template <typename TIO, bool ROUNDED = false, typename Tile>
__device__ __forceinline__ void load_ln_tile(const TIO* x, const Tile& t, const float* lnw,
                                             const float* lnb, bf16_t* sX, int tid, bool skip_ln = false,
                                             float inv_c = 1.f / C, float pad = 0.f) {
  using E = Elem<TIO>;
  constexpr int NB = E::kBatch;
  const int chunk = tid & 15, prow = tid >> 4;
  float w[8], b[8];
  load_param8(lnw ? lnw + chunk * 8 : nullptr, 1.f, w);
  load_param8(lnb ? lnb + chunk * 8 : nullptr, 0.f, b);
  const bool full = t.full();
#pragma unroll
  for (int base = 0; base < 8; base += NB) {
    typename E::Raw raw[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int p = (base + i) * 16 + prow;
      raw[i] = E::load_raw(x + t.pix(p) * C + chunk * 8);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int p = (base + i) * 16 + prow;
      u32x4 pk = ln_pixel8<TIO, 16, ROUNDED>(raw[i], w, b, skip_ln, inv_c, pad);
      if (!full && !t.valid(p)) pk = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(sX + p * LDX + chunk * 8) = pk;
    }
  }
}

// Channel sums of the LayerNorm of a contraction's result: eight channels one after the other, then the eight k-steps of a
// half (channels 16 ks + 8 half ..) in this order, then the two halves.  sum_k_steps: all k-steps in one lane;
// sum_chunks: 16 lanes, lane 2 ks + half of a row of 16, the halves included.
__device__ __forceinline__ float sum_k_steps(const float* s) {
  return ((s[0] + s[1]) + (s[4] + s[5])) + ((s[2] + s[3]) + (s[6] + s[7]));
}
__device__ __forceinline__ float sum_chunks(float s) {
  s += dpp_mov<0x4E>(s);   // quad_perm [2,3,0,1]: ks ^ 1
  s += dpp_mov<0x128>(s);  // row_ror:8: ks ^ 4
  s += dpp_mov<0x124>(s);  // row_ror:4: the other two of these sums, ks ^ 2 (either way round: the lanes 8 apart agree)
  return s + dpp_mov<0xB1>(s);  // quad_perm [1,0,3,2]: the halves
}

// In-place LayerNorm of the rows of sX (bf16 in LDS), same thread mapping.
__device__ __forceinline__ void ln_inplace_tile(bf16_t* sX, const float* lnw, const float* lnb, int tid) {
  const int chunk = tid & 15, prow = tid >> 4;
  float w[8], b[8];
  load_param8(lnw + chunk * 8, 1.f, w);
  load_param8(lnb + chunk * 8, 0.f, b);
#pragma unroll
  for (int it = 0; it < 8; ++it) {
    const int p = it * 16 + prow;
    float v[8];
    unpack8(*reinterpret_cast<const u32x4*>(sX + p * LDX + chunk * 8), v);
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += v[e];
    const float mean = group16_sum(s) * (1.f / C);
    float q = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { const float d = v[e] - mean; q += d * d; }
    const float rstd = rsqrtf(group16_sum(q) * (1.f / C) + LN_EPS);
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (v[e] - mean) * rstd * w[e] + b[e];
    *reinterpret_cast<u32x4*>(sX + p * LDX + chunk * 8) = pack8(o);
  }
}

// Copy `rows` x 128 bf16 weights (row-major, contiguous) into sW[row][LDX].
__device__ __forceinline__ void load_w_rows(const bf16_t* gW, bf16_t* sW, int rows, int tid) {
  for (int idx = tid; idx < rows * 16; idx += 256) {
    const int row = idx >> 4, ch = idx & 15;
    *reinterpret_cast<u32x4*>(sW + row * LDX + ch * 8) =
        *reinterpret_cast<const u32x4*>(gW + row * C + ch * 8);
  }
}

// The wave's 32 pixels as 8 k-step fragments (k = 128 channels).
__device__ __forceinline__ void load_x_frags(const bf16_t* sX, int wave, int lane, bf16x8* xf) {
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) xf[ks] = lds_frag(sX, LDX, wave * 32, ks * 16, lane);
}

// acc[nt] = tile nt (32 weight rows) of  X * W^T  (D form) or  W * X^T  (T form)
template <bool TFORM, int NT>
__device__ __forceinline__ void mfma_chunk(const bf16x8* xf, const bf16_t* sW, int lane, f32x16* acc) {
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nt][r] = 0.f;
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ks = 0; ks < 8; ++ks)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const bf16x8 wf = lds_frag(sW, LDX, nt * 32, ks * 16, lane);
      acc[nt] = TFORM ? mfma32(wf, xf[ks], acc[nt]) : mfma32(xf[ks], wf, acc[nt]);
    }
  // Weight fragments are read four ahead of the MFMAs that use them (left to
  // itself the compiler reads each one right in front of its MFMA and waits).
  __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
  for (int i = 0; i < 8 * NT - 4; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
  __builtin_amdgcn_sched_barrier(0);
}

// T-form accumulators (lane = pixel, 4 consecutive channels per register
// quad) -> fp32 staging tile sS[px][LDS_F].
__device__ __forceinline__ void stage_t_f32(const f32x16* acc, float* sS, int wave, int lane) {
  const int px = wave * 32 + (lane & 31);
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int ch = nt * 32 + 8 * g + 4 * (lane >> 5);
      f32x4 v = {acc[nt][4 * g], acc[nt][4 * g + 1], acc[nt][4 * g + 2], acc[nt][4 * g + 3]};
      *reinterpret_cast<f32x4*>(sS + px * LDS_F + ch) = v;
    }
}

// T-form accumulators -> bf16 staging tile sS[px][LDX]
__device__ __forceinline__ void stage_t_bf16(const f32x16* acc, bf16_t* sS, int wave, int lane) {
  const int px = wave * 32 + (lane & 31);
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int ch = nt * 32 + 8 * g + 4 * (lane >> 5);
      u32x2 v;
      v.x = pack2bf(acc[nt][4 * g], acc[nt][4 * g + 1]);
      v.y = pack2bf(acc[nt][4 * g + 2], acc[nt][4 * g + 3]);
      *reinterpret_cast<u32x2*>(sS + px * LDX + ch) = v;
    }
}

// Staged fp32 tile -> residual stream: out[pix] = (res ? res[pix] : 0) + tile.
// The residual rows of a batch of pixels are loaded (unconditionally, from a
// clamped pixel) before the batch's first store: out may alias res, so the
// compiler cannot move a load above a store on its own.
template <typename TIO, typename Tile>
__device__ __forceinline__ void store_tile_f32(const float* sS, const Tile& t, TIO* out, const TIO* res, int tid) {
  using E = Elem<TIO>;
  constexpr int NB = E::kBatch;
  const int chunk = tid & 15, prow = tid >> 4;
#pragma unroll
  for (int base = 0; base < 8; base += NB) {
    typename E::Raw raw[NB];
    if (res) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int p = (base + i) * 16 + prow;
        raw[i] = E::load_raw(res + t.pix(p) * C + chunk * 8);
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int p = (base + i) * 16 + prow;
      float v[8];
      const f32x4 a = *reinterpret_cast<const f32x4*>(sS + p * LDS_F + chunk * 8);
      const f32x4 b = *reinterpret_cast<const f32x4*>(sS + p * LDS_F + chunk * 8 + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
      if (res) {
        float rr[8];
        E::unpack_raw(raw[i], rr);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += rr[e];
      }
      if (t.valid(p)) E::store8(out + t.pix(p) * C + chunk * 8, v);
    }
  }
}


// 128 x 128 bf16 weight chunk held in registers between a global load and the
// LDS store, so the load overlaps the MFMA work on the previous chunk.
struct WChunkRegs {
  u32x4 r[8];
  // SWAP23: register row rho receives weight row swap23(rho) (bits 2 and 3 exchanged)
  template <bool SWAP23 = false>
  __device__ __forceinline__ void load(const bf16_t* gW, int tid) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int idx = tid + 256 * i, rho = idx >> 4;
      const int row = SWAP23 ? ((rho & ~12) | ((rho & 4) << 1) | ((rho & 8) >> 1)) : rho;
      r[i] = *reinterpret_cast<const u32x4*>(gW + row * C + (idx & 15) * 8);
    }
  }
  __device__ __forceinline__ void store(bf16_t* sW, int tid) const {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<u32x4*>(sW + (idx >> 4) * LDX + (idx & 15) * 8) = r[i];
    }
  }
};

// element `off` (32 bits: every array here is below 2 GB) of an array
template <typename T>
__device__ __forceinline__ T* at32(T* base, uint32_t off) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ const T* at32(const T* base, uint32_t off) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off * (uint32_t)sizeof(T));
}

template <typename TIO> __device__ __forceinline__ typename Elem<TIO>::Raw pack_raw(const float* v);
template <> __device__ __forceinline__ Elem<bf16_t>::Raw pack_raw<bf16_t>(const float* v) { return {pack8(v)}; }
template <> __device__ __forceinline__ Elem<float>::Raw pack_raw<float>(const float* v) {
  return {f32x4{v[0], v[1], v[2], v[3]}, f32x4{v[4], v[5], v[6], v[7]}};
}
template <typename TIO> __device__ __forceinline__ void store_raw(TIO* p, const typename Elem<TIO>::Raw& r);
template <> __device__ __forceinline__ void store_raw<bf16_t>(bf16_t* p, const Elem<bf16_t>::Raw& r) { *reinterpret_cast<u32x4*>(p) = r.v; }
template <> __device__ __forceinline__ void store_raw<float>(float* p, const Elem<float>::Raw& r) {
  *reinterpret_cast<f32x4*>(p) = r.a;
  *reinterpret_cast<f32x4*>(p + 4) = r.b;
}

// 64 lanes x 16 bytes from memory (uniform base, a byte offset per lane) to 1 KB of LDS at `lds`.  Inline assembly, because the
// compiler's own form makes later LDS reads wait for every such load in flight; the panel is read behind a wait of its own.
__device__ __forceinline__ void load_to_lds(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:0" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}

// fragments of 32 weight rows (block `blk`) for `n` k-steps from k-step k0 on, of a matrix with `nks` k-steps
template <int n>
__device__ __forceinline__ void load_frags(const bf16_t* w, int blk, int nks, int k0, int lane, bf16x8* f) {
  const bf16_t* p = w + (blk * nks + k0) * 512;  // (uniform)
#pragma unroll
  for (int i = 0; i < n; ++i) f[i] = as_frag(*reinterpret_cast<const u32x4*>(at32(p + i * 512, (uint32_t)lane * 8u)));
}

}  // namespace
