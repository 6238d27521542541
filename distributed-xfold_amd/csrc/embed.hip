// Element-wise passes between the kernels: the trunk's input embedding and the diffusion head's scaling and blending.
// Each stands for a run of single operations (ten to forty launches of 2 to 5 us, most of them on a few kilobytes, and
// as many passes over the pair tensor), and rounds as they do: every operation of its own, nothing fused into an FMA.
//
// Trunk pass at 160 tokens, 128 MSA rows: embedding 380 us in 78 launches before.  The head's atom conditioning at 384 tokens: 75
// launches less, whose host time (1060 us, 590 now) the GPU had nothing else to do in; a new batch 4460 -> 4080 us.
#pragma clang fp contract(off)
#include "common.h"
#include "kernels.h"

namespace {

template <typename F>
__global__ __launch_bounds__(256) void each_kernel(int64_t n, F f) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) f(i);
}
template <typename F>
int launch_each(int64_t n, hipStream_t s, F f) {
  const int64_t blocks = (n + 255) / 256;
  if (n <= 0 || blocks > 0x7fffffff) return AF3_ERR_BAD_ARG;
  hipLaunchKernelGGL(each_kernel<F>, dim3((unsigned)blocks), dim3(256), 0, s, n, f);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

// eight channels: o = (((left + right + prev) + w_offset) + w_token_offset), + same * w_entity + w_chain, + bond * w_bond
template <typename T>
struct PairEmbed {
  PairEmbedArgs a;
  __device__ __forceinline__ void operator()(int64_t item) const {
    const int c = (int)(item & 15) * 8, n = a.n;
    const uint32_t pix = (uint32_t)(item >> 4);  // (n <= 8192)
    const int i = (int)(pix / (uint32_t)n), j = (int)(pix - (uint32_t)i * (uint32_t)n);
    auto clip = [](int64_t d, int r) { return (int)(d + r < 0 ? 0 : d + r > 2 * r ? 2 * r : d + r); };
    const int64_t *res = a.residue_index, *tok = a.token_index;
    const bool chain = a.asym_id[i] == a.asym_id[j], entity = a.entity_id[i] == a.entity_id[j];
    const int off = chain ? clip(res[i] - res[j], 32) : 65;
    const int toff = chain && res[i] == res[j] ? clip(tok[i] - tok[j], 32) : 65;
    const int coff = entity ? clip(a.sym_id[i] - a.sym_id[j], 2) : 5;
    float o[8], x[8];
    Elem<float>::load8(a.lr + (int64_t)i * a.ld_lr + c, o);
    Elem<float>::load8(a.lr + (int64_t)j * a.ld_lr + 128 + c, x);
    auto add = [&](float f = 1.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = o[e] + f * x[e];
    };
    add();
    Elem<float>::load8(a.prev + (int64_t)pix * 128 + c, x);
    add();
    Elem<float>::load8(a.w_pos + off * 128 + c, x);
    add();
    Elem<float>::load8(a.w_pos + (66 + toff) * 128 + c, x);
    add();
    Elem<float>::load8(a.w_pos + 132 * 128 + c, x);
    add(entity ? 1.f : 0.f);
    Elem<float>::load8(a.w_pos + (133 + coff) * 128 + c, x);
    add();
    Elem<float>::load8(a.w_bond + c, x);
    add(a.contact[pix]);
    Elem<T>::store8(reinterpret_cast<T*>(a.out) + (int64_t)pix * 128 + c, o);
  }
};

// contact[i][j] = 1 for every bond (i, j) whose two ends exist, but [0][0]
struct Contacts {
  const int64_t *idx[2];
  const uint8_t *ok[2];
  int count[2], n;
  float* contact;
  __device__ __forceinline__ void operator()(int64_t t) const {
    const int l = t < count[0] ? 0 : 1;
    const int64_t k = l ? t - count[0] : t;
    int64_t i = idx[l][2 * k], j = idx[l][2 * k + 1];
    if (!ok[l][2 * k] || !ok[l][2 * k + 1]) return;
    i += i < 0 ? n : 0;
    j += j < 0 ? n : 0;
    if (i < 0 || j < 0 || i >= n || j >= n || (i == 0 && j == 0)) return;
    contact[i * n + j] = 1.f;
  }
};

// out[r] = a[r] + b[r % mod], rows of `channels`
template <typename T>
struct AddRows {
  const float *a, *b;
  T* out;
  int64_t ld_b, mod;
  int chunks;
  __device__ __forceinline__ void operator()(int64_t item) const {
    const int64_t row = item / chunks;
    const int c = (int)(item - row * chunks) * 8;
    float x[8], y[8];
    Elem<float>::load8(a + item * 8, x);
    Elem<float>::load8(b + (row % mod) * ld_b + c, y);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = x[e] + y[e];
    Elem<T>::store8(out + item * 8, x);
  }
};

// x[r] *= bf16(mask[r % mod])
struct MaskRows {
  bf16_t* x;
  const float* mask;
  int64_t mod;
  int chunks;
  __device__ __forceinline__ void operator()(int64_t item) const {
    const float m = bf2f(f2bf(mask[item / chunks % mod]));
    float v[8];
    Elem<bf16_t>::load8(x + item * 8, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] * m;
    Elem<bf16_t>::store8(x + item * 8, v);
  }
};

// eight channels of an atom: ((((p0 w0 + p1 w1) + p2 w2) + mask w) + element) + asinh(charge) w, + four characters, * mask.  The weights
// as a linear layer holds them, [channel][input]: 200 KB that stay in L2.  9216 atoms: 11 us in place of 23 launches of 3 to 8.
struct AtomEmbed {
  AtomEmbedArgs a;
  __device__ __forceinline__ void operator()(int64_t item) const {
    const int chunks = a.channels / 8;
    const int64_t atom = item / chunks;
    const int c0 = (int)(item - atom * chunks) * 8;
    auto index = [](int64_t v, int size) { return v + (v < 0 ? size : 0); };
    const float m = a.mask[atom], charge = asinhf(a.charge[atom]), *const p = a.positions + atom * 3;
    const int64_t element = index(a.element[atom], 128);
    int64_t chars[4];
    bool ok = element >= 0 && element < 128;  // (else the atom is not a number)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      chars[j] = index(a.chars[atom * 4 + j], 64);
      ok = ok && chars[j] >= 0 && chars[j] < 64;
    }
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int c = c0 + e;
      float x = p[0] * a.w_pos[c * 3];
      x = x + p[1] * a.w_pos[c * 3 + 1];
      x = x + p[2] * a.w_pos[c * 3 + 2];
      x = x + m * a.w_mask[c];
      x = x + (ok ? a.w_element[c * 128 + element] : __builtin_nanf(""));
      x = x + charge * a.w_charge[c];
#pragma unroll
      for (int j = 0; j < 4; ++j) x = x + (ok ? a.w_chars[c * 256 + 64 * j + chars[j]] : 0.f);
      o[e] = x * m;
    }
    Elem<float>::store8(a.out + item * 8, o);
  }
};

// Atoms gathered into another layout, eight channels of a row: out = src * mask [+ add * add_mask], and what else an atom has.
// (One pass each for queries and keys in place of nine gathers of three or four launches.)
struct GatherAtoms {
  GatherAtomsArgs a;
  __device__ __forceinline__ void operator()(int64_t item) const {
    const int chunks = a.channels / 8;
    const int64_t row = item / chunks;
    const int c = (int)(item - row * chunks) * 8;
    const int64_t at = a.idx[row], add_at = a.add ? a.add_idx[row] : 0;
    const bool ok = at >= 0 && at < a.slots && add_at >= 0 && add_at < a.add_rows;  // (else the row is not a number, its uid 0)
    const float m = a.exists[row] ? 1.f : 0.f;
    float o[8], x[8];
    Elem<float>::load8(a.cond + (ok ? at : 0) * a.channels + c, o);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = ok ? o[e] * m : __builtin_nanf("");
    if (a.add) {
      const float am = a.add_exists[row] ? 1.f : 0.f;
      Elem<float>::load8(a.add + (ok ? add_at : 0) * a.channels + c, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float t = x[e] * am;
        o[e] = o[e] + t;
      }
    }
    Elem<float>::store8(a.out_cond + item * 8, o);
    if (c != 0) return;
    const int64_t from = ok ? at : 0;
    a.out_mask[row] = ok ? a.mask[from] * m : __builtin_nanf("");
#pragma unroll
    for (int e = 0; e < 3; ++e) a.out_pos[row * 3 + e] = ok ? a.pos[from * 3 + e] * m : __builtin_nanf("");
    a.out_uid[row] = ok && a.exists[row] && at < a.uids ? (int)a.uid[at] : 0;
  }
};

constexpr float SIGMA2 = 256.f, SIGMA = 16.f;  // of the data

// positions [samples][atoms][3] against mask [atoms]
struct ScalePositions {
  const float *pos, *mask, *level;
  float* out;
  int64_t atoms;
  __device__ __forceinline__ void operator()(int64_t i) const {
    const float t = *level, d = sqrtf(t * t + SIGMA2);
    out[i] = pos[i] * mask[i / 3 % atoms] / d;
  }
};
struct BlendPositions {
  const float *pos, *update, *mask, *level;
  float* out;
  int64_t atoms;
  __device__ __forceinline__ void operator()(int64_t i) const {
    const float t = *level, v = t * t + SIGMA2;
    const float skip = 1.f / v * SIGMA2, f = t * SIGMA / sqrtf(v);
    const float x = skip * pos[i], y = f * update[i];
    out[i] = (x + y) * mask[i / 3 % atoms];
  }
};
// (x + shift) * mask, then + noise (a scalar)
struct PlacePositions {
  const float *x, *shift, *mask, *noise;
  float* out;
  int64_t atoms;
  __device__ __forceinline__ void operator()(int64_t i) const {
    const float v = (x[i] + shift[i % 3]) * mask[i / 3 % atoms];
    out[i] = v + *noise;
  }
};
// noisy + step_scale * (next - level) * ((noisy - denoised) / level)
struct StepPositions {
  const float *noisy, *denoised, *level, *next;
  float step_scale;
  float* out;
  __device__ __forceinline__ void operator()(int64_t i) const {
    const float t = *level, g = (noisy[i] - denoised[i]) / t, f = step_scale * (*next - t);
    const float d = f * g;
    out[i] = noisy[i] + d;
  }
};

// A sampling step's start: a structure's masked centre of mass to the origin, x rot + shift, mask, + noise (a scalar).  A workgroup per
// sample, since all of its atoms make the centre; the first eight of a thread stay in registers between the two passes.  As a
// product, a sum over the atoms, a division, a difference, a product of matrices and the rest: seven launches, 33 us of a step; this: 5 x
// 2400 atoms 4.2 us, 5 x 18432 12.  Bound by its trips and the barrier between them.
constexpr int AUGMENT_THREADS = 1024, AUGMENT_KEPT = 8;
__global__ __launch_bounds__(AUGMENT_THREADS) void augment_positions_kernel(const float* x, const float* rot, const float* shift,
                                                                           const float* mask, const float* noise, float* out, int atoms) {
  __shared__ f32x4 sSum[AUGMENT_THREADS / 64];
  const int tid = threadIdx.x;
  x += (int64_t)blockIdx.x * atoms * 3;
  out += (int64_t)blockIdx.x * atoms * 3;
  float p[AUGMENT_KEPT][3], m[AUGMENT_KEPT], r[3][3], t[3];
#pragma unroll
  for (int k = 0; k < AUGMENT_KEPT; ++k) {
    const int a = min(tid + k * AUGMENT_THREADS, atoms - 1);
    m[k] = tid + k * AUGMENT_THREADS < atoms ? mask[a] : 0.f;
#pragma unroll
    for (int e = 0; e < 3; ++e) p[k][e] = x[(int64_t)a * 3 + e];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    t[i] = shift[i];
#pragma unroll
    for (int j = 0; j < 3; ++j) r[i][j] = rot[3 * i + j];
  }
  const float n = *noise;
  float sum[3] = {0.f, 0.f, 0.f}, count = 0.f;
#pragma unroll
  for (int k = 0; k < AUGMENT_KEPT; ++k) {
    if (tid + k * AUGMENT_THREADS >= atoms) continue;
    count += m[k];
#pragma unroll
    for (int e = 0; e < 3; ++e) sum[e] += m[k] * p[k][e];
  }
  for (int a = tid + AUGMENT_KEPT * AUGMENT_THREADS; a < atoms; a += AUGMENT_THREADS) {
    const float w = mask[a];
    count += w;
#pragma unroll
    for (int e = 0; e < 3; ++e) sum[e] += w * x[(int64_t)a * 3 + e];
  }
  const f32x4 mine = {wave_sum(sum[0]), wave_sum(sum[1]), wave_sum(sum[2]), wave_sum(count)};
  if ((tid & 63) == 0) sSum[tid >> 6] = mine;
  lds_barrier();
  f32x4 all = sSum[0];
#pragma unroll
  for (int w = 1; w < AUGMENT_THREADS / 64; ++w) all += sSum[w];
  const float c = fmaxf(all.w, 1e-6f), centre[3] = {all.x / c, all.y / c, all.z / c};
  auto place = [&](int a, const float* q, float w) {
    float d[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) d[e] = q[e] - centre[e];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const float v = (d[0] * r[0][j] + d[1] * r[1][j] + d[2] * r[2][j] + t[j]) * w;
      out[(int64_t)a * 3 + j] = v + n;
    }
  };
#pragma unroll
  for (int k = 0; k < AUGMENT_KEPT; ++k)
    if (tid + k * AUGMENT_THREADS < atoms) place(tid + k * AUGMENT_THREADS, p[k], m[k]);
  for (int a = tid + AUGMENT_KEPT * AUGMENT_THREADS; a < atoms; a += AUGMENT_THREADS) {
    const float q[3] = {x[(int64_t)a * 3], x[(int64_t)a * 3 + 1], x[(int64_t)a * 3 + 2]};
    place(a, q, mask[a]);
  }
}

// The windows of an atom layout that somebody reads, in their order.  A layout has room for every token's 24 atoms and as many empty
// slots behind the last atom as there are fewer, half of the windows and more.  Asked for are a window with an atom in it (mask) and
// one that the way back reads; and all of them should any key be a row that neither of these names, whose value would then count.
// One workgroup, the rows as bits in LDS, eight loads of a thread on their way at a time: 9216 rows and 36864 keys 17 us (one load
// at a time 32), twice as many 27 (60), once a batch.
constexpr int BATCH = 8, WINDOW_THREADS = 1024, WINDOW_ROWS = 1 << 19;
__global__ __launch_bounds__(WINDOW_THREADS) void atom_windows_kernel(AtomWindowsArgs a) {
  __shared__ uint32_t want[WINDOW_ROWS / 32];
  __shared__ int stray, live_of[WINDOW_THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rows = a.windows * a.queries;
  if (tid == 0) stray = 0;
  for (int r0 = 0; r0 < rows; r0 += BATCH * WINDOW_THREADS) {
    float m[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) m[k] = a.mask[min(r0 + k * WINDOW_THREADS + tid, rows - 1)];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int r = r0 + k * WINDOW_THREADS + tid;
      const uint64_t b = __ballot(r < rows && m[k] != 0.f);
      if ((lane & 31) == 0 && r < rows) want[r >> 5] = (uint32_t)(lane ? b >> 32 : b);
    }
  }
  __syncthreads();
  for (int64_t i0 = 0; i0 < a.slots; i0 += BATCH * WINDOW_THREADS) {
    int64_t r[BATCH];
    bool there[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int64_t i = min(i0 + k * WINDOW_THREADS + tid, a.slots - 1);
      r[k] = a.back_idx[i];
      there[k] = a.back_exists[i];
    }
#pragma unroll
    for (int k = 0; k < BATCH; ++k)  // (the last one again does no harm)
      if (there[k] && r[k] >= 0 && r[k] < rows) atomicOr(&want[r[k] >> 5], 1u << (r[k] & 31));
  }
  __syncthreads();
  const int64_t keys = (int64_t)a.windows * a.keys;
  for (int64_t i0 = 0; i0 < keys; i0 += BATCH * WINDOW_THREADS) {
    int r[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) r[k] = a.key_rows[min(i0 + k * WINDOW_THREADS + tid, keys - 1)];
#pragma unroll
    for (int k = 0; k < BATCH; ++k)
      if (r[k] >= 0 && r[k] < rows && !(want[r[k] >> 5] >> (r[k] & 31) & 1)) stray = 1;
  }
  __syncthreads();
  int before = 0;
  for (int w0 = 0; w0 < a.windows; w0 += WINDOW_THREADS) {
    const int w = w0 + tid;
    bool live = w < a.windows && stray;
    if (w < a.windows)
      for (int r = w * a.queries; r < (w + 1) * a.queries && !live; ++r) live = want[r >> 5] >> (r & 31) & 1;
    const uint64_t b = __ballot(live);
    if (lane == 0) live_of[wave] = __popcll(b);
    __syncthreads();
    int at = before;
    for (int v = 0; v < WINDOW_THREADS / 64; ++v) {
      if (v < wave) at += live_of[v];
      before += live_of[v];
    }
    if (live) a.out[1 + at + __popcll(b & ((1ull << lane) - 1))] = w;
    __syncthreads();
  }
  if (tid == 0) a.out[0] = before;
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

int launch_pair_embed(const PairEmbedArgs& a, hipStream_t s) {
  if (a.n <= 0 || a.n > 8192 || !a.lr || !a.prev || !a.w_pos || !a.w_bond || !a.contact || !a.out || (a.ld_lr & 3) || a.ld_lr < 256)
    return AF3_ERR_BAD_ARG;
  if (!a.asym_id || !a.residue_index || !a.token_index || !a.entity_id || !a.sym_id) return AF3_ERR_BAD_ARG;
  if (!al16(a.lr) || !al16(a.prev) || !al16(a.w_pos) || !al16(a.w_bond) || !al16(a.out)) return AF3_ERR_BAD_ARG;
  const int64_t items = (int64_t)a.n * a.n * 16;
  return a.out_f32 ? launch_each(items, s, PairEmbed<float>{a}) : launch_each(items, s, PairEmbed<bf16_t>{a});
}

int launch_contacts(const int64_t* idx0, const uint8_t* ok0, int n0, const int64_t* idx1, const uint8_t* ok1, int n1, float* contact,
                    int n, hipStream_t s) {
  if (n <= 0 || n0 < 0 || n1 < 0 || !contact || (n0 && (!idx0 || !ok0)) || (n1 && (!idx1 || !ok1))) return AF3_ERR_BAD_ARG;
  if (n0 + n1 == 0) return AF3_OK;
  return launch_each(n0 + n1, s, Contacts{{idx0, idx1}, {ok0, ok1}, {n0, n1}, n, contact});
}

int launch_add_rows(const float* a, const float* b, int64_t ld_b, int64_t mod, void* out, int out_f32, int64_t rows, int channels,
                    hipStream_t s) {
  if (!a || !b || !out || rows <= 0 || mod <= 0 || channels <= 0 || (channels & 7) || (ld_b & 3) || ld_b < channels || !al16(a) ||
      !al16(b) || !al16(out))
    return AF3_ERR_BAD_ARG;
  const int chunks = channels / 8;
  return out_f32 ? launch_each(rows * chunks, s, AddRows<float>{a, b, static_cast<float*>(out), ld_b, mod, chunks})
                 : launch_each(rows * chunks, s, AddRows<bf16_t>{a, b, static_cast<bf16_t*>(out), ld_b, mod, chunks});
}

int launch_mask_rows(bf16_t* x, const float* mask, int64_t mod, int64_t rows, int channels, hipStream_t s) {
  if (!x || !mask || rows <= 0 || mod <= 0 || channels <= 0 || (channels & 7) || !al16(x)) return AF3_ERR_BAD_ARG;
  return launch_each(rows * (channels / 8), s, MaskRows{x, mask, mod, channels / 8});
}

int launch_atom_embed(const AtomEmbedArgs& a, hipStream_t s) {
  if (!a.positions || !a.mask || !a.element || !a.charge || !a.chars || !a.w_pos || !a.w_mask || !a.w_element || !a.w_charge ||
      !a.w_chars || !a.out || a.atoms <= 0 || a.channels <= 0 || (a.channels & 7) || !al16(a.out))
    return AF3_ERR_BAD_ARG;
  return launch_each(a.atoms * (a.channels / 8), s, AtomEmbed{a});
}

int launch_gather_atoms(const GatherAtomsArgs& a, hipStream_t s) {
  if (!a.idx || !a.exists || !a.cond || !a.mask || !a.pos || !a.uid || !a.out_cond || !a.out_mask || !a.out_pos || !a.out_uid ||
      a.rows <= 0 || a.slots <= 0 || a.uids <= 0 || a.channels <= 0 || (a.channels & 7) || !al16(a.cond) || !al16(a.out_cond))
    return AF3_ERR_BAD_ARG;
  if (a.add && (!a.add_idx || !a.add_exists || a.add_rows <= 0 || !al16(a.add))) return AF3_ERR_BAD_ARG;
  GatherAtomsArgs args = a;
  if (!a.add) args.add_rows = 1;
  return launch_each(a.rows * (a.channels / 8), s, GatherAtoms{args});
}

bool atom_windows_apply(const AtomWindowsArgs& a) {
  return a.mask && a.back_idx && a.back_exists && a.slots > 0 && a.key_rows && a.out && a.windows > 0 && a.queries > 0 && a.keys > 0 &&
         (int64_t)a.windows * a.queries <= WINDOW_ROWS;
}

int launch_atom_windows(const AtomWindowsArgs& a, hipStream_t s) {
  if (!atom_windows_apply(a)) return AF3_ERR_BAD_ARG;
  hipLaunchKernelGGL(atom_windows_kernel, dim3(1), dim3(WINDOW_THREADS), 0, s, a);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

int launch_augment_positions(const float* x, const float* rot, const float* shift, const float* mask, const float* noise, float* out,
                             int64_t samples, int64_t atoms, hipStream_t s) {
  if (!x || !rot || !shift || !mask || !noise || !out || x == out || samples <= 0 || samples > 0x7fffffff || atoms <= 0 || atoms > 0x3fffffff)
    return AF3_ERR_BAD_ARG;
  hipLaunchKernelGGL(augment_positions_kernel, dim3((unsigned)samples), dim3(AUGMENT_THREADS), 0, s, x, rot, shift, mask, noise, out, (int)atoms);
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

int launch_positions(int op, const float* x, const float* y, const float* mask, const float* level, const float* other, float f,
                     float* out, int64_t samples, int64_t atoms, hipStream_t s) {
  if (!x || !out || !level || samples <= 0 || atoms <= 0 || (op != POS_STEP && !mask) || (op != POS_SCALE && !y)) return AF3_ERR_BAD_ARG;
  const int64_t n = samples * atoms * 3;
  switch (op) {
    case POS_SCALE: return launch_each(n, s, ScalePositions{x, mask, level, out, atoms});
    case POS_BLEND: return launch_each(n, s, BlendPositions{x, y, mask, level, out, atoms});
    case POS_PLACE: return launch_each(n, s, PlacePositions{x, y, mask, level, out, atoms});
    case POS_STEP: return other ? launch_each(n, s, StepPositions{x, y, level, other, f, out}) : AF3_ERR_BAD_ARG;
  }
  return AF3_ERR_BAD_ARG;
}
