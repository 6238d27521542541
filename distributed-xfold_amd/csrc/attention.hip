// Flash-style pair-biased attention on bf16 MFMA; the [B, H, Sq, Sk] logits
// never reach HBM.
//
// One wave owns 32 queries of one (batch, head).  Logits are computed
// TRANSPOSED, S^T = K Q^T, so that in the MFMA accumulator layout a lane owns
// one query (column) and 16 of the 32 keys of a tile (rows): the online-softmax
// row maximum / row sum are then in-register reductions plus one exchange
// between the two lane halves.  The same registers, rounded to bf16, are
// directly the B fragments of O^T += V^T P^T (the MFMA k index is a summation
// index, so the key order inside a fragment is free as long as the V^T
// fragment uses the same order).  K and V tiles of 64 keys are staged in LDS row
// by row as they lie in memory, double-buffered and shared by the workgroup's
// waves; the V^T fragments come out of the transposing LDS read of this target
// (ds_read_b64_tr_b16), so nothing is transposed on the way in.
//
// Logit = q.k (q pre-scaled) + pair_bias[h][q][k]; then
//   key_mask:  keys with mask 0 are REPLACED by -1e9 (so a fully masked row is
//              uniform over all Sk keys, like the reference's masked_fill);
//   qpad/kpad: +1e9 where both the query and the key are padding (the atom
//              cross-attention convention).
// Keys beyond Sk (tile padding) get -inf and never contribute.
#include "common.h"
#include "kernels.h"

namespace {

constexpr int KT = 64;        // keys per LDS tile
constexpr float NEG_INF = -__builtin_huge_valf();
constexpr int RSRC_RAW = 0x00020000;  // last word of a raw (unstructured, range-checked) buffer descriptor
typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));
// ds_read_b64_tr_b16: four 16-bit elements per lane, transposed within each group of 16 lanes
__device__ __forceinline__ v4s lds_read_tr16(const bf16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)p);
}
constexpr float LOG2E = 1.4426950408889634f;
// per-key code staged in LDS next to the K tile
constexpr int KEY_MASKED = 1, KEY_PAD = 2, KEY_BEYOND = 4;

// maximum of the lane's 32 logits as a tree of three-input maxima
__device__ __forceinline__ float max3_of_32(const f32x16 (&s)[2]) {
  float t3[11];
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    const int e = 3 * i;
    t3[i] = fmaxf(fmaxf(s[e >> 4][e & 15], s[(e + 1) >> 4][(e + 1) & 15]), s[(e + 2) >> 4][(e + 2) & 15]);
  }
  t3[10] = fmaxf(s[1][14], s[1][15]);
  const float t9a = fmaxf(fmaxf(t3[0], t3[1]), t3[2]), t9b = fmaxf(fmaxf(t3[3], t3[4]), t3[5]);
  const float t9c = fmaxf(fmaxf(t3[6], t3[7]), t3[8]), t9d = fmaxf(t3[9], t3[10]);
  return fmaxf(fmaxf(fmaxf(t9a, t9b), t9c), t9d);
}

// FAST: keys are rows of K / V as they stand (no row table) and the pair bias is present and 16-byte
// addressable.  Then every address of the key-tile loop is a wave-uniform base that advances by a
// constant per tile plus a per-lane offset that never changes, and the bias quads are loaded straight
// into the registers in which the matrix unit accumulates K Q^T on top of them: no address arithmetic
// and no bias additions in the loop.  The last tile of a key count that is not a multiple of 64 takes
// the clamped addresses of the general form.
template <int KSTEPS, int DVT, int NW, bool FAST>
// at least two waves per SIMD: the register allocator then keeps everything in
// the 256 architectural VGPRs instead of parking loop state in accumulation
// registers, which would leave a single wave per SIMD (the one-wave workgroup of
// head dimension 48 stages twelve chunks per thread and is given the whole register file)
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(KSTEPS == 3 && NW == 1 ? 1 : 2)))
void flash_kernel(FlashArgs a) {
  args_at_once<FlashArgs>();
  constexpr int KD = KSTEPS * 16;  // padded q/k head dim
  constexpr bool SUM_COLUMN = KSTEPS == 3;  // (heads of 48: KD is the head's, so that the columns behind it are free)
  constexpr int LDK = KD + 8;      // sK row stride (bf16)
  constexpr int NT = NW * 64;
  __shared__ __attribute__((aligned(16))) bf16_t sK[2][KT * LDK];
  // sV row stride (bf16): V rows as they are, padded to the 32 DVT columns the products read.  A transposing
  // read touches 8 rows x 64 bytes; with a row stride of 16 or 48 dwords modulo the 64 banks (32 or 96
  // elements) these tile the banks exactly twice, the minimum for its 512 bytes.
  constexpr int LDV = DVT == 1 ? 32 : 96;
  static_assert(LDV >= DVT * 32, "a row holds every column the products read");
  __shared__ __attribute__((aligned(16))) bf16_t sV[2][KT * LDV];
  __shared__ __attribute__((aligned(16))) int sCode[2][KT];
  __shared__ int sAnyCode[2];  // whether any key of the staged tile carries a code

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int hh = lane >> 5, j = lane & 31;
  const int xaddr = half_swap_addr();
  // Batch entries that share a slab of a non-batched pair bias must meet in one L2 for that slab to be
  // fetched from memory once, and so must the query tiles that share a head's K and V: workgroup ids are dealt
  // round-robin to the 8 XCDs, each with an L2 of its own, so id -> (xcd, slot) -> logical id gives every XCD a
  // contiguous range of logical ids, and logical = (head * query tiles + query tile) * B + batch gives it a few
  // heads, with the entries that share a slab side by side (16 heads x 48, 5 samples of 768: 36.2 -> 35.2 us
  // against query tiles as the slowest index).
  int b, h, q0;
  if (a.bias_mod > 0) {
    // (windows of a few keys: the workgroups are short and the bias slabs small; plain order)
    if ((int)blockIdx.x >= a.n_blocks) return;
    b = blockIdx.x % a.B;
    h = (blockIdx.x / a.B) % a.H;
    q0 = (blockIdx.x / (a.B * a.H)) * (NW * 32) + wave * 32;
  } else {
    const int per_xcd = (gridDim.x + 7) >> 3;
    const int logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (logical >= a.n_blocks) return;  // workgroup-uniform, before any barrier
    const int tiles = (a.Sq + NW * 32 - 1) / (NW * 32), rest = logical / a.B;
    b = logical % a.B;
    h = rest / tiles;
    q0 = rest % tiles * (NW * 32) + wave * 32;
  }
  const int d = a.d;
  const int qi = min(q0 + j, a.Sq - 1);  // clamped for loads; stores are guarded
  const bool q_ok = q0 + j < a.Sq;

  // Q^T fragments: lane (query j, half hh) holds head-dim 16*ks + 8*hh .. +7
  bf16x8 qf[KSTEPS];
  {
    const bf16_t* qp = a.q + (int64_t)b * a.q_sb + (int64_t)qi * a.q_ss + h * d;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const int c = 16 * ks + 8 * hh;
      const u32x4 z = {0, 0, 0, 0};
      const u32x4 v = *reinterpret_cast<const u32x4*>(qp + (c < d ? c : 0));
      qf[ks] = as_frag(c < d ? v : z);
    }
  }
  const bf16x8 onesf = as_frag(u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});

  // With key_rows, K / V are tables of rows shared by bias_mod consecutive batch
  // entries (one table per sample) and the key rows of this batch entry are
  // looked up in key_rows; a negative entry is a key whose K and V rows are zero.
  const int64_t kv_b = a.key_rows ? b / a.bias_mod : b;
  const bf16_t* kg = a.k + kv_b * a.k_sb + h * d;
  const bf16_t* vg = a.v + kv_b * a.v_sb + h * d;
  const int dch = d / 8;  // 16-byte chunks per real key row

  // Tile loaders (global -> registers -> LDS).  Every load is unconditional,
  // from a clamped address, and nothing is decided from a loaded value before
  // the LDS store one tile later: a load under a lane mask, or a value
  // inspected right after its load, costs a full memory round trip per tile.
  //   chunk id = key * (KD/8) + c, c fastest (one key row is contiguous), for K and for V alike: both go to
  //   LDS row by row as they lie in memory
  // The K chunks of a tile and then its V chunks form one list of 2 KCH entries that the threads share out
  // evenly: thread t moves entries t, t + NT, ..  (head dimension 48 with 256 threads: three each, the
  // middle one a K chunk for waves 0 and 1 and a V chunk for waves 2 and 3; whether an entry is K or V is
  // uniform over a wave because KCH is a multiple of 64).
  constexpr int KCH = KT * (KD / 8);
  static_assert((2 * KCH) % NT == 0, "the chunk list divides evenly");
  constexpr int NL = 2 * KCH / NT;
  u32x4 rc[NL];
  bool row_ok[NL];
  float rkm = 1.f, rkp = 1.f;  // key mask / key padding flag of key tid (threads 0..63)
  const int bb = a.bias_mod > 0 ? b % a.bias_mod : b;  // batch index of bias / padding masks
  const int* krows = a.key_rows ? a.key_rows + (int64_t)bb * a.Sk : nullptr;
  const float* kmask = a.key_mask ? a.key_mask + (int64_t)b * a.km_sb : nullptr;
  const float* kpad = a.kpad ? a.kpad + (int64_t)bb * a.kp_sb : nullptr;
  int k0_loaded = 0;
  // entry i of this thread: chunk e (K) or e - KCH (V) of its tile, key = chunk / (KD/8), c = chunk % (KD/8)
  bool is_v[NL];
  int ch_key[NL], ch_c[NL];
  // FAST: byte offset of the chunk from the first key row of a tile (the launcher has checked that 64 rows
  // of K or V span less than 2 GB)
  uint32_t choff[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = tid + i * NT;
    is_v[i] = e >= KCH;
    const int ch = is_v[i] ? e - KCH : e;
    ch_key[i] = ch / (KD / 8);
    ch_c[i] = ch % (KD / 8);
    choff[i] = (uint32_t)(ch_key[i] * (is_v[i] ? a.v_ss : a.k_ss) + (ch_c[i] < dch ? ch_c[i] : 0) * 8) * 2u;
  }
  // Rows of the chunks this thread moves.  With key_rows they are looked
  // up one tile before the chunks themselves are requested, so that a tile
  // costs one memory round trip, not two in a row.
  int row_i[NL];
  auto gidx = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int key = min(k0 + ch_key[i], a.Sk - 1);
      row_i[i] = krows ? krows[key] : key;
    }
  };
  auto gload = [&](int k0) {
    k0_loaded = k0;
    if (FAST && k0 + KT <= a.Sk) {  // (workgroup-uniform)
      const char* kb = reinterpret_cast<const char*>(kg + (int64_t)k0 * a.k_ss);
      const char* vb = reinterpret_cast<const char*>(vg + (int64_t)k0 * a.v_ss);
#pragma unroll
      for (int i = 0; i < NL; ++i) rc[i] = *reinterpret_cast<const u32x4*>((is_v[i] ? vb : kb) + choff[i]);
    } else {
      if constexpr (FAST) gidx(k0);
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int row = row_i[i];
        row_ok[i] = row >= 0;
        rc[i] = *reinterpret_cast<const u32x4*>((is_v[i] ? vg : kg) + (int64_t)max(row, 0) * (is_v[i] ? a.v_ss : a.k_ss) +
                                                (ch_c[i] < dch ? ch_c[i] : 0) * 8);
      }
    }
    if (tid < KT) {
      const int key = min(k0 + tid, a.Sk - 1);
      if (kmask) rkm = kmask[key];
      if (kpad) rkp = kpad[key];
    }
  };
  auto sstore = [&](int buf) {
    const u32x4 z = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int key = ch_key[i], c = ch_c[i];
      const bool ok = k0_loaded + key < a.Sk && c < dch && (FAST || row_ok[i]);  // (FAST: rows are never negative)
      const u32x4 vv = ok ? rc[i] : z;
      if (!is_v[i]) *reinterpret_cast<u32x4*>(&sK[buf][key * LDK + c * 8]) = vv;
      else *reinterpret_cast<u32x4*>(&sV[buf][key * LDV + c * 8]) = vv;
    }
    if (tid < KT) {  // wave 0, all of it (KT = 64)
      const int code = (k0_loaded + tid >= a.Sk ? KEY_BEYOND : 0) | (rkm == 0.f ? KEY_MASKED : 0) | (rkp == 0.f ? KEY_PAD : 0);
      sCode[buf][tid] = code;
      const bool any = __any(code != 0);
      if (tid == 0) sAnyCode[buf] = any ? 1 : 0;
    }
  };
  // V columns that no chunk covers (head dimension padding: columns KD .. 32 DVT - 1 of either buffer) must
  // read as zero; with heads of 48 the first of them as ones, and the row sum comes out of the products with V
  if constexpr (KD < DVT * 32) {
    constexpr int PAD = DVT * 32 - KD;  // a multiple of 16
    for (int idx = tid; idx < 2 * KT * (PAD / 2); idx += NT) {
      const int row = idx / (PAD / 2), w = idx % (PAD / 2);
      reinterpret_cast<uint32_t*>(&sV[row / KT][(row % KT) * LDV + KD])[w] = SUM_COLUMN && w == 0 ? 0x3F80u : 0u;
    }
  }  // (no tile store touches these columns; the barrier after the first tile's stores orders them too)

  f32x16 o[DVT];
#pragma unroll
  for (int t = 0; t < DVT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;
  float m_run = NEG_INF, l_run = 0.f;  // softmax base (a maximum seen so far) in natural units, and row sum

  // Pair bias (fp32, one row per query): the 8 quads of a 64-key tile are
  // fetched one tile ahead, unconditionally, from addresses clamped into the
  // row (a clamped quad belongs to keys >= Sk, which are masked anyway).
  const float* bias_plane = a.bias ? a.bias + (int64_t)bb * a.bias_sb + (int64_t)h * a.bias_sh : nullptr;  // (uniform)
  const float* bias_row = a.bias ? bias_plane + (int64_t)qi * a.bias_sq : nullptr;
  const bool q_is_pad = a.qpad ? (a.qpad[(int64_t)bb * a.qp_sb + qi] == 0.f) : false;
  const bool bias_vec = FAST || (a.bias && a.Sk >= 4 && ((a.bias_sq & 3) == 0) && ((a.bias_sb & 3) == 0) &&
                                 ((a.bias_sh & 3) == 0) && ((a.bias_squad & 3) == 0) && (((uintptr_t)a.bias & 15) == 0));
  // key k of the row: at k (row-major) or, with quads of four keys as the outer
  // index, at (k / 4) * bias_squad + k % 4
  const int64_t quad_step = a.bias_squad ? a.bias_squad : 4;
  const int last_quad = (a.Sk - 1) & ~3;
  // FAST: this lane's byte offset from the tile's first quad of the bias plane (checked by the launcher to fit)
  const uint32_t bias_lane = (uint32_t)((int64_t)qi * a.bias_sq + hh * quad_step) * 4u;
  // the quads of tile k0 into `dst`, laid out like the score accumulators:
  // dst[u][4g + e] = bias(query, key k0 + 32u + 8g + 4hh + e)
  // `part` < 0: all eight quads; 0..3: the two quads (u = part / 2, g = 2 (part % 2) + {0, 1}) only
  auto gload_bias = [&](f32x16 (&dst)[2], int k0, int part = -1) {
    if (!bias_vec) return;  // workgroup-uniform
    const bool fast_addr = FAST && k0 + KT <= a.Sk;
    const char* bt = reinterpret_cast<const char*>(bias_plane + (int64_t)(k0 >> 2) * quad_step);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (part >= 0 && (u != (part >> 1) || (g >> 1) != (part & 1))) continue;
        f32x4 v;
        if (fast_addr) v = *reinterpret_cast<const f32x4*>(bt + (int64_t)(8 * u + 2 * g) * quad_step * 4 + bias_lane);
        else v = *reinterpret_cast<const f32x4*>(bias_row + (int64_t)(min(k0 + u * 32 + 8 * g + 4 * hh, last_quad) >> 2) * quad_step);
        dst[u][4 * g] = v.x; dst[u][4 * g + 1] = v.y; dst[u][4 * g + 2] = v.z; dst[u][4 * g + 3] = v.w;
      }
  };

  const int nkt = (a.Sk + KT - 1) / KT;
  // Two register sets of 2 x 16 values.  FAST: they alternate between the tiles, the set of tile kt + 1
  // receives that tile's bias while tile kt is worked on and is then accumulated on by the matrix unit.
  // Otherwise one set holds the scores and the other the prefetched bias, copied over before the products.
  f32x16 setA[2], setB[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int r = 0; r < 16; ++r) setA[u][r] = setB[u][r] = 0.f;
  if constexpr (!FAST) gidx(0);
  gload(0);
  if constexpr (!FAST) gidx(KT);
  gload_bias(FAST ? setA : setB, 0);
  // the output gate of the lane's query: asked for now, used after the last tile
  u32x2 gate_w[DVT][4];
#pragma unroll
  for (int t = 0; t < DVT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * t + 8 * g + 4 * hh;
      gate_w[t][g] = u32x2{0x3F803F80u, 0x3F803F80u};
      if (a.g) gate_w[t][g] = *reinterpret_cast<const u32x2*>(a.g + (int64_t)b * a.g_sb + (int64_t)qi * a.g_ss + h * d + (dd < d ? dd : 0));
    }
  sstore(0);
  lds_barrier();

  // One key tile.  FAST: `s` holds the tile's bias, `other` takes the next tile's.  Otherwise `other`
  // holds this tile's bias, is copied to `s`, and then takes the next tile's.
  auto tile = [&](int kt, f32x16 (&s)[2], f32x16 (&other)[2]) {
    const int buf = kt & 1;
    const int k0 = kt * KT;
    // next tile's K / V chunks (their rows are known) and the rows of the one after
    gload((kt + 1) * KT);
    if constexpr (!FAST) gidx((kt + 2) * KT);
    // FAST: the next tile's bias is requested in four pieces spread over this tile (below).  A wave that
    // issues a burst of loads sits at them until the CU's address unit, which takes 16 to 64 cycles per wave
    // instruction and serves eight waves, has accepted them all; spread out, the unit works through them
    // while the wave computes.
    auto bias_piece = [&](int part) {
      if constexpr (FAST) {
        __builtin_amdgcn_sched_barrier(0);
        gload_bias(other, (kt + 1) * KT, part);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // both 32-key halves through the matrix unit first (two independent chains);
    // s[u][4g + e] = logit(query j, key k0 + 32u + 8g + 4hh + e)
    // (either form starts the accumulation from the bias, so both give the same bits)
    if constexpr (!FAST) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float bv = 0.f;
            if (bias_vec) bv = other[u][4 * g + e];
            else if (bias_row) {
              const int kc = min(k0 + u * 32 + 8 * g + 4 * hh + e, a.Sk - 1);
              bv = bias_row[(int64_t)(kc >> 2) * quad_step + (kc & 3)];
            }
            s[u][4 * g + e] = bv;
          }
      gload_bias(other, (kt + 1) * KT);  // the next tile's bias into the registers just read
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
        s[u] = mfma32(lds_frag(sK[buf], LDK, u * 32, ks * 16, lane), qf[ks], s[u]);
    bias_piece(0);
    // Masks from the per-key codes; most tiles carry none (a workgroup-uniform
    // test skips the block).  The logits stay in natural units: the maximum
    // does not care, and exp2 takes fma(s, log2 e, -m log2 e).  (For a row
    // whose keys are all masked every s equals m = -1e9 and the fma leaves the
    // rounding error of m log2 e, at most 2^6 in magnitude and the same for
    // every key: the weights stay uniform.)
    if (__builtin_amdgcn_readfirstlane(sAnyCode[buf])) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int* cp = &sCode[buf][u * 32 + 8 * g + 4 * hh];
          const int code[4] = {cp[0], cp[1], cp[2], cp[3]};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = s[u][4 * g + e];
            if (code[e] & KEY_MASKED) v = -1e9f;
            if (q_is_pad && (code[e] & KEY_PAD)) v += 1e9f;
            if (code[e] & KEY_BEYOND) v = NEG_INF;
            s[u][4 * g + e] = v;
          }
        }
    }
    float mx = max3_of_32(s);
    mx = fmaxf(mx, half_swap(xaddr, mx));
    bias_piece(1);
    // The base of the exponentials follows the maximum lazily: it moves only when a tile's maximum
    // exceeds it by more than BASE_SLACK (weights then reach e^BASE_SLACK at most, far inside fp32 and
    // bf16 range; the normalisation at the end takes the common factor out again), so that most tiles
    // leave the output accumulators alone.  The first tile moves it from -inf to its maximum.
    constexpr float BASE_SLACK = 8.f;
    const float m_new = mx - m_run > BASE_SLACK ? mx : m_run;
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);  // 0 on the first tile (m_run = -inf, m_new finite)
    m_run = m_new;
    const float m2 = m_new * LOG2E;
    bf16x8 pf[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        float pv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][8 * half + e], LOG2E, -m2));
        pf[u][half] = as_frag(pack8(pv));
        if (half == 1) bias_piece(2 + u);
      }
    // row sums of the ROUNDED probabilities on the matrix unit (ones * P), so
    // that the weights that multiply V sum to exactly one after normalisation;
    // SUM_COLUMN: a column of ones beside V's, in the products below
    if constexpr (!SUM_COLUMN) {
      f32x16 lsum;
#pragma unroll
      for (int r = 0; r < 16; ++r) lsum[r] = 0.f;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int half = 0; half < 2; ++half) lsum = mfma32(onesf, pf[u][half], lsum);
      l_run = l_run * alpha + lsum[0];
    }
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int t = 0; t < DVT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
    }
    // O^T[dd][query] += sum_key V^T[dd][key] P^T[key][query]; fragment element e
    // of lane-half hh in k-step `half` is key 32u + 16*half + 8*(e>>2) + 4*hh + (e&3).  V lies in LDS as it
    // lies in memory, [key][dd]; the transposing LDS read hands each lane of a group of 16 one column of a
    // 4-row x 16-column block (lane i of the group points at row i / 4, columns 4 (i % 4) .. of the block
    // and receives column i of its four rows): rows = four consecutive keys, columns = the group's 16 dd.
    {
      const int i16 = lane & 15;
      const bf16_t* vbase = &sV[buf][(4 * hh + (i16 >> 2)) * LDV + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3)];
#pragma unroll
      for (int t = 0; t < DVT; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            const bf16_t* vp = vbase + (u * 32 + 16 * half) * LDV + t * 32;
            const v4s lo = lds_read_tr16(vp), hi = lds_read_tr16(vp + 8 * LDV);
            o[t] = mfma32(as_frag(__builtin_bit_cast(u32x4, v8s{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w})),
                          pf[u][half], o[t]);
          }
    }
    if (kt + 1 < nkt) sstore(buf ^ 1);
    lds_barrier();
  };
  if constexpr (FAST) {
    for (int kt = 0; kt < nkt; kt += 2) {
      tile(kt, setA, setB);
      if (kt + 1 < nkt) tile(kt + 1, setB, setA);
    }
  } else {
    for (int kt = 0; kt < nkt; ++kt) tile(kt, setA, setB);
  }

  if constexpr (SUM_COLUMN) {  // row 48 of o, register 8 of the second block's lower half
    const auto sum = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[DVT - 1][8]), __float_as_uint(o[DVT - 1][8]), false, false);
    l_run = __uint_as_float(sum[0]);
  }
  const float inv = 1.f / l_run;  // the ones * P sums cover both half-waves' keys
  if (!q_ok) return;
  // o[t][4g + e] = out(query j, head-dim 32t + 8g + 4hh + e)
#pragma unroll
  for (int t = 0; t < DVT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int dd = 32 * t + 8 * g + 4 * hh;
      if (dd >= d) continue;  // d % 4 == 0, so a quad is all in or all out
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = o[t][4 * g + e] * inv;
      {
        const u32x2 gw = gate_w[t][g];   // ones without a gate
        v[0] *= bflo(gw.x); v[1] *= bfhi(gw.x); v[2] *= bflo(gw.y); v[3] *= bfhi(gw.y);
      }
      const int64_t off = (int64_t)b * a.o_sb + (int64_t)qi * a.o_ss + h * d + dd;
      if (a.out_f32) {
        f32x4 w = {v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + off) = w;
      } else {
        u32x2 w;
        w.x = pack2bf(v[0], v[1]);
        w.y = pack2bf(v[2], v[3]);
        *reinterpret_cast<u32x2*>(reinterpret_cast<bf16_t*>(a.out) + off) = w;
      }
    }
}

// ------------------------------------------------------------------ heads of 48 over plain keys
// The token transformer's attention: 16 heads of 48, an fp32 pair bias, keys as they stand.  At 100 to 768 tokens a SIMD has one
// or two of its waves, each a chain of key tiles, so what counts is the length of the chain: the arithmetic is flash_kernel's,
// in its order (the same bits), with less around it.  K, V and the bias come through range-checked loads (what lies past the
// last key reads as zeros or as whatever the plane holds; its logits become -inf), so a tile that is not full costs nothing
// more; a masked key's logit is replaced by what stands beside it in LDS (two instructions a logit instead of nine); a tile's
// bias is asked for two tiles ahead, into the accumulators as the exponentials empty them, its K and V one tile ahead.
// Of 8.8 us at 100 tokens flash_kernel spent 2.2 before its first tile, 4.4 in two tiles and 1.4 behind them; us, flash_kernel /
// this, 16 heads: 5 x 40 tokens 7.7 / 5.3, 5 x 256 12.0 / 9.4, 1 x 768 25.1 / 20.9, 5 x 1536 106 / 94.
// The row sum is a 49th column of V, of ones, in the product with V (four products a tile and their wait less), and a quarter's
// products stand beside the next quarter's exponentials.  us, the sum by products of its own and all of V's behind the last
// exponential / this: 5 x 40 5.1 / 4.9, 5 x 200 9.9 / 9.4, 1 x 384 11.8 / 11.1, 5 x 384 13.0 / 12.1, 3 x 512 14.8 / 13.8,
// 1 x 768 21.4 / 21.9, 5 x 768 32.6 / 32.3, 5 x 1536 103.7 / 101.2.  What is left of a tile's 2800 cycles at 768 tokens: 330 K
// products, 470 maximum, 980 exponentials and V, 310 (5 samples) to 640 (one) waiting for the bias, which comes from HBM, 510 the next tile's way
// into LDS, 410 barrier.  No faster: a third set of bias registers (over 256, spills), the bias touched three to six tiles
// ahead, the LDS stores in the middle of the tile (5 x 768 and up slower), the keys of a query shared out between two waves
// of 128 registers (from 128 tokens on the same).
constexpr int TOK_D = 48, TOK_LDK = 56, TOK_LDV = 96;
constexpr int TOK_K_BYTES = KT * TOK_LDK * 2, TOK_TILE = TOK_K_BYTES + KT * TOK_LDV * 2;
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void token_attention_kernel(FlashArgs a) {
  args_at_once<FlashArgs>();
  constexpr int CHUNKS = KT * (TOK_D / 8), NL = 2 * CHUNKS / 256;  // 16-byte pieces of a K (V) tile; of both, per thread
  __shared__ __attribute__((aligned(16))) char sTile[2][TOK_TILE];  // [buffer]: K rows, V rows
  __shared__ __attribute__((aligned(16))) float sRep[2][KT];        // what takes the place of a masked key's logit, or 0
  __shared__ int sAny[2];                                           // whether it does for any key of the tile

  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, j = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // flash_kernel's order of workgroups: logical = (head * query tiles + query tile) * B + batch
  const int logical = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (logical >= a.n_blocks) return;
  const int rest = a.B == 1 ? logical : (int)__umulhi((uint32_t)logical, a.magic_b), b = logical - rest * a.B;
  const int h = a.q_tiles == 1 ? rest : (int)__umulhi((uint32_t)rest, a.magic_t);
  const int q0 = (rest - h * a.q_tiles) * 128 + wave * 32, qi = min(q0 + j, a.Sq - 1);  // clamped for loads; stores are guarded
  const int nkt = (a.Sk + KT - 1) / KT;

  // The descriptor of a tile begins at its first key (or quad) and ends where the plane does: a lane's offset never changes, and all
  // of what lies past the last key is past the descriptor's end by that offset alone (the scalar one stays 0: what it may add
  // to a checked offset is not laid down).
  auto from = [](const void* p, int bytes, int at) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(p) + at), 0, max(bytes - at, 0), RSRC_RAW);
  };
  const bf16_t *const kg = a.k + b * a.k_sb + h * TOK_D, *const vg = a.v + b * a.v_sb + h * TOK_D;
  const int k_bytes = ((a.Sk - 1) * (int)a.k_ss + TOK_D) * 2, v_bytes = ((a.Sk - 1) * (int)a.v_ss + TOK_D) * 2;
  const int quad_step = (int)(a.bias_squad ? a.bias_squad : 4), quads = (a.Sk + 3) >> 2;
  const float* const bg = a.bias + (int64_t)b * a.bias_sb + (int64_t)h * a.bias_sh;
  const int b_bytes = ((a.Sq - 1) * (int)a.bias_sq + (quads - 1) * quad_step + 4) * 4, b_step = KT / 4 * quad_step * 4;
  const float* kmask = a.key_mask ? a.key_mask + (int64_t)b * a.km_sb : nullptr;

  // bias of a tile in four parts of two quads: part p = registers 8 p .. of the 32,
  // s[u][4 g + e] = bias(query, key 64 kt + 32 u + 8 g + 4 hh + e)
  uint32_t quad_at[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) quad_at[i] = (uint32_t)(qi * (int)a.bias_sq + (hh + 2 * i) * quad_step) * 4u;
  auto load_bias = [&](f32x16 (&s)[2], int kt, int part) {
    const int u = part >> 1;
    const __amdgpu_buffer_rsrc_t rest = from(bg, b_bytes, kt * b_step);
#pragma unroll
    for (int g = 2 * (part & 1); g < 2 * (part & 1) + 2; ++g) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rest, quad_at[4 * u + g], 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[u][4 * g + e] = __uint_as_float(v[e]);
    }
  };
  // piece i of this thread: K pieces first, then V (which of the two is uniform over a wave: CHUNKS is a multiple of 64)
  u32x4 rc[NL];
  uint32_t choff[NL], lds_at[NL];
  const char* from_key[NL];  // (uniform) of the tile asked for next, and the bytes that are left from there
  int left[NL], step[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int e = tid + i * 256;
    const bool is_v = e >= CHUNKS, wave_v = wave * 64 + i * 256 >= CHUNKS;
    from_key[i] = reinterpret_cast<const char*>(wave_v ? vg : kg);
    left[i] = wave_v ? v_bytes : k_bytes;
    step[i] = KT * 2 * (int)(wave_v ? a.v_ss : a.k_ss);
    const int ch = is_v ? e - CHUNKS : e, c = ch % (TOK_D / 8), key = ch / (TOK_D / 8);
    choff[i] = (uint32_t)(key * (int)(is_v ? a.v_ss : a.k_ss) + c * 8) * 2u;
    lds_at[i] = (is_v ? TOK_K_BYTES + key * (TOK_LDV * 2) : key * (TOK_LDK * 2)) + c * 16;
  }
  float mask_value = 1.f;  // of key tid of the tile asked for last (threads 0..63)
  auto load_tile = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      rc[i] = __builtin_amdgcn_raw_buffer_load_b128(from(from_key[i], left[i], 0), choff[i], 0, 0);
      from_key[i] += step[i];
      left[i] -= step[i];
    }
    if (kmask && tid < KT) mask_value = kmask[min(kt * KT + tid, a.Sk - 1)];
  };
  auto store_tile = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(sTile[kt & 1] + lds_at[i]) = rc[i];
  };
  auto store_mask = [&](int kt) {
    const int buf = kt & 1;
    if (tid < KT) {
      const float rep = kt * KT + tid >= a.Sk ? NEG_INF : (mask_value == 0.f ? -1e9f : 0.f);
      sRep[buf][tid] = rep;
      const bool any = __any(rep != 0.f);
      if (tid == 0) sAny[buf] = any ? 1 : 0;
    }
  };

  f32x16 setA[2], setB[2];
  bf16x8 qf[3];
#pragma unroll
  for (int ks = 0; ks < 3; ++ks)
    qf[ks] = as_frag(*reinterpret_cast<const u32x4*>(a.q + (int64_t)b * a.q_sb + (int64_t)qi * a.q_ss + h * TOK_D + 16 * ks + 8 * hh));
  load_tile(0);
#pragma unroll
  for (int p = 0; p < 4; ++p) load_bias(setA, 0, p);
  // V's columns 48..63 of either buffer, which the products read: ones in the first, whose product is the row sum, and zeros
  for (int idx = tid; idx < 2 * KT * 2; idx += 256) {
    const int row = idx >> 1;
    *reinterpret_cast<u32x4*>(sTile[row / KT] + TOK_K_BYTES + (row % KT) * (TOK_LDV * 2) + TOK_D * 2 + (idx & 1) * 16) =
        u32x4{idx & 1 ? 0u : 0x3F80u, 0u, 0u, 0u};
  }
  f32x16 o[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;
  float m_run = NEG_INF;
  store_tile(0);
  store_mask(0);
  load_tile(1);
#pragma unroll
  for (int p = 0; p < 4; ++p) load_bias(setB, 1, p);
  lds_barrier();

  auto tile = [&](int kt, f32x16 (&s)[2]) {
    const int buf = kt & 1;
    const char* kv = sTile[buf];
    bf16x8 kf[3][2];
#pragma unroll
    for (int ks = 0; ks < 3; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u) kf[ks][u] = lds_frag(reinterpret_cast<const bf16_t*>(kv), TOK_LDK, u * 32, ks * 16, lane);
    if (kt + 1 < nkt) store_mask(kt + 1);  // (the other buffer was last read in front of the barrier)
#pragma unroll
    for (int ks = 0; ks < 3; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u) s[u] = mfma32(kf[ks][u], qf[ks], s[u]);
    // V's fragments, read while the exponentials' base is found (the transposing reads: see flash_kernel)
    const int i16 = lane & 15;
    const bf16_t* vbase = reinterpret_cast<const bf16_t*>(kv + TOK_K_BYTES) + (4 * hh + (i16 >> 2)) * TOK_LDV + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);
    v4s vf[2][2][2];
    auto read_v = [&](int p) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bf16_t* vp = vbase + 16 * p * TOK_LDV + t * 32;
        vf[p & 1][t][0] = lds_read_tr16(vp);
        vf[p & 1][t][1] = lds_read_tr16(vp + 8 * TOK_LDV);
      }
    };
    read_v(0);
    __builtin_amdgcn_sched_barrier(0);
    if (__builtin_amdgcn_readfirstlane(sAny[buf])) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const f32x4 rep = *reinterpret_cast<const f32x4*>(&sRep[buf][8 * q + 4 * hh]);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[q >> 2][4 * (q & 3) + e] = rep[e] != 0.f ? rep[e] : s[q >> 2][4 * (q & 3) + e];
      }
    }
    float mx = max3_of_32(s);
    const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    mx = fmaxf(__uint_as_float(r2[0]), __uint_as_float(r2[1]));
    constexpr float BASE_SLACK = 8.f;  // see flash_kernel
    const float m_new = mx - m_run > BASE_SLACK ? mx : m_run;
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
    m_run = m_new;
    const float m2 = m_new * LOG2E;
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
    }
    // a quarter's products run beside the next one's exponentials
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[p >> 1][8 * (p & 1) + e], LOG2E, -m2));
      const bf16x8 pf = as_frag(pack8(pv));
      __builtin_amdgcn_sched_barrier(0);
      if (p < 3) read_v(p + 1);
      load_bias(s, kt + 2, p);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const v4s lo = vf[p & 1][t][0], hi = vf[p & 1][t][1];
        o[t] = mfma32(as_frag(__builtin_bit_cast(u32x4, v8s{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w})), pf, o[t]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (kt + 1 < nkt) {
      store_tile(kt + 1);
      load_tile(kt + 2);
    }
    lds_barrier();
  };
  // the output gate: asked for in front of the last tile
  u32x2 gate[6];
  const int64_t row = qi;
  auto load_gate = [&]() {
#pragma unroll
    for (int g = 0; g < 6; ++g) gate[g] = u32x2{0x3F803F80u, 0x3F803F80u};
    if (!a.g) return;
    const bf16_t* gp = a.g + (int64_t)b * a.g_sb + row * a.g_ss + h * TOK_D + 4 * hh;
#pragma unroll
    for (int g = 0; g < 6; ++g) gate[g] = *reinterpret_cast<const u32x2*>(gp + 8 * g);
  };
  load_gate();
  for (int kt = 0; kt < nkt; kt += 2) {
    tile(kt, setA);
    if (kt + 1 < nkt) tile(kt + 1, setB);
  }

  // the sum of the rounded probabilities: row 48 of o, register 8 of the second block's lower half
  const auto sum = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[1][8]), __float_as_uint(o[1][8]), false, false);
  const float inv = 1.f / __uint_as_float(sum[0]);
  if (q0 + j >= a.Sq) return;
  const int64_t at = (int64_t)b * a.o_sb + row * a.o_ss + h * TOK_D + 4 * hh;
#pragma unroll
  for (int g = 0; g < 6; ++g) {  // head dimensions 8 g + 4 hh ..
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = o[g >> 2][4 * (g & 3) + e] * inv;
    v[0] *= bflo(gate[g].x); v[1] *= bfhi(gate[g].x); v[2] *= bflo(gate[g].y); v[3] *= bfhi(gate[g].y);
    if (a.out_f32) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + at + 8 * g) = f32x4{v[0], v[1], v[2], v[3]};
    } else {
      u32x2 w;
      w.x = pack2bf(v[0], v[1]);
      w.y = pack2bf(v[2], v[3]);
      *reinterpret_cast<u32x2*>(reinterpret_cast<bf16_t*>(a.out) + at + 8 * g) = w;
    }
  }
}

// ------------------------------------------------------------------ windows of gathered keys
// The atom transformers' attention: many short windows (32 queries, up to 128 keys that are looked up in a table of
// rows), four heads of 32 channels.  There is next to no arithmetic in one (0.5 MFLOP a head); what counts is the CU's
// vector memory path, which takes a cache line every two cycles or so, whole or in part, and the number of round trips
// one after the other.  The form above, a wave per window and head, touches every line many times over (a key's row is
// 64 bytes to a head, the bias of a lane's query 16 bytes to a load) and goes through rows, K and V, LDS twice.  Here a
// workgroup of four waves takes the four heads of a window: K and V rows of all heads come as runs of 256 bytes straight
// into LDS (an empty slot or a key past the end: an offset past the buffer's end, which writes zeros), everything else
// is asked for at the same time, gate and result travel in 16-byte pieces, and the bias, with quads of keys as the outer
// index (bias_squad), in whole lines.  The samples' windows of one place, which share the bias, follow each other on
// one XCD.  The arithmetic is that of flash_kernel, in the same order: the same bits.
// 2880 windows (768 tokens, 5 samples) 46 us (flash_kernel 80), 1440 windows 27 (45), 375 windows 13.5 (17).
// In LDS chunk c (16 bytes) of a key's row lies at position c ^ (key % 4 * 4 + key / 4 % 4): fragment reads of 32 keys
// and the transposing reads of 8 keys x 64 bytes both spread over the banks.
__device__ __forceinline__ u32x4 table_buffer(const void* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return u32x4{lo, hi & 0xffffu, 0x7fffffffu, 0x00020000u};
}
// a's upper half of the wave and b's lower half change places
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// TILES: tiles of 64 keys in LDS at a time.  With both (66 KB, two workgroups on a CU) a window is the shortest chain;
// with one after the other a CU takes four windows, which hide each other's waits.
constexpr int WKEYS = 128;
template <int TILES>
__global__ __launch_bounds__(256, TILES == 2 ? 2 : 4) void window_kernel(FlashArgs a) {
  args_at_once<FlashArgs>();
  __shared__ __attribute__((aligned(1024))) bf16_t sK[64 * TILES * 128];
  __shared__ __attribute__((aligned(1024))) bf16_t sV[64 * TILES * 128];
  __shared__ __attribute__((aligned(16))) int sCode[WKEYS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int h = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, j = lane & 31;
  const int xaddr = half_swap_addr();
  const int samples = a.B / a.bias_mod, work = a.windows ? min(a.windows[0], a.bias_mod) * samples : a.B;
  const int per_xcd = (work + 7) >> 3, logical = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || logical >= work) return;
  const int place = logical / samples, sample = logical - place * samples, bb = a.windows ? a.windows[1 + place] : place;
  if ((unsigned)bb >= (unsigned)a.bias_mod) return;
  const int b = sample * a.bias_mod + bb;
  const int qi = min(j, a.Sq - 1);
  const bool q_ok = j < a.Sq;

  // the wave's share of the key rows, four to a load
  const int* krows = a.key_rows + (int64_t)bb * a.Sk;
  auto key_of = [&](int i) { return (i / (4 * TILES)) * (64 * TILES) + 16 * TILES * h + 4 * (i % (4 * TILES)) + (lane >> 4); };
  int row[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) row[i] = krows[min(key_of(i), a.Sk - 1)];
  if (tid < WKEYS) {
    float pad = 1.f;
    if (a.kpad) pad = a.kpad[(int64_t)bb * a.kp_sb + min(tid, a.Sk - 1)];
    sCode[tid] = (tid >= a.Sk ? KEY_BEYOND : 0) | (pad == 0.f ? KEY_PAD : 0);
  }
  const bool q_is_pad = a.qpad ? (a.qpad[(int64_t)bb * a.qp_sb + qi] == 0.f) : false;
  bf16x8 qf[2];
  u32x4 gate[2];
  const int64_t q_at = (int64_t)qi * a.q_ss + h * 32 + 8 * hh;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    qf[ks] = as_frag(*reinterpret_cast<const u32x4*>(a.q + (int64_t)b * a.q_sb + q_at + 16 * ks));
    gate[ks] = u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
    if (a.g) gate[ks] = *reinterpret_cast<const u32x4*>(a.g + (int64_t)b * a.g_sb + (int64_t)qi * a.g_ss + h * 32 + 8 * hh + 16 * ks);
  }
  const float* bias_row = a.bias + (int64_t)bb * a.bias_sb + (int64_t)h * a.bias_sh + (int64_t)qi * a.bias_sq;
  const int64_t quad_step = a.bias_squad ? a.bias_squad : 4;
  const u32x4 kt = table_buffer(a.k + (int64_t)sample * a.k_sb), vt = table_buffer(a.v + (int64_t)sample * a.v_sb);
  auto lds_of = [&](const bf16_t* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const bf16_t*)p + h * 16 * TILES * 256);
  };
  const uint32_t k_lds = lds_of(sK), v_lds = lds_of(sV);
  const uint32_t swz = (uint32_t)((j & 3) << 2 | (j >> 2 & 3));
  const char* kl = reinterpret_cast<const char*>(sK) + j * 256;
  const int i16 = lane & 15;
  const uint32_t v_chunk = 4 * h + 2 * (lane >> 4 & 1) + (i16 >> 1 & 1), v_swz = (uint32_t)((i16 >> 2) << 2 | hh);
  const char* vl = reinterpret_cast<const char*>(sV) + (4 * hh + (i16 >> 2)) * 256 + 8 * (i16 & 1);
  const uint32_t v_lo = (v_chunk ^ v_swz) << 4, v_hi = ((v_chunk ^ v_swz ^ 2) << 4) + 8 * 256;
  const bf16x8 onesf = as_frag(u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
  f32x16 o;
#pragma unroll
  for (int r = 0; r < 16; ++r) o[r] = 0.f;
  float m_run = NEG_INF, l_run = 0.f;
  bool any = false;
#pragma unroll
  for (int st = 0; st < 2 / TILES; ++st) {
    const int first = 64 * TILES * st;
    if (first >= a.Sk) break;
    if (st > 0) lds_barrier();  // every wave is through with the previous tile
    // s[u][4g + e]: the logit of key first + 32u + 8g + 4hh + e, accumulated on the bias
    f32x16 s[2 * TILES];
#pragma unroll
    for (int u = 0; u < 2 * TILES; ++u)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(bias_row + (min(first + 32 * u + 8 * g + 4 * hh, a.Sk - 4) >> 2) * quad_step);
        s[u][4 * g] = v.x; s[u][4 * g + 1] = v.y; s[u][4 * g + 2] = v.z; s[u][4 * g + 3] = v.w;
      }
#pragma unroll
    for (int i = 0; i < 4 * TILES; ++i) {
      const int r = row[4 * TILES * st + i];
      const bool ok = r >= 0 && key_of(4 * TILES * st + i) < a.Sk;
      const uint32_t chunk = (uint32_t)((lane & 15) ^ ((lane >> 4 & 3) << 2 | (i & 3))) * 16u;
      const uint32_t ko = ok ? (uint32_t)r * (uint32_t)a.k_ss * 2u + chunk : 0x80000000u;
      const uint32_t vo = ok ? (uint32_t)r * (uint32_t)a.v_ss * 2u + chunk : 0x80000000u;
      asm volatile("s_add_u32 m0, %0, %6\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
                   "s_add_u32 m0, %3, %6\n\ts_nop 0\n\tbuffer_load_dwordx4 %4, %5, 0 offen lds" ::"s"(k_lds), "v"(ko), "s"(kt),
                   "s"(v_lds), "v"(vo), "s"(vt), "n"(i * 1024)
                   : "m0", "scc", "memory");
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // key codes (a key of padding, a key past the end): most windows have none
    if (st == 0) any = __any((sCode[lane] | sCode[64 + lane]) != 0);
#pragma unroll
    for (int u = 0; u < 2 * TILES; ++u)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        s[u] = mfma32(as_frag(*reinterpret_cast<const u32x4*>(kl + u * 32 * 256 + (((4 * h + 2 * ks + hh) ^ swz) << 4))), qf[ks], s[u]);
    if (any) {
#pragma unroll
      for (int u = 0; u < 2 * TILES; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int* cp = &sCode[first + u * 32 + 8 * g + 4 * hh];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = s[u][4 * g + e];
            if (q_is_pad && (cp[e] & KEY_PAD)) v += 1e9f;
            if (cp[e] & KEY_BEYOND) v = NEG_INF;
            s[u][4 * g + e] = v;
          }
        }
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {  // tiles of 64 keys, as flash_kernel takes them
      if (first + 64 * t >= a.Sk) break;
      float m4[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x16& x = s[2 * t + (i >> 1)];
        const int r = 8 * (i & 1);
        m4[i] = fmaxf(fmaxf(fmaxf(x[r], x[r + 1]), fmaxf(x[r + 2], x[r + 3])), fmaxf(fmaxf(x[r + 4], x[r + 5]), fmaxf(x[r + 6], x[r + 7])));
      }
      float mx = fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]));
      mx = fmaxf(mx, half_swap(xaddr, mx));
      constexpr float BASE_SLACK = 8.f;
      const float m_new = mx - m_run > BASE_SLACK ? mx : m_run;
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * LOG2E);
      m_run = m_new;
      const float m2 = m_new * LOG2E;
      bf16x8 pf[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          float pv[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) pv[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * t + u][8 * half + e], LOG2E, -m2));
          pf[u][half] = as_frag(pack8(pv));
        }
      f32x16 lsum;
#pragma unroll
      for (int r = 0; r < 16; ++r) lsum[r] = 0.f;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int half = 0; half < 2; ++half) lsum = mfma32(onesf, pf[u][half], lsum);
      l_run = l_run * alpha + lsum[0];
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) o[r] *= alpha;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const char* vp = vl + (64 * t + u * 32 + 16 * half) * 256;
          const v4s lo = lds_read_tr16(reinterpret_cast<const bf16_t*>(vp + v_lo)), hi = lds_read_tr16(reinterpret_cast<const bf16_t*>(vp + v_hi));
          o = mfma32(as_frag(__builtin_bit_cast(u32x4, v8s{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w})), pf[u][half], o);
        }
    }
  }
  // o[4g + e] = out(query j, channel 8g + 4hh + e); gate[ks] holds channels 16 ks + 8 hh .. + 7: exchanging its middle
  // quads with the other half of the wave makes them quads g = 2 ks and 2 ks + 1, and takes the result the other way
  const float inv = 1.f / l_run;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    uint32_t w[4] = {gate[ks].x, gate[ks].y, gate[ks].z, gate[ks].w};
    swap_halves(w[0], w[2]);
    swap_halves(w[1], w[3]);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = o[8 * ks + e] * inv;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      v[4 * g] *= bflo(w[2 * g]); v[4 * g + 1] *= bfhi(w[2 * g]); v[4 * g + 2] *= bflo(w[2 * g + 1]); v[4 * g + 3] *= bfhi(w[2 * g + 1]);
    }
    const int64_t at = (int64_t)b * a.o_sb + (int64_t)qi * a.o_ss + h * 32 + 16 * ks;
    if (a.out_f32) {
      float* out = reinterpret_cast<float*>(a.out) + at + 4 * hh;
      if (q_ok) {
        *reinterpret_cast<f32x4*>(out) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4*>(out + 8) = f32x4{v[4], v[5], v[6], v[7]};
      }
    } else {
      uint32_t p[4] = {pack2bf(v[0], v[1]), pack2bf(v[2], v[3]), pack2bf(v[4], v[5]), pack2bf(v[6], v[7])};
      swap_halves(p[0], p[2]);
      swap_halves(p[1], p[3]);
      if (q_ok) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(a.out) + at + 8 * hh) = u32x4{p[0], p[1], p[2], p[3]};
    }
  }
}

// what window_kernel takes: its shapes, a bias in rows of whole quads, tables whose byte offsets fit 31 bits
bool window_fits(const FlashArgs& a) {
  return a.key_rows && a.bias && !a.key_mask && a.H == 4 && a.d == 32 && a.Sq <= 32 && a.Sk <= WKEYS && (a.Sk & 3) == 0 &&
         ((a.bias_sq | a.bias_sb | a.bias_sh | a.bias_squad) & 3) == 0 && ((uintptr_t)a.bias & 15) == 0 && a.k_ss > 0 && a.v_ss > 0 &&
         a.table_rows > 0 && a.table_rows * (a.k_ss > a.v_ss ? a.k_ss : a.v_ss) < (1ll << 30);
}

// Queries per workgroup: 128 (four waves share the K / V tiles), 64, or 32 for
// the short query windows of the atom cross-attention.
template <int KSTEPS, int DVT>
int launch_nw(const FlashArgs& a, hipStream_t stream) {
  const int64_t heads = (int64_t)a.H * a.B;
  // The form with fixed per-lane offsets: no row table, a bias that can be fetched 16 bytes at a time, and
  // offsets inside a key tile / a bias plane that fit 32 bits.
  const int64_t quad_step = a.bias_squad ? a.bias_squad : 4;
  const bool fast = !a.key_rows && a.bias && a.Sk >= 4 && (a.bias_sq & 3) == 0 && (a.bias_sb & 3) == 0 &&
                    (a.bias_sh & 3) == 0 && (a.bias_squad & 3) == 0 && ((uintptr_t)a.bias & 15) == 0 &&
                    a.k_ss > 0 && a.v_ss > 0 && a.k_ss < (1 << 22) && a.v_ss < (1 << 22) && a.bias_sq >= 0 &&
                    quad_step > 0 && (int64_t)a.Sq * a.bias_sq + quad_step < (1 << 28);
  // Four waves share each staged K / V tile once there are enough 128-query workgroups to cover the chip; below that, two
  // waves per workgroup spread the work over twice as many CUs.  Not with head dimension 48 (and padding flags or a bias
  // shared by batch % bias_mod: without them token_attention_kernel has it), where the form with fixed offsets needs four waves to
  // share the staging registers.
  const int nw = a.Sq <= 32 ? 1 : (((a.Sq + 127) / 128) * heads < 256 && !(KSTEPS == 3 && fast) ? 2 : 4);
  const int64_t n_blocks = (int64_t)((a.Sq + nw * 32 - 1) / (nw * 32)) * heads;
  if (n_blocks <= 0 || n_blocks > 0x7ffffff0) return AF3_ERR_BAD_ARG;
  FlashArgs fa = a;
  if constexpr (KSTEPS == 3) {
    // (padding flags, and a bias that entries share by batch % bias_mod, are flash_kernel's; byte offsets of 31 bits inside a
    // sample's rows and a head's bias plane, two tiles past the end included; products of the workgroups' numbers and their divisors
    // of 32)
    const int64_t keys = (a.Sk + 191) / 64 * 64, limit = (int64_t)1 << 29, tiles = (a.Sq + 127) / 128, blocks = tiles * heads;
    if (fast && !a.qpad && a.bias_mod == 0 && keys * (a.k_ss > a.v_ss ? a.k_ss : a.v_ss) < limit &&
        (int64_t)a.Sq * a.bias_sq + (keys / 4) * quad_step < limit && blocks * a.B < (1ll << 32) && blocks * tiles < (1ll << 32)) {
      fa.n_blocks = (int)blocks;
      fa.per_xcd = (int)((blocks + 7) / 8);
      fa.q_tiles = (int)tiles;
      fa.magic_b = a.B == 1 ? 0u : 0xffffffffu / (uint32_t)a.B + 1u;
      fa.magic_t = tiles == 1 ? 0u : 0xffffffffu / (uint32_t)tiles + 1u;
      hipLaunchKernelGGL(token_attention_kernel, dim3(8u * fa.per_xcd), dim3(256), 0, stream, fa);
      return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
    }
  }
  fa.n_blocks = (int)n_blocks;
  const dim3 grid((unsigned)((n_blocks + 7) / 8 * 8));  // whole rounds over the 8 XCDs; the surplus ids return at once
  // (with a single wave, or with head dimension 48 and fewer than four waves, to share the K / V staging
  // registers between, the second register set of that form no longer fits: those take the general form)
#define AF3_FLASH_LAUNCH(NW_)                                                                                   \
  do {                                                                                                          \
    if constexpr (NW_ == 4 || (KSTEPS < 3 && NW_ == 2)) {                                                       \
      if (fast) {                                                                                               \
        hipLaunchKernelGGL((flash_kernel<KSTEPS, DVT, NW_, true>), grid, dim3(NW_ * 64), 0, stream, fa);        \
        break;                                                                                                  \
      }                                                                                                         \
    }                                                                                                           \
    hipLaunchKernelGGL((flash_kernel<KSTEPS, DVT, NW_, false>), grid, dim3(NW_ * 64), 0, stream, fa);           \
  } while (0)
  if (nw == 1) AF3_FLASH_LAUNCH(1);
  else if (nw == 2) AF3_FLASH_LAUNCH(2);
  else AF3_FLASH_LAUNCH(4);
#undef AF3_FLASH_LAUNCH
  return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
}

}  // namespace

int launch_flash_attention(const FlashArgs& a, hipStream_t stream) {
  if (a.B <= 0 || a.H <= 0 || a.Sq <= 0 || a.Sk <= 0 || !a.q || !a.k || !a.v || !a.out) return AF3_ERR_BAD_ARG;
  if (a.d != 16 && a.d != 24 && a.d != 32 && a.d != 48) return AF3_ERR_UNSUPPORTED;
  const int64_t strides[] = {a.q_sb, a.q_ss, a.k_sb, a.k_ss, a.v_sb, a.v_ss, a.g_sb, a.g_ss, a.o_sb, a.o_ss};
  for (int64_t s : strides)
    if (s & 7) return AF3_ERR_BAD_ARG;
  if (((uintptr_t)a.q & 15) || ((uintptr_t)a.k & 15) || ((uintptr_t)a.v & 15) || ((uintptr_t)a.g & 15) ||
      ((uintptr_t)a.out & 15))
    return AF3_ERR_BAD_ARG;
  if ((a.qpad == nullptr) != (a.kpad == nullptr)) return AF3_ERR_BAD_ARG;
  if (a.bias_mod < 0 || (a.bias_mod > 0 && a.B % a.bias_mod) || (a.key_rows && a.bias_mod <= 0)) return AF3_ERR_BAD_ARG;
  if (a.bias_squad && (a.bias_sq != 4 || (a.bias_squad & 3))) return AF3_ERR_BAD_ARG;
  if (window_fits(a)) {
    const dim3 grid((unsigned)((a.B + 7) / 8 * 8)), block(256);
    if (a.B <= 512) hipLaunchKernelGGL(window_kernel<2>, grid, block, 0, stream, a);  // two on every CU hold them all
    else hipLaunchKernelGGL(window_kernel<1>, grid, block, 0, stream, a);
    return hipGetLastError() == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
  }
  if (a.d == 48) return launch_nw<3, 2>(a, stream);
  if (a.d == 16) return launch_nw<1, 1>(a, stream);
  return launch_nw<2, 1>(a, stream);
}
