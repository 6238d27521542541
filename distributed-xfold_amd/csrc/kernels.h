// Host-side launch interface of the kernels (internal; the public C ABI is in
// include/af3_hip.h and implemented in api.hip).
#pragma once
#include "common.h"

// ------------------------------------------------------------------ gemm.hip
enum { EPI_PLAIN = 0, EPI_SEGMENTED = 1, EPI_SWIGLU = 2, EPI_GATE_RES = 3 };
enum { SEG_PLAIN = 0, SEG_BIAS_SCALE = 1, SEG_SIGMOID = 2 };

struct GemmArgs {
  const bf16_t* A = nullptr;  // [batch][M][lda]
  const bf16_t* B = nullptr;  // [batch][N][ldb]   (C = A * B^T)
  void* C = nullptr;          // [batch][M][ldc]   bf16 or fp32
  int M = 0, N = 0, K = 0, batch = 1;
  int64_t lda = 0, ldb = 0, ldc = 0, sA = 0, sB = 0, sC = 0;
  int out_f32 = 0;
  int epi = EPI_PLAIN;
  float alpha = 1.f;            // PLAIN: (acc + bias) * alpha ; SEG_BIAS_SCALE likewise
  const float* bias = nullptr;  // indexed by output column: entries 0 .. bias_len - 1 exist
  int64_t bias_len = 0;         // a launch whose epilogue would read past it is refused (gemm_bias_span)
  int act_sigmoid = 0;          // PLAIN only
  int seg_len = 0, seg_ops = 0; // SEGMENTED: op of column segment s in bits [4s, 4s+4)
  const float* gate = nullptr;  // GATE_RES: multiply by gate[m % gate_rows][n]
  int gate_rows = 0;
  int gate_per_row = 0;         // GATE_RES: gate is one factor per row, gate[m % gate_rows]
  int64_t ld_gate = 0;
  const float* res_f32 = nullptr;   // GATE_RES: residual added last (either dtype)
  const bf16_t* res_bf16 = nullptr;
  int64_t ld_res = 0, sRes = 0;
  // regroup32 (PLAIN, batch 1, M and N multiples of 32): element (m, n) is stored
  // at [(m / 32, n / 32)][(m % 32, n % 32)], i.e. C is [(M/32)(N/32)][1024]:
  // the outer products of 32-channel rows, one contiguous 1024-vector per pair.
  int regroup32 = 0;
  const bf16_t* w2 = nullptr;  // launch_outer_mean only
  int xcd_m = 0;               // set by the launchers: XcdWalk::rows
  int small_tiles = 0;  // never the 256x256 tile (same sums, same order)
  int split_k = 0;  // the K range may be summed in parts by several waves (another order of summation)
};
int launch_gemm_nt(const GemmArgs& g, hipStream_t stream);
// wide_product.hip: K = 384, fp32 results of very many columns
struct WideWalk {
  int per_xcd = 0, total = 0, parts = 0, panels = 0;  // parts of a strip's rows, and their panels of 32
  unsigned magic_parts = 0;
};
bool wide_product_applies(const GemmArgs& g);
int launch_wide_product(const GemmArgs& g, hipStream_t stream);
// panel.hip: square products of up to a few hundred rows a batch entry; AF3_ERR_UNSUPPORTED for others
int launch_panel_product(const GemmArgs& g, hipStream_t stream);

// Which tiles of a product run on which XCD.  Each XCD has an L2 of its own, 4 MB, and fetches for itself every row of A
// and B that its tiles touch.  rows = 0: the XCDs share the tiles (batch, n, m), m fastest, in eight runs: every XCD
// fetches all of A for an eighth of B, right for few rows and for many small products.  rows = 1, 2, 4 or 8: one
// product's tiles are dealt as a rows x (8 / rows) grid of rectangles, an XCD fetches 1 / rows of A and rows / 8 of B.
struct XcdWalk {
  int rows = 0;
  int64_t slots = 0;  // tiles of the busiest XCD
};
// The walk that fetches least, if that is at least a third less, no XCD gets 4 % more tiles than its share, and its
// tiles take no more rounds.  `per_round`: tiles that an XCD's 32 CUs hold at a time.  An uneven deal costs what it
// saves (1920 x 768 x 1536 in 64 x 64 tiles: 48 tiles against 45, 16.8 us against 15.4), and a whole round where the
// even deal just fits: 33 tiles against 32 on one XCD (5300 x 768 x 1536 with gate and residual in 128 x 128 tiles 35.9 us,
// even 23.8; 3900 x 3072 x 768 in 192 x 256 tiles 42.0, even 27.4, with SwiGLU 32.3 and 22.0).
// 3840 x 768 x 768 14.3 -> 12.4 us, 3840 x 768 x 1536 24.1 -> 22.0.
constexpr int XCD_CUS = 32;
inline XcdWalk xcd_walk(int64_t tiles_m, int64_t tiles_n, int64_t batch, int bm, int bn, int64_t per_round) {
  XcdWalk w;
  w.slots = (tiles_m * tiles_n * batch + 7) / 8;
  if (batch != 1) return w;
  int64_t least = (w.slots < tiles_m ? w.slots : tiles_m) * bm + ((w.slots + tiles_m - 1) / tiles_m) * bn;
  const int64_t limit = least * 2 / 3, rounds = (w.slots + per_round - 1) / per_round;
  for (int rows = 1; rows <= 8; rows *= 2) {
    const int64_t m = (tiles_m + rows - 1) / rows, n = (tiles_n + 8 / rows - 1) / (8 / rows), fetch = m * bm + n * bn;
    if (m * n * 25 > w.slots * 26 || (m * n + per_round - 1) / per_round > rounds || fetch > limit || fetch >= least) continue;
    least = fetch;
    w.rows = rows;
  }
  if (w.rows) w.slots = ((tiles_m + w.rows - 1) / w.rows) * ((tiles_n + 8 / w.rows - 1) / (8 / w.rows));
  return w;
}
// tile number `slot` of an XCD's rectangle; false behind its last
__device__ __forceinline__ bool xcd_rect_tile(int rows, int xcd, int slot, int tiles_m, int tiles_n, int* tm, int* tn) {
  const int cols = 8 / rows, i = xcd & (rows - 1), j = xcd / rows;
  const int m0 = tiles_m * i / rows, mh = tiles_m * (i + 1) / rows - m0;
  const int n0 = tiles_n * j / cols, nh = tiles_n * (j + 1) / cols - n0;
  if (slot >= mh * nh) return false;
  *tm = m0 + slot % mh;
  *tn = n0 + slot / mh;
  return true;
}
// af3_linear_forward and af3_batch_diffusion_self_attention_forward (api.hip) for callers inside the library that do
// not mind the order in which the products sum K (GemmArgs::split_k)
int run_linear(const bf16_t* x, const bf16_t* w, const float* bias, void* y, int y_dtype, int64_t m, int n, int k, int mode,
               float alpha, int sigmoid, const float* gate, int64_t gate_rows, int64_t gate_ld, const void* residual,
               int res_dtype, int split_k, hipStream_t stream);
// run_self_attention's second half, on projections that are there (its workspace holds them, self_projections)
int run_self_attend(const bf16_t* qkvg, const float* key_mask, int64_t mask_batches, const float* nonbatched_bias, int bias_quad_major,
                    int num_head, void* out, int out_dtype, int64_t batch, int64_t seq, int channels, hipStream_t s);
bf16_t* self_projections(void* workspace, size_t workspace_bytes, int64_t rows, int channels);
int run_self_attention(const bf16_t* q_data, const float* key_mask, int64_t mask_batches, const float* nonbatched_bias,
                       int bias_quad_major, const bf16_t* w_qkvg, const float* query_b, int num_head, void* out, int out_dtype,
                       int64_t batch, int64_t seq, int channels, void* workspace, size_t workspace_bytes, int split_k,
                       hipStream_t stream);
// af3_gathered_cross_attention_forward, with the pair logits in rows or (bias_quad_major) in quads of keys
int run_gathered_attention(const bf16_t* q_data, const bf16_t* atom_data, const int32_t* key_rows, const float* pair_logits,
                           int bias_quad_major, const float* mask_q, const float* mask_k, int64_t bias_batches, const bf16_t* w_qg,
                           const bf16_t* w_kv, const float* query_b, int num_head, void* out, int out_dtype, int64_t batch,
                           int64_t sq, int64_t sk, int64_t samples, int64_t n_atoms, int channels, void* workspace,
                           size_t workspace_bytes, hipStream_t stream, const int* windows = nullptr);
// where in its workspace the projections are (false: too small); with q_data and atom_data null they are there already
bool gathered_projections(void* workspace, size_t workspace_bytes, int64_t query_rows, int64_t atom_rows, int channels, bf16_t** qg,
                          bf16_t** kv);
// Which bias entries a launch reads.  Column c takes bias[c] when the epilogue is not segmented, or
// when c lies in a segment whose op is SEG_BIAS_SCALE; the kernels read whole groups of entries
// (gemm_nt_kernel up to 8 from a multiple of 8, the large tile 4 from a multiple of 4, the last
// group pulled back to end at N).  The device code takes its addresses from these functions, the
// host takes the extent it checks against bias_len from them: one formula for both.
__host__ __device__ inline bool gemm_col_uses_bias(const GemmArgs& g, int col) {
  if (!g.bias) return false;
  if (g.epi != EPI_SEGMENTED) return true;
  return ((g.seg_ops >> (4 * (col / g.seg_len))) & 15) == SEG_BIAS_SCALE;
}
// large tile: the 4 entries a lane fetches for columns colb .. colb + 3 of its wave (colb may lie past N)
__host__ __device__ inline bool big_tile_bias_quad(const GemmArgs& g, int colb, int* first) {
  *first = (colb < g.N - 4 ? colb : g.N - 4);
  return gemm_col_uses_bias(g, colb < g.N - 1 ? colb : g.N - 1);
}
// Half-open range [first, last) of bias entries the launch of `g` reads (big: on the large tile);
// first == last: none.
void gemm_bias_span(const GemmArgs& g, bool big, int64_t* first, int64_t* last);
// contract.hip: the same product, plain bf16 output, 256x256 tiles (large M, N)
bool contract_supported(const GemmArgs& g);
int launch_contract(const GemmArgs& g, hipStream_t stream);
// the 256x256 tile with the epilogues of the dense projections (bias / scale /
// sigmoid per column segment, SwiGLU, regrouped output): big_tile_mode names the
// kernel instance that can take `g`, or -1
int big_tile_mode(const GemmArgs& g);
int launch_big_tile(const GemmArgs& g, int mode, hipStream_t stream);
int launch_outer_mean(const GemmArgs& g, hipStream_t stream);
// the large-tile instance launch_gemm_nt hands `g` to, or -1: the kernel of gemm.hip
int gemm_big_tile_choice(const GemmArgs& g);

// ---------------------------------------------------------------- rowops.hip
// y = LN(x) [* weight + bias] ; then, if scale: y = sigmoid(scale[r]) * y + shift[r]
// with r = row % cond_rows (conditioning shared by the sample batch).
struct RowNormArgs {
  const void* x = nullptr;  // [rows][ldx] bf16 or fp32
  int x_f32 = 0;
  bf16_t* y = nullptr;      // [rows][ldy]
  int64_t rows = 0, ldx = 0, ldy = 0;
  int C = 0;
  const float* weight = nullptr;  // [C] or null
  const float* bias = nullptr;    // [C] or null
  const float* scale = nullptr;   // [cond_rows][ld_cond] pre-sigmoid, or null
  const float* shift = nullptr;
  int64_t cond_rows = 0, ld_cond = 0;
  // C <= 128: a second result of the same rows, y2 [rows][ldy] with scale2 / shift2 [cond_rows][ld_cond2]
  const float *scale2 = nullptr, *shift2 = nullptr;
  bf16_t* y2 = nullptr;
  int64_t ld_cond2 = 0;
  // C > 128: memory that the kernels behind this one will read (weights), brought nearer by workgroups of its own;
  // pieces of 128 bytes
  const void* warm[3] = {nullptr, nullptr, nullptr};
  uint32_t warm_lines[3] = {0, 0, 0};
  unsigned row_blocks = 0;  // set by launch_row_norm
  int samples = 1;  // set by launch_row_norm
  int param_vec = 0, cond_vec = 0;  // set by launch_row_norm: arrays aligned for 16-byte loads
};
int launch_row_norm(const RowNormArgs& a, hipStream_t stream);
// out[c][r] = in[r][c], bf16, rows and cols multiples of 8
// out[b][t][:] = sum over slots a, idx[t][a] >= 0, of relu(src[b][idx[t][a]][:]) / count[t]  (fp32 out, <= 32 slots)
int launch_gathered_relu_mean(const bf16_t* src, const int* idx, const float* count, float* out, int64_t batch,
                              int64_t n_src, int64_t n_out, int slots, int channels, hipStream_t stream);
// out[b][q][:] = cond[q][:] + w pos[b][rows[q]]  (3 coordinates -> channels; rows[q] < 0: cond only)
int launch_atom_position_features(const float* pos, const int* rows, const float* w, const float* cond, void* out,
                                  int out_f32, int64_t batch, int64_t n_slots, int64_t n_q, int channels,
                                  hipStream_t stream);
// out[b][q][:] = (rows[q] >= 0 ? src[b][rows[q]][:] : 0) + add[b][q][:]   (all bf16)
int launch_gather_rows_add(const bf16_t* src, const int* rows, const bf16_t* add, bf16_t* out, int64_t batch,
                           int64_t n_src, int64_t n_q, int channels, hipStream_t stream);
// out[b][t][0..2] = w LayerNorm(x[b][rows[t]]) * ln_w  (rows[t] < 0: zeros); channels = 128, fp32 out
int launch_ln_project3_gather(const bf16_t* x, const int* rows, const float* ln_w, const float* w, float* out,
                              int64_t batch, int64_t n_src, int64_t n_out, int channels, hipStream_t stream);
int launch_transpose(const bf16_t* in, bf16_t* out, int64_t rows, int64_t cols, hipStream_t stream);
// y[r][k] = softmax_k(x[r][k] + 1e9 (mask[k] - 1)) as bf16, x [rows][cols] fp32, y rows ldy apart (the tail zero)
int launch_softmax_rows(const float* x, const float* mask, bf16_t* y, int64_t rows, int cols, int64_t ldy,
                        hipStream_t stream);
// y[r][:] = (res ? res[r][:] : 0) + W relu?(x[r][:]), fp32, W [n_out][k], n_out 16 or 3, k % 4 == 0, k <= 128
int launch_narrow_linear_f32(const float* x, const float* w, const float* res, float* y, int64_t rows, int k, int n_out,
                             int relu_in, hipStream_t stream);
int launch_atom_pair_logits(const float* x, const float* ln_w, const float* w, float* out, int64_t n_groups, int64_t queries,
                            int64_t keys, int n_blocks, int n_head, int quad_major, hipStream_t stream);
int launch_atom_pair_cond(const float* row, const float* col, const float* tp, const int* tq, const int* tk, int n_tok,
                          const float* q_pos, const float* k_pos, const int* q_uid, const int* k_uid, const float* w_off,
                          const float* w_dist, const float* w_valid, const float* w1, const float* w2, const float* w3,
                          float* out, int64_t subsets, int queries, int keys, hipStream_t stream);

// -------------------------------------------------------------- pair_tile.hip
// Residual-stream tensors (`pair`, `out`, `x`) are bf16 or fp32 (io_f32).
// LayerNorm over fewer than 128 real channels: the tensor and the weights are zero-padded to 128 and the
// statistics are taken over `valid` channels (sums over all 128 are sums over the valid ones; the padded
// channels' share of the squared deviations, pad * mean^2, is taken out again).  valid = 128: pad = 0,
// the same arithmetic bit for bit.
struct LnWidth {
  float inv_c = 1.f / 128.f;  // 1 / valid channels
  float pad = 0.f;            // channels (128) - valid channels
};
inline LnWidth ln_width(int valid, int channels = 128) {
  LnWidth w;
  w.inv_c = 1.f / (float)valid;
  w.pad = (float)(channels - valid);
  return w;
}

struct TriMulArgs {
  LnWidth lw;
  int valid_c = 128;  // hidden channels 0 .. valid_c - 1 are real: the others are never contracted and count as zero
  const void* pair = nullptr;   // [N][N][128]
  const float* mask = nullptr;  // [N][N] 0/1 or null
  void* out = nullptr;          // [N][N][128]; may alias pair when residual
  int io_f32 = 0, N = 0, Np = 0, outgoing = 1, residual = 0;
  const float *ln_in_w = nullptr, *ln_in_b = nullptr, *ln_c_w = nullptr, *ln_c_b = nullptr;
  const bf16_t* w_pg = nullptr;   // [4][128][128]: per chunk 64 projection rows + 64 gate rows
  const bf16_t* w_gl = nullptr;   // [128][128] gating_linear
  const bf16_t* w_out = nullptr;  // [128][128] output_projection
  // channel-major planes [N][Np], `plane` elements apart (tri_plane: whole tiles of 128 positions)
  bf16_t *a_buf = nullptr, *b_buf = nullptr;  // 128 planes each: operands
  const bf16_t* t_buf = nullptr;              // 128 planes: contraction result
  int64_t plane = 0;
};
inline int64_t tri_plane(int64_t n) { return (n * ((n + 7) / 8 * 8) + 127) / 128 * 128; }
int launch_trimul_prologue(const TriMulArgs& a, hipStream_t s);
int launch_trimul_epilogue(const TriMulArgs& a, hipStream_t s);

struct AttnProjArgs {
  LnWidth lw;
  const void* pair = nullptr;  // [N][N][128]
  int io_f32 = 0, N = 0, transpose = 0;
  int skip_ln = 0;  // pair is already normalised
  const float *ln_w = nullptr, *ln_b = nullptr;
  const bf16_t* w_main = nullptr;  // [n_chunks][128][128]
  int n_chunks = 0, chunk_ops = 0; // SEG_* per chunk, 4 bits each
  float q_scale = 1.f;
  bf16_t* out_main = nullptr;      // [(b*N + s)][ld_main], chunk c at columns 128c..
  int64_t ld_main = 0;
  const bf16_t* w_bias = nullptr;  // [roundup(n_bias, 32)][128]
  int n_bias = 0;
  float* out_bias = nullptr;       // [n_bias][N][N] fp32, or
  int quads = 0;                   // out_bias is [n_bias][ceil(N / 4)][N][4], quads of keys outermost
  bf16_t* out_bias_bf16 = nullptr; // [n_bias][N][ld_bias] bf16 (values times bias_scale)
  int64_t ld_bias = 0;
  float bias_scale = 1.f;
};
int launch_attn_proj(const AttnProjArgs& a, hipStream_t s);

// pair_cond = Linear(LayerNorm([pair | relative encoding of the token pair])) without the concatenated
// tensor (pair_tile.hip).  The relative encoding has n_rel = 4 max_rel_idx + 2 max_rel_chain + 7 one-hot
// channels; g_hot[h][o] = ln_w[128 + h] * W[o][128 + h] and g_sum[o] = sum_h g_hot[h][o].
struct PairCondInitArgs {
  const void* pair = nullptr;  // [N][N][128], fp32 or bf16
  int io_f32 = 1, N = 0;
  float in_scale = 1.f;        // the pair values are multiplied by this first
  const int *asym_id = nullptr, *residue_index = nullptr, *token_index = nullptr, *entity_id = nullptr, *sym_id = nullptr;  // [N]
  int max_rel_idx = 32, max_rel_chain = 2, n_rel = 139;
  const float* ln_w = nullptr;     // [128] LayerNorm weights of the pair channels
  const bf16_t* w_pair = nullptr;  // [128][128] projection weights of the pair channels
  const float* g_hot = nullptr;    // [n_rel][128]
  const float* g_sum = nullptr;    // [128]
  float* out = nullptr;            // [N][N][128] fp32
};
int launch_pair_cond_init(const PairCondInitArgs& a, hipStream_t s);

struct AttnOutArgs {
  LnWidth lw;
  const bf16_t* og = nullptr;  // [(b*N + s)][ld_og] attention output, normalised, not yet gated
  int64_t ld_og = 0;
  const bf16_t* w_gate = nullptr;  // [128][128] gating_query: the gate is sigmoid(LN(pair) w_gate^T)
  const bf16_t* w_out = nullptr;   // [128][128]
  const void* pair = nullptr;      // gate input and residual source
  int skip_ln = 0;                 // pair is already normalised
  const float *ln_w = nullptr, *ln_b = nullptr;
  void* out = nullptr;
  int io_f32 = 0, N = 0, transpose = 0, residual = 0;
};
int launch_attn_out(const AttnOutArgs& a, hipStream_t s);

struct TransitionArgs {
  LnWidth lw;
  const void* x = nullptr;  // [N][128]
  void* out = nullptr;
  int io_f32 = 0, N = 0, hidden = 0, residual = 0;
  int rounded = 0;  // fp32 rows only: see ln_pixel8
  const float *ln_w = nullptr, *ln_b = nullptr;
  const bf16_t* w1 = nullptr;  // [hidden/64][128][128]: 64 a rows then 64 b rows per slab
  const bf16_t* w2 = nullptr;  // [128][hidden]
};
int launch_transition(const TransitionArgs& a, hipStream_t s);

// -------------------------------------------------------------- attention.hip
// q/k/v/g/out are addressed as base + batch * sb + position * ss + head * d.
struct FlashArgs {
  const bf16_t *q = nullptr, *k = nullptr, *v = nullptr, *g = nullptr;  // g: output gate or null
  int64_t q_sb = 0, q_ss = 0, k_sb = 0, k_ss = 0, v_sb = 0, v_ss = 0, g_sb = 0, g_ss = 0;
  void* out = nullptr;
  int out_f32 = 0;
  int64_t o_sb = 0, o_ss = 0;
  int B = 0, H = 0, Sq = 0, Sk = 0, d = 0;
  const float* bias = nullptr;  // [.][H][Sq][Sk], key stride 1
  int64_t bias_sb = 0, bias_sh = 0, bias_sq = 0;
  // bias_squad != 0: quads of four keys are the outer index, [.][H][Sk/4][Sq][4]:
  // key k of query q at q * bias_sq + (k / 4) * bias_squad + k % 4 with bias_sq = 4.
  // The lanes of a wave hold 32 consecutive queries, so a load of one quad per
  // lane is then one contiguous 512-byte run instead of 32 pieces of 16 bytes.
  int64_t bias_squad = 0;
  const float* key_mask = nullptr;  // [B][Sk] (km_sb may be 0): 0 -> logit replaced by -1e9
  int64_t km_sb = 0;
  const float *qpad = nullptr, *kpad = nullptr;  // [B][Sq], [B][Sk]: +1e9 where both are 0
  int64_t qp_sb = 0, kp_sb = 0;
  int bias_mod = 0;  // > 0: bias, qpad and kpad are indexed by batch % bias_mod
  // Gathered keys: key s of batch entry b is row key_rows[(b % bias_mod) * Sk + s]
  // of the K / V table of sample b / bias_mod (k_sb / v_sb: table stride); a
  // negative row is a key with zero K and V.  Null: key s is row s of batch b.
  const int* key_rows = nullptr;
  int64_t table_rows = 0;  // rows of a sample's table: every entry of key_rows is below this
  // window_kernel: the entries b % bias_mod that are asked for, their number first; the others' results are not written.  Null: all.
  const int* windows = nullptr;
  int per_xcd = 0, q_tiles = 0;  // (these and the magic numbers of their divisions by the launcher)
  unsigned magic_b = 0, magic_t = 0;
  int n_blocks = 0;  // workgroups that have work (set by the launcher; the grid is rounded up to a multiple of 8)
};
int launch_flash_attention(const FlashArgs& a, hipStream_t stream);

// ------------------------------------------- triattn.hip, triattn_core.hip
// Scratch of the triangle-attention fast path, in the frame of the (possibly
// transposed) operator, rows b:
//   q, k     bf16 [b][h][s][32]   (q times log2(e)/sqrt(32))
//   vt       bf16 [b][h][32][ldn] V transposed, ldn = N rounded up to 16, columns >= N zero,
//            key k of a row stored at column tri_vt_pos(k): inside every aligned group of 16
//            keys the two middle quads are swapped, which makes the 8 keys one lane feeds to
//            a P.V MFMA (k, k+1, k+2, k+3, k+8, ..., k+11 with k % 8 == 0 or 4) 16 contiguous bytes
//   bias     fp16, pair bias times log2(e) (clamped to the fp16 range), in MFMA-fragment order:
//            the attention core adds it to the scores on the matrix unit, S^T += I * bias^T with an
//            fp16 identity, and wants per (head, 32-query block, 64-key tile) the four B fragments
//            of that product as four contiguous 1 KB runs: run (k % 64) / 16, then [q % 32][k % 16].
//            fp16 rather than fp32: the bias is half of what the attention core pulls in from L2
//            per key tile, and that traffic is a sixth of its run time; fp16's 11 significant
//            bits put its rounding (2^-12 of a logit) below that of the bf16 probabilities (2^-9).
//            Entries whose key is >= N are zero; query rows >= N of the last block are unused.
__host__ __device__ inline int64_t tri_ldn(int64_t n) { return (n + 15) / 16 * 16; }
__host__ __device__ inline int tri_vt_pos(int k) { return (k & ~12) | ((k & 8) >> 1) | ((k & 4) << 1); }
__host__ __device__ inline int64_t tri_bias_qblocks(int64_t n) { return (n + 31) / 32; }
__host__ __device__ inline int64_t tri_bias_ktiles(int64_t n) { return (n + 63) / 64; }
__host__ __device__ inline int64_t tri_bias_elems(int64_t n, int64_t heads) {
  return heads * tri_bias_qblocks(n) * tri_bias_ktiles(n) * 2048;
}
__host__ __device__ inline int64_t tri_bias_offset(int64_t n, int h, int q, int k) {
  return ((((int64_t)h * tri_bias_qblocks(n) + (q >> 5)) * tri_bias_ktiles(n) + (k >> 6)) * 4 + ((k & 63) >> 4)) * 512 +
         (q & 31) * 16 + (k & 15);
}

struct TriAttnProjArgs {
  LnWidth lw;
  const void* pair = nullptr;  // [N][N][128]
  int io_f32 = 0, N = 0, transpose = 0, skip_ln = 0;
  const float *ln_w = nullptr, *ln_b = nullptr;
  const bf16_t* w_qkvg = nullptr;  // [4][128][128]: q, k, v chunks are used here (the gate chunk by attn_out)
  const bf16_t* w_bias = nullptr;  // [32][128], rows >= 4 zero
  int n_bias = 0;                  // 0 or 4
  float q_scale = 1.f, bias_scale = 1.f;
  bf16_t *q = nullptr, *k = nullptr, *vt = nullptr;
  uint16_t* bias = nullptr;  // fp16 bits, fragment order, tri_bias_elems(N, 4) elements
  int64_t ldn = 0;        // tri_ldn(N)
};
int launch_triattn_proj(const TriAttnProjArgs& a, hipStream_t stream);

struct TriAttnArgs {
  const bf16_t *q = nullptr, *k = nullptr, *vt = nullptr;
  const uint16_t* bias = nullptr;  // fp16 bits, fragment order (tri_bias_offset), or null
  const float* mask = nullptr;   // [N][N] 0/1 or null
  bf16_t* og = nullptr;          // [(b*N + s)][128] normalised attention output (the gate is applied by attn_out)
  int N = 0, head_dim = 32;      // head_dim 32 or 16: q, k [b][h][s][head_dim], vt [b][h][head_dim][ldn], og rows of 4 head_dim
  int64_t ldn = 0;
  int tile_blocks = 0, tile_extra = 0;  // (launch_triattn_flash) blocks of 32 queries per query tile, and how many tiles have one more
};
int launch_triattn_flash(const TriAttnArgs& a, hipStream_t stream);

// --------------------------------------------------------------- pair_step.hip
// One run of per-pixel operators between two long products (contraction, attention core), in place on `pair`.
enum {
  PAIR_STEP_FIRST,          // the outgoing prologue alone (64 channels)
  PAIR_STEP_INCOMING,       // outgoing epilogue, incoming prologue
  PAIR_STEP_PROJECT_START,  // incoming epilogue, starting-node projections
  PAIR_STEP_PROJECT_END,    // starting-node output, ending-node projections
  PAIR_STEP_LAST,           // ending-node output, transition (and pair logits)
  PAIR_STEP_NEXT,           // the same, and the outgoing prologue of the block that follows
};
inline int pair_step_max_hidden(int channels) { return channels == 128 ? 512 : 128; }  // hidden units of the transition
struct PairStepArgs {
  LnWidth lw;
  int channels = 128;  // of the pair tensor and the weights, 128 or 64
  int valid_c = 128, io_f32 = 0, N = 0, Np = 0, ldn = 0, hidden = 0, logit_heads = 0;
  int64_t plane = 0;
  void* pair = nullptr;
  // f_*: weights in fragment order (pair_frags of af3_pairformer_block)
  const float *ln1_w = nullptr, *ln1_b = nullptr;  // gate and output projection of the operator before
  const bf16_t *f_gate = nullptr, *f_out = nullptr;
  const float *ln_c_w = nullptr, *ln_c_b = nullptr;
  const bf16_t *t_buf = nullptr, *og = nullptr;
  const float *ln2_w = nullptr, *ln2_b = nullptr;  // transition
  const bf16_t *f_w1 = nullptr, *f_w2 = nullptr;
  const float *ln3_w = nullptr, *ln3_b = nullptr;  // prologue or projections of the operator behind
  const bf16_t *f_next = nullptr, *f_v = nullptr;  // f_next: projection and gate rows, or q and k;  f_v: v, then the pair-bias heads
  const float* mask = nullptr;                     // prologue
  bf16_t *a_buf = nullptr, *b_buf = nullptr;
  bf16_t *q = nullptr, *k = nullptr, *vt = nullptr;
  uint16_t* bias = nullptr;
  float q_scale = 1.f, bias_scale = 1.f;
  const float *sl_ln_w = nullptr, *sl_ln_b = nullptr;  // pair logits of the single track, or none
  const bf16_t* f_logits = nullptr;
  float* logits = nullptr;
};
int launch_pair_step(const PairStepArgs& a, int step, hipStream_t s);
// the long product of a triangle multiplication, between the planes of its prologue and its epilogue (api.hip)
int run_triangle_contraction(const bf16_t* a_buf, const bf16_t* b_buf, bf16_t* t_buf, int n, int valid_channels, int outgoing, hipStream_t s);

// --------------------------------------------------------------- atom_step.hip
// Tail: act [samples][atoms][128] += gate1 (y W_out^T), then += gate2 transition(LN(act)).  Head: the projections of the
// attention behind it, of act's two LayerNorms.  Gates and scale / shift per atom.
constexpr int ATOM_STEP_MAX_HIDDEN = 256;
struct AtomStepArgs {
  void* act = nullptr;
  int io_f32 = 0, atoms = 0, samples = 0, hidden = 0;
  const bf16_t* y = nullptr;                             // [samples][atoms][128]
  const bf16_t *f_out = nullptr, *f_w1 = nullptr, *f_w2 = nullptr;  // weights in fragment order
  const float *gate1 = nullptr, *gate2 = nullptr;        // [atoms][128]
  const float *scale = nullptr, *scale_q = nullptr;      // [atoms][ld_cond]: 128 scales (before their sigmoid), 128 shifts
  const float* scale_k = nullptr;                        // [atoms][ld_cond_k]
  int64_t ld_cond = 0, ld_cond_k = 0;
  const bf16_t* f_head = nullptr;                        // q, gate, k, v
  const float* q_bias = nullptr;                         // [128] or null
  float q_scale = 1.f;
  bf16_t *qg = nullptr, *kv = nullptr;                   // [samples][atoms][256]: q, gate;  k, v
  const int* tiles = nullptr;                            // the runs of 32 atoms that are asked for, their number first; null: all
};
bool atom_steps_apply(const AtomStepArgs& a);
int launch_atom_step(const AtomStepArgs& a, bool tail, bool head, hipStream_t s);

// -------------------------------------------------------------- single_step.hip
// LayerNorm of rows of 384 channels and a product of them, w row-major [N][384]: out[row][..] = queries (bias, scale), keys, values,
// gate (sigmoid), N = 4 x 384, or with swiglu N / 2 hidden units (w in blocks of 32 + 32 rows).
constexpr int SINGLE_STEP_CHANNELS = 384, SINGLE_STEP_ROWS = 400;
struct SingleStepArgs {
  const void* x = nullptr;  // [rows][384]
  int io_f32 = 0, rows = 0, N = 0, swiglu = 0;
  const float *ln_w = nullptr, *ln_b = nullptr;
  const bf16_t* w = nullptr;
  const float* q_bias = nullptr;  // [384] or null
  float q_scale = 1.f;
  bf16_t* out = nullptr;  // [rows][ldc]
  int64_t ldc = 0;
};
bool single_step_applies(const SingleStepArgs& a);
int launch_single_step(const SingleStepArgs& a, hipStream_t s);

// ----------------------------------------------------------- atom_aggregate.hip
// out[b][t] = sum over slots s, idx[t][s] >= 0, of relu(bf16(x[b][idx[t][s]] w^T)) / count[t]; 128 channels to 768, w in fragment order
struct AtomAggregateArgs {
  const bf16_t* x = nullptr;   // [batch][n_src][128]
  const int* idx = nullptr;    // [tokens][slots], below n_src; at most 32 slots
  const float* count = nullptr;
  const bf16_t* w = nullptr;
  float* out = nullptr;        // [batch][tokens][768]
  int64_t n_src = 0;
  int batch = 0, tokens = 0, slots = 0;
};
int launch_atom_aggregate(const AtomAggregateArgs& a, hipStream_t s);

// ----------------------------------------------------------- row_transition.hip
// act += (silu(a) b) w2^T, (a, b) = LayerNorm(act) w1^T, rows of 384 fp32; w1 (rows in blocks of 32 of a and 32 of b) and w2
// [384][hidden] in fragment order, bits 2 and 3 of a row number exchanged; hidden a multiple of 128
constexpr int ROW_TRANSITION_CHANNELS = 384;
struct RowTransitionArgs {
  float* act = nullptr;  // [rows][384]
  const float *ln_w = nullptr, *ln_b = nullptr;
  const bf16_t *w1 = nullptr, *w2 = nullptr;
  int rows = 0, hidden = 0;
};
int launch_row_transition(const RowTransitionArgs& a, hipStream_t s);

// --------------------------------------------------------------- token_step.hip
// Adaptive LayerNorm of rows of 768 channels and a product of them: with w in fragment order, [N][768], out[row][n0 ..] =
// queries (bias, scale), keys, values, gate (sigmoid), N = 4 x 768, or with swiglu N / 2 hidden units (w in blocks of 64 rows).
// Row s tokens + t is token t of sample s; its conditioning is row t.
constexpr int TOKEN_STEP_CHANNELS = 768;
struct NormProductArgs {
  unsigned work_blocks = 0, magic_tiles = 0;  // (these by launch_norm_product)
  int per_xcd = 0, total = 0, tiles = 0, tile_tokens = 0, magic_samples = 0;
  int samples = 0, tokens = 0, N = 0, swiglu = 0;
  int ld_cond = 0;
  const bf16_t* x = nullptr;     // [samples][tokens][768]
  const float* scale = nullptr;  // [tokens][ld_cond]: 768 scales (before their sigmoid), 768 shifts
  const bf16_t* w = nullptr;
  int64_t ldc = 0;
  const float* q_bias = nullptr;  // [768] or null
  float q_scale = 1.f;
  bf16_t* out = nullptr;  // [samples][tokens][ldc]
  const void* warm[3] = {nullptr, nullptr, nullptr};  // as RowNormArgs
  uint32_t warm_lines[3] = {0, 0, 0};
};
// act = (y w^T) gate + act in place: 768 columns, K = 768 or 1536, w in fragment order; gate row: row % cond_rows
struct GatedProductArgs {
  int per_xcd = 0, total = 0, tiles = 0;  // (these and the magic numbers by launch_gated_product)
  unsigned magic_tiles = 0, magic_cond = 0;
  int rows = 0, K = 0, cond_rows = 0;
  const bf16_t *y = nullptr, *w = nullptr;  // [rows][K], [768][K]
  bf16_t* act = nullptr;                    // [rows][768]
  const float* gate = nullptr;              // [cond_rows][ld_gate]
  int64_t ld_gate = 0;
};
// The products of the token transformer's blocks over any number of rows, [rows][K], w in fragment order: with `gate` into `out`
// as above; N = 4 x 768 columns of queries (bias, scale), keys, values, gate (sigmoid), K = 768; or with swiglu N / 2 hidden units.
struct RowsProductArgs {
  int m_chunk = 0, n_chunk = 0, xcd_m = 0, xcd_shift = 0;  // (these and the magic numbers by launch_rows_product)
  unsigned magic_chunk = 0, magic_cond = 0;
  int rows = 0, N = 0, K = 0, swiglu = 0, cond_rows = 0;
  const bf16_t *x = nullptr, *w = nullptr;
  bf16_t* out = nullptr;
  int64_t ldc = 0;
  const float* q_bias = nullptr;
  float q_scale = 1.f;
  const float* gate = nullptr;
  int64_t ld_gate = 0;
};
bool rows_product_applies(const RowsProductArgs& a);
int launch_rows_product(const RowsProductArgs& a, hipStream_t s);
bool gated_product_applies(const GatedProductArgs& a);
int launch_gated_product(const GatedProductArgs& a, hipStream_t s);
bool norm_product_applies(const NormProductArgs& a);
int launch_norm_product(const NormProductArgs& a, hipStream_t s);

// -------------------------------------------------------------------- embed.hip
struct PairEmbedArgs {
  const float* lr = nullptr;    // [n][ld_lr]: left projection, then right
  int64_t ld_lr = 0;
  const float* prev = nullptr;  // [n][n][128]
  const int64_t *asym_id = nullptr, *residue_index = nullptr, *token_index = nullptr, *entity_id = nullptr, *sym_id = nullptr;
  const float* w_pos = nullptr;    // [139][128]
  const float* w_bond = nullptr;   // [128]
  const float* contact = nullptr;  // [n][n]
  void* out = nullptr;             // [n][n][128]
  int out_f32 = 0, n = 0;
};
int launch_pair_embed(const PairEmbedArgs& a, hipStream_t s);
int launch_contacts(const int64_t* idx0, const uint8_t* ok0, int n0, const int64_t* idx1, const uint8_t* ok1, int n1, float* contact,
                    int n, hipStream_t s);
int launch_add_rows(const float* a, const float* b, int64_t ld_b, int64_t mod, void* out, int out_f32, int64_t rows, int channels,
                    hipStream_t s);
int launch_mask_rows(bf16_t* x, const float* mask, int64_t mod, int64_t rows, int channels, hipStream_t s);
struct AtomEmbedArgs {
  const float *positions = nullptr, *mask = nullptr, *charge = nullptr;  // [atoms][3], [atoms], [atoms]
  const int64_t *element = nullptr, *chars = nullptr;                    // [atoms] below 128, [atoms][4] below 64
  // [channels][3], [channels], [channels][128], [channels], [channels][4 * 64]
  const float *w_pos = nullptr, *w_mask = nullptr, *w_element = nullptr, *w_charge = nullptr, *w_chars = nullptr;
  float* out = nullptr;  // [atoms][channels]
  int64_t atoms = 0;
  int channels = 0;
};
int launch_atom_embed(const AtomEmbedArgs& a, hipStream_t s);
// windows of an atom layout that somebody reads (af3_atom_windows_forward)
struct AtomWindowsArgs {
  const float* mask = nullptr;             // [windows][queries]
  const int64_t* back_idx = nullptr;       // [slots] into the windows' rows
  const uint8_t* back_exists = nullptr;    // [slots]
  int64_t slots = 0;
  const int32_t* key_rows = nullptr;       // [windows][keys], negative: none
  int windows = 0, queries = 0, keys = 0;
  int32_t* out = nullptr;                  // [1 + windows]
};
bool atom_windows_apply(const AtomWindowsArgs& a);
int launch_atom_windows(const AtomWindowsArgs& a, hipStream_t s);
struct GatherAtomsArgs {
  const int64_t *idx = nullptr, *add_idx = nullptr, *uid = nullptr;  // [rows], [rows], [uids]
  const uint8_t *exists = nullptr, *add_exists = nullptr;            // [rows]
  const float *cond = nullptr, *add = nullptr;                       // [slots][channels]; [add_rows][channels] or null
  const float *mask = nullptr, *pos = nullptr;                       // [slots], [slots][3]
  float *out_cond = nullptr, *out_mask = nullptr, *out_pos = nullptr;
  int* out_uid = nullptr;
  int64_t rows = 0, slots = 0, add_rows = 0, uids = 0;
  int channels = 0;
};
int launch_gather_atoms(const GatherAtomsArgs& a, hipStream_t s);
enum { POS_SCALE = 0, POS_BLEND = 1, POS_PLACE = 2, POS_STEP = 3 };
int launch_augment_positions(const float* x, const float* rot, const float* shift, const float* mask, const float* noise, float* out,
                             int64_t samples, int64_t atoms, hipStream_t s);
int launch_positions(int op, const float* x, const float* y, const float* mask, const float* level, const float* other, float f,
                     float* out, int64_t samples, int64_t atoms, hipStream_t s);

// ---------------------------------------------------------------------- msa.hip
struct MsaProjectArgs {
  const void* msa = nullptr;  // [rows][n][64]
  int io_f32 = 0, rows = 0, n = 0;
  const float *ln_w = nullptr, *ln_b = nullptr;
  const bf16_t* w = nullptr;      // [64][64]
  const float* mask = nullptr;    // [rows][n]; not for values
  bf16_t* out[2] = {nullptr, nullptr};
  int64_t ld = 0;                 // rows (values: n) rounded up to 8
};
int launch_msa_project(const MsaProjectArgs& a, bool values, hipStream_t s);

struct MsaUpdateArgs {
  const void* msa = nullptr;  // [rows][n][64]
  void* out = nullptr;        // may be msa
  int io_f32 = 0, rows = 0, n = 0, residual = 0;
  const bf16_t* avg = nullptr;  // [8][n][rows][8], or null: no attention part
  const float *att_ln_w = nullptr, *att_ln_b = nullptr;
  const bf16_t *w_g = nullptr, *w_o = nullptr;  // [64][64]
  const float *tr_ln_w = nullptr, *tr_ln_b = nullptr;
  const bf16_t* w1 = nullptr;   // [2 hidden][64], the silu half first, or null: no transition
  const bf16_t* w2 = nullptr;   // [64][hidden]
  int hidden = 0;               // a multiple of 32, at most 256
};
int launch_msa_update(const MsaUpdateArgs& a, hipStream_t s);
int launch_msa_coverage(const float* mask, int rows, int n, float eps, float* inv, float* live, hipStream_t s);
int launch_transpose_f32(const float* in, float* out, int n, hipStream_t s);  // [n][n]

// --------------------------------------------------------------- check_f32.hip
struct CkGemmArgs {
  const float* A = nullptr;  // element (b, m, k) at A[b*sA + m*lda + k*ka]
  const float* B = nullptr;  // element (b, n, k) at B[b*sB + n*ldb + k*kb]
  float* C = nullptr;        // element (b, m, n) at C[b*sC + m*ldc + n]
  int M = 0, N = 0, K = 0, batch = 1;
  int64_t lda = 0, ka = 1, ldb = 0, kb = 1, ldc = 0, sA = 0, sB = 0, sC = 0;
  const float* bias = nullptr;  // y = sigmoid?((acc + bias) * alpha) * mul + add
  float alpha = 1.f;
  int sigmoid = 0;
  const float* mul = nullptr;   // [mul_rows][ld_mul], row m % mul_rows
  int64_t mul_rows = 0, ld_mul = 0;
  const float* add = nullptr;   // [b*s_add + m*ld_add + n]
  int64_t ld_add = 0, s_add = 0;
};
int launch_ck_gemm(const CkGemmArgs& g, hipStream_t s);

struct CkNormArgs {
  const float* x = nullptr;
  float* y = nullptr;
  int64_t rows = 0;
  int C = 0;
  const float *weight = nullptr, *bias = nullptr, *scale = nullptr, *shift = nullptr;
  int64_t cond_rows = 0, ld_cond = 0;
};
int launch_ck_norm(const CkNormArgs& a, hipStream_t s);

enum { CK_TRIMUL_SPLIT = 0, CK_CHAN_TO_PIX = 1, CK_TRANSPOSE_PIX = 2, CK_SWIGLU = 3, CK_BINARY = 4 };
int launch_ck_elementwise(int op, const float* x0, const float* x1, const float* x2, float* y0, float* y1,
                          int64_t n0, int64_t n1, int flag, hipStream_t s);

struct CkAttnArgs {
  const float *q = nullptr, *k = nullptr, *v = nullptr;  // base + batch*sb + pos*ss + head*d
  float* out = nullptr;
  int64_t q_sb = 0, q_ss = 0, k_sb = 0, k_ss = 0, v_sb = 0, v_ss = 0, o_sb = 0, o_ss = 0;
  int B = 0, H = 0, Sq = 0, Sk = 0, d = 0;
  const float* bias = nullptr;  // bias[bb*bias_sb + h*bias_sh + q*bias_sq + k*bias_sk]
  int64_t bias_sb = 0, bias_sh = 0, bias_sq = 0, bias_sk = 1;
  int bias_mod = 0;             // bb = b % bias_mod when > 0 (also indexes qpad / kpad)
  const float* key_mask = nullptr;  // [.][Sk], batch stride km_sb: 0 -> logit replaced by -1e9
  int64_t km_sb = 0;
  const float *qpad = nullptr, *kpad = nullptr;  // [.][Sq], [.][Sk]: +1e9 where both are 0
};
int launch_ck_attention(const CkAttnArgs& a, hipStream_t s);
