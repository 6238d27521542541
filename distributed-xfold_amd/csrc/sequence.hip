// Whole-module entry points: the launches of a run of blocks, enqueued in one call.  Host code only; a step is one of the
// library's own entry points with the arguments a caller would give it, or one kernel for several of them (pair_step.hip,
// atom_step.hip, the Evoformer's msa.hip).
//
// Why it exists: a launch costs 2.7 to 3.7 us of host time from C (by machine, back to back), and about 11 us through
// the Python operator layer (argument checks, tensor allocation, ctypes).  Up to a few hundred tokens the kernels
// themselves take 4 to 10 us, so that the operator layer, not the GPU, set the pace of a block.
#include "../../include/af3_hip.h"
#include "kernels.h"

namespace {

inline size_t align_up(size_t v) { return (v + 255) / 256 * 256; }
inline int64_t up8(int64_t v) { return (v + 7) / 8 * 8; }

// bump allocator over the caller's workspace
struct Carver {
  char* base;
  size_t size, used = 0;
  bool ok = true;
  Carver(void* p, size_t n) : base(static_cast<char*>(p)), size(n) {}
  void* take(size_t bytes) {
    bytes = align_up(bytes);
    if (!base || used + bytes > size) { ok = false; return nullptr; }
    void* r = base + used;
    used += bytes;
    return r;
  }
};

// `waiter` waits for everything enqueued on `on` so far.  An event may be recorded again while waits for its earlier
// recordings are pending, and be destroyed after that: the runtime keeps what a pending wait needs.  (Creating and
// destroying one costs the host as much as a launch: once a call, not once a block.)
struct Event {
  hipEvent_t e = nullptr;
  ~Event() {
    if (e) (void)hipEventDestroy(e);
  }
  int record(hipStream_t on) {
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return AF3_ERR_LAUNCH;
    return hipEventRecord(e, on) == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH;
  }
  int wait(hipStream_t waiter) { return !e || hipStreamWaitEvent(waiter, e, 0) == hipSuccess ? AF3_OK : AF3_ERR_LAUNCH; }
  int order(hipStream_t on, hipStream_t waiter) {
    const int rc = record(on);
    return rc != AF3_OK ? rc : wait(waiter);
  }
};

#define STEP(call)               \
  do {                           \
    const int rc_ = (call);      \
    if (rc_ != AF3_OK) return rc_; \
  } while (0)

// ---- the pair operators in steps: a run of them between two long products in one kernel (pair_step.hip) ----
// Few tokens: a step takes the chain of one tile of 32 or 64 positions where a kernel of its own per operator takes several of
// tiles of 128, and eight launches a block take the place of thirteen.  Many tokens: a step saves the passes over the tensor that
// its operators would make one by one, at the price of the weights, which every tile fetches anew; on an fp32 stream, whose passes
// are twice the bytes, that pays for much longer.  us, kernels per operator (up to 400 tokens with the two steps that end in
// projections) / steps: a stack of 4 blocks on a bf16 stream, one block on it, a stack of 4 on an fp32 stream
//   209 tokens   948 / 897     288 / 277    1003 / 945
//   301         1513 / 1452    431 / 419    1683 / 1560
//   387         2518 / 2456    691 / 675    2817 / 2654
//   512         3971 / 3914   1020 / 1033   4777 / 4333
//   550         5298 / 5204   1361 / 1352   5990 / 5689
//   600         6160 / 6233   1599 / 1609   7035 / 6789
//   768         9686 / 9771   2469 / 2505  11183 / 10607;  3 blocks: 1024 19673 / 18762, 1280 33765 / 32302, 1536 52463 / 52510
// Pair tensors of 64 channels have no other kernels (64 / 301 / 768 / 2048 tokens, bf16, a block on its own: 100 -> 46,
// 345 -> 221, 1940 -> 1460, 22400 -> 18800 against one zero-padded to 128; their 32-bit offsets end at 3072).
// The bf16 line lies below 512 tokens, the first size at which one of the two is behind (a block on its own, by 1 %); 550 is ahead
// once more, by 1 to 2 %, 600 behind.
constexpr int64_t BF16_STEP_POSITIONS = 500 * 500, F32_STEP_POSITIONS = 1280 * 1280;
// The outgoing epilogue and the incoming prologue are one step while its patches are one round of workgroups: it stores transposed
// operands 8 or 16 bytes at a time, which costs more than the pass and the launch it saves beyond (a stack of 4 blocks, us, two
// kernels / one: 128 tokens 495 / 474, 176 673 / 653, 192 735 / 742, 256 1036 / 1064, 387 2456 / 2535; fp32 stream 176 712 / 687).
constexpr int64_t INCOMING_STEP_POSITIONS = 184 * 184;
bool pair_steps_apply(const af3_pairformer_block& b, int64_t n, int dt) {
  const int c = b.pair_channels == 64 ? 64 : 128;
  return b.pair_frags && n <= 8192 &&
         (c == 64 ? n <= AF3_PAIR64_MAX_TOKENS : n * tri_ldn(n) <= (dt == AF3_F32 ? F32_STEP_POSITIONS : BF16_STEP_POSITIONS)) &&
         b.num_head_pair == 4 && b.valid_channels >= 8 && b.valid_channels <= c && b.valid_channels % 4 == 0 &&
         (c == 128 || b.valid_channels == 64) && b.pair_hidden > 0 && b.pair_hidden % 64 == 0 &&
         b.pair_hidden <= pair_step_max_hidden(c);
}
// Scratch.  q, k and the operands of the contraction are never alive together, nor are its result and the attention's.
struct PairStepScratch {
  bf16_t *qa = nullptr, *kb = nullptr, *vt = nullptr, *ogt = nullptr;
  uint16_t* bias = nullptr;
  static size_t plane_bytes(int64_t n, int c) { return (size_t)c * tri_plane(n) * 2; }  // (tri_plane(n) >= n n)
  static size_t vt_bytes(int64_t n, int c) { return (size_t)n * c * tri_ldn(n) * 2; }
  static size_t bytes(int64_t n, int c) {
    return 3 * align_up(plane_bytes(n, c)) + align_up(vt_bytes(n, c)) + align_up((size_t)tri_bias_elems(n, 4) * 2) +
           (c == 128 && n * tri_ldn(n) <= LOGIT_RING_POSITIONS ? LOGIT_RING * logit_bytes(n, 16) : 0);
  }
  // Pair logits of the last blocks, where the single track runs on a stream of its own.  With two buffers every block waits
  // for the attention two blocks back, and an event costs the host some 20 us (recorded 3, waited for 15 to 17), where a launch
  // costs 2.7 to 3.7: at 64 tokens the launches set the pace.  With eight it is one wait in four blocks (runs of 4 blocks, us a
  // block: 93 -> 83).
  static constexpr int LOGIT_RING = 8;
  static constexpr int64_t LOGIT_RING_POSITIONS = 208 * 208;  // (beyond, the kernels set the pace)
  static size_t logit_bytes(int64_t n, int heads) { return align_up((size_t)heads * n * ((n + 3) / 4 * 4) * 4); }
  float* ring(int64_t n) const {
    return reinterpret_cast<float*>(reinterpret_cast<char*>(bias) + align_up((size_t)tri_bias_elems(n, 4) * 2));
  }
  bool carve(int64_t n, int c, void* ws, size_t wsb) {
    Carver w(ws, wsb);
    qa = static_cast<bf16_t*>(w.take(plane_bytes(n, c)));
    kb = static_cast<bf16_t*>(w.take(plane_bytes(n, c)));
    ogt = static_cast<bf16_t*>(w.take(plane_bytes(n, c)));
    vt = static_cast<bf16_t*>(w.take(vt_bytes(n, c)));
    bias = static_cast<uint16_t*>(w.take((size_t)tri_bias_elems(n, 4) * 2));
    return w.ok;
  }
};

// One block's pair operators.  `first`: no step before has made the outgoing prologue.  `next`: the block whose outgoing prologue
// the last step makes, or null.
// `logits`: where the pair logits of the single track go, or null; they are written behind `logits_free`.
int pair_operators_in_steps(const af3_pairformer_block& b, const af3_pairformer_block* next, bool first, void* pair, int dt,
                            const float* mask, const float* mask_in, int64_t n, void* ws, size_t wsb, float* logits,
                            Event* logits_free, hipStream_t s) {
  if (!pair || (dt != AF3_F32 && dt != AF3_BF16) || ((uintptr_t)pair & 15) || ((uintptr_t)mask & 15) || ((uintptr_t)mask_in & 15))
    return AF3_ERR_BAD_ARG;
  PairStepScratch w;
  const int c = b.valid_channels, hidden = b.pair_hidden, wide = b.pair_channels == 64 ? 64 : 128;
  if (!w.carve(n, wide, ws, wsb)) return AF3_ERR_WORKSPACE;
  PairStepArgs a;
  a.channels = wide;
  a.lw = ln_width(c, wide);
  a.valid_c = c; a.io_f32 = dt == AF3_F32; a.N = (int)n; a.Np = (int)up8(n); a.ldn = (int)tri_ldn(n); a.plane = tri_plane(n);
  a.pair = pair; a.hidden = hidden;
  a.t_buf = a.og = w.ogt; a.a_buf = a.q = w.qa; a.b_buf = a.k = w.kb; a.vt = w.vt; a.bias = w.bias;
  a.bias_scale = 1.4426950408889634f;  // base-2 logits, as grid_self_attn_impl
  a.q_scale = a.bias_scale / sqrtf((float)(c / 4));
  // pair_frags, in rows of 128 (64)
  auto qkg = [&](int d, int mat) { return b.pair_frags + (d * 3 + mat) * wide * wide; };
  auto tm = [&](const af3_pairformer_block& x, int d, int mat) { return x.pair_frags + (6 + d * 6 + mat) * wide * wide; };
  auto ta = [&](int d, int row) { return b.pair_frags + (18 * wide + d * (2 * wide + 32) + row) * wide; };
  const uint16_t* const w1 = b.pair_frags + (22 * wide + 64) * wide;
  const int logit_rows = b.with_single ? (b.num_head + 31) / 32 * 32 : 0;
  TriAttnArgs core;
  core.q = w.qa; core.k = w.kb; core.vt = w.vt; core.bias = w.bias; core.mask = mask; core.og = w.ogt; core.N = (int)n; core.ldn = a.ldn;
  core.head_dim = wide / 4;

  auto product = [&](int d) {  // a triangle multiplication's prologue or epilogue as a kernel of its own
    TriMulArgs p;
    p.lw = a.lw; p.valid_c = c; p.pair = p.out = pair; p.mask = d == 1 && mask_in ? mask_in : mask; p.io_f32 = a.io_f32;
    p.N = a.N; p.Np = a.Np; p.plane = a.plane; p.outgoing = d == 0; p.residual = 1;
    p.ln_in_w = b.tm_ln_in_w[d]; p.ln_in_b = b.tm_ln_in_b[d]; p.ln_c_w = b.tm_ln_c_w[d]; p.ln_c_b = b.tm_ln_c_b[d];
    p.w_pg = b.tm_w_proj_gate[d]; p.w_gl = b.tm_w_gating[d]; p.w_out = b.tm_w_out[d];
    p.a_buf = w.qa; p.b_buf = w.kb; p.t_buf = w.ogt;
    return p;
  };
  if (first && wide == 64) {
    a.ln3_w = b.tm_ln_in_w[0]; a.ln3_b = b.tm_ln_in_b[0]; a.f_next = tm(b, 0, 2); a.mask = mask;
    STEP(launch_pair_step(a, PAIR_STEP_FIRST, s));
  } else if (first) {
    STEP(launch_trimul_prologue(product(0), s));
  }
  for (int d = 0; d < 2; ++d) {
    STEP(run_triangle_contraction(w.qa, w.kb, w.ogt, (int)n, c, d == 0, s));
    a.ln1_w = b.tm_ln_in_w[d]; a.ln1_b = b.tm_ln_in_b[d]; a.f_gate = tm(b, d, 0); a.f_out = tm(b, d, 1);
    a.ln_c_w = b.tm_ln_c_w[d]; a.ln_c_b = b.tm_ln_c_b[d];
    if (d == 0 && wide == 128 && n * tri_ldn(n) > INCOMING_STEP_POSITIONS) {
      STEP(launch_trimul_epilogue(product(0), s));
      STEP(launch_trimul_prologue(product(1), s));
    } else if (d == 0) {
      a.ln3_w = b.tm_ln_in_w[1]; a.ln3_b = b.tm_ln_in_b[1]; a.f_next = tm(b, 1, 2); a.mask = mask_in ? mask_in : mask;
      STEP(launch_pair_step(a, PAIR_STEP_INCOMING, s));
    } else {
      a.ln3_w = b.ta_ln_w[0]; a.ln3_b = b.ta_ln_b[0]; a.f_next = qkg(0, 0); a.f_v = ta(0, 0);
      STEP(launch_pair_step(a, PAIR_STEP_PROJECT_START, s));
    }
  }
  STEP(launch_triattn_flash(core, s));
  a.ln1_w = b.ta_ln_w[0]; a.ln1_b = b.ta_ln_b[0]; a.f_gate = qkg(0, 2); a.f_out = ta(0, wide + 32);
  a.ln3_w = b.ta_ln_w[1]; a.ln3_b = b.ta_ln_b[1]; a.f_next = qkg(1, 0); a.f_v = ta(1, 0);
  STEP(launch_pair_step(a, PAIR_STEP_PROJECT_END, s));
  STEP(launch_triattn_flash(core, s));
  a.ln1_w = b.ta_ln_w[1]; a.ln1_b = b.ta_ln_b[1]; a.f_gate = qkg(1, 2); a.f_out = ta(1, wide + 32);
  a.ln2_w = b.pt_ln_w; a.ln2_b = b.pt_ln_b; a.f_w1 = w1; a.f_w2 = w1 + (2 * hidden + logit_rows) * wide;
  if (logits) {
    a.sl_ln_w = b.sl_ln_w; a.sl_ln_b = b.sl_ln_b; a.f_logits = w1 + 2 * hidden * wide; a.logit_heads = b.num_head; a.logits = logits;
    if (logits_free) STEP(logits_free->wait(s));
  }
  if (!next) return launch_pair_step(a, PAIR_STEP_LAST, s);
  a.ln3_w = next->tm_ln_in_w[0]; a.ln3_b = next->tm_ln_in_b[0]; a.f_next = tm(*next, 0, 2); a.mask = mask;
  return launch_pair_step(a, PAIR_STEP_NEXT, s);
}

// one block by itself
int pair_operators(const af3_pairformer_block& b, void* pair, int dt, const float* mask, const float* mask_in, int64_t n,
                   void* ws, size_t wsb, hipStream_t s) {
  if (pair_steps_apply(b, n, dt))
    return pair_operators_in_steps(b, nullptr, true, pair, dt, mask, mask_in, n, ws, wsb, nullptr, nullptr, s);
  for (int d = 0; d < 2; ++d)
    STEP(af3_triangle_multiplication_forward_padded(pair, dt, d == 1 && mask_in ? mask_in : mask, d, b.tm_ln_in_w[d], b.tm_ln_in_b[d],
                                                    b.tm_w_proj_gate[d], b.tm_ln_c_w[d], b.tm_ln_c_b[d], b.tm_w_out[d],
                                                    b.tm_w_gating[d], pair, 1, n, b.valid_channels, ws, wsb, s));
  for (int d = 0; d < 2; ++d)
    STEP(af3_grid_self_attn_forward_padded(pair, dt, mask, d, b.ta_ln_w[d], b.ta_ln_b[d], b.ta_w_bias[d], nullptr,
                                           b.ta_w_qkvg[d], b.ta_w_out[d], b.num_head_pair, pair, 1, n, b.valid_channels, ws,
                                           wsb, s));
  return af3_transition_forward_padded(pair, dt, b.pt_ln_w, b.pt_ln_b, b.pt_w1, b.pt_w2, b.pair_hidden, pair, 1, n * n,
                                       b.valid_channels, s);
}

int single_update(const af3_pairformer_block& b, void* single, int dt, const float* mask, const float* logits, int64_t n,
                  void* ws, size_t wsb, af3_stream_t s) {
  const int c = b.c_single, h = b.single_hidden;
  Carver w(ws, wsb);
  uint16_t* x = static_cast<uint16_t*>(w.take((size_t)n * c * 2));
  uint16_t* y = static_cast<uint16_t*>(w.take((size_t)n * (c > h ? c : h) * 2));
  const size_t ab = af3_batch_diffusion_self_attention_workspace_bytes(1, n, c);
  void* aw = w.take(ab);
  if (!w.ok) return AF3_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(s);
  // The products here are a few hundred rows: their K range may be split between waves (nothing compares one
  // sequence's bits with a batch's).
  auto product = [&](const uint16_t* in, const uint16_t* wt, void* out, int out_dt, int n_out, int k, int mode, const void* res) {
    return run_linear(in, wt, nullptr, out, out_dt, n, n_out, k, mode, 1.f, 0, nullptr, 0, 0, res, dt, 1, st);
  };
  // Up to SINGLE_STEP_ROWS rows either norm and the product behind it are one kernel.
  const int d = b.num_head > 0 && c % b.num_head == 0 ? c / b.num_head : 0;
  bf16_t* const qkvg = self_projections(aw, ab, n, c);
  SingleStepArgs in, hidden;
  in.x = hidden.x = single; in.io_f32 = hidden.io_f32 = dt == AF3_F32; in.rows = hidden.rows = n <= SINGLE_STEP_ROWS ? (int)n : 0;
  in.ln_w = b.sa_ln_w; in.ln_b = b.sa_ln_b; in.w = b.sa_w_qkvg; in.N = 4 * c; in.ldc = 4 * c; in.out = qkvg;
  in.q_bias = b.sa_q_b; in.q_scale = 1.0f / sqrtf((float)d);
  hidden.ln_w = b.st_ln_w; hidden.ln_b = b.st_ln_b; hidden.w = b.st_w1; hidden.N = 2 * h; hidden.swiglu = 1; hidden.ldc = h; hidden.out = y;
  const bool steps = c == SINGLE_STEP_CHANNELS && (dt == AF3_F32 || dt == AF3_BF16) && (d == 16 || d == 24 || d == 32 || d == 48) &&
                     single_step_applies(in) && single_step_applies(hidden);
  if (steps) {
    STEP(launch_single_step(in, st));
    STEP(run_self_attend(qkvg, mask, 1, logits, 1, b.num_head, y, AF3_BF16, 1, n, c, st));
  } else {
    STEP(af3_layer_norm_forward(single, dt, x, n, c, b.sa_ln_w, b.sa_ln_b, nullptr, nullptr, 0, 0, s));
    STEP(run_self_attention(x, mask, 1, logits, 1, b.sa_w_qkvg, b.sa_q_b, b.num_head, y, AF3_BF16, 1, n, c, aw, ab, 1, st));
  }
  STEP(product(y, b.sa_w_out, single, dt, c, c, AF3_LINEAR_GATE_RES, single));
  if (steps) {
    STEP(launch_single_step(hidden, st));
  } else {
    STEP(af3_layer_norm_forward(single, dt, x, n, c, b.st_ln_w, b.st_ln_b, nullptr, nullptr, 0, 0, s));
    STEP(product(x, b.st_w1, y, AF3_BF16, 2 * h, c, AF3_LINEAR_SWIGLU, nullptr));
  }
  return product(y, b.st_w2, single, dt, c, h, AF3_LINEAR_GATE_RES, single);
}

inline bool msa_size_ok(int64_t rows, int64_t n) { return rows > 0 && n > 0 && n <= 8192 && rows <= (1ll << 30) / n; }

size_t opm_bytes(int64_t rows, int64_t n) {
  return 2 * align_up((size_t)n * 32 * up8(rows) * 2);
}
size_t msa_attention_bytes(int64_t rows, int64_t n) {
  return align_up((size_t)8 * n * n * 4) + align_up((size_t)8 * n * up8(n) * 2) + align_up((size_t)64 * rows * up8(n) * 2) +
         align_up((size_t)64 * rows * n * 2);
}
size_t msa_mask_bytes(int64_t n) { return align_up((size_t)n * n * 4) + align_up((size_t)n * 4); }

// pair (+)= (outer product W + b) / (eps + coverage)
int outer_product_mean(const af3_msa_block& b, const void* msa, int msa_dt, const float* msa_mask, const float* inv, void* pair,
                       int pair_dt, int residual, int64_t rows, int64_t n, Carver w, hipStream_t s) {
  MsaProjectArgs p;
  p.msa = msa; p.io_f32 = msa_dt == AF3_F32; p.rows = (int)rows; p.n = (int)n; p.ld = up8(rows);
  p.ln_w = b.opm_ln_w; p.ln_b = b.opm_ln_b; p.w = b.opm_w_lr; p.mask = msa_mask;
  for (bf16_t*& o : p.out) o = static_cast<bf16_t*>(w.take((size_t)n * 32 * p.ld * 2));
  if (!w.ok) return AF3_ERR_WORKSPACE;
  STEP(launch_msa_project(p, false, s));
  GemmArgs g;
  g.A = p.out[0]; g.B = p.out[1]; g.C = pair; g.out_f32 = pair_dt == AF3_F32;
  g.M = g.N = (int)n * 32; g.K = (int)p.ld; g.lda = g.ldb = p.ld;
  g.w2 = b.opm_w_out; g.bias = b.opm_b_out; g.gate = inv;
  if (residual && g.out_f32) g.res_f32 = static_cast<const float*>(pair);
  else if (residual) g.res_bf16 = static_cast<const bf16_t*>(pair);
  return launch_outer_mean(g, s);
}

// The weighted average of the MSA's values, [head][token][row][8]
int msa_average(const af3_msa_block& b, const void* msa, int msa_dt, const float* live, const float* logits, int64_t rows, int64_t n,
                Carver& w, const bf16_t** avg_out, hipStream_t s) {
  MsaProjectArgs p;
  p.msa = msa; p.io_f32 = msa_dt == AF3_F32; p.rows = (int)rows; p.n = (int)n; p.ld = up8(n);
  p.ln_w = b.ma_ln_w; p.ln_b = b.ma_ln_b; p.w = b.ma_w_v;
  bf16_t* weights = static_cast<bf16_t*>(w.take((size_t)8 * n * p.ld * 2));
  p.out[0] = static_cast<bf16_t*>(w.take((size_t)64 * rows * p.ld * 2));
  bf16_t* avg = static_cast<bf16_t*>(w.take((size_t)64 * rows * n * 2));
  if (!w.ok) return AF3_ERR_WORKSPACE;
  STEP(launch_msa_project(p, true, s));
  STEP(launch_softmax_rows(logits, live, weights, 8 * n, (int)n, p.ld, s));
  *avg_out = avg;
  return af3_batched_nt_product_forward(weights, p.out[0], avg, 8, n, 8 * rows, p.ld, s);
}

void msa_attention_args(const af3_msa_block& b, const bf16_t* avg, MsaUpdateArgs& u) {
  u.avg = avg; u.att_ln_w = b.ma_ln_w; u.att_ln_b = b.ma_ln_b; u.w_g = b.ma_w_g; u.w_o = b.ma_w_o;
}
void msa_transition_args(const float* ln_w, const float* ln_b, const uint16_t* w1, const uint16_t* w2, int hidden, MsaUpdateArgs& u) {
  u.tr_ln_w = ln_w; u.tr_ln_b = ln_b; u.w1 = w1; u.w2 = w2; u.hidden = hidden;
}

}  // namespace

extern "C" {

size_t af3_msa_workspace_bytes(int64_t rows, int64_t n) {
  if (!msa_size_ok(rows, n)) return 0;
  const size_t a = opm_bytes(rows, n), b = msa_attention_bytes(rows, n);
  return msa_mask_bytes(n) + align_up((size_t)n * n * 4) + (a > b ? a : b);
}

int af3_outer_product_mean_forward(const af3_msa_block* block, const void* msa, int msa_dtype, const float* msa_mask, void* pair,
                                   int pair_dtype, int residual, int64_t rows, int64_t n, void* workspace,
                                   size_t workspace_bytes, af3_stream_t stream) {
  if (!block || !msa || !msa_mask || !pair || !msa_size_ok(rows, n)) return AF3_ERR_BAD_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  Carver w(workspace, workspace_bytes);
  float *inv = static_cast<float*>(w.take((size_t)n * n * 4)), *live = static_cast<float*>(w.take((size_t)n * 4));
  if (!w.ok) return AF3_ERR_WORKSPACE;
  STEP(launch_msa_coverage(msa_mask, (int)rows, (int)n, block->epsilon, inv, live, s));
  return outer_product_mean(*block, msa, msa_dtype, msa_mask, inv, pair, pair_dtype, residual, rows, n, w, s);
}

int af3_msa_attention_forward(const af3_msa_block* block, const void* msa, int msa_dtype, const float* msa_mask, const void* pair,
                              int pair_dtype, void* out, int residual, int64_t rows, int64_t n, void* workspace,
                              size_t workspace_bytes, af3_stream_t stream) {
  if (!block || !msa || !msa_mask || !pair || !out || !msa_size_ok(rows, n)) return AF3_ERR_BAD_ARG;
  hipStream_t s = static_cast<hipStream_t>(stream);
  Carver w(workspace, workspace_bytes);
  float *inv = static_cast<float*>(w.take((size_t)n * n * 4)), *live = static_cast<float*>(w.take((size_t)n * 4));
  float* logits = static_cast<float*>(w.take((size_t)8 * n * n * 4));
  if (!w.ok) return AF3_ERR_WORKSPACE;
  STEP(launch_msa_coverage(msa_mask, (int)rows, (int)n, block->epsilon, inv, live, s));
  STEP(af3_pair_logits_forward(pair, pair_dtype, block->ma_pn_w, block->ma_pn_b, block->ma_w_logits, 8, logits, n, stream));
  MsaUpdateArgs u;
  u.msa = msa; u.out = out; u.io_f32 = msa_dtype == AF3_F32; u.rows = (int)rows; u.n = (int)n; u.residual = residual;
  const bf16_t* avg;
  STEP(msa_average(*block, msa, msa_dtype, live, logits, rows, n, w, &avg, s));
  msa_attention_args(*block, avg, u);
  return launch_msa_update(u, s);
}

int af3_transition64_forward(const void* x, int io_dtype, const float* ln_w, const float* ln_b, const uint16_t* w1,
                             const uint16_t* w2, int hidden, void* out, int residual, int64_t rows, af3_stream_t stream) {
  if (!x || !out || rows <= 0 || rows > (1ll << 30) || (io_dtype != AF3_F32 && io_dtype != AF3_BF16)) return AF3_ERR_BAD_ARG;
  MsaUpdateArgs u;
  u.msa = x; u.out = out; u.io_f32 = io_dtype == AF3_F32; u.rows = (int)rows; u.n = 1; u.residual = residual;
  msa_transition_args(ln_w, ln_b, w1, w2, hidden, u);
  return launch_msa_update(u, static_cast<hipStream_t>(stream));
}

int af3_evoformer_stack_forward(const af3_msa_block* const* blocks, int num_blocks, void* msa, int msa_dtype, const float* msa_mask,
                                void* pair, int pair_dtype, const float* pair_mask, int64_t rows, int64_t n, void* workspace,
                                size_t workspace_bytes, void* pair_workspace, size_t pair_workspace_bytes, af3_stream_t stream) {
  if (!blocks || num_blocks <= 0 || !msa || !msa_mask || !pair || !msa_size_ok(rows, n)) return AF3_ERR_BAD_ARG;
  if ((msa_dtype != AF3_F32 && msa_dtype != AF3_BF16) || (pair_dtype != AF3_F32 && pair_dtype != AF3_BF16)) return AF3_ERR_BAD_ARG;
  for (int i = 0; i < num_blocks; ++i)
    if (!blocks[i] || blocks[i]->epsilon != blocks[0]->epsilon || blocks[i]->pair.pair_channels == 64) return AF3_ERR_BAD_ARG;
  if (workspace_bytes < af3_msa_workspace_bytes(rows, n)) return AF3_ERR_WORKSPACE;  // (in place: before the first launch)
  for (int i = 0; i < num_blocks; ++i)
    if (pair_workspace_bytes < af3_pairformer_stack_workspace_bytes(n, blocks[i]->pair.num_head_pair)) return AF3_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  Carver w(workspace, workspace_bytes);
  float *inv = static_cast<float*>(w.take((size_t)n * n * 4)), *live = static_cast<float*>(w.take((size_t)n * 4));
  float* mask_in = static_cast<float*>(w.take((size_t)n * n * 4));
  if (!w.ok) return AF3_ERR_WORKSPACE;
  // what depends on the masks alone: once for all blocks
  STEP(launch_msa_coverage(msa_mask, (int)rows, (int)n, blocks[0]->epsilon, inv, live, s));
  if (pair_mask) STEP(launch_transpose_f32(pair_mask, mask_in, (int)n, s));
  for (int i = 0; i < num_blocks; ++i) {
    const af3_msa_block& b = *blocks[i];
    STEP(outer_product_mean(b, msa, msa_dtype, msa_mask, inv, pair, pair_dtype, 1, rows, n, w, s));
    Carver v = w;  // the outer product's operands are done with
    float* logits = static_cast<float*>(v.take((size_t)8 * n * n * 4));
    if (!v.ok) return AF3_ERR_WORKSPACE;
    STEP(af3_pair_logits_forward(pair, pair_dtype, b.ma_pn_w, b.ma_pn_b, b.ma_w_logits, 8, logits, n, stream));
    MsaUpdateArgs u;
    u.msa = u.out = msa; u.io_f32 = msa_dtype == AF3_F32; u.rows = (int)rows; u.n = (int)n; u.residual = 1;
    const bf16_t* avg;
    STEP(msa_average(b, msa, msa_dtype, live, logits, rows, n, v, &avg, s));
    msa_attention_args(b, avg, u);
    msa_transition_args(b.mt_ln_w, b.mt_ln_b, b.mt_w1, b.mt_w2, b.mt_hidden, u);
    STEP(launch_msa_update(u, s));
    STEP(pair_operators(b.pair, pair, pair_dtype, pair_mask, pair_mask ? mask_in : nullptr, n, pair_workspace, pair_workspace_bytes, s));
  }
  return AF3_OK;
}

size_t af3_pairformer_stack_workspace_bytes(int64_t n, int num_head_pair) {
  const size_t a = af3_triangle_multiplication_workspace_bytes(n), b = af3_grid_self_attn_workspace_bytes(n, num_head_pair);
  size_t most = a > b ? a : b;
  if (n > 0 && n * tri_ldn(n) <= F32_STEP_POSITIONS && PairStepScratch::bytes(n, 128) > most) most = PairStepScratch::bytes(n, 128);
  if (n > 0 && n <= AF3_PAIR64_MAX_TOKENS && PairStepScratch::bytes(n, 64) > most) most = PairStepScratch::bytes(n, 64);
  return most;
}

size_t af3_pairformer_single_workspace_bytes(int64_t n, int c_single, int single_hidden) {
  if (n <= 0 || c_single <= 0 || single_hidden <= 0) return 0;
  return align_up((size_t)n * c_single * 2) + align_up((size_t)n * (c_single > single_hidden ? c_single : single_hidden) * 2) +
         align_up(af3_batch_diffusion_self_attention_workspace_bytes(1, n, c_single));
}

int af3_pairformer_stack_forward(
    const af3_pairformer_block* const* blocks, int num_blocks, void* pair, int pair_dtype, const float* pair_mask,
    const float* pair_mask_incoming, void* single, int single_dtype, const float* seq_mask, int64_t n, float* logits,
    void* workspace, size_t workspace_bytes, void* single_workspace, size_t single_workspace_bytes, af3_stream_t stream,
    af3_stream_t single_stream, int join) {
  if (!blocks || num_blocks <= 0 || !pair || n <= 0) return AF3_ERR_BAD_ARG;
  // all of it before the first launch: the blocks work in place
  for (int i = 0; i < num_blocks; ++i) {
    if (!blocks[i]) return AF3_ERR_BAD_ARG;
    const af3_pairformer_block& b = *blocks[i];
    if (workspace_bytes < af3_pairformer_stack_workspace_bytes(n, b.num_head_pair)) return AF3_ERR_WORKSPACE;
    // (a pair tensor of 64 channels is what the step kernels alone take)
    if ((b.pair_channels != 0 && b.pair_channels != 128 && b.pair_channels != 64) ||
        (b.pair_channels == 64) != (blocks[0]->pair_channels == 64) ||
        (b.pair_channels == 64 && (!pair_steps_apply(b, n, pair_dtype) || b.with_single)))
      return AF3_ERR_BAD_ARG;
    if (!b.with_single) continue;
    if (!single || !logits || b.num_head != blocks[0]->num_head || b.c_single != blocks[0]->c_single) return AF3_ERR_BAD_ARG;
    if (single_workspace_bytes < af3_pairformer_single_workspace_bytes(n, b.c_single, b.single_hidden)) return AF3_ERR_WORKSPACE;
  }
  hipStream_t main_s = static_cast<hipStream_t>(stream);
  hipStream_t side_s = single_stream ? static_cast<hipStream_t>(single_stream) : main_s;
  const bool two = side_s != main_s;
  // The pair logits of the run's k-th single track are in buffer k % buffers: two, the caller's, or at few tokens more of
  // them in the workspace (which nothing else uses before the streams have been joined).
  float* first = logits;
  int buffers = num_blocks > 1 ? 2 : 1;
  size_t logit_size = logits ? (size_t)blocks[0]->num_head * ((n + 3) / 4 * 4) * n : 0;
  if (two && join) {
    bool all = n * tri_ldn(n) <= PairStepScratch::LOGIT_RING_POSITIONS;
    for (int i = 0; i < num_blocks; ++i) all = all && pair_steps_apply(*blocks[i], n, pair_dtype) && blocks[i]->num_head <= 16;
    PairStepScratch w;
    if (all && workspace_bytes >= PairStepScratch::bytes(n, 128) && w.carve(n, 128, workspace, workspace_bytes)) {
      first = w.ring(n);
      logit_size = PairStepScratch::logit_bytes(n, 16) / 4;
      buffers = PairStepScratch::LOGIT_RING;
    }
  }
  const int half = buffers > 1 ? buffers / 2 : 1;
  Event ready, read_done[2];  // behind the pair logits; behind the last attention that reads a buffer of either half
  int singles = 0;
  for (int i = 0; i < num_blocks; ++i) singles += blocks[i]->with_single ? 1 : 0;
  // (the wait in front of the first update of `single` is for what `stream` holds on entry, too)
  if (two && singles == 0) STEP(ready.order(main_s, side_s));
  // Where launches set the pace the updates of two blocks wait for the streams' meeting together, but for the last one, which has no
  // pair operators to run beside.  With the wait on entry, that is four meetings for four blocks instead of six: 64 tokens 381 -> 343
  // us (321 -> 308 in a process that launches faster), 45 382 -> 339, 128 464 -> 454; past 144 tokens the pair operators are longer
  // than what an update waits for (176, two together: 683 -> 689).
  const bool by_two = buffers == PairStepScratch::LOGIT_RING && n * tri_ldn(n) <= 144 * 144;
  int rc = AF3_OK, k = 0, done = 0, from = 0;  // single tracks whose logits are on their way, those enqueued; the block of the next one
  for (int i = 0; i < num_blocks && rc == AF3_OK; ++i) {
    const af3_pairformer_block& b = *blocks[i];
    float* lg = nullptr;
    Event* free = nullptr;
    if (b.with_single) {
      lg = first + (k % buffers) * logit_size;
      if (k % half == 0) free = &read_done[k / half & 1];
    }
    // the pair logits are the only thing the single track reads of `pair`: they are made in front of whatever updates it next
    if (pair_steps_apply(b, n, pair_dtype)) {
      const bool chained = i > 0 && pair_steps_apply(*blocks[i - 1], n, pair_dtype);
      const af3_pairformer_block* next = i + 1 < num_blocks && pair_steps_apply(*blocks[i + 1], n, pair_dtype) ? blocks[i + 1] : nullptr;
      rc = pair_operators_in_steps(b, next, !chained, pair, pair_dtype, pair_mask, pair_mask_incoming, n, workspace, workspace_bytes,
                                   lg, free, main_s);
      if (rc != AF3_OK || !b.with_single) continue;
    } else {
      rc = pair_operators(b, pair, pair_dtype, pair_mask, pair_mask_incoming, n, workspace, workspace_bytes, main_s);
      if (rc != AF3_OK || !b.with_single) continue;
      if (free) rc = free->wait(main_s);
      if (rc == AF3_OK)
        rc = af3_pair_logits_quads_forward(pair, pair_dtype, b.sl_ln_w, b.sl_ln_b, b.sl_w, b.num_head, lg, n, stream);
    }
    ++k;
    if (rc != AF3_OK || (by_two && k % 2 == 1 && k + 1 < singles)) continue;
    if (two) rc = ready.order(main_s, side_s);
    for (; from <= i && rc == AF3_OK; ++from) {
      const af3_pairformer_block& t = *blocks[from];
      if (!t.with_single) continue;
      rc = single_update(t, single, single_dtype, seq_mask, first + (done % buffers) * logit_size, n, single_workspace,
                         single_workspace_bytes, side_s);
      if (rc == AF3_OK && two && done % half == half - 1 && from + half + 1 < num_blocks) rc = read_done[done / half & 1].record(side_s);
      ++done;
    }
  }
  if (two && join) {
    const int jrc = ready.order(side_s, main_s);
    if (rc == AF3_OK) rc = jrc;
  }
  return rc;
}

size_t af3_diffusion_transformer_workspace_bytes(int64_t batch, int64_t seq, int channels, int hidden) {
  if (batch <= 0 || seq <= 0 || channels <= 0 || hidden <= 0) return 0;
  const size_t rows = (size_t)batch * seq;
  return align_up(rows * channels * 2) + align_up(rows * (channels > hidden ? channels : hidden) * 2) +
         align_up(af3_batch_diffusion_self_attention_workspace_bytes(batch, seq, channels));
}

static constexpr size_t WARM_LOGIT_BYTES = (size_t)4 << 20;
int af3_diffusion_transformer_forward(
    const af3_diffusion_block* blocks, int num_blocks, void* act, int act_dtype, int64_t batch, int64_t seq, int channels,
    int hidden, int num_head, const float* key_mask, const float* const* pair_logits, int bias_quad_major,
    const float* scale_shift, const float* gate, int64_t cond_rows, void* workspace, size_t workspace_bytes,
    af3_stream_t stream) {
  if (!blocks || num_blocks <= 0 || !act || !pair_logits || !scale_shift || !gate || cond_rows <= 0 || batch <= 0 || seq <= 0 ||
      channels <= 0 || hidden <= 0 || num_head <= 0 || channels % num_head)
    return AF3_ERR_BAD_ARG;
  const int c = channels;
  const int64_t rows = batch * seq, ld_ss = (int64_t)2 * num_blocks * 2 * c, ld_g = (int64_t)2 * num_blocks * c;
  Carver w(workspace, workspace_bytes);
  uint16_t* x = static_cast<uint16_t*>(w.take((size_t)rows * c * 2));
  uint16_t* y = static_cast<uint16_t*>(w.take((size_t)rows * (c > hidden ? c : hidden) * 2));
  const size_t ab = af3_batch_diffusion_self_attention_workspace_bytes(batch, seq, c);
  void* aw = w.take(ab);
  if (!w.ok) return AF3_ERR_WORKSPACE;
  for (int i = 0; i < num_blocks; ++i)  // (`frags` stand beside the weights, not in their place)
    if (!blocks[i].w_q || !blocks[i].w_out || !blocks[i].w_tr1 || !blocks[i].w_tr2) return AF3_ERR_BAD_ARG;
  // Adaptive LayerNorm of act, with the weights of the products up to the next one on their way into the last-level cache
  // (rowops.hip), and the pair logits where they are no more than the weights.  The conditioning of those products, rows of
  // 6 KB some 300 KB apart, costs more that way than it saves.
  struct Range {
    const void* p;
    size_t bytes;
  };
  auto norm = [&](const float* ss, Range r0, Range r1, Range r2) -> int {
    RowNormArgs a;
    if (act_dtype != AF3_F32 && act_dtype != AF3_BF16) return AF3_ERR_BAD_ARG;
    a.x = act; a.x_f32 = act_dtype == AF3_F32; a.y = x; a.rows = rows; a.ldx = a.ldy = c; a.C = c;
    a.scale = ss; a.shift = ss + c; a.cond_rows = cond_rows; a.ld_cond = ld_ss;
    int k = 0;
    for (const Range& r : {r0, r1, r2})
      if (r.p) { a.warm[k] = r.p; a.warm_lines[k] = (uint32_t)(r.bytes / 128); ++k; }
    return launch_row_norm(a, static_cast<hipStream_t>(stream));
  };
  // The norm and the product behind it in one kernel, where all blocks' weights are there in its order; it warms what the kernels
  // up to the next one read, the next one's weights among it.
  bf16_t* const qkvg = self_projections(aw, ab, rows, c);
  const bool act_ok = act_dtype == AF3_BF16 && c == TOKEN_STEP_CHANNELS && cond_rows == seq && rows <= 0x7fffffff;
  auto step = [&](int i, bool transition) {
    const af3_diffusion_block& b = blocks[i];
    NormProductArgs a;
    a.x = static_cast<const bf16_t*>(act); a.samples = (int)batch; a.tokens = (int)seq;
    a.scale = scale_shift + ((int64_t)2 * i + transition) * 2 * c; a.ld_cond = (int)ld_ss;
    a.w = b.frags ? b.frags + (transition ? (int64_t)4 * c * c : 0) : nullptr;
    a.swiglu = transition; a.N = transition ? 2 * hidden : 4 * c; a.ldc = transition ? hidden : 4 * c;
    a.out = transition ? y : qkvg;
    if (!transition) { a.q_bias = b.q_b; a.q_scale = 1.0f / sqrtf((float)(c / num_head)); }
    return a;
  };
  // Where the norm stands by itself, the products that token_step.hip takes over any number of rows.
  auto product = [&](int i, bool transition) {
    const af3_diffusion_block& b = blocks[i];
    RowsProductArgs a;
    a.rows = (int)rows; a.x = reinterpret_cast<const bf16_t*>(x); a.K = c; a.swiglu = transition; a.N = transition ? 2 * hidden : 4 * c;
    a.ldc = transition ? hidden : 4 * c; a.out = transition ? reinterpret_cast<bf16_t*>(y) : qkvg;
    a.w = act_ok && b.frags ? b.frags + (transition ? (int64_t)4 * c * c : 0) : nullptr;
    if (!transition) { a.q_bias = b.q_b; a.q_scale = 1.0f / sqrtf((float)(c / num_head)); }
    return a;
  };
  // The product behind either, with its gate, into the stream.
  auto back = [&](int i, bool transition) {
    const af3_diffusion_block& b = blocks[i];
    RowsProductArgs a;
    a.rows = (int)rows; a.x = reinterpret_cast<const bf16_t*>(y); a.N = c; a.K = transition ? hidden : c; a.ldc = c;
    a.out = static_cast<bf16_t*>(act); a.gate = gate + ((int64_t)2 * i + transition) * c; a.ld_gate = ld_g; a.cond_rows = (int)cond_rows;
    a.w = act_ok && b.frags ? b.frags + (int64_t)(transition ? 5 * c + 2 * hidden : 4 * c + 2 * hidden) * c : nullptr;
    return a;
  };
  auto few_rows = [](const RowsProductArgs& r) {
    GatedProductArgs a;
    a.rows = r.rows; a.K = r.K; a.cond_rows = r.cond_rows; a.y = r.x; a.act = r.out; a.w = r.w; a.gate = r.gate; a.ld_gate = r.ld_gate;
    return a;
  };
  // (the fragments that product_back reads, or the weights as they were given)
  auto weights_back = [&](int i, bool transition) -> const void* {
    const RowsProductArgs a = back(i, transition);
    return gated_product_applies(few_rows(a)) || rows_product_applies(a) ? (const void*)a.w : transition ? blocks[i].w_tr2 : blocks[i].w_out;
  };
  auto product_back = [&](int i, bool transition) -> int {
    const RowsProductArgs a = back(i, transition);
    const GatedProductArgs few = few_rows(a);
    if (gated_product_applies(few)) return launch_gated_product(few, static_cast<hipStream_t>(stream));
    if (rows_product_applies(a)) return launch_rows_product(a, static_cast<hipStream_t>(stream));
    const af3_diffusion_block& b = blocks[i];
    return af3_linear_forward(y, transition ? b.w_tr2 : b.w_out, nullptr, act, act_dtype, rows, c, transition ? hidden : c,
                              AF3_LINEAR_GATE_RES, 1.f, 0, gate + ((int64_t)2 * i + transition) * c, cond_rows, ld_g, act, act_dtype, stream);
  };
  bool steps = act_ok && qkvg;
  for (int i = 0; i < num_blocks && steps; ++i) steps = norm_product_applies(step(i, false)) && norm_product_applies(step(i, true));
  if (bias_quad_major != 0 && (bias_quad_major != 1 || (seq & 3))) return AF3_ERR_BAD_ARG;
  const size_t all_logits = (size_t)num_head * seq * seq * 4, logit_bytes = all_logits <= WARM_LOGIT_BYTES ? all_logits : 0;
  for (int i = 0; i < num_blocks; ++i) {
    const af3_diffusion_block& b = blocks[i];
    const float* ss = scale_shift + (int64_t)2 * i * 2 * c;
    if (steps) {
      auto warm = [](NormProductArgs& a, int k, const void* p, size_t bytes) {  // (a null entry of pair_logits is no bias)
        if (p) { a.warm[k] = p; a.warm_lines[k] = (uint32_t)(bytes / 128); }
      };
      NormProductArgs a = step(i, false);
      warm(a, 0, weights_back(i, false), (size_t)c * c * 2);
      warm(a, 1, b.frags + (int64_t)4 * c * c, (size_t)2 * hidden * c * 2);
      warm(a, 2, pair_logits[i], logit_bytes);
      STEP(launch_norm_product(a, static_cast<hipStream_t>(stream)));
      STEP(run_self_attend(qkvg, key_mask, 1, pair_logits[i], bias_quad_major, num_head, y, AF3_BF16, batch, seq, c,
                           static_cast<hipStream_t>(stream)));
      STEP(product_back(i, false));
      a = step(i, true);
      warm(a, 0, weights_back(i, true), (size_t)hidden * c * 2);
      if (i + 1 < num_blocks) warm(a, 1, blocks[i + 1].frags, (size_t)4 * c * c * 2);
      STEP(launch_norm_product(a, static_cast<hipStream_t>(stream)));
      STEP(product_back(i, true));
      continue;
    }
    const RowsProductArgs in = product(i, false), hidden_in = product(i, true);
    const bool in_rows = qkvg && rows_product_applies(in), hidden_rows = rows_product_applies(hidden_in);
    STEP(norm(ss, {in_rows ? (const void*)in.w : b.w_q, (size_t)4 * c * c * 2}, {weights_back(i, false), (size_t)c * c * 2},
              {pair_logits[i], logit_bytes}));
    if (in_rows) {
      STEP(launch_rows_product(in, static_cast<hipStream_t>(stream)));
      STEP(run_self_attend(qkvg, key_mask, 1, pair_logits[i], bias_quad_major, num_head, y, AF3_BF16, batch, seq, c,
                           static_cast<hipStream_t>(stream)));
    } else {
      STEP(af3_batch_diffusion_self_attention_forward(x, key_mask, 1, pair_logits[i], bias_quad_major, b.w_q, b.q_b, num_head, y,
                                                      AF3_BF16, batch, seq, c, aw, ab, stream));
    }
    STEP(product_back(i, false));
    STEP(norm(ss + 2 * c, {hidden_rows ? (const void*)hidden_in.w : b.w_tr1, (size_t)2 * hidden * c * 2},
              {weights_back(i, true), (size_t)hidden * c * 2}, {nullptr, 0}));
    if (hidden_rows) STEP(launch_rows_product(hidden_in, static_cast<hipStream_t>(stream)));
    else
      STEP(af3_linear_forward(x, b.w_tr1, nullptr, y, AF3_BF16, rows, 2 * hidden, c, AF3_LINEAR_SWIGLU, 1.f, 0, nullptr, 0, 0, nullptr, 0,
                              stream));
    STEP(product_back(i, true));
  }
  return AF3_OK;
}

size_t af3_atom_transformer_workspace_bytes(int64_t samples, int64_t subsets, int64_t queries, int channels, int hidden) {
  if (samples <= 0 || subsets <= 0 || queries <= 0 || channels <= 0 || hidden <= 0) return 0;
  const size_t rows = (size_t)samples * subsets * queries;
  return 2 * align_up(rows * channels * 2) + align_up(rows * (channels > hidden ? channels : hidden) * 2) +
         align_up(af3_gathered_cross_attention_workspace_bytes(samples * subsets, queries, samples, subsets * queries, channels));
}

static int atom_transformer(
    const af3_diffusion_block* blocks, int num_blocks, void* act, int act_dtype, int64_t samples, int64_t subsets,
    int64_t queries, int64_t keys, int channels, int hidden, int num_head, const int32_t* key_rows, const float* mask_q,
    const float* mask_k, const float* pair_logits, int bias_quad_major, const float* scale_shift_q, const float* scale_shift_k,
    const float* gate, const int32_t* windows, void* workspace, size_t workspace_bytes, af3_stream_t stream) {
  if (!blocks || num_blocks <= 0 || !act || !key_rows || !scale_shift_q || !scale_shift_k || !gate || samples <= 0 ||
      subsets <= 0 || queries <= 0 || keys <= 0 || channels <= 0 || hidden <= 0 || num_head <= 0)
    return AF3_ERR_BAD_ARG;
  const int c = channels;
  const int64_t atoms = subsets * queries, rows = samples * atoms;
  const int64_t ld_q = (int64_t)2 * num_blocks * 2 * c, ld_k = (int64_t)num_blocks * 2 * c;
  Carver w(workspace, workspace_bytes);
  uint16_t* xq = static_cast<uint16_t*>(w.take((size_t)rows * c * 2));
  uint16_t* xk = static_cast<uint16_t*>(w.take((size_t)rows * c * 2));
  uint16_t* y = static_cast<uint16_t*>(w.take((size_t)rows * (c > hidden ? c : hidden) * 2));
  const size_t ab = af3_gathered_cross_attention_workspace_bytes(samples * subsets, queries, samples, atoms, c);
  void* aw = w.take(ab);
  if (!w.ok) return AF3_ERR_WORKSPACE;
  // everything between two attentions in one kernel, where all blocks' weights are there in its order
  auto step_args = [&](int i) {
    const af3_diffusion_block& b = blocks[i];
    const float *ss = scale_shift_q + (int64_t)2 * i * 2 * c, *g = gate + (int64_t)2 * i * atoms * c;
    AtomStepArgs a;
    a.act = act; a.io_f32 = act_dtype == AF3_F32; a.atoms = (int)atoms; a.samples = (int)samples; a.hidden = hidden;
    a.y = y; a.gate1 = g; a.gate2 = g + atoms * c; a.scale = ss + 2 * c; a.ld_cond = ld_q;
    a.f_out = b.frags; a.tiles = windows;
    if (b.frags) { a.f_w1 = b.frags + c * c; a.f_w2 = a.f_w1 + 2 * hidden * c; }
    return a;
  };
  auto attention_args = [&](AtomStepArgs& a, int i) {  // the attention behind the step is block i's
    const af3_diffusion_block& b = blocks[i];
    a.f_head = b.frags ? b.frags + (c + 3 * hidden) * c : nullptr;
    a.scale_q = scale_shift_q + (int64_t)2 * i * 2 * c;
    a.scale_k = scale_shift_k + (int64_t)i * 2 * c; a.ld_cond_k = ld_k;
    a.q_bias = b.q_b; a.q_scale = 1.0f / sqrtf((float)(c / num_head));
    (void)gathered_projections(aw, ab, rows, rows, c, &a.qg, &a.kv);
  };
  bool steps = c == 128 && rows <= 0x7fffffff && (act_dtype == AF3_F32 || act_dtype == AF3_BF16);
  for (int i = 0; i < num_blocks && steps; ++i) {
    AtomStepArgs a = step_args(i);
    attention_args(a, i);
    steps = atom_steps_apply(a);
  }
  // (a window's queries are a tile of the steps, and its attention is window_kernel's: what makes neither takes all of them)
  if (!steps || queries != 32 || num_head != 4 || keys > 128 || (keys & 3) || !pair_logits || ((uintptr_t)pair_logits & 15) ||
      atoms >= 1 << 22)
    windows = nullptr;
  for (int i = 0; i < num_blocks; ++i) {
    const af3_diffusion_block& b = blocks[i];
    const float* pl = pair_logits ? pair_logits + (int64_t)i * subsets * num_head * queries * keys : nullptr;
    if (steps) {
      AtomStepArgs a = step_args(i);
      if (i == 0) {
        attention_args(a, 0);
        STEP(launch_atom_step(a, false, true, static_cast<hipStream_t>(stream)));
      }
      STEP(run_gathered_attention(nullptr, nullptr, key_rows, pl, bias_quad_major, mask_q, mask_k, subsets, b.w_q, b.w_kv, b.q_b, num_head, y,
                                  AF3_BF16, samples * subsets, queries, keys, samples, atoms, c, aw, ab,
                                  static_cast<hipStream_t>(stream), windows));
      const bool more = i + 1 < num_blocks;
      attention_args(a, more ? i + 1 : i);
      STEP(launch_atom_step(a, true, more, static_cast<hipStream_t>(stream)));
      continue;
    }
    const float *ss = scale_shift_q + (int64_t)2 * i * 2 * c, *sk = scale_shift_k + (int64_t)i * 2 * c;
    const float* g = gate + (int64_t)2 * i * atoms * c;
    if (c <= 128) {
      RowNormArgs ln;
      ln.x = act; ln.x_f32 = act_dtype == AF3_F32; ln.rows = rows; ln.ldx = ln.ldy = ln.C = c;
      ln.y = xq; ln.scale = ss; ln.shift = ss + c; ln.cond_rows = atoms; ln.ld_cond = ld_q;
      ln.y2 = xk; ln.scale2 = sk; ln.shift2 = sk + c; ln.ld_cond2 = ld_k;
      STEP(launch_row_norm(ln, static_cast<hipStream_t>(stream)));
    } else {
      STEP(af3_layer_norm_forward(act, act_dtype, xq, rows, c, nullptr, nullptr, ss, ss + c, atoms, ld_q, stream));
      STEP(af3_layer_norm_forward(act, act_dtype, xk, rows, c, nullptr, nullptr, sk, sk + c, atoms, ld_k, stream));
    }
    STEP(run_gathered_attention(xq, xk, key_rows, pl, bias_quad_major, mask_q, mask_k, subsets, b.w_q, b.w_kv, b.q_b, num_head, y,
                                AF3_BF16, samples * subsets, queries, keys, samples, atoms, c, aw, ab,
                                static_cast<hipStream_t>(stream)));
    STEP(af3_linear_forward(y, b.w_out, nullptr, act, act_dtype, rows, c, c, AF3_LINEAR_GATE_RES, 1.f, 0, g, atoms, 0, act, act_dtype,
                            stream));
    STEP(af3_layer_norm_forward(act, act_dtype, xq, rows, c, nullptr, nullptr, ss + 2 * c, ss + 3 * c, atoms, ld_q, stream));
    STEP(af3_linear_forward(xq, b.w_tr1, nullptr, y, AF3_BF16, rows, 2 * hidden, c, AF3_LINEAR_SWIGLU, 1.f, 0, nullptr, 0, 0, nullptr,
                            0, stream));
    STEP(af3_linear_forward(y, b.w_tr2, nullptr, act, act_dtype, rows, c, hidden, AF3_LINEAR_GATE_RES, 1.f, 0, g + atoms * c, atoms, 0,
                            act, act_dtype, stream));
  }
  return AF3_OK;
}
int af3_atom_transformer_forward(
    const af3_diffusion_block* blocks, int num_blocks, void* act, int act_dtype, int64_t samples, int64_t subsets,
    int64_t queries, int64_t keys, int channels, int hidden, int num_head, const int32_t* key_rows, const float* mask_q,
    const float* mask_k, const float* pair_logits, int bias_quad_major, const float* scale_shift_q, const float* scale_shift_k,
    const float* gate, void* workspace, size_t workspace_bytes, af3_stream_t stream) {
  return atom_transformer(blocks, num_blocks, act, act_dtype, samples, subsets, queries, keys, channels, hidden, num_head, key_rows, mask_q,
                          mask_k, pair_logits, bias_quad_major, scale_shift_q, scale_shift_k, gate, nullptr, workspace, workspace_bytes,
                          stream);
}
int af3_atom_transformer_windows_forward(
    const af3_diffusion_block* blocks, int num_blocks, void* act, int act_dtype, int64_t samples, int64_t subsets,
    int64_t queries, int64_t keys, int channels, int hidden, int num_head, const int32_t* key_rows, const float* mask_q,
    const float* mask_k, const float* pair_logits, int bias_quad_major, const float* scale_shift_q, const float* scale_shift_k,
    const float* gate, const int32_t* windows, void* workspace, size_t workspace_bytes, af3_stream_t stream) {
  if (!windows) return AF3_ERR_BAD_ARG;
  return atom_transformer(blocks, num_blocks, act, act_dtype, samples, subsets, queries, keys, channels, hidden, num_head, key_rows, mask_q,
                          mask_k, pair_logits, bias_quad_major, scale_shift_q, scale_shift_k, gate, windows, workspace, workspace_bytes,
                          stream);
}

// ------------------------------------------------------------- element-wise passes
int af3_contact_matrix_forward(const int64_t* idx0, const uint8_t* exists0, int count0, const int64_t* idx1, const uint8_t* exists1,
                               int count1, float* contact, int64_t n, af3_stream_t stream) {
  if (n <= 0 || n > 8192) return AF3_ERR_BAD_ARG;
  return launch_contacts(idx0, exists0, count0, idx1, exists1, count1, contact, (int)n, static_cast<hipStream_t>(stream));
}

int af3_pair_embed_forward(const float* lr, int64_t ld_lr, const float* prev, const int64_t* asym_id, const int64_t* residue_index,
                           const int64_t* token_index, const int64_t* entity_id, const int64_t* sym_id, const float* w_pos,
                           const float* w_bond, const float* contact, void* out, int out_dtype, int64_t n, af3_stream_t stream) {
  if (n <= 0 || n > 8192 || (out_dtype != AF3_F32 && out_dtype != AF3_BF16)) return AF3_ERR_BAD_ARG;
  PairEmbedArgs a;
  a.lr = lr; a.ld_lr = ld_lr; a.prev = prev;
  a.asym_id = asym_id; a.residue_index = residue_index; a.token_index = token_index; a.entity_id = entity_id; a.sym_id = sym_id;
  a.w_pos = w_pos; a.w_bond = w_bond; a.contact = contact; a.out = out; a.out_f32 = out_dtype == AF3_F32; a.n = (int)n;
  return launch_pair_embed(a, static_cast<hipStream_t>(stream));
}

int af3_add_rows_forward(const float* a, const float* b, int64_t ld_b, int64_t mod, void* out, int out_dtype, int64_t rows,
                         int channels, af3_stream_t stream) {
  if (out_dtype != AF3_F32 && out_dtype != AF3_BF16) return AF3_ERR_BAD_ARG;
  return launch_add_rows(a, b, ld_b, mod, out, out_dtype == AF3_F32, rows, channels, static_cast<hipStream_t>(stream));
}

int af3_atom_windows_forward(const float* mask, const int64_t* back_idx, const uint8_t* back_exists, int64_t slots, const int32_t* key_rows,
                             int64_t subsets, int64_t queries, int64_t keys, int32_t* windows, af3_stream_t stream) {
  if (subsets <= 0 || subsets > 0x7fffffff || queries <= 0 || queries > 0x7fffffff || keys <= 0 || keys > 0x7fffffff) return AF3_ERR_BAD_ARG;
  AtomWindowsArgs a;
  a.mask = mask; a.back_idx = back_idx; a.back_exists = back_exists; a.slots = slots; a.key_rows = key_rows;
  a.windows = (int)subsets; a.queries = (int)queries; a.keys = (int)keys; a.out = windows;
  return launch_atom_windows(a, static_cast<hipStream_t>(stream));
}
int af3_mask_rows_forward(uint16_t* x, const float* mask, int64_t mod, int64_t rows, int channels, af3_stream_t stream) {
  return launch_mask_rows(x, mask, mod, rows, channels, static_cast<hipStream_t>(stream));
}

int af3_atom_embed_forward(const float* positions, const float* mask, const int64_t* element, const float* charge,
                           const int64_t* atom_name_chars, const float* w_pos, const float* w_mask, const float* w_element,
                           const float* w_charge, const float* w_chars, float* out, int64_t atoms, int channels, af3_stream_t stream) {
  AtomEmbedArgs a;
  a.positions = positions; a.mask = mask; a.element = element; a.charge = charge; a.chars = atom_name_chars;
  a.w_pos = w_pos; a.w_mask = w_mask; a.w_element = w_element; a.w_charge = w_charge; a.w_chars = w_chars;
  a.out = out; a.atoms = atoms; a.channels = channels;
  return launch_atom_embed(a, static_cast<hipStream_t>(stream));
}

int af3_gather_atoms_forward(const int64_t* idx, const uint8_t* exists, int64_t rows, const float* cond, const float* mask,
                             const float* positions, int64_t slots, const int64_t* uid, int64_t uids, const int64_t* add_idx,
                             const uint8_t* add_exists, const float* add, int64_t add_rows, float* out_cond, float* out_mask,
                             float* out_positions, int32_t* out_uid, int channels, af3_stream_t stream) {
  GatherAtomsArgs a;
  a.idx = idx; a.exists = exists; a.rows = rows; a.cond = cond; a.mask = mask; a.pos = positions; a.slots = slots;
  a.uid = uid; a.uids = uids; a.add_idx = add_idx; a.add_exists = add_exists; a.add = add; a.add_rows = add_rows;
  a.out_cond = out_cond; a.out_mask = out_mask; a.out_pos = out_positions; a.out_uid = out_uid; a.channels = channels;
  return launch_gather_atoms(a, static_cast<hipStream_t>(stream));
}

int af3_augment_positions_forward(const float* x, const float* rot, const float* shift, const float* mask, const float* noise, float* out,
                                  int64_t samples, int64_t atoms, af3_stream_t stream) {
  return launch_augment_positions(x, rot, shift, mask, noise, out, samples, atoms, static_cast<hipStream_t>(stream));
}
int af3_positions_forward(int op, const float* x, const float* y, const float* mask, const float* level, const float* next,
                          float factor, float* out, int64_t samples, int64_t atoms, af3_stream_t stream) {
  return launch_positions(op, x, y, mask, level, next, factor, out, samples, atoms, static_cast<hipStream_t>(stream));
}

}  // extern "C"
