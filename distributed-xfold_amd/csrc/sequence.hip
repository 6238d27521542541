// Whole-module entry points: the launches of a run of blocks, enqueued in one call.  Host code only; every step is
// one of the library's own entry points with the same arguments a caller would give it.
//
// Why it exists: a launch costs about 3.7 us of host time from C (measured, back to back), and about 11 us through
// the Python operator layer (argument checks, tensor allocation, ctypes).  Up to a few hundred tokens the kernels
// themselves take 4 to 10 us, so that the operator layer, not the GPU, set the pace of a block.
#include "../../include/af3_hip.h"
#include "kernels.h"

namespace {

inline size_t align_up(size_t v) { return (v + 255) / 256 * 256; }

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

// `waiter` waits for everything enqueued on `on` so far.  The event lives only for the two calls: the runtime keeps
// what a pending wait needs.
int order_streams(hipStream_t on, hipStream_t waiter) {
  hipEvent_t e;
  if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return AF3_ERR_LAUNCH;
  const bool ok = hipEventRecord(e, on) == hipSuccess && hipStreamWaitEvent(waiter, e, 0) == hipSuccess;
  return hipEventDestroy(e) == hipSuccess && ok ? AF3_OK : AF3_ERR_LAUNCH;
}

#define STEP(call)               \
  do {                           \
    const int rc_ = (call);      \
    if (rc_ != AF3_OK) return rc_; \
  } while (0)

int pair_operators(const af3_pairformer_block& b, void* pair, int dt, const float* mask, const float* mask_in, int64_t n,
                   void* ws, size_t wsb, af3_stream_t s) {
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
  STEP(af3_layer_norm_forward(single, dt, x, n, c, b.sa_ln_w, b.sa_ln_b, nullptr, nullptr, 0, 0, s));
  STEP(run_self_attention(x, mask, 1, logits, 0, b.sa_w_qkvg, b.sa_q_b, b.num_head, y, AF3_BF16, 1, n, c, aw, ab, 1, st));
  STEP(product(y, b.sa_w_out, single, dt, c, c, AF3_LINEAR_GATE_RES, single));
  STEP(af3_layer_norm_forward(single, dt, x, n, c, b.st_ln_w, b.st_ln_b, nullptr, nullptr, 0, 0, s));
  STEP(product(x, b.st_w1, y, AF3_BF16, 2 * h, c, AF3_LINEAR_SWIGLU, nullptr));
  return product(y, b.st_w2, single, dt, c, h, AF3_LINEAR_GATE_RES, single);
}

}  // namespace

extern "C" {

size_t af3_pairformer_stack_workspace_bytes(int64_t n, int num_head_pair) {
  const size_t a = af3_triangle_multiplication_workspace_bytes(n), b = af3_grid_self_attn_workspace_bytes(n, num_head_pair);
  return a > b ? a : b;
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
  for (int i = 0; i < num_blocks; ++i)
    if (!blocks[i] || (blocks[i]->with_single && (!single || !logits || blocks[i]->num_head != blocks[0]->num_head)))
      return AF3_ERR_BAD_ARG;
  hipStream_t main_s = static_cast<hipStream_t>(stream);
  hipStream_t side_s = single_stream ? static_cast<hipStream_t>(single_stream) : main_s;
  const bool two = side_s != main_s;
  if (two) STEP(order_streams(main_s, side_s));
  hipEvent_t read_done[2] = {nullptr, nullptr};  // behind the attention that reads logits buffer 0 / 1
  int rc = AF3_OK;
  for (int i = 0; i < num_blocks && rc == AF3_OK; ++i) {
    const af3_pairformer_block& b = *blocks[i];
    rc = pair_operators(b, pair, pair_dtype, pair_mask, pair_mask_incoming, n, workspace, workspace_bytes, stream);
    if (rc != AF3_OK || !b.with_single) continue;
    // the only reader of `pair` on the single path: it stays in front of whatever updates `pair` next
    float* lg = logits + (size_t)(num_blocks > 1 ? i & 1 : 0) * b.num_head * n * n;
    hipEvent_t& done = read_done[i & 1];
    if (done && hipStreamWaitEvent(main_s, done, 0) != hipSuccess) rc = AF3_ERR_LAUNCH;
    if (rc == AF3_OK)
      rc = af3_pair_logits_forward(pair, pair_dtype, b.sl_ln_w, b.sl_ln_b, b.sl_w, b.num_head, lg, n, stream);
    if (rc == AF3_OK && two) rc = order_streams(main_s, side_s);
    if (rc == AF3_OK)
      rc = single_update(b, single, single_dtype, seq_mask, lg, n, single_workspace, single_workspace_bytes, side_s);
    if (rc == AF3_OK && two && i + 2 < num_blocks) {
      if (!done && hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess) rc = AF3_ERR_LAUNCH;
      else if (hipEventRecord(done, side_s) != hipSuccess) rc = AF3_ERR_LAUNCH;
    }
  }
  for (hipEvent_t e : read_done)
    if (e && hipEventDestroy(e) != hipSuccess && rc == AF3_OK) rc = AF3_ERR_LAUNCH;
  if (two && join) {
    const int jrc = order_streams(side_s, main_s);
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

int af3_diffusion_transformer_forward(
    const af3_diffusion_block* blocks, int num_blocks, void* act, int act_dtype, int64_t batch, int64_t seq, int channels,
    int hidden, int num_head, const float* key_mask, const float* const* pair_logits, int bias_quad_major,
    const float* scale_shift, const float* gate, int64_t cond_rows, void* workspace, size_t workspace_bytes,
    af3_stream_t stream) {
  if (!blocks || num_blocks <= 0 || !act || !pair_logits || !scale_shift || !gate || cond_rows <= 0 || batch <= 0 || seq <= 0 ||
      channels <= 0 || hidden <= 0)
    return AF3_ERR_BAD_ARG;
  const int c = channels;
  const int64_t rows = batch * seq, ld_ss = (int64_t)2 * num_blocks * 2 * c, ld_g = (int64_t)2 * num_blocks * c;
  Carver w(workspace, workspace_bytes);
  uint16_t* x = static_cast<uint16_t*>(w.take((size_t)rows * c * 2));
  uint16_t* y = static_cast<uint16_t*>(w.take((size_t)rows * (c > hidden ? c : hidden) * 2));
  const size_t ab = af3_batch_diffusion_self_attention_workspace_bytes(batch, seq, c);
  void* aw = w.take(ab);
  if (!w.ok) return AF3_ERR_WORKSPACE;
  for (int i = 0; i < num_blocks; ++i) {
    const af3_diffusion_block& b = blocks[i];
    const float *ss = scale_shift + (int64_t)2 * i * 2 * c, *g = gate + (int64_t)2 * i * c;
    STEP(af3_layer_norm_forward(act, act_dtype, x, rows, c, nullptr, nullptr, ss, ss + c, cond_rows, ld_ss, stream));
    STEP(af3_batch_diffusion_self_attention_forward(x, key_mask, 1, pair_logits[i], bias_quad_major, b.w_q, b.q_b, num_head, y,
                                                    AF3_BF16, batch, seq, c, aw, ab, stream));
    STEP(af3_linear_forward(y, b.w_out, nullptr, act, act_dtype, rows, c, c, AF3_LINEAR_GATE_RES, 1.f, 0, g, cond_rows, ld_g, act,
                            act_dtype, stream));
    STEP(af3_layer_norm_forward(act, act_dtype, x, rows, c, nullptr, nullptr, ss + 2 * c, ss + 3 * c, cond_rows, ld_ss, stream));
    STEP(af3_linear_forward(x, b.w_tr1, nullptr, y, AF3_BF16, rows, 2 * hidden, c, AF3_LINEAR_SWIGLU, 1.f, 0, nullptr, 0, 0, nullptr, 0,
                            stream));
    STEP(af3_linear_forward(y, b.w_tr2, nullptr, act, act_dtype, rows, c, hidden, AF3_LINEAR_GATE_RES, 1.f, 0, g + c, cond_rows, ld_g,
                            act, act_dtype, stream));
  }
  return AF3_OK;
}

size_t af3_atom_transformer_workspace_bytes(int64_t samples, int64_t subsets, int64_t queries, int channels, int hidden) {
  if (samples <= 0 || subsets <= 0 || queries <= 0 || channels <= 0 || hidden <= 0) return 0;
  const size_t rows = (size_t)samples * subsets * queries;
  return 2 * align_up(rows * channels * 2) + align_up(rows * (channels > hidden ? channels : hidden) * 2) +
         align_up(af3_gathered_cross_attention_workspace_bytes(samples * subsets, queries, samples, subsets * queries, channels));
}

int af3_atom_transformer_forward(
    const af3_diffusion_block* blocks, int num_blocks, void* act, int act_dtype, int64_t samples, int64_t subsets,
    int64_t queries, int64_t keys, int channels, int hidden, int num_head, const int32_t* key_rows, const float* mask_q,
    const float* mask_k, const float* pair_logits, const float* scale_shift_q, const float* scale_shift_k, const float* gate,
    void* workspace, size_t workspace_bytes, af3_stream_t stream) {
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
  for (int i = 0; i < num_blocks; ++i) {
    const af3_diffusion_block& b = blocks[i];
    const float *ss = scale_shift_q + (int64_t)2 * i * 2 * c, *sk = scale_shift_k + (int64_t)i * 2 * c;
    const float* g = gate + (int64_t)2 * i * atoms * c;
    const float* pl = pair_logits ? pair_logits + (int64_t)i * subsets * num_head * queries * keys : nullptr;
    STEP(af3_layer_norm_forward(act, act_dtype, xq, rows, c, nullptr, nullptr, ss, ss + c, atoms, ld_q, stream));
    STEP(af3_layer_norm_forward(act, act_dtype, xk, rows, c, nullptr, nullptr, sk, sk + c, atoms, ld_k, stream));
    STEP(af3_gathered_cross_attention_forward(xq, xk, key_rows, pl, mask_q, mask_k, subsets, b.w_q, b.w_kv, b.q_b, num_head, y,
                                              AF3_BF16, samples * subsets, queries, keys, samples, atoms, c, aw, ab, stream));
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

}  // extern "C"
