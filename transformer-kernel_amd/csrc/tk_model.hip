// The layer loop of the forward as one host call (no kernels of its own).
//
// One forward is 1 + 4..7 launches per layer.  Issued one by one from Python,
// each cost 10-12 us of host time (argument conversion, output views, one
// allocation per intermediate), more than most kernels of a single short
// sequence run: a one-layer forward at B1 S512 D1024 took 94 us of host
// time for ~65 us of kernels, B2 S64 D384 85 us for ~35.  Here the same launches, in
// the same order with the same arguments, cost the runtime's launch itself.
//
// The schedule is a list of steps, so a caller that times each launch runs
// it one step at a time and the order is written down once.
#include "tk_common.hpp"

namespace tk {
namespace {

enum StepKind {
  kLnIn, kQkv, kAttn, kQkvAttn, kOutLn, kOutResid, kLn2, kUp, kDownLn, kDownResid, kLnNext, kLnFinal, kLnQkv, kTail
};
const char* const kStepNames[] = {"ln_in", "qkv", "flash_attn", "qkv_attn", "out_proj_ln", "out_proj_resid",
                                  "ln2", "ffn_up_gelu", "ffn_down_ln", "ffn_down_resid", "ln_next", "ln_final",
                                  "ln_qkv", "block_tail"};

struct Schedule {
  bool fused_qa;  // QKV projection and attention in one kernel
  bool fuse;      // residual GEMM + LayerNorm as one step (tk_gemm_bias_add_ln)
  bool narrow;    // every row-local part of a block in one kernel
  int per_layer;
  int64_t layers;
  int64_t steps() const { return (narrow ? 0 : 1) + layers * per_layer; }
  int64_t layer_of(int64_t step) const {
    return narrow ? step / per_layer : step == 0 ? 0 : (step - 1) / per_layer;
  }
  StepKind kind(int64_t step) const {
    if (narrow) return step == 0 ? kLnQkv : step % per_layer == 0 ? kQkv : step % per_layer == 1 ? kAttn : kTail;
    if (step == 0) return kLnIn;
    const int64_t layer = (step - 1) / per_layer;
    int k = (int)((step - 1) % per_layer);
    if (fused_qa) {
      if (k == 0) return kQkvAttn;
      --k;
    } else {
      if (k < 2) return k == 0 ? kQkv : kAttn;
      k -= 2;
    }
    if (fuse) return k == 0 ? kOutLn : k == 1 ? kUp : kDownLn;
    if (k < 4) return k == 0 ? kOutResid : k == 1 ? kLn2 : k == 2 ? kUp : kDownResid;
    return layer + 1 < layers ? kLnNext : kLnFinal;
  }
};

Schedule schedule(const tk_model& m, int64_t batch, int64_t seq, bool dense, int flags) {
  Schedule s;
  // The fused kernel reads h as [T, heads * head_dim]: unpadded head dims only.
  s.fused_qa = dense && (flags & TK_FWD_QKV_ATTENTION) && m.heads * m.head_dim == m.d_model &&
               tk_qkv_attention_supported(batch, seq, m.heads, m.head_dim);
  s.fuse = (flags & TK_FWD_FUSED_NORM) && tk_gemm_ln_supported(m.d_model);
  // The narrow kernels read b_1 in 16-byte vectors; the separate launches take it at any address
  // (a parameter that is a view into a flat buffer).
  bool packed = true;
  for (int64_t i = 0; i < m.num_layers; ++i)
    packed = packed && m.layers[i].w_qkv_packed && m.layers[i].w_o_packed && m.layers[i].w_1_packed &&
             m.layers[i].w_2_packed && ((uintptr_t)m.layers[i].b_1 & 15) == 0;
  s.narrow = packed && (flags & TK_FWD_FUSED_NORM) &&
             tk_narrow_supported(m.d_model, m.heads * m.head_dim, m.ffn_dim);
  // Which of the two runs where both take the model depends on the batch (the fused kernel takes
  // even ones), and their LayerNorm statistics and residual sums round differently.
  if (flags & TK_FWD_BATCH_INVARIANT) s.fused_qa = s.fused_qa && !s.narrow;
  else s.narrow = s.narrow && !s.fused_qa;
  s.per_layer = s.narrow ? 3 : (s.fused_qa ? 1 : 2) + (s.fuse ? 3 : 5);
  s.layers = m.num_layers;
  return s;
}

// Intermediates of a forward, 256-byte aligned in the caller's workspace.  The
// q|k|v rows are dead once attention has run and the FFN's hidden rows live
// from the FFN-up to the FFN-down GEMM, so the two share their bytes.
struct Layout {
  int64_t resid, h, ctx, shared, bytes;
};
Layout layout(const tk_model& m, int64_t t, const Schedule& s) {
  auto up = [](int64_t b) { return (b + 255) & ~(int64_t)255; };
  const int64_t dp = m.heads * m.head_dim;
  Layout l;
  l.resid = 0;
  l.h = l.resid + up(t * m.d_model * 4);
  l.ctx = l.h + up(t * m.d_model * 2);
  l.shared = l.ctx + up(t * dp * 2);
  const int64_t qkv = s.fused_qa ? 0 : t * 3 * dp * 2, u = t * m.ffn_dim * 2;
  l.bytes = l.shared + up(qkv > u ? qkv : u);
  return l;
}

int check_model(const tk_model* m, int64_t batch, int64_t seq, const char* who) {
  TK_REQUIRE(m && m->layers && m->nf_w && m->nf_b, TK_ERR_ARG, "%s: null model", who);
  TK_REQUIRE(m->d_model > 0 && m->heads > 0 && m->head_dim > 0 && m->ffn_dim > 0 && m->num_layers > 0 &&
                 m->d_model < (1ll << 24) && m->heads < (1ll << 24) && m->head_dim < (1ll << 24) &&
                 m->ffn_dim < (1ll << 24),
             TK_ERR_ARG, "%s: bad model sizes", who);
  TK_REQUIRE(batch >= 0 && seq >= 0 && batch < (1ll << 31) && seq < (1ll << 31) && batch * seq < (1ll << 31),
             TK_ERR_ARG, "%s: bad batch=%lld seq=%lld", who, (long long)batch, (long long)seq);
  return TK_OK;
}

}  // namespace
}  // namespace tk

using namespace tk;

extern "C" int64_t tk_forward_workspace(const tk_model* m, int64_t batch, int64_t seq, int dense, int flags) {
  if (int rc = check_model(m, batch, seq, "tk_forward_workspace")) return rc;
  return layout(*m, batch * seq, schedule(*m, batch, seq, dense != 0, flags)).bytes;
}

extern "C" int64_t tk_forward_steps(const tk_model* m, int64_t batch, int64_t seq, int dense, int flags) {
  if (int rc = check_model(m, batch, seq, "tk_forward_steps")) return rc;
  return schedule(*m, batch, seq, dense != 0, flags).steps();
}

extern "C" const char* tk_forward_step_name(const tk_model* m, int64_t batch, int64_t seq, int dense, int flags,
                                            int64_t step) {
  if (check_model(m, batch, seq, "tk_forward_step_name")) return nullptr;
  const Schedule s = schedule(*m, batch, seq, dense != 0, flags);
  return step >= 0 && step < s.steps() ? kStepNames[s.kind(step)] : nullptr;
}

extern "C" int tk_forward(const tk_model* m, const void* x, void* out, int64_t batch, int64_t seq,
                          const uint8_t* valid, void* workspace, int64_t workspace_bytes, int flags,
                          int64_t first_step, int64_t num_steps, void* stream) {
  if (int rc = check_model(m, batch, seq, "tk_forward")) return rc;
  TK_REQUIRE(x && out && workspace, TK_ERR_ARG, "tk_forward: null pointer");
  const Schedule s = schedule(*m, batch, seq, valid == nullptr, flags);
  const int64_t t = batch * seq, d = m->d_model, f = m->ffn_dim, nh = m->heads, hd = m->head_dim, dp = nh * hd;
  const Layout l = layout(*m, t, s);
  TK_REQUIRE(workspace_bytes >= l.bytes && ((uintptr_t)workspace & 255) == 0, TK_ERR_ARG,
             "tk_forward: workspace of %lld bytes at %p; %lld bytes, 256-byte aligned, needed",
             (long long)workspace_bytes, workspace, (long long)l.bytes);
  TK_REQUIRE((flags & ~31) == 0, TK_ERR_ARG, "tk_forward: unknown flags %d", flags);
  const bool io16 = flags & (TK_FWD_IO_F16 | TK_FWD_IO_BF16), bf16 = flags & TK_FWD_IO_BF16;
  TK_REQUIRE(!io16 || (!s.fuse && !s.narrow), TK_ERR_UNSUPPORTED,
             "tk_forward: 16-bit x and out need the schedule without TK_FWD_FUSED_NORM");
  TK_REQUIRE((flags & (TK_FWD_IO_F16 | TK_FWD_IO_BF16)) != (TK_FWD_IO_F16 | TK_FWD_IO_BF16), TK_ERR_ARG,
             "tk_forward: x is either fp16 or bf16");
  const int64_t steps = s.steps();
  if (num_steps < 0) num_steps = steps - first_step;
  TK_REQUIRE(first_step >= 0 && num_steps >= 0 && first_step + num_steps <= steps, TK_ERR_ARG,
             "tk_forward: steps [%lld, %lld) of %lld", (long long)first_step, (long long)(first_step + num_steps),
             (long long)steps);
  char* ws = static_cast<char*>(workspace);
  float* resid = reinterpret_cast<float*>(ws + l.resid);
  tk_half* h = reinterpret_cast<tk_half*>(ws + l.h);
  tk_half* ctx = reinterpret_cast<tk_half*>(ws + l.ctx);
  tk_half* qkv = reinterpret_cast<tk_half*>(ws + l.shared);
  tk_half* u = qkv;
  const bool invariant = flags & TK_FWD_BATCH_INVARIANT;
  const int64_t in_st[3] = {seq * 3 * dp, hd, 3 * dp}, out_st[3] = {seq * dp, hd, dp};
  for (int64_t i = first_step; i < first_step + num_steps; ++i) {
    const int64_t li = s.layer_of(i);
    const tk_layer& w = m->layers[li];
    const bool last = li + 1 == m->num_layers;
    // Residual input of the first layer's attention update: the caller's x, which is never
    // written (16-bit: its fp32 copy, left by the first LayerNorm).
    const float* x32 = static_cast<const float*>(x);
    const float* src = li == 0 && !io16 ? x32 : resid;
    // What the LayerNorm after the FFN is: the next block's first, or the final one (fp32, into out).
    const float* nw = last ? m->nf_w : m->layers[li + 1].n1_w;
    const float* nb = last ? m->nf_b : m->layers[li + 1].n1_b;
    const float ne = last ? m->nf_eps : m->layers[li + 1].n1_eps;
    void* ndst = last ? out : static_cast<void*>(h);
    const int ndt = last && !io16 ? TK_F32 : TK_F16;
    int rc = TK_OK;
    switch (s.kind(i)) {
      case kLnIn:
        if (io16) rc = ln_first16(x, bf16, w.n1_w, w.n1_b, resid, h, t, d, w.n1_eps, stream);
        else rc = tk_ln_cast(x32, w.n1_w, w.n1_b, h, TK_F16, t, d, w.n1_eps, nullptr, stream);
        break;
      case kQkv:
        rc = gemm(h, d, w.w_qkv, d, w.b_qkv, nullptr, 0, qkv, 3 * dp, t, 3 * dp, d, TK_EPI_BIAS, nullptr, 0, invariant,
                  stream);
        break;
      case kAttn:
        rc = flash_attn(qkv, qkv + dp, qkv + 2 * dp, ctx, batch, nh, seq, hd, in_st, in_st, in_st, out_st, m->scale,
                        m->causal, valid, seq, invariant, stream);
        break;
      case kQkvAttn:
        rc = tk_qkv_attention(h, d, w.w_qkv, d, w.b_qkv, ctx, dp, batch, seq, nh, hd, m->scale, m->causal, stream);
        break;
      case kOutLn:
        rc = gemm_bias_add_ln(ctx, dp, w.w_o, dp, w.b_o, src, w.n2_w, w.n2_b, resid, h, TK_F16, t, d, dp, w.n2_eps,
                              valid, valid ? TK_ROWS_KEEP_RESID : 0, invariant, stream);
        break;
      case kOutResid:
        rc = gemm(ctx, dp, w.w_o, dp, w.b_o, src, d, resid, d, t, d, dp, TK_EPI_BIAS_RESID, valid,
                  valid ? TK_ROWS_KEEP_RESID : 0, invariant, stream);
        break;
      case kLn2:
        rc = tk_ln_cast(resid, w.n2_w, w.n2_b, h, TK_F16, t, d, w.n2_eps, nullptr, stream);
        break;
      case kUp:
        rc = gemm(h, d, w.w_1, d, w.b_1, nullptr, 0, u, f, t, f, d, TK_EPI_BIAS_GELU, nullptr, 0, invariant, stream);
        break;
      case kDownLn:
        rc = gemm_bias_add_ln(u, f, w.w_2, f, w.b_2, resid, nw, nb, resid, ndst, ndt, t, d, f, ne, valid,
                              valid ? (last ? TK_ROWS_ZERO_ALL : TK_ROWS_ZERO) : 0, invariant, stream);
        break;
      case kDownResid:
        rc = gemm(u, f, w.w_2, f, w.b_2, resid, d, resid, d, t, d, f, TK_EPI_BIAS_RESID, valid,
                  valid ? TK_ROWS_ZERO : 0, invariant, stream);
        break;
      case kLnQkv:
        rc = tk_narrow_qkv(x32, w.n1_w, w.n1_b, w.n1_eps, w.w_qkv_packed, w.b_qkv, qkv, t, stream);
        break;
      case kTail:
        rc = tk_narrow_tail(ctx, src, w.w_o_packed, w.b_o, w.n2_w, w.n2_b, w.n2_eps, w.w_1_packed, w.b_1,
                            w.w_2_packed, w.b_2, f, nw, nb, ne, last ? nullptr : resid, ndst, ndt, t, valid,
                            valid ? (last ? TK_ROWS_ZERO_ALL : TK_ROWS_ZERO) : 0, stream);
        break;
      case kLnNext:
      case kLnFinal:
        if (last && bf16) rc = ln_last_bf16(resid, nw, nb, ndst, t, d, ne, valid, stream);
        else rc = tk_ln_cast(resid, nw, nb, ndst, ndt, t, d, ne, last ? valid : nullptr, stream);
        break;
    }
    if (rc != TK_OK) return rc;
  }
  return TK_OK;
}
