// One transformer block from one host call: the launches of BasicTransformerBlock.forward in their order.
//
// Bound by the host before: about ten launches per block, each through its own wrapper (argument checks, an allocation per
// result, a 20-argument foreign call), 230 us of Python per block where the launches themselves take 3 us each -- more than
// the block's GPU time for images up to 768 x 768.  Everything that does not change from call to call (operands, shapes,
// flags) is laid out once in a KhBlockDesc; a call brings the activations, one workspace and the counters.  The kernels, their
// arguments and their order are those of the single entry points, which are what runs here.  A linear that is called by itself
// (kh_lora_linear_desc_bf16) saves the same checks.
#include "kh_common.h"
#include "../../include/katz_hip.h"

namespace {

struct Layout {   // byte offsets into the workspace
  int64_t wide, att, h1, h2, norm, k, v, t, bytes;
};

int64_t rank_columns(const KhLinearDesc& l) { return l.R == 0 ? 0 : l.n_split > 0 ? l.N / l.n_split * l.R : l.R; }

Layout layout(const KhBlockDesc& d, int64_t M, int64_t Mc, bool cross, bool own_kv) {
  const auto up = [](int64_t n) { return (n + 255) / 256 * 256; };
  const int64_t C = d.ff.N;
  int64_t t = 0;
  const auto rows = [&](const KhLinearDesc& l, int64_t m) { t = t > m * rank_columns(l) ? t : m * rank_columns(l); };
  rows(d.qkv, M); rows(d.out1, M); rows(d.geglu, M); rows(d.ff, M);
  if (cross) { rows(d.q2, M); rows(d.out2, M); }
  if (own_kv) { rows(d.k2, Mc); rows(d.v2, Mc); }
  const int64_t widest = d.qkv.N > d.geglu.N / 2 ? d.qkv.N : d.geglu.N / 2;   // q | k | v, then q alone, then the feed-forward's hidden rows
  Layout w{};
  int64_t at = 0;
  const auto take = [&](int64_t elements) { const int64_t p = at; at += up(elements * 2); return p; };
  w.wide = take(M * widest);
  w.att = take(M * (d.qkv.N / 3));
  w.h1 = take(M * C);
  w.h2 = take(cross ? M * C : 0);
  w.norm = take(d.folded ? 0 : M * C);
  w.k = take(own_kv ? Mc * d.k2.N : 0);
  w.v = take(own_kv ? Mc * d.v2.N : 0);
  w.t = take(t);
  w.bytes = at;
  return w;
}

int64_t counters_of(const KhLinearDesc& l, int64_t rows) { return l.R == 0 ? 0 : KH_SPLIT_COUNTER_INTS(rows); }

int64_t counter_ints(const KhBlockDesc& d, int64_t M, int64_t Mc, bool cross, bool own_kv) {
  int64_t n = counters_of(d.qkv, M) + counters_of(d.out1, M) + counters_of(d.geglu, M) + counters_of(d.ff, M);
  if (cross) n += counters_of(d.q2, M) + counters_of(d.out2, M);
  if (own_kv) n += counters_of(d.k2, Mc) + counters_of(d.v2, Mc);
  return n;
}

// The operands of the linear behind the one that is launched next, for kh_set_weight_prefetch.
void hint(const KhLinearDesc& next) {
  kh_set_weight_prefetch(nullptr, 0);
  if (next.hint_weight) kh_set_weight_prefetch(next.w, next.N * next.K * 2);
  if (next.R > 0) {
    kh_set_weight_prefetch(next.a_cat, rank_columns(next) * next.K * 2);
    kh_set_weight_prefetch(next.b_cat, next.N * next.R * 2);
  }
}

struct Run {
  const KhBlockCall& c;
  void* stream;
  char* ws;
  const Layout w;
  int32_t* counters;

  int32_t* take(const KhLinearDesc& l, int64_t rows) {   // (none where every linear is two launches)
    if (counters == nullptr) return nullptr;
    int32_t* p = l.R == 0 ? nullptr : counters;
    counters += counters_of(l, rows);
    return p;
  }
  int flags(const KhLinearDesc& l) const { return (l.geglu ? 1 : 0) | (l.R > 0 ? (int)(l.r_used / 16) << 16 : 0) | (int)c.flags; }

  int linear(const KhLinearDesc& l, const void* x, const void* residual, void* y, int64_t rows, const float* ln, float* stats,
             const KhLinearDesc* next) {
    if (c.hints) {
      if (next) hint(*next);
      else {
        kh_set_weight_prefetch(nullptr, 0);
        for (int i = 0; i < 3; ++i)
          if (c.tail_hint[2 * i]) kh_set_weight_prefetch((const void*)(uintptr_t)c.tail_hint[2 * i], (int64_t)c.tail_hint[2 * i + 1]);
      }
    }
    if (ln || stats)
      return kh_lora_linear_norm_bf16(x, l.w, ln ? nullptr : l.bias, l.a_cat, l.col_scale, l.b_cat, l.R ? ws + w.t : nullptr, take(l, rows), residual,
                                      y, ln, ln ? l.c1 : nullptr, ln ? l.c2 : nullptr, ln ? l.ca1 : nullptr, ln ? l.ca2 : nullptr, ln ? (float)l.eps : 0.f,
                                      stats, rows, l.N, l.K, l.R, l.R ? l.n_split : 0, flags(l), stream);
    if (l.R == 0) return kh_lora_linear_bf16(x, l.w, l.bias, nullptr, nullptr, nullptr, residual, y, rows, l.N, l.K, 0, l.geglu ? 1 : 0, stream);
    return kh_lora_linear_split_bf16(x, l.w, l.bias, l.a_cat, l.col_scale, l.b_cat, ws + w.t, take(l, rows), residual, y, rows, l.N, l.K, l.R,
                                     l.n_split, flags(l), stream);
  }
};

#define KH_STEP(call) \
  if (const int rc__ = (call); rc__ != KH_OK) return rc__

}  // namespace

KH_EXPORT int kh_lora_linear_desc_bf16(const KhLinearDesc* l, const void* x, const void* residual, void* y, void* t_scratch, int32_t* counters,
                                       int64_t M, int flags, void* stream) {
  if (!l) return KH_ERR_INVALID_ARG;
  if (l->R == 0) return kh_lora_linear_bf16(x, l->w, l->bias, nullptr, nullptr, nullptr, residual, y, M, l->N, l->K, 0, l->geglu ? 1 : 0, stream);
  return kh_lora_linear_split_bf16(x, l->w, l->bias, l->a_cat, l->col_scale, l->b_cat, t_scratch, counters, residual, y, M, l->N, l->K, l->R, l->n_split,
                                   (l->geglu ? 1 : 0) | (int)(l->r_used / 16) << 16 | flags, stream);
}

KH_EXPORT int kh_transformer_block_needs(const KhBlockDesc* d, int64_t B, int64_t T, int64_t S, int own_kv, int64_t* workspace_bytes, int64_t* counters) {
  if (!d || B <= 0 || T <= 0 || S < 0 || !workspace_bytes || !counters) return KH_ERR_INVALID_ARG;
  const bool cross = d->q2.w != nullptr;
  *workspace_bytes = layout(*d, B * T, B * S, cross, cross && own_kv).bytes;
  *counters = counter_ints(*d, B * T, B * S, cross, cross && own_kv);
  return KH_OK;
}

KH_EXPORT int kh_transformer_block_bf16(const KhBlockDesc* desc, const KhBlockCall* call, void* stream) {
  if (!desc || !call) return KH_ERR_INVALID_ARG;
  const KhBlockDesc& d = *desc;
  const KhBlockCall& c = *call;
  const bool cross = d.q2.w != nullptr, own_kv = cross && c.ctx != nullptr;
  const int64_t M = c.B * c.T, Mc = c.B * c.S, C = d.ff.N, inner = d.qkv.N / 3;
  if (!c.x || !c.y || !c.workspace || c.B <= 0 || c.T <= 0 || (d.folded && !c.stats)) return KH_ERR_INVALID_ARG;
  if (cross && (c.S <= 0 || (!own_kv && (!c.k || !c.v)))) return KH_ERR_INVALID_ARG;
  // the shapes the chain assumes: every width is checked once more by the entry point that uses it
  if (d.qkv.N % 3 != 0 || inner != d.heads * 64 || d.qkv.K != C || d.out1.K != inner || d.out1.N != C || d.geglu.K != C || d.ff.K * 2 != d.geglu.N ||
      (cross && (d.q2.K != C || d.q2.N != inner || d.out2.K != inner || d.out2.N != C)) ||
      (own_kv && (d.k2.N != inner || d.v2.N != inner || d.v2.K != d.k2.K)))
    return KH_ERR_INVALID_ARG;
  const Layout w = layout(d, M, Mc, cross, own_kv);
  if (w.bytes > c.workspace_bytes || !kh_aligned16(c.workspace)) return KH_ERR_INVALID_ARG;
  const bool waits = (c.flags & ((1 << 8) | (1 << 24))) == 0;
  const int64_t ints = waits ? counter_ints(d, M, Mc, cross, own_kv) : 0;
  if (ints > c.counter_ints || (ints > 0 && !c.counters)) return KH_ERR_INVALID_ARG;
  Run r{c, stream, (char*)c.workspace, w, waits ? c.counters : nullptr};
  char* const ws = r.ws;
  const float* const ln = d.folded ? c.stats : nullptr;
  float* const stats = d.folded ? c.stats : nullptr;
  // a norm that is not folded into the linear behind it is a launch of its own
  const void* x = c.x;
  const auto normed = [&](const void* rows, const void* weight, const void* bias, float eps, const void** out) {
    *out = rows;
    if (d.folded) return KH_OK;
    *out = ws + w.norm;
    return kh_layer_norm_bf16(rows, ws + w.norm, weight, bias, M, C, eps, stream);
  };
  const KhLinearDesc* const after_out1 = !cross ? &d.geglu : own_kv ? &d.k2 : &d.q2;
  const void* n;
  // self-attention
  KH_STEP(normed(x, d.n1_w, d.n1_b, (float)d.n1_eps, &n));
  KH_STEP(r.linear(d.qkv, n, nullptr, ws + w.wide, M, ln, nullptr, &d.out1));
  const int64_t ld3 = d.qkv.N;
  KH_STEP(kh_attention_bf16(ws + w.wide, ws + w.wide + 2 * inner, ws + w.wide + 4 * inner, ws + w.att, c.B, d.heads, c.T, c.T, 64, ld3, ld3, ld3, inner,
                            ld3 * c.T, ld3 * c.T, ld3 * c.T, inner * c.T, (float)d.scale1, stream));
  KH_STEP(r.linear(d.out1, ws + w.att, x, ws + w.h1, M, nullptr, stats, after_out1));
  const void* h = ws + w.h1;
  // attention over the context
  if (cross) {
    KH_STEP(normed(h, d.n2_w, d.n2_b, (float)d.n2_eps, &n));
    const void *k = c.k, *v = c.v;
    int64_t ldk = c.ldk, ldv = c.ldv, bsk = c.bsk, bsv = c.bsv;
    if (own_kv) {
      KH_STEP(r.linear(d.k2, c.ctx, nullptr, ws + w.k, Mc, nullptr, nullptr, &d.v2));
      KH_STEP(r.linear(d.v2, c.ctx, nullptr, ws + w.v, Mc, nullptr, nullptr, &d.q2));
      k = ws + w.k; v = ws + w.v; ldk = ldv = inner; bsk = bsv = inner * c.S;
    }
    const KhLinearDesc& q = d.q2;
    if (d.fuse_xattn && kh_lora_linear_xattn_ok(M, q.N, q.K, q.R, c.T, c.S)) {
      if (c.hints) hint(d.out2);
      KH_STEP(kh_lora_linear_xattn_bf16(n, q.w, ln ? nullptr : q.bias, q.a_cat, q.col_scale, q.b_cat, q.R ? ws + w.t : nullptr, r.take(q, M), ln,
                                        ln ? q.c1 : nullptr, ln ? q.c2 : nullptr, ln ? q.ca1 : nullptr, ln ? q.ca2 : nullptr, ln ? (float)q.eps : 0.f, k, v,
                                        ws + w.att, M, q.N, q.K, q.R, c.T, c.S, ldk, ldv, inner, bsk, bsv, (float)d.scale2, r.flags(q), stream));
    } else {
      KH_STEP(r.linear(q, n, nullptr, ws + w.wide, M, ln, nullptr, &d.out2));
      KH_STEP(kh_attention_bf16(ws + w.wide, k, v, ws + w.att, c.B, d.heads, c.T, c.S, 64, inner, ldk, ldv, inner, inner * c.T, bsk, bsv, inner * c.T,
                                (float)d.scale2, stream));
    }
    KH_STEP(r.linear(d.out2, ws + w.att, h, ws + w.h2, M, nullptr, stats, &d.geglu));
    h = ws + w.h2;
  }
  // feed-forward
  KH_STEP(normed(h, d.n3_w, d.n3_b, (float)d.n3_eps, &n));
  KH_STEP(r.linear(d.geglu, n, nullptr, ws + w.wide, M, ln, nullptr, &d.ff));
  return r.linear(d.ff, ws + w.wide, h, c.y, M, nullptr, c.last ? nullptr : stats, nullptr);
}
