// Whole-step entry points of the layered language models: a list of layers, each a token mixer and a gated feed-forward or a mixture
// of experts, as a sequence of this library's launches.  Nothing here allocates or synchronises.
//
// Prefill (more than 128 rows):  residual add + norm | input projection | mixer kernels | output projection | residual add + norm |
//   gate/up GEMM with silu(gate) * up | down GEMM, the adds deferred into the next norm so that the fp32 residual is read and written
//   once per half layer.
// Where the tiles of a projection leave CUs idle (bf16), it leaves fp32 K-slice partials (md_gemm_partial_rows) which the row-wise step
//   behind it sums: out / down -> residual add + norm; up to 128 rows also gate_up -> silu(gate) * up (otherwise the product's epilogue).
// Few rows (LM_STEP_ROWS, bf16):  gemm_step.hip's products, which go on with the row-wise step themselves.
// Experts:  router + choice | rows grouped by expert | grouped gate/up product with silu(gate) * up | grouped down product; the weighted sum
//   of a row's experts is taken by the row-wise step that follows, as the sums of K-slice partials are.  Few rows per expert: gemm_experts.hip's
//   products, which take the choices as they are.
//   A step of few rows norms nothing whole there either: the router and the experts' first product take the rows' factors themselves.
// Residual streams:  the row-wise step between two sublayers mixes them (streams.hip); x is then [streams][rows][width_pad].
#include "gemm_internal.hpp"
#include "lm_internal.hpp"
#include "stage_common.hpp"

#include <algorithm>

namespace {

int g_lm_kernels = 3;

constexpr int DECODE_ROWS = 128;  // most rows of the decode regime

inline size_t esize(const md_lm_model* m) { return m->dtype == MD_DTYPE_F32 ? 4 : 2; }

struct LmWs {
  float* x;
  char *h, *proj, *q, *att, *y, *gu, *act;
  float *part, *qf, *kf, *of, *ret_seg, *attn_part;
  char *c_rows, *kv, *q_lat, *conv_out;
  float *latent_part, *dt, *seg, *seg_decay, *route_weight, *sumsq, *row_factor, *head_sumsq;
  int32_t *chosen, *slot_of, *row_of, *offsets;
  void* splitk;
  size_t splitk_bytes;
  int64_t part_floats;
  size_t total;
};

inline bool decode_regime(const md_lm_model* m, int rows) { return m->dtype == MD_DTYPE_BF16 && rows <= DECODE_ROWS; }

// products that go on with the row-wise step behind them (gemm_step.hip)
// (Experts: where their own products take the step.  The first token's retention is its value times q . k, normed: only
// the sign of q . k is left, so a rounding of the norm at another place turns it over where q . k is small.  A step in which any sequence may
// begin keeps the rounding of long prompts where a layer has retention: 12 tokens 1.78 ms, 1.29 this way.  Their sums and gates take no bias.)
inline bool step_regime(const md_lm_model* m, const md_lm_batch* b) {
  if (m->dtype != MD_DTYPE_BF16 || b->n_rows > lm_step_most_rows(m->width_pad)) return false;
  for (int i = 0; i < m->n_layers; ++i) {
    const md_lm_layer& l = m->layers[i];
    if (l.experts > 0 && !lm_expert_step_takes(b->n_rows, l.top, l.experts)) return false;
    if (l.out_proj.b || (l.ff > 0 && (l.gate_up.b || l.down.b))) return false;
    if (b->n_going != b->n_seq && l.mixer == MD_MIXER_RETENTION) return false;
  }
  return true;
}

inline bool own_row_steps(const md_lm_model* m) { return m->streams > 0 || m->pos || m->embed_norm.w; }
inline int n_streams(const md_lm_model* m) { return m->streams > 0 ? m->streams : 1; }
inline int conv_columns(const md_lm_layer& l) { return l.heads * l.vdim_pad + 2 * l.groups * l.dim_pad; }

// What splits its sums wants more memory at fewer rows: there is room for what any smaller step of the same kind (one token per sequence, or
// prompts) would want, so that a workspace of the largest step serves all.
LmWs layout(const md_lm_model* m, const md_lm_batch* b, int n_logits, void* base) {
  const int rows = b->n_rows, n_seq = b->n_seq, max_len = b->max_len, max_ctx = b->max_ctx;
  const size_t es = esize(m), M = rows;
  size_t in = 0, q = 0, att = 0, gu = 0, act = 0, qf = 0, of = 0, rs = 0, ap = 0, sk = 0, part = 0, y = M * m->width_pad;
  size_t c_rows = 0, kv = 0, q_lat = 0, lp = 0, conv = 0, dt = 0, seg = 0, segs = 0, slots = 0, experts = 0;
  size_t sk_room = 0, ssm_heads = 0;
  auto splitk = [&](const md_linear& l, int n) {
    if (m->dtype != MD_DTYPE_BF16 || !l.w || n <= 0) return;
    sk = std::max(sk, md_gemm_workspace_bytes(&l, n, 1));
    sk_room = std::max(sk_room, md_gemm_workspace_bytes(&l, std::min(n, DECODE_ROWS), 1));
  };
  auto partial = [&](const md_linear& l, bool residual) {
    if (m->dtype == MD_DTYPE_BF16 && l.w) part = std::max(part, md_gemm_partial_most(l, residual ? rows : std::min(rows, DECODE_ROWS)));
  };
  for (int i = 0; i < m->n_layers; ++i) {
    const md_lm_layer& l = m->layers[i];
    in = std::max(in, (size_t)l.in_proj.n_pad);
    att = std::max(att, (size_t)l.out_proj.k_pad);
    partial(l.in_proj, true);
    partial(l.out_proj, true);
    if (l.experts > 0) {
      const size_t T = M * l.top;
      slots = std::max(slots, T);
      experts = std::max(experts, (size_t)l.experts);
      if (m->dtype == MD_DTYPE_F32) gu = std::max(gu, T * l.gate_up.n_pad);
      act = std::max(act, T * l.down.k_pad);
      y = std::max(y, T * m->width_pad);
      const int most = std::min(rows, DECODE_ROWS) * l.top;
      if (m->dtype == MD_DTYPE_BF16)
        part = std::max(part, std::max(md_gemm_grouped_most(l.gate_up, l.experts, most), md_gemm_grouped_most(l.down, l.experts, most)));
    } else if (l.ff > 0) {
      if (m->dtype == MD_DTYPE_F32 || l.gate_up.b) gu = std::max(gu, M * l.gate_up.n_pad);
      act = std::max(act, M * l.down.k_pad);
      partial(l.gate_up, false);
      partial(l.down, true);
    }
    if (l.mixer == MD_MIXER_ATTENTION) {
      q = std::max(q, (size_t)l.heads * l.dim_pad);
      const int span = l.chunk > 0 ? std::min(l.chunk, max_ctx) : max_ctx;
      if (max_len > 1 && m->dtype == MD_DTYPE_BF16)
        ap = std::max({ap, lm_attn_mfma_part_floats_most(rows, n_seq, span, l.heads, l.vdim_pad), lm_attn_pairs_floats_most(rows, n_seq, span, l.heads, l.dim_pad, l.vdim_pad)});
      if (max_len == 1) {
        int keys;
        const int ns = lm_attn_decode_splits(n_seq, span, &keys);
        ap = std::max(ap, lm_attn_decode_part_floats(n_seq, ns, l.heads, l.vdim_pad));
        ap = std::max(ap, lm_attn_heads_floats(n_seq, span, l.heads, l.kv_heads, l.dim_pad, l.vdim_pad, l.taps, l.kv_layer == i));
      }
    } else if (l.mixer == MD_MIXER_LATENT) {
      if (m->dtype != MD_DTYPE_BF16) continue;
      if (max_len > 1) {
        c_rows = std::max(c_rows, (size_t)b->ctx_rows * l.rank_pad);
        kv = std::max(kv, (size_t)b->ctx_rows * l.up_kv.n_pad);
        splitk(l.up_kv, b->ctx_rows);
      } else {
        const int ns = lm_latent_decode_splits(n_seq, l.heads, max_ctx);
        q_lat = std::max(q_lat, (size_t)n_seq * l.heads * l.rank_pad);
        lp = std::max(lp, lm_latent_decode_part_floats(n_seq, ns, l.heads, l.rank_pad));
      }
    } else if (l.mixer == MD_MIXER_STATE_SPACE) {
      conv = std::max(conv, M * conv_columns(l));
      dt = std::max(dt, M * l.heads);
      ssm_heads = std::max(ssm_heads, (size_t)l.heads);
      if (m->dtype == MD_DTYPE_BF16) {
        const size_t ns = lm_ssm_most_segments(n_seq, l.heads, max_len);
        segs = std::max(segs, ns * l.heads);
        seg = std::max(seg, ns * l.heads * l.dim_pad * l.vdim_pad);
      }
    } else {
      qf = std::max(qf, (size_t)l.heads * l.dim_pad);
      of = std::max(of, (size_t)l.heads * l.vdim_pad);
      if (m->dtype == MD_DTYPE_BF16) rs = std::max(rs, (size_t)lm_ret_most_states(n_seq, l.heads, l.dim_pad, l.vdim_pad, max_len) * l.heads * l.dim_pad * l.vdim_pad);
    }
  }
  splitk(m->head, n_logits);
  Arena a{(char*)base, 0};
  LmWs w;
  w.x = (float*)a.take(n_streams(m) * M * m->width_pad * 4);
  w.h = (char*)a.take(std::max(M, (size_t)n_logits) * m->width_pad * es);
  w.proj = (char*)a.take(M * in * es);
  w.q = (char*)a.take(M * q * es);
  w.att = (char*)a.take(M * att * es);
  w.y = (char*)a.take(y * es);
  w.gu = (char*)a.take(gu * es);
  w.act = (char*)a.take(act * es);
  w.part = (float*)a.take(part * 4);
  w.part_floats = (int64_t)part;
  w.splitk = a.take(sk_room);
  w.splitk_bytes = sk;
  w.attn_part = (float*)a.take(ap * 4);
  // the plain retention kernels' rotated rows and the matrix-core kernels' segment states are never live together
  float* r = (float*)a.take(std::max(M * (2 * qf + of), rs) * 4);
  w.qf = r;
  w.kf = r + M * qf;
  w.of = r + 2 * M * qf;
  w.ret_seg = r;
  w.c_rows = (char*)a.take(c_rows * es);
  w.kv = (char*)a.take(kv * es);
  w.q_lat = (char*)a.take(q_lat * es);
  w.latent_part = (float*)a.take(lp * 4);
  w.conv_out = (char*)a.take(conv * es);
  w.dt = (float*)a.take(dt * 4);
  w.seg = (float*)a.take(seg * 4);
  w.seg_decay = (float*)a.take(segs * 4);
  w.route_weight = (float*)a.take(slots * 4);
  w.chosen = (int32_t*)a.take(slots * 4);
  w.slot_of = (int32_t*)a.take(slots * 4);
  w.row_of = (int32_t*)a.take(slots * 4);
  w.offsets = (int32_t*)a.take(slots ? (experts + 1) * 4 : 0);
  w.sumsq = (float*)a.take(m->dtype == MD_DTYPE_BF16 ? (size_t)std::min(rows, LM_STEP_ROWS) * (m->width_pad / 8) * 4 : 0);
  w.row_factor = (float*)a.take(slots ? (size_t)std::min(rows, LM_STEP_ROWS) * 4 : 0);
  w.head_sumsq = (float*)a.take(conv && m->dtype == MD_DTYPE_BF16 ? (size_t)std::min(rows, LM_STEP_ROWS) * ssm_heads * 4 : 0);
  w.total = a.off;
  return w;
}

md_status check_linear(const md_linear& l, int k_pad) {
  MD_CHECK_ARG(l.w && l.n == l.n_pad && l.n_pad > 0 && l.n_pad % 64 == 0 && l.k_pad == k_pad);
  return MD_OK;
}

md_status check_model(const md_lm_model* m, const md_lm_state* st) {
  MD_CHECK_ARG(m && m->layers && m->n_layers > 0 && m->embed && m->final_norm.w);
  MD_CHECK_ARG(m->dtype == MD_DTYPE_BF16 || m->dtype == MD_DTYPE_F32);
  MD_CHECK_ARG(m->width > 0 && m->width_pad >= m->width && m->width_pad % 64 == 0 && m->vocab > 0);
  MD_TRY(check_linear(m->head, m->width_pad));
  MD_CHECK_ARG(m->head.n_pad >= m->vocab && m->streams >= 0 && m->streams <= MD_LM_MAX_STREAMS && (!m->pos || m->positions > 0));
  for (int i = 0; i < m->n_layers; ++i) {
    const md_lm_layer& l = m->layers[i];
    MD_CHECK_ARG(l.heads > 0 && l.dim > 0 && l.vdim > 0 && l.dim_pad % 32 == 0 && l.vdim_pad % 32 == 0 && l.dim_pad >= l.dim && l.vdim_pad >= l.vdim);
    MD_CHECK_ARG(l.norm1.w && l.col_q >= 0 && l.col_q + (l.mixer == MD_MIXER_STATE_SPACE ? l.groups : l.heads) * l.dim_pad <= l.in_proj.n_pad && l.col_q % 4 == 0);
    MD_TRY(check_linear(l.in_proj, m->width_pad));
    MD_CHECK_ARG(l.out_proj.w && l.out_proj.n == l.out_proj.n_pad && l.out_proj.n_pad == m->width_pad && l.out_proj.k_pad >= l.heads * l.vdim_pad && l.out_proj.k_pad % 64 == 0);
    MD_CHECK_ARG(l.ff == 0 || (l.norm2.w && l.ff_pad >= l.ff && l.ff_pad % 64 == 0));
    if (l.ff > 0) {
      MD_TRY(check_linear(l.gate_up, m->width_pad));
      MD_TRY(check_linear(l.down, l.ff_pad));
      MD_CHECK_ARG(l.gate_up.n_pad == 2 * l.ff_pad && l.down.n_pad == m->width_pad);
    }
    if (l.experts > 0) {
      MD_TRY(check_linear(l.router, m->width_pad));
      MD_CHECK_ARG(l.ff > 0 && l.top > 0 && l.top <= l.experts && l.router.n_pad >= l.experts && l.router_bias);
    }
    MD_CHECK_ARG(m->streams == 0 || (l.mix1 && (l.ff == 0 || l.mix2)));
    if (l.mixer == MD_MIXER_ATTENTION) {
      MD_CHECK_ARG(l.kv_heads > 0 && l.heads % l.kv_heads == 0 && l.taps >= 1 && l.conv && l.q_norm && l.slope && l.head_mix && l.chunk >= 0);
      MD_CHECK_ARG(l.kv_layer >= 0 && l.kv_layer <= i && m->layers[l.kv_layer].mixer == MD_MIXER_ATTENTION);
      const md_lm_layer& o = m->layers[l.kv_layer];
      MD_CHECK_ARG(o.kv_layer == l.kv_layer && o.kv_heads == l.kv_heads && o.dim_pad == l.dim_pad && o.vdim_pad == l.vdim_pad);
      if (l.kv_layer == i)
        MD_CHECK_ARG(l.k_norm && l.col_k >= 0 && l.col_v >= 0 && l.col_k % 4 == 0 && l.col_v % 4 == 0 &&
                     l.col_k + l.kv_heads * l.dim_pad <= l.in_proj.n_pad && l.col_v + l.kv_heads * l.vdim_pad <= l.in_proj.n_pad);
      MD_CHECK_ARG(st->layers[l.kv_layer].k && st->layers[l.kv_layer].v && (l.taps == 1 || st->layers[i].conv));
    } else if (l.mixer == MD_MIXER_RETENTION) {
      MD_CHECK_ARG(l.decay && (l.rot_dims == 0 || l.rope) && l.rot_dims >= 0 && l.rot_dims % 2 == 0 && l.rot_dims <= l.dim && st->layers[i].ret);
      MD_CHECK_ARG(l.col_k >= 0 && l.col_v >= 0 && l.col_g >= 0 && l.col_k % 4 == 0 && l.col_v % 4 == 0 && l.col_g % 4 == 0 &&
                   l.col_k + l.heads * l.dim_pad <= l.in_proj.n_pad && l.col_v + l.heads * l.vdim_pad <= l.in_proj.n_pad &&
                   l.col_g + l.heads * l.vdim_pad <= l.in_proj.n_pad);
    } else if (l.mixer == MD_MIXER_LATENT) {
      MD_TRY(check_linear(l.up_kv, l.rank_pad));
      MD_CHECK_ARG(l.rank > 0 && l.rank_pad >= l.rank && l.rank_pad % 64 == 0 && l.latent_norm && l.up_k_t && st->layers[i].k);
      MD_CHECK_ARG(l.up_kv.n_pad >= l.heads * (l.dim_pad + l.vdim_pad) && l.col_k >= 0 && l.col_k % 32 == 0 && l.col_k + l.rank_pad <= l.in_proj.n_pad);
      MD_CHECK_ARG(l.col_g < 0 || (l.col_g % 32 == 0 && l.col_g + l.heads * l.vdim_pad <= l.in_proj.n_pad));
      MD_CHECK_ARG(l.col_q % 32 == 0);
    } else if (l.mixer == MD_MIXER_STATE_SPACE) {
      const int x = l.heads * l.vdim_pad, bc = l.groups * l.dim_pad;
      MD_CHECK_ARG(l.groups > 0 && l.heads % l.groups == 0 && l.taps >= 1 && l.norm_groups > 0 && l.heads * l.vdim % l.norm_groups == 0);
      MD_CHECK_ARG(l.conv && l.conv_bias && l.dt_bias && l.decay && l.skip && l.out_norm && st->layers[i].ret && (l.taps == 1 || st->layers[i].conv));
      MD_CHECK_ARG(l.col_v >= 0 && l.col_v % 32 == 0 && l.col_k == l.col_v + x && l.col_q == l.col_k + bc && l.col_q + bc <= l.in_proj.n_pad);
      MD_CHECK_ARG(l.col_g >= 0 && l.col_g % 32 == 0 && l.col_g + x <= l.in_proj.n_pad && l.col_dt >= 0 && l.col_dt % 8 == 0 && l.col_dt + (l.heads + 7) / 8 * 8 <= l.in_proj.n_pad);
    } else {
      return MD_ERR_UNSUPPORTED;
    }
  }
  return MD_OK;
}

// one step's launches; carries the pending addend of the residual stream from one row-wise step to the next
struct Step {
  const md_lm_model* m;
  const md_lm_batch* b;
  const md_lm_state* st;
  LmWs w;
  hipStream_t s;
  bool dec;
  LmAddend add = {};           // pending addend of the residual stream(s)
  const float* mix = nullptr;  // streams: the weights around the sublayer that made it
  bool few = false;            // a step of few rows
  bool chain = false;          // fp32: the products' order of sums (gemm_f32.hip)
  bool ready = false;          // w.h holds the next sublayer's input already ...
  const md_lm_layer* unnormed = nullptr;  // few rows: the state-space layer whose outputs lie before their norm in w.att
  const float* sumsq = nullptr;  // ... but for the factor that these give its rows, in the order of the matrix operand

  // ordered: the rows of `a` lie as another of these products left them
  LmStepGemm step_gemm(const void* a, int64_t lda, const md_linear& lin, bool ordered) const {
    LmStepGemm g = {};
    g.a = (const bf16_t*)a;
    g.lda = ordered ? 8 : lda;
    g.chunk = ordered ? 8 * b->n_rows : 8;
    g.ldo = 8;
    g.out_chunk = 8 * b->n_rows;
    g.w = (const bf16_t*)lin.w;
    g.k = lin.k_pad;
    g.rows = b->n_rows;
    g.sumsq = sumsq;
    g.sumsq_n = m->width_pad / 8;
    g.eps = m->eps;
    g.width = m->width;
    g.bias = (const bf16_t*)lin.b;
    return g;
  }

  md_status linear(const void* a, int64_t lda, const md_linear& lin, void* c, int64_t ldc, int rows, bool split = true) {
    if (m->dtype == MD_DTYPE_F32) return lm_gemm_f32(a, lda, lin, c, ldc, rows, chain, s);
    md_gemm_args g = {};
    g.a = a;
    g.lda = lda;
    g.lin = lin;
    g.c = c;
    g.ldc = ldc;
    g.m = rows;
    g.epilogue = MD_EPI_BIAS;
    g.store_pad_cols = 1;
    g.splitk_ws = split && w.splitk_bytes ? w.splitk : nullptr;
    g.splitk_ws_bytes = split ? w.splitk_bytes : 0;
    g.tile_policy = rows > 64 && rows <= DECODE_ROWS ? MD_TILE_DECODE_TALL : MD_TILE_BY_SHAPE;
    return md_gemm_bf16(&g, s);
  }

  // a mixer's projection -> w.proj.  Few rows: one product of whole columns; up to 128 and short prompts: K-slice partials and their sum in two launches, unless one
  // slice fills the chip
  md_status project(const md_linear& lin) {
    if (few) {
      LmStepGemm g = step_gemm(w.h, m->width_pad, lin, sumsq != nullptr);
      g.out = (bf16_t*)w.proj;
      g.ldo = lin.n_pad;
      return lm_step_rows(g, lin.n_pad, s);
    }
    int sl = m->dtype == MD_DTYPE_BF16 ? md_gemm_partial_count(lin, b->n_rows) : 0;
    if (!dec && sl < 3) sl = 1;  // (two slices save about what the second launch takes)
    if (sl == 1) return linear(w.h, m->width_pad, lin, w.proj, lin.n_pad, b->n_rows, !dec);
    const int64_t stride = (int64_t)b->n_rows * lin.n_pad;
    MD_TRY(md_gemm_partial_rows(w.h, m->width_pad, lin, b->n_rows, sl, w.part, lin.n_pad, stride, s));
    return lm_reduce_rows(w.part, sl, lin.n_pad, stride, lin.b, w.proj, lin.n_pad, b->n_rows, lin.n_pad, s);
  }

  // a projection whose result is the next addend
  md_status to_residual(const void* a, int64_t lda, const md_linear& lin) {
    add = {};
    add.ld = m->width_pad;
    const int sl = m->dtype == MD_DTYPE_BF16 && !lin.b ? md_gemm_partial_count(lin, b->n_rows) : 0;  // (slices carry no bias)
    if (sl > 0) {
      add.slices = sl;
      add.slice_stride = (int64_t)b->n_rows * lin.n_pad;
      add.src = w.part;
      return md_gemm_partial_rows(a, lda, lin, b->n_rows, sl, w.part, lin.n_pad, add.slice_stride, s);
    }
    add.src = w.y;
    return linear(a, lda, lin, w.y, m->width_pad, b->n_rows);
  }

  // a sublayer's last projection.  Few rows: the residual stream(s) and the input of the next sublayer in the same launch
  // (plain: rows for a router and experts)
  md_status finish(const void* a, int64_t lda, const md_linear& lin, bool ordered, const float* prev, const md_rms_weight& nw, const float* next, bool plain = false) {
    mix = prev;
    if (!few) return to_residual(a, lda, lin);
    LmStepGemm g = step_gemm(a, lda, lin, ordered);
    g.out = (bf16_t*)w.h;
    if (plain) {
      g.ldo = m->width_pad;
      g.out_chunk = 8;
    }
    g.x = w.x;
    g.stride = (int64_t)b->n_rows * m->width_pad;
    g.streams = n_streams(m);
    g.width_pad = m->width_pad;
    g.prev = prev;
    g.next = next;
    g.norm = nw;
    g.sumsq_out = w.sumsq;
    if (unnormed) {
      g.head_sumsq = w.head_sumsq;
      g.heads = unnormed->heads;
      g.groups = unnormed->norm_groups;
      g.normed = unnormed->heads * unnormed->vdim / unnormed->norm_groups;
      unnormed = nullptr;
    }
    sumsq = w.sumsq;
    ready = true;
    return lm_step_resid(g, s);
  }

  // a sublayer's input -> w.h
  md_status input(const md_rms_weight& nw, const float* next) {
    if (ready) {
      ready = false;
      return MD_OK;
    }
    sumsq = nullptr;
    if (!few || (m->streams == 0 && add.top == 0)) return add_norm(nw, w.h, next, nullptr, true, b->n_rows);
    LmStreams a = streams(nw, w.h, next);
    a.out_chunk = 8 * b->n_rows;
    a.sumsq_out = w.sumsq;
    sumsq = w.sumsq;
    add = {};
    return lm_stream_split(a, b->n_rows, s);
  }

  LmStreams streams(const md_rms_weight& nw, void* y, const float* next) const {
    LmStreams a = {};
    a.x = w.x;
    a.stride = (int64_t)b->n_rows * m->width_pad;
    a.streams = n_streams(m);
    a.add = add;
    a.prev = mix;
    a.next = next;
    a.w = nw;
    a.eps = m->eps;
    a.width = m->width; a.width_pad = m->width_pad;
    a.y = y;
    return a;
  }

  // x += pending;  y = norm(x).  Streams: mixed with the weights around the pending sublayer, then u = their sum weighted for the next one
  // (next == nullptr: plain sum);  y = norm(u).  sum_out: u itself
  md_status add_norm(const md_rms_weight& nw, void* y, const float* next, const int32_t* rows_idx, bool write_x, int rows, float* sum_out = nullptr) {
    md_status r;
    if (m->streams > 0 || add.top > 0) {
      LmStreams a = streams(nw, y, next);
      a.sum_out = sum_out;
      a.rows_idx = rows_idx;
      a.write_x = write_x;
      r = lm_stream_step(m->dtype, a, rows, s);
    } else if (add.slices > 0) {
      r = lm_reduce_resid_norm(w.x, m->width_pad, (const float*)add.src, add.slices, m->width_pad, add.slice_stride, nw, m->eps, m->width, m->width_pad, y,
                               m->width_pad, rows_idx, write_x, rows, s);
    } else {
      r = lm_resid_norm(m->dtype, w.x, m->width_pad, add.src, m->width_pad, nw, m->eps, m->width, m->width_pad, y, m->width_pad, rows_idx, write_x, rows, s);
    }
    if (write_x) add = {};
    return r;
  }

  LmRows rows() const {
    return LmRows{b->n_seq, b->n_rows, b->max_len, b->max_ctx, b->row_seq, b->row_pos, b->seq_row0, b->seq_pos0, b->seq_slot};
  }

  md_status attention(int i) {
    const md_lm_layer& l = m->layers[i];
    LmAttn a = {};
    a.r = rows();
    a.proj = w.proj;
    a.ldp = l.in_proj.n_pad;
    a.col_q = l.col_q; a.col_k = l.col_k; a.col_v = l.col_v;
    a.heads = l.heads; a.kv_heads = l.kv_heads; a.dim = l.dim; a.vdim = l.vdim; a.dp = l.dim_pad; a.vp = l.vdim_pad;
    a.taps = l.taps;
    a.conv = l.conv; a.q_norm = l.q_norm; a.k_norm = l.k_norm;
    a.conv_ld = l.in_proj.n_pad;
    a.value_norm = l.value_norm;
    a.eps = m->eps; a.scale = l.scale;
    a.slope = l.slope; a.mix = l.head_mix;
    a.chunk = l.chunk;
    a.own_kv = l.kv_layer == i;
    a.k = st->layers[l.kv_layer].k;
    a.v = st->layers[l.kv_layer].v;
    a.conv_state = st->layers[i].conv;
    a.ctx = st->ctx;
    a.q = w.q;
    a.out = w.att;
    a.ldo = few ? 8 : l.out_proj.k_pad;
    a.out_chunk = few ? 8 * b->n_rows : 8;
    a.part = w.attn_part;
    const int span = l.chunk > 0 ? std::min(l.chunk, b->max_ctx) : b->max_ctx;
    if (m->dtype == MD_DTYPE_BF16 && b->max_len == 1 && (g_lm_kernels & 2) && lm_attn_heads_takes(a, span)) return lm_attn_heads(a, span, s);
    if (m->dtype == MD_DTYPE_BF16 && b->max_len == 1 && (g_lm_kernels & 2) && lm_attn_decode_takes(a)) {
      a.n_split = lm_attn_decode_splits(b->n_seq, span, &a.split_keys);
      return lm_attn_decode(a, s);
    }
    if (m->dtype == MD_DTYPE_BF16 && b->max_len > 1 && (g_lm_kernels & 5) == 1 && lm_attn_pairs_takes(a, span)) return lm_attn_pairs(a, span, s);
    MD_TRY(lm_attn_prep(m->dtype, a, s));
    if (m->dtype == MD_DTYPE_BF16 && b->max_len > 1 && (g_lm_kernels & 1) && lm_attn_mfma_takes(a)) {
      a.n_split = lm_attn_mfma_parts(a.r, b->ctx_rows, span, l.heads, l.vdim_pad, &a.split_keys);
      return lm_attn_mfma(a, s);
    }
    return lm_attn_plain(m->dtype, a, s);
  }

  md_status retention(int i) {
    const md_lm_layer& l = m->layers[i];
    LmRet a = {};
    a.r = rows();
    a.proj = w.proj;
    a.ldp = l.in_proj.n_pad;
    a.col_q = l.col_q; a.col_k = l.col_k; a.col_v = l.col_v; a.col_g = l.col_g;
    a.heads = l.heads; a.dim = l.dim; a.vdim = l.vdim; a.dp = l.dim_pad; a.vp = l.vdim_pad;
    a.eps = m->eps; a.scale = l.scale;
    a.decay = l.decay; a.rope = l.rope;
    a.rot_dims = l.rot_dims;
    a.state = st->layers[i].ret;
    a.out = w.att;
    a.ldo = few ? 8 : l.out_proj.k_pad;
    a.out_chunk = few ? 8 * b->n_rows : 8;
    a.qf = w.qf; a.kf = w.kf; a.of = w.of;
    a.seg = w.ret_seg;
    a.n_seg = lm_ret_segments(b->n_seq, l.heads, l.dim_pad, l.vdim_pad, b->max_len, &a.seg_chunks);
    if (m->dtype == MD_DTYPE_BF16) {
      if (b->max_len == 1 && (g_lm_kernels & 2) && lm_ret_decode_takes(a)) return lm_ret_decode(a, s);
      if (b->max_len > 1 && (g_lm_kernels & 1) && lm_ret_mfma_takes(a)) return lm_ret_mfma(a, s);
    }
    return lm_ret_plain(m->dtype, a, s);
  }

  md_status latent(int i) {
    const md_lm_layer& l = m->layers[i];
    LmLatent a = {};
    a.r = rows();
    a.proj = w.proj;
    a.ldp = l.in_proj.n_pad;
    a.col_q = l.col_q; a.col_c = l.col_k; a.col_g = l.col_g;
    a.heads = l.heads; a.dim = l.dim; a.vdim = l.vdim; a.dp = l.dim_pad; a.vp = l.vdim_pad; a.rank = l.rank; a.rp = l.rank_pad;
    a.eps = m->eps; a.scale = l.scale;
    a.norm = l.latent_norm;
    a.up_k_t = l.up_k_t;
    a.up_kv = l.up_kv;
    a.cache = st->layers[i].k;
    a.ctx = st->ctx;
    a.out = w.att;
    a.ldo = few ? 8 : l.out_proj.k_pad;
    a.out_chunk = few ? 8 * b->n_rows : 8;
    a.ctx_rows = b->ctx_rows;
    a.seq_ctx0 = b->seq_ctx0;
    a.c_rows = w.c_rows; a.kv = w.kv; a.q_lat = w.q_lat; a.part = w.latent_part;
    if (m->dtype == MD_DTYPE_BF16 && b->max_len == 1 && (g_lm_kernels & 2) && lm_latent_decode_takes(a)) {
      a.n_split = lm_latent_decode_splits(b->n_seq, l.heads, b->max_ctx);
      return lm_latent_decode(a, s);
    }
    if (m->dtype == MD_DTYPE_BF16 && b->max_len > 1 && (g_lm_kernels & 1) && lm_latent_mfma_takes(a)) {
      MD_TRY(lm_latent_rows(MD_DTYPE_BF16, a, true, s));
      MD_TRY(linear(w.c_rows, l.rank_pad, l.up_kv, w.kv, l.up_kv.n_pad, b->ctx_rows));
      return lm_latent_mfma(a, s);
    }
    return lm_latent_plain(m->dtype, a, s);
  }

  md_status state_space(int i) {
    const md_lm_layer& l = m->layers[i];
    LmSsm a = {};
    a.r = rows();
    a.proj = w.proj;
    a.ldp = l.in_proj.n_pad;
    a.col_z = l.col_g; a.col_x = l.col_v; a.col_b = l.col_k; a.col_c = l.col_q; a.col_dt = l.col_dt;
    a.heads = l.heads; a.groups = l.groups; a.dim = l.dim; a.vdim = l.vdim; a.dp = l.dim_pad; a.vp = l.vdim_pad; a.taps = l.taps;
    a.norm_groups = l.norm_groups;
    a.conv = l.conv; a.conv_bias = l.conv_bias; a.dt_bias = l.dt_bias; a.decay = l.decay; a.skip = l.skip; a.out_norm = l.out_norm;
    a.eps = m->eps;
    a.conv_state = st->layers[i].conv;
    a.state = st->layers[i].ret;
    a.out = w.att;
    a.ldo = few ? 8 : l.out_proj.k_pad;
    a.out_chunk = few ? 8 * b->n_rows : 8;
    a.u = w.conv_out; a.dt = w.dt; a.seg = w.seg; a.seg_decay = w.seg_decay;
    if (m->dtype == MD_DTYPE_BF16) {
      if (b->max_len == 1 && (g_lm_kernels & 2) && lm_ssm_decode_takes(a)) {
        // (the product's waves take an eighth of K each)
        const bool eighths = (l.norm_groups == 2 || l.norm_groups == 4 || l.norm_groups == 8) && l.heads % 8 == 0 && l.vdim == l.vdim_pad &&
                             l.out_proj.k_pad == l.heads * l.vdim && l.out_proj.k_pad % 512 == 0;
        if (few && (l.norm_groups == 1 || eighths)) {
          a.sumsq = w.head_sumsq;
          unnormed = &l;
        }
        return lm_ssm_decode(a, s);
      }
      a.n_seg = lm_ssm_segments(b->n_seq, l.heads, b->max_len, &a.seg_chunks);
      if (b->max_len > 1 && (g_lm_kernels & 1) && lm_ssm_mfma_takes(a)) return lm_ssm_mfma(a, s);
    }
    return lm_ssm_plain(m->dtype, a, s);
  }

  md_status mixer(int i) {
    switch (m->layers[i].mixer) {
      case MD_MIXER_ATTENTION: return attention(i);
      case MD_MIXER_LATENT: return latent(i);
      case MD_MIXER_STATE_SPACE: return state_space(i);
      default: return retention(i);
    }
  }

  md_status feed_forward(const md_lm_layer& l, const md_rms_weight& nw, const float* next) {
    if (l.experts > 0) {
      mix = l.mix2;
      return expert_forward(l);
    }
    if (few) {
      LmStepGemm g = step_gemm(w.h, m->width_pad, l.gate_up, sumsq != nullptr);
      g.out = (bf16_t*)w.act;
      g.ff_pad = l.ff_pad;
      MD_TRY(lm_step_silu(g, s));
    } else if (m->dtype == MD_DTYPE_F32 || l.gate_up.b) {
      MD_TRY(linear(w.h, m->width_pad, l.gate_up, w.gu, l.gate_up.n_pad, b->n_rows));
      MD_TRY(lm_silu_mul(m->dtype, w.gu, l.gate_up.n_pad, w.act, l.down.k_pad, b->n_rows, l.ff_pad, s));
    } else if (!dec || md_gemm_partial_count(l.gate_up, b->n_rows) == 1) {
      MD_TRY(md_gemm_silu_bf16(w.h, m->width_pad, l.gate_up, w.act, l.down.k_pad, b->n_rows, s));
    } else {
      const int sl = md_gemm_partial_count(l.gate_up, b->n_rows);
      const int64_t ld = l.gate_up.n_pad, stride = (int64_t)b->n_rows * ld;
      MD_TRY(md_gemm_partial_rows(w.h, m->width_pad, l.gate_up, b->n_rows, sl, w.part, ld, stride, s));
      MD_TRY(lm_reduce_silu_mul(w.part, sl, ld, stride, w.act, l.down.k_pad, b->n_rows, l.ff_pad, s));
    }
    return finish(w.act, l.down.k_pad, l.down, few, l.mix2, nw, next);
  }

  md_status expert_forward(const md_lm_layer& l) {
    const int rows = b->n_rows, slots = rows * l.top;
    const bool step = dec && lm_expert_step_takes(rows, l.top, l.experts);
    LmRoute r = {w.h, rows, m->width_pad, l.experts, l.top, l.router.w, l.router_bias, w.chosen, w.route_weight};
    if (step) {
      r.sumsq = sumsq;
      r.sumsq_n = m->width_pad / 8;
      r.width = m->width;
      r.eps = m->eps;
      r.factor = w.row_factor;
    } else {
      r.offsets = w.offsets;
      r.row_of = w.row_of;
      r.slot_of = w.slot_of;
    }
    MD_TRY(lm_route(m->dtype, r, s));
    const int64_t ld = l.gate_up.n_pad;
    add = {};
    add.ld = m->width_pad;
    add.top = l.top;
    add.slot_of = r.slot_of;
    add.weight = w.route_weight;
    if (step) {
      add.src = w.part;
      add.slices = 1;
      LmExpertGemm g = {(const bf16_t*)w.h, m->width_pad, rows, l.top, (const bf16_t*)l.gate_up.w, ld * l.gate_up.k_pad, l.gate_up.k_pad, l.experts,
                        w.chosen, slots, l.ff_pad, sumsq ? w.row_factor : nullptr, w.act, l.down.k_pad};
      MD_TRY(lm_expert_silu(g, s));
      g = {(const bf16_t*)w.act, l.down.k_pad, slots, 1, (const bf16_t*)l.down.w, (int64_t)l.down.n_pad * l.down.k_pad, l.down.k_pad, l.experts,
           w.chosen, slots, 0, nullptr, w.part, m->width_pad};
      return lm_expert_rows(g, l.down.n_pad, s);
    }
    if (dec) {
      const int64_t stride = slots * ld;
      const int sl = md_gemm_grouped_slices(l.gate_up, l.experts, slots);
      if (sl == 1) {
        MD_TRY(md_gemm_grouped_bf16(w.h, m->width_pad, w.row_of, l.gate_up, l.experts, w.offsets, w.act, l.down.k_pad, slots, true, false, s));
      } else {
        MD_TRY(md_gemm_grouped_partial(w.h, m->width_pad, w.row_of, l.gate_up, l.experts, w.offsets, w.part, ld, stride, slots, s));
        MD_TRY(lm_reduce_silu_mul(w.part, sl, ld, stride, w.act, l.down.k_pad, slots, l.ff_pad, s));
      }
      add.src = w.part;
      add.slices = md_gemm_grouped_slices(l.down, l.experts, slots);
      add.slice_stride = (int64_t)slots * l.down.n_pad;
      return md_gemm_grouped_partial(w.act, l.down.k_pad, nullptr, l.down, l.experts, w.offsets, w.part, l.down.n_pad, add.slice_stride, slots, s);
    }
    add.src = w.y;
    if (m->dtype == MD_DTYPE_F32) {
      MD_TRY(lm_grouped_gemm_f32(w.h, m->width_pad, w.row_of, l.gate_up, l.experts, w.offsets, w.gu, ld, slots, chain, s));
      MD_TRY(lm_silu_mul(m->dtype, w.gu, ld, w.act, l.down.k_pad, slots, l.ff_pad, s));
      return lm_grouped_gemm_f32(w.act, l.down.k_pad, nullptr, l.down, l.experts, w.offsets, w.y, m->width_pad, slots, chain, s);
    }
    MD_TRY(md_gemm_grouped_bf16(w.h, m->width_pad, w.row_of, l.gate_up, l.experts, w.offsets, w.act, l.down.k_pad, slots, true, true, s));
    return md_gemm_grouped_bf16(w.act, l.down.k_pad, nullptr, l.down, l.experts, w.offsets, w.y, m->width_pad, slots, false, false, s);
  }

  // the residual stream behind everything so far -> out (fp32 [n_rows][width_pad]); streams: their sum
  md_status tap(float* out) {
    if (m->streams > 0 || add.top > 0) return add_norm(m->final_norm, nullptr, nullptr, nullptr, false, b->n_rows, out);
    MD_TRY(add_norm(m->final_norm, nullptr, nullptr, nullptr, true, b->n_rows));
    const size_t bytes = (size_t)b->n_rows * m->width_pad * 4;
    return hipMemcpyAsync(out, w.x, bytes, hipMemcpyDeviceToDevice, s) == hipSuccess ? MD_OK : MD_ERR_LAUNCH;
  }

  md_status run(const int32_t* logit_rows, int n_logits, void* logits, int64_t ld_logits, float* layer_out) {
    if (w.splitk_bytes) MD_TRY(zero_fill(w.splitk, 8192, s));  // arrival tickets
    const int64_t row_floats = (int64_t)b->n_rows * m->width_pad;
    if (own_row_steps(m)) MD_TRY(lm_embed_streams(m, b->tokens, b->row_pos, w.x, row_floats, b->n_rows, s));
    else MD_TRY(lm_embed(m->dtype, m->embed, m->width_pad, b->tokens, w.x, b->n_rows, m->vocab, s));
    const bool few_logits = n_logits > 0 && n_logits <= LM_STEP_ROWS;
    for (int i = 0; i < m->n_layers; ++i) {
      const md_lm_layer& l = m->layers[i];
      // what follows this layer: the next one's mixer, or the head
      const md_lm_layer* after = i + 1 < m->n_layers ? &m->layers[i + 1] : nullptr;
      const md_rms_weight& nw = after ? after->norm1 : m->final_norm;
      const float* next = after ? after->mix1 : nullptr;
      MD_TRY(input(l.norm1, l.mix1));
      MD_TRY(project(l.in_proj));
      if (l.out_proj.k_pad != l.heads * l.vdim_pad) MD_TRY(zero_fill(w.att, (size_t)b->n_rows * l.out_proj.k_pad * esize(m), s));
      MD_TRY(mixer(i));
      if (l.ff > 0) {
        MD_TRY(finish(w.att, l.out_proj.k_pad, l.out_proj, few, l.mix1, l.norm2, l.mix2, l.experts > 0));
        MD_TRY(input(l.norm2, l.mix2));
        MD_TRY(feed_forward(l, nw, next));
      } else {
        MD_TRY(finish(w.att, l.out_proj.k_pad, l.out_proj, few, l.mix1, nw, next));
      }
      if (layer_out) MD_TRY(tap(layer_out + i * row_floats));
    }
    if (n_logits == 0) return MD_OK;
    ready = ready && few_logits;
    if (!ready) {
      sumsq = nullptr;
      MD_TRY(add_norm(m->final_norm, w.h, nullptr, logit_rows, false, n_logits));
    }
    if (!few || !few_logits) return linear(w.h, m->width_pad, m->head, logits, ld_logits, n_logits);
    LmStepGemm g = step_gemm(w.h, m->width_pad, m->head, ready);
    g.rows = n_logits;
    g.rows_idx = ready ? logit_rows : nullptr;  // (otherwise w.h holds the wanted rows only)
    g.out = (bf16_t*)logits;
    g.ldo = ld_logits;
    return lm_step_rows(g, m->head.n_pad, s);
  }
};

}  // namespace

extern "C" void md_lm_set_kernels(int32_t mask) { g_lm_kernels = mask; }

extern "C" size_t md_lm_workspace_bytes(const md_lm_model* m, const md_lm_batch* b, int32_t n_logits) {
  if (!m || !m->layers || !b || b->n_rows <= 0 || b->n_seq <= 0 || b->max_len <= 0 || n_logits < 0) return 0;
  return layout(m, b, n_logits, nullptr).total;
}

extern "C" md_status md_lm_forward(const md_lm_model* m, const md_lm_batch* b, const md_lm_state* st, const int32_t* logit_rows,
                                   int32_t n_logits, void* logits, int64_t ld_logits, float* layer_out, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  MD_CHECK_ARG(m && b && st && st->layers && st->slots > 0 && st->ctx > 0 && st->ctx % 64 == 0 && workspace);
  MD_CHECK_ARG(b->n_seq > 0 && b->n_rows >= b->n_seq && b->max_len > 0 && b->max_len <= b->n_rows && b->max_ctx <= st->ctx && b->max_ctx >= b->max_len);
  MD_CHECK_ARG(b->tokens && b->row_seq && b->row_pos && b->seq_row0 && b->seq_pos0 && b->seq_slot);
  MD_CHECK_ARG(b->max_len > 1 || b->n_rows == b->n_seq);
  MD_CHECK_ARG(b->max_len == 1 || (b->seq_ctx0 && b->ctx_rows >= b->n_rows));
  MD_CHECK_ARG(n_logits >= 0 && (n_logits == 0 || (logits && ld_logits >= m->head.n_pad && ld_logits % 8 == 0)));
  MD_CHECK_ARG(logit_rows || n_logits <= b->n_rows);
  MD_TRY(check_model(m, st));
  const LmWs w = layout(m, b, n_logits, workspace);
  if (workspace_bytes < w.total) return MD_ERR_WORKSPACE;
  Step step{m, b, st, w, (hipStream_t)stream, decode_regime(m, b->n_rows)};
  step.few = step_regime(m, b);
  for (int i = 0; i < m->n_layers; ++i) step.chain = step.chain || m->layers[i].mixer == MD_MIXER_RETENTION;
  return step.run(logit_rows, n_logits, logits, ld_logits, layer_out);
}

extern "C" md_status md_lm_decode_step(const md_lm_model* m, const md_lm_batch* b, const md_lm_state* st, int32_t* next, int32_t* pos,
                                       int32_t suppress_id, void* logits, int64_t ld_logits, void* workspace, size_t workspace_bytes,
                                       void* stream) {
  MD_CHECK_ARG(next && pos && b && b->row_pos == pos && b->seq_pos0 == pos && b->max_len == 1 && logits);
  MD_TRY(md_lm_forward(m, b, st, nullptr, b->n_seq, logits, ld_logits, nullptr, workspace, workspace_bytes, stream));
  hipStream_t s = (hipStream_t)stream;
  return m->dtype == MD_DTYPE_F32 ? md_argmax_advance_f32(logits, ld_logits, b->n_seq, m->vocab, suppress_id, next, pos, s)
                                  : md_argmax_advance(logits, ld_logits, b->n_seq, m->vocab, suppress_id, next, pos, s);
}
