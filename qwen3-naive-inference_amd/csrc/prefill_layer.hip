// One decoder layer of a prefill step, launched by one call (gfx950).
//
// Reference semantics: Qwen3DecoderLayer.forward_prefill (qwen3_naive.py:
// 597-645, :692-702, :719-745).  The layer is a chain of 8 to 10 short
// kernels on one stream; from Python each cost 10-27 us of host time
// (argument checks, ctypes, torch's library GEMM dispatch), so a layer of up
// to 2,048 tokens took 200 us of host time for 55-130 us of GPU work.  This
// entry point enqueues the chain through the library's own entry points.
// Host code only: every launch is the callee's.
#include <algorithm>

#include "qmi_common.h"

namespace {

constexpr int64_t kAlign = 256;

int64_t padded(int64_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

// Rows up to which the decode-batch kernel is the faster projection: it reads
// 16 weight rows per tile (qkv at 16 rows: 4.8 us against 5.9; at 77 rows 6.6
// against 6.2).
constexpr int64_t kRowsForm = 64;

int linear(const uint16_t* x, int64_t xs, const uint16_t* w, int64_t ws, int64_t m, int64_t n,
           int64_t k, int32_t act, uint16_t* y, void* st) {
  if (m <= kRowsForm && k % 128 == 0)
    return qmi_linear_rows(x, xs, w, ws, m, n, k, act, y, n, st);
  return qmi_linear_tiles(x, xs, w, ws, m, n, k, act, y, n, st);
}

struct Layout {
  int64_t h, r1, qkv, q, o, proj, act, total;
};

// o_proj and down_proj have few columns; up to 256 rows their K range is
// split (fp32 partial products) to fill the chip: at 77 rows o_proj 4.9 us
// and down_proj 5.9 us, against 8.9 and 11.8 us for 64 x 64 tiles.
int64_t parts_of(int64_t m, int64_t n, int64_t k) {
  return k % 128 ? 0 : qmi_linear_rows_parts_count(m, n, k);
}

Layout layout(int64_t t, int64_t hidden, int64_t qkv_n, int64_t q_n, int64_t inter) {
  Layout l;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t p = at;
    at += padded(bytes);
    return p;
  };
  l.h = take(2 * t * hidden);
  l.r1 = take(2 * t * hidden);
  l.qkv = take(2 * t * qkv_n);
  l.q = take(2 * t * q_n);
  l.o = take(2 * t * q_n);
  const int64_t parts = std::max(parts_of(t, hidden, q_n), parts_of(t, hidden, inter));
  l.proj = take(std::max<int64_t>(2 * t * hidden, 4 * parts * t * hidden));
  l.act = take(2 * t * inter);
  l.total = at;
  return l;
}

}  // namespace

extern "C" int64_t qmi_prefill_layer_workspace_bytes(int64_t n_tok, int64_t hidden,
                                                     int64_t num_q_heads, int64_t num_kv_heads,
                                                     int64_t head_dim, int64_t inter) {
  if (n_tok <= 0 || hidden <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || inter <= 0)
    return 0;
  return layout(n_tok, hidden, (num_q_heads + 2 * num_kv_heads) * head_dim, num_q_heads * head_dim,
                inter).total;
}

#define QMI_TRY(call)                 \
  do {                                \
    const int _s = (call);            \
    if (_s != QMI_OK) return _s;      \
  } while (0)

extern "C" int qmi_prefill_layer(const qmi_prefill_layer_args* a, void* stream) {
  if (!a) return QMI_E_NULL_POINTER;
  const int64_t t = a->n_tok, hidden = a->hidden, d = a->head_dim;
  const int64_t hq = a->num_q_heads, hkv = a->num_kv_heads, inter = a->inter;
  if (t < 0 || hidden <= 0 || hq <= 0 || hkv <= 0 || d <= 0 || inter <= 0) return QMI_E_BAD_SHAPE;
  if (t == 0) return QMI_OK;
  if (!a->x || !a->input_norm || !a->post_norm || !a->out || !a->residual_out || !a->workspace)
    return QMI_E_NULL_POINTER;
  const int64_t q_n = hq * d, qkv_n = q_n + 2 * hkv * d;
  const Layout l = layout(t, hidden, qkv_n, q_n, inter);
  if (a->workspace_bytes < l.total) return QMI_E_WORKSPACE_TOO_SMALL;
  if (reinterpret_cast<uintptr_t>(a->workspace) % 16) return QMI_E_BAD_STRIDE;
  char* ws = static_cast<char*>(a->workspace);
  auto at = [&](int64_t off) { return reinterpret_cast<uint16_t*>(ws + off); };
  uint16_t *h = at(l.h), *r1 = at(l.r1), *qkv = at(l.qkv), *q = at(l.q), *o = at(l.o);
  uint16_t *proj = at(l.proj), *act = at(l.act);
  float* parts = reinterpret_cast<float*>(ws + l.proj);

  // Input norm; the residual it adds up to is x itself, or x + residual.
  const uint16_t* res = a->x;
  int64_t res_stride = a->x_stride;
  if (a->residual) {
    QMI_TRY(qmi_add_rms_norm(a->x, a->x_stride, a->residual, a->residual_stride, r1, hidden,
                             a->input_norm, h, hidden, t, hidden, a->eps, stream));
    res = r1;
    res_stride = hidden;
  } else {
    QMI_TRY(qmi_rms_norm(a->x, a->x_stride, a->input_norm, h, hidden, t, hidden, a->eps, stream));
  }
  QMI_TRY(linear(h, hidden, a->qkv_weight, a->qkv_stride, t, qkv_n, hidden, 0, qkv, stream));
  QMI_TRY(qmi_qk_norm_rope_store(qkv, qkv_n, t, hq, hkv, d, a->q_norm, a->k_norm, a->positions,
                                 a->cos_sin_cache, a->max_position, q, q_n, a->k_cache, a->v_cache,
                                 a->slot_mapping, a->num_blocks * a->block_size, a->qk_eps, stream));
  QMI_TRY(qmi_varlen_prefill_attention(
      q, q_n, d, a->k_cache, a->v_cache, a->num_blocks, a->block_size, hq, hkv, d, a->cu_seqlens_q,
      a->cu_seqlens_k, a->block_table, a->bt_stride, a->bt_width, a->batch, a->max_seqlen_q,
      a->max_seqlen_k, t, a->scale, o, q_n, d, a->attn_workspace, a->attn_workspace_bytes, 0, stream));
  int64_t s = parts_of(t, hidden, q_n);
  if (s > 0) {
    QMI_TRY(qmi_linear_rows_parts(o, q_n, a->o_weight, a->o_stride, t, hidden, q_n, parts, s, stream));
    QMI_TRY(qmi_add_rms_norm_parts(parts, s, t, res, res_stride, a->residual_out, hidden,
                                   a->post_norm, h, hidden, hidden, a->post_eps, stream));
  } else {
    QMI_TRY(qmi_linear_tiles(o, q_n, a->o_weight, a->o_stride, t, hidden, q_n, 0, proj, hidden, stream));
    QMI_TRY(qmi_add_rms_norm(proj, hidden, res, res_stride, a->residual_out, hidden, a->post_norm, h,
                             hidden, t, hidden, a->post_eps, stream));
  }
  QMI_TRY(linear(h, hidden, a->gate_up_weight, a->gate_up_stride, t, inter, hidden, 1, act, stream));
  s = parts_of(t, hidden, inter);
  if (s > 0) {
    QMI_TRY(qmi_linear_rows_parts(act, inter, a->down_weight, a->down_stride, t, hidden, inter, parts,
                                  s, stream));
    return qmi_sum_parts(parts, s, t, hidden, a->out, hidden, stream);
  }
  return qmi_linear_tiles(act, inter, a->down_weight, a->down_stride, t, hidden, inter, 0, a->out,
                          hidden, stream);
}
