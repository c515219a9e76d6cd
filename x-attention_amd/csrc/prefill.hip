// The prefill operator as one call: antidiagonal estimate, block selection and
// block-sparse attention enqueued back to back on one stream (what
// Xattention_prefill, xattn/src/Xattention.py:302-402, runs for a sequence
// whose temporaries fit one launch per stage).
//
// A short prompt is bound by what happens around the kernels.  As three calls
// from Python with a tensor each for the estimator's workspace, the
// thresholds (a fill kernel of their own), the column lists, the counts and
// the output, a 1000-token prompt took 75 us of host time for 40-60 us of GPU
// work.  Here the temporaries share one caller-provided buffer, thresholds that
// live on the host travel in the kernel arguments, and the rows the padding to
// chunk_size adds are left out of all three stages.
#include "estimate.h"
#include "xattn_hip.h"

using namespace xattn;

namespace {
struct PrefillLayout {
  size_t est_bytes, cnt_off, idx_off, queue_off, totals_bytes, plan_off, total;
  int nqb, nkb;
  PlanShape plan;
};

size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

// false if the estimator refuses the geometry
bool prefill_layout(int num_heads, int q_len, int k_len, int stride, int chunk_size, PrefillLayout* l) {
  l->est_bytes = estimate_real_rows_bytes(num_heads, q_len, k_len, stride, 128, chunk_size);
  if (l->est_bytes == 0) return false;
  l->nqb = (q_len + 127) / 128;
  l->nkb = (k_len + 127) / 128;
  l->cnt_off = up256(l->est_bytes);
  l->idx_off = l->cnt_off + up256((size_t)num_heads * l->nqb * sizeof(int32_t));
  l->queue_off = l->idx_off + up256((size_t)num_heads * l->nqb * l->nkb * sizeof(int32_t));
  l->totals_bytes = up256((size_t)l->nqb * 128);
  l->plan_off = l->queue_off + kQueueBytes + l->totals_bytes;                  // (cleared together)
  const int64_t units = (int64_t)num_heads * l->nqb;
  l->plan = plan_shape(num_heads, q_len, k_len);
  l->total = l->plan_off + plan_bytes(l->plan, units, l->nqb);
  return true;
}
}  // namespace

extern "C" size_t xattn_prefill_workspace_bytes(int num_heads, int q_len, int k_len, int stride, int chunk_size) {
  PrefillLayout l;
  return prefill_layout(num_heads, q_len, k_len, stride, chunk_size, &l) ? l.total : 0;
}

extern "C" size_t xattn_prefill_least_workspace_bytes(int num_heads, int q_len, int k_len, int stride, int chunk_size) {
  PrefillLayout l;
  return prefill_layout(num_heads, q_len, k_len, stride, chunk_size, &l) ? l.plan_off : 0;
}

extern "C" int xattn_prefill_fwd(const void* q, const void* k, const void* v, void* out, void* workspace,
                                 size_t workspace_bytes, int num_heads, int num_kv_heads, int q_len, int k_len,
                                 int head_dim, int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_h,
                                 int64_t k_stride_n, int64_t v_stride_h, int64_t v_stride_n, int64_t o_stride_h,
                                 int64_t o_stride_n, int stride, int chunk_size, int causal, int own_chunk_only,
                                 float estimate_scale, int zero_rows_from, const double* tau_host, int tau_host_count,
                                 const double* tau_device, int keep_sink, int keep_recent, float softmax_scale,
                                 void* stream) {
  if (!workspace || !v || !out) return XATTN_ERR_NULL;
  PrefillLayout l;
  if (!prefill_layout(num_heads, q_len, k_len, stride, chunk_size, &l)) return XATTN_ERR_SHAPE;
  if (workspace_bytes < l.plan_off) return XATTN_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(workspace) & 255) return XATTN_ERR_ALIGN;
  char* ws = static_cast<char*>(workspace);
  SelectArgs sel{};
  sel.tau = tau_device;
  sel.tau_host = tau_host;
  sel.tau_host_count = tau_host_count;
  sel.col_cnt = reinterpret_cast<int32_t*>(ws + l.cnt_off);
  sel.col_idx = reinterpret_cast<int32_t*>(ws + l.idx_off);
  sel.idx_pitch = l.nkb;
  sel.keep_sink = keep_sink;
  sel.keep_recent = keep_recent;
  sel.real_q_blocks_only = 1;
  sel.stages = 3;
  const int64_t units = (int64_t)num_heads * l.nqb;
  if (workspace_bytes < l.total) l.plan = PlanShape{};      // lists stay whole
  const AttnPlan plan = plan_at(l.plan, ws + l.plan_off, units, l.nqb);
  // (with zero_rows_from 0 no row is estimated, and no MFMA pass would clear what is noted: noted afterwards)
  // Where no list can be long enough to be cut, nothing is noted (nor planned below): then the selection may follow the
  // estimate in the same kernel.
  const int q_chunks = (int)(((int64_t)q_len + chunk_size - 1) / chunk_size), k_chunks = (int)(((int64_t)k_len + chunk_size - 1) / chunk_size);
  const int64_t last_token = (int64_t)l.nqb * 128 - 1 + (int64_t)(k_chunks - q_chunks) * chunk_size;   // on the key axis, both padded
  const bool may_cut = l.plan.per_qb && (!causal || keep_sink || last_token / 128 + 1 > l.plan.min_piece);
  if (may_cut && zero_rows_from != 0) sel.plan = &plan;
  // Ahead of what is noted lie the attention's queue and the q-blocks' totals; the estimate clears them together.
  const bool cleared = zero_rows_from != 0, queued = cleared && attention_queued(num_heads, q_len, k_len, causal);
  int32_t* const queue = queued ? reinterpret_cast<int32_t*>(ws + l.queue_off) : nullptr;
  if (cleared && attention_asks_totals(num_heads, q_len, k_len, causal)) sel.totals = reinterpret_cast<uint32_t*>(ws + l.queue_off + kQueueBytes);
  if (queue || sel.totals || sel.plan) {
    const size_t from = queue ? l.queue_off : sel.totals ? l.queue_off + kQueueBytes : l.plan_off;
    const size_t noted = sel.plan ? plan_noted_bytes(l.nqb) + plan_round((size_t)units * 4) : 0;
    sel.clear = reinterpret_cast<unsigned long long*>(ws + from);
    sel.clear_words = (int)((l.plan_off - from + noted) / 8);
  }
  int rc = estimate_impl(q, k, nullptr, ws, l.est_bytes, nullptr, num_heads, num_kv_heads, q_len, k_len, head_dim,
                         q_stride_h, q_stride_n, k_stride_h, k_stride_n, stride, 128, chunk_size, 0, q_chunks, causal,
                         own_chunk_only, estimate_scale, nullptr, 0, 1, 1, zero_rows_from, 0, l.nqb, stream, &sel);
  if (rc != XATTN_OK) return rc;
  return block_sparse_impl(q, k, v, out, sel.col_idx, sel.col_cnt, l.nkb, l.nqb, 0, num_heads, num_kv_heads, q_len,
                           k_len, head_dim, q_stride_h, q_stride_n, k_stride_h, k_stride_n, v_stride_h, v_stride_n,
                           o_stride_h, o_stride_n, 0, l.nqb, causal, softmax_scale, stream, may_cut ? &plan : nullptr, !sel.plan, queue, sel.totals, true);
}

extern "C" int xattn_estimate_fwd(const void* q, const void* k, void* block_sums, uint8_t* mask, void* workspace,
                                  size_t workspace_bytes, int num_heads, int num_kv_heads, int q_len, int k_len,
                                  int head_dim, int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_h,
                                  int64_t k_stride_n, int stride, int chunk_size, int causal, int own_chunk_only,
                                  float estimate_scale, int zero_rows_from, const double* tau_host, int tau_host_count,
                                  const double* tau_device, int keep_sink, int keep_recent, void* stream) {
  if (!workspace || !block_sums || !mask) return XATTN_ERR_NULL;
  if (reinterpret_cast<uintptr_t>(block_sums) & 1) return XATTN_ERR_ALIGN;
  if (q_len <= 0 || chunk_size <= 0) return XATTN_ERR_SHAPE;
  SelectArgs sel{};
  sel.tau = tau_device;
  sel.tau_host = tau_host;
  sel.tau_host_count = tau_host_count;
  sel.mask = mask;
  sel.sums_out = block_sums;
  sel.keep_sink = keep_sink;
  sel.keep_recent = keep_recent;
  sel.stages = 3;
  const int q_chunks = (int)(((int64_t)q_len + chunk_size - 1) / chunk_size);
  return estimate_impl(q, k, nullptr, workspace, workspace_bytes, nullptr, num_heads, num_kv_heads, q_len, k_len, head_dim,
                       q_stride_h, q_stride_n, k_stride_h, k_stride_n, stride, 128, chunk_size, 0, q_chunks, causal,
                       own_chunk_only, estimate_scale, nullptr, 0, 1, 1, zero_rows_from, 0, 0, stream, &sel);
}
