// Host side of the estimator as the library's own entry points call it (estimate.hip, prefill.hip).
#pragma once
#include "attn_plan.h"
#include "lds_limit.h"
#include "xattn_common.h"

namespace xattn {

// what the fused normalise-and-select pass needs beside the estimator's own arguments
struct SelectArgs {
  const double* tau;        // per head, on the device; or null and
  const double* tau_host;   // one value, or one per head (at most kMaxTauHost), copied into the kernel's arguments
  int tau_host_count;
  uint8_t* mask;
  void* sums_out;           // bf16 [H][rows][nkb] block sums, or null
  int32_t* col_idx;
  int32_t* col_cnt;
  int64_t idx_pitch;
  int keep_sink, keep_recent;
  int real_q_blocks_only;   // leave out the rows of q-blocks past the sequence end
  const AttnPlan* plan;     // null, or where to note long lists for the attention (lists of all q-blocks of a head)
  uint32_t* totals;         // null, or where to find blocks of each q-block's lists, and of its longest, at 32 * (row)
  unsigned long long* clear;   // words set to zero for what follows, or null
  int clear_words;
  int stages;               // bit 0: run the GEMM pass, bit 1: run the normalise-and-select pass
};

int estimate_impl(const void* q, const void* k, float* block_sums, void* workspace, size_t workspace_size,
                  float* scores_out, int num_heads, int num_kv_heads, int q_len, int k_len, int head_dim,
                  int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_h, int64_t k_stride_n, int stride,
                  int block_size, int chunk_size, int chunk_begin, int chunk_end, int causal, int own_chunk_only,
                  float scale, const int32_t* slab_pairs, int num_slab_pairs, int softmax, int kdb,
                  int zero_rows_from, int window_row0, int window_rows, void* stream, const SelectArgs* sel);

// CUs of the current device, rounded down to a multiple of 8
int resident_workgroups();

// estimator workspace of one launch over every query chunk when only the rows of real q-blocks are computed; 0 if the
// geometry is not accepted
size_t estimate_real_rows_bytes(int num_heads, int q_len, int k_len, int stride, int block_size, int chunk_size);

// xattn_block_sparse_fwd, with a plan (null: no list is cut) whose long lists are noted or still to be noted, and a queue of
// kQueueBytes zeros (null: a workgroup for each list and piece) and the q-blocks' totals - or, not ready, room for them
constexpr size_t kQueueBytes = 4096;
bool attention_queued(int num_heads, int q_len, int k_len, int causal);
// whether the attention asks for the blocks of each q-block's lists and of its longest, 128 bytes apart (null: it finds them)
bool attention_asks_totals(int num_heads, int q_len, int k_len, int causal);
int block_sparse_impl(const void* q, const void* k, const void* v, void* out, const int32_t* col_idx, const int32_t* col_cnt,
                      int64_t idx_pitch, int idx_rows, int idx_row0, int num_heads, int num_kv_heads, int q_len, int k_len,
                      int head_dim, int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_h, int64_t k_stride_n,
                      int64_t v_stride_h, int64_t v_stride_n, int64_t o_stride_h, int64_t o_stride_n, int q_block_begin,
                      int q_block_end, int causal, float softmax_scale, void* stream, const AttnPlan* plan, bool note,
                      int32_t* queue, uint32_t* totals, bool ready);

}  // namespace xattn
