// Block-sparse FlashAttention forward for gfx950 (bf16 MFMA, fp32 softmax).
//
// Replaces the reference's call to the third-party CUDA kernel
// block_sparse_attn_func (xattn/src/Xattention.py:377-391): for every query
// block of 128 tokens only the key/value blocks named by a per-(head, q-block)
// column list are visited, with token-level causal masking (bottom-right
// aligned when k_len > q_len) and grouped-query attention by KV-head sharing.
// With no column list the same kernels visit every visible block, which is the
// dense FlashAttention baseline the speedup is quoted against.
#include "attn_rows32.h"
#include "attn_rows64.h"
#include "attn_wide.h"
#include "lds_limit.h"
#include "estimate.h"
#include "xattn_hip.h"

namespace xattn {

// Notes the lists of q-blocks [qb_begin, qb_end) of every head, where the pass that made them has not (or, without
// lists, the visible blocks of each).  One workgroup, which counts the pieces in LDS.
__global__ __launch_bounds__(1024) void note_lists_kernel(AttnParams p) {
  __shared__ unsigned long long pieces;
  if (threadIdx.x == 0) pieces = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  for (int qb = p.qb_begin + (int)(threadIdx.x >> 6); qb < p.qb_end; qb += 16) {
    const int row = qb - p.idx_row0;
    const int q_last = (qb * kBlk + kBlk - 1 < p.Lq ? qb * kBlk + kBlk - 1 : p.Lq - 1) + p.kv_off;
    int visible = p.causal ? (q_last < 0 ? 0 : q_last / kBlk + 1) : p.nkb;
    visible = visible < p.nkb ? visible : p.nkb;
    auto count = [&](int h) {
      if (!p.col_cnt) return visible;
      const int n = p.col_cnt[(int64_t)h * p.idx_rows + row];
      return n < 0 ? 0 : n > p.idx_pitch ? (int)p.idx_pitch : n;
    };
    int total = 0;
    for (int h = lane; h < p.H; h += 64) total += count(h) < 65536 ? count(h) : 65536;   // (a sum of at most 8192)
    note_q_block(p.plan, qb, p.H, __builtin_amdgcn_readlane(wave_scan(total), 63), row, p.idx_rows, lane, count,
                 [&](unsigned long long x) { return __hip_atomic_fetch_add(&pieces, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); });
  }
  __syncthreads();
  if (threadIdx.x == 0) *p.plan.noted = pieces;
}

static_assert(kQueueBytes == kQueueWords * 4, "estimate.h");
// What no pass before the launch has made ready: a work queue (or null), and of each q-block the blocks of its lists and of the
// longest (or null).  A wavefront per q-block.
__global__ __launch_bounds__(64) void ready_kernel(AttnParams p, int32_t* queue, uint32_t* totals) {
  const int lane = threadIdx.x;
  if (queue)
    for (int i = (int)blockIdx.x * 64 + lane; i < kQueueWords; i += (int)gridDim.x * 64) queue[i] = 0;
  if (!totals) return;
  const int row = p.qb_begin + (int)blockIdx.x - p.idx_row0;
  int total = 0, longest = 0;
  for (int h = lane; h < p.H; h += 64) {
    int n = p.col_cnt[(int64_t)h * p.idx_rows + row];
    n = n < 0 ? 0 : n > p.idx_pitch ? (int)p.idx_pitch : n;
    total += n;
    longest = longest > n ? longest : n;
  }
  total = wave_scan(total);
  longest = (int)wave_max((uint32_t)longest);
  if (lane == 63) {
    totals[32 * row] = (uint32_t)total;
    totals[32 * row + 1] = (uint32_t)longest;
  }
}

}  // namespace xattn

using namespace xattn;

// Whether the kernel of 64 rows per wavefront takes all q-blocks (else lists_decide).  It depends on the whole problem alone, so
// results do not depend on how a problem is spread over launches.
// 64 rows are for long lists: mostly without causality.  Whole calls, us, 32 / 64 rows: field 4000 276 / 257, 8000 832 / 757, 20000
// 4855 / 4344, 30000 with 2 heads 1037 / 921.
// Few units leave CUs to a single workgroup, where four wavefronts finish a list sooner than two: 1000 tokens 29.9 / 33.1, long
// text with few heads (64 rows from the 15th q-block on) 65536 with 4 241 / 273, 50000 with 8 257 / 299, 131072 with 2 339 / 367.
// On a cache lists are cut, and each piece starts with 32 keys that say little about the others: rows outgrow their reference
// maxima often, and nothing is gained over all.  Text of three seeds, 2048 on 63488 479, 271, 429 / 455, 274, 420 (with a queue),
// 500 on 60000 189, 132, 180 / 191, 129, 187, 8000 on 100000 665, 490, 495 / 659, 511, 517.
static bool all_rows64(int H, int nqb, int nkb, int causal) {
  return !causal && nkb < 2 * nqb && ((int64_t)H * nqb > 512 || nkb >= 192);
}

// Of prompts by themselves, with units enough that a second launch costs little (3 us without a q-block of its own, 50 for
// 32768 units that are the other's), the lists decide, q-block for q-block (long_lists).  Where q-blocks see fewer than 384
// blocks: 64 rows where lists have 8 blocks on average and the longest is less than twice that, as of video - unlike lists would
// give two launches with an end of their own each, and one long list takes twice as long (32768 tokens, few long heads, with a
// line on the total alone: 1340 us with 32 rows / 1640).  Whole calls, us, 32 rows / by the lists: video of 18000 tokens
// 1425 / 1274, of 32000 4180 / 3700; text of 32768, which stays with 32 rows, 535 / 533.  Longer ones outlast such ends: from 8
// blocks on average - but below 18432 units, where a prompt in which some heads keep a few long lists would lose, from 24.  Text of
// six seeds with 32 heads, 32 rows / from 24 / from 8: 131072 tokens 7443, 4753, 4846, 25027, 4709, 13684 / 7358, 4731, 4833, 22174,
// 4685, 12697 / 7149, 4728, 4831, 21813, 4684, 12264; 100000 4838, 3063, 3132, 15030, 3027, 8746 / 4768, 3045, 3115, 13150, 3012,
// 7945 / 4629, 3040, 3116, 12974, 3006, 7729; 80000 (20000 units) 3315, 2107, 2167, 9887, 2089, 5921 / 3316, 2107, 2158, 8947, 2075,
// 5748 / 3330, 2098, 2155, 8404, 2069, 5316; 64000 (16000) 2320, 1452, 1504, 6522, 1433, 3981 / 2312, 1456, 1493, 5846, 1424, 3973 /
// 2369, 1445, 1490, 5509, 1426, 3621; 50000 1666, 1033, 1059, 4172, 1017, 2653 / 1630, 1028, 1053, 3852, 1021, 2524 / 1726, 1038, 1068,
// 3517, 1014, 2442.
static int lists_decide(int H, int nqb, int nkb, int kv_off, int causal) {
  const int64_t units = (int64_t)H * nqb;
  if (!causal || kv_off >= 128 * kBlk || units < 3584) return kNot;
  return nkb < 384 ? kFrom8Alike : units < 18432 ? kFrom24 : kFrom8;
}

// Whether the 64-row kernel has a work queue: where units go several times through the places (us without / with: video of
// 65536 16840 / 15880; but a field of 4000, 768 like units, 229 / 235: dealt by the launch, the second round's find CUs of
// their own).
bool xattn::attention_queued(int num_heads, int q_len, int k_len, int causal) {
  const int nqb = (int)(((int64_t)q_len + kBlk - 1) / kBlk), nkb = (int)(((int64_t)k_len + kBlk - 1) / kBlk);
  const int64_t units = (int64_t)num_heads * nqb;
  return units > 1024 && (all_rows64(num_heads, nqb, nkb, causal) || lists_decide(num_heads, nqb, nkb, k_len - q_len, causal));
}

// Whether a unit is two workgroups', of 64 rows each, with a wavefront for half of every tile's keys: where units leave half of the
// CUs idle.  Only up to 16 key blocks, where no list is ever cut (plan_shape); it depends on the whole problem alone.  A prompt of 500
// tokens 23.3 -> 21.5 us, 1000 with 8 heads 25.9 -> 23.1, 900 with 16 29.2 -> 25.6.  (From there to the CUs' number: in_wide.)
// Dense attention without lists has whole units always: the sums' order differs, and its q-blocks are those of a longer prompt to the
// bit.  (With lists they are not, across this line: the same q-blocks in a call of more heads or tokens may differ in the last bits.)
static bool in_halves(int H, int nqb, int nkb) { return nkb <= 16 && (int64_t)H * nqb <= 128; }

// Whether a unit is a workgroup of eight wavefronts (attn_wide.h), one to a CU: where no XCD gets more of them than it has CUs (a prompt of
// 1100 tokens with 28 heads, whose 252 units the dispatch deals 36 to an XCD, 27.7 -> 31.5 us).  Only up to 16 key blocks: a workgroup
// that has the CU alone leaves it idle at a piece's start and end (500 tokens on 60000 151.5 -> 157.6, 1000 on 30000 182 -> 200; uncut
// 500 on 8700 gained 0.7 of 22.3), and cut or not the choice has to be one.  It depends on the whole problem alone, too.
static bool in_wide(int H, int Hkv, int nqb, int nkb) {
  return nkb <= 16 && (int64_t)H * nqb <= 256 && fullest_xcd(dispatch_shape(H, Hkv, nqb), nqb) <= kUnit / 2;
}

// Bytes of output from which the 32-row kernel stores its rows not temporal: they then leave the memory-side cache to q, k and v, which
// the estimate has just read.  Prompts, us: 4096 tokens of 32 / 32 heads 88.5 -> 87.1, 6500 134.8 -> 132.3, 5000 of 32 / 8 124.3 -> 117.1, 6500 of
// 28 / 4 124.1 -> 118.6, video of 7000 274.8 -> 270.3, 10000 of 32 / 8 258 -> 256; from 16000 tokens on they are equal.  The product that
// reads the output next finds a small one in that cache (a layer's 900 tokens on 3000 135.6 -> 137.3 us if stored so, 2100 on
// 6000 312.5 -> 313.9); with larger ones it is bound by its arithmetic (layers of 3500 to 12000 tokens are equal or gain).
// Not in the 64-row kernel, whose lists are long: video of 65536 tokens 15306 -> 15366 us, text of 131072 14373 -> 14405, of 50000 2650 ->
// 2675, fields equal.
constexpr int64_t kOutNtBytes = 24 << 20;
// Calls that load their queries so, too, where the estimate has read them and the attention reads them for the last time.  With a KV
// head per query head from so many bytes of output on, of 32 heads, text at two strides: 3100 tokens 67.1 -> 70.8, 68.7 -> 71.4, 3500 75.5 ->
// 76.2, 76.4 -> 77.9, 3900 86.4 -> 86.3, 83.1 -> 82.0, 4300 101.5 -> 97.5, 98.8 -> 97.5, 5500 123.7 -> 121.2, 116.5 -> 115.4, 8000 183.9 -> 183.0,
// 161.7 -> 160.4, 13000 327.6 -> 327.0, 294.1 -> 292.2; of 24 5000 equal, 6500 117.5 -> 116.7.
constexpr int64_t kQueriesNtBytes = 30 << 20;
// With fewer KV heads from so many bytes of q, k, v and output on: below, all of a call stays in the memory-side cache beside what
// came before it, and queries loaded so leave it (28 / 4 2000 tokens 41.2 -> 45.0, video of 6000 204.9 -> 211.2, of 8000 332 -> 338, 32 / 8 5000
// 117.1 -> 124.8, 3500 on 5000 112.6 -> 116.7; 97 to 140 MiB).  Above, three or six inputs in turn: 9000 of 32 / 8 206.9 -> 201.2, 11000
// 240 -> 236, 14000 of 28 / 4 219 -> 211, 5836 on 13528 136.9 -> 131.5, 4000 on 30000 145.4 -> 141.9, 7000 on 20000 215.0 -> 210.6; 8000 on 20000,
// 4000 on 60000 and video of 10000 to 16000 equal.  (One input again and again, up to 256 MiB of which stay, would be 3 to 10 % slower.)
constexpr int64_t kCallNtBytes = 160 << 20;

static int not_temporal(const AttnParams& p, bool lists) {
  const int64_t bytes = (int64_t)p.H * p.Lq * kHeadDim * 2, call = 2 * bytes + (int64_t)p.Hkv * p.Lk * kHeadDim * 4;
  if (bytes <= kOutNtBytes) return kNtNone;
  return lists && (p.H == p.Hkv ? bytes > kQueriesNtBytes : call > kCallNtBytes) ? kNtQueriesToo : kNtOutput;
}

// `p` for the 64-row kernel, `p32` for the 32-row one (they may deal units differently), `pieces` ids ahead of the units'; with a queue,
// `places` workgroups of the 64-row kernel.
template <bool kHasList, bool kPlanned>
static int launch_fwd(const AttnParams& p, const AttnParams& p32, int64_t pieces, int places, hipStream_t s) {
  const int64_t ids = pieces + p32.unit_ids;
  const bool all64 = all_rows64(p.H, p.nqb, p.nkb, p.causal);
  if (all64 || p.lists_decide) {
    hipLaunchKernelGGL((block_sparse_fwd64_kernel<kHasList, kPlanned>), dim3((unsigned)(p.queue ? places : pieces + p.unit_ids)), dim3(128), 0, s, p);
    if (hipGetLastError() != hipSuccess) return XATTN_ERR_LAUNCH;
  }
  if (all64) return XATTN_OK;
  if (kHasList && !kPlanned && in_halves(p.H, p.nqb, p.nkb)) {
    hipLaunchKernelGGL((block_sparse_fwd_kernel<true, false, true, kNtNone>), dim3((unsigned)(2 * ids)), dim3(256), 0, s, p32);
  } else if (kHasList && !kPlanned && in_wide(p.H, p.Hkv, p.nqb, p.nkb)) {
    static LdsLimit limit;
    if (limit.raise(reinterpret_cast<const void*>(&block_sparse_wide_kernel)) != hipSuccess) return XATTN_ERR_LAUNCH;
    hipLaunchKernelGGL(block_sparse_wide_kernel, dim3((unsigned)ids), dim3(512), kWideLds, s, p32);
  } else {
    auto kernel = block_sparse_fwd_kernel<kHasList, kPlanned, false, kNtNone>;
    const int nt = not_temporal(p, kHasList);
    if (nt == kNtOutput) kernel = block_sparse_fwd_kernel<kHasList, kPlanned, false, kNtOutput>;
    if (kHasList && nt == kNtQueriesToo) kernel = block_sparse_fwd_kernel<true, kPlanned, false, kNtQueriesToo>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)ids), dim3(256), 0, s, p32);
  }
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int xattn::block_sparse_impl(const void* q, const void* k, const void* v, void* out,
                                      const int32_t* col_idx, const int32_t* col_cnt, int64_t idx_pitch,
                                      int idx_rows, int idx_row0, int num_heads, int num_kv_heads, int q_len, int k_len,
                                      int head_dim,
                                      int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_h,
                                      int64_t k_stride_n, int64_t v_stride_h, int64_t v_stride_n,
                                      int64_t o_stride_h, int64_t o_stride_n, int q_block_begin, int q_block_end,
                                      int causal, float softmax_scale, void* stream,
                                      const AttnPlan* plan, bool note, int32_t* queue,
                                      uint32_t* totals, bool ready) {
  if (!q || !k || !v || !out) return XATTN_ERR_NULL;
  if (head_dim != kHeadDim) return XATTN_ERR_HEAD_DIM;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads) return XATTN_ERR_HEADS;
  if (q_len <= 0 || k_len <= 0) return XATTN_ERR_SHAPE;
  if ((col_idx == nullptr) != (col_cnt == nullptr)) return XATTN_ERR_NULL;
  const int64_t strides[] = {q_stride_h, q_stride_n, k_stride_h, k_stride_n,
                             v_stride_h, v_stride_n, o_stride_h, o_stride_n};
  for (int64_t s : strides)
    if (s % 8) return XATTN_ERR_ALIGN;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return XATTN_ERR_ALIGN;
  if (!tile_stride_ok(k_stride_n) || !tile_stride_ok(v_stride_n) || !tile_stride_ok(q_stride_n) || !tile_stride_ok(o_stride_n))
    return XATTN_ERR_SHAPE;
  if (!scale_ok(softmax_scale)) return XATTN_ERR_SHAPE;

  AttnParams p;
  p.q = static_cast<const __bf16*>(q);
  p.k = static_cast<const __bf16*>(k);
  p.v = static_cast<const __bf16*>(v);
  p.o = static_cast<__bf16*>(out);
  p.q_sh = q_stride_h; p.q_sn = q_stride_n; p.k_sh = k_stride_h; p.k_sn = k_stride_n;
  p.v_sh = v_stride_h; p.v_sn = v_stride_n; p.o_sh = o_stride_h; p.o_sn = o_stride_n;
  p.col_idx = col_idx; p.col_cnt = col_cnt; p.idx_pitch = idx_pitch;
  p.H = num_heads; p.Hkv = num_kv_heads; p.Lq = q_len; p.Lk = k_len;
  p.nqb = (q_len + kBlk - 1) / kBlk;
  p.nkb = (k_len + kBlk - 1) / kBlk;
  p.causal = causal ? 1 : 0;
  p.kv_off = k_len - q_len;
  p.scale_log2 = softmax_scale * kLog2e;
  if (q_block_end < 0) q_block_end = p.nqb;
  if (q_block_begin < 0 || q_block_begin >= q_block_end || q_block_end > p.nqb) return XATTN_ERR_SHAPE;
  // the lists may hold a window of q-block rows only; the q-blocks of this launch must lie inside it
  if (col_idx && (idx_pitch < 1 || idx_row0 < 0 || q_block_begin < idx_row0 || q_block_end > idx_row0 + idx_rows))
    return XATTN_ERR_SHAPE;
  p.idx_rows = idx_rows;
  p.idx_row0 = idx_row0;
  p.qb_begin = q_block_begin;
  p.qb_end = q_block_end;
  p.plan = plan ? *plan : AttnPlan{};
  p.lists_decide = lists_decide(p.H, p.nqb, p.nkb, p.kv_off, p.causal);
  const int q_blocks = q_block_end - q_block_begin;
  const DispatchShape alike = dispatch_shape(p.H, p.Hkv, q_blocks);
  const DispatchShape unlike = col_idx && p.causal ? unlike_lists_shape(p.H, p.Hkv, q_blocks) : alike;
  p.shape = p.lists_decide == kFrom8 || p.lists_decide == kFrom24 ? unlike : alike;      // (else the 64-row kernel's lists are much alike)
  const int64_t grid = grid_for(p.shape, q_blocks), grid32 = grid_for(unlike, q_blocks);
  const int64_t pieces = plan ? piece_ids_room((int64_t)plan_pieces(plan->shape, q_blocks)) : 0;
  if (pieces + (grid > grid32 ? grid : grid32) > 0x7fffffff) return XATTN_ERR_SHAPE;
  p.unit_ids = (int)grid;
  const int cus = resident_workgroups();
  if (cus <= 0) return XATTN_ERR_LAUNCH;
  const int places = 2 * cus / kQueues * kQueues;
  if (places == 0) queue = nullptr;
  p.queue = queue;
  p.totals = totals;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!ready && (queue || totals))
    hipLaunchKernelGGL(ready_kernel, dim3((unsigned)(q_block_end - q_block_begin)), dim3(64), 0, s, p, queue, totals);
  AttnParams p32 = p;
  p32.shape = unlike;
  p32.unit_ids = (int)grid32;
  if (plan) {
    if (note) hipLaunchKernelGGL(note_lists_kernel, dim3(1), dim3(1024), 0, s, p);
    return col_idx ? launch_fwd<true, true>(p, p32, pieces, places, s) : launch_fwd<false, true>(p, p32, pieces, places, s);
  }
  return col_idx ? launch_fwd<true, false>(p, p32, pieces, places, s) : launch_fwd<false, false>(p, p32, pieces, places, s);
}

extern "C" int xattn_block_sparse_fwd(const void* q, const void* k, const void* v, void* out,
                                      const int32_t* col_idx, const int32_t* col_cnt, int64_t idx_pitch,
                                      int idx_rows, int idx_row0, int num_heads, int num_kv_heads, int q_len, int k_len,
                                      int head_dim,
                                      int64_t q_stride_h, int64_t q_stride_n, int64_t k_stride_h,
                                      int64_t k_stride_n, int64_t v_stride_h, int64_t v_stride_n,
                                      int64_t o_stride_h, int64_t o_stride_n, int q_block_begin, int q_block_end,
                                      int causal, float softmax_scale, void* stream) {
  return block_sparse_impl(q, k, v, out, col_idx, col_cnt, idx_pitch, idx_rows, idx_row0, num_heads, num_kv_heads, q_len, k_len,
                           head_dim, q_stride_h, q_stride_n, k_stride_h, k_stride_n, v_stride_h, v_stride_n, o_stride_h,
                           o_stride_n, q_block_begin, q_block_end, causal, softmax_scale, stream, nullptr, false, nullptr, nullptr, true);
}

namespace {
PlanShape shape_of(int num_heads, int q_len, int k_len, bool listed) {
  PlanShape s = plan_shape(num_heads, q_len, k_len);
  if (listed) return s;
  s.last = -1;                          // all lists of a q-block alike, and the last q-block's like the others'
  if (s.units > kEvenUnits) s.per_qb = 0;
  return s;
}
}  // namespace

// Whether a launch over some of the q-blocks has the problem's queue, and totals: not where its units fit the places at once, for
// which another launch ahead, and memory, cost more than they give (us per window of text, with / without: 4 q-blocks of 32 heads
// 25.7 / 18.8, 16 29.4 / 27.4; video, 16 of 28 heads 165.5 / 162).
static bool launch_queued(int num_heads, int q_len, int k_len, int q_blocks, int causal) {
  return (int64_t)num_heads * q_blocks > 512 && attention_queued(num_heads, q_len, k_len, causal);
}

static size_t totals_bytes(int64_t rows, bool asked) { return asked ? plan_round((size_t)rows * 128) : 0; }

extern "C" size_t xattn_block_sparse_workspace_bytes(int num_heads, int q_len, int k_len, int idx_rows, int q_blocks) {
  if (num_heads <= 0 || q_len <= 0 || k_len <= 0 || idx_rows < 0 || q_blocks <= 0) return 0;
  const int64_t rows = idx_rows ? idx_rows : ((int64_t)q_len + kBlk - 1) / kBlk;
  const size_t plan = plan_bytes(shape_of(num_heads, q_len, k_len, idx_rows != 0), num_heads * rows, q_blocks);
  const bool queued = launch_queued(num_heads, q_len, k_len, q_blocks, 0) || launch_queued(num_heads, q_len, k_len, q_blocks, 1);
  return plan_round(plan) + (queued ? kQueueBytes + totals_bytes(rows, idx_rows != 0 && attention_asks_totals(num_heads, q_len, k_len, 1)) : 0);
}

extern "C" int xattn_block_sparse_fwd_ws(const void* q, const void* k, const void* v, void* out, void* workspace,
                                         size_t workspace_bytes, const int32_t* col_idx, const int32_t* col_cnt,
                                         int64_t idx_pitch, int idx_rows, int idx_row0, int num_heads, int num_kv_heads,
                                         int q_len, int k_len, int head_dim, int64_t q_stride_h, int64_t q_stride_n,
                                         int64_t k_stride_h, int64_t k_stride_n, int64_t v_stride_h, int64_t v_stride_n,
                                         int64_t o_stride_h, int64_t o_stride_n, int q_block_begin, int q_block_end,
                                         int causal, float softmax_scale, void* stream) {
  if (q_len <= 0 || k_len <= 0) return XATTN_ERR_SHAPE;
  if (q_block_end < 0) q_block_end = (q_len + kBlk - 1) / kBlk;
  const int nqb = (q_len + kBlk - 1) / kBlk, q_blocks = q_block_end - q_block_begin;
  const size_t need = xattn_block_sparse_workspace_bytes(num_heads, q_len, k_len, col_idx ? idx_rows : 0, q_blocks);
  const PlanShape shape = num_heads > 0 ? shape_of(num_heads, q_len, k_len, col_idx != nullptr) : PlanShape{};
  if (!col_idx) idx_rows = nqb, idx_row0 = 0;
  AttnPlan plan{};
  int32_t* queue = nullptr;
  if (shape.per_qb && need) {
    if (!workspace) return XATTN_ERR_NULL;
    if (workspace_bytes < need) return XATTN_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) & 255) return XATTN_ERR_ALIGN;
    plan = plan_at(shape, static_cast<char*>(workspace), (int64_t)num_heads * idx_rows, q_blocks);
  }
  uint32_t* totals = nullptr;
  if (workspace && workspace_bytes >= need && need >= kQueueBytes && !(reinterpret_cast<uintptr_t>(workspace) & 255) &&
      launch_queued(num_heads, q_len, k_len, q_blocks, causal)) {
    const bool asked = col_idx && attention_asks_totals(num_heads, q_len, k_len, 1);
    char* at = static_cast<char*>(workspace) + need - kQueueBytes - totals_bytes(idx_rows, asked);
    queue = reinterpret_cast<int32_t*>(at);
    if (asked && causal) totals = reinterpret_cast<uint32_t*>(at + kQueueBytes);
  }
  return block_sparse_impl(q, k, v, out, col_idx, col_cnt, idx_pitch, idx_rows, idx_row0, num_heads, num_kv_heads, q_len, k_len,
                           head_dim, q_stride_h, q_stride_n, k_stride_h, k_stride_n, v_stride_h, v_stride_n, o_stride_h,
                           o_stride_n, q_block_begin, q_block_end, causal, softmax_scale, stream, plan.noted ? &plan : nullptr, true, queue, totals, false);
}

bool xattn::attention_asks_totals(int num_heads, int q_len, int k_len, int causal) {
  return lists_decide(num_heads, (int)(((int64_t)q_len + kBlk - 1) / kBlk), (int)(((int64_t)k_len + kBlk - 1) / kBlk), k_len - q_len, causal) != 0;
}
