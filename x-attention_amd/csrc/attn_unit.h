// What the block-sparse attention kernels share: parameters, which (head, q-block) and list a workgroup has, masking, and
// how results leave.
#pragma once
#include "attn_plan.h"
#include "attn_tiles.h"
#include "xattn_common.h"

namespace xattn {

// Which q-blocks are the 64-row kernel's: all of a problem's or none; those whose lists have so many blocks on average (and are much
// alike).
enum ListsDecide { kNot, kFrom8, kFrom8Alike, kFrom24 };

struct AttnParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  __bf16* o;
  int64_t q_sh, q_sn, k_sh, k_sn, v_sh, v_sn, o_sh, o_sn;  // element strides (head, token)
  const int32_t* col_idx;   // [H, idx_rows, idx_pitch] ascending k-block ids, or null = all visible
  const int32_t* col_cnt;   // [H, idx_rows]
  int64_t idx_pitch;
  int idx_rows;             // q-block rows per head in col_idx / col_cnt
  int idx_row0;             // q-block held by their row 0
  int H, Hkv, Lq, Lk, nqb, nkb;
  int qb_begin, qb_end;     // q-blocks handled by this launch
  int causal, kv_off;       // kv_off = Lk - Lq
  float scale_log2;         // softmax_scale * log2(e)
  DispatchShape shape;      // dispatch_shape of the launch, computed on the host
  AttnPlan plan;            // kPlanned only
  int32_t* queue;           // this launch's work queue (kQueueWords, zero), or null: one workgroup per id
  int unit_ids;             // ids of units, grid_for()
  int lists_decide;         // ListsDecide: q-blocks with long lists are the 64-row kernel's, others the 32-row's
  const uint32_t* totals;   // blocks of a q-block's lists and of the longest at 32 * (q-block - idx_row0), or null: to be found
};

// The kernel's parameters, read anew: between two units nothing that is computed from them is kept, which would take more
// scalar registers than there are.
__device__ __forceinline__ const AttnParams& reread_params() {
  auto at = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const AttnParams*)at;
}

// Requests every line of the kernel's parameters, so that none is waited for on its own.
__device__ __forceinline__ void touch_params() {
  typedef const __attribute__((address_space(4))) uint32_t* word_ptr;
  const word_ptr at = (word_ptr)__builtin_amdgcn_kernarg_segment_ptr();
  uint32_t w[(sizeof(AttnParams) + 63) / 64];
#pragma unroll
  for (uint32_t i = 0; i < sizeof(w) / 4; ++i) w[i] = at[16 * i];
#pragma unroll
  for (uint32_t i = 0; i < sizeof(w) / 4; ++i) asm volatile("" ::"s"(w[i]));
}

__device__ __forceinline__ int clamp_block(int kb, int nkb) { return kb < 0 ? 0 : (kb < nkb ? kb : nkb - 1); }

typedef const __attribute__((address_space(4))) int32_t* const_i32_ptr;

// Blocks that a q-block sees without lists.
__device__ __forceinline__ int visible_blocks(const AttnParams& p, int qb) {
  const int q_last = (qb * kBlk + kBlk - 1 < p.Lq ? qb * kBlk + kBlk - 1 : p.Lq - 1) + p.kv_off;
  const int visible = p.causal ? (q_last < 0 ? 0 : q_last / kBlk + 1) : p.nkb;
  return visible < p.nkb ? visible : p.nkb;
}

// Whether q-block qb is the 64-row kernel's, where its lists decide.  By whole wavefronts, the same for all.
__device__ __forceinline__ bool long_lists(const AttnParams& p, int total, int longest) {
  return total >= (p.lists_decide == kFrom24 ? 24 : 8) * p.H && (p.lists_decide != kFrom8Alike || longest * p.H < 2 * total);
}
template <bool kHasList>
__device__ __forceinline__ bool has_rows64(const AttnParams& p, int qb) {
  if (!kHasList) return long_lists(p, p.H * visible_blocks(p, qb), visible_blocks(p, qb));
  if (p.totals) {
    const const_i32_ptr of = (const_i32_ptr)(uintptr_t)(p.totals + 32 * (qb - p.idx_row0));
    return long_lists(p, of[0], of[1]);
  }
  int total = 0, longest = 0;
  for (int h = (int)(threadIdx.x & 63); h < p.H; h += 64) {
    int n = p.col_cnt[(int64_t)h * p.idx_rows + (qb - p.idx_row0)];
    n = n < 0 ? 0 : n > p.idx_pitch ? (int)p.idx_pitch : n;
    total += n;
    longest = longest > n ? longest : n;
  }
  return long_lists(p, __builtin_amdgcn_readlane(wave_scan(total), 63), (int)wave_max((uint32_t)longest));
}

// What an id stands for.
struct Unit {
  int head, qb, kvh;
  int piece;                 // which piece of its list, or -1: all of it
  int skip;                  // ids ahead of the units'
  int n_blocks, first;       // blocks of the list or piece; first: where it starts among the visible blocks (no list)
  const_i32_ptr list;        // the column list is read through the scalar cache (uniform, read-only)
  int cuts, part0;           // pieces of this list, the first one's place in the plan
  int kb, kb_next;           // the sweep's first two blocks
};

// The same in scalar registers: from one turn of a loop to the next the compiler does not see that all lanes have the same.
__device__ __forceinline__ Unit uniform(const Unit& u) {
  auto one = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  Unit v;
  v.head = one(u.head), v.qb = one(u.qb), v.kvh = one(u.kvh), v.piece = one(u.piece), v.skip = one(u.skip);
  v.n_blocks = one(u.n_blocks), v.first = one(u.first), v.cuts = one(u.cuts), v.part0 = one(u.part0), v.kb = one(u.kb), v.kb_next = one(u.kb_next);
  const uintptr_t list = (uintptr_t)u.list;
  v.list = (const_i32_ptr)((uintptr_t)(uint32_t)one((int)list) | (uintptr_t)(uint32_t)one((int)(list >> 32)) << 32);
  return v;
}

__device__ __forceinline__ PieceIds pieces_noted(const AttnParams& p) {
  const const_i32_ptr at = (const_i32_ptr)(uintptr_t)p.plan.noted;
  return PieceIds{at[0], at[1]};
}

// The (head, q-block) with this id; false: there is none.
template <bool kPlanned>
__device__ __forceinline__ bool find_place(const AttnParams& p, int id, Unit& u) {
  u.piece = -1;
  u.skip = 0;
  if (kPlanned) {
    const PieceIds noted = pieces_noted(p);
    u.skip = noted.ids();
    if (id < u.skip) {
      int i = id, pieces = noted.whole;
      const bool rest = id >= noted.whole_ids();
      if (rest) i -= noted.whole_ids(), pieces = noted.rests;
      const int at = p.plan.shape.in_turn ? i : (i & 7) * ((pieces + 7) / 8) + (i >> 3);
      if (at >= pieces) return false;
      const_i32_ptr entry = (const_i32_ptr)(uintptr_t)p.plan.pieces + 2 * (rest ? p.plan.room - 1 - at : at);
      const int unit = entry[0];
      u.piece = entry[1];
      u.head = unit / p.idx_rows;
      u.qb = unit - u.head * p.idx_rows + p.idx_row0;
      u.kvh = (int)divided((uint32_t)u.head, p.shape.by_group);
      return true;
    }
    // Where pieces are most of the work, what stays whole are short lists, often of the same few KV heads: they go to the XCDs in
    // turn, each q-block's heads from another one on (as units of the dispatch, 64 more on some XCDs than on others).
    const uint32_t rows = (uint32_t)(p.qb_end - p.qb_begin), heads = (uint32_t)p.H, kv_heads = (uint32_t)p.Hkv;
    if (p.plan.shape.rests_last && 2 * (uint32_t)noted.whole >= rows * heads) {
      const uint32_t w = (uint32_t)(id - u.skip), row = w / heads;
      if (row >= rows) return false;
      const uint32_t turned = (w - row * heads + row) % heads, of = turned / kv_heads;
      u.kvh = (int)(turned - of * kv_heads);
      u.head = (int)((uint32_t)u.kvh * (heads / kv_heads) + of);
      u.qb = p.qb_end - 1 - (int)row;
      return true;
    }
  }
  return map_workgroup(id - u.skip, p.shape, p.qb_begin, p.qb_end, &u.head, &u.qb, &u.kvh);
}
// ... or it is the other kernel's.
template <bool kHasList, bool kPlanned, bool kRows64>
__device__ __forceinline__ bool find_unit(const AttnParams& p, int id, Unit& u) {
  return find_place<kPlanned>(p, id, u) && (!p.lists_decide || has_rows64<kHasList>(p, u.qb) == kRows64);
}
__device__ __forceinline__ int64_t unit_slot(const AttnParams& p, const Unit& u) { return (int64_t)u.head * p.idx_rows + (u.qb - p.idx_row0); }

// The work queue.  Workgroups of a launch are dealt to the XCDs in turn, one XCD's are never another's, and a workgroup keeps
// its place until its stores are acknowledged.  So XCDs with like numbers of workgroups ended far apart (video of 65536 14.5 to
// 16.0 ms, where only clocks differ), and a tenth of the places stood empty.  With a queue as many workgroups are launched as fit.
// Workgroup b starts with id b and goes on with those of its queue, b % 32: ids that leave the same rest, which its XCD has
// anyway.  (An answer takes 1 to 2 us, and a counter gives four in a us: with one per XCD the wait was 4 us of a short list's 15.)
// queue[32 c]: what queue c has handed out beyond the ids that its workgroups start with.
constexpr int kQueues = 32, kQueueWords = kQueues * 32;
// Takes the next id of this workgroup's queue; one lane (resolved by next_id).
__device__ __forceinline__ int ask_next(const AttnParams& p) {
  return __hip_atomic_fetch_add(p.queue + (blockIdx.x % kQueues) * 32, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The id that lane 0 was given, or that another queue has left, or -1.  By a whole wavefront.  Short lists (`few` blocks the
// last time) are left to their own workgroups where a queue has a single one left; so are others after four vain tries.
template <bool kPlanned>
__device__ __forceinline__ int next_id(const AttnParams& p, int ticket, int lane, bool few) {
  const int ids = (kPlanned ? pieces_noted(p).ids() : 0) + p.unit_ids, first = (int)(gridDim.x / kQueues);
  const int id = (first + __builtin_amdgcn_readfirstlane(ticket)) * kQueues + (int)(blockIdx.x % kQueues);
  if (id < ids) return id;
  for (int i = 0; i < 4; ++i) {
    int left = 0;
    if (lane < kQueues)
      left = (ids - lane + kQueues - 1) / kQueues - first - __hip_atomic_load(p.queue + lane * 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t most = wave_max(left > (few ? 1 : 0) ? (uint32_t)left * kQueues + (uint32_t)lane : 0u);
    if (most == 0) return -1;
    const int c = (int)(most % kQueues);
    int taken = 0;
    if (lane == 0) taken = __hip_atomic_fetch_add(p.queue + c * 32, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int other = (first + __builtin_amdgcn_readfirstlane(taken)) * kQueues + c;
    if (other < ids) return other;
  }
  return -1;
}

// Its list; false: others have it.
template <bool kHasList, bool kPlanned>
__device__ __forceinline__ bool find_list(const AttnParams& p, Unit& u) {
  const int64_t slot = unit_slot(p, u);
  u.list = nullptr;
  u.first = u.cuts = u.part0 = 0;
  if (kHasList) {
    u.list = (const_i32_ptr)(uintptr_t)(p.col_idx + slot * p.idx_pitch);
    const int n = ((const_i32_ptr)(uintptr_t)p.col_cnt)[slot];
    u.n_blocks = n < 0 ? 0 : (n > p.idx_pitch ? (int)p.idx_pitch : n);
  } else {
    u.n_blocks = visible_blocks(p, u.qb);
  }
  if (kPlanned) {
    const uint32_t cut = u.n_blocks > p.plan.shape.min_piece ? (uint32_t)((const_i32_ptr)(uintptr_t)p.plan.cut)[slot] : 0;
    if (cut != 0) {
      if (u.piece < 0) return false;
      u.cuts = cut_pieces(cut);
      u.part0 = cut_at(cut);
      const int length = cut_length(cut);
      if (kHasList) u.list += u.piece * length;
      else u.first = u.piece * length;
      u.n_blocks = u.piece + 1 < u.cuts ? length : u.n_blocks - u.piece * length;
    }
  }
  return true;
}

// The unit of id `id` and its list for the 32-row kernel, with the list's first two blocks; false: there is nothing for this workgroup.
// What is read from memory - the totals that choose the kernel, the list's length, its head, where it is cut - is requested
// together: each is an answer of about 0.4 us, and one after the other they were most of the 1 to 1.5 us ahead of a unit's first
// copies.  (With the parameters' lines, the map's divisions and the list's next entry in the sweep, calls, us: 1000 tokens 30.8 -> 30.4, 4096
// of 32 / 32 heads 71.3 -> 70.5, a layer's 500 tokens 97.1 -> 96.3; attention of 500 tokens 11.7 -> 11.1; 131072 and chunks equal.)
template <bool kHasList, bool kPlanned>
__device__ __forceinline__ bool find_work(const AttnParams& p, int id, Unit& u) {
  if (!kHasList) {
    if (!find_unit<false, kPlanned, false>(p, id, u) || !find_list<false, kPlanned>(p, u)) return false;
    u.kb = u.first;
    u.kb_next = u.first + 1;
    return true;
  }
  if (!find_place<kPlanned>(p, id, u)) return false;
  const int64_t slot = unit_slot(p, u);
  const int last = p.idx_pitch > 0x7fffffff ? 0x7fffffff : (int)p.idx_pitch - 1, second = last > 0 ? 1 : 0;
  const bool by_totals = p.lists_decide && p.totals;
  u.list = (const_i32_ptr)(uintptr_t)(p.col_idx + slot * p.idx_pitch);
  const const_i32_ptr of = by_totals ? (const_i32_ptr)(uintptr_t)(p.totals + 32 * (u.qb - p.idx_row0)) : u.list;
  int n = ((const_i32_ptr)(uintptr_t)p.col_cnt)[slot], head0 = u.list[0], head1 = u.list[second];
  int total = of[0], longest = of[by_totals ? 1 : second], word = kPlanned ? ((const_i32_ptr)(uintptr_t)p.plan.cut)[slot] : 0;
  asm volatile("" : "+s"(n), "+s"(head0), "+s"(head1), "+s"(total), "+s"(longest), "+s"(word));      // (not each where it is needed)
  if (p.lists_decide && (p.totals ? long_lists(p, total, longest) : has_rows64<true>(p, u.qb))) return false;
  u.n_blocks = n < 0 ? 0 : n > p.idx_pitch ? (int)p.idx_pitch : n;
  u.first = u.cuts = u.part0 = 0;
  u.kb = clamp_block(head0, p.nkb);
  u.kb_next = clamp_block(head1, p.nkb);
  if (kPlanned && u.n_blocks > p.plan.shape.min_piece && word != 0) {
    if (u.piece < 0) return false;
    u.cuts = cut_pieces((uint32_t)word);
    u.part0 = cut_at((uint32_t)word);
    const int length = cut_length((uint32_t)word);
    u.n_blocks = u.piece + 1 < u.cuts ? length : u.n_blocks - u.piece * length;
    u.list += u.piece * length;
    u.kb = clamp_block(u.list[0], p.nkb);
    u.kb_next = clamp_block(u.list[u.n_blocks > 1 ? 1 : 0], p.nkb);
  }
  return true;
}

// The next id that has work, from the ticket of thread 0, the same for all wavefronts; -1: there is none.
template <bool kHasList, bool kPlanned>
__device__ __forceinline__ int hand_out(const AttnParams& p, int ticket, int wave, int lane, bool few, char* scratch) {
  if (wave == 0) {
    int next;
    for (;;) {
      next = next_id<kPlanned>(p, ticket, lane, few);
      Unit u;
      if (next < 0 || (find_unit<kHasList, kPlanned, true>(p, next, u) && find_list<kHasList, kPlanned>(p, u))) break;
      if (lane == 0) ticket = ask_next(p);
    }
    if (lane == 0) *reinterpret_cast<int*>(scratch) = next;
  }
  __syncthreads();
  const int id = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(scratch));
  __syncthreads();
  return id;
}

// A lane's place in the fragments of a tile in LDS.
struct FragAddr {
  int kaddr[8];             // K fragment of k-step s: row r of 32 keys, logical chunk 2s + hh
  int vaddr[4][2];          // V^T fragment of 16 keys (feature tile dt, half a)
};
__device__ __forceinline__ void frag_addressing(int lane, FragAddr& a) {
  const int r = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int s = 0; s < 8; ++s) a.kaddr[s] = r * 256 + (((2 * s + hh) ^ swz(r)) << 4);
  // the transposing read hands lane l the feature dt*32 + (l % 32) of keys
  // 16ks + 8a + 4hh + {0..3}; as a source lane it points at key e = (l%16)/4 of
  // that quad, features dt*32 + 16*((l/16)%2) + 4*(l%4) .. +3.
  const int e = (lane & 15) >> 2, j = lane & 3, g2 = (lane >> 4) & 1;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      const int row = 8 * h2 + 4 * hh + e;                       // + 16*ks
      const int c = dt * 4 + 2 * g2 + (j >> 1);
      a.vaddr[dt][h2] = row * 256 + ((c ^ swz(row)) << 4) + (j & 1) * 8;
    }
}

// token-level masking of the scores of 32 keys from key0 on: keys past the sequence end, and (causal) keys after the query.
// The lane's last visible key is taken relative to its first key of the step once, so that each score costs one
// compare against a constant and one select.
__device__ __forceinline__ void mask_step(f32x16& s, int key0, int hh, int q_pos, int Lk, int causal) {
  int last = Lk - 1;
  if (causal) last = last < q_pos ? last : q_pos;
  const int lim = last - key0 - hh * 4;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int c = (v >> 2) * 8 + (v & 3);     // key offset inside the step, without the lane's hh * 4
    s[v] = c > lim ? -INFINITY : s[v];
  }
}

// Normalises 32 output rows (group `wave` of the q-block's four) and stores them through LDS.  Lane (r, hh) holds half of row r in
// 8-byte pieces; written straight to memory those are 512 sixteen-byte requests per wavefront, and a
// workgroup's registers and LDS stay allocated until its last store is acknowledged - on lists of a few blocks
// that wait was a quarter of a workgroup's life.  Staged through 8 KiB of LDS,
// 16 lanes write one 256-byte row: 64 full-line requests.
constexpr int kOutStage = 8192;      // bytes per wavefront
template <bool kNt = false>
__device__ __forceinline__ void store_out(const AttnParams& p, int head, int qb, int wave, int lane, int r, int hh,
                                          const f32x16 (&oacc)[4], float l_run, char* stage) {
  const float l_tot = half_sum(l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      u32x2 w;
      w[0] = pack_bf16(oacc[dt][g * 4 + 0] * inv, oacc[dt][g * 4 + 1] * inv);
      w[1] = pack_bf16(oacc[dt][g * 4 + 2] * inv, oacc[dt][g * 4 + 3] * inv);
      const int c = dt * 4 + g;                          // 16-byte chunk of the row; XOR-swizzled against bank conflicts
      *reinterpret_cast<u32x2*>(stage + r * 256 + ((c ^ (r & 15)) << 4) + hh * 8) = w;
    }
  // written and read by the same wavefront: the LDS keeps a wavefront's accesses in order, no barrier.
  // The rows leave through a buffer resource that ends with the sequence (rows past it are dropped), rebased to
  // the q-block so that a lane's offset is one 32-bit product plus a multiple of four rows.
  const int rows_left = p.Lq - qb * kBlk;
  const int rows = rows_left < kBlk ? rows_left : kBlk;
  const __amdgpu_buffer_rsrc_t ores = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.o + (int64_t)head * p.o_sh + (int64_t)qb * kBlk * p.o_sn), 0, (int)((int64_t)rows * p.o_sn * 2), 0x00020000);
  const int c = lane & 15;
  const uint32_t row_bytes = (uint32_t)p.o_sn * 2u;
  const uint32_t voff0 = (uint32_t)(wave * 32 + (lane >> 4)) * row_bytes + (uint32_t)c * 16u;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = i * 4 + (lane >> 4);
    const u32x4 w = *reinterpret_cast<const u32x4*>(stage + row * 256 + ((c ^ (row & 15)) << 4));
    __builtin_amdgcn_raw_buffer_store_b128(w, ores, (int)(voff0 + (uint32_t)(i * 4) * row_bytes), 0, kNt ? kNotTemporal : 0);
  }
}

// What a piece of a cut list leaves behind: accumulators as the lanes hold them (1 KiB per store), row maxima and sums.
// Pieces of a list run on any XCD, each with an L2 of its own: stores and loads are at device scope (kDeviceScope: they go
// through to, and come from, memory that all of them share).
constexpr int kDeviceScope = 16;   // sc1
__device__ __forceinline__ __amdgpu_buffer_rsrc_t part_resource(float* part) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, kPartFloats * 4, 0x00020000);
}
__device__ __forceinline__ void store_partial(float* part, int wave, int lane, int r, int hh, const f32x16 (&oacc)[4], float m_run,
                                              float l_run) {
  const __amdgpu_buffer_rsrc_t res = part_resource(part);
  const float l_tot = half_sum(l_run);
  const int dst = (wave * 16 * 64 + lane) * 16;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 w;
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = oacc[dt][g * 4 + u];
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, w), res, dst + (dt * 4 + g) * 1024, 0, kDeviceScope);
    }
  if (hh == 0) {
    const int at = (128 * 128 + wave * 32 + r) * 4;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, m_run), res, at, 0, kDeviceScope);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, l_tot), res, at + 512, 0, kDeviceScope);
  }
}
// The pieces' results combined into the registers of a finished sweep, in the order of the list.  One workgroup reads up to
// 16 x 66 KiB here while the others may be done: a piece's 16 KiB per wavefront are requested while the one before it is added
// up (each load behind the last one's sum: 160 us for 16 pieces).  A piece's place is the loads' scalar offset, which the
// buffer's bounds check does not see: only pieces of the list are named, and nothing else is added, not even times 0.
__device__ __forceinline__ void load_partials(float* part, int pieces, int wave, int lane, int r, int hh, f32x16 (&oacc)[4], float& l_run) {
  const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc((void*)part, 0, pieces * kPartFloats * 4, 0x00020000);
  const int at = (128 * 128 + wave * 32 + r) * 4, from = (wave * 16 * 64 + lane) * 16;
  auto ml = [&](int s, int which) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(res, at + which * 512, s * kPartFloats * 4, kDeviceScope));
  };
  struct Piece {
    float m, l;
    f32x4 o[16];
  } a, b;
  auto request = [&](Piece& x, int s) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    x.m = ml(s, 0);
    x.l = ml(s, 1);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      x.o[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(res, from + i * 1024, s * kPartFloats * 4, kDeviceScope));
    __builtin_amdgcn_sched_barrier(0);
  };
  float tops[kMostPieces], m = -INFINITY, l = 0.f;
#pragma unroll
  for (int s = 0; s < kMostPieces; ++s) tops[s] = ml(s < pieces ? s : pieces - 1, 0);
#pragma unroll
  for (int s = 0; s < kMostPieces; ++s) m = fmaxf(m, tops[s]);
  const float safe = m == -INFINITY ? 0.f : m;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[i][v] = 0.f;
  auto add = [&](const Piece& x) __attribute__((always_inline)) {
    const float w = fast_exp2(x.m - safe);      // 0 where the piece saw no key of this row
    l += w * x.l;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) oacc[i >> 2][(i & 3) * 4 + u] += w * x.o[i][u];
  };
  read_ahead(pieces, a, b, request, add);
  l_run = hh == 0 ? l : 0.f;
}

}  // namespace xattn
