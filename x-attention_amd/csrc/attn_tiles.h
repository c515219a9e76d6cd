// K/V tile movement and workgroup dispatch shared by the attention-shaped
// kernels (block-sparse forward, block-mass profiler).
#pragma once
#include "xattn_common.h"

namespace xattn {

constexpr int kBlk = 128;          // block_size of the operator
constexpr int kTileBytes = kBlk * 256;   // one K or V tile in LDS
constexpr int kUnit = 64;                // workgroups resident on one XCD (32 CUs x 2)

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4;

// LDS tile layout: row n at byte n*256, its 16-byte chunk c stored at chunk
// c ^ swz(n).  swz takes all 16 values over 16 consecutive rows (row-per-lane
// b128 reads of one logical chunk are conflict-free) and moves rows n..n+3 into
// different 64-byte groups (the 4-row x 32-byte gathers of the transposing read
// are conflict-free too).
__device__ __forceinline__ int swz(int n) { return ((n & 3) << 2) | ((n >> 2) & 3); }

// Copies key block kb of one head (row stride sn elements) into an LDS tile.
// Wavefront w issues 8 instructions of 1 KiB (4 rows) each; voff[i] is the
// lane's byte offset inside the block for instruction i.  kPolicy: the loads' cache policy.
template <int kPolicy = 0>
__device__ __forceinline__ void copy_tile(const __bf16* base, int64_t sn, int len, int kb, const int (&voff)[8],
                                          char* tile, int wave) {
  const int rows_left = len - kb * kBlk;
  const int rows = rows_left < kBlk ? rows_left : kBlk;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(base + (int64_t)kb * kBlk * sn), 0, (int)((int64_t)rows * sn * 2), 0x00020000);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(tile + (wave * 8 + i) * 1024), 16, voff[i], 0, 0, kPolicy);
}

// The same copy issued from one assembly block, M0 (the LDS destination) included.  The compiler makes the
// transposing LDS reads wait for every buffer load into LDS it knows of (the two might alias), which exposes
// the whole copy latency at the next fragment read; loads issued this way are not counted by the compiler, so
// the caller waits for them itself (wait_vm0) before the barrier that publishes the tile.  Loads return in
// order, so the compiler's own vmcnt waits for its own loads stay sufficient.
__device__ __forceinline__ void copy_tile_async(const __bf16* base, int64_t sn, int len, int kb, const int (&voff)[8],
                                                char* tile, int wave) {
  const int rows_left = len - kb * kBlk;
  const int rows = rows_left < kBlk ? rows_left : kBlk;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(base + (int64_t)kb * kBlk * sn), 0, (int)((int64_t)rows * sn * 2), 0x00020000);
  const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)(tile + wave * 8 * 1024));
  asm volatile(
      "s_mov_b32 m0, %[dst]\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v0], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v1], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v2], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v3], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v4], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v5], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v6], %[rs], 0 offen lds\n\ts_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %[v7], %[rs], 0 offen lds"
      :
      : [dst] "s"(dst), [rs] "s"(rsrc), [v0] "v"(voff[0]), [v1] "v"(voff[1]), [v2] "v"(voff[2]), [v3] "v"(voff[3]),
        [v4] "v"(voff[4]), [v5] "v"(voff[5]), [v6] "v"(voff[6]), [v7] "v"(voff[7])
      : "memory", "m0", "scc");
}

__device__ __forceinline__ void tile_offsets(int64_t sn, int lane, int wave, int (&voff)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 4 * (wave * 8 + i) + (lane >> 4);
    const int c = (lane & 15) ^ swz(row);
    voff[i] = (int)(row * sn * 2) + (c << 4);
  }
}

// Division of numbers below 2^31 by the same divisor again and again: the high half of a product, and a shift.
struct Divisor {
  uint32_t mul;      // 0: the divisor is 1
  uint32_t shift;
};
inline Divisor divisor(uint32_t d) {
  Divisor v{0, 0};
  if (d <= 1) return v;
  while ((2ull << v.shift) < d) ++v.shift;            // 2^shift < d <= 2^(shift + 1)
  v.mul = (uint32_t)(((1ull << (32 + v.shift)) + d - 1) / d);
  return v;
}
__host__ __device__ inline uint32_t divided(uint32_t x, const Divisor& v) {
  return v.mul ? (uint32_t)((uint64_t)x * v.mul >> 32) >> v.shift : x;
}

// Workgroup ids are dealt round-robin to the 8 XCDs, and an XCD (32 CUs, two
// workgroups each, one L2) starts its workgroups in id order.  The ids, up to
// 64, that land on one XCD one after the other form a unit: the query heads of
// ONE KV head times a run of adjacent q-blocks, so what is resident on the XCD
// together streams the same K/V through its L2 at about the same place.  A KV
// head with more than 64 query heads is dealt as several head sets of equal
// size (each a dispatch group of its own).  Units are dealt to XCDs in turn;
// the dispatch group of a unit rotates with the q-block run, so every XCD sees
// every head equally often (heads differ by orders of magnitude in list
// length).  Runs go out last (longest, when causal) first, so of eight runs an
// XCD that sees a head in the first has more of it than one that sees it in the
// eighth: of the next eight it sees it that much later, the rotation runs
// backwards.  (Where two of 8 groups keep long lists of 256 q-blocks, an XCD
// had 20 % more than its share: text of 32768 tokens 1986 us, 1738 with the
// turn.)  Groups fewer than XCDs rotate every second or fourth run, or half the
// XCDs would never see a group.
struct DispatchShape {
  int group;       // query heads per KV head
  int sets;        // head sets per KV head (1 unless group > kUnit)
  int set_heads;   // query heads per set (<= kUnit)
  int n_groups;    // dispatch groups: Hkv * sets
  int unit_rows;   // q-blocks per unit
  int turn_shift;  // groups rotate once per 1 << turn_shift runs
  uint32_t unit_size;   // ids of a unit: kUnit, or as many as it needs where runs are few and that is at most half, or units are halved
  uint32_t unit_inv;    // 2^31 / unit_size, rounded up: ids are divided by a product
  Divisor by_groups, by_heads, by_group;   // n_groups, set_heads, group
};
// (head, q-block)s of the XCD that has most of them, units being dealt to the XCDs in turn.
inline int64_t fullest_xcd(const DispatchShape& d, int n_qblocks) {
  int64_t on[8] = {}, most = 0;
  unsigned unit = 0;
  for (int left = n_qblocks; left > 0; left -= d.unit_rows)
    for (int g = 0; g < d.n_groups; ++g) on[unit++ & 7] += left < d.unit_rows ? left : d.unit_rows;
  for (int64_t n : on) most = n > most ? n : most;
  return most * d.set_heads;
}

// Where a launch has fewer than eight runs, some XCDs may have a unit more than others, or the only ones.  There the number of runs
// is rounded up to one of which every XCD has as many, if the fullest XCD then has an eighth less to do (q-blocks per unit are rounded up,
// too, which may leave fewer runs than that, or a short last one).
// Prompts, us, whole units / rounded up: 650 tokens with 28 / 4 heads 29.1 / 26.9, 1150 33.7 / 32.0, 3000 (105 workgroups on the fullest XCD, 84)
// 62.3 / 60.6, video 84.9 / 79.6; lists of about 4 blocks: 8000 tokens of one head 31.3 / 23.3, 4000 of 4 / 1 30.6 / 23.1, 5000 of 12 / 12
// 38.5 / 33.8.  But 2800 tokens with 28 / 4 (91 and 84) 58.7 / 60.1, such lists 34.6 / 39.7, 5000 (154 and 147) 92.8 / 94.1, 52.8 / 56.4;
// and where the fullest has more than before, 4224 tokens with 16 / 2 (72 and 80), lists of 8 blocks 42.4 / 53.8.  Units of more than 32
// ids that a launch goes round in several times straddle an XCD's 64 places, which costs long lists 2 to 8 % of what evenness gives short ones
// (3000 of 28 / 4: lists of about 2 blocks 29.5 / 28.0, 4 39.5 / 42.9).  40003 tokens of 24 heads without causality, runs even
// already, in units of 63 instead of 64 15.57 -> 15.68 ms.
// And a unit of at most 32 workgroups then has no more ids than it needs.  An XCD deals its workgroups to its 32 CUs in turn, also those without work, so
// units rounded up to 16 or 32 ids put their work on the same CUs and left others idle (us, 64 ids / a power of two / now, text: 600
// tokens of 64 / 16 heads 29.0 / 32.6 / 28.9, 1240 of 32 / 16 36.3 / 39.5 / 36.3, 1112 of 32 / 32 38.9 / 39.7 / 36.2, 1240 of 24 / 24 40.0 / 41.0 /
// 37.0, 984 of 32 / 32 35.0 / 33.4 / 33.4); from 600 units on, of more
// than 32 ids, and with 8 / 8, 32 / 8, 28 / 4 and 40 / 8 heads, the three are within 1 or 2 %.
inline DispatchShape dispatch_shape(int H, int Hkv, int n_qblocks) {
  DispatchShape d;
  d.group = H / Hkv;
  d.sets = (d.group + kUnit - 1) / kUnit;
  d.set_heads = (d.group + d.sets - 1) / d.sets;
  d.n_groups = Hkv * d.sets;
  d.unit_rows = kUnit / d.set_heads;
  d.turn_shift = d.n_groups == 4 ? 1 : d.n_groups == 2 ? 2 : 0;
  const int runs = (n_qblocks + d.unit_rows - 1) / d.unit_rows;
  const int even = d.n_groups % 8 == 0 ? 1 : d.n_groups % 4 == 0 ? 2 : d.n_groups % 2 == 0 ? 4 : 8;
  const int wanted = (runs + even - 1) / even * even;
  if (runs < 8 && wanted != runs) {
    DispatchShape e = d;
    e.unit_rows = (n_qblocks + wanted - 1) / wanted;
    if (8 * fullest_xcd(e, n_qblocks) <= 7 * fullest_xcd(d, n_qblocks)) d = e;
  }
  if (d.unit_rows > n_qblocks) d.unit_rows = n_qblocks;
  const int work = d.set_heads * d.unit_rows;
  d.unit_size = (uint32_t)(runs < 8 && work <= kUnit / 2 ? work : kUnit);
  d.unit_inv = ((1u << 31) + d.unit_size - 1) / d.unit_size;
  d.by_groups = divisor((uint32_t)d.n_groups);
  d.by_heads = divisor((uint32_t)d.set_heads);
  d.by_group = divisor((uint32_t)d.group);
  return d;
}

// The same for q-blocks that keep lists of their own: heads' lists differ many times over, and an XCD that has a head's units of 64
// q-blocks has all of its long lists.  Units are halved, down to 16 workgroups, until there are 16 runs, over which a KV group goes round
// the XCDs twice.  Text, us, whole units / halved: 32 / 32 heads 9000 tokens 173 / 170.5, 17000 406 / 342, 32768 815 / 704, 65536 2210 / 1940,
// 100000 4640 / 4549; 32 / 8 8000 126.5 / 121.7, 10000 154 / 147, 13000 234.5 / 228.5, 17000 324 / 308; 28 / 4 8000 97 / 91.5.  Until there
// are 32 runs, or down to 32 workgroups only: 17000 of 32 / 32 342, 364.  Below 48 q-blocks lists are cut and shorter: 5000 of 32 / 32
// 96.3 / 98.5, 4500 of 28 / 4 equal.  Lists that are alike gain where units are few (video of 12000 of 28 / 4 687 / 661, 8000 of 32 / 32
// 397 / 385, of 32 / 8 357 / 358) and lose the XCD's common keys where they are many (20000 of 32 / 32, by the 64-row kernel, 1806 / 1850).  A
// halved unit has as many ids as work, also where that is more than half of kUnit (groups of 7: 35 workgroups in 64 ids, a mean of five inputs
// each, 28 / 4 11000 tokens 192.2 / 190.5, 13000 219.5 / 217.7, 16000 284.4 / 282.2, 56 / 8 13000 418 / 413, 9300 and 17900 equal).
inline DispatchShape unlike_lists_shape(int H, int Hkv, int n_qblocks) {
  DispatchShape d = dispatch_shape(H, Hkv, n_qblocks);
  if (n_qblocks < 48) return d;
  const int rows = d.unit_rows;
  while ((n_qblocks + d.unit_rows - 1) / d.unit_rows < 16 && d.unit_rows > 1 && d.unit_rows * d.set_heads > 16) d.unit_rows = (d.unit_rows + 1) / 2;
  if (d.unit_rows == rows) return d;
  d.unit_size = (uint32_t)(d.set_heads * d.unit_rows);
  d.unit_inv = ((1u << 31) + d.unit_size - 1) / d.unit_size;
  return d;
}

// Returns false for ids that carry no work.  The shape is computed once on the host (dispatch_shape) and the
// arithmetic is unsigned: this runs at the start of every workgroup, where its divisions are a measurable part
// of what a short unit costs.
__host__ __device__ inline bool map_workgroup(int id, const DispatchShape& d, int qb_begin, int qb_end, int* head,
                                              int* qb, int* kv_head) {
  if (id < 0) return false;
  const uint32_t x = (uint32_t)id & 7u, s = (uint32_t)id >> 3;
  const uint32_t at = (uint32_t)((uint64_t)s * d.unit_inv >> 31);      // s / unit_size (exact: s < 2^25 where it is not kUnit)
  const uint32_t unit = at * 8u + x, w = s - at * d.unit_size;
  const uint32_t ng = (uint32_t)d.n_groups, sh = (uint32_t)d.set_heads;
  const uint32_t run = divided(unit, d.by_groups);
  const uint32_t turn = (run & 8u ? ~run : run) & 7u;
  const uint32_t rotated = unit - run * ng + (turn >> d.turn_shift);
  const uint32_t dg = rotated - divided(rotated, d.by_groups) * ng;      // the unit's group, rotated by its run
  const uint32_t w_row = divided(w, d.by_heads), w_head = w - w_row * sh;
  const uint32_t from_end = run * (uint32_t)d.unit_rows + w_row;
  uint32_t set = 0, kvh = dg;
  if (d.sets != 1) {
    kvh = dg / (uint32_t)d.sets;
    set = dg - kvh * (uint32_t)d.sets;
  }
  const uint32_t in_group = set * sh + w_head;             // head index inside its KV group
  if (w >= sh * (uint32_t)d.unit_rows || from_end >= (uint32_t)(qb_end - qb_begin) || in_group >= (uint32_t)d.group)
    return false;
  *qb = qb_end - 1 - (int)from_end;
  *head = (int)(kvh * (uint32_t)d.group + in_group);
  *kv_head = (int)kvh;
  return true;
}
inline bool map_workgroup(int id, int H, int Hkv, int qb_begin, int qb_end, int* head, int* qb) {
  int kv_head;
  return map_workgroup(id, dispatch_shape(H, Hkv, qb_end - qb_begin), qb_begin, qb_end, head, qb, &kv_head);
}

// grid size of a launch over n_qblocks q-blocks
inline int64_t grid_for(const DispatchShape& d, int n_qblocks) {
  const int64_t runs = (n_qblocks + d.unit_rows - 1) / d.unit_rows;
  return (runs * d.n_groups + 7) / 8 * 8 * d.unit_size;
}
inline int64_t grid_for(int H, int Hkv, int n_qblocks) { return grid_for(dispatch_shape(H, Hkv, n_qblocks), n_qblocks); }

// Token strides of K and V the tile copies can address (byte offsets inside a
// 128-row tile are held in 32 bits), and a usable softmax scale.
inline bool tile_stride_ok(int64_t sn) { return sn >= kHeadDim && sn <= ((int64_t)1 << 22); }
inline bool scale_ok(float s) { return s > 0.f && s < 1e30f; }

}  // namespace xattn
