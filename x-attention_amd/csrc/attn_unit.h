// What the block-sparse attention kernels share: parameters, which (head, q-block) and list a workgroup has, masking, and
// how results leave.
#pragma once
#include "attn_plan.h"
#include "attn_tiles.h"
#include "xattn_common.h"

namespace xattn {

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
  DispatchShape shape;      // dispatch_shape(H, Hkv), computed on the host
  AttnPlan plan;            // kPlanned only
};

__device__ __forceinline__ int clamp_block(int kb, int nkb) { return kb < 0 ? 0 : (kb < nkb ? kb : nkb - 1); }

typedef const __attribute__((address_space(4))) int32_t* const_i32_ptr;

// What a workgroup works on.
struct Unit {
  int head, qb, kvh;
  int piece;                 // which piece of its list, or -1: all of it
  int skip;                  // workgroups ahead of the units'
  int n_blocks, first;       // blocks of the list or piece; first: where it starts among the visible blocks (no list)
  const_i32_ptr list;        // the column list is read through the scalar cache (uniform, read-only)
  int cuts, part0;           // pieces of this list, the first one's place in the plan
};

// The (head, q-block) of this workgroup; false: nothing is left for it.
template <bool kPlanned>
__device__ __forceinline__ bool find_unit(const AttnParams& p, Unit& u) {
  u.piece = -1;
  u.skip = 0;
  if (kPlanned) {
    const int pieces = ((const_i32_ptr)(uintptr_t)p.plan.noted)[0], per_xcd = (pieces + 7) / 8;   // (the low half)
    u.skip = per_xcd * 8;
    if ((int)blockIdx.x < u.skip) {
      const int at = p.plan.shape.in_turn ? (int)blockIdx.x : (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
      if (at >= pieces) return false;
      const_i32_ptr entry = (const_i32_ptr)(uintptr_t)p.plan.pieces + 2 * at;
      const int unit = entry[0];
      u.piece = entry[1];
      u.head = unit / p.idx_rows;
      u.qb = unit - u.head * p.idx_rows + p.idx_row0;
      u.kvh = u.head / p.shape.group;
      return u.qb >= p.qb_begin && u.qb < p.qb_end;      // (q-blocks may be shared among two launches)
    }
  }
  return map_workgroup((int)blockIdx.x - u.skip, p.shape, p.qb_begin, p.qb_end, &u.head, &u.qb, &u.kvh);
}
__device__ __forceinline__ int64_t unit_slot(const AttnParams& p, const Unit& u) { return (int64_t)u.head * p.idx_rows + (u.qb - p.idx_row0); }

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
    const int q_last = (u.qb * kBlk + kBlk - 1 < p.Lq ? u.qb * kBlk + kBlk - 1 : p.Lq - 1) + p.kv_off;
    const int visible = p.causal ? (q_last < 0 ? 0 : q_last / kBlk + 1) : p.nkb;
    u.n_blocks = visible < p.nkb ? visible : p.nkb;
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
// that wait was a quarter of a workgroup's life.  Staged through 8 KiB of LDS
// (free once the sweep is over), 16 lanes write one 256-byte row: 64 full-line requests.
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
    __builtin_amdgcn_raw_buffer_store_b128(w, ores, (int)(voff0 + (uint32_t)(i * 4) * row_bytes), 0, 0);
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
// The pieces' results combined into the registers of a finished sweep, in the order of the list.
__device__ __forceinline__ void load_partials(float* part, int pieces, int wave, int lane, int r, int hh, f32x16 (&oacc)[4], float& l_run) {
  const int at = (128 * 128 + wave * 32 + r) * 4;
  auto ml = [&](int s, int which) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(part_resource(part + (int64_t)s * kPartFloats), at + which * 512, 0, kDeviceScope));
  };
  float m = -INFINITY, l = 0.f;
#pragma unroll 4
  for (int s = 0; s < pieces; ++s) m = fmaxf(m, ml(s, 0));
  const float safe = m == -INFINITY ? 0.f : m;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[i][v] = 0.f;
  for (int s = 0; s < pieces; ++s) {
    const __amdgpu_buffer_rsrc_t res = part_resource(part + (int64_t)s * kPartFloats);
    const float w = fast_exp2(ml(s, 0) - safe);      // 0 where the item saw no key of this row
    l += w * ml(s, 1);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 o = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(res, (wave * 16 * 64 + lane) * 16 + (dt * 4 + g) * 1024, 0, kDeviceScope));
#pragma unroll
        for (int u = 0; u < 4; ++u) oacc[dt][g * 4 + u] += w * o[u];
      }
  }
  l_run = hh == 0 ? l : 0.f;
}

}  // namespace xattn
