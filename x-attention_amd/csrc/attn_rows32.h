// Block-sparse attention with 32 query rows per wavefront, where lists may be short or units few (all_rows64 and lists_decide
// have the rule).
//
// Work decomposition: one workgroup (4 wavefronts) per (head, q-block); each
// wavefront owns 32 query rows.  Scores are produced transposed,
// S^T = K Q^T, so that one lane owns one query row (softmax statistics need a
// single cross-lane exchange) and the fp32 accumulator registers of S^T are,
// unchanged, the B operand of O^T += V^T P^T.  K and V tiles (128 keys x 128
// features, row-major, XOR-swizzled 16-byte chunks) are copied global -> LDS by
// buffer loads that write LDS directly; keys past the sequence end fall outside
// the buffer resource and arrive as zeros.  K fragments are read with
// ds_read_b128, V^T fragments with the transposing ds_read_b64_tr_b16, both
// issued one k-step ahead of the MFMAs that consume them.  The copy of the next
// K tile overlaps softmax and P.V, the copy of the next V tile overlaps Q.K^T
// (both issued from assembly, see copy_tile_async: the compiler would make the
// transposing reads wait for every copy it knows of).
// Two workgroups fit per CU (64 KiB LDS each) so one's softmax overlaps the
// other's MFMA.  The query block enters and the output block leaves through
// the same LDS tiles as full 256-byte rows (the q-block is copied like a K
// tile before V_0 is requested; the output is staged in the K tile after the
// sweep): row-per-lane accesses to global memory would be hundreds of partial
// line requests per wavefront, and a workgroup keeps its registers and LDS
// until the last of its stores is acknowledged.
#pragma once
#include "attn_unit.h"

namespace xattn {

// S^T = K_j Q^T on NT x 32 keys: lane owns query row r, key rows 8g + 4hh + t of each 32-row tile
template <int NT>
__device__ __forceinline__ void qk_tile(const char* Ks, const int (&kaddr)[8], const bf16x8 (&qreg)[8], f32x16 (&sacc)[NT]) {
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) sacc[i][v] = 0.f;
  bf16x8 kf[2][NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) kf[0][nt] = *reinterpret_cast<const bf16x8*>(Ks + kaddr[0] + nt * 8192);
  __builtin_amdgcn_sched_group_barrier(0x100, NT, 0);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if (s < 7) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        kf[(s + 1) & 1][nt] = *reinterpret_cast<const bf16x8*>(Ks + kaddr[s + 1] + nt * 8192);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sacc[nt] = mfma32(kf[s & 1][nt], qreg[s], sacc[nt]);
    if (s < 7) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    } else {
      __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
    }
  }
}

// Online softmax in the exp2 domain on the scores of one tile; leaves the bf16
// probabilities in pfrag (already in the B-operand layout of O^T += V^T P^T).
// The reference maximum m_run is only moved when a row's maximum outgrows it
// by more than 2^8 (or on the row's first visible key): exp2 arguments then
// stay <= 8, which fp32 sums and bf16 probabilities hold without loss, and
// the rescaling of l and of the 64 output accumulators is skipped for the
// wavefront whenever no row needs it.  O / l does not depend on the choice.
template <int NT>
__device__ __forceinline__ void softmax_tile(f32x16 (&sacc)[NT], f32x16 (&oacc)[4], float& m_run, float& l_run,
                                             float scale_log2, bf16x8 (&pfrag)[NT * 2]) {
  float mx = -INFINITY;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sacc[nt][v]);
  mx = half_max(mx) * scale_log2;
  const bool move = mx > m_run + 8.f || (m_run == -INFINITY && mx > -INFINITY);
  if (__any(move)) {
    const float m_new = move ? mx : m_run;
    const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v) oacc[dt][v] *= alpha;
  }
  const float m_safe = (m_run == -INFINITY) ? 0.f : m_run;
  float psum = 0.f;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float e = fast_exp2(__builtin_fmaf(sacc[nt][v], scale_log2, -m_safe));
      psum += e;
      pfrag[nt * 2 + (v >> 3)][v & 7] = (__bf16)e;
    }
  l_run += psum;
}

// O^T += V_j^T P^T on KS x 16 keys
template <int KS>
__device__ __forceinline__ void pv_tile(const char* Vs, const int (&vaddr)[4][2], const bf16x8 (&pfrag)[KS], f32x16 (&oacc)[4]) {
  i16x4 vf[2][4][2];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int a = 0; a < 2; ++a)
      vf[0][dt][a] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) i16x4*)(Vs + vaddr[dt][a]));
  __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (ks < KS - 1) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int a = 0; a < 2; ++a)
          vf[(ks + 1) & 1][dt][a] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(Vs + vaddr[dt][a] + (ks + 1) * 4096));
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      typedef __attribute__((__vector_size__(8 * sizeof(short)))) short i16x8;
      i16x8 av;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        av[u] = vf[ks & 1][dt][0][u];
        av[4 + u] = vf[ks & 1][dt][1][u];
      }
      oacc[dt] = mfma32(__builtin_bit_cast(bf16x8, av), pfrag[ks], oacc[dt]);
    }
    if (ks < KS - 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
    } else {
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    }
  }
}

// What is loaded and stored not temporal (the rule: not_temporal in block_sparse_attn.hip)
enum { kNtNone, kNtOutput, kNtQueriesToo };

// A unit's sweep.  kHalves: the workgroup has 64 rows of the q-block; wavefront (rg, kh) takes row group rg of them and the keys of
// half kh of every tile, and the two halves' results meet in LDS at the end.  A tile is then half as long a chain of matrix and
// vector work, which is what bounds a workgroup alone on its CU: a prompt of 500 tokens, lists of up to 4 blocks, 23.3 -> 21.5 us in
// all, 2000 with 4 heads 25.2 -> 23.1 (figures of the rule: in_halves).
template <bool kHasList, bool kPlanned, bool kHalves, int kNt>
__device__ __forceinline__ void sweep_unit(const AttnParams& p, const Unit& u, int half, char* Ks, char* Vs) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, hh = lane >> 5;
  const int kh = kHalves ? wave & 1 : 0;
  const int rows = kHalves ? half * 2 + (wave >> 1) : wave;        // this wavefront's 32 rows of the q-block
  constexpr int NT = kHalves ? 2 : 4;                              // ... and 32-key steps of a tile, from kh * NT on
  const int n_blocks = u.n_blocks;
  const __bf16* qbase = p.q + (int64_t)u.head * p.q_sh;
  const __bf16* kbase = p.k + (int64_t)u.kvh * p.k_sh;
  const __bf16* vbase = p.v + (int64_t)u.kvh * p.v_sh;
  const int q_pos = u.qb * kBlk + rows * 32 + r + p.kv_off;   // position of this lane's query token on the key axis

  bf16x8 qreg[8];   // Q^T fragments stay in registers for the whole sweep
  FragAddr la;
  frag_addressing(lane, la);
  int voffK[8], voffV[8];   // tile copies: byte offsets of the lane's rows
  tile_offsets(p.k_sn, lane, wave, voffK);
  tile_offsets(p.v_sn, lane, wave, voffV);

  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[i][v] = 0.f;
  float m_run = -INFINITY;   // running row maximum, already multiplied by scale_log2
  float l_run = 0.f;         // this lane's share of the running row sum

  int kb = u.kb, kb_next = u.kb_next;
  {
    // The q-block is a tile like any other: copied row-wise (full lines) into the V tile, where each wavefront's
    // eighth-of-a-tile copies are its own 32 query rows, and read back as fragments before V_0 is requested.
    int voffQ[8];
    tile_offsets(p.q_sn, lane, rows, voffQ);
    copy_tile<kNt == kNtQueriesToo ? kNotTemporal : 0>(qbase, p.q_sn, p.Lq, u.qb, voffQ, Vs, wave);
    if (n_blocks > 0) copy_tile(kbase, p.k_sn, p.Lk, kb, voffK, Ks, wave);
    wait_vm0();
#pragma unroll
    for (int s = 0; s < 8; ++s) qreg[s] = *reinterpret_cast<const bf16x8*>(Vs + wave * 8192 + la.kaddr[s]);
    __builtin_amdgcn_s_waitcnt(0xC07F);      // the fragments are in registers before V_0 may overwrite them
    asm volatile("" ::: "memory");
    if (n_blocks > 0) copy_tile_async(vbase, p.v_sn, p.Lk, kb, voffV, Vs, wave);
  }
  // K_0 landed before the fragments were read (every wavefront waited for its share); V_0 stays in flight during
  // the first Q.K^T and is waited for with the tile's own barrier
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  for (int j = 0; j < n_blocks; ++j) {
    const bool more = j + 1 < n_blocks;
    f32x16 sacc[NT];
    qk_tile<NT>(Ks + kh * NT * 8192, la.kaddr, qreg, sacc);
    wait_vm0();
    __syncthreads();                       // everyone is done with K_j; V_j landed and visible
    if (more) copy_tile_async(kbase, p.k_sn, p.Lk, kb_next, voffK, Ks, wave);

    const bool need_mask = (kb * kBlk + kBlk > p.Lk) || (p.causal && kb * kBlk + kBlk - 1 > u.qb * kBlk + p.kv_off);
    if (need_mask) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mask_step(sacc[nt], kb * kBlk + (kh * NT + nt) * 32, hh, q_pos, p.Lk, p.causal);
    }
    bf16x8 pfrag[NT * 2];
    softmax_tile<NT>(sacc, oacc, m_run, l_run, p.scale_log2, pfrag);
    pv_tile<NT * 2>(Vs + kh * NT * 8192, la.vaddr, pfrag, oacc);
    // the list's next entry is on its way while this wavefront waits (in flight beside LDS reads it would make each of them wait for all)
    int kb_then = kHasList ? u.list[j + 2 < n_blocks ? j + 2 : j] : kb + 2;
    __builtin_amdgcn_sched_barrier(0);
    wait_vm0();
    __syncthreads();                       // everyone is done with V_j; K_{j+1} landed and visible
    if (kHasList) asm volatile("" : "+s"(kb_then));
    if (more) copy_tile_async(vbase, p.v_sn, p.Lk, kb_next, voffV, Vs, wave);
    kb = kb_next;
    kb_next = kHasList ? clamp_block(kb_then, p.nkb) : kb_then;
  }
  // the last barrier of the sweep (or the one before it, for an empty list) left both tiles unused
  if (kPlanned && u.cuts > 0) {
    float* const part = p.plan.part + (int64_t)u.part0 * kPartFloats;
    store_partial(part + (int64_t)u.piece * kPartFloats, wave, lane, r, hh, oacc, m_run, l_run);
    wait_vm0();                              // written through to memory
    __syncthreads();
    int* const scratch = reinterpret_cast<int*>(Ks);
    if (tid == 0) scratch[0] = __hip_atomic_fetch_add(p.plan.done + unit_slot(p, u), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (scratch[0] != u.cuts - 1) return;      // the piece that comes last combines them
    __syncthreads();
    load_partials(part, u.cuts, wave, lane, r, hh, oacc, l_run);
  }
  if (kHalves) {
    char* const o1 = Ks + (wave >> 1) * 16384 + lane * 16;
    float* const ml = reinterpret_cast<float*>(Vs) + (wave >> 1) * 128 + lane;
    if (kh == 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        f32x4 w;
#pragma unroll
        for (int t = 0; t < 4; ++t) w[t] = oacc[i >> 2][(i & 3) * 4 + t];
        *reinterpret_cast<f32x4*>(o1 + i * 1024) = w;
      }
      ml[0] = m_run;
      ml[64] = l_run;
    }
    __syncthreads();
    if (kh == 1) return;
    const float m1 = ml[0], m = fmaxf(m_run, m1), safe = m == -INFINITY ? 0.f : m;
    const float w0 = fast_exp2(m_run - safe), w1 = fast_exp2(m1 - safe);      // 0 where a half saw no key of this row
    l_run = w0 * l_run + w1 * ml[64];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const f32x4 o = *reinterpret_cast<const f32x4*>(o1 + i * 1024);
#pragma unroll
      for (int t = 0; t < 4; ++t) oacc[i >> 2][(i & 3) * 4 + t] = w0 * oacc[i >> 2][(i & 3) * 4 + t] + w1 * o[t];
    }
    store_out(p, u.head, u.qb, rows, lane, r, hh, oacc, l_run, Ks + (wave >> 1) * 16384);
    return;
  }
  store_out<kNt != kNtNone>(p, u.head, u.qb, wave, lane, r, hh, oacc, l_run, Ks + wave * 8192);
}

// kHasList = false visits every visible block, the dense baseline (its own symbol, so profiles tell the two apart);
// kPlanned: long lists are cut (attn_plan.h); kHalves: a unit is two workgroups', of 64 rows each; kNt: what is
// not temporal (a parameter since the choice made in the kernel costs a call of 700 tokens 0.15 of 26.8 us)
template <bool kHasList, bool kPlanned, bool kHalves, int kNt>
__global__ __launch_bounds__(256, 2) void block_sparse_fwd_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(1024))) char Ks[kTileBytes];
  __shared__ __attribute__((aligned(1024))) char Vs[kTileBytes];

  touch_params();
  // (both halves on the same XCD, one after the other)
  const int id = kHalves ? (int)(blockIdx.x >> 4 << 3 | (blockIdx.x & 7)) : (int)blockIdx.x;
  const int half = kHalves ? (int)(blockIdx.x >> 3 & 1) : 0;
  Unit u;
  if (!find_work<kHasList, kPlanned>(p, id, u)) return;
  if (kHalves && u.qb * kBlk + half * 64 >= p.Lq) return;
  sweep_unit<kHasList, kPlanned, kHalves, kNt>(p, u, half, Ks, Vs);
}

}  // namespace xattn
