// Single-token decode attention over a KV cache for gfx950.
//
// Replaces the reference's call to the third-party
// flashinfer.single_decode_with_kv_cache(q[H,d], k[Hkv,L,d], v[Hkv,L,d],
// kv_layout="HND") in its Llama attention forward
// (xattn/src/load_llama.py:191-196): out[h] = softmax(q[h] K[h/g]^T / sqrt(d)) V[h/g].
//
// The step reads every key and value once and does four flops per byte, so it
// is bound by HBM bandwidth; the design keeps as many bytes in flight per CU as
// LDS can hold.  One workgroup of four wavefronts per CU owns all 160 KiB of
// LDS; every wavefront streams its own contiguous range of 32-key tiles through
// a private ring of five 8 KiB slots (K_i, V_i, K_i+1, V_i+1, K_i+2) filled by
// buffer loads that write LDS directly, so four tiles per wavefront are always
// in flight and no workgroup barrier is needed.  A KV head's query heads (the
// GQA group, at most 32) are the columns of one MFMA tile: S^T = K Q^T gives
// each lane one query head, the softmax is the same lane-owns-a-row form as in
// the prefill kernel and its accumulators feed O^T += V^T P^T unchanged.  The
// four wavefronts combine (max, sum, unnormalised output) of their key ranges in
// LDS and write one partial result per workgroup; a second small kernel merges
// the workgroups of a head.  Short caches take one launch (decode_short_kernel).
//
// Keys and values of large caches are loaded "not temporal" (kNtBytes).
#include <mutex>

#include "lds_limit.h"
#include "xattn_common.h"
#include "xattn_hip.h"

namespace xattn {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4;
typedef __attribute__((__vector_size__(8 * sizeof(short)))) short i16x8;

constexpr int kDecKeys = 32;                  // keys per tile
constexpr int kDecTileBytes = kDecKeys * 256;
constexpr int kDecSlots = 5;
constexpr int kDecWaves = 4;
constexpr int kDecLds = kDecWaves * kDecSlots * kDecTileBytes;   // 160 KiB
constexpr int kPartStride = 132;              // floats per (range, query head): 128 outputs, max, sum, 2 pad
constexpr int kDecCUs = 256;

struct DecodeParams {
  const __bf16* q;
  const __bf16* k;
  const __bf16* v;
  __bf16* o;
  float* part;
  int64_t q_sh, k_sh, k_sn, v_sh, v_sn, o_sh;   // element strides
  int H, Hkv, group, Lk;
  int n_tiles, wgs;            // tiles of the cache, workgroups of a KV head
  int per_wave, longer;        // tiles of a wavefront, and how many wavefronts of a head have one more
  float scale_log2;
};

__device__ __forceinline__ int dec_swz(int n) { return ((n & 3) << 2) | ((n >> 2) & 3); }

// waits until at most kLeft of this wavefront's buffer loads are outstanding (loads complete in order); other counters untouched
template <int kLeft>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (kLeft & 15) | (kLeft >> 4) << 14);
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_lgkm0() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
}

// One 32-key tile, global -> this wavefront's LDS slot.
template <bool kNt>
__device__ __forceinline__ void dec_copy(const __bf16* base, int64_t sn, int len, int tile, const int (&voff)[8], char* slot) {
  const int rows_left = len - tile * kDecKeys;
  const int rows = rows_left < kDecKeys ? rows_left : kDecKeys;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(base + (int64_t)tile * kDecKeys * sn), 0, (int)((int64_t)rows * sn * 2), 0x00020000);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(slot + i * 1024), 16, voff[i], 0, 0, kNt ? kNotTemporal : 0);
}

template <bool kNt>
__global__ __launch_bounds__(256, 1) void decode_partial_kernel(DecodeParams p) {
  extern __shared__ __attribute__((aligned(1024))) char ring_all[];

  const int tid = threadIdx.x, lane = tid & 63;
  // the wavefront number in a scalar register: tile ranges, buffer resources and
  // LDS slots derived from it are then uniform values for the compiler too
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;
  const int kvh = blockIdx.x / p.wgs, wg = blockIdx.x - kvh * p.wgs;
  // the wavefronts' ranges differ by a tile at most, and a workgroup's lie apart (131072 keys of 4 KV heads 54.7 us with its four one
  // after the other, 50.9 so; the longer ones are spread over the workgroups)
  const int range = wave * p.wgs + wg;
  const int t0 = range * p.per_wave + (range < p.longer ? range : p.longer);
  const int n = p.per_wave + (range < p.longer ? 1 : 0);

  char* ring = ring_all + wave * (kDecSlots * kDecTileBytes);
  // the same place as an LDS byte address
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring_all +
                            (uint32_t)(wave * (kDecSlots * kDecTileBytes));
  const __bf16* kbase = p.k + (int64_t)kvh * p.k_sh;
  const __bf16* vbase = p.v + (int64_t)kvh * p.v_sh;

  int voffK[8], voffV[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 4 * i + (lane >> 4);
    const int c = (lane & 15) ^ dec_swz(row);
    voffK[i] = (int)(row * p.k_sn * 2) + (c << 4);
    voffV[i] = (int)(row * p.v_sn * 2) + (c << 4);
  }
  int kaddr[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) kaddr[s] = r * 256 + (((2 * s + hh) ^ dec_swz(r)) << 4);
  int vaddr[4][2];
  {
    const int e = (lane & 15) >> 2, j = lane & 3, g2 = (lane >> 4) & 1;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int row = 8 * a + 4 * hh + e;                       // + 16*ks
        const int c = dt * 4 + 2 * g2 + (j >> 1);
        vaddr[dt][a] = row * 256 + ((c ^ dec_swz(row)) << 4) + (j & 1) * 8;
      }
  }

  f32x16 oacc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[i][v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // The query heads' rows, then load number j of the sequence K_0 V_0 K_1 V_1 ... to slot j % 5.  A CU takes a load of 1 KiB every 20
  // clk, whether it moves anything or not, so none is issued past the range's end (with loads of empty resources there, and the queries
  // read row by row, 32 loads a wavefront ahead of the first tile, a step on 1100 keys took 7.6 us instead of 7.0).
  bf16x8 qreg[8];
  if (n > 0) {
    char* const rows = ring + 4 * kDecTileBytes;
#pragma unroll 1
    for (int i = 0; i < p.group; i += 4) {
      const int row = i + (lane >> 4), src = row < p.group ? row : p.group - 1;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p.q + (int64_t)(kvh * p.group + src) * p.q_sh + ((lane & 15) ^ dec_swz(row)) * 8),
                                       (lds_ptr_t)(rows + i * 256), 16, 0, 0);
    }
    dec_copy<kNt>(kbase, p.k_sn, p.Lk, t0, voffK, ring + 0 * kDecTileBytes);
    dec_copy<kNt>(vbase, p.v_sn, p.Lk, t0, voffV, ring + 1 * kDecTileBytes);
    if (n > 1) {
      dec_copy<kNt>(kbase, p.k_sn, p.Lk, t0 + 1, voffK, ring + 2 * kDecTileBytes);
      dec_copy<kNt>(vbase, p.v_sn, p.Lk, t0 + 1, voffV, ring + 3 * kDecTileBytes);
      wait_vm<32>();
    } else {
      wait_vm<16>();
    }
    // Q^T fragments: lane r holds query head kvh*group + r (zeros beyond the group)
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(rows + kaddr[s]);
#pragma unroll
      for (int e = 0; e < 8; ++e) qreg[s][e] = r < p.group ? x[e] : (__bf16)0.f;
    }
  }

  int slot = 0;   // slot of K_i
  for (int i = 0; i < n; ++i) {
    const int tile = t0 + i, behind = n - 1 - i;
    char* Kt = ring + slot * kDecTileBytes;
    const int sv = slot + 1 >= kDecSlots ? slot + 1 - kDecSlots : slot + 1;
    const int s4 = slot + 4 >= kDecSlots ? slot + 4 - kDecSlots : slot + 4;   // freed by V_{i-1}, at first by the queries

    wait_lgkm0();   // this wavefront's reads of the slot about to be refilled have returned
    if (behind > 1) {
      dec_copy<kNt>(kbase, p.k_sn, p.Lk, tile + 2, voffK, ring + s4 * kDecTileBytes);
      wait_vm<32>();    // K_i landed
    } else if (behind == 1) {
      wait_vm<24>();
    } else {
      wait_vm<8>();
    }

    f32x16 sacc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sacc[v] = 0.f;
    {
      bf16x8 kf[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(Kt + kaddr[s]);
#pragma unroll
      for (int s = 0; s < 8; ++s) sacc = mfma32(kf[s], qreg[s], sacc);
    }
    if (tile * kDecKeys + kDecKeys > p.Lk) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int kpos = tile * kDecKeys + (v >> 2) * 8 + hh * 4 + (v & 3);
        sacc[v] = kpos >= p.Lk ? -INFINITY : sacc[v];
      }
    }
    // K_i is in registers (the MFMAs above consumed every fragment): its slot takes V_{i+2}
    wait_lgkm0();
    if (behind > 1) dec_copy<kNt>(vbase, p.v_sn, p.Lk, tile + 2, voffV, Kt);

    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sacc[v]);
    mx = half_max(mx) * p.scale_log2;
    const float m_new = fmaxf(m_run, mx);          // finite: every tile holds at least one real key
    const float alpha = fast_exp2(m_run - m_new);  // 0 on the first tile
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v) oacc[dt][v] *= alpha;
    float psum = 0.f;
    bf16x8 pfrag[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float e = fast_exp2(__builtin_fmaf(sacc[v], p.scale_log2, -m_run));
      psum += e;
      pfrag[v >> 3][v & 7] = (__bf16)e;
    }
    l_run += psum;

    // V_i landed
    if (behind > 1) wait_vm<32>();
    else if (behind == 1) wait_vm<16>();
    else wait_vm<0>();
    {
      // The sixteen transposing reads of V_i are issued from one asm statement:
      // an LDS read the compiler can see would make it wait for EVERY buffer
      // load in flight (it cannot tell the ring's slots apart), which would
      // empty the ring on each iteration.
      i16x4 t[4][2][2];   // [feature tile][half a][k-step]
      const uint32_t vt = ring_lds + (uint32_t)(sv * kDecTileBytes);
      uint32_t a[4][2];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) a[dt][h2] = vt + (uint32_t)vaddr[dt][h2];
      asm volatile(
          "ds_read_b64_tr_b16 %0, %16\n\t"
          "ds_read_b64_tr_b16 %1, %16 offset:4096\n\t"
          "ds_read_b64_tr_b16 %2, %17\n\t"
          "ds_read_b64_tr_b16 %3, %17 offset:4096\n\t"
          "ds_read_b64_tr_b16 %4, %18\n\t"
          "ds_read_b64_tr_b16 %5, %18 offset:4096\n\t"
          "ds_read_b64_tr_b16 %6, %19\n\t"
          "ds_read_b64_tr_b16 %7, %19 offset:4096\n\t"
          "ds_read_b64_tr_b16 %8, %20\n\t"
          "ds_read_b64_tr_b16 %9, %20 offset:4096\n\t"
          "ds_read_b64_tr_b16 %10, %21\n\t"
          "ds_read_b64_tr_b16 %11, %21 offset:4096\n\t"
          "ds_read_b64_tr_b16 %12, %22\n\t"
          "ds_read_b64_tr_b16 %13, %22 offset:4096\n\t"
          "ds_read_b64_tr_b16 %14, %23\n\t"
          "ds_read_b64_tr_b16 %15, %23 offset:4096\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(t[0][0][0]), "=&v"(t[0][0][1]), "=&v"(t[0][1][0]), "=&v"(t[0][1][1]),
            "=&v"(t[1][0][0]), "=&v"(t[1][0][1]), "=&v"(t[1][1][0]), "=&v"(t[1][1][1]),
            "=&v"(t[2][0][0]), "=&v"(t[2][0][1]), "=&v"(t[2][1][0]), "=&v"(t[2][1][1]),
            "=&v"(t[3][0][0]), "=&v"(t[3][0][1]), "=&v"(t[3][1][0]), "=&v"(t[3][1][1])
          : "v"(a[0][0]), "v"(a[0][1]), "v"(a[1][0]), "v"(a[1][1]),
            "v"(a[2][0]), "v"(a[2][1]), "v"(a[3][0]), "v"(a[3][1])
          : "memory");
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          i16x8 av;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            av[u] = t[dt][0][ks][u];
            av[4 + u] = t[dt][1][ks][u];
          }
          oacc[dt] = mfma32(__builtin_bit_cast(bf16x8, av), pfrag[ks], oacc[dt]);
        }
    }
    slot = slot + 2 >= kDecSlots ? slot + 2 - kDecSlots : slot + 2;
  }
  // The four wavefronts' results meet in LDS (each uses the start of its own,
  // now idle, ring) and leave as one partial result per workgroup.
  const float l_tot = half_sum(l_run);
  float* mine = reinterpret_cast<float*>(ring);
  if (r < p.group) {
    float* dst = mine + r * kPartStride;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 w;
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = oacc[dt][g * 4 + u];
        *reinterpret_cast<f32x4*>(dst + dt * 32 + g * 8 + hh * 4) = w;
      }
    if (hh == 0) {
      dst[128] = m_run;    // -inf for an empty range
      dst[129] = l_tot;    // 0 for an empty range
    }
  }
  __syncthreads();
  {
    constexpr int kWaveFloats = kDecSlots * kDecTileBytes / 4;
    const float* all = reinterpret_cast<const float*>(ring_all);
    float* out = p.part + (int64_t)blockIdx.x * p.group * kPartStride;
    for (int e = tid; e < p.group * 128; e += 256) {
      const int g = e >> 7, d = e & 127;
      float mw[kDecWaves], m = -INFINITY;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) {
        mw[w] = all[w * kWaveFloats + g * kPartStride + 128];
        m = fmaxf(m, mw[w]);
      }
      float acc = 0.f, l = 0.f;
#pragma unroll
      for (int w = 0; w < kDecWaves; ++w) {
        const float wt = mw[w] == -INFINITY ? 0.f : fast_exp2(mw[w] - m);
        acc += wt * all[w * kWaveFloats + g * kPartStride + d];
        l += wt * all[w * kWaveFloats + g * kPartStride + 129];
      }
      out[g * kPartStride + d] = acc;
      if (d == 0) {
        out[g * kPartStride + 128] = m;
        out[g * kPartStride + 129] = l;
      }
    }
  }
}

// out[h][d] = sum_s w_s O_s[d] / sum_s w_s l_s,  w_s = 2^(m_s - max m), over the
// head's workgroups s (at most 256).  Bound by the latency of one dependent
// chain, so everything a thread needs from memory is requested at once: lane i
// holds (m_s, l_s) of partial results i, i + 64, .. for the weights, which every
// wavefront finds for itself (no barrier), and features 4*(t%32).. of every
// eighth partial result, eight of them in flight, which do not wait for the
// weights.  (With a running maximum the loads of one trip waited for the branch
// of the one before: 7.1 -> 4.8 us for the merge of 64.)
__global__ __launch_bounds__(256) void decode_merge_kernel(DecodeParams p) {
  __shared__ __attribute__((aligned(16))) float accs[8][128];
  __shared__ float wt[4][256];
  const int head = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kvh = head / p.group, g = head % p.group;
  const int wgs = p.wgs;
  const float* base = p.part + ((int64_t)kvh * wgs * p.group + g) * kPartStride;
  const int64_t step = (int64_t)p.group * kPartStride;
  const int slot = tid >> 5, dg = tid & 31;

  float m[4], l[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int s = lane + 64 * u;
    m[u] = s < wgs ? base[s * step + 128] : -INFINITY;
    l[u] = s < wgs ? base[s * step + 129] : 0.f;
  }
  constexpr int kAhead = 8;
  f32x4 o[kAhead];
  auto load = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int s = s0 + 8 * u;
      o[u] = s < wgs ? *reinterpret_cast<const f32x4*>(base + s * step + dg * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  load(slot);
  const float mx = wave_maxf(fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3])));
  float den = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float w = m[u] == -INFINITY ? 0.f : fast_exp2(m[u] - mx);   // 0 for an empty range
    wt[wave][lane + 64 * u] = w;
    den += w * l[u];
  }
  den = wave_sumf(den);
  __builtin_amdgcn_wave_barrier();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = slot; s0 < wgs; s0 += 8 * kAhead) {
    if (s0 != slot) load(s0);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const float ws = s0 + 8 * u < wgs ? wt[wave][s0 + 8 * u] : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += ws * o[u][e];
    }
  }
  *reinterpret_cast<f32x4*>(&accs[slot][dg * 4]) = acc;
  __syncthreads();
  if (tid < 128) {
    float num = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) num += accs[s][tid];
    p.o[(int64_t)head * p.o_sh + tid] = (__bf16)(den > 0.f ? num / den : 0.f);
  }
}

// A step over a short cache, in one launch.  Partial results of several workgroups would need a second one, 3 us on the GPU and as much
// on the host, so a KV head is four workgroups', each of which goes over all keys for a quarter of the features.  They are on one XCD,
// and each begins at another quarter of the keys, so the keys are fetched into its L2 once, by all four together.  Its wavefronts take
// every twelfth tile each: 8 KiB of keys and 2 KiB of values, requested anew as soon as the last ones are in registers.  Bound by what
// a CU takes in, 10 KiB per tile at 110 GB/s from the L2 and 70 from memory, behind 3.4 us of latencies (launch, first tile, softmax, the
// wavefronts' results, store).
constexpr int kShortWaves = 12, kShortParts = 4;
constexpr int kShortSlot = kDecTileBytes + kDecTileBytes / kShortParts;
constexpr int kShortLds = kShortWaves * kShortSlot + kDecTileBytes;      // the queries last
constexpr int kShortStride = 36;              // floats per (wavefront, query head): 32 outputs, max, sum, 2 pad

__global__ __launch_bounds__(64 * kShortWaves) void decode_short_kernel(DecodeParams p) {
  extern __shared__ __attribute__((aligned(1024))) char ring_all[];
  const int stride = (p.Hkv + 7) & ~7;
  const int part = blockIdx.x / stride, kvh = blockIdx.x - part * stride;
  if (kvh >= p.Hkv) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, hh = lane >> 5;
  char* const mine = ring_all + wave * kShortSlot;
  char* const queries = ring_all + kShortWaves * kShortSlot;
  const uint32_t slot = (uint32_t)(uintptr_t)(lds_char_ptr)ring_all + (uint32_t)(wave * kShortSlot);
  const int turn = part * p.n_tiles / kShortParts;
  auto tile_of = [&](int i) {
    const int t = wave + i * kShortWaves + turn;
    return t < p.n_tiles ? t : t - p.n_tiles;
  };
  const int n = wave < p.n_tiles ? (p.n_tiles - 1 - wave) / kShortWaves + 1 : 0;

  if (wave * 4 < p.group) {
    const int row = wave * 4 + (lane >> 4), src = row < p.group ? row : p.group - 1;
    const __bf16* const from = p.q + (int64_t)(kvh * p.group + src) * p.q_sh + ((lane & 15) ^ dec_swz(row)) * 8;
    // (from assembly, as the tiles: the compiler would wait for a copy that it knows of, and for all behind it, at the first
    // transposing read of every tile)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"((uint32_t)(uintptr_t)(lds_char_ptr)(queries + wave * 1024)), "v"(from) : "memory", "m0");
  }
  uint32_t voffK[8], voffV[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 4 * i + (lane >> 4);
    voffK[i] = (uint32_t)(row * p.k_sn * 2) + (uint32_t)(((lane & 15) ^ dec_swz(row)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) voffV[i] = (uint32_t)((16 * i + (lane >> 2)) * p.v_sn * 2) + (uint32_t)(part * 64 + (lane & 3) * 16);
  auto resource = [&](const __bf16* base, int64_t sn, int tile) {
    const int rows_left = p.Lk - tile * kDecKeys, rows = rows_left < kDecKeys ? rows_left : kDecKeys;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)tile * kDecKeys * sn), 0, (int)((int64_t)rows * sn * 2), 0x00020000);
  };
  auto copy_k = [&](int tile) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t res = resource(p.k + (int64_t)kvh * p.k_sh, p.k_sn, tile);
#pragma unroll
    for (int i = 0; i < 8; ++i) slab_copy_1k(res, voffK[i], slot + i * 1024);
  };
  auto copy_v = [&](int tile) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t res = resource(p.v + (int64_t)kvh * p.v_sh, p.v_sn, tile);
#pragma unroll
    for (int i = 0; i < 2; ++i) slab_copy_1k(res, voffV[i], slot + kDecTileBytes + i * 1024);
  };
  if (n > 0) {
    copy_k(tile_of(0));
    copy_v(tile_of(0));
    asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  int kaddr[8], vaddr[2];
#pragma unroll
  for (int s = 0; s < 8; ++s) kaddr[s] = r * 256 + (((2 * s + hh) ^ dec_swz(r)) << 4);
#pragma unroll
  for (int a = 0; a < 2; ++a)
    vaddr[a] = kDecTileBytes + (8 * a + 4 * hh + ((lane & 15) >> 2)) * 64 + (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) * 16 + (lane & 1) * 8;
  f32x16 oacc;
#pragma unroll
  for (int v = 0; v < 16; ++v) oacc[v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  asm volatile("s_barrier" ::: "memory");      // the queries, of whoever copied them
  bf16x8 qreg[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const bf16x8 x = *reinterpret_cast<const bf16x8*>(queries + kaddr[s]);
#pragma unroll
    for (int e = 0; e < 8; ++e) qreg[s][e] = r < p.group ? x[e] : (__bf16)0.f;
  }

  for (int i = 0; i < n; ++i) {
    const int tile = tile_of(i);
    const bool more = i + 1 < n;
    asm volatile("s_waitcnt vmcnt(2)" ::: "memory");      // K_i; V_i may be on its way
    bf16x8 kf[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(mine + kaddr[s]);
    wait_lgkm0();
    if (more) copy_k(tile_of(i + 1));
    f32x16 sacc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sacc[v] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) sacc = mfma32(kf[s], qreg[s], sacc);
    if (tile * kDecKeys + kDecKeys > p.Lk) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int kpos = tile * kDecKeys + (v >> 2) * 8 + hh * 4 + (v & 3);
        sacc[v] = kpos >= p.Lk ? -INFINITY : sacc[v];
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sacc[v]);
    mx = half_max(mx) * p.scale_log2;
    // A tile's probabilities are relative to its own maximum, so that its largest is 1 and not rounded, and its output is
    // weighted in 32 bits: relative to the wavefront's maximum so far, the rounding of later tiles' to bf16 made the result's error
    // against 64 bits up to 4 % larger than that of a wavefront per tile (700 to 1500 keys).
    const float m_new = fmaxf(m_run, mx), top = m_new == -INFINITY ? 0.f : m_new, base = mx == -INFINITY ? 0.f : mx;
    const float alpha = fast_exp2(m_run - top), beta = fast_exp2(mx - top);      // alpha is 0 on the first tile
    m_run = m_new;
    float psum = 0.f;
    bf16x8 pfrag[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float e = fast_exp2(__builtin_fmaf(sacc[v], p.scale_log2, -base));
      psum += e;
      pfrag[v >> 3][v & 7] = (__bf16)e;
    }
    l_run = l_run * alpha + psum * beta;
    if (more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");      // V_i
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    i16x4 t[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int a = 0; a < 2; ++a)
        t[ks][a] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(mine + vaddr[a] + ks * 1024));
    wait_lgkm0();
    if (more) copy_v(tile_of(i + 1));
    f32x16 own;
#pragma unroll
    for (int v = 0; v < 16; ++v) own[v] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      i16x8 av;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        av[u] = t[ks][0][u];
        av[4 + u] = t[ks][1][u];
      }
      own = mfma32(__builtin_bit_cast(bf16x8, av), pfrag[ks], own);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[v] = __builtin_fmaf(own[v], beta, oacc[v] * alpha);
  }

  // the wavefronts' results meet in LDS, each in its own slot
  const float l_tot = half_sum(l_run);
  if (r < p.group) {
    float* const dst = reinterpret_cast<float*>(mine) + r * kShortStride;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 w;
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = oacc[g * 4 + u];
      *reinterpret_cast<f32x4*>(dst + g * 8 + hh * 4) = w;
    }
    if (hh == 0) {
      dst[32] = m_run;
      dst[33] = l_tot;
    }
  }
  __syncthreads();
  for (int e = tid; e < p.group * 32; e += 64 * kShortWaves) {
    const int g = e >> 5, d = e & 31;
    const float* const src = reinterpret_cast<const float*>(ring_all) + g * kShortStride;
    float m[kShortWaves], top = -INFINITY, acc = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < kShortWaves; ++w) {
      m[w] = src[w * (kShortSlot / 4) + 32];
      top = fmaxf(top, m[w]);
    }
#pragma unroll
    for (int w = 0; w < kShortWaves; ++w) {
      const float wt = m[w] == -INFINITY ? 0.f : fast_exp2(m[w] - top);      // 0 for a wavefront without tiles
      acc += wt * src[w * (kShortSlot / 4) + d];
      l += wt * src[w * (kShortSlot / 4) + 33];
    }
    p.o[(int64_t)(kvh * p.group + g) * p.o_sh + part * 32 + d] = (__bf16)(l > 0.f ? acc / l : 0.f);
  }
}

// Bytes of keys and values from which they are loaded "not temporal": such a cache does not stay in the memory-side cache (256 MB)
// beside what else a step reads, and a stream from memory is faster by a sixth (100003 keys of 8 KV heads 75.9 -> 68.0 us, 6.1 TB/s;
// 40000 34.5 -> 31.7; 70000 of 4 32.7 -> 29.8).  A smaller one may be there still from the call before (two or three in turn,
// without / with: 82 MB 19.0 / 19.4 us, 38 MB 12.8 / 13.1).
constexpr int64_t kNtBytes = 96 << 20;

// Tiles of the longest cache that decode_short_kernel takes: 1280 keys where every workgroup has a CU of its own, 128 where some wait for
// another's (more than 64 KV heads).  A step's cache comes from memory, the weights of all layers having passed since its last one, and
// so were these measured, over caches of 640 MB in turn.  us, two launches / one:
//                                            100          500          800          1100         1300         1500 keys
//   in a captured graph, 1 KV head           9.1 / 4.2    9.4 / 6.5    9.7 / 8.4    9.8 / 9.8    9.8 / 10.7   9.8 / 11.6
//                        2                   7.6 / 4.2    8.2 / 6.6    8.3 / 8.2    8.3 / 9.7    8.4 / 10.5   8.4 / 11.4
//                        4                   7.2 / 4.0    7.5 / 6.4    7.6 / 8.1    7.6 / 9.7    7.7 / 10.4   7.7 / 11.4
//                        8                   7.2 / 4.4    7.2 / 6.6    7.3 / 8.3    7.4 / 9.9    7.5 / 10.7   7.6 / 11.7
//                        32                  7.1 / 4.5    7.5 / 7.0    8.5 / 8.8    10.3 / 10.8  11.1 / 11.9  11.4 / 12.9
//                        64                  7.2 / 4.6    8.9 / 8.1    11.8 / 10.6  13.9 / 13.0  14.6 / 14.6  15.7 / 17.0
//                        72                  7.2 / 6.9    10.4 / 11.6  12.9 / 14.7  14.1 / 17.9  16.3 / 21.0  18.6 / 23.8
//                        128                 7.4 / 7.2    12.8 / 13.8  16.8 / 18.9  20.0 / 24.6  22.5 / 28.5  24.8 / 32.6
//   in a loop of calls, 8                    8.2 / 4.7    8.3 / 6.6    8.1 / 8.1    8.2 / 9.7    8.5 / 10.5   8.9 / 11.6
//                       128                  8.7 / 7.4    13.6 / 13.9  17.2 / 19.3  20.8 / 26.0  23.7 / 29.1  25.5 / 33.2
//   a layer's whole step, 8, graph           29.4 / 27.8 (300 keys)    29.6 / 29.5  29.7 / 30.7               30.0 / 32.0
//                         as Python calls it 43.1 / 39.3 (300)         42.4 / 38.7  41.7 / 38.1               42.0 / 38.3
// (32 / 32 heads the same: 37.3 / 36.0, 39.4 / 39.9, 41.6 / 41.6, 42.5 / 43.6 and 43.0 / 39.5, 42.6 / 40.2, 42.4 / 42.1, 43.5 / 43.2.)
// Beyond 800 keys the GPU is done sooner with two launches and a layer that is called from Python later, the host having one more to make;
// the line is where the loss of the one and the gain of the other are equal.  (A cache still in the L2, graph, 8: 500 keys 6.8 / 5.1, 1100
// 7.0 / 7.1, 1500 6.9 / 8.1.)  A word of every later row of values asked for at the start made one launch 0.4 to 0.8 slower.
constexpr int kShortTiles = 40, kShortTilesInTurns = 4;

struct DecodeGeometry {
  int n_tiles, wgs;
};

// One workgroup per CU at most: a KV head gets 256 / H_kv workgroups (at least one), unless that leaves them fewer than two tiles (2200
// keys of 8 KV heads: with four, a wavefront's each, 7.6 us, with two 7.3).
static DecodeGeometry decode_geometry(int num_kv_heads, int k_len) {
  DecodeGeometry g;
  g.n_tiles = (k_len + kDecKeys - 1) / kDecKeys;
  int most = kDecCUs / num_kv_heads;
  if (most < 1) most = 1;
  const int wanted = (g.n_tiles + 1) / 2;
  g.wgs = wanted < most ? wanted : most;
  return g;
}

}  // namespace xattn

using namespace xattn;

extern "C" size_t xattn_decode_workspace_bytes(int num_heads, int num_kv_heads, int k_len) {
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || k_len <= 0) return 0;
  const DecodeGeometry g = decode_geometry(num_kv_heads, k_len);
  return (size_t)g.wgs * num_heads * kPartStride * sizeof(float);
}

namespace {
// Validates, fills the launch parameters and enqueues both kernels; `part` holds
// part_bytes bytes of per-range partial results.
int decode_launch(const void* q, const void* k, const void* v, void* out, void* part, size_t part_bytes,
                  int num_heads, int num_kv_heads, int k_len, int head_dim, int64_t q_stride_h,
                  int64_t k_stride_h, int64_t k_stride_n, int64_t v_stride_h, int64_t v_stride_n,
                  int64_t o_stride_h, float softmax_scale, void* stream) {
  if (!q || !k || !v || !out || !part) return XATTN_ERR_NULL;
  if (head_dim != kHeadDim) return XATTN_ERR_HEAD_DIM;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads) return XATTN_ERR_HEADS;
  if (num_heads / num_kv_heads > 32) return XATTN_ERR_HEADS;
  if (k_len <= 0) return XATTN_ERR_SHAPE;
  const int64_t strides[] = {q_stride_h, k_stride_h, k_stride_n, v_stride_h, v_stride_n};
  for (int64_t s : strides)
    if (s % 8) return XATTN_ERR_ALIGN;
  auto a16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  if (!a16(q) || !a16(k) || !a16(v) || !a16(part)) return XATTN_ERR_ALIGN;
  // a tile's byte offsets are held in 32 bits
  if (k_stride_n > (1 << 22) || v_stride_n > (1 << 22) || k_stride_n < kHeadDim || v_stride_n < kHeadDim)
    return XATTN_ERR_SHAPE;
  if (part_bytes < xattn_decode_workspace_bytes(num_heads, num_kv_heads, k_len)) return XATTN_ERR_WORKSPACE;

  const DecodeGeometry g = decode_geometry(num_kv_heads, k_len);
  DecodeParams p;
  p.q = static_cast<const __bf16*>(q);
  p.k = static_cast<const __bf16*>(k);
  p.v = static_cast<const __bf16*>(v);
  p.o = static_cast<__bf16*>(out);
  p.part = static_cast<float*>(part);
  p.q_sh = q_stride_h; p.k_sh = k_stride_h; p.k_sn = k_stride_n;
  p.v_sh = v_stride_h; p.v_sn = v_stride_n; p.o_sh = o_stride_h;
  p.H = num_heads; p.Hkv = num_kv_heads; p.group = num_heads / num_kv_heads; p.Lk = k_len;
  p.n_tiles = g.n_tiles; p.wgs = g.wgs;
  p.per_wave = g.n_tiles / (g.wgs * kDecWaves); p.longer = g.n_tiles % (g.wgs * kDecWaves);
  p.scale_log2 = softmax_scale * kLog2e;

  hipStream_t s = static_cast<hipStream_t>(stream);
  static LdsLimit limit[3];
  if (g.n_tiles <= (kShortParts * num_kv_heads <= kDecCUs ? kShortTiles : kShortTilesInTurns)) {
    if (limit[2].raise(reinterpret_cast<const void*>(decode_short_kernel)) != hipSuccess) return XATTN_ERR_LAUNCH;
    hipLaunchKernelGGL(decode_short_kernel, dim3((unsigned)(kShortParts * ((num_kv_heads + 7) & ~7))), dim3(64 * kShortWaves), kShortLds, s, p);
    return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
  }
  const bool nt = (int64_t)num_kv_heads * k_len * kHeadDim * 4 > kNtBytes;
  const auto kernel = nt ? decode_partial_kernel<true> : decode_partial_kernel<false>;
  if (limit[nt].raise(reinterpret_cast<const void*>(kernel)) != hipSuccess) return XATTN_ERR_LAUNCH;
  const unsigned grid = (unsigned)(num_kv_heads * g.wgs);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), kDecLds, s, p);
  hipLaunchKernelGGL(decode_merge_kernel, dim3((unsigned)num_heads), dim3(256), 0, s, p);
  return hipGetLastError() == hipSuccess ? XATTN_OK : XATTN_ERR_LAUNCH;
}
}  // namespace

extern "C" int xattn_decode_fwd(const void* q, const void* k, const void* v, void* out, void* workspace,
                                size_t workspace_bytes, int num_heads, int num_kv_heads, int k_len, int head_dim,
                                int64_t q_stride_h, int64_t k_stride_h, int64_t k_stride_n, int64_t v_stride_h,
                                int64_t v_stride_n, int64_t o_stride_h, float softmax_scale, void* stream) {
  return decode_launch(q, k, v, out, workspace, workspace_bytes, num_heads, num_kv_heads, k_len, head_dim, q_stride_h,
                       k_stride_h, k_stride_n, v_stride_h, v_stride_n, o_stride_h, softmax_scale, stream);
}

// ---------------------------------------------------------------------------
// The same decode step for callers that may not allocate: the partial results
// live in a device array that is part of this library's code object.  Every GPU
// the library runs on holds its own copy of the array at its own address; the
// address is looked up once per device and kept.  In host code the array's name
// is only a handle for that lookup, never a pointer a kernel could use.
namespace {
// (256 / H_kv workgroups per KV head) x H query heads is at most 256 * 32
// (range, head) pairs while H_kv <= 256 and H <= 32 H_kv.
constexpr size_t kDecScratchBytes = (size_t)kDecCUs * 32 * kPartStride * sizeof(float);   // 4.125 MiB
static_assert(kDecScratchBytes == XATTN_DECODE_STATIC_SCRATCH_BYTES, "header and kernel disagree on the scratch size");
constexpr int kMaxDevices = 64;
}  // namespace
static __device__ __align__(256) unsigned char scratch[kDecScratchBytes];
namespace {
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (looked up on first use).
int scratch_of_current_device(void** ptr_out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return XATTN_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return XATTN_ERR_LAUNCH;
    g_scratch_ptr[dev] = ptr;
  }
  *ptr_out = g_scratch_ptr[dev];
  return XATTN_OK;
}
}  // namespace

extern "C" int xattn_decode_fwd_static(const void* q, const void* k, const void* v, void* out, int num_heads,
                                       int num_kv_heads, int k_len, int head_dim, int64_t q_stride_h,
                                       int64_t k_stride_h, int64_t k_stride_n, int64_t v_stride_h,
                                       int64_t v_stride_n, int64_t o_stride_h, float softmax_scale, void* stream) {
  const size_t need = xattn_decode_workspace_bytes(num_heads, num_kv_heads, k_len);
  if (need == 0) {
    if (num_heads <= 0 || num_kv_heads <= 0 || (num_kv_heads > 0 && num_heads % num_kv_heads)) return XATTN_ERR_HEADS;
    return XATTN_ERR_SHAPE;
  }
  if (need > kDecScratchBytes) return XATTN_ERR_WORKSPACE;   // more (range, head) pairs than the array holds
  void* ptr = nullptr;
  const int rc = scratch_of_current_device(&ptr);
  if (rc != XATTN_OK) return rc;
  return decode_launch(q, k, v, out, ptr, kDecScratchBytes, num_heads, num_kv_heads, k_len, head_dim, q_stride_h,
                       k_stride_h, k_stride_n, v_stride_h, v_stride_n, o_stride_h, softmax_scale, stream);
}
