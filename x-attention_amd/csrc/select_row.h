// Threshold block selection of one q-block row by one wavefront: shared by the stand-alone selection kernel
// (block sums from memory) and the estimator's fused normalise-and-select kernel (block sums from LDS).
#pragma once
#include <type_traits>

#include "attn_plan.h"
#include "xattn_common.h"

namespace xattn {

constexpr int kMaxTauHost = 64;   // per-head thresholds that fit the kernel arguments

struct SelParams {
  const float* sums;
  const double* tau;               // per head on the device, or null: tau_val[head * tau_step]
  double tau_val[kMaxTauHost];
  int tau_step;
  uint8_t* mask;
  __bf16* sums_out;                // block sums for the caller, or null
  int32_t* col_idx;
  int32_t* col_cnt;
  int64_t idx_pitch;
  int H, nqb, nkb, row_begin, row_end, diag_offset;
  int win_row0, win_rows;   // the arrays hold q-block rows [win_row0, win_row0 + win_rows) of every head
  int causal, keep_sink, keep_recent, list_cols, q_len, kv_off;
  int blocks_per_chunk;
  int npow2;   // LDS key capacity (power of two >= nkb)
  AttnPlan plan;   // per_qb 0: nothing is noted
  uint32_t* totals;   // null, or where blocks of each q-block's lists, and of its longest, are found: 32 * (row - win_row0)
};

constexpr int kMostSlots = 16;    // candidates per lane held in registers (rows up to 1024 candidates)
constexpr int kMaxExtract = 32;   // blocks pulled out one by one before falling back to the sort in LDS
constexpr int kBeforeSearch = 2;  // blocks pulled out of more than 64 before the search for where a long list ends

// value encoded in a sort key (0 for forced blocks and padding)
__device__ __forceinline__ double key_value(uint64_t key) {
  const uint32_t hi = (uint32_t)(key >> 32);
  return hi ? (double)__uint_as_float(hi - 1u) : 0.0;
}

template <int kCtrl, int kRows>
__device__ __forceinline__ double lane_move(double x) {            // 0 where no lane is moved from
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  return __builtin_bit_cast(double, ((uint64_t)lane_move<kCtrl, kRows>(0u, (uint32_t)(b >> 32)) << 32) | lane_move<kCtrl, kRows>(0u, (uint32_t)b));
}
__device__ __forceinline__ double wave_sum(double x) {
  x += lane_move<0x111, 0xf>(x);
  x += lane_move<0x112, 0xf>(x);
  x += lane_move<0x114, 0xf>(x);
  x += lane_move<0x118, 0xf>(x);
  x += lane_move<0x142, 0xa>(x);
  x += lane_move<0x143, 0xc>(x);
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), 63) << 32) |
                                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 63));
}

// value of the lane whose number differs in bit J
template <int J>
__device__ __forceinline__ uint32_t other_lane(uint32_t x, int lane) {
  if (J == 1) return lane_move<0xB1, 0xf>(x, x);                                  // within four: 1 0 3 2
  if (J == 2) return lane_move<0x4E, 0xf>(x, x);                                  // 2 3 0 1
  if (J == 4) {
    const uint32_t y = lane_move<0x141, 0xf>(x, x);                               // eight mirrored, then each four
    return lane_move<0x1B, 0xf>(y, y);
  }
  if (J == 8) return lane_move<0x128, 0xf>(x, x);                                 // sixteen rotated by eight
  uint32_t a = x, b = x;      // a ends up with the lanes whose bit J is 0 in both places, b with the others
  if (J == 16) asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  else asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return lane & J ? a : b;
}
// sum over groups of kLanes lanes, in each of them: with the lane next to it, then two, then four apart
template <int kLanes>
__device__ __forceinline__ float sum_lanes(float x, int lane) {
  auto other = [&](auto j) { return __builtin_bit_cast(float, other_lane<decltype(j)::value>(__builtin_bit_cast(uint32_t, x), lane)); };
  x += other(std::integral_constant<int, 1>());
  if (kLanes > 2) x += other(std::integral_constant<int, 2>());
  if (kLanes > 4) x += other(std::integral_constant<int, 4>());
  return x;
}
template <int K, int J>
__device__ __forceinline__ void sort_step(uint32_t& hi, uint32_t& lo, int lane) {
  const uint32_t oh = other_lane<J>(hi, lane), ol = other_lane<J>(lo, lane);
  const bool less = (((uint64_t)hi << 32) | lo) < (((uint64_t)oh << 32) | ol);
  const bool largest = ((lane & J) == 0) == ((lane & K) == 0);
  const bool take = less == largest;
  hi = take ? oh : hi;
  lo = take ? ol : lo;
  if constexpr (J > 1) sort_step<K, J / 2>(hi, lo, lane);
}
// the first n lanes' (at most kMost) 64-bit keys in descending order, by a bitonic network of 6 (up to 8 lanes) to 21 steps of some ten
// instructions; the other lanes' are 0
template <int kMost>
__device__ __forceinline__ void sort_lanes(uint32_t& hi, uint32_t& lo, int lane, int n) {
  sort_step<2, 1>(hi, lo, lane);
  sort_step<4, 2>(hi, lo, lane);
  if (kMost > 4) sort_step<8, 4>(hi, lo, lane);
  if (kMost > 8 && n > 8) sort_step<16, 8>(hi, lo, lane);
  if (kMost > 16 && n > 16) sort_step<32, 16>(hi, lo, lane);
  if (kMost > 32 && n > 32) sort_step<64, 32>(hi, lo, lane);
}
// sum of the lanes before the lane's own
__device__ __forceinline__ double wave_sum_before(double x) {
  x += lane_move<0x111, 0xf>(x);
  x += lane_move<0x112, 0xf>(x);
  x += lane_move<0x114, 0xf>(x);
  x += lane_move<0x118, 0xf>(x);
  x += lane_move<0x142, 0xa>(x);
  x += lane_move<0x143, 0xc>(x);
  return lane_move<0x138, 0xf>(x);
}

// M(i + ahead) from the masses before the i-th ordinary block (b0), before its predecessor (b1) and before
// the one ahead of that (b2); ranks 0 and 1 carry no mass
__device__ __forceinline__ double rank_mass(int i, int ahead, double b0, double b1, double b2) {
  const int back = 2 - ahead;          // 0, 1 or 2 ordinary blocks fewer than all those ahead of it
  if (i < back) return 0.0;
  return back == 0 ? b0 : (back == 1 ? b1 : b2);
}

// a row's block sums for the caller
__device__ __forceinline__ void store_sums(const SelParams& p, const float* x, int head, int row, int lane) {
  __bf16* out = p.sums_out + ((int64_t)head * p.win_rows + (row - p.win_row0)) * p.nkb;
  for (int c = lane; c < p.nkb; c += 64) out[c] = (__bf16)x[c];
}

// How much of a row is decided at once.  Bound by one wavefront's chain of instructions, and by the longest list where rows are few.
//  - Up to 64 candidates, one per lane: a sort of the lanes and a prefix sum.  (Four pulled out one by one, 1 us each, and the rest
//    ranked against each other, 0.09 us each: selection of a prompt of 4096 tokens 13.6 us, 8.8 so.)
//  - More, in registers, with as many as there are for 128, 256, 512 and 1024: two are pulled out (most rows of text end there), then a
//    search leaves at most 63, which are sorted.  (Six pulled out first, the search down to four that were pulled out, 16 registers
//    always: 2048 tokens on 63488 37.5 -> 24.4 us, video of 65536 159 -> 98, text of 15000 19 -> 15.7, of 32768 53 -> 47.  With one and three
//    pulled out first 23.7 and 25.4, 97 and 101, 16.2 and 14.7, 46.9 and 46.7.)
//  - Beyond 1024, and rows whose sums outrank forced blocks after 32 pulled out: a sort in LDS.
//
// Selection for q-block row `row` of `head` by ONE wavefront (lane = its lane number).  x: the row's nkb block
// sums (global or LDS), at most kMost of them candidates (with all of the ways above in it a kernel of a few candidates had 30 KB more
// code); keys (npow2 entries) and flags (nkb bytes): LDS scratch of this wavefront.  All LDS
// traffic is the wavefront's own, which the LDS keeps in program order: the points where the lanes exchange
// data through it need no workgroup barrier.  x may occupy the LAST 4 * nkb bytes of the key array (rounded up
// to 64 bytes): key c then lands on sums 2c - (2 npow2 - nkb) and the one after, both below c, i.e. sums that
// the loops which fill the keys (ascending c, a whole wavefront's reads before its writes) have read already.
template <int kMost = 1 << 30>
__device__ __forceinline__ void select_row(const SelParams& p, const float* x, int head, int row, uint64_t* keys,
                                           uint8_t* flags, int lane) {
  const int64_t slot = (int64_t)head * p.win_rows + (row - p.win_row0);   // this row's place in the arrays
  const int diag = row + p.diag_offset;
  // Column index of the first diagonal of the row's query chunk.  When it is 0
  // the reference's eye() assignment overwrites the forced sink column
  // (utils.py:100-106), leaving the diagonal as the only forced block while
  // the [0, forced_sum, ...] prefix (utils.py:115-124) still reserves two
  // slots: the largest other block is then always kept and every later one is
  // judged against the mass gathered before its predecessor.
  const int chunk_first = p.diag_offset + (row / p.blocks_per_chunk) * p.blocks_per_chunk;
  const bool one_forced = p.causal && chunk_first == 0;

  // candidates: columns [0, ncand); when causal nothing beyond the diagonal can be kept
  int ncand = p.nkb;
  if (p.causal) ncand = diag + 1 < p.nkb ? diag + 1 : p.nkb;
  if (ncand < 0) ncand = 0;
  int np2 = 64;
  while (np2 < ncand) np2 <<= 1;

  // (the forced blocks' sums are read before any sort key is written: x may share its memory with the tail of
  // the key array, see below)
  double forced_sum = 0.0;
  // sort keys of the forced blocks (utils.py:126-130); key_hi >= key_lo, equal when only one block is forced
  double key_lo = 0.0, key_hi = 0.0;
  auto sum_of = [&](int c) { return (double)__uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(x[c]))); };
  if (p.causal && ncand > 0) {
    if (!one_forced || diag == 0) forced_sum = sum_of(0);
    if (diag != 0 && diag < p.nkb) forced_sum += sum_of(diag);
    const double kd = 100000.0 * (1.0 + sum_of(diag < p.nkb ? diag : 0));
    const double k0 = one_forced ? kd : 100000.0 * (1.0 + sum_of(0));
    key_lo = kd < k0 ? kd : k0;
    key_hi = kd < k0 ? k0 : kd;
  }
  // value bits of candidate c (0 for forced blocks and columns past the candidates)
  auto load_one = [&](int c, double& sum) -> uint32_t {
    uint32_t bits = 0;
    if (c < ncand) {
      const float v = x[c];
      sum += (double)v;
      const bool forced = p.causal && (c == diag || (c == 0 && !one_forced));
      // block sums are >= 0, so their bit pattern orders like the value (+1
      // keeps every candidate ahead of the forced blocks, which sort last)
      bits = forced ? 0u : __float_as_uint(v > 0.f ? v : 0.f) + 1u;
    }
    return bits;
  };
  // sort key: low word = ~column makes equal sums come out by ascending column; padding (c >= ncand) sorts
  // last and carries an out-of-range column
  auto sort_key = [&](int c, uint32_t bits) -> uint64_t {
    return c < ncand ? (((uint64_t)bits << 32) | (uint32_t)(~(uint32_t)c)) : 0ull;
  };
  const int n_forced = one_forced ? 1 : 2;
  // forced keys ranked ahead of an ordinary block of sum v (all of them unless v is beyond 100000)
  auto forced_ahead = [&](double v) -> int {
    if (!(v > key_lo)) return n_forced;
    return one_forced ? 0 : (v > key_hi ? 0 : 1);
  };
  double required = 0.0;
  // no block sum can exceed a forced key unless the row's total does: otherwise the forced blocks rank first
  // and a decision does not need the block's own value
  bool may_outrank = false;
  auto total_is = [&](double total) {
    required = total * (p.tau ? p.tau[head] : p.tau_val[head * p.tau_step]);
    may_outrank = p.causal && total > key_lo;
  };
  int dropped = 0;
  bool finished = false;
  // At most 64 candidates, one key in each of the first n lanes, behind `taken` others: `before` is the mass ahead of them and prev_before that ahead
  // of the last one taken.  Sorted, each lane finds the mass ahead of its own in a prefix sum.
  auto decide_lanes = [&](uint64_t key, int n, double before, double prev_before, int taken) {
    uint32_t hi = (uint32_t)(key >> 32), lo = (uint32_t)key;
    sort_lanes<kMost>(hi, lo, lane, n);
    const double v = hi ? (double)__uint_as_float(hi - 1u) : 0.0;
    double mass = before + wave_sum_before(v);
    if (may_outrank) {                     // (then they are all of the row's, and nothing was taken)
      const double b1 = lane_move<0x138, 0xf>(mass), b2 = lane_move<0x138, 0xf>(b1);
      mass = rank_mass(lane, forced_ahead(v), mass, b1, b2);
    } else if (one_forced) {
      const double b1 = lane_move<0x138, 0xf>(mass);
      mass = lane > 0 ? b1 : taken > 0 ? prev_before : 0.0;
    }
    if (hi != 0) {
      if (mass < required) flags[~lo] = 1;
      else dropped = 1;
    }
    finished = true;
  };
  // More than 64 candidates, in registers: slot u of a lane holds column u*64 + lane.
  auto decide_slots = [&](auto slots) {
    constexpr int S = decltype(slots)::value;
    uint32_t vals[S];
    double total = 0.0;
    int n_others = 0;
#pragma unroll
    for (int u = 0; u < S; ++u) {
      vals[u] = load_one(u * 64 + lane, total);
      n_others += __popcll(__ballot(vals[u] != 0));
    }
    total_is(wave_sum(total));
    // the largest that is left, and it taken from the lowest column that holds it
    auto largest = [&]() {
      uint32_t best = 0;
#pragma unroll
      for (int u = 0; u < S; ++u) best = vals[u] > best ? vals[u] : best;
      return wave_max(best);
    };
    auto pull = [&](uint32_t best) {
      uint32_t col = 0xffffffffu;
#pragma unroll
      for (int u = S - 1; u >= 0; --u) col = vals[u] == best ? (uint32_t)(u * 64 + lane) : col;
      col = wave_min(col);
#pragma unroll
      for (int u = 0; u < S; ++u) vals[u] = (uint32_t)(u * 64 + lane) == col ? 0u : vals[u];
      return col;
    };
    // ---- extraction: keep pulling out the largest remaining block while the rule says "keep"
    double before = forced_sum, prev_before = 0.0, prev2_before = 0.0;
    int taken = 0;               // blocks kept so far
    for (int it = 0; it < kMaxExtract; ++it) {
      if (it == kBeforeSearch && n_others > 0 && !may_outrank) {
        // ---- a long list: bisection on the value for hi > lo with  before + (sum of values >= hi) < required  and
        // before + (sum of values >= lo) >= required.  Everything from hi on is kept, and at most 63 blocks are left to decide.
        uint32_t hi = largest() + 1;
        uint32_t lo = 0, step = 1u << 22;        // (lo 0: not known yet; first the search goes down by growing steps)
        int above = 0, from_lo = n_others;       // candidates >= hi, >= lo
        double mass_hi = 0.0;
        while (hi - lo > 1 && from_lo - above > 63) {
          const uint32_t mid = lo ? lo + (hi - lo) / 2 : (hi > step + 1 ? hi - step : 1);
          int n = 0;
          double sum = 0.0;
#pragma unroll
          for (int u = 0; u < S; ++u) {
            uint32_t w = vals[u];
            asm volatile("" : "+v"(w));          // (else every value is kept as a double across the loop)
            const bool in = w >= mid;
            n += __popcll(__ballot(in));
            sum += in ? (double)__uint_as_float(w - 1u) : 0.0;
          }
          sum = wave_sum(sum);
          if (before + sum < required) {
            hi = mid;
            mass_hi = sum;
            above = n;
            step <<= 1;
          } else {
            lo = mid;
            from_lo = n;
          }
        }
        if (above > 0) {
          uint32_t least = 0xffffffffu;          // the last of the blocks taken
#pragma unroll
          for (int u = 0; u < S; ++u) {
            const bool in = vals[u] >= hi;
            least = in && vals[u] < least ? vals[u] : least;
            if (in) flags[u * 64 + lane] = 1;
            vals[u] = in ? 0u : vals[u];
          }
          least = wave_min(least);
          before += mass_hi;
          prev_before = before - (double)__uint_as_float(least - 1u);
          n_others -= above;
          taken += above;
        }
        if (from_lo - above <= 63) {
          // they come together in the key array, with the largest of those below, which may be judged by the mass ahead of its
          // predecessor; the others below are dropped
          int n = 0;
#pragma unroll
          for (int u = 0; u < S; ++u) {
            const bool in = vals[u] != 0 && vals[u] >= lo;
            const uint64_t ballot = __ballot(in);
            if (in) keys[n + __popcll(ballot & ((1ull << lane) - 1ull))] = sort_key(u * 64 + lane, vals[u]);
            vals[u] = in ? 0u : vals[u];
            n += __popcll(ballot);
          }
          if (n < n_others) {
            const uint32_t best = largest(), col = pull(best);
            if (lane == 0) keys[n] = sort_key((int)col, best);
            if (++n < n_others) dropped = 1;
          }
          __builtin_amdgcn_wave_barrier();
          decide_lanes(lane < n ? keys[lane] : 0ull, n, before, prev_before, taken);
          return;
        }
        // a run of equal sums: they come out by ascending column, each adding the same mass
        const double t = (double)__uint_as_float(lo - 1u);
        const int shift = one_forced && taken > 0 ? 1 : 0;     // judged against the mass before its predecessor
        int seen = 0, kept = 0;
#pragma unroll
        for (int u = 0; u < S; ++u) {
          const bool in = vals[u] == lo;
          const uint64_t tied = __ballot(in);
          const int i = seen + __popcll(tied & ((1ull << lane) - 1ull));
          const double mass = shift && i == 0 ? prev_before : before + (double)(i - shift) * t;
          const bool keep = in && mass < required;
          if (keep) flags[u * 64 + lane] = 1;
          vals[u] = keep ? 0u : vals[u];
          kept += __popcll(__ballot(keep));
          seen += __popcll(tied);
        }
        if (kept < seen) {
          finished = true;
          dropped = 1;
          return;
        }
        before += (double)kept * t;
        prev_before = before - t;
        n_others -= kept;
        taken += kept;
      }
      if (n_others == 0) {
        finished = true;
        return;
      }
      if (!may_outrank) {
        const double mass = p.causal ? rank_mass(taken, n_forced, before, prev_before, prev2_before) : before;
        if (!(mass < required)) {
          finished = true;
          dropped = 1;
          return;
        }
      }
      const uint32_t best = largest();
      const double best_val = (double)__uint_as_float(best - 1u);
      if (may_outrank) {
        const double mass = rank_mass(taken, forced_ahead(best_val), before, prev_before, prev2_before);
        if (!(mass < required)) {
          finished = true;
          dropped = 1;
          return;
        }
      }
      const uint32_t col = pull(best);
      if (lane == 0) flags[col] = 1;
      prev2_before = prev_before;
      prev_before = before;
      before += best_val;
      --n_others;
      ++taken;
    }
  };
  for (int c = lane; c < p.nkb; c += 64) flags[c] = 0;
  __builtin_amdgcn_wave_barrier();
  const bool small = np2 <= kMostSlots * 64;
  if (kMost <= 64 || np2 == 64) {
    double total = 0.0;
    const uint32_t bits = load_one(lane, total);
    total_is(wave_sum(total));
    decide_lanes(sort_key(lane, bits), ncand, forced_sum, 0.0, 0);
  } else if constexpr (kMost > 64) {
    if (np2 == 128) {
      decide_slots(std::integral_constant<int, 2>{});
    } else if (np2 == 256) {
      decide_slots(std::integral_constant<int, 4>{});
    } else if (np2 == 512) {
      decide_slots(std::integral_constant<int, 8>{});
    } else if (small) {
      decide_slots(std::integral_constant<int, kMostSlots>{});
    } else {
      double total = 0.0;
      for (int c = lane; c < np2; c += 64) keys[c] = sort_key(c, load_one(c, total));
      total_is(wave_sum(total));
      __builtin_amdgcn_wave_barrier();
    }
  }

  if (kMost > 64 && !finished) {
  if (small) {
    double again = 0.0;
    for (int c = lane; c < np2; c += 64) keys[c] = sort_key(c, load_one(c, again));
    __builtin_amdgcn_wave_barrier();
  }
  // ---- bitonic sort, descending
  for (int k = 2; k <= np2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = lane; t < (np2 >> 1); t += 64) {
        const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
        const int l = i | j;
        const uint64_t a = keys[i], b = keys[l];
        const bool up = (i & k) == 0;        // this pair's run is descending
        if ((a < b) == up) {
          keys[i] = b;
          keys[l] = a;
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }

  // fp64 exclusive prefix over the sorted values; rank kept while mass before it < required
  const int per = np2 >> 6;
  double local = 0.0;
  for (int u = 0; u < per; ++u) local += key_value(keys[lane * per + u]);
  double incl = local;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const double o = __shfl_up(incl, d, 64);
    if (lane >= d) incl += o;
  }
  double before = forced_sum + (incl - local);
  for (int u = 0; u < per; ++u) {
    const int rank = lane * per + u;
    const uint64_t key = keys[rank];
    const uint32_t col = ~(uint32_t)key;
    if (col < (uint32_t)ncand && (key >> 32) != 0) {
      double mass = before;
      if (may_outrank) {
        const double b1 = rank > 0 ? before - key_value(keys[rank - 1]) : 0.0;
        const double b2 = rank > 1 ? b1 - key_value(keys[rank - 2]) : 0.0;
        mass = rank_mass(rank, forced_ahead(key_value(key)), before, b1, b2);
      } else if (one_forced) {
        mass = rank == 0 ? 0.0 : before - key_value(keys[rank - 1]);
      }
      if (mass < required) flags[col] = 1;
      else dropped = 1;
    }
    before += key_value(key);
  }
  }   // sort path
  const bool any_dropped = __any(dropped);
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    if (p.causal) {
      if (p.nkb > 0) flags[0] = 1;
      if (diag >= 0 && diag < p.nkb) flags[diag] = 1;
    } else if (any_dropped) {
      flags[0] = 1;     // unselected ranks scatter to column 0 (utils.py:164)
    }
    if (p.keep_recent && diag >= 0 && diag < p.nkb) flags[diag] = 1;
  }
  __builtin_amdgcn_wave_barrier();
  if (p.keep_sink && row == 0)
    for (int c = lane; c < p.nkb; c += 64) flags[c] = 1;
  __builtin_amdgcn_wave_barrier();

  if (p.mask) {
    uint8_t* mrow = p.mask + slot * p.nkb;
    for (int c = lane; c < p.nkb; c += 64) mrow[c] = flags[c];
  }

  if (p.col_idx) {
    int32_t* list = p.col_idx + slot * p.idx_pitch;
    const int q_last = (row * 128 + 127 < p.q_len ? row * 128 + 127 : p.q_len - 1) + p.kv_off;
    int count = 0;
    for (int c0 = 0; c0 < p.nkb; c0 += 64) {
      const int c = c0 + lane;
      bool keep = c < p.nkb && flags[c] && c < p.list_cols;
      if (p.causal) keep = keep && (c * 128 <= q_last);
      const uint64_t ballot = __ballot(keep);
      const int pos = count + __popcll(ballot & ((1ull << lane) - 1ull));
      if (keep && pos < p.idx_pitch) list[pos] = c;
      count += __popcll(ballot);
    }
    count = count < p.idx_pitch ? count : (int)p.idx_pitch;
    if (lane == 0) p.col_cnt[slot] = count;
    if (lane == 0 && p.totals) {
      uint32_t* const of = p.totals + 32 * (row - p.win_row0);
      __hip_atomic_fetch_add(of, (uint32_t)count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_max(of + 1, (uint32_t)count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (kMost > 64 && p.plan.shape.per_qb && (p.causal ? q_last / 128 + 1 : p.list_cols) > p.plan.shape.min_piece)   // else too few blocks to be cut
      list_made(p.plan, p.H, p.win_rows, row - p.win_row0, head, count, lane);
  }
}

}  // namespace xattn
