// Load-balanced work plan of the decode kernels, computed on the device.
//
// The work of a call is the list of 32-token blocks of every row (GQA row =
// (sequence, kv head), MLA row = sequence), rows in order.  With
// nb(b) = ceil(len_b / 32) blocks per row of sequence b and R rows per
// sequence, T = sum_b R * nb(b).  A grid of n workgroups gives workgroup g
// the blocks [floor(g T / n), floor((g + 1) T / n)), so every workgroup
// streams the same amount of KV whatever the lengths (n is capped at T, so
// no range is empty).  A workgroup walks its range as row segments; a row
// covered by several workgroups gets one partial per workgroup, stored in
// slot g + row: along the block order both g and row are non-decreasing, so
// g + row is distinct for every (workgroup, row) pair and slots stay below
// n + rows.
#pragma once

#include "ws_common.h"

namespace ws {

// Most sequences a call takes (the per-sequence prefix lives in LDS).
constexpr int kMaxSeqs = 2048;
// Most splits a call takes: plan_start's products stay below 2^24, plan_align's
// counts within 16 bits, and plan_owner's quotients exact.
constexpr int kMaxSplits = 4096;

struct Plan {
  int T;  // total blocks (the host keeps it below 2^31 / grid)
  int n;  // workgroups with work (min(grid, T)), at most kMaxSplits
  int q, r;  // T = q n + r
  // The calling split's range [begin, end) and the sequence of block `begin`.
  bool has_work;
  int begin, end, b0;
};

// Wave-wide inclusive prefix sum from the ROCm device library (ockl), a
// DPP sequence: every lane of the wave must be active.
extern "C" __device__ int __ockl_wfscan_add_i32(int, bool);

// Most sequences the sequence-aligned plan takes (four a lane).
constexpr int kSeqPlanMax = 256;
// Step of the block counts per split the sequence-aligned plan tries over
// ceil(T / n): up to three steps are accepted.  A split whose range enters a
// second sequence restarts its load stream there, which costs the 16-head MLA
// step about four blocks' time and the wide one (queries of 128 heads in, 128
// KB of outputs out) about ten.
constexpr int kAlignStep = 1;
constexpr int kAlignStepWide = 3;

// Workgroup-uniform value moved to a scalar register.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// A length the call can serve: 0 <= l <= cap - add (room for the appended
// token when add == 1).  A length outside that range (a caller's mistake, or
// the -1 a fused step leaves after one) is not clamped: the sequence gets no
// blocks, its outputs are NaN and a fused step writes len_out = -1.
__device__ __forceinline__ bool len_ok(int l, int add, int cap) {
  return l >= 0 && l <= cap - add;
}

// Sequence length used by the kernels: len_in[b] + add (1 when the call
// appends the step's new token), or 0 for a length outside the valid range.
__device__ __forceinline__ int plan_len(const int32_t* len_in, int b, int add, int cap) {
  const int l = len_in[b];
  return len_ok(l, add, cap) ? l + add : 0;
}

// Length slot of plan sequence v.  A call whose sequences carry ng groups
// of 16 query heads over one shared latent (absorbed MLA with H = 16 ng)
// plans over v = b ng + group: each group is its own plan sequence with
// sequence b's length.
__device__ __forceinline__ int seq_of(int v, int ng) { return ng == 1 ? v : v / ng; }

// len_out of a fused step: the new length, or -1 for an invalid len_in.
__device__ __forceinline__ int step_len_out(const int32_t* len_in, int b, int add, int cap) {
  const int l = len_in[b];
  return len_ok(l, add, cap) ? l + add : -1;
}

__device__ __forceinline__ Plan plan_of(int T, int grid) {
  Plan p;
  p.T = T;
  p.n = min(grid, T);
  p.q = p.n > 0 ? (int)((unsigned)T / (unsigned)p.n) : 0;
  p.r = T - p.q * p.n;
  p.has_work = false;
  p.begin = p.end = 0;
  p.b0 = -1;
  return p;
}

// floor(g T / n) as g q + floor(g r / n): 32-bit products (g r < n^2 <= 2^24)
// and one 32-bit division, for 0 <= g <= n.
__device__ __forceinline__ int plan_start(const Plan& p, int g) {
  return g * p.q + (int)((unsigned)(g * p.r) / (unsigned)p.n);
}

// Splits of a sequence of nb blocks at M blocks per split (rM: v_rcp_f32's 1 / M,
// good to an ulp): ceil(nb / M), or one fewer where nb - 1 is a multiple of M and
// the product rounds below it (a split then takes M + 1 blocks).  At least 1 and
// at most nb for nb > 0 (nb < 2^19), and the same in every kernel, which is what
// the plan needs.
__device__ __forceinline__ int plan_nsplits(int nb, float rM) {
  return nb > 0 ? (int)((float)(nb - 1) * rM) + 1 : 0;
}

// The sequence-aligned plan's blocks per split: the first M of base, base +
// step, base + 2 step, base + 3 step, base = ceil(T / n), at which the
// sequences (nb: the blocks of a lane's K sequences) need at most n splits, or
// 0 if there is none.  The four candidates are counted in one pass, summed
// over the wave as 16-bit halves (each count is at most n + 2 B).  Every lane
// must call it.
template <int K>
__device__ __forceinline__ int plan_align(const int (&nb)[K], const Plan& p, int step) {
  const int base = (p.T + p.n - 1) / p.n;
  float rM[4];
  uint32_t cnt[2] = {0, 0};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    rM[c] = __builtin_amdgcn_rcpf((float)(base + c * step));
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) sum += plan_nsplits(nb[k], rM[c]);
    cnt[c >> 1] += sum << (16 * (c & 1));
  }
  cnt[0] = __ockl_wfred_add_u32(cnt[0]);
  cnt[1] = __ockl_wfred_add_u32(cnt[1]);
  int M = 0;
#pragma unroll
  for (int c = 3; c >= 0; --c)
    if (uniform((cnt[c >> 1] >> (16 * (c & 1))) & 0xffffu) <= p.n) M = base + c * step;
  return M;
}

// plan_build for at most 64 K sequences, K consecutive ones a lane.
template <int K>
__device__ __forceinline__ Plan plan_build_k(const int32_t* len_in, int add, int cap, int B, int R,
                                             int grid, int* s_pref, int* s_len, int g, int ng,
                                             int step) {
  const int lane = threadIdx.x & 63;
  const int v0 = K * lane;
  int l[K], nb[K], sum = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    l[k] = K > 1 || lane < B ? plan_len(len_in, seq_of(min(v0 + k, B - 1), ng), add, cap) : 0;
    if (v0 + k >= B) l[k] = 0;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    nb[k] = R * ((l[k] + 31) >> 5);
    sum += nb[k];
  }
  const int incl = __ockl_wfscan_add_i32(sum, true);
  int run = incl - sum;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (v0 + k < B) {
      s_pref[v0 + k] = run;
      s_len[v0 + k] = l[k];
    }
    run += nb[k];
  }
  const int T = __builtin_amdgcn_readlane(incl, 63);
  if (lane == 0) s_pref[B] = T;
  Plan p = plan_of(T, grid);
  const int M = R == 1 && B >= 2 && p.n > 0 ? plan_align<K>(nb, p, step) : 0;
  if (M > 0) {
    const float rM = __builtin_amdgcn_rcpf((float)M);
    int ns[K], nsum = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      ns[k] = plan_nsplits(nb[k], rM);
      nsum += ns[k];
    }
    const int w = __ockl_wfscan_add_i32(nsum, true);
    if (g >= 0 && g < __builtin_amdgcn_readlane(w, 63)) {
      // split g: its lane (the first with w > g), the lane's sequence and the
      // split's number j of that sequence's
      const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(w > g));
      int j = g - __builtin_amdgcn_readlane(w - nsum, at);
      int first = __builtin_amdgcn_readlane(incl - sum, at);
      int nbb = __builtin_amdgcn_readlane(nb[0], at);
      int nsb = __builtin_amdgcn_readlane(ns[0], at);
      p.b0 = K * at;
#pragma unroll
      for (int k = 1; k < K; ++k) {
        const int nbk = __builtin_amdgcn_readlane(nb[k], at);
        const int nsk = __builtin_amdgcn_readlane(ns[k], at);
        if (p.b0 == K * at + k - 1 && j >= nsb) {
          j -= nsb;
          first += nbb;
          nbb = nbk;
          nsb = nsk;
          p.b0 = K * at + k;
        }
      }
      p.has_work = true;
      p.begin = first + j * nbb / nsb;
      p.end = first + (j + 1) * nbb / nsb;
    }
    return p;
  }
  if (g >= 0 && g < p.n) {
    p.has_work = true;
    p.begin = plan_start(p, g);
    p.end = plan_start(p, g + 1);
    // the lane of the first sequence that ends past block `begin`, and which
    const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(incl > p.begin));
    int last = __builtin_amdgcn_readlane(incl - sum, at);
    p.b0 = K * at;
#pragma unroll
    for (int k = 0; k + 1 < K; ++k) {
      last += __builtin_amdgcn_readlane(nb[k], at);
      if (last <= p.begin) p.b0 = K * at + k + 1;
    }
  }
  return p;
}

// Builds s_pref[0..B] (exclusive prefix of blocks per sequence, R rows each)
// and the lengths s_len[0..B) (plan_len), and returns the plan.  Every wave
// of the workgroup calls it with all its lanes, builds the whole plan by
// itself (B <= 64: lane b is sequence b; above, ceil(B / 64) consecutive
// ones a lane) and writes the same values, reading back only what it wrote:
// no barrier between the kernel start and its first loads.  (With more than
// 64 sequences built together by the workgroup, behind three barriers and a
// chain of one load per sequence of a lane, GQA B = 256 took 204.7 us a step,
// against 187.5 with every wave on its own here and in the merge.)
//
// With one row per sequence (R == 1) and 2 to kSeqPlanMax sequences, the plan
// may instead be sequence-aligned: sequence b gets n_b = plan_nsplits(nb(b), M)
// splits, M the first block count per split of plan_align with sum_b n_b <= n,
// which take equal shares of its blocks, so no split spans two sequences.
// Every kernel of a call (step and merge) passes the same arguments and so
// makes the same choice.
//
// Split g (g >= 0) gets its range in has_work / begin / end and the sequence
// of its first block in b0.
//
// ng > 1: B counts plan sequences v = b ng + group, whose lengths are
// len_in[v / ng] (seq_of).  step: kAlignStep or kAlignStepWide.
__device__ __forceinline__ Plan plan_build(const int32_t* len_in, int add, int cap, int B, int R,
                                           int grid, int* s_pref, int* s_len, int g, int ng,
                                           int step) {
  if (__builtin_expect(B >= 1 && B <= 64, 1))
    return plan_build_k<1>(len_in, add, cap, B, R, grid, s_pref, s_len, g, ng, step);
  if (B <= kSeqPlanMax)
    return plan_build_k<4>(len_in, add, cap, B, R, grid, s_pref, s_len, g, ng, step);
  // lane: sequences c * lane .. c * lane + c - 1, four loads at a time
  const int lane = threadIdx.x & 63;
  const int c = (B + 63) >> 6;
  const int v0 = c * lane;
  int sum = 0;
  for (int k0 = 0; k0 < c; k0 += 4) {
    int l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      l[k] = plan_len(len_in, seq_of(min(v0 + k0 + k, B - 1), ng), add, cap);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k0 + k >= c || v0 + k0 + k >= B) continue;
      s_len[v0 + k0 + k] = l[k];
      sum += R * ((l[k] + 31) >> 5);
    }
  }
  const int incl = __ockl_wfscan_add_i32(sum, true);
  // (only final values go to LDS: the workgroup's waves all write them)
  int run = incl - sum;
  for (int k = 0; k < min(c, B - v0); ++k) {
    s_pref[v0 + k] = run;
    run += R * ((s_len[v0 + k] + 31) >> 5);
  }
  const int T = __builtin_amdgcn_readlane(incl, 63);
  if (lane == 0) s_pref[B] = T;
  Plan p = plan_of(T, grid);
  if (g >= 0 && g < p.n) {
    p.has_work = true;
    p.begin = plan_start(p, g);
    p.end = plan_start(p, g + 1);
    // the lane with the first sequence that ends past block `begin`, then the
    // sequence among its c <= 32
    const int vb = c * __builtin_ctzll(__builtin_amdgcn_ballot_w64(incl > p.begin));
    const bool past = lane < c && vb + lane < B && s_pref[min(vb + lane + 1, B)] <= p.begin;
    p.b0 = vb + __builtin_popcountll(__builtin_amdgcn_ballot_w64(past));
  }
  return p;
}

// Workgroup whose range holds block blk: ceil((blk + 1) n / T) - 1.  The
// double quotient is exact enough: the operands are integers below 2^53, and
// a quotient that is not an integer lies at least 1 / T > 2^-31 below the
// next one, far above the rounding error of a quotient of at most 4096.
__device__ __forceinline__ int plan_owner(const Plan& p, int blk) {
  return (int)ceil((double)(blk + 1) * (double)p.n / (double)p.T) - 1;
}

// What a merge needs of the plan: the pieces of one row.
struct RowSplits {
  int nbb;      // the row's blocks (0: no pieces, its partial is in out / lse)
  int w_first;  // its first split
  int nseg;     // and how many splits hold it
};

// The pieces of row r of plan sequence v under plan_build's plan, from wave
// sums over the lengths: no prefix in LDS and no barrier, so a merge's start
// costs one coalesced load of the lengths, whatever the batch (a merge
// workgroup per output row that rebuilt the whole prefix made the merge of
// 256 sequences x 32 heads 24 us, and of 96 sequences x 8 head groups 116).
// Every lane of the wave must be active; v and r are wave-uniform.
template <int K>
__device__ __forceinline__ RowSplits plan_row_k(const int32_t* len_in, int add, int cap, int B,
                                                int R, int grid, int v, int r, int ng,
                                                int step) {
  const int lane = threadIdx.x & 63;
  int nb[K];
  uint32_t sum = 0, before = 0;
  RowSplits rs{0, 0, 0};
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int u = lane + 64 * k;
    int l = plan_len(len_in, seq_of(min(u, B - 1), ng), add, cap);
    if (u >= B) l = 0;
    nb[k] = (l + 31) >> 5;
    sum += nb[k];
    before += u < v ? nb[k] : 0;
    if (k == (v >> 6)) rs.nbb = __builtin_amdgcn_readlane(nb[k], v & 63);
  }
  if (rs.nbb == 0) return rs;
  const Plan p = plan_of(R * uniform((int)__ockl_wfred_add_u32(sum)), grid);
  const int M = R == 1 && B >= 2 ? plan_align<K>(nb, p, step) : 0;
  if (M > 0) {
    const float rM = __builtin_amdgcn_rcpf((float)M);
    uint32_t ns = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) ns += lane + 64 * k < v ? plan_nsplits(nb[k], rM) : 0;
    rs.w_first = uniform((int)__ockl_wfred_add_u32(ns));
    rs.nseg = uniform(plan_nsplits(rs.nbb, rM));
  } else {
    const int start = R * uniform((int)__ockl_wfred_add_u32(before)) + r * rs.nbb;
    rs.w_first = plan_owner(p, start);
    rs.nseg = plan_owner(p, start + rs.nbb - 1) - rs.w_first + 1;
  }
  return rs;
}
__device__ __forceinline__ RowSplits plan_row(const int32_t* len_in, int add, int cap, int B,
                                              int R, int grid, int v, int r, int ng,
                                              int step) {
  if (B <= 64) return plan_row_k<1>(len_in, add, cap, B, R, grid, v, r, ng, step);
  if (B <= kSeqPlanMax) return plan_row_k<4>(len_in, add, cap, B, R, grid, v, r, ng, step);
  const int lane = threadIdx.x & 63;
  uint32_t sum = 0, before = 0;
#pragma unroll 4
  for (int u = lane; u < B; u += 64) {
    const int nb = (plan_len(len_in, seq_of(u, ng), add, cap) + 31) >> 5;
    sum += nb;
    before += u < v ? nb : 0;
  }
  RowSplits rs{(plan_len(len_in, seq_of(v, ng), add, cap) + 31) >> 5, 0, 0};
  const uint32_t tot = __ockl_wfred_add_u32(sum);
  const uint32_t bef = __ockl_wfred_add_u32(before);
  if (rs.nbb == 0) return rs;
  const Plan p = plan_of(R * uniform((int)tot), grid);
  const int start = R * uniform((int)bef) + r * rs.nbb;
  rs.w_first = plan_owner(p, start);
  rs.nseg = plan_owner(p, start + rs.nbb - 1) - rs.w_first + 1;
  return rs;
}

// Sequence holding block blk: the last b with s_pref[b] <= blk (B >= 1).
__device__ __forceinline__ int plan_seq(const int* s_pref, int B, int blk) {
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (uniform(s_pref[mid]) <= blk) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

}  // namespace ws
