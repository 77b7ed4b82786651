// LSE merges, fused with the final normalisation and the bf16 cast:
//   lse_merge_kernel       a GPU partial with a second (host) partial: one
//                          workgroup per row, one float4 of the output per thread
//   merge_split_kernel     a split step's pieces, with or without a host partial
//   merge_split_uv_kernel  the same of an absorbed-MLA step, through W_UV
// The host partial may arrive in any of the reference CPU kernels' output
// conventions, so no conversion launch is needed after its host-to-device copy,
// and may be pinned host memory, read in place.
#include <math.h>

#include <algorithm>

#include "ws_plan.h"
#include "ws_reduce.h"

namespace ws {

template <int FMT>
__device__ __forceinline__ void load_b(const void* b_out, const void* aux0,
                                       const void* aux1, int row, int Dv, int c,
                                       float& lse_b, float4& o_b) {
  if (FMT == WS_PARTIAL_LSE_F32) {
    lse_b = ((const float*)aux0)[row];
    o_b = ((const float4*)((const float*)b_out + (size_t)row * Dv))[c];
  } else if (FMT == WS_PARTIAL_LSE_BF16) {
    lse_b = ((const float*)aux0)[row];
    const uint2 raw = ((const uint2*)((const uint16_t*)b_out + (size_t)row * Dv))[c];
    o_b = make_float4(bf16_to_f32(raw.x & 0xffffu), bf16_to_f32(raw.x >> 16),
                      bf16_to_f32(raw.y & 0xffffu), bf16_to_f32(raw.y >> 16));
  } else if (FMT == WS_TRIPLE_UNNORM_F32 || FMT == WS_TRIPLE_NORM_F32) {
    const float m = ((const float*)aux0)[row];
    const float s = ((const float*)aux1)[row];
    lse_b = (s == 0.f) ? neg_inf() : m + __logf(s);
    o_b = ((const float4*)((const float*)b_out + (size_t)row * Dv))[c];
    if (FMT == WS_TRIPLE_UNNORM_F32) {
      const float inv = (s > 0.f) ? 1.f / s : 0.f;
      o_b.x *= inv;
      o_b.y *= inv;
      o_b.z *= inv;
      o_b.w *= inv;
    }
  } else {  // WS_TRIPLE_NORM_BF16
    const float m = bf16_to_f32(((const uint16_t*)aux0)[row]);
    const float s = bf16_to_f32(((const uint16_t*)aux1)[row]);
    lse_b = (s == 0.f) ? neg_inf() : m + __logf(s);
    const uint2 raw =
        ((const uint2*)((const uint16_t*)b_out + (size_t)row * Dv))[c];
    o_b = make_float4(bf16_to_f32(raw.x & 0xffffu), bf16_to_f32(raw.x >> 16),
                      bf16_to_f32(raw.y & 0xffffu), bf16_to_f32(raw.y >> 16));
  }
}

template <int FMT>
__global__ __launch_bounds__(128) void lse_merge_kernel(
    const float* __restrict__ out_g, const float* __restrict__ lse_g,
    const void* __restrict__ b_out, const void* __restrict__ b_aux0,
    const void* __restrict__ b_aux1, uint16_t* __restrict__ out_bf16,
    float* __restrict__ out_f32, float* __restrict__ lse_out, int Dv) {
  const int row = blockIdx.x;
  const int c = threadIdx.x;
  if (c >= Dv / 4) return;
  const float la = lse_g[row];
  float lb;
  float4 ob;
  load_b<FMT>(b_out, b_aux0, b_aux1, row, Dv, c, lb, ob);
  const float M = max_nan(la, lb);
  float4 r;
  float lse_r;
  if (M == neg_inf()) {
    r = make_float4(0.f, 0.f, 0.f, 0.f);
    lse_r = neg_inf();
  } else {
    const float wa = __expf(la - M);
    const float wb = __expf(lb - M);
    const float inv = 1.f / (wa + wb);
    const float4 oa = ((const float4*)(out_g + (size_t)row * Dv))[c];
    // An empty side has weight 0; its (0) output must not turn into NaN.
    const float fa = wa * inv, fb = wb * inv;
    r = make_float4(fa * oa.x + fb * ob.x, fa * oa.y + fb * ob.y,
                    fa * oa.z + fb * ob.z, fa * oa.w + fb * ob.w);
    lse_r = M + __logf(wa + wb);
  }
  if (out_f32) ((float4*)(out_f32 + (size_t)row * Dv))[c] = r;
  if (out_bf16) {
    uint2 packed;
    packed.x = pack_bf16x2(r.x, r.y);
    packed.y = pack_bf16x2(r.z, r.w);
    ((uint2*)(out_bf16 + (size_t)row * Dv))[c] = packed;
  }
  if (lse_out && c == 0) lse_out[row] = lse_r;
}

// ---------------------------------------------------------------------------
// Split combine + host merge of a deferred-combine decode step.
//
// It rebuilds the step's plan from the post-step lengths (ws_plan.h) to find
// the GPU pieces of a plan row (kv row): the final (out, lse) the step wrote
// when one workgroup held the row, else the partials of the row's workgroups
// (slots w + kv row), then LSE-combines them with the host partial (format FMT,
// or none when FMT < 0) and writes the normalised result.  Runs after the step
// on the same stream, so plain loads see its writes.
//
// A wave owns a group of up to 64 float4 columns: the whole output rows (heads)
// of the plan row that fit, or a part of one row wider than 256.  What bounds a
// merge is the chain of round trips (lengths, then pieces) and, for rows of
// many pieces, how many piece loads are in flight.  So the lse values travel
// with the pieces' columns (piece_batch keeps running weights; no pass over
// the lse values first), and PS waves share a column group, wave i taking
// pieces i, i + PS, ... and the first combining them through LDS.  With few
// pieces a row (PS = 1) a wave walks several groups of its plan row on one plan.
//   (weights first, one wave a row and 256 columns: 32 rows of 64 pieces x 128
//   columns 6.8 us, 128 rows of 32 pieces x 512 columns 6.0, 12288 rows of two
//   to three pieces and a host partial x 512 columns 30, 8192 rows of one piece
//   x 128 columns 25.0; now 4.7, 4.6, 25.5 and 7.1)
struct MergeSplitParams {
  const int32_t* gpu_len;
  // B: plan sequences; ng > 1 for absorbed MLA with H = 16 ng heads, whose
  // plan sequences are (sequence, 16-head group) pairs (ws_plan.h seq_of).
  int B, ng, R, heads, Dv, cap, grid;
  int step;       // the plan's alignment step
  bool f32_pieces;
  bool in_place;  // out_g / lse_g are the outputs: rows of one piece stay as they are
  int add;  // lengths are gpu_len[b] + add (1 when gpu_len is a fused step's len_in)
  const float* out_g;
  const float* lse_g;
  const uint16_t* part_out;  // bf16 pieces (fp32 ones with f32_pieces)
  const float* part_lse;
  const void* b_out;
  const void* b_aux0;
  const void* b_aux1;
  uint16_t* out_bf16;
  float* out_f32;
  float* lse_out;
};

// Waves that share a column group: 1, or more where the rows have many pieces
// on average (n splits over rows plan rows, about n / rows + 1 each) and the
// column groups alone do not fill the chip.  Merge launches alone, captured, us
// with 1 / 2 / 4 / 8 waves (the rule's choice in brackets):
//     16 groups of 64 pieces    9.4   5.9   4.9  [4.5]
//    256 groups of 256         16.0   8.7   6.4  [5.6]
//    256 groups of 32           6.5   4.5   4.0  [4.2]
//    512 groups of 64           5.1   4.3  [4.2]  5.0
//   1024 groups of 64          11.0   8.3  [7.6]  8.8
//   1024 groups of 8            4.0   4.0  [4.8]  6.6
//   2048 groups of 32          [7.6]  7.2   7.8  11.2
//  12288 groups of 2 to 3     [18.9] 36.0  61.6 123
// 1024 groups of 8 equal pieces alone would do with one; ragged batches of that
// average have rows of dozens.
constexpr int kMergeMaxStreams = 8;
static int merge_streams(int n, long long rows, int groups) {
  if (n >= 24 * rows && rows * groups <= 512) return kMergeMaxStreams;
  return n >= 4 * rows && rows * groups <= 1024 ? 4 : 1;
}
// Waves of a merge launch with PS = 1 (32 a CU); further groups are walked.
constexpr long long kMergeWaves = 8192;
constexpr int kMergeWgWaves = 4;

// A thread's place in column group `grp` of a plan row: head h of the row and
// float4 column c of the head (ok: inside the row).
struct MergeCol {
  int h, c;
  bool ok;
};
__device__ __forceinline__ MergeCol merge_col(int grp, int lane, int heads, int Dv4) {
  MergeCol m;
  if (Dv4 <= 64) {  // 64 / Dv4 whole rows
    const int per = 64 / Dv4;
    const int r = lane / Dv4;
    m.h = grp * per + r;
    m.c = lane - r * Dv4;
    m.ok = r < per && m.h < heads;
  } else {
    const int parts = (Dv4 + 63) >> 6;
    m.h = grp / parts;
    m.c = 64 * (grp - m.h * parts) + lane;
    m.ok = m.c < Dv4;
  }
  if (!m.ok) {
    m.h = min(m.h, heads - 1);
    m.c = 0;
  }
  return m;
}
__host__ __device__ inline int merge_groups(int heads, int Dv4) {
  return Dv4 <= 64 ? (heads + 64 / Dv4 - 1) / (64 / Dv4) : heads * ((Dv4 + 63) >> 6);
}

// What stream `st` of PS adds to the row's output: its share of the pieces (VT:
// four columns of one, bf16 or fp32), or (the first stream) the final partial of
// a row that one split held.
template <class VT>
__device__ __forceinline__ PieceAcc merge_stream(const MergeSplitParams& p, const RowSplits& rs,
                                                 size_t krow, int h, int c, int heads, int st,
                                                 int PS) {
  if (rs.nseg > 1) {
    const size_t slot0 = ((size_t)rs.w_first + krow) * heads + h;
    const size_t row = (size_t)(p.Dv >> 2) * sizeof(VT);  // bytes of a piece's row
    return piece_stream<VT>((const char*)p.part_out + slot0 * row + c * sizeof(VT), heads * row,
                            p.part_lse + slot0, heads, st, PS, rs.nseg);
  }
  PieceAcc x = piece_acc_empty();
  if (st == 0) {
    const size_t q = krow * heads + h;
    const float4 v = ((const float4*)(p.out_g + q * p.Dv))[c];
    x.m = p.lse_g[q];
    if (x.m != neg_inf()) {
      x.sum = 1.f;
      x.a = v;
    }
  }
  return x;
}

// The finished row's columns from n accumulators acc(i) and the host partial
// (lb, ob): the output in o and the row's lse.
template <class F>
__device__ __forceinline__ void merge_finish(const F& acc, int n, float lb, const float4& ob,
                                             float4& o, float& lse) {
  float M = lb;
  for (int i = 0; i < n; ++i) M = fmaxf(M, acc(i).m);
  const float wb = piece_weight(lb, M);
  // an empty host side has weight 0 and must not turn its output into NaN
  float4 a = wb > 0.f ? make_float4(wb * ob.x, wb * ob.y, wb * ob.z, wb * ob.w)
                      : make_float4(0.f, 0.f, 0.f, 0.f);
  float L = wb;
  for (int i = 0; i < n; ++i) {
    const PieceAcc x = acc(i);
    const float f = acc_factor(x.m, M);
    L += x.sum * f;
    a.x += x.a.x * f; a.y += x.a.y * f; a.z += x.a.z * f; a.w += x.a.w * f;
  }
  const float inv = L == 0.f ? 0.f : 1.f / L;
  o = make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
  lse = L == 0.f ? neg_inf() : M + __logf(L);
}

template <int FMT, int PS, class VT>
__global__ __launch_bounds__(64 * (PS > kMergeWgWaves ? PS : kMergeWgWaves)) void
merge_split_kernel(const MergeSplitParams p) {
  __shared__ PieceAcc s_acc[PS > 1 ? PS : 1][64];
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const size_t krow = blockIdx.x;
  const int b = uniform(blockIdx.x / p.R);
  const int r = blockIdx.x - b * p.R;
  const int Dv4 = p.Dv >> 2;
  const int groups = merge_groups(p.heads, Dv4);
  const int waves = blockDim.x >> 6;
  int grp = PS > 1 ? blockIdx.y : blockIdx.y * waves + wave;
  if (PS == 1 && grp >= groups) return;
  // The host partial's address depends on nothing the plan computes: its
  // loads go out first, once per column group (of PS waves the first uses them;
  // the operand may be host memory, read over the link).
  MergeCol mc = merge_col(grp, lane, p.heads, Dv4);
  float lb = neg_inf();
  float4 ob = make_float4(0.f, 0.f, 0.f, 0.f);
  auto host = [&]() {
    if (FMT >= 0)
      load_b<(FMT >= 0 ? FMT : 0)>(p.b_out, p.b_aux0, p.b_aux1, (int)(krow * p.heads + mc.h),
                                   p.Dv, mc.c, lb, ob);
  };
  if (PS == 1 || wave == 0) host();
  const RowSplits rs = plan_row(p.gpu_len, p.add, p.cap, p.B, p.R, p.grid, b, r, p.ng, p.step);
  if (p.in_place && rs.nseg <= 1) return;  // out / lse hold the row
  auto store = [&](const float4& o, float lse) {
    if (!mc.ok) return;
    const size_t q = krow * p.heads + mc.h;
    if (p.out_f32) ((float4*)(p.out_f32 + q * p.Dv))[mc.c] = o;
    if (p.out_bf16)
      ((uint2*)(p.out_bf16 + q * p.Dv))[mc.c] =
          make_uint2(pack_bf16x2(o.x, o.y), pack_bf16x2(o.z, o.w));
    if (p.lse_out && mc.c == 0) p.lse_out[q] = lse;
  };
  float4 o;
  float lse;
  if constexpr (PS > 1) {
    s_acc[wave][lane] = merge_stream<VT>(p, rs, krow, mc.h, mc.c, p.heads, wave, PS);
    __syncthreads();
    if (wave != 0) return;
    merge_finish([&](int i) { return s_acc[i][lane]; }, PS, lb, ob, o, lse);
    store(o, lse);
  } else {
    for (;;) {
      const PieceAcc x = merge_stream<VT>(p, rs, krow, mc.h, mc.c, p.heads, 0, 1);
      merge_finish([&](int) { return x; }, 1, lb, ob, o, lse);
      store(o, lse);
      grp += waves * gridDim.y;
      if (grp >= groups) break;
      mc = merge_col(grp, lane, p.heads, Dv4);
      host();
    }
  }
}

// Launches merge_split_kernel<FMT> over rows plan rows.  (fp32 pieces come with
// at least 1024 output rows of 512 columns, mla_layout: 2048 column groups, so
// one wave each.)
template <int FMT>
static void launch_merge(const MergeSplitParams& p, long long rows, hipStream_t s) {
  const int groups = merge_groups(p.heads, p.Dv / 4);
  const int PS = merge_streams(p.grid, rows, groups);
  if (PS == kMergeMaxStreams) {
    hipLaunchKernelGGL((merge_split_kernel<FMT, kMergeMaxStreams, uint2>),
                       dim3((unsigned)rows, groups), dim3(64 * kMergeMaxStreams), 0, s, p);
  } else if (PS == 4) {
    hipLaunchKernelGGL((merge_split_kernel<FMT, 4, uint2>), dim3((unsigned)rows, groups), dim3(256),
                       0, s, p);
  } else {
    // (a grid dimension holds fewer than 2^32 threads: two waves at 2^24 rows)
    const int most = rows * 64 * kMergeWgWaves < (1LL << 32) ? kMergeWgWaves : 2;
    const int waves = std::min(groups, most);
    const long long fit = std::max(kMergeWaves / (rows * waves), 1LL);
    const int wgs = (int)std::min<long long>((groups + waves - 1) / waves, fit);
    const dim3 grid((unsigned)rows, wgs), block(64 * waves);
    if (p.f32_pieces)
      hipLaunchKernelGGL((merge_split_kernel<FMT, 1, float4>), grid, block, 0, s, p);
    else
      hipLaunchKernelGGL((merge_split_kernel<FMT, 1, uint2>), grid, block, 0, s, p);
  }
}

// ---------------------------------------------------------------------------
// Split combine + host merge + the W_UV epilogue of absorbed MLA
// (system/deepseek.py:397-407): the merged latent row of (sequence b, head h)
// is normalised, rounded to bf16 as the reference rounds it before its bmm,
// and projected onto W_UV[h] ([Dout][512] bf16), giving out_v[b][h * Dout + v].
//
// One 256-thread workgroup per (b, h) row: the waves merge its two column groups
// as merge_split_kernel does (the same streams in the same order, so the
// optional latent output is bit-identical to it), two waves a group, into an
// LDS row; then eight lanes per W_UV row read it 128 contiguous bytes at a time
// and reduce by shuffles, 32 rows per pass.  W_UV[h] is shared by the B rows
// of head h through L2.
constexpr int kUvThreads = 256;
constexpr int kUvGroup = 2;  // passes of 32 W_UV rows whose loads are in flight together

template <int FMT, int PS, class VT>
__global__ __launch_bounds__(kUvThreads) void merge_split_uv_kernel(
    const MergeSplitParams p, const uint16_t* __restrict__ w_uv, int Dout,
    uint16_t* __restrict__ out_v) {
  constexpr int Dv = 512;
  constexpr int kGroupWaves = kUvThreads / 128;  // waves of a column group
  __shared__ PieceAcc s_acc[PS > 1 ? PS : 1][Dv / 4];
  __shared__ float s_row[Dv];
  const int qrow = blockIdx.x;  // b * heads + h
  const int t = threadIdx.x;
  const int b = qrow / p.heads;
  const int h = qrow - b * p.heads;
  const int hp = p.heads / p.ng;  // heads of a piece: 16, or all (wide layout)
  const int pv_seq = qrow / hp;   // plan sequence (b, head group) and head in it
  const int h16 = qrow - pv_seq * hp;
  // The W_UV rows of the first kUvGroup passes do not depend on the merge:
  // their loads go out first and land while the plan and the merge run.
  const int lane8 = t & 7;
  const int rsub = t >> 3;  // kUvThreads / 8 rows per pass
  u32x4 wv[kUvGroup][8];
#pragma unroll
  for (int g = 0; g < kUvGroup; ++g) {
    const int v = min(g * (kUvThreads / 8) + rsub, Dout - 1);
    const u32x4* wrow = (const u32x4*)(w_uv + ((size_t)h * Dout + v) * 512);
#pragma unroll
    for (int j = 0; j < 8; ++j) wv[g][j] = wrow[j * 8 + lane8];
  }
  // So do the host partial's.
  const int c = t & (Dv / 4 - 1);    // float4 column
  const int first = uniform(t / (Dv / 4));  // the first stream of this wave
  float lb = neg_inf();
  float4 ob = make_float4(0.f, 0.f, 0.f, 0.f);
  if (FMT >= 0 && first == 0)
    load_b<(FMT >= 0 ? FMT : 0)>(p.b_out, p.b_aux0, p.b_aux1, qrow, Dv, c, lb, ob);
  const RowSplits rs = plan_row(p.gpu_len, p.add, p.cap, p.B, 1, p.grid, pv_seq, 0, p.ng, p.step);
  PieceAcc x;
#pragma unroll
  for (int i = 0; i < PS; i += kGroupWaves)
    if (first + i < PS) {
      x = merge_stream<VT>(p, rs, pv_seq, h16, c, hp, first + i, PS);
      if (PS > 1) s_acc[first + i][c] = x;
    }
  if (PS > 1) __syncthreads();
  float lse = 0.f;
  if (first == 0) {
    float4 o;
    if constexpr (PS > 1)
      merge_finish([&](int i) { return s_acc[i][c]; }, PS, lb, ob, o, lse);
    else
      merge_finish([&](int) { return x; }, 1, lb, ob, o, lse);
    uint2 packed;
    packed.x = pack_bf16x2(o.x, o.y);
    packed.y = pack_bf16x2(o.z, o.w);
    if (p.out_bf16) ((uint2*)(p.out_bf16 + (size_t)qrow * Dv))[c] = packed;
    s_row[4 * c + 0] = bf16_to_f32(packed.x & 0xffffu);
    s_row[4 * c + 1] = bf16_to_f32(packed.x >> 16);
    s_row[4 * c + 2] = bf16_to_f32(packed.y & 0xffffu);
    s_row[4 * c + 3] = bf16_to_f32(packed.y >> 16);
  }
  __syncthreads();
  // (here, where both waves have read the row's lse_g: lse_out may be lse_g)
  if (p.lse_out && t == 0) p.lse_out[qrow] = lse;
  // out_v[b][h * Dout + v] = sum_k s_row[k] * W_UV[h][v][k]: eight lanes per
  // W_UV row, kUvThreads / 8 rows per pass, kUvGroup passes per group of loads
  for (int v0 = 0; v0 < Dout; v0 += kUvGroup * (kUvThreads / 8)) {
    if (v0 > 0) {  // groups after the first load here
#pragma unroll
      for (int g = 0; g < kUvGroup; ++g) {
        const int v = min(v0 + g * (kUvThreads / 8) + rsub, Dout - 1);
        const u32x4* wrow = (const u32x4*)(w_uv + ((size_t)h * Dout + v) * 512);
#pragma unroll
        for (int j = 0; j < 8; ++j) wv[g][j] = wrow[j * 8 + lane8];
      }
    }
#pragma unroll
    for (int g = 0; g < kUvGroup; ++g) {
      const int v = v0 + g * (kUvThreads / 8) + rsub;
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const u32x4 w = wv[g][j];
        const float* r = s_row + 8 * (j * 8 + lane8);
        acc += bf16_to_f32(w.x & 0xffffu) * r[0] + bf16_to_f32(w.x >> 16) * r[1];
        acc += bf16_to_f32(w.y & 0xffffu) * r[2] + bf16_to_f32(w.y >> 16) * r[3];
        acc += bf16_to_f32(w.z & 0xffffu) * r[4] + bf16_to_f32(w.z >> 16) * r[5];
        acc += bf16_to_f32(w.w & 0xffffu) * r[6] + bf16_to_f32(w.w >> 16) * r[7];
      }
      acc += __shfl_xor(acc, 1);
      acc += __shfl_xor(acc, 2);
      acc += __shfl_xor(acc, 4);
      if (lane8 == 0 && v < Dout)
        out_v[(size_t)b * p.heads * Dout + (size_t)h * Dout + v] = f32_to_bf16(acc);
    }
  }
}


// Launches merge_split_uv_kernel<FMT> (the plan rows are p.B: R = 1).
template <int FMT>
static void launch_merge_uv(const MergeSplitParams& p, const uint16_t* w_uv, int Dout,
                            uint16_t* out_v, hipStream_t s) {
  const dim3 grid((unsigned)(p.B / p.ng * p.heads)), block(kUvThreads);
  const int PS = merge_streams(p.grid, p.B, merge_groups(p.heads / p.ng, p.Dv / 4));
  if (PS == kMergeMaxStreams)
    hipLaunchKernelGGL((merge_split_uv_kernel<FMT, kMergeMaxStreams, uint2>), grid, block, 0, s, p,
                       w_uv, Dout, out_v);
  else if (PS == 4)
    hipLaunchKernelGGL((merge_split_uv_kernel<FMT, 4, uint2>), grid, block, 0, s, p, w_uv, Dout,
                       out_v);
  else if (p.f32_pieces)
    hipLaunchKernelGGL((merge_split_uv_kernel<FMT, 1, float4>), grid, block, 0, s, p, w_uv, Dout,
                       out_v);
  else
    hipLaunchKernelGGL((merge_split_uv_kernel<FMT, 1, uint2>), grid, block, 0, s, p, w_uv, Dout,
                       out_v);
}

// Split combine without a host partial (the one-launch entry points).
int merge_split_pieces(const int32_t* len, int len_add, const MlaLayout& lay, int R, int heads,
                       int Dv, int cap, int n, float* out, float* lse, const SplitWorkspace& w,
                       uint16_t* out_bf16, hipStream_t stream) {
  MergeSplitParams prm;
  prm.gpu_len = len;
  prm.B = lay.plan_seqs;
  prm.ng = lay.ng;
  prm.step = lay.step;
  prm.f32_pieces = lay.f32_pieces;
  prm.in_place = out_bf16 == nullptr;
  prm.R = R;
  prm.heads = heads;
  prm.Dv = Dv;
  prm.cap = cap;
  prm.grid = n;
  prm.add = len_add;
  prm.out_g = out;
  prm.lse_g = lse;
  prm.part_out = w.part_out;
  prm.part_lse = w.part_lse;
  prm.b_out = nullptr;
  prm.b_aux0 = nullptr;
  prm.b_aux1 = nullptr;
  prm.out_bf16 = out_bf16;
  prm.out_f32 = out;
  prm.lse_out = lse;
  launch_merge<-1>(prm, (long long)lay.plan_seqs * R, stream);
  return WS_OK;
}

// The host-partial formats: whether a format is known, and whether it needs
// b_aux1 (the triples' sum).
static bool fmt_known(int f) {
  return f == WS_PARTIAL_LSE_F32 || f == WS_TRIPLE_UNNORM_F32 || f == WS_TRIPLE_NORM_BF16 ||
         f == WS_TRIPLE_NORM_F32 || f == WS_PARTIAL_LSE_BF16;
}
static bool fmt_has_sum(int f) { return f != WS_PARTIAL_LSE_F32 && f != WS_PARTIAL_LSE_BF16; }

}  // namespace ws

using namespace ws;

extern "C" int ws_merge_split(const int32_t* gpu_len, int B, int rows_per_seq, int heads,
                              int Dv, int page_capacity, int n_workgroups,
                              const float* out_g, const float* lse_g,
                              const void* workspace, size_t workspace_bytes,
                              const void* b_out, const void* b_aux0, const void* b_aux1,
                              int fmt_b, uint16_t* out_bf16, float* out_f32,
                              float* lse_out, void* stream) {
  if (!gpu_len || !out_g || !lse_g || !workspace)
    return set_error(WS_EINVAL, "ws_merge_split: null input pointer");
  if (!out_bf16 && !out_f32)
    return set_error(WS_EINVAL, "ws_merge_split: no output");
  // an absorbed-MLA step with H = 16 ng heads planned (sequence, head group)
  // pairs, unless its layout is wide (ws_reduce.h mla_layout)
  const bool mla = Dv == 512 && rows_per_seq == 1 && heads > 16 && heads % 16 == 0;
  const MlaLayout lay = mla_layout(B, heads);
  const int ng = mla ? lay.ng : 1;
  // (a step takes at most kMaxSeqs (sequence, 16-head group) pairs in any layout)
  if (B < 0 || (long long)B * (mla ? heads / 16 : 1) > kMaxSeqs || rows_per_seq <= 0 ||
      heads <= 0 || (heads > 16 && !mla) || Dv <= 0 || Dv % 4 || Dv > 512 || page_capacity <= 0 ||
      n_workgroups <= 0)
    return set_error(WS_EINVAL, "ws_merge_split: bad sizes");
  const int Bp = B * ng;      // plan sequences
  heads /= ng;                // heads per plan row
  if (b_out && (!b_aux0 || (fmt_has_sum(fmt_b) && !b_aux1)))
    return set_error(WS_EINVAL, "ws_merge_split: host partial without its lse / max / sum");
  if (b_out && !fmt_known(fmt_b))
    return set_error(WS_EINVAL, "ws_merge_split: unknown format %d", fmt_b);
  if (n_workgroups > kMaxSplits)
    return set_error(WS_EINVAL, "ws_merge_split: %d workgroups exceed %d", n_workgroups,
                     kMaxSplits);
  if (((uintptr_t)workspace & 255u) || ((uintptr_t)out_g | (uintptr_t)out_f32 |
                                         (uintptr_t)b_out) & 15u || ((uintptr_t)out_bf16 & 7u))
    return set_error(WS_EINVAL, "ws_merge_split: misaligned buffer");
  const long long rows_kv = (long long)Bp * rows_per_seq;
  if (rows_kv > (1 << 24))
    return set_error(WS_EINVAL, "ws_merge_split: %lld rows exceed %d", rows_kv, 1 << 24);
  const bool f32_pieces = mla && lay.f32_pieces;
  const size_t need = ws::workspace_bytes((int)rows_kv, heads, Dv, n_workgroups, f32_pieces);
  if (workspace_bytes < need)
    return set_error(WS_EWORKSPACE, "ws_merge_split: workspace %zu < %zu bytes",
                     workspace_bytes, need);
  if (B == 0) return WS_OK;
  const SplitWorkspace w = carve_workspace((void*)workspace, (int)rows_kv, heads, n_workgroups);
  MergeSplitParams prm;
  prm.gpu_len = gpu_len;
  prm.B = Bp;
  prm.ng = ng;
  prm.R = rows_per_seq;
  prm.heads = heads;
  prm.Dv = Dv;
  prm.step = mla ? lay.step : kAlignStep;
  prm.f32_pieces = f32_pieces;
  prm.cap = page_capacity;
  prm.grid = n_workgroups;
  prm.add = 0;
  prm.out_g = out_g;
  prm.lse_g = lse_g;
  prm.part_out = w.part_out;
  prm.part_lse = w.part_lse;
  prm.b_out = b_out;
  prm.b_aux0 = b_aux0;
  prm.b_aux1 = b_aux1;
  prm.out_bf16 = out_bf16;
  prm.out_f32 = out_f32;
  prm.lse_out = lse_out;
  prm.in_place = false;
  hipStream_t s = (hipStream_t)stream;
  if (!b_out) {
    launch_merge<-1>(prm, rows_kv, s);
  } else {
    switch (fmt_b) {
      case WS_PARTIAL_LSE_F32: launch_merge<WS_PARTIAL_LSE_F32>(prm, rows_kv, s); break;
      case WS_TRIPLE_UNNORM_F32: launch_merge<WS_TRIPLE_UNNORM_F32>(prm, rows_kv, s); break;
      case WS_TRIPLE_NORM_BF16: launch_merge<WS_TRIPLE_NORM_BF16>(prm, rows_kv, s); break;
      case WS_PARTIAL_LSE_BF16: launch_merge<WS_PARTIAL_LSE_BF16>(prm, rows_kv, s); break;
      default: launch_merge<WS_TRIPLE_NORM_F32>(prm, rows_kv, s); break;
    }
  }
  return check_launch("ws_merge_split");
}

extern "C" int ws_lse_merge(const float* out_g, const float* lse_g,
                            const void* b_out, const void* b_aux0,
                            const void* b_aux1, int fmt_b, uint16_t* out_bf16,
                            float* out_f32, float* lse_out, int rows, int Dv,
                            void* stream) {
  if (!out_g || !lse_g || !b_out || !b_aux0)
    return set_error(WS_EINVAL, "ws_lse_merge: null input pointer");
  if (!fmt_known(fmt_b))
    return set_error(WS_EINVAL, "ws_lse_merge: unknown format %d", fmt_b);
  if (fmt_has_sum(fmt_b) && !b_aux1)
    return set_error(WS_EINVAL, "ws_lse_merge: triple format needs b_aux1 (sum)");
  if (rows < 0 || Dv <= 0 || Dv % 4 || Dv > 512)
    return set_error(WS_EINVAL, "ws_lse_merge: bad sizes rows=%d Dv=%d", rows, Dv);
  if (((uintptr_t)out_g | (uintptr_t)b_out | (uintptr_t)out_f32) & 15u ||
      ((uintptr_t)out_bf16 & 7u))
    return set_error(WS_EINVAL, "ws_lse_merge: misaligned buffer");
  if (rows == 0) return WS_OK;
  const int threads = ((Dv / 4 + 63) / 64) * 64;
  hipStream_t s = (hipStream_t)stream;
  switch (fmt_b) {
#define WS_MERGE_CASE(F)                                                         \
  case F:                                                                        \
    hipLaunchKernelGGL(lse_merge_kernel<F>, dim3(rows), dim3(threads), 0, s,     \
                       out_g, lse_g, b_out, b_aux0, b_aux1, out_bf16, out_f32,   \
                       lse_out, Dv);                                             \
    break;
    WS_MERGE_CASE(WS_PARTIAL_LSE_F32)
    WS_MERGE_CASE(WS_TRIPLE_UNNORM_F32)
    WS_MERGE_CASE(WS_TRIPLE_NORM_BF16)
    WS_MERGE_CASE(WS_TRIPLE_NORM_F32)
    WS_MERGE_CASE(WS_PARTIAL_LSE_BF16)
#undef WS_MERGE_CASE
    default:
      return set_error(WS_EINVAL, "ws_lse_merge: unknown format %d", fmt_b);
  }
  return check_launch("ws_lse_merge");
}

extern "C" int ws_mla_merge_split_uv(const int32_t* gpu_len, int B, int heads,
                                     int page_capacity, int n_workgroups, const float* out_g,
                                     const float* lse_g, const void* workspace,
                                     size_t workspace_bytes, const void* b_out,
                                     const void* b_aux0, const void* b_aux1, int fmt_b,
                                     const uint16_t* w_uv, int Dout, uint16_t* out_latent,
                                     uint16_t* out_v, float* lse_out, void* stream) {
  constexpr int Dv = 512;
  if (!gpu_len || !out_g || !lse_g || !workspace || !w_uv || !out_v)
    return set_error(WS_EINVAL, "ws_mla_merge_split_uv: null pointer");
  if (B < 0 || heads < 16 || heads % 16 || (long long)B * (heads / 16) > kMaxSeqs ||
      page_capacity <= 0 || n_workgroups <= 0 || Dout <= 0 || Dout % 32 || Dout > 512)
    return set_error(WS_EINVAL, "ws_mla_merge_split_uv: bad sizes B=%d heads=%d Dout=%d", B,
                     heads, Dout);
  const MlaLayout lay = mla_layout(B, heads);
  const int ng = lay.ng;
  const int Bp = lay.plan_seqs;  // plan sequences (sequence, head group)
  if (b_out && (!b_aux0 || (fmt_has_sum(fmt_b) && !b_aux1)))
    return set_error(WS_EINVAL, "ws_mla_merge_split_uv: host partial without its lse / max / sum");
  if (b_out && !fmt_known(fmt_b))
    return set_error(WS_EINVAL, "ws_mla_merge_split_uv: unknown format %d", fmt_b);
  if (n_workgroups > kMaxSplits)
    return set_error(WS_EINVAL, "ws_mla_merge_split_uv: %d workgroups exceed %d", n_workgroups,
                     kMaxSplits);
  if (((uintptr_t)workspace & 255u) || ((uintptr_t)out_g | (uintptr_t)b_out |
                                         (uintptr_t)w_uv) & 15u ||
      ((uintptr_t)out_latent & 7u) || ((uintptr_t)out_v & 1u))
    return set_error(WS_EINVAL, "ws_mla_merge_split_uv: misaligned buffer");
  const size_t need =
      ws::workspace_bytes(Bp, lay.piece_heads, Dv, n_workgroups, lay.f32_pieces);
  if (workspace_bytes < need)
    return set_error(WS_EWORKSPACE, "ws_mla_merge_split_uv: workspace %zu < %zu bytes",
                     workspace_bytes, need);
  if (B == 0) return WS_OK;
  const SplitWorkspace w =
      carve_workspace((void*)workspace, Bp, lay.piece_heads, n_workgroups);
  MergeSplitParams prm;
  prm.gpu_len = gpu_len;
  prm.B = Bp;
  prm.ng = ng;
  prm.R = 1;
  prm.heads = heads;
  prm.Dv = Dv;
  prm.step = lay.step;
  prm.f32_pieces = lay.f32_pieces;
  prm.cap = page_capacity;
  prm.grid = n_workgroups;
  prm.add = 0;
  prm.out_g = out_g;
  prm.lse_g = lse_g;
  prm.part_out = w.part_out;
  prm.part_lse = w.part_lse;
  prm.b_out = b_out;
  prm.b_aux0 = b_aux0;
  prm.b_aux1 = b_aux1;
  prm.out_bf16 = out_latent;
  prm.out_f32 = nullptr;
  prm.lse_out = lse_out;
  prm.in_place = false;
  hipStream_t s = (hipStream_t)stream;
  if (!b_out) {
    launch_merge_uv<-1>(prm, w_uv, Dout, out_v, s);
  } else {
    switch (fmt_b) {
      case WS_PARTIAL_LSE_F32: launch_merge_uv<WS_PARTIAL_LSE_F32>(prm, w_uv, Dout, out_v, s); break;
      case WS_TRIPLE_UNNORM_F32:
        launch_merge_uv<WS_TRIPLE_UNNORM_F32>(prm, w_uv, Dout, out_v, s);
        break;
      case WS_TRIPLE_NORM_BF16:
        launch_merge_uv<WS_TRIPLE_NORM_BF16>(prm, w_uv, Dout, out_v, s);
        break;
      case WS_PARTIAL_LSE_BF16:
        launch_merge_uv<WS_PARTIAL_LSE_BF16>(prm, w_uv, Dout, out_v, s);
        break;
      default: launch_merge_uv<WS_TRIPLE_NORM_F32>(prm, w_uv, Dout, out_v, s); break;
    }
  }
  return check_launch("ws_mla_merge_split_uv");
}
