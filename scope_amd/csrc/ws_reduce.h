// Split pieces shared by the decode kernels and the merges.
//
// A decode call cuts every row's blocks between its splits (ws_plan.h).  A
// split that holds a whole row writes the row's final partial (out
// normalised fp32, lse natural log) straight to the caller's out / lse; a
// row spread over several splits leaves one piece per split in the
// workspace, and a later launch on the same stream (merge_split_kernel,
// merge_split_uv_kernel) rebuilds the plan to find and LSE-combine them.
//
// Workspace layout (ws_decode_plan), for a call over rows_kv rows of `heads`
// output rows each, run by n splits:
//   [slot lse f32 x (n + rows_kv) x heads, padded to 256 B]
//   [slot out bf16 (some wide MLA calls: fp32, mla_layout) x (n + rows_kv) x heads x Dv]
// (slot = split + row, ws_plan.h).  Pieces are normalised and rounded to
// bf16 (their weights stay fp32): a 32-token block carries 36 KB of latent
// and an MLA piece 16 x 512 outputs, so at 256 splits fp32 pieces cost
// 8 MB of writes and reads per call.  Every call writes the slots it reads
// back, so the workspace needs no initial contents.
#pragma once

#include "ws_common.h"
#include "ws_plan.h"

namespace ws {

__host__ __device__ inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

struct SplitWorkspace {
  float* part_lse;
  uint16_t* part_out;  // bf16 (f32_pieces calls: the fp32 values' address)
};

__host__ __device__ inline size_t workspace_bytes(int rows_kv, int heads, int Dv, int n,
                                                  bool f32_pieces = false) {
  const size_t slots = (size_t)n + rows_kv;
  return align256(slots * heads * 4) + slots * heads * Dv * (f32_pieces ? 4 : 2);
}

__host__ __device__ inline SplitWorkspace carve_workspace(void* base, int rows_kv,
                                                          int heads, int n) {
  SplitWorkspace w;
  char* p = (char*)base;
  const size_t slots = (size_t)n + rows_kv;
  w.part_lse = (float*)p;
  p += align256(slots * heads * 4);
  w.part_out = (uint16_t*)p;
  return w;
}

// Layout of an absorbed-MLA call with B sequences of H heads (H a multiple
// of 16).  The wide kernel (ws_mla_wide.h) reads a latent block once for up to
// 128 heads; its plan sequences are the sequences and a piece holds all H
// heads.  Other calls plan (sequence, 16-head group) pairs with 16-head pieces
// and read a block once per group.  The step, the merges and the workspace
// query of a call all take their layout from here, so they agree.
//
// 128 heads always run wide.  Fewer do from B * H = 1024 on: the wide kernel has
// a longer start and end per sequence, the group layout reads every block H / 16
// times.  Captured steps with their merge, equal lengths, us, group -> wide:
//   B  32 x H 32   64 tokens 11.5 -> 15.6   1001 25.5 -> 29.1   4096 59.0 -> 45.6
//   B  16 x H 64   64 tokens 11.9 -> 15.8   1001 23.1 -> 27.2  16384 142 -> 83
//   B 128 x H 32   64 tokens 17.5 -> 20.5   1001 60.3 -> 48.1
//   B  64 x H 96   64 tokens 26.9 -> 20.3   1001 92.6 -> 47.7
//   B 512 x H 32   64 tokens 46.7 -> 38.8   1001  226 -> 149
// so short contexts lose 3 to 5 us near the line and longer ones gain up to half.
// The line is on rows alone because the merges, which must agree, know no bound
// on the lengths.  Below it: B 8 x H 64 of 2048 tokens 23.2 -> 26.3.
//
// The group layout holds more of these calls' rows whole (fp32), having H / 16
// times the plan sequences; the wide one cuts nearly every row over workgroups.
// A bf16 piece rounds its outputs once more, which would show in the error
// against 64 bits (B 128 x H 32 of 2048 tokens: 0.00133 -> 0.00200 of the output's
// norm), so these calls leave fp32 pieces.  128 heads over at most 64 sequences
// cut nearly every row in either layout and keep bf16 ones.
constexpr int kWideHeads = 128;    // heads of the wide kernel's four waves
constexpr int kWideMinHeads = 32;
constexpr int kWideMinRows = 1024;  // B * H from which fewer than 128 heads run it
constexpr int kWideBf16Seqs = 64;  // sequences up to which 128 heads leave bf16 pieces
// (a call takes B * H / 16 <= kMaxSeqs)
constexpr int kWideMaxSeqs = 16 * kMaxSeqs / kWideMinHeads;
struct MlaLayout {
  bool wide;
  int ng;           // plan sequences per sequence
  int piece_heads;  // heads of one piece
  int plan_seqs;    // B * ng
  int step;         // the plan's alignment step (ws_plan.h)
  bool f32_pieces;  // fp32 pieces instead of bf16 ones
};
__host__ __device__ inline MlaLayout mla_layout(int B, int H) {
  MlaLayout l;
  l.wide = H == kWideHeads ||
           (H >= kWideMinHeads && H < kWideHeads && (long long)B * H >= kWideMinRows);
  l.ng = l.wide ? 1 : H / 16;
  l.piece_heads = l.wide ? H : 16;
  l.plan_seqs = B * l.ng;
  l.step = l.wide ? kAlignStepWide : kAlignStep;
  l.f32_pieces = l.wide && (H < kWideHeads || B > kWideBf16Seqs);
  return l;
}

// Workgroups of a decode call: n_workgroups, or the library's choice (0):
// `per_cu` resident workgroups on every CU of the current device, but no more
// than the call's 32-token blocks can feed with `min_blocks` each.
int choose_workgroups(int n_workgroups, int per_cu, long long max_blocks, int min_blocks);
// Workgroups of an MLA call (ws_mla.hip).
int mla_workgroups(int n_workgroups, int B, int max_len);
// Combines the pieces of a split decode step with no host partial: rows held
// by several splits are LSE-combined from the workspace into out / lse, which
// already hold the others; out_bf16, when not null, receives every row's output
// in bf16.  lay gives the plan (B plan sequences of R rows; for absorbed MLA
// the layout's); lengths are len[b] + len_add.  Launches on `stream`; returns
// WS_OK or an error code (ws_merge.hip).
int merge_split_pieces(const int32_t* len, int len_add, const MlaLayout& lay, int R, int heads,
                       int Dv, int cap, int n, float* out, float* lse, const SplitWorkspace& w,
                       uint16_t* out_bf16, hipStream_t stream);

// Eight outputs of a piece, rounded to bf16, as one 16-byte store.
__device__ __forceinline__ void store_piece8(uint16_t* dst, float a0, float a1, float a2,
                                             float a3, float a4, float a5, float a6,
                                             float a7) {
  u32x4 v;
  v[0] = pack_bf16x2(a0, a1);
  v[1] = pack_bf16x2(a2, a3);
  v[2] = pack_bf16x2(a4, a5);
  v[3] = pack_bf16x2(a6, a7);
  *(u32x4*)dst = v;
}

// Four bf16 piece outputs (8 bytes) as floats.
__device__ __forceinline__ float4 piece4_f32(uint2 v) {
  return make_float4(__builtin_bit_cast(float, v.x << 16),
                     __builtin_bit_cast(float, v.x & 0xffff0000u),
                     __builtin_bit_cast(float, v.y << 16),
                     __builtin_bit_cast(float, v.y & 0xffff0000u));
}

// Running LSE combine of part of a row's pieces in one thread's four columns:
// sum and a are relative to m.
struct PieceAcc {
  float m, sum;
  float4 a;
};
__device__ __forceinline__ PieceAcc piece_acc_empty() {
  return PieceAcc{neg_inf(), 0.f, make_float4(0.f, 0.f, 0.f, 0.f)};
}

// exp(x - m): 0 for x = -inf (no weight) also where m is -inf, NaN for a NaN x.
__device__ __forceinline__ float piece_weight(float x, float m) {
  return x == neg_inf() ? 0.f : __expf(x - m);
}
// Factor that takes an accumulator from reference m to M >= m (an empty one, m
// = -inf, holds only zeros, or the NaN of a bad piece, which stays).
__device__ __forceinline__ float acc_factor(float m, float M) {
  return m == neg_inf() ? 1.f : __expf(m - M);
}

// Four columns of a piece as loaded: VT is uint2 (bf16) or float4 (fp32).
__device__ __forceinline__ float4 piece4_f32(float4 v) { return v; }

// Adds the pieces s, s + step, ... (U of them, those below n; piece s's columns
// at pieces + s * stride bytes) to an accumulator: all U lse values and columns
// are requested before the first is used (past n the last piece again, a cache
// hit).
template <int U, class VT>
__device__ __forceinline__ void piece_batch(PieceAcc& x, const char* pieces, size_t stride,
                                            const float* lse, int lstride, int s, int step,
                                            int n) {
  float l[U];
  VT v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) l[u] = lse[(size_t)min(s + u * step, n - 1) * lstride];
#pragma unroll
  for (int u = 0; u < U; ++u)
    v[u] = *(const VT*)(pieces + (size_t)min(s + u * step, n - 1) * stride);
  float m = x.m;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (s + u * step >= n) l[u] = neg_inf();
    m = fmaxf(m, l[u]);
  }
  const float f = acc_factor(x.m, m);
  x.m = m;
  x.sum *= f;
  x.a.x *= f; x.a.y *= f; x.a.z *= f; x.a.w *= f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (s + u * step >= n) continue;
    const float w = piece_weight(l[u], m);
    const float4 o = piece4_f32(v[u]);
    x.sum += w;
    x.a.x += w * o.x; x.a.y += w * o.y; x.a.z += w * o.z; x.a.w += w * o.w;
  }
}

// The pieces first, first + step, ... of a row's n.
template <class VT>
__device__ __forceinline__ PieceAcc piece_stream(const char* pieces, size_t stride,
                                                 const float* lse, int lstride, int first,
                                                 int step, int n) {
  PieceAcc x = piece_acc_empty();
  int s = first;
  for (; s + 8 * step < n; s += 16 * step)
    piece_batch<16, VT>(x, pieces, stride, lse, lstride, s, step, n);
  if (s + 4 * step < n)
    piece_batch<8, VT>(x, pieces, stride, lse, lstride, s, step, n);
  else if (s < n)
    piece_batch<4, VT>(x, pieces, stride, lse, lstride, s, step, n);
  return x;
}

}  // namespace ws
