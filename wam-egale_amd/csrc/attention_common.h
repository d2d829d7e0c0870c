// Shared by the attention kernels: LDS tile layouts, row clamping and the
// per-query RMS factor.
#pragma once
#include "wam_common.h"

namespace wam {

constexpr int kAttnHD = 128;
constexpr int kAttnKT = 64;                          // keys per LDS stage
constexpr int kAttnTile = kAttnKT * kAttnHD * 2;     // 16 KB per K or V tile
constexpr int kAttnStage = 2 * kAttnTile;            // K tile + V tile
constexpr int kAttnStages = 3;

// LDS layouts (64 banks x 4 bytes; 256-byte rows = one bank line).
// K [64 keys][128 d]: an S^T operand fetch reads 16 consecutive keys at one
// 16-byte chunk per cycle, so chunk XOR (key mod 16).
__device__ inline int k_off(int key, int c) { return key * 256 + ((c ^ (key & 15)) << 4); }
// V [64 keys][128 d] in natural layout: a transposed read fetches 4
// consecutive keys x 64 bytes per 32 lanes, so the 64-byte segment XOR
// (key mod 4).
__device__ inline int v_off(int key, int c) { return key * 256 + ((c ^ ((key & 3) << 2)) << 4); }

__device__ inline int clamp_row(int r, int n) { return r < 0 ? 0 : (r >= n ? n - 1 : r); }

// Per-query RMS factor of queries written by wam_linear's norm epilogue:
// rsqrt(sum of the row's q_ssq_n partial sums of squares / q_norm_dim + eps)
// for query row b * Mq + qi (clamped into range).  The RMSNorm across heads
// is model.py:609-612; the rotation after it is linear and commutes.  The
// pipelined kernel stages the partial sums through LDS instead (see there).
constexpr int kQssqMax = 16;
__device__ inline float q_rms_factor(const wam_attention_args& a, int b, int qi) {
  const float* p = a.q_ssq + ((int64_t)b * a.Mq + min(qi, a.Mq - 1)) * a.q_ssq_n;
  float s = 0.f;
  for (int t = 0; t < a.q_ssq_n; ++t) s += p[t];
  return rsqrtf(s / (float)a.q_norm_dim + a.q_eps);
}

constexpr int kFewGroupMax = 8;  // batch rows per group of attention_few_kernel
// The kernel for calls with few queries per key source: query waves per
// workgroup (1, 2 or 4 of 32 queries; 0: not this kernel), batch rows per
// group and key-tile ranges (each a workgroup of its own, merged by a second
// pass), and its predicted time in us.
struct FewPlan {
  int qw, group, ranges;
  double cost;
};
// `sharing`: batch rows per pool row (1 without a row map or history).
FewPlan attention_few_plan(int B, int Mq, int H, int64_t keys, int sharing, int64_t max_bytes);
int64_t attention_few_bytes(const FewPlan& p, int B, int Mq, int H);
int attention_few(const wam_attention_args* a, const FewPlan& p, float* part, hipStream_t s);

}  // namespace wam
