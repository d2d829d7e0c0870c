// Tile GEMM shared by gemm.hip and gemm_small.hip: launch parameters, the
// direct-to-LDS tile kernel (gemm_bf16_kernel) and the epilogue arithmetic.
// Each source file instantiates the kernel for its own tile configurations.
#pragma once
#include <type_traits>
#include "wam_common.h"

namespace wam {

struct LinearParams {
  const bf16* a; int64_t lda; int M, K;
  int seg_n, n_tiles_per_seg, m_tiles, n_tiles, n_seg_count;
  const void* w[3]; int64_t ldw;      // ldw in elements of the weight dtype
  const bf16* bias[3];
  void* out[3]; int64_t ldo;
  int epi;
  const void* res; int64_t ldr; int res_f32, out_f32;
  wam_modulation gate; int gate_index;
  const float* wscale[3];  // per-output-column fp32 scales of fp8 weights (else unused)
  int mod_d;   // row length of the modulation table (the full output width)
  int n_off;   // column of this launch's first output column in that table
  // Split-K launches: k range kp of k_split writes its raw fp32 sums to
  // part[kp][m][seg * seg_n + n] (row stride part_ld = all segments' columns);
  // a reduce pass adds the ranges in order and applies the epilogue.
  int k_split;
  float* part;
  int part_ld;
  // q/k-norm epilogue (kEpiBiasNorm): per segment, the sums of squares of
  // the bf16 outputs per 256-column group (row stride ssq_ld), the gamma the
  // outputs are multiplied by, and the RoPE table (nfreq, or none).
  float* ssq[3]; const bf16* ngamma[3];
  const float2* nfreq; int nfreq_batch, ntokens, nhd, ssq_ld;
  // fp8 e4m3 activations (the fp8 MFMA mode): A is [M, K] bytes with one
  // fp32 scale per row
  const float* ascale;
  // MX activations: A is e4m3 [M, K] with one e8m0 exponent per row and 32
  // consecutive k (abscale, row stride K / 32 bytes); MX output: out[0] is
  // e4m3 [M, seg_n] (row stride ldo bytes) with one e8m0 exponent per row and
  // 32 consecutive columns (oscale, row stride seg_n / 32 bytes).
  const uint8_t* abscale;
  uint8_t* oscale;
};

// Cost of a launch, and of reducing `bytes` of partial sums in a pass of its
// own or in a row pass that runs anyway, us.
constexpr double kSmallLaunch = 2.6;
inline double split_reduce_us(int64_t bytes, bool fused) { return (fused ? 0.0 : 4.1) + 0.28e-6 * (double)bytes; }
// Tile (an index into the small-grid plan's table) and k ranges of a launch.
struct SplitPlan {
  int tile, ks;
};
SplitPlan split_plan(int M, int seg_n, int n_seg, int K, int wb, int64_t ws_bytes, bool fused = false);
int64_t split_plan_bytes(const SplitPlan& g, int M, int seg_n, int n_seg);
int split_tiles(LinearParams& p, const SplitPlan& g, int wb, hipStream_t s);
int split_reduce(const LinearParams& p, int wb, hipStream_t s);
// A linear whose small-grid plan has several k ranges: `split` is set and the
// partial sums written, the reduction left to the caller (split_reduce,
// split_rms_rope or split_ln on *p).  Otherwise nothing is launched.
int linear_partials(const wam_linear_args* a, hipStream_t s, LinearParams* p, bool* split);
int split_rms_rope(const LinearParams& p, const wam_rms_rope_args& r, const wam_kv_layout_args* kv, hipStream_t s);
// commit (may be null): the new K/V rows' copy to the pool, by workgroups of
// the same launch (the gated residual without fp8 rows).
int split_ln(const LinearParams& p, const wam_ln_args& l, const wam_kv_commit_args* commit, hipStream_t s);
// One launch of the four-wave kernel on tm-row tiles (128 to 256; fp8 weights
// 224 or 256); with p.k_split > 1 its partial sums only.
int w4_tiles(LinearParams& p, int tm, int wb, hipStream_t s);

constexpr int kEpiPartial = 100;   // kernel epilogue of a split-K range: raw fp32 sums
constexpr int kEpiBiasNorm = 101;  // bias, then the q/k-norm epilogue (four-wave kernel; eight-wave without RoPE)

template <int BM_, int BN_, int BK_, int WGM_, int WGN_, int STAGES_, int BLOCKS_ = 1, int SCHED_ = 0,
          int WB_ = 2, int SPLIT_ = 1>
struct GemmCfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WGM = WGM_, WGN = WGN_, STAGES = STAGES_;
  static constexpr int WB = WB_;          // bytes per weight element: 2 (bf16) or 1 (fp8 e4m3)
  static constexpr bool kW4 = false;
  // SPLIT > 1: a stage's loads are issued in SPLIT parts, one at the barrier
  // and the others before the MFMAs of the next k-step's first sub-steps, so
  // the load issue does not stall the waves all at once.  With two stages
  // the later parts have most of a k-step to land before the next barrier.
  static constexpr int SPLIT = SPLIT_;
  static constexpr int BLOCKS = BLOCKS_;  // resident workgroups per CU
  static constexpr int EPI_ROWS = 1 << 30;  // cap on the epilogue's fp32 rows per stage buffer
  static constexpr int SCHED = SCHED_;    // 2: all DS reads of the next k-step, then this
                                          // step's MFMAs; 0: the compiler's order
  static constexpr int kWaves = WGM * WGN;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int WTM = BM / WGM, WTN = BN / WGN;
  static constexpr int TM = WTM / 32, TN = WTN / 32;
  static constexpr int KCH = BK / 8;                     // 16-byte chunks per LDS row
  static constexpr int ROW_BYTES = BK * 2;
  static constexpr int W_ROW_BYTES = BK * WB;
  static constexpr int KCH_W = W_ROW_BYTES / 16;         // 16-byte chunks per LDS weight row
  static constexpr int A_BYTES = BM * ROW_BYTES, B_BYTES = BN * W_ROW_BYTES;
  static constexpr int STAGE = A_BYTES + B_BYTES;
  static constexpr int ROWS_PER_LOAD = 1024 / ROW_BYTES;    // A rows per wave-wide 16 B/lane load
  static constexpr int W_ROWS_PER_LOAD = 1024 / W_ROW_BYTES;
  static constexpr int A_LOADS = BM / ROWS_PER_LOAD, W_LOADS = BN / W_ROWS_PER_LOAD;
  static constexpr int LOADS = A_LOADS + W_LOADS;          // per stage, whole workgroup
  static constexpr int LOADS_PER_WAVE = LOADS / kWaves;
  static_assert(KCH == 8 || KCH == 4, "BK must be 64 or 32");
  static_assert(WB == 2 || (WB == 1 && BK == 64), "fp8 weights use 64-deep k-steps");
  static_assert(A_LOADS % kWaves == 0 && W_LOADS % kWaves == 0 && kWaves % 2 == 0,
                "loads per wave: A then W");
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile");
  static_assert(STAGES >= 2 && BLOCKS * (STAGES * STAGE + (5 - STAGES) * 1024) <= 160 * 1024, "LDS budget");
  static_assert(SPLIT == 1 || (STAGES >= 2 && LOADS_PER_WAVE % SPLIT == 0 && SPLIT - 1 <= BK / 16 - 1),
                "split load issue");
};

// Byte offset of logical 16-byte chunk `c` of LDS row `r`.  The gfx950 LDS
// has 64 banks of 4 bytes (256 bytes per cycle), and a ds_read_b128 serves 16
// lanes per cycle.  An MFMA operand fetch reads 32 consecutive rows at one
// logical chunk, so any 16 consecutive rows must land on 16 distinct 16-byte
// bank slots: rows sharing a 256-byte bank line (2 rows of 128 bytes, 4 of 64)
// are separated by the XOR of the row's index within its bank-line group.
template <int KCH>
__device__ inline int lds_off(int r, int c) {
  if constexpr (KCH == 8) return r * 128 + ((c ^ ((r >> 1) & 7)) << 4);
  else return r * 64 + ((c ^ ((r >> 2) & 3)) << 4);
}

__device__ inline void widen4_bf16(u32x2 t, float out[4]) {
  out[0] = __uint_as_float(t[0] << 16);
  out[1] = __uint_as_float(t[0] & 0xffff0000u);
  out[2] = __uint_as_float(t[1] << 16);
  out[3] = __uint_as_float(t[1] & 0xffff0000u);
}

// 4 consecutive values of a bf16 or fp32 vector in two unconditional 8-byte
// loads (for bf16 the second repeats the first), so that none sits in a
// branch; widen4 makes fp32 values of them.
struct Raw4 {
  u32x2 a, b;
};
__device__ inline Raw4 ld4_raw(const void* p, bool f32, int64_t off) {
  const char* base = static_cast<const char*>(p) + off * (f32 ? 4 : 2);
  return Raw4{*reinterpret_cast<const u32x2*>(base), *reinterpret_cast<const u32x2*>(base + (f32 ? 8 : 0))};
}
__device__ inline void widen4(const Raw4& r, bool f32, float out[4]) {
  float h[4];
  widen4_bf16(r.a, h);
  out[0] = f32 ? __uint_as_float(r.a[0]) : h[0];
  out[1] = f32 ? __uint_as_float(r.a[1]) : h[1];
  out[2] = f32 ? __uint_as_float(r.b[0]) : h[2];
  out[3] = f32 ? __uint_as_float(r.b[1]) : h[3];
}

// The temb part of the gate of token row m, columns n .. n + 3.
__device__ inline Raw4 gate_raw(const LinearParams& p, int m, int n) {
  const int64_t trow = p.gate.temb_len == p.gate.tokens ? m : temb_row(p.gate, m);
  return ld4_raw(p.gate.temb, p.gate.temb_dtype == WAM_F32, temb_off(p.gate, trow, p.gate_index, p.mod_d, n));
}

__device__ inline void ld_mod4(const wam_modulation m, int D, int64_t row, int idx,
                               int d, float out[4]) {
  const int64_t toff = temb_off(m, temb_row(m, row), idx, D, d);
  const int64_t tab = (int64_t)idx * D + d;
  if (m.table_dtype == WAM_F32) {
    float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(m.table) + tab);
    out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
  } else {
    bf16x4 v = *reinterpret_cast<const bf16x4*>(static_cast<const bf16*>(m.table) + tab);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = static_cast<float>(v[e]);
  }
  if (m.temb_dtype == WAM_F32) {
    float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(m.temb) + toff);
    out[0] += v.x; out[1] += v.y; out[2] += v.z; out[3] += v.w;
  } else {
    bf16x4 v = *reinterpret_cast<const bf16x4*>(static_cast<const bf16*>(m.temb) + toff);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] += static_cast<float>(v[e]);
  }
}

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding:
// vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Issue the direct-to-LDS loads of k-tile `kt` into LDS stage `stage`.  Load
// g (0 <= g < LOADS) fills the 1 KB LDS block g, i.e. rows ROWS_PER_LOAD*g ..
// +ROWS_PER_LOAD of the stacked [A rows; W rows] tile.  Wave w issues loads
// g = w + i * kWaves; whether a load reads A or W depends on i only, so the
// unrolled sequence has no branches.  a_lane / b_lane already include the
// swizzle term of the wave's block parity (the wave count is even).
template <class C, int NPARTS = 1>
__device__ __forceinline__ void issue_stage(char* base, i32x4 ra, i32x4 rb, int wave, int a_lane,
                                            int b_lane, int a_pitch, int b_pitch, int kt, int part = 0) {
  const int ko = kt * C::BK * 2, ko_w = kt * C::BK * C::WB;
  constexpr int A_ITERS = C::A_LOADS / C::kWaves;
  constexpr int PER = C::LOADS_PER_WAVE / NPARTS;
#pragma unroll
  for (int ip = 0; ip < PER; ++ip) {
    const int i = part * PER + ip;  // part is a constant wherever the caller is unrolled
    const int g = wave + i * C::kWaves;
    char* dst = base + g * 1024;
    if (i < A_ITERS)
      asm_ld16_lds(ra, dst, a_lane + g * C::ROWS_PER_LOAD * a_pitch + ko);
    else
      asm_ld16_lds(rb, dst, b_lane + (g - C::A_LOADS) * C::W_ROWS_PER_LOAD * b_pitch + ko_w);
  }
}

// MFMA operand fragments of one 16-deep k-step (logical chunk c of each row).
template <class C>
__device__ __forceinline__ void fetch_frags(const char* abase, const char* bbase, int wm, int wn,
                                            int l32, int c, bf16x8 (&fa)[C::TM], bf16x8 (&fb)[C::TN]) {
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
    fa[i] = ld_bf16x8(abase + lds_off<C::KCH>(wm * C::WTM + i * 32 + l32, c));
#pragma unroll
  for (int j = 0; j < C::TN; ++j) {
    const int r = wn * C::WTN + j * 32 + l32;
    if constexpr (C::WB == 2) {
      fb[j] = ld_bf16x8(bbase + lds_off<C::KCH>(r, c));
    } else {
      // 8 fp8 weights (8 bytes: half c & 1 of 16-byte chunk c >> 1 of a
      // 64-byte row), widened exactly to bf16; the per-column scale is
      // applied to the accumulator in the epilogue.
      const u32x2 q = *reinterpret_cast<const u32x2*>(bbase + lds_off<4>(r, c >> 1) + (c & 1) * 8);
      fb[j] = fp8x8_to_bf16x8(q);
    }
  }
}

// The epilogue of 4 consecutive outputs (m, n..n+3) from their fp32 sums v:
// fp8 column scale, bias, then GELU-tanh, or the (gated) residual with an
// fp32 or bf16 output.  The caller loads the residual rv (fp32) of the
// residual epilogues.  With gate_held the gate of these columns is
// gate_pre (every row the caller handles reads the same modulation row);
// otherwise it is read for row m.
template <int EPI, int WB>
__device__ __forceinline__ void epi_apply(const LinearParams& p, void* out, int m, int n, const f32x4 v,
                                          const float (&bv)[4], const float (&wsc)[4],
                                          const float (&gate)[4], const float (&rv)[4]) {
  float y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = WB == 1 ? v[e] * wsc[e] + bv[e] : v[e] + bv[e];
  if constexpr (EPI == WAM_EPI_BIAS_GELU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = gelu_tanh(y[e]);
  } else if constexpr (EPI == WAM_EPI_BIAS_GATE_RES || EPI == WAM_EPI_BIAS_RES) {
    if constexpr (EPI == WAM_EPI_BIAS_GATE_RES) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = rv[e] + y[e] * gate[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = rv[e] + y[e];
    }
    if (p.out_f32) {
      *reinterpret_cast<float4*>(static_cast<float*>(out) + (int64_t)m * p.ldo + n) =
          make_float4(y[0], y[1], y[2], y[3]);
      return;
    }
  }
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16>(y[e]);
  *reinterpret_cast<bf16x4*>(static_cast<bf16*>(out) + (int64_t)m * p.ldo + n) = o;
}

template <class C, int EPI, int RF32 = 0>
__global__ __launch_bounds__(C::kThreads, C::BLOCKS) void gemm_bf16_kernel(LinearParams p) {
  // One __shared__ object per pipeline stage: the compiler tracks the
  // direct-to-LDS loads per object, so reading one stage while another is
  // being filled needs no wait on the outstanding loads.
  __shared__ __attribute__((aligned(1024))) char lds0[C::STAGE];
  __shared__ __attribute__((aligned(1024))) char lds1[C::STAGE];
  __shared__ __attribute__((aligned(1024))) char lds2[C::STAGES > 2 ? C::STAGE : 16];
  __shared__ __attribute__((aligned(1024))) char lds3[C::STAGES > 3 ? C::STAGE : 16];
  __shared__ __attribute__((aligned(1024))) char lds4[C::STAGES > 4 ? C::STAGE : 16];
  static_assert(C::STAGES <= 5, "at most five stage objects");
#define WAM_GEMM_BUF(st) ((st) == 0 ? lds0 : (st) == 1 ? lds1 : (st) == 2 ? lds2 : (st) == 3 ? lds3 : lds4)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WGN, wn = wave % C::WGN;

  // Tile order: XCD-contiguous ranges, then groups of 8 m-tiles swept along n
  // so that one XCD's L2 holds a few A row-panels and W column-panels.
  int tile = xcd_remap(blockIdx.x, gridDim.x);
  int kp = 0;  // k range of a split-K launch: pieces are (k range, tile), tiles fastest
  if constexpr (EPI == kEpiPartial) {
    const int tiles = p.m_tiles * p.n_tiles;
    kp = __builtin_amdgcn_readfirstlane(tile / tiles);
    tile -= kp * tiles;
  }
  constexpr int G = 8;
  const int per_group = G * p.n_tiles;
  const int group = tile / per_group, in_group = tile - group * per_group;
  const int first_m = group * G;
  const int gsize = min(p.m_tiles - first_m, G);
  const int tm = __builtin_amdgcn_readfirstlane(first_m + in_group % gsize);
  const int tn = __builtin_amdgcn_readfirstlane(in_group / gsize);
  const int seg = __builtin_amdgcn_readfirstlane(tn / p.n_tiles_per_seg);
  const int n0 = (tn - seg * p.n_tiles_per_seg) * C::BN;
  const int m0 = tm * C::BM;

  const bf16* A = p.a;
  const char* wseg = static_cast<const char*>(seg == 0 ? p.w[0] : (seg == 1 ? p.w[1] : p.w[2]));
  const char* W = wseg + (int64_t)n0 * p.ldw * C::WB;

  // Direct-to-LDS staging.  Load g (0 <= g < LOADS) of a stage fills the
  // 1 KB LDS block g, i.e. rows ROWS_PER_LOAD*g .. +ROWS_PER_LOAD of the
  // stacked [A rows; W rows] tile; lane L lands at byte 16 L of that block,
  // which is physical chunk L % KCH of row L / KCH, so it fetches the logical
  // chunk that the swizzle maps there.  Rows of A past M fall outside the
  // buffer resource and load as zeros.
  // A split-K range starts kb k-tiles in: both resources start there, and
  // their byte bounds shrink by the same amount.
  int nk = p.K / C::BK, kb = 0;
  if constexpr (EPI == kEpiPartial) {
    kb = (int)((int64_t)kp * nk / p.k_split);
    nk = (int)((int64_t)(kp + 1) * nk / p.k_split) - kb;
  }
  const uint32_t ka = (uint32_t)kb * C::BK * 2u, kw = (uint32_t)kb * C::BK * C::WB;
  const uint32_t a_bytes = (uint32_t)(p.M - m0) * (uint32_t)p.lda * 2u;
  const i32x4 ra = make_rsrc4(A + (int64_t)m0 * p.lda + (int64_t)kb * C::BK, a_bytes - ka);
  // Weight rows past N (a partial last n-tile) load as zeros.
  const int n_rows = min(C::BN, p.seg_n - n0);
  const i32x4 rb = make_rsrc4(W + kw, (uint32_t)((int64_t)n_rows * p.ldw * C::WB) - kw);
  const int lrow = lane / C::KCH, pchunk = lane % C::KCH;
  // The swizzle term of row r = ROWS_PER_LOAD * g + lrow: for 128-byte rows
  // (8 rows per block) it depends on the parity of g, for 64-byte rows (16
  // rows per block) on lrow only.  With an even wave count every block a wave
  // loads has the wave's parity.
  const int r1 = C::ROWS_PER_LOAD + lrow;
  const int chunk0 = C::KCH == 8 ? (pchunk ^ ((lrow >> 1) & 7)) : (pchunk ^ ((lrow >> 2) & 3));
  const int chunk1 = C::KCH == 8 ? (pchunk ^ ((r1 >> 1) & 7)) : (pchunk ^ ((r1 >> 2) & 3));
  const int lchunk = (wave & 1) ? chunk1 : chunk0;
  const int a_lane = (lrow * (int)p.lda + lchunk * 8) * 2;
  const int a_pitch = (int)p.lda * 2, b_pitch = (int)p.ldw * C::WB;
  int b_lane;
  if constexpr (C::WB == 2) {
    b_lane = lrow * b_pitch + lchunk * 16;
  } else {
    // 64-byte weight rows, 16 per block: the swizzle term (r >> 2) & 3 of row
    // r = 16 g + lane / 4 depends on the lane only.
    const int wrow = lane >> 2, wch = (lane & 3) ^ ((wrow >> 2) & 3);
    b_lane = wrow * b_pitch + wch * 16;
  }

  // The epilogue's per-column operands are loaded before the k loop, so that
  // their latency is not at the end of the tile.
  constexpr int RPO_FIT = (C::STAGE / (C::BN * 4)) / 32 * 32;
  constexpr int RPO = RPO_FIT < C::EPI_ROWS ? RPO_FIT : C::EPI_ROWS;  // fp32 rows per buffer
  static_assert(RPO >= 32, "a stage buffer must hold 32 fp32 rows of the tile");
  constexpr int ROUND = RPO * C::STAGES < C::BM ? RPO * C::STAGES : C::BM;  // rows staged per round
  constexpr int NROUNDS = (C::BM + ROUND - 1) / ROUND;
  constexpr int QPR = C::BN / 4;                         // 16-byte chunks per fp32 row
  constexpr int RPI = 64 / QPR;                          // rows per wave-wide access
  static_assert(QPR == 64 || QPR == 32 || QPR == 16, "BN must be 256, 128 or 64");
  constexpr int ROW_B = C::BN * 4;
  void* out = seg == 0 ? p.out[0] : (seg == 1 ? p.out[1] : p.out[2]);
  const bf16* __restrict__ bias = seg == 0 ? p.bias[0] : (seg == 1 ? p.bias[1] : p.bias[2]);
  const int q = lane % QPR;  // this lane's chunk of a row in the read phase
  const int n = n0 + 4 * q;
  const bool n_ok = n < p.seg_n;  // N is a multiple of 4: a lane's 4 columns are all in or all out
  float bv[4] = {0.f, 0.f, 0.f, 0.f};
  if (bias && n_ok) {
    const bf16x4 t = *reinterpret_cast<const bf16x4*>(bias + n);
#pragma unroll
    for (int e = 0; e < 4; ++e) bv[e] = static_cast<float>(t[e]);
  }
  float wsc[4] = {1.f, 1.f, 1.f, 1.f};
  if constexpr (C::WB == 1) {
    const float* ws = seg == 0 ? p.wscale[0] : (seg == 1 ? p.wscale[1] : p.wscale[2]);
    const float4 t = n_ok ? *reinterpret_cast<const float4*>(ws + n) : make_float4(1.f, 1.f, 1.f, 1.f);
    wsc[0] = t.x; wsc[1] = t.y; wsc[2] = t.z; wsc[3] = t.w;
  }
  f32x16 acc[C::TN][C::TM];
#pragma unroll
  for (int j = 0; j < C::TN; ++j)
#pragma unroll
    for (int i = 0; i < C::TM; ++i) acc[j][i] = f32x16{};

  const int half = lane >> 5, l32 = lane & 31;
  constexpr int KSTEPS = C::BK / 16;
  constexpr int MF = C::TM * C::TN, R = C::TM + C::TN;
  static_assert(KSTEPS % 2 == 0, "fragment double buffer alternates per k-step");

  // Prologue: all STAGES buffers in flight, wait for the first.
#pragma unroll
  for (int st = 0; st < C::STAGES; ++st)
    if (st < nk) issue_stage<C>(WAM_GEMM_BUF(st), ra, rb, wave, a_lane, b_lane, a_pitch, b_pitch, st);
  if (nk >= C::STAGES) wait_vmcnt<(C::STAGES - 1) * C::LOADS_PER_WAVE>();
  else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();

  bf16x8 fa[2][C::TM], fb[2][C::TN];
  fetch_frags<C>(lds0, lds0 + C::A_BYTES, wm, wn, l32, half, fa[0], fb[0]);

  // The k loop is unrolled by STAGES so that every buffer reference is to a
  // fixed __shared__ object.
  for (int kt0 = 0; kt0 < nk; kt0 += C::STAGES) {
#pragma unroll
    for (int st = 0; st < C::STAGES; ++st) {
      const int kt = kt0 + st;
      if (kt >= nk) break;
      const char* abase = WAM_GEMM_BUF(st);
      const char* bbase = abase + C::A_BYTES;
      // k-steps 0 .. KSTEPS-2: read the next step's fragments, then this
      // step's MFMAs.
#pragma unroll
      for (int ks = 0; ks + 1 < KSTEPS; ++ks) {
        if constexpr (C::SPLIT > 1) {
          // the remaining parts of the loads issued at the previous barrier
          // (tile kt - 1 + STAGES into the previous stage's buffer)
          if (ks + 1 < C::SPLIT && kt >= 1 && kt - 1 + C::STAGES < nk)
            issue_stage<C, C::SPLIT>(WAM_GEMM_BUF((st + C::STAGES - 1) % C::STAGES), ra, rb, wave, a_lane,
                                     b_lane, a_pitch, b_pitch, kt - 1 + C::STAGES, ks + 1);
        }
        fetch_frags<C>(abase, bbase, wm, wn, l32, (ks + 1) * 2 + half, fa[(ks + 1) & 1], fb[(ks + 1) & 1]);
#pragma unroll
        for (int j = 0; j < C::TN; ++j)
#pragma unroll
          for (int i = 0; i < C::TM; ++i)
            acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][j], fa[ks & 1][i], acc[j][i],
                                                                0, 0, 0);
        if constexpr (C::SCHED == 2) {
          __builtin_amdgcn_sched_group_barrier(0x100, R, 0);   // all DS reads of step ks+1
          __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);  // then the MFMAs of step ks
        }
      }
      // Every LDS read of this stage is done (the last step's fragments are
      // in registers), so the barrier goes here: the next stage's data is
      // then visible, this stage's buffer can be refilled, and the next
      // stage's first reads overlap this stage's last MFMAs.
      if (kt + 1 < nk) {
        if (kt + C::STAGES - 1 < nk) wait_vmcnt<(C::STAGES - 2) * C::LOADS_PER_WAVE>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_s_barrier();
        if (kt + C::STAGES < nk)
          issue_stage<C, C::SPLIT>(WAM_GEMM_BUF(st), ra, rb, wave, a_lane, b_lane, a_pitch, b_pitch,
                                   kt + C::STAGES, 0);
        const char* na = WAM_GEMM_BUF((st + 1) % C::STAGES);
        fetch_frags<C>(na, na + C::A_BYTES, wm, wn, l32, half, fa[0], fb[0]);
      }
      constexpr int LAST = (KSTEPS - 1) & 1;
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
          acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[LAST][j], fa[LAST][i], acc[j][i], 0, 0, 0);
    }
  }

  // Epilogue, staged through LDS.  The accumulators are in MFMA layout (a
  // lane holds one row and 4 columns per fragment), which would make every
  // global store and residual read touch 32 rows at 16 bytes each.  Instead
  // the fp32 tile goes to the (now idle) stage buffers, RPO rows per buffer,
  // and is read back row-wise: a wave covers whole rows, so bias, modulation,
  // residual and output accesses are contiguous and fill whole cache lines.
  // Rows are 16-byte chunks XOR-swizzled by (row & 15), which keeps both the
  // column-wise writes and the row-wise reads free of bank conflicts.
  // The residual of a round's rows is loaded into registers before the round
  // is staged through LDS (16 bytes per row chunk: 4 fp32, or 4 bf16 in the
  // low half), so the whole round's loads are in flight together.
  constexpr bool RES = EPI == WAM_EPI_BIAS_GATE_RES || EPI == WAM_EPI_BIAS_RES;
  constexpr int ITERS = ROUND / (C::kWaves * RPI);
  constexpr int RB = RF32 ? 4 : 2;  // residual bytes per element
  typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));
  typedef unsigned int u32x2v __attribute__((ext_vector_type(2)));
  // The residual through a buffer resource over the tile's rows from column
  // n0 (rows past M read zeros), so the prefetch has no branch: a load inside
  // a branch, or a dtype chosen at run time, left the compiler waiting for
  // all memory operations (the previous rows' stores included) before every
  // row of the epilogue.
  const int rows_left = min(p.M - m0, C::BM);
  const __amdgpu_buffer_rsrc_t rres =
      RES ? make_rsrc(static_cast<const char*>(p.res) + ((int64_t)m0 * p.ldr + n0) * RB,
                      (uint32_t)((rows_left - 1) * (uint32_t)p.ldr + (uint32_t)min(C::BN, p.seg_n - n0)) * RB)
          : make_rsrc(p.a, 0u);
  std::conditional_t<RF32 != 0, u32x4v, u32x2v> rraw[RES ? ITERS : 1];
  auto res_prefetch = [&](int rd) {
    if constexpr (RES) {
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int row = rd * ROUND + (it * C::kWaves + wave) * RPI + lane / QPR;
        const int off = (row * (int)p.ldr + 4 * q) * RB;
        if constexpr (RF32)
          rraw[it] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(rres, off, 0, 0));
        else
          rraw[it] = __builtin_bit_cast(u32x2v, __builtin_amdgcn_raw_buffer_load_b64(rres, off, 0, 0));
      }
    }
  };
  res_prefetch(0);
  // The gate of this lane's 4 columns, loaded once per tile (after the k
  // loop, which has no registers to spare for it) when the tile's rows read
  // at most two consecutive modulation rows (one or two samples, or latent
  // frames): gate for the rows before gate_split, gate2 from there on.  Rows
  // that read more (one modulation row per token) load theirs per row, those
  // of kGateBatch iterations together (a row at a time each was a memory round
  // trip: 2325 x 3072 x 3072, one modulation row per token, 70 -> 64 us; the
  // four-wave kernel's fp8 2325 x 14336 x 3072 134 -> 120).
  float gate[4] = {0.f, 0.f, 0.f, 0.f}, gate2[4] = {0.f, 0.f, 0.f, 0.f};
  constexpr int kGateBatch = 4;
  Raw4 gtab{};
  bool gate_held = false;
  int gate_split = 0;  // first tile row served by the second modulation row
  if constexpr (EPI == WAM_EPI_BIAS_GATE_RES) {
    const int m_last = min(m0 + C::BM, p.M) - 1;
    const int64_t tr0 = temb_row(p.gate, m0), tr1 = temb_row(p.gate, m_last);
    gate_held = tr1 - tr0 <= 1;
    gate_split = (int)(temb_first_row(p.gate, tr1) - m0);
    // columns clamped into the row: both loads unconditional, in flight with
    // the residual's
    const int nc = min(n, p.seg_n - 4) + p.n_off;
    ld_mod4(p.gate, p.mod_d, m0, p.gate_index, nc, gate);
    ld_mod4(p.gate, p.mod_d, m_last, p.gate_index, nc, gate2);
    gtab = ld4_raw(p.gate.table, p.gate.table_dtype == WAM_F32, (int64_t)p.gate_index * p.mod_d + nc);
  }
  // q-norm epilogue (no RoPE here): the gamma of the lane's 4 columns and the
  // segment's sums-of-squares array.  With 256-column tiles a wave holds one
  // whole row of the tile per pass, so a row's sum is one wave reduction.
  constexpr bool NORM = EPI == kEpiBiasNorm;
  static_assert(!NORM || C::BN == 256, "the q-norm epilogue needs 256-column tiles");
  float gm[4] = {1.f, 1.f, 1.f, 1.f};
  float* nssq = nullptr;
  if constexpr (NORM) {
    nssq = seg == 0 ? p.ssq[0] : (seg == 1 ? p.ssq[1] : p.ssq[2]);
    const bf16* g = seg == 0 ? p.ngamma[0] : (seg == 1 ? p.ngamma[1] : p.ngamma[2]);
    const bf16x4 tg = *reinterpret_cast<const bf16x4*>(g + min(n, p.seg_n - 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) gm[e] = static_cast<float>(tg[e]);
  }
  // Every wave is done reading the last stage (its fragments are in
  // registers and consumed); only LDS operations are waited for, so the
  // residual loads stay in flight.
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int rd = 0; rd < NROUNDS; ++rd) {
#pragma unroll
    for (int i = 0; i < C::TM; ++i) {
      const int r = wm * C::WTM + i * 32;  // first tile row of this fragment row (uniform)
      if (r / ROUND != rd) continue;
      const int obj = (r % ROUND) / RPO;
      char* buf = WAM_GEMM_BUF(obj);
      const int lr = r % RPO + l32;
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int qq = (wn * C::WTN + j * 32 + 8 * g) / 4 + half;
          const f32x4 v = {acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]};
          *reinterpret_cast<f32x4*>(buf + lr * ROW_B + ((qq ^ (lr & 15)) << 4)) = v;
        }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's LDS writes are done
    __builtin_amdgcn_s_barrier();
    // the round's residual rows have landed (one wait per round, which also
    // drains the previous round's stores)
    if constexpr (RES) wait_vmcnt<0>();
    Raw4 graw[kGateBatch];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int rr = (it * C::kWaves + wave) * RPI + lane / QPR;  // row within the round
      const int row = rd * ROUND + rr;
      const int m = m0 + row;
      if constexpr (EPI == WAM_EPI_BIAS_GATE_RES) {
        if (it % kGateBatch == 0 && !gate_held) {
#pragma unroll
          for (int k = 0; k < kGateBatch; ++k)
            graw[k] = gate_raw(p, min(m + k * C::kWaves * RPI, p.M - 1), min(n, p.seg_n - 4) + p.n_off);
        }
      }
      if constexpr (NORM) {
        // y = bf16(acc + b) as the bias epilogue rounds it; the row's sum of
        // y^2 over the tile's 256 columns (every lane of the wave takes part
        // in the reduction); the stored value bf16(y * gamma), one rounding.
        const bool row_ok = row < C::BM && m < p.M;
        const int lrr = rr % RPO;
        const f32x4 v = *reinterpret_cast<const f32x4*>(WAM_GEMM_BUF(rr / RPO) + lrr * ROW_B + ((q ^ (lrr & 15)) << 4));
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16>(v[e] + bv[e]);
        const bf16x2 o01 = {o[0], o[1]}, o23 = {o[2], o[3]};
        const float ss = __builtin_amdgcn_fdot2_f32_bf16(o23, o23, __builtin_amdgcn_fdot2_f32_bf16(o01, o01, 0.f, false),
                                                         false);
        const float tot = wave_sum(row_ok && n_ok ? ss : 0.f);
        if (row_ok && lane == 0) nssq[(int64_t)m * p.ssq_ld + (n0 >> 8)] = tot;
        if (row_ok && n_ok) {
          bf16x4 t;
#pragma unroll
          for (int e = 0; e < 4; ++e) t[e] = static_cast<bf16>(static_cast<float>(o[e]) * gm[e]);
          *reinterpret_cast<bf16x4*>(static_cast<bf16*>(out) + (int64_t)m * p.ldo + n) = t;
        }
        continue;
      }
      if (row >= C::BM || m >= p.M || !n_ok) continue;
      const int obj = rr / RPO, lr = rr % RPO;
      const char* buf = WAM_GEMM_BUF(obj);
      const f32x4 v = *reinterpret_cast<const f32x4*>(buf + lr * ROW_B + ((q ^ (lr & 15)) << 4));
      if constexpr (EPI == kEpiPartial) {
        *reinterpret_cast<f32x4*>(p.part + ((int64_t)kp * p.M + m) * p.part_ld + seg * p.seg_n + n) = v;
      } else {
        float rv[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (RES) {
          const auto t = rraw[it];
          if constexpr (RF32) {
#pragma unroll
            for (int e = 0; e < 4; ++e) rv[e] = __uint_as_float(t[e]);  // by value: a vector element has no address
          } else {
            rv[0] = __uint_as_float(t[0] << 16);
            rv[1] = __uint_as_float(t[0] & 0xffff0000u);
            rv[2] = __uint_as_float(t[1] << 16);
            rv[3] = __uint_as_float(t[1] & 0xffff0000u);
          }
        }
        float gsel[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) gsel[e] = row >= gate_split ? gate2[e] : gate[e];
        if constexpr (EPI == WAM_EPI_BIAS_GATE_RES) {
          if (!gate_held) {
            float gb[4];
            widen4(gtab, p.gate.table_dtype == WAM_F32, gsel);
            widen4(graw[it % kGateBatch], p.gate.temb_dtype == WAM_F32, gb);
#pragma unroll
            for (int e = 0; e < 4; ++e) gsel[e] += gb[e];
          }
        }
        epi_apply<EPI, C::WB>(p, out, m, n, v, bv, wsc, gsel, rv);
      }
    }
    if (rd + 1 < NROUNDS) {
      res_prefetch(rd + 1);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // this round's LDS reads are done
      __builtin_amdgcn_s_barrier();
    }
  }
#undef WAM_GEMM_BUF
}

// ------------------------------------------------ partial sums of a split
// Sums of the k_split partial ranges at byte offsets off[c] of a plane, in
// range order.  Up to R ranges of every chunk are in flight together: read one
// chunk and four ranges at a time they were up to nine memory round trips in a
// row, and the row passes took 9 to 12 us in a block instead of 7.5 to 8.6.
// A place past the last range reads zeros beyond the resource's bound (a
// workspace of partial sums is smaller than 2 GiB).
template <int R, int NCH>
__device__ inline void add_ranges(const LinearParams& p, int r0, const int (&off)[NCH], f32x4 (&v)[NCH]) {
  const uint32_t plane = (uint32_t)p.M * (uint32_t)p.part_ld * 4u;
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.part, plane * (uint32_t)p.k_split);
  f32x4 t[NCH][R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t base = r0 + r < p.k_split ? (uint32_t)(r0 + r) * plane : 0x80000000u;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      t[c][r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(base + (uint32_t)off[c]), 0, 0));
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < NCH; ++c) v[c] += t[c][r];
}

template <int NCH>
__device__ inline void sum_ranges(const LinearParams& p, const int (&off)[NCH], f32x4 (&v)[NCH]) {
#pragma unroll
  for (int c = 0; c < NCH; ++c) v[c] = f32x4{};
  if (p.k_split <= 4) return add_ranges<4, NCH>(p, 0, off, v);
  for (int r0 = 0; r0 < p.k_split; r0 += 8) add_ranges<8, NCH>(p, r0, off, v);
}

}  // namespace wam
