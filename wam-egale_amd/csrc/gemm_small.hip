// GEMMs whose 256x256 tiles would leave most of the chip idle: few rows (the
// action tokens of a policy step, a text context) or few columns.  The plan
// picks a tile and a number of k ranges so that one round of workgroups
// covers the CUs; with several ranges the tiles write fp32 partial sums and a
// reduce pass adds them in range order and applies the epilogue, alone or
// together with the row pass that follows the projection in the block
// (RMSNorm + RoPE, or the residual stream and its LayerNorm).
#include <string.h>
#include "gemm_tile.h"

namespace wam {

// ------------------------------------------------------------------- tiles
// With weights from HBM a CU takes operands in at 50-60 GB/s (about 32 KB of
// loads in flight), whatever the tile or the way to LDS (224 x 14336 x 3072 on
// 128x128 tiles: 34 us staged through LDS by direct loads or through
// registers, 3 or 5 stages): fewer operand bytes per output (a larger tile)
// and more CUs at work help, k ranges trade the second against partial-sum
// traffic.  That is not all that bounds them: with the weights in the
// last-level cache the same product takes 31 us of 37.
using Small32 = GemmCfg<32, 128, 64, 1, 4, 3, 2>;
using Small64 = GemmCfg<64, 128, 64, 1, 4, 5>;
using Small64n64 = GemmCfg<64, 64, 64, 2, 2, 5>;
using Small128 = GemmCfg<128, 128, 64, 2, 4, 5, 1, 2>;
using Small192 = GemmCfg<192, 128, 64, 2, 4, 3, 1, 2>;
using Small256 = GemmCfg<256, 128, 64, 4, 2, 3, 1, 2>;
// fp8 e4m3 weights (64-byte LDS rows widened at the fragment read)
using Small64f8 = GemmCfg<64, 128, 64, 1, 4, 5, 1, 0, 1>;
using Small128f8 = GemmCfg<128, 128, 64, 2, 4, 5, 1, 0, 1>;
using Small256f8 = GemmCfg<256, 128, 64, 4, 2, 3, 1, 0, 1>;

// Cost model, in us: kSmallLaunch + rounds * (round + steps * step), rounds being
// dispatch rounds of one workgroup per CU and steps the 64-deep k-steps of
// one range; at least the weights' time from HBM; and for several ranges the
// reduce pass (split_reduce_us of the partial sums' bytes, written and read).
// Fitted to 34 shapes (96 to 2325 rows, K 1536 to 14336, N 1536 to 14336, 1
// to 32 ranges, weights cold): 6% rms, and the plan it picks is within 3% of
// the fastest measured one but for 400 x 3072 x 14336 (8%) and 224 x 9216 x
// 3072 (13%).  Against 128x128 or 256x128 tiles over the whole k:
//   32 x 3072 x 14336 107 -> 22 us     780 x 3072 x 14336 114 -> 80
//   224 x 3072 x 3072  30 -> 18        1024 x 9216 x 3072 104 -> 60
//   224 x 3072 x 14336 125 -> 37       1560 x 3072 x 14336 227 -> 122
//   1024 x 1536 x 8960  82 -> 40       2325 x 3072 x 14336 218 -> 182
// 64x64 tiles, against the best of the wider ones with their reduce pass (us):
// 64 x 14336 x 3072 24.3 -> 21.7 and 32 rows 21.9 -> 18.8 (whole k on 224
// CUs), 224 x 3072 x 3072 17.7 -> 14.8, 32 x 3072 x 3072 10.6 -> 9.6.
// The four-wave kernel's tiles of 128 to 192 rows, against the best of the
// others (us): 2325 x 3072 x 3072 51 -> 45, 1024 x 8960 x 1536 35 -> 31, 1024 x
// 1536 x 8960 40.3 -> 39.5.  A reduction that a
// row pass does anyway costs its traffic only (fused): 224 x 9216 x 3072 in
// three ranges with the q/k norm's row pass 33 us, whole and then the pass 39.
// fp8 weights (wb 1) are priced with the same steps, fitted to bf16 weights
// only; of 90 random fp8 shapes (1 to 2600 rows) none is slower than with
// tiles of 128 or 256 rows over the whole k.
struct TileCost {
  int bm, bn;
  double round, step;
};
constexpr TileCost kTiles[] = {
    {32, 128, 0.3, 0.47},  {64, 128, 1.9, 0.42},  {128, 128, 3.0, 0.49}, {192, 128, 2.2, 0.64}, {256, 128, 2.7, 0.88},
    {128, 256, 2.3, 0.83}, {160, 256, 4.5, 0.90}, {192, 256, 6.0, 1.03}, {224, 256, 4.7, 1.05}, {256, 256, 4.4, 1.21},
    {64, 64, 0.5, 0.28},
};
constexpr int kTile32 = 0, kTile192 = 3, kTileW4 = 5, kTileW224 = 8, kTile64n64 = 10, kTileCount = 11;
constexpr double kHbmBytesPerUs = 6.6e6;
constexpr int kMaxRanges = 32;

SplitPlan split_plan(int M, int seg_n, int n_seg, int K, int wb, int64_t ws_bytes, bool fused) {
  const int cus = device_cu_count(), nk = K / 64;
  const double hbm = (double)seg_n * n_seg * K * wb / kHbmBytesPerUs;
  SplitPlan best{0, 1};
  double best_cost = 1e30;
  for (int c = 0; c < kTileCount; ++c) {
    const TileCost& t = kTiles[c];
    const bool w4 = c >= kTileW4 && c < kTile64n64;
    // 256-column tiles hold whole tiles of one segment; the fp8-weight small
    // tiles are 128 columns wide
    if ((w4 && seg_n % 256 != 0) || (n_seg > 1 && seg_n % t.bn != 0)) continue;
    // fp8 weights: 64 and 128 rows, 256 x 128 (a 32-row stage would not hold a
    // 32-row slab of the fp32 epilogue), and the two largest
    if (wb == 1 && (c == kTile32 || c == kTile192 || c == kTile64n64 || (w4 && c < kTileW224))) continue;
    // a shorter tile holds all rows
    if (c > (wb == 1 ? 1 : 0) && kTiles[c - 1].bm >= M && kTiles[c - 1].bn == t.bn) continue;
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((seg_n + t.bn - 1) / t.bn) * n_seg;
    // one range, or as many as fill one or two rounds
    const int64_t cand[3] = {1, cus / tiles, 2 * cus / tiles};
    for (int64_t ks : cand) {
      if (ks > kMaxRanges) ks = kMaxRanges;
      if (ks > nk) ks = nk;
      if (ks < 1) continue;
      const int64_t rounds = (tiles * ks + cus - 1) / cus, steps = (nk + ks - 1) / ks;
      const int64_t bytes = ks > 1 ? ks * (int64_t)M * seg_n * n_seg * 4 : 0;
      if (bytes > ws_bytes || bytes >= INT32_MAX) continue;  // (32-bit offsets in the reduce passes)
      double cost = (double)rounds * (t.round + (double)steps * t.step);
      cost = kSmallLaunch + (cost > hbm ? cost : hbm);
      if (ks > 1) cost += split_reduce_us(bytes, fused);
      if (cost < best_cost - 1e-9) best_cost = cost, best = SplitPlan{c, (int)ks};
    }
  }
  return best;
}

int64_t split_plan_bytes(const SplitPlan& g, int M, int seg_n, int n_seg) {
  return g.ks > 1 ? g.ks * (int64_t)M * seg_n * n_seg * 4 : 0;
}

template <class C>
static int launch_small(LinearParams& p, hipStream_t s) {
  p.n_tiles_per_seg = (p.seg_n + C::BN - 1) / C::BN;
  p.m_tiles = (p.M + C::BM - 1) / C::BM;
  p.n_tiles = p.n_tiles_per_seg * p.n_seg_count;
  p.part_ld = p.seg_n * p.n_seg_count;
  const dim3 grid((unsigned)(p.m_tiles * p.n_tiles * p.k_split)), block(C::kThreads);
  if (p.k_split > 1) {
    hipLaunchKernelGGL((gemm_bf16_kernel<C, kEpiPartial>), grid, block, 0, s, p);
  } else {
    switch (p.epi) {
      case WAM_EPI_BIAS:
        hipLaunchKernelGGL((gemm_bf16_kernel<C, WAM_EPI_BIAS>), grid, block, 0, s, p);
        break;
      case WAM_EPI_BIAS_GELU:
        hipLaunchKernelGGL((gemm_bf16_kernel<C, WAM_EPI_BIAS_GELU>), grid, block, 0, s, p);
        break;
      case WAM_EPI_BIAS_GATE_RES:
        if (p.res_f32) hipLaunchKernelGGL((gemm_bf16_kernel<C, WAM_EPI_BIAS_GATE_RES, 1>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((gemm_bf16_kernel<C, WAM_EPI_BIAS_GATE_RES, 0>), grid, block, 0, s, p);
        break;
      default:
        if (p.res_f32) hipLaunchKernelGGL((gemm_bf16_kernel<C, WAM_EPI_BIAS_RES, 1>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((gemm_bf16_kernel<C, WAM_EPI_BIAS_RES, 0>), grid, block, 0, s, p);
        break;
    }
  }
  WAM_LAUNCHED("gemm_bf16_kernel");
  return WAM_OK;
}

// The tiles of a plan: with several ranges only the partial sums are written.
int split_tiles(LinearParams& p, const SplitPlan& g, int wb, hipStream_t s) {
  p.k_split = g.ks;
  WAM_REQUIRE(g.ks == 1 || (p.part && g.ks <= p.K / 64), "wam_linear: bad split-K launch");
  if (g.tile == kTile64n64) return launch_small<Small64n64>(p, s);
  if (g.tile >= kTileW4) return w4_tiles(p, kTiles[g.tile].bm, wb, s);
  if (wb == 1) {
    switch (g.tile) {
      case 1: return launch_small<Small64f8>(p, s);
      case 2: return launch_small<Small128f8>(p, s);
      default: return launch_small<Small256f8>(p, s);
    }
  }
  switch (g.tile) {
    case 0: return launch_small<Small32>(p, s);
    case 1: return launch_small<Small64>(p, s);
    case 2: return launch_small<Small128>(p, s);
    case kTile192: return launch_small<Small192>(p, s);
    default: return launch_small<Small256>(p, s);
  }
}

// ------------------------------------------------------------------ reduce
// The launch's epilogue over the partial sums, one thread per 4 consecutive
// outputs of one segment.  W1: fp8 weights (per-column scales).  A8: fp8
// activations with row scales; MXO: e4m3 output with an exponent per 32
// columns (8 lanes), as the four-wave kernel writes it.
template <int EPI, bool W1, bool A8 = false, bool MXO = false>
__global__ __launch_bounds__(256) void split_reduce_kernel(LinearParams p) {
  const int q4 = p.part_ld / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)p.M * q4) return;
  const int m = (int)(i / q4), c = (int)(i - (int64_t)m * q4) * 4;
  const int seg = c >= p.seg_n ? (c >= 2 * p.seg_n ? 2 : 1) : 0, n = c - seg * p.seg_n;
  const bf16* bias = seg == 0 ? p.bias[0] : (seg == 1 ? p.bias[1] : p.bias[2]);
  void* out = seg == 0 ? p.out[0] : (seg == 1 ? p.out[1] : p.out[2]);
  float bv[4] = {0.f, 0.f, 0.f, 0.f}, wsc[4] = {1.f, 1.f, 1.f, 1.f}, rv[4] = {0.f, 0.f, 0.f, 0.f};
  const u32x2 braw = *reinterpret_cast<const u32x2*>(bias ? static_cast<const void*>(bias + n) : p.part);
  if constexpr (W1) {
    const float* ws = seg == 0 ? p.wscale[0] : (seg == 1 ? p.wscale[1] : p.wscale[2]);
    const float4 t = *reinterpret_cast<const float4*>(ws + n);
    wsc[0] = t.x; wsc[1] = t.y; wsc[2] = t.z; wsc[3] = t.w;
  }
  constexpr bool RES = EPI == WAM_EPI_BIAS_GATE_RES || EPI == WAM_EPI_BIAS_RES;
  Raw4 rraw{};
  if constexpr (RES) rraw = ld4_raw(p.res, p.res_f32 != 0, (int64_t)m * p.ldr + n);
  Raw4 gtab{}, graw{};
  if constexpr (EPI == WAM_EPI_BIAS_GATE_RES) {
    gtab = ld4_raw(p.gate.table, p.gate.table_dtype == WAM_F32, (int64_t)p.gate_index * p.mod_d + n + p.n_off);
    graw = gate_raw(p, m, n + p.n_off);
  }
  const int off[1] = {(m * p.part_ld + c) * 4};
  f32x4 v[1];
  sum_ranges<1>(p, off, v);
  if (bias) widen4_bf16(braw, bv);
  if constexpr (RES) widen4(rraw, p.res_f32 != 0, rv);
  if constexpr (A8) {
    const float sr = p.ascale[m];
#pragma unroll
    for (int e = 0; e < 4; ++e) wsc[e] = sr * wsc[e];
  }
  if constexpr (MXO) {
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = v[0][e] * wsc[e] + bv[e];
      if constexpr (EPI == WAM_EPI_BIAS_GELU) y[e] = gelu_tanh(y[e]);
    }
    const int X = mx_exponent(max8_lanes(fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3])))));
    const float inv = __uint_as_float((uint32_t)(127 - X) << 23);
    int pk = 0;
    pk = __builtin_amdgcn_cvt_pk_fp8_f32(y[0] * inv, y[1] * inv, pk, false);
    pk = __builtin_amdgcn_cvt_pk_fp8_f32(y[2] * inv, y[3] * inv, pk, true);
    *reinterpret_cast<int*>(static_cast<uint8_t*>(out) + (int64_t)m * p.ldo + n) = pk;
    if ((threadIdx.x & 7) == 0) p.oscale[(int64_t)m * (p.seg_n / 32) + n / 32] = (uint8_t)(X + 127);
    return;
  }
  float gate[4] = {0.f, 0.f, 0.f, 0.f}, gb[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (EPI == WAM_EPI_BIAS_GATE_RES) {
    widen4(gtab, p.gate.table_dtype == WAM_F32, gate);
    widen4(graw, p.gate.temb_dtype == WAM_F32, gb);
#pragma unroll
    for (int e = 0; e < 4; ++e) gate[e] += gb[e];
  }
  epi_apply<EPI, W1 ? 1 : 2>(p, out, m, n, v[0], bv, wsc, gate, rv);
}

int split_reduce(const LinearParams& p, int wb, hipStream_t s) {
  const dim3 grid((unsigned)(((int64_t)p.M * (p.part_ld / 4) + 255) / 256)), block(256);
  const bool w1 = wb == 1;
#define WAM_REDUCE(E)                                                                             \
  if (w1) hipLaunchKernelGGL((split_reduce_kernel<E, true>), grid, block, 0, s, p);               \
  else hipLaunchKernelGGL((split_reduce_kernel<E, false>), grid, block, 0, s, p)
  if (p.ascale) {  // bias or GELU, whole 256-column tiles
    const bool gelu = p.epi == WAM_EPI_BIAS_GELU, mxo = p.oscale != nullptr;
    auto kernel = gelu ? (mxo ? split_reduce_kernel<WAM_EPI_BIAS_GELU, true, true, true>
                              : split_reduce_kernel<WAM_EPI_BIAS_GELU, true, true, false>)
                       : (mxo ? split_reduce_kernel<WAM_EPI_BIAS, true, true, true>
                              : split_reduce_kernel<WAM_EPI_BIAS, true, true, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, s, p);
    WAM_LAUNCHED("split_reduce_kernel");
    return WAM_OK;
  }
  switch (p.epi) {
    case WAM_EPI_BIAS: WAM_REDUCE(WAM_EPI_BIAS); break;
    case WAM_EPI_BIAS_GELU: WAM_REDUCE(WAM_EPI_BIAS_GELU); break;
    case WAM_EPI_BIAS_GATE_RES: WAM_REDUCE(WAM_EPI_BIAS_GATE_RES); break;
    default: WAM_REDUCE(WAM_EPI_BIAS_RES); break;
  }
#undef WAM_REDUCE
  WAM_LAUNCHED("split_reduce_kernel");
  return WAM_OK;
}

}  // namespace wam
