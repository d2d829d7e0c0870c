// The row passes of the block that follow a projection split over k, with the
// reduction of its partial sums in them: q/k/v bias + RMSNorm + RoPE, and the
// (gated) residual stream with the LayerNorm that reads it.  One workgroup
// per row (and segment): a few rows give too few waves to hide a reduce pass,
// its launch and a row pass one after the other (2 x 16 rows: 4 + 6 us for
// the reduce and the LayerNorm, 5.5 us together).  The same kernel without
// partial sums is the LayerNorm of few rows.
#include "gemm_tile.h"
#include "kv_layout.h"

namespace wam {

constexpr int kRowThreads = 256;

// Sum over the workgroup of each thread's v (every thread gets it).  slot:
// which of the kernel's reductions this is, so that consecutive ones need one
// barrier each.
__device__ inline float block_sum(float v, float (*sh)[4], int slot) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[slot][threadIdx.x >> 6] = v;
  __syncthreads();
  return (sh[slot][0] + sh[slot][1]) + (sh[slot][2] + sh[slot][3]);
}

// q/k/v: y = bf16(sum + bias) as the projection rounds it; segments with a
// gamma (s < r.n_tensors) are then normalised over the row and rotated, as
// rms_rope_kernel does.  NCH chunks of 4 columns per thread, 1024 apart.
// KV: the first workgroup does the KV pool's bookkeeping instead.
template <int NCH, bool KV>
__global__ __launch_bounds__(kRowThreads) void split_rms_rope_kernel(LinearParams p, wam_rms_rope_args r,
                                                                     wam_kv_layout_args kv) {
  __shared__ float sh[1][4];
  if constexpr (KV)
    if (blockIdx.x == 0) return kv_layout_pool<kRowThreads>(kv);
  const int tid = threadIdx.x, D = p.seg_n, job = blockIdx.x - (KV ? 1 : 0);
  const int row = __builtin_amdgcn_readfirstlane(job / p.n_seg_count);
  const int seg = __builtin_amdgcn_readfirstlane(job - row * p.n_seg_count);
  const bf16* bias = seg == 0 ? p.bias[0] : (seg == 1 ? p.bias[1] : p.bias[2]);
  bf16* out = static_cast<bf16*>(seg == 0 ? p.out[0] : (seg == 1 ? p.out[1] : p.out[2])) + (int64_t)row * p.ldo;
  const bool norm = seg < r.n_tensors;
  const void* gamma = norm ? (seg ? r.gamma[1] : r.gamma[0]) : p.part;
  const float2* f = nullptr;
  if (norm && r.freq) {
    const int b = row / r.tokens, t = row - b * r.tokens;
    f = static_cast<const float2*>(r.freq) + ((int64_t)(r.freq_batch == 1 ? 0 : b) * r.tokens + t) * (r.head_dim / 2);
  }
  // (columns past the row repeat its last four and are masked)
  Raw4 braw[NCH], graw[NCH];
  float4 fr[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int n = min((tid + kRowThreads * c) * 4, D - 4);
    braw[c] = ld4_raw(bias ? static_cast<const void*>(bias) : p.part, false, n);
    graw[c] = ld4_raw(gamma, false, n);
    const float2* fp = f ? f + ((n % r.head_dim) >> 1) : reinterpret_cast<const float2*>(p.part);
    const float2 f0 = fp[0], f1 = fp[1];
    fr[c] = make_float4(f0.x, f0.y, f1.x, f1.y);
  }
  int off[NCH];
  f32x4 v[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) off[c] = (row * p.part_ld + seg * D + min((tid + kRowThreads * c) * 4, D - 4)) * 4;
  sum_ranges<NCH>(p, off, v);
  float y[NCH][4], ss = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const bool in = (tid + kRowThreads * c) * 4 < D;
    float bv[4];
    widen4(braw[c], false, bv);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[c][e] = static_cast<float>(static_cast<bf16>(bias ? v[c][e] + bv[e] : v[c][e]));
      ss += in ? y[c][e] * y[c][e] : 0.f;
    }
  }
  const float eps = seg ? r.eps[1] : r.eps[0];
  const float rstd = norm ? rsqrtf(block_sum(ss, sh, 0) / D + eps) : 1.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int n = (tid + kRowThreads * c) * 4;
    float z[4];
    if (norm) {
      float gv[4];
      widen4(graw[c], false, gv);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[c][e] = y[c][e] * rstd * gv[e];
    }
    z[0] = y[c][0] * fr[c].x - y[c][1] * fr[c].y;
    z[1] = y[c][0] * fr[c].y + y[c][1] * fr[c].x;
    z[2] = y[c][2] * fr[c].z - y[c][3] * fr[c].w;
    z[3] = y[c][2] * fr[c].w + y[c][3] * fr[c].z;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16>(f ? z[e] : y[c][e]);
    if (n < D) *reinterpret_cast<bf16x4*>(out + n) = o;
  }
}

// LayerNorm of one row.  SRC: what the row is.
enum { kRowInput = 0, kRowResidual = 1, kRowGated = 2 };  // l.x, res + sum + b, res + (sum + b) * gate
// With partial sums the row goes to p.out[0] in fp32 too.  Q8 as in
// ln_modulate_kernel.  COMMIT: the workgroups past the rows copy new K/V rows
// to the pool (256 rows: a launch of its own 4.9 us, here the pass takes 9.4
// instead of 8.6; the block 238.5 -> 236.7).
template <int NCH, int SRC, bool Q8, bool COMMIT>
__global__ __launch_bounds__(kRowThreads) void row_ln_kernel(LinearParams p, wam_ln_args l, wam_kv_commit_args kv) {
  __shared__ float sh[3][4];
  if constexpr (COMMIT)
    if ((int)blockIdx.x >= l.rows) return kv_commit_rows<kRowThreads>(kv, blockIdx.x - l.rows, gridDim.x - l.rows);
  const int tid = threadIdx.x, D = l.D, row = blockIdx.x;
  const bool xf32 = SRC == kRowInput ? l.x_dtype == WAM_F32 : p.res_f32 != 0;
  const void* x = SRC == kRowInput ? l.x : p.res;
  const int64_t x_at = SRC == kRowInput ? (int64_t)row * D : (int64_t)row * p.ldr;
  // add = s0 + s1, mul = s2 + s3 + 1 of the modulation; beta and gamma alone
  // with affine parameters (s1, s3 then repeat them unused).
  const wam_modulation& m = l.mod;
  const bool affine = l.affine != 0;
  const bool f0 = (affine ? l.gb_dtype : m.table_dtype) == WAM_F32, f1 = (affine ? l.gb_dtype : m.temb_dtype) == WAM_F32;
  const int64_t trow = affine ? 0 : temb_row(m, row);
  const int64_t a0 = affine ? 0 : (int64_t)l.shift_index * D, a1 = affine ? 0 : temb_off(m, trow, l.shift_index, D, 0);
  const int64_t b0 = affine ? 0 : a0 + D, b1 = affine ? 0 : temb_off(m, trow, l.shift_index + 1, D, 0);
  const void *s0 = affine ? l.beta : m.table, *s1 = affine ? l.beta : m.temb, *s2 = affine ? l.gamma : m.table,
             *s3 = affine ? l.gamma : m.temb;
  const wam_modulation& gm = p.gate;
  const bool gf0 = gm.table_dtype == WAM_F32, gf1 = gm.temb_dtype == WAM_F32;
  const int64_t g0 = (int64_t)p.gate_index * D, g1 = SRC == kRowGated ? temb_off(gm, temb_row(gm, row), p.gate_index, D, 0) : 0;
  Raw4 xr[NCH], c0[NCH], c1[NCH], c2[NCH], c3[NCH], gr0[NCH], gr1[NCH], br[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int n = min((tid + kRowThreads * c) * 4, D - 4);
    xr[c] = ld4_raw(x, xf32, x_at + n);
    c0[c] = ld4_raw(s0, f0, a0 + n);
    c1[c] = ld4_raw(s1, f1, a1 + n);
    c2[c] = ld4_raw(s2, f0, b0 + n);
    c3[c] = ld4_raw(s3, f1, b1 + n);
    if constexpr (SRC != kRowInput) br[c] = ld4_raw(p.bias[0] ? static_cast<const void*>(p.bias[0]) : x, false, n);
    if constexpr (SRC == kRowGated) {
      gr0[c] = ld4_raw(gm.table, gf0, g0 + n);
      gr1[c] = ld4_raw(gm.temb, gf1, g1 + n);
    }
  }
  f32x4 sums[NCH];
  if constexpr (SRC != kRowInput) {
    int off[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) off[c] = (row * p.part_ld + min((tid + kRowThreads * c) * 4, D - 4)) * 4;
    sum_ranges<NCH>(p, off, sums);
  }
  float v[NCH][4], s = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const bool in = (tid + kRowThreads * c) * 4 < D;
    const int n = min((tid + kRowThreads * c) * 4, D - 4);
    widen4(xr[c], xf32, v[c]);
    if constexpr (SRC != kRowInput) {
      const f32x4 y = sums[c];
      float bv[4], ga[4], gb[4];
      widen4(br[c], false, bv);
      if constexpr (SRC == kRowGated) {
        widen4(gr0[c], gf0, ga);
        widen4(gr1[c], gf1, gb);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float t = p.bias[0] ? y[e] + bv[e] : y[e];
        v[c][e] = SRC == kRowGated ? v[c][e] + t * (ga[e] + gb[e]) : v[c][e] + t;
      }
      if (in)
        *reinterpret_cast<float4*>(static_cast<float*>(p.out[0]) + (int64_t)row * p.ldo + n) =
            make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s += in ? v[c][e] : 0.f;
  }
  const float mean = block_sum(s, sh, 0) / D;
  float q = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = (tid + kRowThreads * c) * 4 < D ? v[c][e] - mean : 0.f;
      q += d * d;
    }
  const float rstd = rsqrtf(block_sum(q, sh, 1) / D + l.eps);
  bf16x4 o[NCH];
  float mx = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int n = (tid + kRowThreads * c) * 4;
    float w0[4], w1[4], w2[4], w3[4];
    widen4(c0[c], f0, w0);
    widen4(c1[c], f1, w1);
    widen4(c2[c], f0, w2);
    widen4(c3[c], f1, w3);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float add = affine ? w0[e] : w0[e] + w1[e], mul = affine ? w2[e] : (w2[e] + w3[e]) + 1.f;
      o[c][e] = static_cast<bf16>((v[c][e] - mean) * rstd * mul + add);
      if constexpr (Q8) mx = n < D ? fmaxf(mx, fabsf(static_cast<float>(o[c][e]))) : mx;
    }
    if (n < D && (!Q8 || l.y)) *reinterpret_cast<bf16x4*>(static_cast<bf16*>(l.y) + (int64_t)row * D + n) = o[c];
  }
  if constexpr (Q8) {
    mx = wave_max(mx);
    if ((tid & 63) == 0) sh[2][tid >> 6] = mx;
    __syncthreads();
    const float amax = fmaxf(fmaxf(sh[2][0], sh[2][1]), fmaxf(sh[2][2], sh[2][3]));
    const float sc = amax > 0.f ? amax / 448.0f : 1.0f;
    const float inv = amax > 0.f ? 448.0f / amax : 1.0f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int n = (tid + kRowThreads * c) * 4;
      int w = 0;
      w = __builtin_amdgcn_cvt_pk_fp8_f32(static_cast<float>(o[c][0]) * inv, static_cast<float>(o[c][1]) * inv, w, false);
      w = __builtin_amdgcn_cvt_pk_fp8_f32(static_cast<float>(o[c][2]) * inv, static_cast<float>(o[c][3]) * inv, w, true);
      if (n < D) *reinterpret_cast<int*>(static_cast<uint8_t*>(l.y8) + (int64_t)row * D + n) = w;
    }
    if (tid == 0) l.y8_scale[row] = sc;
  }
}

template <int NCH>
static void launch_rms_rope(const LinearParams& p, const wam_rms_rope_args& r, const wam_kv_layout_args* kv, hipStream_t s) {
  const dim3 grid((unsigned)(p.M * p.n_seg_count + (kv ? 1 : 0))), block(kRowThreads);
  if (kv) hipLaunchKernelGGL((split_rms_rope_kernel<NCH, true>), grid, block, 0, s, p, r, *kv);
  else hipLaunchKernelGGL((split_rms_rope_kernel<NCH, false>), grid, block, 0, s, p, r, wam_kv_layout_args{});
}

int rms_rope_check(const wam_rms_rope_args*);

int split_rms_rope(const LinearParams& p, const wam_rms_rope_args& r, const wam_kv_layout_args* kv, hipStream_t s) {
  WAM_TRY(rms_rope_check(&r));
  switch ((p.seg_n + 1023) / 1024) {
    case 1: launch_rms_rope<1>(p, r, kv, s); break;
    case 2: launch_rms_rope<2>(p, r, kv, s); break;
    case 3: launch_rms_rope<3>(p, r, kv, s); break;
    default: launch_rms_rope<4>(p, r, kv, s); break;
  }
  WAM_LAUNCHED("split_rms_rope_kernel");
  return WAM_OK;
}

template <int SRC, bool Q8, bool COMMIT = false>
static void launch_row_ln(const LinearParams& p, const wam_ln_args& l, const wam_kv_commit_args& kv, hipStream_t s) {
  const int64_t n = COMMIT ? (int64_t)kv.B * kv.tokens * (kv.D / 8) : 0;
  const int64_t copies = (n + kRowThreads - 1) / kRowThreads;
  const dim3 grid((unsigned)(l.rows + (copies < 1024 ? copies : 1024))), block(kRowThreads);
  switch ((l.D + 1023) / 1024) {
    case 1: hipLaunchKernelGGL((row_ln_kernel<1, SRC, Q8, COMMIT>), grid, block, 0, s, p, l, kv); break;
    case 2: hipLaunchKernelGGL((row_ln_kernel<2, SRC, Q8, COMMIT>), grid, block, 0, s, p, l, kv); break;
    case 3: hipLaunchKernelGGL((row_ln_kernel<3, SRC, Q8, COMMIT>), grid, block, 0, s, p, l, kv); break;
    default: hipLaunchKernelGGL((row_ln_kernel<4, SRC, Q8, COMMIT>), grid, block, 0, s, p, l, kv); break;
  }
}

int split_ln(const LinearParams& p, const wam_ln_args& l, const wam_kv_commit_args* commit, hipStream_t s) {
  const wam_kv_commit_args none{};
  const bool gated = p.epi == WAM_EPI_BIAS_GATE_RES, q8 = l.y8 != nullptr;
  WAM_REQUIRE(!commit || (gated && !q8), "split_ln: a commit rides with the gated residual only");
  if (commit) launch_row_ln<kRowGated, false, true>(p, l, *commit, s);
  else if (gated) q8 ? launch_row_ln<kRowGated, true>(p, l, none, s) : launch_row_ln<kRowGated, false>(p, l, none, s);
  else q8 ? launch_row_ln<kRowResidual, true>(p, l, none, s) : launch_row_ln<kRowResidual, false>(p, l, none, s);
  WAM_LAUNCHED("row_ln_kernel");
  return WAM_OK;
}

int row_ln(const wam_ln_args& l, hipStream_t s) {
  const LinearParams none{};
  l.y8 ? launch_row_ln<kRowInput, true>(none, l, wam_kv_commit_args{}, s)
       : launch_row_ln<kRowInput, false>(none, l, wam_kv_commit_args{}, s);
  WAM_LAUNCHED("row_ln_kernel");
  return WAM_OK;
}

}  // namespace wam
