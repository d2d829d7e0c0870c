// Attention for calls with few queries per key source (the 16 action tokens
// of a policy step and its candidates, one video latent, a short text
// context): a workgroup takes 32, 64 or 128 queries of one head, deals their
// keys to its eight waves in 32-key tiles and merges the waves' partial
// results through LDS.
//
// What bounds such a call: a CU keeps about 32 KB of loads in flight, 50-60
// GB/s while K and V come from HBM, so the key rows that all workgroups read
// together set the time.  Batch rows that share a pool row (the candidates of
// one CFG branch) therefore go through one workgroup as a group: the history
// is read once for the group, each row's own keys are masked to its own
// queries.  The measured choice is at attention_few_plan.
#include <algorithm>
#include <type_traits>
#include "attention_common.h"

namespace wam {

constexpr int kFewKeys = 32;                      // keys per tile
constexpr int kFewTile = kFewKeys * kAttnHD * 2;  // 8 KB of K or V
constexpr int kFewWaves = 8;
constexpr int kFewMaxRanges = 8;

// Running maximum of a query without a finite score: finite, so that a score
// of -inf less it is -inf (less -inf it would be NaN), and below any other.
constexpr float kNoMax = -__FLT_MAX__;

// Maximum of three (a NaN in any gives NaN, as a score that is NaN must).
__device__ inline float max3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}

// QW waves along the queries, KW = 8 / QW along the keys.  A unit is (query
// block of 32 QW, group of G batch rows, head), query block fastest, groups of
// one head adjacent; G > 1 needs B % G == 0 and G * Mq <= 32 QW.  Queries of a
// group are numbered batch row by batch row.  The unit's tiles are those of
// each distinct pool row of the group, then of each distinct own row; with
// gridDim.x > units, tile range blockIdx / units, whose unnormalised O and
// (max, sum) go to `part` for few_combine_kernel.
//
// A tile's K and V rows come in as whole 256-byte rows, 4 per load, into
// registers one tile ahead (the QW waves of the tile share the loads), go to
// LDS and are read back as MFMA fragments in the layouts of attention.hip:
// one barrier per tile and two LDS stages; with QW = 1 a tile is the wave's
// own and needs neither.
template <int QW, bool GROUP>
__global__ __launch_bounds__(64 * kFewWaves, 2) void attention_few_kernel(wam_attention_args a, int group, int units,
                                                                         int ranges, float* __restrict__ part) {
  constexpr int KW = kFewWaves / QW, NLD = 8 / QW, QB = 32 * QW;
  const int G = GROUP ? group : 1;
  constexpr int kStage = KW * 2 * kFewTile;
  static_assert(QW == 1 || 2 * kStage <= kFewWaves * 2 * kFewTile, "two stages fit the merge's LDS");
  __shared__ __attribute__((aligned(1024))) char lds[kFewWaves * 2 * kFewTile];
  __shared__ float s_ml[2][kFewWaves][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = wave % QW, kw = wave / QW;
  const int l32 = lane & 31, half = lane >> 5;
  const int piece = xcd_remap(blockIdx.x, gridDim.x);
  const int range = __builtin_amdgcn_readfirstlane(piece / units);
  const int unit = __builtin_amdgcn_readfirstlane(piece - range * units);
  const int nq = G * a.Mq, nqb = (nq + QB - 1) / QB, groups = a.B / G;
  const int qb = unit % nqb, gh = unit / nqb;
  const int b0 = (gh % groups) * G, h = gh / groups;
  const int n_hist = a.n_hist_dev ? __builtin_amdgcn_readfirstlane(*a.n_hist_dev) : 0;
  // consecutive history slots start at base; otherwise they are listed
  const int base = a.n_hist_dev && a.hist_base_dev ? __builtin_amdgcn_readfirstlane(*a.hist_base_dev) : -1;
  // Lane i holds the pool and own row of batch row b0 + i (repeated past G);
  // a group's distinct ones, in batch row order, go to the lanes of list.
  const int bi = b0 + min(lane, G - 1);
  const int rp = clamp_row(a.pool_rows ? (int)a.pool_rows[bi] : bi, a.n_hist_dev ? a.pool_batch : 1);
  const int ro = clamp_row(a.kv_rows ? (int)a.kv_rows[bi] : bi, a.kv_batch);
  // This lane's query and its rows.
  const int vq = qb * QB + qw * 32 + l32;
  const int vc = min(vq, nq - 1), bl = vc / a.Mq, b = b0 + bl, qi = vc - bl * a.Mq;
  const int my_pool = __shfl(rp, bl, 64), my_own = __shfl(ro, bl, 64);
  int n_pool = 1, n_own = 1, list_p = rp, list_o = ro;
  if constexpr (GROUP) {
    auto distinct = [&](int r, int& list) {
      bool first = lane < G;
#pragma unroll
      for (int j = 0; j < kFewGroupMax; ++j) first &= j >= lane || __builtin_amdgcn_readlane(r, j) != r;
      const uint64_t bits = __builtin_amdgcn_ballot_w64(first);
      const int pos = __popcll(bits & ((1ull << lane) - 1));
      list = __builtin_amdgcn_ds_permute((first ? pos : 63) * 4, r);
      return (int)__popcll(bits);
    };
    n_pool = distinct(rp, list_p);
    n_own = distinct(ro, list_o);
  }
  const int hist_tiles = (n_hist + kFewKeys - 1) / kFewKeys, own_tiles = (a.Mk + kFewKeys - 1) / kFewKeys;
  const int n_pool_tiles = n_pool * hist_tiles, all = n_pool_tiles + n_own * own_tiles;
  const int t0 = (int)((int64_t)range * all / ranges), t1 = (int)((int64_t)(range + 1) * all / ranges);

  // Tile t: its source (history or own keys of row `row`), first key, key count.
  struct Tile {
    bool hist;
    int row, key0, n;
  };
  auto tile_of = [&](int t) {
    Tile x;
    x.hist = t < n_pool_tiles;
    const int u = x.hist ? t : t - n_pool_tiles, per = x.hist ? hist_tiles : own_tiles;
    const int src = GROUP ? u / per : 0;
    x.key0 = (u - src * per) * kFewKeys;
    x.row = __builtin_amdgcn_readlane(x.hist ? list_p : list_o, src);
    x.n = x.hist ? n_hist : a.Mk;
    return x;
  };
  // Load i of this wave covers tile rows 4 (qw NLD + i) + lane / 16, as byte
  // offsets into the source's rows of this head (host: below 2^31 / 2^32).
  // Keys past the source's end, and tiles past the range, read zeros through
  // the resources' bound; a listed slot (read a tile before its row) past the
  // end repeats the last one.  Their scores are masked.
  const int lrow = 4 * qw * NLD + (lane >> 4), pch = lane & 15;
  const bool listed = base < 0 && n_hist > 0;
  const int prs = (int)a.pool_rstride * 2, krs = (int)a.kv_rstride * 2;
  int sl[NLD];
  auto slots_of = [&](int t) {
    const Tile x = tile_of(t);
#pragma unroll
    for (int i = 0; i < NLD; ++i) sl[i] = a.slots[min(x.key0 + 4 * i + lrow, n_hist - 1)];
  };
  u32x4 kr[NLD], vr[NLD];
  Tile next{};  // the tile in kr and vr
  auto load = [&](int t) {
    const Tile x = next = tile_of(t);
    const int64_t at = (int64_t)x.row * (x.hist ? a.pool_bstride : a.kv_bstride) + h * kAttnHD;
    const int rs = x.hist ? prs : krs, skip = x.hist && base >= 0 ? base : 0;
    const uint32_t end = x.hist && listed ? (uint32_t)(a.pool_bstride * 2 - h * kAttnHD * 2)
                                          : (uint32_t)(skip + x.n - 1) * (uint32_t)rs + kAttnHD * 2;
    const uint32_t bytes = t < t1 ? end : 0u;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(static_cast<const bf16*>(x.hist ? a.pool_k : a.k) + at, bytes);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(static_cast<const bf16*>(x.hist ? a.pool_v : a.v) + at, bytes);
    int off[NLD];
    if (x.hist && listed) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) off[i] = sl[i] * rs + pch * 16;
    } else {
#pragma unroll
      for (int i = 0; i < NLD; ++i) off[i] = (skip + x.key0 + lrow) * rs + pch * 16 + i * 4 * rs;
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      kr[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off[i], 0, 0));
      vr[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, off[i], 0, 0));
    }
  };
  int t = t0 + kw;
  if (listed) slots_of(t);
  // Q fragments (B operand of S^T = K Q^T): query qi, d = 16 ks + 8 half .. +8.
  bf16x8 qf[8];
  {
    const bf16* q = static_cast<const bf16*>(a.q) + (int64_t)b * a.q_bstride + h * kAttnHD + (int64_t)qi * a.q_rstride +
                    8 * half;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = ld_bf16x8(q + 16 * ks);
  }
  float sc = a.scale * kLog2e;
  if (a.q_ssq) sc *= q_rms_factor(a, b, qi);
  load(t);
  if (listed) slots_of(t + KW);

  // The lane's offsets in a tile, k_off and v_off with their exclusive-ors
  // taken apart: K fragment ks at kfrag0 ^ (ks << 5); V^T fragment (ks, dt, p),
  // keys 16 ks + 4 half + 8 p + (lane % 16) / 4, d = 32 dt + 16 ((lane / 16) %
  // 2) + 4 (lane % 4), at (vfrag0 ^ (dt << 6)) + 4096 ks + 2048 p; the row
  // chunk that load i writes at (krow0 ^ ((qw NLD + i) % 4 << 6)) + 1024 i for
  // K and vrow + 1024 i for V.
  const int tr_i = lane & 15, tr_gh = (lane >> 4) & 1;
  const int kfrag0 = k_off(l32, half), vfrag0 = v_off(4 * half + (tr_i >> 2), 2 * tr_gh + ((tr_i & 3) >> 1)) + (tr_i & 1) * 8;
  const int krow0 = lrow * 256 + ((pch ^ (lane >> 4)) << 4), vrow = v_off(lrow, pch);
  float m_run = kNoMax, l_run = 0.f;
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x16{};
  const int iters = (t1 - t0 + KW - 1) / KW;
  for (int it = 0; it < iters; ++it, t += KW) {
    const int stage = (QW > 1 && (it & 1) ? kStage : 0) + kw * 2 * kFewTile;
    // opaque once per tile: the lane's offsets are a few exclusive-ors away
    // and would otherwise be held in 30 registers across the loop
    int kfrag = kfrag0, vfrag = vfrag0, krow = krow0;
    asm volatile("" : "+v"(kfrag), "+v"(vfrag), "+v"(krow));
    const Tile x = next;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      *reinterpret_cast<u32x4*>(lds + stage + (krow ^ (((qw * NLD + i) & 3) << 6)) + i * 1024) = kr[i];
      *reinterpret_cast<u32x4*>(lds + stage + kFewTile + vrow + i * 1024) = vr[i];
    }
    load(t + KW);
    if (listed) slots_of(t + 2 * KW);
    if constexpr (QW > 1) __syncthreads();  // the tile is whole; the other stage's readers are past it
    if (t >= t1) continue;
    const bool mine = !GROUP || (x.hist ? my_pool : my_own) == x.row;
    if (GROUP && !__builtin_amdgcn_ballot_w64(mine)) continue;
    // K fragments four ahead of their MFMAs.
    constexpr int KA = 4;
    f32x16 s = f32x16{};
    bf16x8 kf[8];
    auto kload = [&](int ks) { kf[ks] = ld_bf16x8(lds + stage + (kfrag ^ (ks << 5))); };
#pragma unroll
    for (int ks = 0; ks < KA; ++ks) kload(ks);
    __builtin_amdgcn_sched_group_barrier(0x100, KA, 0);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      if (ks + KA < 8) kload(ks + KA);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], qf[ks], s, 0, 0, 0);
      if (ks + KA < 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    if (x.key0 + kFewKeys > x.n || GROUP) {
      const int last = mine ? x.n - x.key0 - 4 * half : 0;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (8 * (v >> 2) + (v & 3) >= last) s[v] = -INFINITY;
    }
    // Lazy rescaling as in attention_kernel: the running max (log2 units,
    // equal in both lane halves of a query) moves by more than 8 or not at
    // all.  It stays at kNoMax while the query has seen scores of -inf only
    // (another row's keys among them), whose weights are then zeros.
    float mx = max3(max3(max3(s[0], s[1], s[2]), max3(s[3], s[4], s[5]), max3(s[6], s[7], s[8])),
                    max3(s[9], s[10], s[11]), max3(max3(s[12], s[13], s[14]), s[15], s[15]));
    if (__builtin_amdgcn_ballot_w64(mx * sc > m_run + 8.0f)) {
      const float mt = fmaxf(mx, __shfl_xor(mx, 32, 64)) * sc;
      const bool grow = mt > m_run + 8.0f;
      const float m_new = grow ? mt : m_run;
      const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
      m_run = m_new;
    }
    bf16x8 pb[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      pb[v >> 3][v & 7] = static_cast<bf16>(__builtin_amdgcn_exp2f(s[v] * sc - m_run));
    }
    // the sum of the weights O accumulates
    const bf16x2 one = {static_cast<bf16>(1.f), static_cast<bf16>(1.f)};
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int v = 0; v < 8; v += 2) {
      l0 = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{pb[0][v], pb[0][v + 1]}, one, l0, false);
      l1 = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{pb[1][v], pb[1][v + 1]}, one, l1, false);
    }
    l_run += l0 + l1;
    // V^T fragments (two transposed reads each), VA ahead of their MFMAs.
    auto vload = [&](int i) {
      const int ks = i >> 2, dt = i & 3;
      bf16x8 va;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const bf16x4 t4 = ld_tr16(lds + stage + kFewTile + (vfrag ^ (dt << 6)) + ks * 4096 + p * 2048);
        va[4 * p + 0] = t4[0]; va[4 * p + 1] = t4[1];
        va[4 * p + 2] = t4[2]; va[4 * p + 3] = t4[3];
      }
      return va;
    };
    if constexpr (GROUP) {
      // Queries of another row must not see this one's values at all, not
      // even times zero (infinities): the tile's sum is formed apart and
      // added for its own queries only.  (For every tile: a second path for
      // the tiles that all queries share made the allocator copy O and spill.)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        f32x16 u = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vload(dt), pb[0], f32x16{}, 0, 0, 0);
        u = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vload(4 + dt), pb[1], u, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] += mine ? u[v] : 0.f;
      }
      continue;
    }
    constexpr int VA = 3;
    bf16x8 vf[VA + 1];
#pragma unroll
    for (int i = 0; i < VA; ++i) vf[i] = vload(i);
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * VA, 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i + VA < 8) vf[(i + VA) % (VA + 1)] = vload(i + VA);
      o[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % (VA + 1)], pb[i >> 2], o[i & 3], 0, 0, 0);
      if (i + VA < 8) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  }

  // Merge over the KW key waves of a query block: each wave scales its O by
  // 2^(m - max m), the rows [query][d] go through LDS (16-byte chunks
  // XOR-swizzled by the query) and are summed.  A wave without a tile has m =
  // kNoMax, l = 0, O = 0.
  const float l = l_run + __shfl_xor(l_run, 32, 64);
  if (half == 0) {
    s_ml[0][wave][l32] = m_run;
    s_ml[1][wave][l32] = l;
  }
  __syncthreads();
  float m = kNoMax, den = 0.f;
#pragma unroll
  for (int w = 0; w < KW; ++w) m = fmaxf(m, s_ml[0][w * QW + qw][l32]);
#pragma unroll
  for (int w = 0; w < KW; ++w) den += __builtin_amdgcn_exp2f(s_ml[0][w * QW + qw][l32] - m) * s_ml[1][w * QW + qw][l32];
  const float scale = __builtin_amdgcn_exp2f(m_run - m);
  const float f = ranges > 1 ? scale : scale / den;
  char* const ob = lds + wave * 2 * kFewTile;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int c = 8 * dt + 2 * g + half;  // d = 4 c
      *reinterpret_cast<f32x4*>(ob + l32 * 512 + ((c ^ l32) << 4)) =
          f32x4{o[dt][4 * g] * f, o[dt][4 * g + 1] * f, o[dt][4 * g + 2] * f, o[dt][4 * g + 3] * f};
    }
  __syncthreads();
#pragma unroll
  for (int i = tid; i < QB * 32; i += 64 * kFewWaves) {
    const int ql = i >> 5, c = i & 31, q32 = ql & 31;
    f32x4 v = f32x4{};
#pragma unroll
    for (int w = 0; w < KW; ++w)
      v += *reinterpret_cast<const f32x4*>(lds + (w * QW + (ql >> 5)) * 2 * kFewTile + q32 * 512 + ((c ^ q32) << 4));
    const int row = qb * QB + ql;
    if (row >= nq) continue;
    if (ranges > 1) {
      *reinterpret_cast<f32x4*>(part + (((int64_t)range * units + unit) * QB + ql) * kAttnHD + 4 * c) = v;
    } else {
      bf16x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = static_cast<bf16>(v[e]);
      const int rb = row / a.Mq;
      *reinterpret_cast<bf16x4*>(static_cast<bf16*>(a.o) + (int64_t)(b0 + rb) * a.o_bstride +
                                 (int64_t)(row - rb * a.Mq) * a.o_rstride + h * kAttnHD + 4 * c) = r;
    }
  }
  if (ranges > 1 && kw == 0 && half == 0 && vq < nq) {
    float* ml = part + (int64_t)ranges * units * QB * kAttnHD + (((int64_t)range * units + unit) * QB + qw * 32 + l32) * 2;
    *reinterpret_cast<float2*>(ml) = make_float2(m, den);
  }
}

// The tile ranges' partial results of each query row, merged: one wave per
// row, two of the 128 outputs per lane, every range's loads issued together.
__global__ __launch_bounds__(256) void few_combine_kernel(wam_attention_args a, int G, int QB, int units, int ranges,
                                                          const float* __restrict__ part) {
  const int lane = threadIdx.x & 63;
  const int64_t rows = (int64_t)units * QB, row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int unit = (int)(row / QB), ql = (int)(row - (int64_t)unit * QB);
  const int nq = G * a.Mq, nqb = (nq + QB - 1) / QB, groups = a.B / G;
  const int gh = unit / nqb, vq = (unit % nqb) * QB + ql;
  if (vq >= nq) return;
  const int bl = vq / a.Mq, b = (gh % groups) * G + bl, h = gh / groups;
  const float* ml = part + (int64_t)ranges * rows * kAttnHD;
  float2 mlv[kFewMaxRanges], ov[kFewMaxRanges];
#pragma unroll
  for (int i = 0; i < kFewMaxRanges; ++i) {
    const int64_t at = (int64_t)min(i, ranges - 1) * rows + row;
    mlv[i] = *reinterpret_cast<const float2*>(ml + at * 2);
    ov[i] = *reinterpret_cast<const float2*>(part + at * kAttnHD + 2 * lane);
    if (i >= ranges) mlv[i] = make_float2(-INFINITY, 0.f);
  }
  float m = -INFINITY, den = 0.f, n0 = 0.f, n1 = 0.f;
#pragma unroll
  for (int i = 0; i < kFewMaxRanges; ++i) m = fmaxf(m, mlv[i].x);
#pragma unroll
  for (int i = 0; i < kFewMaxRanges; ++i) {
    const float w = mlv[i].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mlv[i].x - m);
    den += w * mlv[i].y;
    n0 += w * ov[i].x;
    n1 += w * ov[i].y;
  }
  const float inv = 1.f / den;
  bf16x2 r;
  r[0] = static_cast<bf16>(n0 * inv);
  r[1] = static_cast<bf16>(n1 * inv);
  *reinterpret_cast<bf16x2*>(static_cast<bf16*>(a.o) + (int64_t)b * a.o_bstride +
                             (int64_t)(vq - bl * a.Mq) * a.o_rstride + h * kAttnHD + 2 * lane) = r;
}

// (64-bit: the size query and the plan take any shape, a launch has at most a
// dispatch round of units)
static int64_t few_units(int qw, int group, int B, int Mq, int H) {
  return ((int64_t)group * Mq + 32 * qw - 1) / (32 * qw) * (B / group) * H;
}

int64_t attention_few_bytes(const FewPlan& p, int B, int Mq, int H) {
  return p.ranges > 1 ? p.ranges * few_units(p.qw, p.group, B, Mq, H) * 32 * p.qw * (kAttnHD + 2) * 4 : 0;
}

// The workgroups must fit one dispatch round (one per CU): more queries per
// workgroup while they do not, more key ranges while CUs are left and the
// keys are long enough to pay for the merge.  Time per tile round (8, 4 or 2
// tiles with 1, 2 or 4 query waves) and of the merge as measured, 24 heads,
// against 256-query units with their own splits (us, launches included):
//   2 x 16 queries, 304 keys   13.4 -> 8.9      14 x 16, 1168 keys  47 -> 29
//   2 x 16, 512 shared keys    13.5 -> 10.2     14 x 16, 512 shared 24 -> 11
//   2 x 128, 512 shared        20.2 -> 11.1     780, 780 keys       36 -> 24
//   1024 (12 heads), 1024      28.3 -> 19.9     780, 512            31 -> 18
//   16, 6016 keys (8 ranges)   28.4 -> 19.7     1560, 512           22 -> 35 (not taken)
// Batch rows of one pool row may be grouped as far as a wave's 32 queries
// (g divides B), which reads their history once and leaves CUs for more
// workgroups or key ranges.  A group that straddles two pool rows (g does not
// divide the rows per pool row: 7 in pairs) has twice the history, and the
// masks of other rows' keys make a round 2.3 us instead of 2: one workgroup
// per row where that fits a dispatch round and the keys are not many.  16
// queries a row, 24 heads, all slots valid (us: in pairs, one by one, and the
// 256-query units):
//   8 rows of 2, 1333 slots   24.9  20.1  31.8     10 rows of 2, 1333  33.3  20.1  32.0
//   8 rows of 2, 6000 slots   53.4  61.8 113       4 rows of 1, 6000   29.4  37.0  74.4
//   14 rows of 2, 1168 slots  30 (336 rows x heads do not fit one by one)
// Plans go by the pool's slots, whatever is valid of them: over 16 valid ones
// of 1333 one by one takes 7.2 us, in pairs 8.8, the units 5.9, and ranges,
// whose merge does not depend on the keys, 13.6 (8 rows of 2, 3000 slots);
// from a third of the slots on all of these are faster than the units.
FewPlan attention_few_plan(int B, int Mq, int H, int64_t keys, int sharing, int64_t max_bytes) {
  const int cus = device_cu_count();
  FewPlan best{0, 1, 1, 1e30};
  if (B < 1 || Mq < 1 || B > (1 << 20) || Mq > 128 * cus || keys > (1 << 24)) return best;
  const int tiles = (int)((keys + kFewKeys - 1) / kFewKeys);
  for (int qw = 1; qw <= 4; qw *= 2) {
    if (qw > 1 && Mq <= 16 * qw) continue;
    for (int g = 1; g == 1 || (qw == 1 && g <= kFewGroupMax && g <= sharing && g * Mq <= 32); ++g) {
      const int64_t units = few_units(qw, g, B, Mq, H);
      if (B % g != 0 || units > cus) continue;
      // the largest group's tiles (own rows of few keys: a tile each)
      const int most = g > 1 ? tiles * (sharing % g != 0 ? 2 : 1) + g - 1 : tiles;
      const double per = qw == 4 ? 1.16 : (qw == 2 ? 1.45 : (g > 1 ? 2.3 : 2.0));
      for (int r = 1; r <= kFewMaxRanges && units * r <= cus; ++r) {
        if (r > 1 && r * kFewWaves / qw > tiles) break;
        const FewPlan p{qw, g, r, 0};
        const int64_t bytes = attention_few_bytes(p, B, Mq, H);
        if (bytes > max_bytes) break;
        const int rounds = ((most + r - 1) / r + kFewWaves / qw - 1) / (kFewWaves / qw);
        const double cost = 8.3 + (g > 1 ? 1.0 : 0.0) + rounds * per + (r > 1 ? 6.0 + 0.45e-6 * (double)bytes : 0.0);
        if (cost < best.cost - 1e-9) best = FewPlan{qw, g, r, cost};
      }
    }
  }
  return best;
}

int attention_few(const wam_attention_args* a, const FewPlan& p, float* part, hipStream_t s) {
  const int QB = 32 * p.qw, units = (int)few_units(p.qw, p.group, a->B, a->Mq, a->H);
  const dim3 grid((unsigned)(units * p.ranges)), block(64 * kFewWaves);
  auto kernel = p.qw == 4   ? attention_few_kernel<4, false>
                : p.qw == 2 ? attention_few_kernel<2, false>
                : p.group > 1 ? attention_few_kernel<1, true> : attention_few_kernel<1, false>;
  hipLaunchKernelGGL(kernel, grid, block, 0, s, *a, p.group, units, p.ranges, part);
  WAM_LAUNCHED("attention_few_kernel");
  if (p.ranges > 1) {
    const int64_t rows = (int64_t)units * QB;
    hipLaunchKernelGGL(few_combine_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, *a, p.group, QB, units,
                       p.ranges, static_cast<const float*>(part));
    WAM_LAUNCHED("few_combine_kernel");
  }
  return WAM_OK;
}

}  // namespace wam
