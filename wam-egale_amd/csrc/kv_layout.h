// The KV pool's bookkeeping by one workgroup, for pools of up to
// kLayoutSlots slots per thread (what it computes: kv_cache.hip).
#pragma once
#include "wam_common.h"

namespace wam {

constexpr int kLayoutSlots = 32;  // slots of a thread, their valid flags the bits of one word

// T threads; slot = j T + thread, so a wave's slots of one j are 64 in a row
// (a chunk): loads and list writes are coalesced, and a slot's place in the
// ascending lists is the valid count of the chunks before it, plus the bits
// below its own in the chunk's ballot.  Free slots need no scan of their own
// (a slot has slot - (valid before it) free ones before it), and evicting
// smallest ids first leaves the largest id in place, so a call that evicts
// nothing makes one exchange through LDS.  (Runs of slots per thread, and a
// block scan or reduction of its own for each of the five results, took 9.5
// to 11 us a call in a block at 6240 slots.)
template <int T>
__device__ inline void kv_layout_pool(const wam_kv_layout_args& a) {
  constexpr int W = T / 64, CH = kLayoutSlots * W, CPL = CH / 64, G = T > 256 ? 8 : 16;
  __shared__ int sh_cnt[CH];
  __shared__ long long sh_id[W];
  __shared__ int sh_bad[W], sh_run[2];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int P = a.pool, nj = (P + T - 1) / T;
  const bool cand = a.candidate != 0;

  int bad = 0;
  if (cand)
    for (int b = tid; b < a.batch; b += T) bad |= (a.rows[b] < 0 || a.rows[b] >= a.pool_batch) ? 1 : 0;
  // Valid flags and the largest valid id: G slots' loads in flight together.
  uint32_t bits = 0;  // bit j: slot j T + tid is valid
  long long mx = -1;
  for (int j0 = 0; j0 < nj; j0 += G) {
    uint8_t m[G];
    long long id[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int slot = min((j0 + j) * T + tid, P - 1);
      m[j] = a.mask[slot];
      id[j] = cand ? 0 : (long long)a.ids[slot];
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const bool v = (j0 + j) * T + tid < P && m[j] != 0;
      bits |= v ? 1u << ((j0 + j) & 31) : 0u;
      mx = v && id[j] > mx ? id[j] : mx;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const long long y = __shfl_xor(mx, o, 64);
    mx = y > mx ? y : mx;
    bad |= __shfl_xor(bad, o, 64);
  }
  if (lane == 0) {
    sh_id[w] = mx;
    sh_bad[w] = bad;
  }

  // Chunk counts of a flag word, exchanged: every wave scans all of them (CPL
  // chunks a lane).  before(j): flags in the chunks before this wave's j-th,
  // which is the (w % CPL)-th chunk of lane 2 j + w / CPL.
  static_assert(W == 2 * CPL, "a wave's chunks have one place in their lanes");
  int excl = 0, total = 0;
  auto scan = [&](uint32_t flags) {
    for (int j = 0; j < nj; ++j) {
      const int n = __popcll(__ballot((flags >> j) & 1u));
      if (lane == 0) sh_cnt[j * W + w] = n;
    }
    __syncthreads();
    int x = 0, mine = 0;  // the lane's flags, and those before its (w % CPL)-th chunk
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const int n = CPL * lane + i < nj * W ? sh_cnt[CPL * lane + i] : 0;
      mine += i < w % CPL ? n : 0;
      x += n;
    }
    const int own = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      x += lane >= o ? y : 0;
    }
    excl = x - own + mine;
    total = __builtin_amdgcn_readlane(x, 63);
    __syncthreads();
  };
  auto before = [&](int j) { return __builtin_amdgcn_readlane(excl, 2 * j + w / CPL); };
  auto below = [&](unsigned long long b) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
  };

  scan(bits);
#pragma unroll
  for (int i = 0; i < W; ++i) {
    mx = sh_id[i] > mx ? sh_id[i] : mx;
    bad |= sh_bad[i];
  }
  int error = cand && bad ? 2 : 0;
  // Eviction of the oldest ids (allocate_slots), one id a round.
  int need = cand ? 0 : a.tokens - (P - total);
  if (need > 0) {
    while (need > 0) {
      long long mn = 0x7fffffffffffffffLL;
      uint32_t eq = 0;  // this thread's slots with its smallest id
      for (int j0 = 0; j0 < nj; j0 += G) {
        long long id[G];
#pragma unroll
        for (int j = 0; j < G; ++j) id[j] = (long long)a.ids[min((j0 + j) * T + tid, P - 1)];
#pragma unroll
        for (int j = 0; j < G; ++j) {
          const uint32_t bit = bits & (1u << ((j0 + j) & 31));
          eq = bit && id[j] < mn ? bit : (bit && id[j] == mn ? eq | bit : eq);
          mn = bit && id[j] < mn ? id[j] : mn;
        }
      }
      const long long own = mn;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const long long y = __shfl_xor(mn, o, 64);
        mn = y < mn ? y : mn;
      }
      __syncthreads();
      if (lane == 0) sh_id[w] = mn;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < W; ++i) mn = sh_id[i] < mn ? sh_id[i] : mn;
      eq = own == mn ? eq : 0u;
      scan(eq);
      for (int j = 0; j < nj; ++j) {
        const bool oldest = (eq >> j) & 1u;
        const int pos = before(j) + below(__ballot(oldest));
        if (oldest && pos < need) {
          bits &= ~(1u << j);
          a.mask[j * T + tid] = 0;
          a.ids[j * T + tid] = -1;
        }
      }
      need -= total;
      if (total == 0) {  // no valid slot left to evict: the host checks make this unreachable
        error = 1;
        break;
      }
    }
    scan(bits);
  }
  // Next id over the remaining valid slots (_next_cache_id), the history list
  // and the new slots, both in ascending slot order.
  const long long next = total > 0 ? mx + 1 : 0;
  if (tid == 0) sh_run[0] = sh_run[1] = 0;
  __syncthreads();
  for (int j = 0; j < nj; ++j) {
    const int slot = j * T + tid;
    const bool v = (bits >> j) & 1u;
    const int pv = before(j) + below(__ballot(v));
    if (v) {
      a.hist_slots[pv] = slot;
      if (pv == 0) sh_run[0] = slot;
      if (pv == total - 1) sh_run[1] = slot;
    } else if (!cand && slot < P && slot - pv < a.tokens) {
      a.new_slots[slot - pv] = slot;
      a.mask[slot] = a.update != 0 ? 1 : 0;
      a.ids[slot] = next;
      a.is_pred[slot] = a.update == 1 ? 1 : 0;
    }
  }
  __syncthreads();
  if (tid == 0) {
    a.info[0] = total;
    a.info[1] = error;
    a.info[2] = total > 0 && sh_run[1] - sh_run[0] + 1 == total ? sh_run[0] : -1;
  }
}

// New K/V rows to their pool slots, 16 bytes a thread and step, by `blocks`
// workgroups of T threads.
template <int T>
__device__ inline void kv_commit_rows(const wam_kv_commit_args& a, int block, int blocks) {
  const int chunks = a.D >> 3;
  const int64_t n = (int64_t)a.B * a.tokens * chunks;
  for (int64_t i = (int64_t)block * T + threadIdx.x; i < n; i += (int64_t)blocks * T) {
    int64_t row, cc;
    split_row(i, chunks, row, cc);  // i < 2^31: B * tokens * D / 8 elements
    const int c = (int)cc;
    int64_t b, t;
    split_row(row, a.tokens, b, t);
    const int64_t src = row * a.ld + c * 8;
    const int64_t dst = b * a.pool_bstride + (int64_t)a.new_slots[t] * a.pool_rstride + c * 8;
    st_bf16x8(static_cast<bf16*>(a.pool_k) + dst, ld_bf16x8(static_cast<const bf16*>(a.k) + src));
    st_bf16x8(static_cast<bf16*>(a.pool_v) + dst, ld_bf16x8(static_cast<const bf16*>(a.v) + src));
  }
}

}  // namespace wam
