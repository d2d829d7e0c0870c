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
// nothing makes one exchange through LDS.
template <int T>
__device__ inline void kv_layout_pool(const wam_kv_layout_args& a) {
  constexpr int W = T / 64, CH = kLayoutSlots * W, CPL = CH / 64, G = T > 256 ? 8 : 16, BINS = 256;
  __shared__ __attribute__((aligned(16))) int sh_cnt[CH];
  __shared__ __attribute__((aligned(16))) int sh_hist[BINS];
  __shared__ long long sh_id[W];
  __shared__ int sh_bad[W], sh_n[W], sh_first[W], sh_last[W];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int P = a.pool, nj = (P + T - 1) / T;
  const bool cand = a.candidate != 0;

  bool bad = false;
  if (cand)
    for (int b = tid; b < a.batch; b += T) bad |= a.rows[b] < 0 || a.rows[b] >= a.pool_batch;
  // Valid flags and the largest valid id: G slots' loads in flight together,
  // through buffer resources (a 32-bit offset each; zeros past the pool's
  // end).
  const __amdgpu_buffer_rsrc_t rmask = make_rsrc(a.mask, (uint32_t)P), rids = make_rsrc(a.ids, (uint32_t)P * 8);
  auto load_id = [&](int j) {
    return __builtin_bit_cast(long long, __builtin_amdgcn_raw_buffer_load_b64(rids, (j * T + tid) * 8, 0, 0));
  };
  uint32_t bits = 0;  // bit j: slot j T + tid is valid
  long long mx = -1, id[G];
  for (int j0 = 0; j0 < nj; j0 += G) {
    uint8_t m[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      m[j] = __builtin_amdgcn_raw_buffer_load_b8(rmask, (j0 + j) * T + tid, 0, 0);
      id[j] = cand ? 0 : load_id(j0 + j);
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const bool v = m[j] != 0;
      bits |= v ? 1u << ((j0 + j) & 31) : 0u;
      mx = v && id[j] > mx ? id[j] : mx;
    }
  }
  bad = __ballot(bad) != 0;
  if (!cand) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const long long y = __shfl_xor(mx, o, 64);
      mx = y > mx ? y : mx;
    }
  }
  if (lane == 0) {
    sh_id[w] = mx;
    sh_bad[w] = bad;
  }

  // Chunk counts of a flag word, exchanged: every wave scans all of them (CPL
  // chunks a lane).  before(j): flags in the chunks before this wave's j-th,
  // which is the (w % CPL)-th chunk of lane 2 j + w / CPL.  A barrier parts
  // one scan's reads from the next one's writes.
  static_assert(W == 2 * CPL, "a wave's chunks have one place in their lanes");
  int excl = 0, total = 0;
  auto scan = [&](uint32_t flags) {
    int first = P, last = -1;  // flagged slots of this wave
    for (int j = 0; j < nj; ++j) {
      const unsigned long long b = __ballot((flags >> j) & 1u);
      if (lane == 0) sh_cnt[j * W + w] = __popcll(b);
      if (b) {
        const int at = j * T + w * 64;
        first = last < 0 ? at + __builtin_ctzll(b) : first;
        last = at + 63 - __builtin_clzll(b);
      }
    }
    if (lane == 0) {
      sh_first[w] = first;
      sh_last[w] = last;
    }
    __syncthreads();
    int n[CPL], x = 0, mine = 0;  // the lane's flags, and those before its (w % CPL)-th chunk
#pragma unroll
    for (int i = 0; i < CPL; ++i) n[i] = sh_cnt[CPL * lane + i];  // (past the pool: not written, not counted)
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      n[i] = CPL * lane + i < nj * W ? n[i] : 0;
      mine += i < w % CPL ? n[i] : 0;
      x += n[i];
    }
    const int own = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      x += lane >= o ? y : 0;
    }
    excl = x - own + mine;
    total = __builtin_amdgcn_readlane(x, 63);
  };
  auto before = [&](int j) { return __builtin_amdgcn_readlane(excl, 2 * j + w / CPL); };
  auto below = [&](unsigned long long b) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
  };

  scan(bits);
#pragma unroll
  for (int i = 0; i < W; ++i) {
    mx = sh_id[i] > mx ? sh_id[i] : mx;
    bad |= sh_bad[i] != 0;
  }
  int error = cand && bad ? 2 : 0;
  // Eviction of the oldest ids (allocate_slots).
  int need = cand ? 0 : a.tokens - (P - total);
  if (need > 0) {
    // fn(slot's bit or 0, its id) for each of the thread's slots.  The larger
    // workgroup has up to G ids per thread in registers still; in the smaller
    // one, part of a row pass, they would cost that pass a wave per SIMD.
    auto each = [&](auto fn) {
      for (int j0 = 0; j0 < nj; j0 += G) {
        long long e[G];
#pragma unroll
        for (int j = 0; j < G; ++j) e[j] = T > 256 && nj <= G ? id[j] : load_id(j0 + j);
#pragma unroll
        for (int j = 0; j < G; ++j) fn(bits & (1u << ((j0 + j) & 31)), e[j]);
      }
    };
    auto free_slot = [&](int j) {
      bits &= ~(1u << j);
      a.mask[j * T + tid] = 0;
      a.ids[j * T + tid] = -1;
    };
    auto count = [&](uint32_t flags) {
      int c = __popc(flags);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
      if (lane == 0) sh_n[w] = c;
      __syncthreads();
      c = 0;
#pragma unroll
      for (int i = 0; i < W; ++i) c += sh_n[i];
      return __builtin_amdgcn_readfirstlane(c);
    };
    // The first n of the c flagged slots.  (A place in the order is needed
    // only where a chunk goes in part.)
    auto evict = [&](uint32_t flags, int c, int n) {
      if (c > n) scan(flags);
      for (int j = 0; j < nj; ++j) {
        const bool f = (flags >> j) & 1u;
        if (c > n) {
          const int pos = before(j) + below(__ballot(f));
          if (f && pos < n) free_slot(j);
        } else if (f) {
          free_slot(j);
        }
      }
    };
    // The smallest id, which is all of it when one chunk makes room.
    long long mn = 0x7fffffffffffffffLL;
    uint32_t eq = 0;  // this thread's slots with its smallest id
    each([&](uint32_t bit, long long i) {
      eq = bit && i < mn ? bit : (bit && i == mn ? eq | bit : eq);
      mn = bit && i < mn ? i : mn;
    });
    const long long own = mn;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const long long y = __shfl_xor(mn, o, 64);
      mn = y < mn ? y : mn;
    }
    __syncthreads();
    if (lane == 0) sh_id[w] = mn;
    for (int i = tid; i < BINS; i += T) sh_hist[i] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; ++i) mn = sh_id[i] < mn ? sh_id[i] : mn;
    eq = own == mn ? eq : 0u;
    int flagged = count(eq);
    if (need > total) {  // not enough valid slots: the host checks make this unreachable
      error = 1;
      need = total;
    }
    if (need > flagged) {
      // More ids: the id of the last slot to go, 8 bits of its distance from
      // the smallest at a time, by a count of the slots per digit; then all
      // slots below it, and its own in ascending order.  1024 threads, 784
      // slots of 1, 2, 3, 14 and 49 ids out of 6240 (us a call, 7 of them for
      // restoring the state): a round per id 20, 23, 27, 51 and 132, now 18,
      // 22, 23, 23 and 25; 309 ids out of 2361: 720, now 22.
      const uint64_t range = (uint64_t)mx - (uint64_t)mn;
      uint64_t key = 0;
      const int top = 64 - __builtin_clzll(range);  // (two ids at least: range > 0)
      for (int shift = top; shift > 0;) {
        const int up = shift, digit = up < 8 ? up : 8;
        shift -= digit;
        if (up < top) {
          __syncthreads();
          for (int i = tid; i < BINS; i += T) sh_hist[i] = 0;
          __syncthreads();
        }
        each([&](uint32_t bit, long long i) {
          const uint64_t k = (uint64_t)i - (uint64_t)mn;
          const bool v = bit && (up == 64 || k >> (up & 63) == key);
          const int bin = (int)(k >> shift) & ((1 << digit) - 1);
          // 64 slots in a row mostly hold one id: one lane adds for all
          const unsigned long long any = __ballot(v);
          if (!any) return;
          const int lead = __builtin_ctzll(any), b0 = __builtin_amdgcn_readlane(bin, lead);
          const unsigned long long same = __ballot(v && bin == b0);
          if (lane == lead) atomicAdd(&sh_hist[b0], __popcll(same));
          else if (v && bin != b0) atomicAdd(&sh_hist[bin], 1);
        });
        __syncthreads();
        // the digit whose slots hold the need-th, in every wave
        static_assert(BINS == 4 * 64, "four digits a lane");
        int c[5], x = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) x += c[i + 1] = sh_hist[4 * lane + i];
        const int sum = x;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int y = __shfl_up(x, o, 64);
          x += lane >= o ? y : 0;
        }
        c[0] = x - sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i + 1] += c[i];
        const int i = need <= c[1] ? 0 : (need <= c[2] ? 1 : (need <= c[3] ? 2 : 3));
        const int less = i == 0 ? c[0] : (i == 1 ? c[1] : (i == 2 ? c[2] : c[3]));
        const int at = __builtin_ctzll(__ballot(c[0] < need && need <= c[4]));
        key = key << digit | (uint64_t)__builtin_amdgcn_readlane(4 * lane + i, at);
        need -= __builtin_amdgcn_readlane(less, at);
      }
      eq = 0;
      uint32_t lower = 0;
      each([&](uint32_t bit, long long i) {
        const uint64_t k = (uint64_t)i - (uint64_t)mn;
        eq |= k == key ? bit : 0u;
        lower |= k < key ? bit : 0u;
      });
      for (int j = 0; j < nj; ++j)
        if ((lower >> j) & 1u) free_slot(j);
      flagged = count(eq);
    }
    evict(eq, flagged, need);
    __syncthreads();
    scan(bits);
  }
  // Next id over the remaining valid slots (_next_cache_id), the history list
  // and the new slots, both in ascending slot order.
  const long long next = total > 0 ? mx + 1 : 0;
  for (int j = 0; j < nj; ++j) {
    const int slot = j * T + tid;
    const bool v = (bits >> j) & 1u;
    const int pv = before(j) + below(__ballot(v));
    if (v) {
      a.hist_slots[pv] = slot;
    } else if (!cand && slot < P && slot - pv < a.tokens) {
      a.new_slots[slot - pv] = slot;
      a.mask[slot] = a.update != 0 ? 1 : 0;
      a.ids[slot] = next;
      a.is_pred[slot] = a.update == 1 ? 1 : 0;
    }
  }
  if (tid == 0) {
    int first = P, last = -1;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      first = min(first, sh_first[i]);
      last = max(last, sh_last[i]);
    }
    a.info[0] = total;
    a.info[1] = error;
    a.info[2] = total > 0 && last - first + 1 == total ? first : -1;
  }
}

// Whether the bookkeeping runs as a workgroup of 256 threads of the q/k row
// pass.  That pass in us with it, 2 x 16 rows (alone 4):
//   slots  read only  none evicted  one id  three ids
//    2288     4.2         5.9         9.6     16
//    4096     6.1         7.2        10.8     19
//    6240     8.0         9.2        14.6     31
// A launch of its own (1024 threads) adds its gap and, at 6240 slots, 5, 6.2,
// 12.6 and 20 us: pools that may evict take that beyond 16 slots per thread,
// read-only ones ride as far as the flags fit.
inline bool kv_layout_rides(int pool, bool candidate) { return pool <= (candidate ? kLayoutSlots : 16) * 256; }

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
