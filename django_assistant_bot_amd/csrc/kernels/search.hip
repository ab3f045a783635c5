// The small steps around the index scan: unit-length query rows, the threshold of a search from the scores of
// the row sample, the ranking of the candidates, and the ids / documents of the hits.  (The search they belong to
// replaces pgvector's CosineDistance ORDER BY ... LIMIT: reference rag/services/search_service.py:185-196.)
//
// All of them are chains of a few memory round trips on little data, so what counts is one launch each and no
// host round trip between them: the ranking reads the candidate counts on the device and says in a status word
// whether the threshold held.
#include <type_traits>

#include "common.h"
#include "launchers.h"
#include "select.h"

namespace dab {

// Values that a search's caller holds on the host, in the launch's arguments: a copy of them is a launch of its own, 4 us
// on the card and some 8 of the host (a search of 109 queries in 6,185 rows of a group 46 -> 37 us).
struct HostGroups {
  int v[kHostValues];
};
struct HostLimits {
  int64_t v[kHostValues];
};
struct NoGroups {};

// x / max(|x|, 1e-12), rounded to bf16.  One workgroup a row (rows are an embedding's width, read twice: L1 / L2).  What else a
// search begins with: the first workgroup writes the queries' groups out of the arguments, those behind the rows clear
// the mask that the lists set bits in (a fill of its own: 3 us, and 5 of the host).  GROUPS: HostGroups, or NoGroups, whose 512 bytes
// of arguments less are 0.4 us of a launch (a search of 2 queries in 202,640 rows 64.8 -> 64.3).
template <typename GROUPS>
__global__ __launch_bounds__(256) void unit_rows_kernel(const float* __restrict__ x, long ldx, bf16* __restrict__ out, int cols, int rows,
                                                        GROUPS groups, int n_groups, int* __restrict__ groups_out,
                                                        uint32_t* __restrict__ clear, long words) {
  __shared__ float red[4];
  if ((int)blockIdx.x >= rows) {  // whole workgroup
    const long w = ((long)((int)blockIdx.x - rows) * 256 + threadIdx.x) * 4;
    for (int i = 0; i < 4; ++i)
      if (w + i < words) clear[w + i] = 0u;
    return;
  }
  if constexpr (std::is_same_v<GROUPS, HostGroups>) {
    if (blockIdx.x == 0 && (int)threadIdx.x < n_groups) groups_out[threadIdx.x] = groups.v[threadIdx.x];
  }
  const float* r = x + (size_t)blockIdx.x * ldx;
  bf16* o = out + (size_t)blockIdx.x * cols;
  float s = 0.f;
  for (int i = threadIdx.x; i < cols; i += 256) s = fmaf(r[i], r[i], s);
  const float norm = fmaxf(sqrtf(block_sum<256>(s, red)), 1e-12f);
  for (int i = threadIdx.x; i < cols; i += 256) o[i] = f2bf(r[i] / norm);
}

// groups: n_groups <= kHostValues ints of the host, written to groups_out; clear: so many words set to zero
int unit_rows(const float* x, long ldx, void* out, int rows, int cols, hipStream_t s, const int* groups, int n_groups, int* groups_out,
              uint32_t* clear, long words) {
  if (rows <= 0) return 0;
  if (cols <= 0 || n_groups < 0 || n_groups > kHostValues || (n_groups && (!groups || !groups_out)) || words < 0 || (words && !clear))
    return hipErrorInvalidValue;
  const long blocks = rows + (words + 1023) / 1024;
  if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks);
  if (!n_groups) {
    hipLaunchKernelGGL(unit_rows_kernel<NoGroups>, grid, dim3(256), 0, s, x, ldx, (bf16*)out, cols, rows, NoGroups{}, 0, nullptr, clear, words);
    return hipGetLastError();
  }
  HostGroups g = {};
  for (int i = 0; i < n_groups; ++i) g.v[i] = groups[i];
  hipLaunchKernelGGL(unit_rows_kernel<HostGroups>, grid, dim3(256), 0, s, x, ldx, (bf16*)out, cols, rows, g, n_groups, groups_out, clear,
                     words);
  return hipGetLastError();
}

constexpr int RV_NT = 1024;
constexpr int RV_MAX = 256;  // maxima ranked: one of every four neighbouring threads
constexpr int RV_CAP = 512;
constexpr int RV_HELD = 4;

// thr[row] = the r-th largest of the row's n scores less `slack` (r <= kRankMax; -inf when r > n), cnt[row] = 0.
//
// The r-th largest of 256 maxima over disjoint parts is a lower bound that at least r scores reach, and with the r
// of a search (7-41 of thousands) only a few more do: those are ranked.  Two looks at the row, the first 16,384 scores
// held in registers between them; ranks by ballots (a wave compares 64 at once, no chain of LDS reads).  15,625 scores
// of one query: 8.6 us, of 128 queries 9.6 (two reads of the row and ranks by LDS loops: 14.5 and 16.5; a radix select's
// four passes with wave-aggregated histograms: 61 and 91).
__global__ __launch_bounds__(RV_NT) void rank_value_kernel(const float* __restrict__ scores, long ld, int n, int r,
                                                           float slack, float* __restrict__ thr, int* __restrict__ cnt) {
  __shared__ uint32_t tmax[RV_MAX];
  __shared__ uint32_t kept[RV_CAP];
  __shared__ uint32_t n_kept, bound;
  __shared__ uint32_t hist[256];
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* s = scores + (size_t)row * ld;
  if (tid == 0) cnt[row] = 0;
  if (r > n) {
    if (tid == 0) thr[row] = -INFINITY;
    return;
  }
  const bool vec = (reinterpret_cast<uintptr_t>(s) & 15) == 0;
  const int n4 = vec ? n / 4 : 0, lane = tid & 63, w = tid >> 6;
  // the first RV_HELD vectors of a thread stay in registers for the second look
  f32x4 held[RV_HELD];
  uint32_t m = 0;
#pragma unroll
  for (int j = 0; j < RV_HELD; ++j) {
    const int i = tid + RV_NT * j;
    if (i < n4) held[j] = reinterpret_cast<const f32x4*>(s)[i];
  }
  const int rest = 4 * n4 < n ? 4 * n4 + tid : n;
  auto each = [&](auto f) {
#pragma unroll
    for (int j = 0; j < RV_HELD; ++j)
      if (tid + RV_NT * j < n4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f(float_key(held[j][e]));
      }
#pragma unroll 4
    for (int i = tid + RV_NT * RV_HELD; i < n4; i += RV_NT) {
      const f32x4 v = reinterpret_cast<const f32x4*>(s)[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) f(float_key(v[e]));
    }
    for (int i = rest; i < n; i += RV_NT) f(float_key(s[i]));
  };
  each([&](uint32_t key) { m = max(m, key); });
  m = max(m, (uint32_t)__shfl_xor((int)m, 1, 64));
  m = max(m, (uint32_t)__shfl_xor((int)m, 2, 64));
  if ((tid & 3) == 0) tmax[tid >> 2] = m;
  if (tid == 0) {
    n_kept = 0;
    bound = 0;
  }
  __syncthreads();
  // rank of maximum a: the waves take 16 each, against all 256 by ballots
  uint32_t all[RV_MAX / 64];
#pragma unroll
  for (int c = 0; c < RV_MAX / 64; ++c) all[c] = tmax[64 * c + lane];
#pragma unroll 4
  for (int j = 0; j < RV_MAX / (RV_NT / 64); ++j) {
    const int a = w * (RV_MAX / (RV_NT / 64)) + j;
    const uint32_t key = tmax[a];
    int rank = 0;
#pragma unroll
    for (int c = 0; c < RV_MAX / 64; ++c)
      rank += __popcll(__ballot(all[c] > key || (all[c] == key && 64 * c + lane < a)));
    if (rank == r - 1 && lane == 0) bound = key;
  }
  __syncthreads();
  const uint32_t t = bound;
  each([&](uint32_t key) {
    if (key >= t) {
      const uint32_t at = atomicAdd(&n_kept, 1u);
      if (at < RV_CAP) kept[at] = key;
    }
  });
  __syncthreads();
  const int nk = (int)n_kept;
  if (nk <= RV_CAP) {
    for (int a = w; a < nk; a += RV_NT / 64) {
      const uint32_t key = kept[a];
      int above = 0, same = 0;  // equal keys share one value: any of them may name it
      for (int c = 0; c < nk; c += 64) {
        const bool in = c + lane < nk;
        const uint32_t o = kept[min(c + lane, nk - 1)];
        above += __popcll(__ballot(in && o > key));
        same += __popcll(__ballot(in && o == key));
      }
      if (lane == 0 && above < r && r <= above + same) thr[row] = key_float(key) - slack;
    }
    return;
  }
  // many equal scores at the bound: radix select, most significant byte first
  uint32_t prefix = 0, mask = 0, need = (uint32_t)r;
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += RV_NT) {
      const uint32_t key = float_key(s[i]);
      if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 255u], 1u);
    }
    __syncthreads();
    uint32_t above = 0, digit = 0;
    for (int d = 255; d >= 0; --d) {  // every thread walks the same bins
      if (above + hist[d] >= need) {
        digit = (uint32_t)d;
        break;
      }
      above += hist[d];
    }
    need -= above;
    prefix |= digit << shift;
    mask |= 255u << shift;
    __syncthreads();
  }
  if (tid == 0) thr[row] = key_float(prefix) - slack;
}

int rank_value(const float* scores, long ld, int rows, int n, int r, float slack, float* thr, int* cnt, hipStream_t s) {
  if (rows <= 0) return 0;
  if (n <= 0 || r < 1 || r > kRankMax) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rank_value_kernel, dim3(rows), dim3(RV_NT), 0, s, scores, ld, n, r, slack, thr, cnt);
  return hipGetLastError();
}

constexpr int RK_SORT = 4096;  // candidates of a list held in LDS
constexpr int RK_BINS = SEL_NT;
constexpr int RK_FEW = 512;    // entries ranked by counting
constexpr int RK_MANY = 2048;  // entries behind the histogram's cut that are held

template <int CAP>
struct RankShared {
  unsigned long long key[CAP];  // ordered bits of the score, ~row
  __attribute__((aligned(16))) unsigned long long few[RK_MANY];
  uint32_t hist[RK_BINS];
  uint32_t rank[RK_FEW];
  uint32_t lo[SEL_NT / 64], hi[SEL_NT / 64], total[SEL_NT / 64];
  uint32_t bin, in_bin, upto, n;
};

// The bin in which the count from the top reaches `kept`, for all threads (the last one where there are fewer entries); in_bin:
// the entries in it, upto: those and the ones above.
template <int CAP>
__device__ __forceinline__ uint32_t cut_bin(RankShared<CAP>& sh, uint32_t kept) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint32_t h = sh.hist[RK_BINS - 1 - tid];
  uint32_t incl = h;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  if (lane == 63) sh.total[w] = incl;
  __syncthreads();
  for (int j = 0; j < w; ++j) incl += sh.total[j];
  if (incl - h < kept && (kept <= incl || tid == RK_BINS - 1)) {
    sh.bin = RK_BINS - 1 - tid;
    sh.in_bin = h;
    sh.upto = incl;
  }
  __syncthreads();
  return sh.bin;
}

// The block's least and greatest value.
template <int CAP>
__device__ __forceinline__ void block_range(RankShared<CAP>& sh, uint32_t& lo, uint32_t& hi) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  lo = wave_fold_bits(lo, [](uint32_t x, uint32_t y) { return min(x, y); });
  hi = wave_fold_bits(hi, [](uint32_t x, uint32_t y) { return max(x, y); });
  if (lane == 0) {
    sh.lo[w] = lo;
    sh.hi[w] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < SEL_NT / 64; ++j) {
    lo = min(lo, sh.lo[j]);
    hi = max(hi, sh.hi[j]);
  }
}

// Shift after which steps of (key - lo) fall into RK_BINS bins: monotone for any scores.  (__clz(0) = 32)
__device__ __forceinline__ int bin_shift(uint32_t lo, uint32_t hi) { return max(0, 22 - __clz(hi - lo)); }

// A bound in lo .. hi that at least `need` of the entries reach (all of them, where they are fewer) and at most `most` (need <=
// most).  each(f) hands this thread's entries to f; those of the block differ from each other (ordered bits << 32 | ~place), so
// the histograms of ever narrower ranges end at the latest with one entry a bin.  Leaves hist cleared.
template <int CAP, typename F>
__device__ __forceinline__ unsigned long long bound_of(RankShared<CAP>& sh, unsigned long long lo, unsigned long long hi,
                                                       uint32_t need, uint32_t most, F each) {
  for (uint32_t above = 0;;) {
    const int shift = max(0, 54 - __clzll((long long)(hi - lo)));  // (hi - lo) >> shift < RK_BINS
    sh.hist[threadIdx.x] = 0;
    __syncthreads();
    each([&](unsigned long long e) {
      const int bin = e >= lo && e <= hi ? (int)((e - lo) >> shift) : -1;
      const unsigned long long in = __ballot(bin >= 0);
      if (!in) return;
      // the lanes of one bin by one atomic: 64 on an address are 64 steps (equal scores)
      const int leader = __ffsll((long long)in) - 1, first = __builtin_amdgcn_readlane(bin, leader);
      const unsigned long long same = __ballot(bin == first);
      if (bin >= 0 && (bin != first || (int)(threadIdx.x & 63) == leader))
        atomicAdd(&sh.hist[bin], bin == first ? (uint32_t)__popcll(same) : 1u);
    });
    __syncthreads();
    const uint32_t bin = cut_bin(sh, need - above);
    lo += (unsigned long long)bin << shift;
    sh.hist[threadIdx.x] = 0;
    if (above + sh.upto <= most || shift == 0) return lo;
    above += sh.upto - sh.in_bin;
    hi = min(hi, lo + ((1ull << shift) - 1));
  }
}

// Bitonic, greatest first; P a power of two, at least 64.  A wave's 64 consecutive pairs lie in its own 128 entries where
// the stride is 64 or less: no workgroup barrier there.
__device__ __forceinline__ void sort_desc(unsigned long long* key, int P) {
  for (int size = 2; size <= P; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int p = threadIdx.x; p < P / 2; p += SEL_NT) {
        const int a = 2 * p - (p & (stride - 1)), b = a + stride;
        const unsigned long long ka = key[a], kb = key[b];
        if ((ka > kb) != ((a & size) == 0)) {
          key[a] = kb;
          key[b] = ka;
        }
      }
      if (stride > 64 || (stride == 1 && size >= 128))
        __syncthreads();  // (the next size's first stride is `size`: across waves from size 128 on)
      else
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // a wave's own LDS operations, in order
    }
  __syncthreads();
}

// sh.key[0 .. c) in any order -> emit(place, entry, id, document) for the `kept` (1 .. c) greatest.  lo, hi: of the entries
// this thread has written; the caller has cleared hist, rank and n and no barrier is due.
template <int CAP, typename F>
__device__ void rank_list(RankShared<CAP>& sh, int c, int kept, uint32_t lo, uint32_t hi, const int64_t* row_ids,
                          const int64_t* row_docs, F emit) {
  const int tid = threadIdx.x;
  block_range(sh, lo, hi);
  const int shift = bin_shift(lo, hi);
  auto bin_of = [&](unsigned long long e) { return ((uint32_t)(e >> 32) - lo) >> shift; };
  for (int i = tid; i < c; i += SEL_NT) atomicAdd(&sh.hist[bin_of(sh.key[i])], 1u);
  __syncthreads();
  const uint32_t least = cut_bin(sh, (uint32_t)kept);
  for (int i = tid; i < c; i += SEL_NT) {
    const unsigned long long e = sh.key[i];
    if (bin_of(e) < least) continue;
    const uint32_t at = atomicAdd(&sh.n, 1u);
    if (at < RK_MANY) sh.few[at] = e;
  }
  __syncthreads();
  int m = (int)sh.n;
  if (m > RK_MANY) {  // (equal scores in one bin): cut among them by their rows
    const unsigned long long bound =
        bound_of(sh, (unsigned long long)lo << 32, ((unsigned long long)hi << 32) | ~0u, (uint32_t)kept,
                 (uint32_t)(kept <= RK_FEW ? RK_FEW : RK_MANY), [&](auto f) __attribute__((always_inline)) {
                   for (int i = tid; i < c; i += SEL_NT) f(sh.key[i]);
                 });
    if (tid == 0) sh.n = 0;
    __syncthreads();
    for (int i = tid; i < c; i += SEL_NT) {
      const unsigned long long e = sh.key[i];
      const int at = wave_append(&sh.n, e >= bound);
      if (at >= 0 && at < RK_MANY) sh.few[at] = e;
    }
    __syncthreads();
    m = (int)sh.n;
  }
  if (m <= RK_FEW) {  // every entry against all m, m / parts of them a thread
    const int E = (m + 63) & ~63, parts = SEL_NT / E, part = tid / E, e = tid - part * E;
    const bool own = part < parts && e < m;
    const unsigned long long mine = own ? sh.few[e] : 0ull;
    int64_t id = 0, doc = 0;
    const uint32_t r = ~(uint32_t)mine;
    if (own && part == 0) {  // (requested ahead of the ranks)
      id = row_ids[r];
      doc = row_docs[r];
    }
    if (own) {
      const int step = (m + 2 * parts - 1) / (2 * parts) * 2, j0 = part * step, j1 = min(m, j0 + step);
      uint32_t above = 0;
      for (int j = j0; j + 1 < j1; j += 2) {
        const u32x4 two = *reinterpret_cast<const u32x4*>(&sh.few[j]);
        above += (((unsigned long long)two[1] << 32) | two[0]) > mine;
        above += (((unsigned long long)two[3] << 32) | two[2]) > mine;
      }
      if (j0 < j1 && ((j1 - j0) & 1)) above += sh.few[j1 - 1] > mine;
      atomicAdd(&sh.rank[e], above);
    }
    __syncthreads();
    if (own && part == 0 && (int)sh.rank[e] < kept) emit((int)sh.rank[e], mine, id, doc);
    return;
  }
  unsigned long long* list = m <= RK_MANY ? sh.few : sh.key;  // (else: a list that names a row more than once)
  const int n = m <= RK_MANY ? m : c;
  int P = 64;
  while (P < n) P <<= 1;
  for (int i = n + tid; i < P; i += SEL_NT) list[i] = 0ull;
  __syncthreads();
  sort_desc(list, P);
  for (int i = tid; i < kept; i += SEL_NT) {
    const uint32_t r = ~(uint32_t)list[i];
    emit(i, list[i], row_ids[r], row_docs[r]);
  }
}

// One row's candidates (unordered, cnt[row] of them) -> its k best: score, item id, document id, best first, equal
// scores in row order (lists above 4096: in the list's, which its appends leave open); -inf / -1 past the last.
// status[row] = 1 where the list cannot be trusted: it overflowed, or it holds fewer than k entries although a threshold cut rows off.
//
// A search's lists hold 1-2 thousand entries for some 250 hits.  A histogram of 1024 bins between the list's least and
// greatest score leaves little more than the hits (bins are equal steps of the ordered bits: monotone for any scores),
// and up to 512 entries are ranked by counting the greater ones: one chain of LDS reads instead of the 66 steps of a
// bitonic sort of the list.  Where more remain (k above some 400, many near-equal scores) they are sorted, up to 2048, or
// cut by score and row to as many first.  Lists above 4096 are radix-selected.  With the ids and documents in the same
// launch 7.9 us for 1,300 candidates of one query and 9.8 for 128 queries (sorted whole: 22 and 31; radix select of 16,000 and five
// element-wise launches behind it: 61 and 91).
__global__ __launch_bounds__(SEL_NT) void rank_hits_kernel(const float* __restrict__ cand_val,
                                                           const int* __restrict__ cand_idx,
                                                           const int* __restrict__ cnt, const float* __restrict__ thr,
                                                           int cap, int k, const int64_t* __restrict__ row_ids,
                                                           const int64_t* __restrict__ row_docs,
                                                           float* __restrict__ out_vals, int64_t* __restrict__ out_ids,
                                                           int64_t* __restrict__ out_docs, int* __restrict__ status) {
  __shared__ union {
    RankShared<RK_SORT> list;
    SelShared sel;
  } sh;
  const int row = blockIdx.x, tid = threadIdx.x;
  const int c = cnt[row];
  const bool bad = c > cap || (c < k && !(thr[row] == -INFINITY));  // (a NaN threshold passes nothing)
  if (tid == 0) status[row] = bad;
  if (bad) return;
  const float* cv = cand_val + (size_t)row * cap;
  const int* ci = cand_idx + (size_t)row * cap;
  out_vals += (size_t)row * k;
  out_ids += (size_t)row * k;
  out_docs += (size_t)row * k;
  const int kept = min(k, c);
  for (int i = kept + tid; i < k; i += SEL_NT) {
    out_vals[i] = -INFINITY;
    out_ids[i] = -1;
    out_docs[i] = -1;
  }
  if (c > RK_SORT) {
    select_topk([&](int i) -> uint32_t { return float_key(cv[i]); }, c, kept, sh.sel);
    for (int i = tid; i < kept; i += SEL_NT) {
      const int r = ci[sh.sel.cand_idx[i]];
      out_vals[i] = key_float(sh.sel.cand_key[i]);
      out_ids[i] = row_ids[r];
      out_docs[i] = row_docs[r];
    }
    return;
  }
  if (kept == 0) return;
  uint32_t lo = ~0u, hi = 0u;
  for (int i = tid; i < c; i += SEL_NT) {
    const uint32_t key = float_key(cv[i]);
    sh.list.key[i] = ((unsigned long long)key << 32) | (uint32_t)~ci[i];
    lo = min(lo, key);
    hi = max(hi, key);
  }
  sh.list.hist[tid] = 0;
  if (tid < RK_FEW) sh.list.rank[tid] = 0;
  if (tid == 0) sh.list.n = 0;
  rank_list(sh.list, c, kept, lo, hi, row_ids, row_docs, [&](int i, unsigned long long e, int64_t id, int64_t doc) {
    out_vals[i] = key_float((uint32_t)(e >> 32));
    out_ids[i] = id;
    out_docs[i] = doc;
  });
}

int rank_hits(const float* cand_val, const int* cand_idx, const int* cnt, const float* thr, int cap, int rows, int k,
              const int64_t* row_ids, const int64_t* row_docs, float* out_vals, int64_t* out_ids, int64_t* out_docs,
              int* status, hipStream_t s) {
  if (rows <= 0) return 0;
  if (k < 1 || k > SEL_MAXK || cap < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rank_hits_kernel, dim3(rows), dim3(SEL_NT), 0, s, cand_val, cand_idx, cnt, thr, cap, k, row_ids,
                     row_docs, out_vals, out_ids, out_docs, status);
  return hipGetLastError();
}

constexpr int TH_CAND = 8192;   // candidates held in LDS, and the scores of a row that need no parts
constexpr int TH_PARTS = 4096;  // parts looked into (4 k at most, or 1024)
constexpr int TH_HELD = 16;     // 16-B vectors of part maxima a thread keeps in registers between its looks
constexpr int TH_FEW = 2;       // threads with a score that passes, as a multiple of k, from which their maxima give the bound

// The k best of every row of scores [n] -> score, item id, document id, best first, equal scores in row order; -inf / -1
// where fewer rows pass the filters.  One workgroup a row; parts: the greatest ordered bits of every 16 scores.
//
// The k-th greatest of maxima over disjoint parts is a bound that at least k scores reach, and where the parts are many
// times k few more do.  So the scores themselves are read only in the parts that reach it: 64 KB of maxima and some 20 KB
// of scores for 250 of 262,144, and the rest is the ranking of about 300 candidates.  The bound is the lower end of a
// bin of a 1024-bin histogram: of the threads' maxima, one atomic each, where 2 k threads have a score that passes, else (k
// above 500, up to 128 k rows, groups that lie together) of the parts' own, (key, place) in as many rounds as leave 2 k or
// 1024 of them.  Where those hold more than 8192 scores that reach it (k near the number of parts, equal scores) the bound is
// raised over these scores in the same way.  Rows of up to 8192 scores are ranked as they are.
//
// us, against a radix select by one workgroup a query (up to 32,768 scores) or selection in chunks and a merge, and the
// ids' launch: 42 queries of 31,098 rows 9.8 (188), 4 of 60,001 9.5 (34), 10 of 142,939 10.1 (40); 1 of 1,000,003 17.3.
// From the parts, against the same: 250 of 12,000 13.8 (54), 500 of 30,000 21 (115), 1000 of 50,000 29 (85), 1024 of 1,000,000
// 75 (244), 250 of 600,000 with 12,000 that pass together 21 (66); all scores equal, 1000 of 60,000 43 (62).  (A row that the
// threads' bound alone did not cut was radix-selected whole by its workgroup: 1024 of 1,000,000 some 2,800.)
__global__ __launch_bounds__(SEL_NT) void top_hits_kernel(const float* __restrict__ scores, int n,
                                                          const uint32_t* __restrict__ parts, int ldp, int k,
                                                          const int64_t* __restrict__ row_ids,
                                                          const int64_t* __restrict__ row_docs,
                                                          float* __restrict__ out_vals, int64_t* __restrict__ out_ids,
                                                          int64_t* __restrict__ out_docs) {
  __shared__ struct {
    RankShared<TH_CAND> list;
    uint32_t part[TH_PARTS];
    uint32_t n_part, n_cand;
  } sh;
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* s = scores + (size_t)row * n;
  out_vals += (size_t)row * k;
  out_ids += (size_t)row * k;
  out_docs += (size_t)row * k;
  auto emit = [&](int i, unsigned long long e, int64_t id, int64_t doc) {
    const float v = key_float((uint32_t)(e >> 32));
    const bool hit = !isinf(v);
    out_vals[i] = v;
    out_ids[i] = hit ? id : -1;
    out_docs[i] = hit ? doc : -1;
  };
  auto entry = [](uint32_t key, int at) { return ((unsigned long long)key << 32) | (uint32_t)~at; };
  sh.list.hist[tid] = 0;
  if (tid < RK_FEW) sh.list.rank[tid] = 0;
  if (tid == 0) {
    sh.list.n = 0;
    sh.n_part = 0;
    sh.n_cand = 0;
  }
  uint32_t lo = ~0u, hi = 0u;
  // a score at or above the bound takes a slot (n % 4 == 0: whole vectors)
  auto take = [&](int i, unsigned long long bound) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(s + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t key = float_key(v[e]);
      const unsigned long long x = entry(key, i + e);
      const int at = wave_append(&sh.n_cand, x >= bound && key != kNegInfKey);
      if (at >= 0 && at < TH_CAND) {
        sh.list.key[at] = x;
        lo = min(lo, key);
        hi = max(hi, key);
      }
    }
  };
  if (n <= TH_CAND) {
    __syncthreads();
    for (int i = 4 * tid; i < n; i += 4 * SEL_NT) take(i, 0ull);
  } else {
    const u32x4* pv = reinterpret_cast<const u32x4*>(parts + (size_t)row * ldp);
    const int np = (n + 15) / 16, nv = (np + 3) / 4;
    u32x4 held[TH_HELD];
    uint32_t m = 0;
    auto look = [&](int v) {  // past the last part: zeros
      u32x4 x = pv[min(v, nv - 1)];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = 4 * v + e < np ? x[e] : 0u;
      return x;
    };
#pragma unroll
    for (int j = 0; j < TH_HELD; ++j) held[j] = look(tid + j * SEL_NT);
#pragma unroll
    for (int j = 0; j < TH_HELD; ++j) m = max(max(m, max(held[j][0], held[j][1])), max(held[j][2], held[j][3]));
#pragma unroll 4
    for (int v = tid + TH_HELD * SEL_NT; v < nv; v += SEL_NT) {
      const u32x4 x = look(v);
      m = max(max(m, max(x[0], x[1])), max(x[2], x[3]));
    }
    auto each_vector = [&](int from, auto f) __attribute__((always_inline)) {
#pragma unroll 4
      for (int v = from + tid; v < nv; v += SEL_NT) f(look(v), v);
    };
    auto each_part = [&](auto f) __attribute__((always_inline)) {
      each_vector(0, [&](const u32x4& x, int v) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f(entry(x[e], 4 * v + e));
      });
    };
    const int live = __syncthreads_count(m > kNegInfKey);
    unsigned long long top = entry(m, 0), bound = 0;
    auto keep = [&](const u32x4& x, int v, auto reaches) __attribute__((always_inline)) {
      if (!__ballot(max(max(x[0], x[1]), max(x[2], x[3])) >= (uint32_t)(bound >> 32))) return;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int at = wave_append(&sh.n_part, reaches(x[e], 4 * v + e));
        if (at >= 0 && at < TH_PARTS) sh.part[at] = 4 * v + e;
      }
    };
    auto by_key = [&](uint32_t key, int) { return key >= (uint32_t)(bound >> 32); };
    auto by_entry = [&](uint32_t key, int at) { return entry(key, at) >= bound; };
    if (live >= TH_FEW * k) {
      uint32_t mlo = m > kNegInfKey ? m : ~0u, mhi = m;
      block_range(sh.list, mlo, mhi);
      top = entry(mhi, 0);
      const int shift = bin_shift(mlo, mhi);
      if (m > kNegInfKey) atomicAdd(&sh.list.hist[(m - mlo) >> shift], 1u);
      __syncthreads();
      bound = (unsigned long long)(mlo + (cut_bin(sh.list, (uint32_t)k) << shift)) << 32;
      sh.list.hist[tid] = 0;
#pragma unroll
      for (int j = 0; j < TH_HELD; ++j) keep(held[j], tid + j * SEL_NT, by_key);
      each_vector(TH_HELD * SEL_NT, [&](const u32x4& x, int v) __attribute__((always_inline)) { keep(x, v, by_key); });
    } else if (live) {
      uint32_t mlo = ~0u, mhi = m;
      each_vector(0, [&](const u32x4& x, int) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) mlo = min(mlo, x[e] > kNegInfKey ? x[e] : ~0u);
      });
      block_range(sh.list, mlo, mhi);
      top = entry(mhi, 0);
      const unsigned long long least = entry(mlo, np - 1);
      bound = bound_of(sh.list, least, top, (uint32_t)k, (uint32_t)max(2 * k, 1024), each_part);
      if (bound == least) bound = (unsigned long long)(kNegInfKey + 1) << 32;  // all parts, perhaps fewer than k
      each_vector(0, [&](const u32x4& x, int v) __attribute__((always_inline)) { keep(x, v, by_entry); });
    }
    __syncthreads();
    int chosen = (int)sh.n_part;
    static_assert(TH_PARTS >= 4 * SEL_MAXK && TH_PARTS >= 1024, "room for the parts");
    if (chosen > max(4 * k, 1024)) {  // the threads' bound says little
      bound = bound_of(sh.list, entry((uint32_t)(bound >> 32), np - 1), top, (uint32_t)k, (uint32_t)max(2 * k, 1024), each_part);
      if (tid == 0) sh.n_part = 0;
      __syncthreads();
      each_vector(0, [&](const u32x4& x, int v) __attribute__((always_inline)) { keep(x, v, by_entry); });
      __syncthreads();
      chosen = (int)sh.n_part;
    }
    auto each_chosen = [&](auto f) __attribute__((always_inline)) {
      for (int e = tid; e < 4 * chosen; e += SEL_NT) {
        const int i = 16 * (int)sh.part[e >> 2] + 4 * (e & 3);
        if (i < n) f(i);
      }
    };
    bound = bound >> 32 << 32;
    each_chosen([&](int i) { take(i, bound); });
    __syncthreads();
    if (sh.n_cand > TH_CAND) {  // to what rank_list ranks by counting, or sorts alone
      auto each_score = [&](auto f) __attribute__((always_inline)) {
        each_chosen([&](int i) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(s + i);
#pragma unroll
          for (int e = 0; e < 4; ++e) f(entry(float_key(v[e]), i + e));
        });
      };
      bound = bound_of(sh.list, entry((uint32_t)(bound >> 32), n - 1), top, (uint32_t)k,
                       (uint32_t)(k <= RK_FEW ? RK_FEW : RK_MANY), each_score);
      if (tid == 0) sh.n_cand = 0;
      lo = ~0u, hi = 0u;
      __syncthreads();
      each_chosen([&](int i) { take(i, bound); });
    }
  }
  __syncthreads();
  const int c = (int)sh.n_cand, kept = min(k, c);
  for (int i = kept + tid; i < k; i += SEL_NT) emit(i, (unsigned long long)kNegInfKey << 32, -1, -1);
  if (kept) rank_list(sh.list, c, kept, lo, hi, row_ids, row_docs, emit);
}

int top_hits(const float* scores, int rows, int n, const void* parts, int ldp, int k, const int64_t* row_ids,
             const int64_t* row_docs, float* out_vals, int64_t* out_ids, int64_t* out_docs, hipStream_t s) {
  if (rows <= 0) return 0;
  if (n <= 0 || n % 4 || k < 1 || k > n || k > SEL_MAXK || (uintptr_t)scores % 16) return hipErrorInvalidValue;
  if (n > TH_CAND && (!parts || (uintptr_t)parts % 16 || ldp % 4 || ldp < (n + 15) / 16)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(top_hits_kernel, dim3(rows), dim3(SEL_NT), 0, s, scores, n, (const uint32_t*)parts, ldp, k, row_ids,
                     row_docs, out_vals, out_ids, out_docs);
  return hipGetLastError();
}

// Item and document ids of ranked rows; -1 where the score is infinite (filtered rows past the last hit).
__global__ __launch_bounds__(256) void hit_ids_kernel(const float* __restrict__ vals, const int* __restrict__ rows,
                                                      const int64_t* __restrict__ row_ids,
                                                      const int64_t* __restrict__ row_docs, int64_t* __restrict__ ids,
                                                      int64_t* __restrict__ docs, int n, int n_rows) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int r = rows[i];
  const bool hit = !isinf(vals[i]) && r >= 0 && r < n_rows;
  ids[i] = hit ? row_ids[r] : -1;
  docs[i] = hit ? row_docs[r] : -1;
}

int hit_ids(const float* vals, const int* rows, const int64_t* row_ids, const int64_t* row_docs, int64_t* ids,
            int64_t* docs, int n, int n_rows, hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(hit_ids_kernel, dim3((n + 255) / 256), dim3(256), 0, s, vals, rows, row_ids, row_docs, ids, docs,
                     n, n_rows);
  return hipGetLastError();
}

// Filter bitmasks of a search, bit r of row q set where query q may see row r.
//
// Allow-lists of item ids: list q is ids[off[q] .. off[q + 1]), looked up by binary search in the index's ids sorted
// with their rows (16-20 dependent reads, all in L2); ids that are not in the index set nothing.
__global__ __launch_bounds__(256) void allow_bits_kernel(const int64_t* __restrict__ ids, const int64_t* __restrict__ off,
                                                         const int64_t* __restrict__ keys, const int64_t* __restrict__ rows,
                                                         int n_keys, uint32_t* __restrict__ mask, int words) {
  const int q = blockIdx.y;
  const int64_t i = off[q] + (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= off[q + 1]) return;
  const int64_t id = ids[i];
  int lo = 0, hi = n_keys;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (keys[mid] < id) lo = mid + 1;
    else hi = mid;
  }
  if (lo < n_keys && keys[lo] == id) {
    const int64_t r = rows[lo];
    if (r >= 0 && r < (int64_t)words * 32) atomicOr(mask + (size_t)q * words + (r >> 5), 1u << (r & 31));
  }
}

int allow_bits(const int64_t* ids, const int64_t* off, const int64_t* keys, const int64_t* rows, int n_keys,
               uint32_t* mask, int words, int queries, int longest, hipStream_t s) {
  if (queries <= 0 || longest <= 0 || n_keys <= 0) return 0;
  if (words <= 0 || queries > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(allow_bits_kernel, dim3((longest + 255) / 256, queries), dim3(256), 0, s, ids, off, keys, rows, n_keys,
                     mask, words);
  return hipGetLastError();
}

// Rows whose document id is below the query's bound; AND: intersected with the mask that is there.
// LIMITS: const int64_t*, or HostLimits.
__device__ __forceinline__ int64_t limit_of(const int64_t* limit, int q) { return limit[q]; }
__device__ __forceinline__ int64_t limit_of(const HostLimits& limit, int q) { return limit.v[q]; }

template <bool AND, typename LIMITS>
__global__ __launch_bounds__(256) void doc_lt_bits_kernel(const int64_t* __restrict__ docs, LIMITS limit, int n,
                                                          uint32_t* __restrict__ mask, int words) {
  const int q = blockIdx.y, r = blockIdx.x * 256 + threadIdx.x;
  const unsigned long long b = __ballot(r < n && docs[min(r, n - 1)] < limit_of(limit, q));
  const int lane = threadIdx.x & 63, w = r / 32;  // lanes 0 and 32 write the wave's two words
  if ((lane & 31) == 0 && w < words) {
    uint32_t* m = mask + (size_t)q * words + w;
    const uint32_t v = (uint32_t)(lane ? b >> 32 : b);
    *m = AND ? *m & v : v;
  }
}

template <typename LIMITS>
static int doc_lt_launch(const int64_t* docs, const LIMITS& limit, int n, uint32_t* mask, int words, int queries, int intersect,
                         hipStream_t s) {
  const dim3 grid((n + 255) / 256, queries);
  if (intersect) hipLaunchKernelGGL((doc_lt_bits_kernel<true, LIMITS>), grid, dim3(256), 0, s, docs, limit, n, mask, words);
  else hipLaunchKernelGGL((doc_lt_bits_kernel<false, LIMITS>), grid, dim3(256), 0, s, docs, limit, n, mask, words);
  return hipGetLastError();
}

// host: the limits are the host's, at most kHostValues
int doc_lt_bits(const int64_t* docs, const int64_t* limit, int n, uint32_t* mask, int words, int queries, int intersect, int host,
                hipStream_t s) {
  if (queries <= 0 || words <= 0) return 0;
  if (n <= 0 || words != (n + 31) / 32 || queries > (host ? kHostValues : 65535)) return hipErrorInvalidValue;
  if (!host) return doc_lt_launch(docs, limit, n, mask, words, queries, intersect, s);
  HostLimits values = {};
  for (int i = 0; i < queries; ++i) values.v[i] = limit[i];
  return doc_lt_launch(docs, values, n, mask, words, queries, intersect, s);
}

// Everything a search that selects from its scores launches, in one call: unit queries (with the groups and the cleared mask),
// the masks' bits, scores and maxima, selection.  Up to some 30k rows a search is bound by its host time, and a third of that
// were the calls from Python with their checks and buffers: 1 query in 5,000 rows of a group 35 -> 25 us, document bounds of
// 16 in 20k rows 40 -> 27, lists of 16 in 3,000 rows 62 -> 50, of 4 in 60k rows 67 with 46 instead of 66 of the host.
//
// One workspace, in pieces of whole pages of 4 KB: unit queries, groups, mask, scores, maxima.  (In pieces of 256 bytes, as one
// buffer behind the other, 1 query in 500,000 rows took 134.9 instead of 133.4 us, 16 in 300,000 100.5 instead of 99.8.)
SearchSpace search_space(int queries, int cols, int n, int n_groups, int masked) {
  SearchSpace w = {};
  const auto piece = [&](long bytes) {
    const long at = w.bytes;
    w.bytes += (bytes + 4095) / 4096 * 4096;
    return at;
  };
  w.ldp = ((n + 15) / 16 + 3) / 4 * 4;
  w.words = (n + 31) / 32;
  w.unit = piece((long)queries * cols * 2);
  w.groups = piece((long)n_groups * 4);
  w.mask = piece(masked ? (long)queries * w.words * 4 : 0);
  w.scores = piece((long)queries * n * 4);
  w.parts = piece((long)queries * w.ldp * 4);
  return w;
}

int selected_search(const SearchCall& c, hipStream_t s) {
  if (c.queries <= 0 || c.k <= 0 || c.k > c.n || c.rows <= 0 || c.rows > c.n || c.n % 4) return hipErrorInvalidValue;
  if (c.host_groups && (c.n_groups < c.queries || c.n_groups > kHostValues)) return hipErrorInvalidValue;
  if (c.limits && c.queries > kHostValues) return hipErrorInvalidValue;
  const bool masked = c.lists || c.limits;
  const SearchSpace w = search_space(c.queries, c.cols, c.n, c.host_groups ? c.n_groups : 0, masked);
  if (c.space_bytes < w.bytes) return hipErrorInvalidValue;
  char* const base = (char*)c.space;
  uint32_t* const mask = masked ? (uint32_t*)(base + w.mask) : nullptr;
  int* const groups = c.host_groups ? (int*)(base + w.groups) : nullptr;
  const int words = (c.rows + 31) / 32;  // (of the rows rounded up to fours: as many)
  if (words != w.words) return hipErrorInvalidValue;
  int rc = unit_rows(c.x, c.ldx, base + w.unit, c.queries, c.cols, s, c.host_groups, c.host_groups ? c.n_groups : 0, groups,
                     c.lists ? mask : nullptr, c.lists ? (long)c.queries * words : 0);
  if (!rc && c.lists) rc = allow_bits(c.ids, c.offsets, c.keys, c.key_rows, c.n_keys, mask, words, c.queries, c.longest, s);
  if (!rc && c.limits) rc = doc_lt_bits(c.row_docs, c.limits, c.rows, mask, words, c.queries, c.lists, 1, s);
  if (!rc)
    rc = index_scan_scores_shuf(base + w.unit, c.cols, c.vecs, c.queries, c.n, c.cols, c.row_group, groups, mask, (float*)(base + w.scores),
                                base + w.parts, w.ldp, s);
  if (!rc)
    rc = top_hits((const float*)(base + w.scores), c.queries, c.n, base + w.parts, w.ldp, c.k, c.row_ids, c.row_docs, c.vals, c.out_ids,
                  c.out_docs, s);
  return rc;
}

// Rows first, first + step, ... of a matrix in the shuffle_weights layout, row-major (the search's row sample, rows of
// a snapshot): a thread a 16-B piece, piece (c, g) of row r at [r / 16][c][g][r % 16].
__global__ __launch_bounds__(256) void gather_rows_kernel(const u32x4* __restrict__ src, const int64_t* __restrict__ rows,
                                                          u32x4* __restrict__ out, int n, int pieces) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)n * pieces) return;
  const int64_t r = rows[i / pieces];
  const int p = (int)(i % pieces);  // 32-wide chunk p / 4, 8-wide piece p % 4
  out[i] = src[((r / 16) * pieces + p) * 16 + r % 16];
}

int gather_rows(const void* src, const int64_t* rows, void* out, int n, int K, hipStream_t s) {
  if (n <= 0) return 0;
  if (K <= 0 || K % 32) return hipErrorInvalidValue;
  const int pieces = K / 8;
  const int64_t blocks = ((int64_t)n * pieces + 255) / 256;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, s, (const u32x4*)src, rows, (u32x4*)out, n, pieces);
  return hipGetLastError();
}

}  // namespace dab
