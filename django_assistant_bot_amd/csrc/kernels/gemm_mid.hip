// Mid-M bf16 GEMM  C[M,N] = A[M,K] . B[N,K]^T  (+ residual, or fused SwiGLU over 8-row [gate | up]
// groups) for up to 4096 rows: the token counts of mixed prefill + decode serving steps and of
// request-at-a-time prompts (the reference runs one HF ``generate`` per request:
// ai/providers/transformers.py:57-66, served by gunicorn_conf.py:9 workers).  B is in the
// ops.shuffle_weights fragment layout (the one copy of every projection the decoder keeps).
//
// Two kernels: gemm_mid_kernel with tiles of 128 x 256, described here, and gemm_wide_kernel with tiles of 256 or 192 x 256 for
// longer prompts (what differs stands there; which of them a product takes: mid_pick, and the caller for 192 rows).
//
// Why a third GEMM: at these M the 256x256 phased kernel (gemm256.hip) has 12-64 tiles for 256 CUs
// and the 128x128 kernel (gemm.hip) runs at ~20 % of the MFMA rate (profiles/gemm_mid_r5.md).
// Design (cdna_hip_programming.md section 5, "Projection GEMM at M = 256"; stream-K):
//   * tile 128 (rows of A) x 256 (weight rows), K-tile 64; 8 waves = 2 (M) x 4 (N), each wave a
//     64 x 64 piece = 4 x 4 v_mfma_f32_16x16x32_bf16 accumulators, 32 MFMAs per K-tile;
//   * A / B staged by LDS-DMA (buffer_load ... lds, 16 B per lane) into a ring of 3 K-tile stages
//     of 48 KB (A 16 KB | B0 16 KB | B1 16 KB); one phase per K-tile: [fragment reads, DMA of the
//     K-tile two ahead, counted vmcnt] barrier [32 MFMAs] barrier; the two wave groups (wr = 0 / 1)
//     run one barrier apart (one group's MFMAs beside the other's LDS reads), as in gemm256;
//   * work decomposition: the tiles_m workgroups of one "group" (one per 128-row tile of A) march
//     in lockstep through the SAME range of the (weight tile, K-tile) iteration space, so a weight
//     K-tile is fetched from HBM once and served to the group's other workgroups from their XCD's
//     L2 (groups are formed from blocks that share blockIdx % 8; the slots that whole groups leave over on
//     the XCDs are joined into further groups, whose weights come from HBM or MALL once for each of their two or
//     three XCDs).  The iteration space tiles_n x (K / 64) is split evenly over the groups, floor(256 / tiles_m) or
//     fewer (gemm_mid_groups; stream-K in the N x K plane): every working CU gets the same number of MFMAs whatever
//     the tile count;
//   * a tile whose K range spans several groups is combined in-launch by its OWNER, the group
//     holding the tile's first K-steps: that segment ends the owner's range, so in time it finishes
//     last.  The other segments store their fp32 partial (write-through sc1 stores, 1 KB per
//     wave-instruction) and count themselves in at the tile two K-steps later, when the pipeline's own
//     counted wait has retired the stores (no drain); the owner keeps its partial in registers,
//     waits until all are in, adds the partials with sc1 loads in segment order (no
//     fence needed: cdna_hip_programming.md section 5 item 2), clears the count and runs the
//     epilogue;
//   * no workgroup waits without end.  The parts an owner waits for may stand on any XCD and behind it in the order of
//     placement, and workgroups of another stream's launch that wait in the same way can hold the CUs they need (16 row
//     tiles: two launches with half of each XCD's CUs each).  So after some 0.1 ms an owner stores its sum too, counts itself
//     in and goes on, and the workgroup whose part comes last adds them all, in the same order: the same bits.  One count a
//     tile instead of a flag a part: 0.98-1.06 times the speed over 136 sizes of Llama-3-8B's and 1B's projections, 1.01 in the mean.
//     A last-arriver combine for every tile (every segment stored and drained, then an atomic ticket) cost 5-9 us
//     per launch on the small projections (profiles/gemm_mid_r6.md).
#include <cmath>

#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

enum { MID_NONE = 0, MID_SWIGLU8 = 4, MID_GEGLU8 = 6, MID_REGLU8 = 7 };

struct GMid {
  const bf16* A;
  const bf16* B;  // shuffle_weights layout, [N][K]
  bf16* C;
  const bf16* residual;   // GLU epilogues with RES: fp32 bias [gate N / 2 | up N / 2] instead
  float* slabs;  // [tiles_m][gn][2] partial tiles of 128 x 256 fp32 (in accumulator order): a range's first part, and the sum
                 // that an owner handed over
  int* cnt;      // zero at rest.  128 rows: [8 spx ..) the parts of a divided tile that are in, by its owner, [tiles_m][gn]; 256 rows:
                 // [.. 8 spx) ready flags (the launch that stored a partial tile)
  unsigned* ended;  // [8][32]: workgroups of an XCD label that ended, over all launches on this workspace, a line each
  long spin_limit;
  int M, N, K;
  long lda, ldc, ldr;
  int tiles_m, tiles_n, kt;
  int spx;  // blocks per XCD label (grid / 8)
  int gpx;  // whole groups per XCD label
  int gn;   // groups: 8 * gpx and those of the slots left over
  int q, r;  // tiles_n * kt = q * gn + r iterations: group j owns q (+1 for j < r)
  unsigned b_bytes, slab_bytes;
  int bgrp;  // row blocks per group of the B copy: 1 (plain) or 8 (shuffle_weights(w, 8))
};

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mk_rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

template <int VMC>
__device__ __forceinline__ void wait_vmc() {
  static_assert(VMC >= 0 && VMC <= 63, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(VMC) : "memory");
}

__device__ __forceinline__ void mbar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// the barrier after a phase's LDS reads: they are retired first (s_barrier waits for no counter)
__device__ __forceinline__ void mread_bar() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  mbar();
}

// ring geometry per K-step width BK (64: 3 stages of 48 KB, DMA distance 2; 32: 6 stages of 24 KB,
// distance 5 -- the same LDS, two and a half times the latency cover in cycles)
template <int BK>
struct MidGeo {
  static constexpr int kA = 128 * BK * 2;        // A bytes per stage
  static constexpr int kStage = 384 * BK * 2;    // A | B (256 weight rows)
  static constexpr int kStages = BK == 64 ? 3 : 6;
  static constexpr int kDist = kStages - 1;     // stage issued kDist iterations ahead
  static constexpr int kDma = BK == 64 ? 6 : 3;  // LDS-DMA instructions per wave per stage
  static constexpr int kSmem = kStages * kStage;
  static_assert(kSmem + 512 <= 163840, "LDS");
};
constexpr int kE = 8;                  // VMEM stores per wave in every epilogue variant
constexpr int kSlabSt = 16;            // VMEM stores per wave of a published partial tile
constexpr int kSlabFloats = 512 * 64;  // one partial tile: 512 threads x 16 f32x4

// group start of the balanced split of the iteration space
__device__ __forceinline__ int grp_start(int j, int q, int r) { return j * q + min(j, r); }
__device__ __forceinline__ int grp_owner(int i, int q, int r) {
  const int big = r * (q + 1);
  return i < big ? i / (q + 1) : r + (i - big) / q;
}

}  // namespace

// BK: K-step width (see MidGeo); DIAG (timing only, benchmarks/gemm_bench.py): 1 = partial tiles
// are stored and counted but never combined (the output of split tiles is left unwritten)
template <int EPI, bool RES, int BK, int DIAG = 0>
__global__ __launch_bounds__(512) void gemm_mid_kernel(GMid p) {
  using Geo = MidGeo<BK>;
  constexpr int kStage = Geo::kStage, kStages = Geo::kStages, kDist = Geo::kDist, kDma = Geo::kDma;
  constexpr int kA = Geo::kA;
  __shared__ __attribute__((aligned(16))) char smem[Geo::kSmem];

  // ---- which group / row tile this block is: blocks b, b + 8, ... share an XCD label.  The slots of an XCD that whole
  // groups leave over are joined, XCD after XCD, into further groups
  const int bid = blockIdx.x, tid = threadIdx.x;
  const int x = bid & 7, slot = bid >> 3;
  unsigned* const ended = p.ended + 32 * x;
  auto count_out = [&]() {
    if (tid == 0) __hip_atomic_fetch_add(ended, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  int g = slot / p.tiles_m, mt = slot - g * p.tiles_m, j = x * p.gpx + g;
  if (g >= p.gpx) {
    const int over = p.spx - p.gpx * p.tiles_m, u = x * over + slot - p.gpx * p.tiles_m;
    g = u / p.tiles_m;
    mt = u - g * p.tiles_m;
    j = 8 * p.gpx + g;
    if (j >= p.gn) return count_out();  // whole workgroup (uniform)
  }
  const int start = grp_start(j, p.q, p.r);
  const int end = start + p.q + (j < p.r ? 1 : 0);
  if (end <= start) return count_out();

  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w >> 2, wc = w & 3;
  const int li = lane & 15, gq = lane >> 4;
  const int m0 = mt * 128;
  const int kt = p.kt;  // K-steps of BK per tile

  // ---- LDS-DMA staging (per-lane parts in VOFFSET, the K / panel offset in SOFFSET).
  // A: BK = 64: rows of 128 B, 16-B chunk c of row r at c ^ ((r >> 1) & 7), wave w stages rows
  //    8w..8w+7 (+64);  BK = 32: rows of 64 B, chunk c at c ^ ((r >> 2) & 3), wave w rows 16w..16w+15.
  //    (conflict-free for the 4 x 16-lane groups of ds_read_b128; the swizzle goes on the SOURCE
  //    address since LDS-DMA writes lane-linearly)
  // B: the fragment layout: a 16-row x 32-k block is 1 KB in lane order; BK = 64 stages blocks
  //    (rb, 2kk) and (rb, 2kk + 1) back to back (2 KB per row block), BK = 32 block (rb, kk).
  unsigned vA0, vA1 = 0;
  if constexpr (BK == 64) {
    const int sw = (4 * (w & 1) + (lane >> 4)) & 7;
    const int cc = (lane & 7) ^ sw;
    const int srow = 8 * w + (lane >> 3);
    vA0 = (unsigned)((srow * p.lda + 8 * cc) * 2);
    vA1 = vA0 + (unsigned)(64 * p.lda * 2);
  } else {
    const int srow = 16 * w + (lane >> 2);
    const int cc = (lane & 3) ^ ((srow >> 2) & 3);
    vA0 = (unsigned)((srow * p.lda + 8 * cc) * 2);
  }
  const unsigned kblk = (unsigned)(p.K / 32) * 1024u;  // bytes of one 16-row block over all of K
  // grouped copy (p.bgrp = 8, shuffle_weights(w, 8)): the 8 blocks of a 128-row half adjacent per k
  // chunk, so block w of a half is w KB in and a k chunk is 8 KB on (the half itself starts where
  // the plain layout's does)
  const bool bgrp = p.bgrp == 8;
  const unsigned cb = bgrp ? 8192u : 1024u;  // bytes per 32-deep k chunk of a block
  const unsigned vB0 = (unsigned)(lane * 16) + (unsigned)w * (bgrp ? 1024u : kblk), vB2 = vB0 + 8u * kblk;
  const long a_rows = min(128, p.M - m0);
  const __amdgpu_buffer_rsrc_t rA = mk_rsrc(p.A + (size_t)m0 * p.lda, (unsigned)(((a_rows - 1) * p.lda + p.K) * 2));
  const __amdgpu_buffer_rsrc_t rB = mk_rsrc(p.B, p.b_bytes);

  auto stage = [&](int buf, int nt, int kk) {
    char* dst = smem + buf * kStage;
    const unsigned sa = (unsigned)kk * (unsigned)(BK * 2);
    const unsigned sb = (unsigned)nt * 16u * kblk + (unsigned)kk * (unsigned)(BK / 32) * cb;
    if constexpr (BK == 64) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void*)(dst + w * 1024), 16, vA0, sa, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void*)(dst + 8192 + w * 1024), 16, vA1, sa, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + kA + w * 2048), 16, vB0, sb, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + kA + w * 2048 + 1024), 16, vB0 + cb, sb, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + kA + 16384 + w * 2048), 16, vB2, sb, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + kA + 16384 + w * 2048 + 1024), 16, vB2 + cb, sb,
                                               0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void*)(dst + w * 1024), 16, vA0, sa, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + kA + w * 1024), 16, vB0, sb, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + kA + 8192 + w * 1024), 16, vB2, sb, 0, 0);
    }
  };

  // ---- fragment reads: A rows 64 wr + 16 i + li, B row blocks 4 wc + jn
  constexpr int KS = BK / 32;  // MFMA k-steps per stage
  int rdA[KS];
  if constexpr (BK == 64) {
    const int swr = li >> 1;
    rdA[0] = (64 * wr + li) * 128 + 16 * (gq ^ swr);
    rdA[KS - 1] = (64 * wr + li) * 128 + 16 * ((4 + gq) ^ swr);
  } else {
    rdA[0] = (64 * wr + li) * 64 + 16 * (gq ^ ((li >> 2) & 3));
  }
  constexpr int kRowBlk = BK * 32;  // LDS bytes of one 16-row block of A / B in a stage
  const int rdB = kA + wc * 4 * kRowBlk + lane * 16;

  bf16x8 af[4][KS];
  bf16x8 bfr[4][KS];
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int jn = 0; jn < 4; ++jn) acc[i][jn] = f32x4{0.f, 0.f, 0.f, 0.f};

  // staging cursor: the iteration kDist ahead of the one being computed
  int s_nt = start / kt, s_kk = start - s_nt * kt;
  int s_it = start;
  auto advance = [&]() {
    ++s_it;
    if (++s_kk == kt) {
      s_kk = 0;
      ++s_nt;
    }
  };
  // prologue: iterations start .. start + kDist - 1 in flight (buffers 0 ..), the first landed
#pragma unroll
  for (int d = 0; d < kDist; ++d)
    if (s_it < end) {
      stage(d, s_nt, s_kk);
      advance();
    }
  {
    const int beyond = s_it - start - 1;  // issued stages past the first
    if (beyond >= 4) wait_vmc<4 * kDma>();
    else if (beyond == 3) wait_vmc<3 * kDma>();
    else if (beyond == 2) wait_vmc<2 * kDma>();
    else if (beyond == 1) wait_vmc<kDma>();
    else wait_vmc<0>();
  }
  mbar();

  int it = start;
  int b = 0;  // ring buffer of iteration `it`
  // VMEM stores issued since the last phase's wait (younger than the DMA in flight): an epilogue's
  // kE or a published partial's kSlabSt; the next phase's counted wait lets them stay in flight
  int after_st = 0;
  // the tile of a partial stored by this workgroup that is not counted in yet: counted at the second phase after the
  // stores, when that phase's vmcnt(kDma) has retired them (no drain)
  int pend = -1, pend_phases = 0;
  int before = -1;  // lane 0: how many of its tile's parts were in before this workgroup's first one
  const __amdgpu_buffer_rsrc_t rS = mk_rsrc(p.slabs, p.slab_bytes);
  auto slab_off = [&](int jj, int side) { return (unsigned)(((mt * p.gn + jj) * 2 + side) * kSlabFloats) * 4u; };
  auto count_in = [&](int at) {  // after every wave's stores retired and a barrier
    return tid == 0 ? __hip_atomic_fetch_add(p.cnt + at, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -1;
  };
  auto publish = [&](int side) {
    const unsigned own = slab_off(j, side);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jn = 0; jn < 4; ++jn)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][jn]), rS, (unsigned)(tid * 16),
                                               own + (unsigned)((i * 4 + jn) * 8192), 16);
  };
  auto add_partial = [&](int jj, int side) {
    const unsigned off = slab_off(jj, side);
    u32x4 v[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jn = 0; jn < 4; ++jn)
        v[i][jn] = __builtin_amdgcn_raw_buffer_load_b128(rS, (unsigned)(tid * 16), off + (unsigned)((i * 4 + jn) * 8192), 16);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jn = 0; jn < 4; ++jn) acc[i][jn] += __builtin_bit_cast(f32x4, v[i][jn]);
  };
  for (;;) {
    // behind its range a workgroup whose part of the first tile came last finishes that tile (a round without K-steps)
    const bool late = it >= end;
    const int nt = (late ? start : it) / kt;
    const int j_lo = grp_owner(nt * kt, p.q, p.r), j_hi = grp_owner(nt * kt + kt - 1, p.q, p.r);
    if (late && (j == j_lo || !__syncthreads_or(before == j_hi - j_lo))) break;
    const int k0 = late ? 0 : it - nt * kt;
    const int k1 = late ? 0 : min(kt, k0 + (end - it));
    if (wr == 1) mbar();  // group 1 one barrier behind through the K-loop (ping-pong)
    for (int kk = k0; kk < k1; ++kk, ++it) {
      const char* sb = smem + b * kStage;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) af[i][ks] = *reinterpret_cast<const bf16x8*>(sb + i * 16 * (BK * 2) + rdA[ks]);
#pragma unroll
      for (int jn = 0; jn < 4; ++jn)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          bfr[jn][ks] = *reinterpret_cast<const bf16x8*>(sb + rdB + jn * kRowBlk + ks * 1024);
      // the stage kDist ahead goes into the buffer read one phase ago
      if (s_it < end) {
        stage(b == 0 ? kStages - 1 : b - 1, s_nt, s_kk);
        advance();
        if (after_st == kSlabSt) wait_vmc<(kDist - 1) * kDma + kSlabSt>();
        else if (after_st == kE) wait_vmc<(kDist - 1) * kDma + kE>();
        else wait_vmc<(kDist - 1) * kDma>();
      } else {
        // tail: the stages after `it + 1` that are still in flight may stay so
        const int beyond = after_st ? 0 : s_it - it - 2;
        if (beyond >= 4) wait_vmc<4 * kDma>();
        else if (beyond == 3) wait_vmc<3 * kDma>();
        else if (beyond == 2) wait_vmc<2 * kDma>();
        else if (beyond == 1) wait_vmc<kDma>();
        else wait_vmc<0>();
      }
      after_st = 0;
      mread_bar();
      if (pend >= 0 && ++pend_phases >= 2) {  // this phase's wait retired the stores
        before = count_in(pend);
        pend = -1;
      }
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int jn = 0; jn < 4; ++jn) acc[i][jn] = mfma16(bfr[jn][ks], af[i][ks], acc[i][jn]);
      __builtin_amdgcn_s_setprio(0);
      mbar();
      b = b == kStages - 1 ? 0 : b + 1;
    }
    if (wr == 0) mbar();  // pairs with group 1's last K-loop barrier
    if (pend >= 0) {  // (a one-phase segment followed: drain and count now)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      before = count_in(pend);
      pend = -1;
    }

    // ---- segment end.  A whole tile goes straight to the epilogue.  A split tile's segments are
    // held by groups j_lo .. j_hi in K order; its OWNER is j_lo, whose segment (the tile's first
    // K-steps) ends its own range, so in time it finishes last.  The other segments store their
    // fp32 partial (sc1, write-through) and count themselves in; the owner waits until all are in
    // and adds them in segment order, its registers first.  Where they stay out it stores its own as well: of all of
    // them one counts itself in last, and that workgroup adds them.
    const int n0 = nt * 256;
    bool write = true;
    if (k0 != 0 || k1 != kt) {
      const int at = 8 * p.spx + mt * p.gn + j_lo;  // where the tile's parts are counted
      if (late) {
        add_partial(j_lo, 1);
      } else if (j != j_lo) {
        publish(0);
        after_st = kSlabSt;
        if (!DIAG) {  // (DIAG: the owner reads nothing, so nothing may be counted)
          pend = at;
          pend_phases = 0;
          if (it >= end) {  // nothing left to hide the drain behind
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            before = count_in(at);
            pend = -1;
          }
        }
        write = false;
      } else if (DIAG) {
        write = false;
      } else {
        bool in = true;
        if (tid == 0) {
          long spins = 0;
          while (__hip_atomic_load(p.cnt + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != j_hi - j_lo) {
            if (++spins > p.spin_limit) {
              in = false;
              break;
            }
            __builtin_amdgcn_s_sleep(2);
          }
        }
        if (!__syncthreads_and(in)) {  // (every thread loads only after lane 0 saw the count)
          publish(1);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          __syncthreads();
          write = __syncthreads_or(count_in(at) == j_hi - j_lo);
        }
      }
      if (write) {
        for (int jj = j_lo + 1; jj <= j_hi; ++jj) add_partial(jj, 0);
        if (tid == 0) __hip_atomic_store(p.cnt + at, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (write) {
      // ---- epilogue: acc[i][jn][r] = C[m0 + 64 wr + 16 i + li][n0 + 64 wc + 16 jn + 4 gq + r];
      // exactly kE stores per wave (rows >= M fall outside the descriptor and are dropped)
      int e_li = li, e_g = gq, e_wc = wc;
      asm volatile("" : "+v"(e_li), "+v"(e_g), "+v"(e_wc));
      const long c_rows = min(128, p.M - m0);
      const __amdgpu_buffer_rsrc_t rC = mk_rsrc(p.C + (size_t)m0 * p.ldc, (unsigned)(c_rows * p.ldc * 2));
      if constexpr (glu8_epilogue(EPI)) {
        // 8-row [gate | up] groups inside each 16-row block: one permlane32_swap of the (jn, jn + 1)
        // pair gives lanes 0-31 block jn's gate / up rows and lanes 32-63 block jn + 1's
        f32x4 bg[2], bu[2];
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
          bg[pr] = bu[pr] = f32x4{0.f, 0.f, 0.f, 0.f};
          if constexpr (RES) {
            const float* fb = reinterpret_cast<const float*>(p.residual) + (n0 + 64 * e_wc + 32 * pr) / 2 + 4 * e_g;
            bg[pr] = *reinterpret_cast<const f32x4*>(fb);
            bu[pr] = *reinterpret_cast<const f32x4*>(fb + p.N / 2);
          }
        }
        if constexpr (RES) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mr = 64 * wr + 16 * i + e_li;
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][2 * pr][r]),
                                                              __float_as_uint(acc[i][2 * pr + 1][r]), false, false);
              o[r] = glu_act<glu8_act(EPI)>(__uint_as_float(s[0]) + bg[pr][r]) * (__uint_as_float(s[1]) + bu[pr][r]);
            }
            u32x2 v;
            v[0] = pack2bf(o[0], o[1]);
            v[1] = pack2bf(o[2], o[3]);
            const int oc = (n0 + 64 * e_wc + 32 * pr) / 2 + 4 * e_g;
            __builtin_amdgcn_raw_buffer_store_b64(v, rC, (unsigned)((mr * p.ldc + oc) * 2), 0, 0);
          }
        }
      } else {
        // permlane16_swap of the (jn, jn + 1) pair: each lane then holds 8 contiguous columns
        // n0 + 64 wc + 32 pr + cq -> one 16-B store
        const int cq = 16 * (e_g & 1) + 8 * (e_g >> 1);
        u32x4 rv[4][2];
        if constexpr (RES) {
          const __amdgpu_buffer_rsrc_t rR = mk_rsrc(p.residual + (size_t)m0 * p.ldr, (unsigned)(c_rows * p.ldr * 2));
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int pr = 0; pr < 2; ++pr)
              rv[i][pr] = __builtin_amdgcn_raw_buffer_load_b128(
                  rR, (unsigned)(((64 * wr + 16 * i + e_li) * p.ldr + n0 + 64 * e_wc + 32 * pr + cq) * 2), 0, 0);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mr = 64 * wr + 16 * i + e_li;
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            float o[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][2 * pr][r]),
                                                              __float_as_uint(acc[i][2 * pr + 1][r]), false, false);
              o[r] = __uint_as_float(s[0]);
              o[4 + r] = __uint_as_float(s[1]);
            }
            if constexpr (RES) {
              const u32x4 rw = rv[i][pr];
#pragma unroll
              for (int qd = 0; qd < 4; ++qd) {  // round like a bf16 GEMM output, then the bf16 add (HF)
                o[2 * qd] = bf2f(f2bf(o[2 * qd])) + __uint_as_float(rw[qd] << 16);
                o[2 * qd + 1] = bf2f(f2bf(o[2 * qd + 1])) + __uint_as_float(rw[qd] & 0xffff0000u);
              }
            }
            u32x4 v;
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) v[qd] = pack2bf(o[2 * qd], o[2 * qd + 1]);
            const int nc = n0 + 64 * e_wc + 32 * pr + cq;
            __builtin_amdgcn_raw_buffer_store_b128(v, rC, (unsigned)((mr * p.ldc + nc) * 2), 0, 0);
          }
        }
      }
      after_st = kE;
    }
    if (late) break;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int jn = 0; jn < 4; ++jn) acc[i][jn] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  count_out();
}

// Tiles of 256 x 256 with the same split of the iteration space (in pairs of K-steps), partial tiles and owners, which wait for a
// flag of each part (they hand nothing over: the workgroups they wait for have been placed before them).  What bounds
// the kernel above is the way of its loads into a CU: 48 KB a K-step (64 B a cycle at best, 43 measured from L2) against 1024
// cycles of MFMAs; with both operands' addresses held still its K-step takes as long, and weights straight into registers
// instead of LDS gain nothing.  A tile of 256 rows loads 32 KB for the same MFMAs.  Loop, staging and LDS layout are those of
// gemm256: two buffers of K-steps, a phase of two quadrants of 128 x 128, pieces of 16 KB restaged one phase after their last
// read and waited for three phases later.
namespace {
constexpr int kWHalf = 16384;                // a K-step: A0 | A1 | B0 | B1, 128 rows of 128 B each (A1: the tile's rows past 128)
constexpr int kWSlabFloats = 256 * 256;      // one a workgroup: only the first part of its range can be another's tile
static_assert(kWSlabFloats == 2 * kSlabFloats, "the partial tiles of both kernels take the same workspace");
}  // namespace

// ROWS 256, or 192 (the second half of A is 64 rows, its phases of half the products) where that leaves fewer rows past the
// prompt's end: a pair of K-steps 1.45-2.2 us against 1.83-2.7, partial tiles of 192 KB.  us of a call of Llama-3-8B without -> with
// it: 560 tokens 10,220 -> 9,789, 1,093 15,949 -> 15,754, 1,300 18,085 -> 17,349; Llama-3.2-1B, 1,300 3,709 -> 3,483.
template <int EPI, bool RES, int ROWS>
__global__ __launch_bounds__(512) void gemm_wide_kernel(GMid p) {
  static_assert(ROWS == 256 || ROWS == 192, "a second half of 128 or 64 rows");
  constexpr int H2 = ROWS - 128, I2 = H2 / 32;               // rows of the second half, 16-row blocks of a wave in it
  constexpr int kWBuf = 3 * kWHalf + H2 * 128;
  constexpr int NE = 16 + 4 * I2, kWSlabSt = NE, kWE = NE / 2;  // accumulators; VMEM stores per wave of a published partial tile, of an epilogue
  constexpr int kFly = 6 + H2 / 64;                          // copies that a phase's wait leaves in flight
  // behind the buffers: the count the launch's number comes from, and whether an owner's waits ended well
  __shared__ __attribute__((aligned(16))) char smem[2 * kWBuf + 256];

  const int bid = blockIdx.x, tid = threadIdx.x;
  const int x = bid & 7, slot = bid >> 3;
  unsigned* const ended = p.ended + 32 * x;
  auto count_out = [&]() {
    if (tid == 0) __hip_atomic_fetch_add(ended, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // Each XCD takes p.tiles_n column tiles of its own, whose parts its groups share: later blocks hold earlier parts.  An owner
  // waits for groups of its XCD alone, whose workgroups stand in front of its own in the order of placement.  The first
  // workgroup of an XCD that has not ended so waits for nobody, and the launch ends however few of its workgroups are
  // resident and whatever other launches hold some XCDs (they fill a CU, and fit beside none).
  const int g = slot / p.tiles_m, mt = slot - g * p.tiles_m, j = p.gpx - 1 - g;
  if (j < 0) return count_out();  // whole workgroup (uniform)
  const int start = grp_start(j, p.q, p.r);
  const int end = start + p.q + (j < p.r ? 1 : 0);
  if (end <= start) return count_out();
  const int nt0 = x * p.tiles_n;

  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w >> 2, wc = w & 3;
  const int li = lane & 15, gq = lane >> 4;
  const int m0 = mt * ROWS;
  const int kt = p.kt;  // pairs of K-steps per tile

  // ---- LDS-DMA staging, as the kernel above: piece = 128 rows of A (16-B chunk c of row r at c ^ ((r >> 1) & 7), swizzled
  // at the source) or 8 blocks of 16 weight rows, 2 KB each
  const int cc = (lane & 7) ^ ((4 * (w & 1) + (lane >> 4)) & 7);
  const unsigned vA0 = (unsigned)(((8 * w + (lane >> 3)) * p.lda + 8 * cc) * 2), rowsA = (unsigned)(64 * p.lda * 2);
  const unsigned kblk = (unsigned)(p.K / 32) * 1024u;
  const bool bgrp = p.bgrp == 8;
  const unsigned cb = bgrp ? 8192u : 1024u;
  const unsigned vB0 = (unsigned)(lane * 16) + (unsigned)w * (bgrp ? 1024u : kblk);
  const long a_rows = min(ROWS, p.M - m0);
  const __amdgpu_buffer_rsrc_t rA = mk_rsrc(p.A + (size_t)m0 * p.lda, (unsigned)(((a_rows - 1) * p.lda + p.K) * 2));
  const __amdgpu_buffer_rsrc_t rB = mk_rsrc(p.B, p.b_bytes);
  auto stage_a = [&](int buf, int half, int ks) {
    char* dst = smem + buf * kWBuf + half * kWHalf + w * 1024;
    const unsigned v0 = vA0 + (half ? 2u * rowsA : 0u), v1 = v0 + rowsA, so = (unsigned)ks * 128u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void*)dst, 16, v0, so, 0, 0);
    if (half == 0 || H2 == 128) __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void*)(dst + 8192), 16, v1, so, 0, 0);
  };
  auto stage_b = [&](int buf, int half, int nt, int ks) {
    char* dst = smem + buf * kWBuf + (1 + half) * kWHalf + H2 * 128 + w * 2048;
    const unsigned v0 = vB0 + (half ? 8u * kblk : 0u), v1 = v0 + cb, so = (unsigned)(nt0 + nt) * 16u * kblk + (unsigned)ks * 2u * cb;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)dst, 16, v0, so, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, (lds_void*)(dst + 1024), 16, v1, so, 0, 0);
  };

  // ---- fragment reads
  // (buffer 1's offsets in registers of their own: past the 64 KB of an instruction's offset hipcc adds each read's anew)
  int rdA[2][2], rdB[2];
#pragma unroll
  for (int buf = 0; buf < 2; ++buf) {
    rdA[buf][0] = buf * kWBuf + (64 * wr + li) * 128 + 16 * (gq ^ (li >> 1));
    rdA[buf][1] = buf * kWBuf + (64 * wr + li) * 128 + 16 * ((4 + gq) ^ (li >> 1));
    rdB[buf] = buf * kWBuf + kWHalf + H2 * 128 + wc * 4096 + lane * 16;
    asm volatile("" : "+v"(rdA[buf][0]), "+v"(rdA[buf][1]), "+v"(rdB[buf]));
  }
  const int second = kWHalf - (64 - H2 / 2) * 128 * wr;  // from a wave's rows in the first half to those in the second
  bf16x8 af[4][2], bfr[2][2][2];
  f32x4 acc[2][2][4][2];  // (192 rows: [1][..] of two row blocks)
#define WIDE_ACC(E) \
  acc[(E) >> 4][(E) < 16 ? ((E) >> 3) & 1 : ((E)-16) / (2 * I2)][(E) < 16 ? ((E) >> 1) & 3 : ((E)-16) / 2 % I2][(E)&1]
  auto zero_acc = [&]() {
#pragma unroll
    for (int e = 0; e < NE; ++e) WIDE_ACC(e) = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  zero_acc();
#define WIDE_READ_A(BUF, IH)                                                                  \
  _Pragma("unroll") for (int i = 0; i < ((IH) ? I2 : 4); ++i) {                               \
    const char* base = smem + ((IH) ? second : 0) + i * 2048;                                 \
    af[i][0] = *reinterpret_cast<const bf16x8*>(base + rdA[BUF][0]);                          \
    af[i][1] = *reinterpret_cast<const bf16x8*>(base + rdA[BUF][1]);                          \
  }
#define WIDE_READ_B(BUF)                                                                      \
  _Pragma("unroll") for (int jh = 0; jh < 2; ++jh)                                            \
  _Pragma("unroll") for (int jn = 0; jn < 2; ++jn) {                                          \
    const char* base = smem + jh * kWHalf + jn * 2048 + rdB[BUF];                             \
    bfr[jh][jn][0] = *reinterpret_cast<const bf16x8*>(base);                                  \
    bfr[jh][jn][1] = *reinterpret_cast<const bf16x8*>(base + 1024);                           \
  }
#define WIDE_MFMA(IH, JH1)                                                                    \
  __builtin_amdgcn_s_setprio(1);                                                              \
  _Pragma("unroll") for (int jj = 0; jj < 2; ++jj)                                            \
  _Pragma("unroll") for (int ks = 0; ks < 2; ++ks)                                            \
  _Pragma("unroll") for (int i = 0; i < ((IH) ? I2 : 4); ++i)                                 \
  _Pragma("unroll") for (int jn = 0; jn < 2; ++jn)                                            \
    acc[IH][JH1 ^ jj][i][jn] = mfma16(bfr[JH1 ^ jj][jn][ks], af[i][ks], acc[IH][JH1 ^ jj][i][jn]); \
  __builtin_amdgcn_s_setprio(0);

  int it = start;
  int nt = start / kt, k0 = start - nt * kt;
  // The launch's number, the same for all of its workgroups: this one has not ended yet, so its launch has added less
  // than the label's p.spx workgroups to their count (which may wrap: 2^32 is a multiple of 32; the 128-row kernel counts its
  // own there too).  What a launch that gave up left raised, or raised late, so means nothing to the next.  Wave 0 copies the count
  // to LDS ahead of the first stage, so that it has landed when that has (in the 128-row kernel a scalar load in front, and one
  // count for all labels, cost 0.8 to 2 us a launch; the addition behind the prologue instead of at the end 1 to 3 us where a
  // group takes few K-steps).  The number is read by an asm statement: before an ordinary read hipcc drains the copies in flight.
  if (w == 0)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(mk_rsrc(ended, 4), (lds_void*)(smem + 2 * kWBuf), 4, 0u, 0u, 0, 0);
  // prologue: K-step 0 complete, A0 / B0 / B1 of K-step 1 in flight
  stage_a(0, 0, 2 * k0);
  stage_b(0, 0, nt, 2 * k0);
  stage_b(0, 1, nt, 2 * k0);
  stage_a(0, 1, 2 * k0);
  stage_a(1, 0, 2 * k0 + 1);
  stage_b(1, 0, nt, 2 * k0 + 1);
  stage_b(1, 1, nt, 2 * k0 + 1);
  wait_vmc<kFly>();
  mbar();
  unsigned before;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
               : "=v"(before)
               : "v"((unsigned)(uintptr_t)(lds_void*)(smem + 2 * kWBuf))
               : "memory");
  const int launch = (int)((unsigned)__builtin_amdgcn_readfirstlane((int)before) / (unsigned)p.spx) + 1;

  const __amdgpu_buffer_rsrc_t rS = mk_rsrc(p.slabs, p.slab_bytes);
  auto block_of = [&](int jj) { return ((p.gpx - 1 - jj) * p.tiles_m + mt) * 8 + x; };
  auto slab_off = [&](int jj) { return (unsigned)(block_of(jj) * kWSlabFloats) * 4u + (unsigned)(tid * 16); };
  auto flag_of = [&](int jj) { return p.cnt + block_of(jj); };
  bool pending = false;  // the first part is stored as a partial tile, its flag not raised yet
  auto raise_flag = [&]() {  // after every wave's stores retired and a barrier
    if (tid == 0) __hip_atomic_store(flag_of(j), launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    pending = false;
  };
  int after_st = 0;  // VMEM stores younger than the copies in flight
  while (it < end) {
    const int k1 = min(kt, k0 + (end - it));
    it += k1 - k0;
    const bool more = it < end;
    if (wr == 1) mbar();  // group 1 one barrier behind through the K-loop (ping-pong)
    for (int k = k0; k < k1; ++k) {
      const bool last = k == k1 - 1;
      const bool st = !last || more;
      const int ks = 2 * k + 1, kn = last ? 0 : 2 * k + 2, nn = last ? nt + 1 : nt;
      // phase 1
      WIDE_READ_A(0, 0)
      WIDE_READ_B(0)
      stage_a(1, 1, ks);
      if (after_st == kWSlabSt) wait_vmc<kFly + kWSlabSt>();
      else if (after_st == kWE) wait_vmc<kFly + kWE>();
      else wait_vmc<kFly>();
      mread_bar();
      WIDE_MFMA(0, 0)
      mbar();
      // phase 2
      WIDE_READ_A(0, 1)
      if (st) {
        stage_a(0, 0, kn);
        stage_b(0, 0, nn, kn);
        stage_b(0, 1, nn, kn);
        if (after_st == kWSlabSt) wait_vmc<kFly + kWSlabSt>();
        else if (after_st == kWE) wait_vmc<kFly + kWE>();
        else wait_vmc<kFly>();
      } else {
        wait_vmc<0>();
      }
      after_st = 0;
      mread_bar();
      WIDE_MFMA(1, 1)
      mbar();
      // phase 3
      WIDE_READ_A(1, 0)
      WIDE_READ_B(1)
      if (st) {
        stage_a(0, 1, kn);
        wait_vmc<kFly>();
      }
      mread_bar();
      WIDE_MFMA(0, 0)
      mbar();
      if (pending) raise_flag();  // both groups are past phase 3's wait, which retired the stores
      // phase 4
      WIDE_READ_A(1, 1)
      if (st) {
        stage_a(1, 0, kn + 1);
        stage_b(1, 0, nn, kn + 1);
        stage_b(1, 1, nn, kn + 1);
        wait_vmc<kFly>();
      }
      mread_bar();
      WIDE_MFMA(1, 1)
      mbar();
    }
    if (wr == 0) mbar();  // pairs with group 1's last K-loop barrier

    // ---- end of a part: stored with a flag behind it, or the owner adds what the others stored
    const int n0 = (nt0 + nt) * 256;
    bool write = true;
    if (k0 != 0 || k1 != kt) {
      const int j_lo = grp_owner(nt * kt, p.q, p.r), j_hi = grp_owner(nt * kt + kt - 1, p.q, p.r);
      if (j != j_lo) {
        const unsigned own = slab_off(j);
#pragma unroll
        for (int e = 0; e < NE; ++e)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, WIDE_ACC(e)), rS, own, (unsigned)(e * 8192), 16);
        after_st = kWSlabSt;
        pending = true;
        if (!more) {  // nothing left to hide the drain behind
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          mbar();
          raise_flag();
        }
        write = false;
      } else {
        bool ok = true;
        for (int jj = j_lo + 1; jj <= j_hi; ++jj) {
          int* fl = flag_of(jj);
          if (tid == 0) {
            long spins = 0;
            while (__hip_atomic_load(fl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != launch) {
              if (++spins > p.spin_limit) {
                ok = false;  // a producer never published (cannot happen in a healthy launch)
                break;
              }
              __builtin_amdgcn_s_sleep(2);
            }
            if (ok) __hip_atomic_store(fl, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          mbar();  // every thread loads only after lane 0 saw the flag
          const unsigned off = slab_off(jj);
          u32x4 v[NE / 2];  // a window: half of the partial tile
#pragma unroll
          for (int e = 0; e < NE / 2; ++e) v[e] = __builtin_amdgcn_raw_buffer_load_b128(rS, off, (unsigned)(e * 8192), 16);
#pragma unroll
          for (int e = 0; e < NE; ++e) {
            WIDE_ACC(e) += __builtin_bit_cast(f32x4, v[e % (NE / 2)]);
            if (e < NE / 2) v[e] = __builtin_amdgcn_raw_buffer_load_b128(rS, off, (unsigned)((NE / 2 + e) * 8192), 16);
          }
        }
        // Lane 0 tells the others, by asm statements on the one LDS array: __syncthreads_and brings an object of its own, and
        // with two of them hipcc waits for every copy in flight ahead of each fragment read
        const unsigned told = (unsigned)(uintptr_t)(lds_void*)(smem + 2 * kWBuf + 64);
        if (tid == 0) asm volatile("ds_write_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" ::"v"(told), "v"((int)ok) : "memory");
        mbar();
        int all;
        asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(all) : "v"(told) : "memory");
        if (!__builtin_amdgcn_readfirstlane(all)) {
          const float nan = __builtin_nanf("");
#pragma unroll
          for (int e = 0; e < NE; ++e) WIDE_ACC(e) = f32x4{nan, nan, nan, nan};
        }
      }
    }
    if (write) {
      // ---- epilogue: acc[ih][jh][i][jn][r] = C[m0 + 128 ih + (64 or H2 / 2) wr + 16 i + li][n0 + 128 jh + 32 wc + 16 jn + 4 gq + r];
      // exactly kWE stores per wave (rows >= M fall outside the descriptor and are dropped)
      int e_lane = tid & 63;  // (opaque, so that nothing derived from it stays live across the K-loop)
      asm volatile("" : "+v"(e_lane));
      const int e_li = e_lane & 15, e_g = e_lane >> 4;
      const long c_rows = min(ROWS, p.M - m0);
      const __amdgpu_buffer_rsrc_t rC = mk_rsrc(p.C + (size_t)m0 * p.ldc, (unsigned)(c_rows * p.ldc * 2));
      if constexpr (glu8_epilogue(EPI)) {
        f32x4 bg[2], bu[2];
#pragma unroll
        for (int jh = 0; jh < 2; ++jh) {
          bg[jh] = bu[jh] = f32x4{0.f, 0.f, 0.f, 0.f};
          if constexpr (RES) {
            const float* fb = reinterpret_cast<const float*>(p.residual) + (n0 + 128 * jh + 32 * wc) / 2 + 4 * e_g;
            bg[jh] = *reinterpret_cast<const f32x4*>(fb);
            bu[jh] = *reinterpret_cast<const f32x4*>(fb + p.N / 2);
          }
        }
        if constexpr (RES) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int ih = 0; ih < 2; ++ih)
#pragma unroll
          for (int i = 0; i < (ih ? I2 : 4); ++i)
#pragma unroll
            for (int jh = 0; jh < 2; ++jh) {
              const int mr = 128 * ih + (ih ? H2 / 2 : 64) * wr + 16 * i + e_li;
              float o[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[ih][jh][i][0][r]),
                                                                __float_as_uint(acc[ih][jh][i][1][r]), false, false);
                o[r] = glu_act<glu8_act(EPI)>(__uint_as_float(s[0]) + bg[jh][r]) * (__uint_as_float(s[1]) + bu[jh][r]);
              }
              u32x2 v;
              v[0] = pack2bf(o[0], o[1]);
              v[1] = pack2bf(o[2], o[3]);
              const int oc = (n0 + 128 * jh + 32 * wc) / 2 + 4 * e_g;
              __builtin_amdgcn_raw_buffer_store_b64(v, rC, (unsigned)((mr * p.ldc + oc) * 2), 0, 0);
              __builtin_amdgcn_sched_barrier(0);
            }
      } else {
        const int cq = 16 * (e_g & 1) + 8 * (e_g >> 1);
        const __amdgpu_buffer_rsrc_t rR =
            mk_rsrc(RES ? p.residual + (size_t)m0 * p.ldr : p.residual, RES ? (unsigned)(c_rows * p.ldr * 2) : 0u);
#pragma unroll
        for (int ih = 0; ih < 2; ++ih) {
          u32x4 rv[4][2];
          if constexpr (RES) {
#pragma unroll
            for (int i = 0; i < (ih ? I2 : 4); ++i)
#pragma unroll
              for (int jh = 0; jh < 2; ++jh)
                rv[i][jh] = __builtin_amdgcn_raw_buffer_load_b128(
                    rR, (unsigned)(((128 * ih + (ih ? H2 / 2 : 64) * wr + 16 * i + e_li) * p.ldr + n0 + 128 * jh + 32 * wc + cq) * 2), 0, 0);
          }
#pragma unroll
          for (int i = 0; i < (ih ? I2 : 4); ++i)
#pragma unroll
            for (int jh = 0; jh < 2; ++jh) {
              const int mr = 128 * ih + (ih ? H2 / 2 : 64) * wr + 16 * i + e_li;
              float o[8];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[ih][jh][i][0][r]),
                                                                __float_as_uint(acc[ih][jh][i][1][r]), false, false);
                o[r] = __uint_as_float(s[0]);
                o[4 + r] = __uint_as_float(s[1]);
              }
              if constexpr (RES) {
                const u32x4 rw = rv[i][jh];
#pragma unroll
                for (int qd = 0; qd < 4; ++qd) {  // round like a bf16 GEMM output, then the bf16 add (HF)
                  o[2 * qd] = bf2f(f2bf(o[2 * qd])) + __uint_as_float(rw[qd] << 16);
                  o[2 * qd + 1] = bf2f(f2bf(o[2 * qd + 1])) + __uint_as_float(rw[qd] & 0xffff0000u);
                }
              }
              u32x4 v;
#pragma unroll
              for (int qd = 0; qd < 4; ++qd) v[qd] = pack2bf(o[2 * qd], o[2 * qd + 1]);
              const int nc = n0 + 128 * jh + 32 * wc + cq;
              __builtin_amdgcn_raw_buffer_store_b128(v, rC, (unsigned)((mr * p.ldc + nc) * 2), 0, 0);
            }
        }
      }
      after_st = kWE;
    }
    zero_acc();
    k0 = 0;
    ++nt;
  }
#undef WIDE_ACC
#undef WIDE_READ_A
#undef WIDE_READ_B
#undef WIDE_MFMA
  count_out();
}

namespace {
int cu_count() {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return cus;
}
}  // namespace

// Eligible: N % 256 == 0, K % 64 == 0, 16-B aligned A rows, ceil(M / 128) row tiles <= blocks per
// XCD label (32 on MI355X: M <= 4096), 32-bit buffer offsets.
int gemm_mid_ok(int M, int N, int K, long lda) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 256 || K % 64 || lda % 8 || lda < K) return 0;
  const int spx = cu_count() / 8;
  if ((M + 127) / 128 > spx) return 0;
  if ((long)N * K * 2 >= (1L << 32) || (127L * lda + K) * 2 >= (1L << 31)) return 0;
  return 1;
}

// Estimated us of a product on `groups` groups.  Its K-steps take 0.7 each, from some 120 working workgroups on 0.5 +
// 0.00165 a workgroup, or the weights' way from memory (4.5 TB/s), whichever is longer; its ends 5.6 for whole tiles, 8.1
// and 1.56 a part where every tile is cut into parts of as many K-steps, 10.5 and 1.56 a part otherwise, and 2.5 for each
// further tile of a group.  (Fitted to 1,480 launches of 1-32 row tiles, N 256-28,672, K 256-14,336: half of them within 5
// %, nine of ten within 16 %.)
static double mid_us(int M, int N, int K, int groups) {
  const int tm = (M + 127) / 128, tn = N / 256, kt = K / 64;
  const double iters = (double)tn * kt, q = iters / groups;
  const double step = fmax(0.7, 0.5 + 0.00165 * (groups < iters ? groups : iters) * tm);
  const double weights = (double)tn * 512 * K / 4.5e6;
  double ends, steps = q * step;
  if (tn % groups == 0) {
    ends = 5.6;
  } else if (groups % tn == 0 && kt % (groups / tn) == 0) {
    ends = 8.1 + 1.56 * (groups / tn);
  } else {
    ends = 10.5 + 1.56 * (groups > tn ? ceil(kt / (q > 1. ? q : 1.)) : 1.);
    steps = ceil(q) * step;
  }
  if (tn > groups) ends += 2.5 * ((double)tn / groups - 1.);
  return ends + (steps > weights ? steps : weights);
}

// Groups of ceil(M / 128) workgroups: the whole ones of each XCD, and those joined from the slots left over where they
// gain 3 % by the estimate (or no group has two K-steps).  More workgroups are no gain where the whole groups divide the
// tiles evenly.  us, whole groups -> with the joined ones: gate_up of Llama-3-8B at M 1093 272 -> 238, down 138 -> 128, down
// at M 1300 175 -> 156, 2200 338 -> 242, qkv at M 2600 158 -> 120; but qkv at M 1093 (24 tiles, 24 groups) 53.9 -> 63.4, o at
// M 1700 55.0 -> 60.7.
// Fewer groups an XCD where that gains 6 % by the estimate: every part of a tile costs its owner a partial tile of 128 KB,
// and unequal parts an end of their own, so a short K is better cut into few equal parts while much of the chip idles (K
// below 768 has too few K-steps to choose from).  us, all the groups that fit -> those taken: (130, 2048, 2048) 38.4 on 128
// groups -> 20.0 on 32, (300, 2048, 2048) 35.3 -> 20.5, (130, 3072, 2048) 31.1 -> 20.3 on 48, (1000, 3072, 2048) 28.6 -> 24.4
// on 24, (130, 2048, 8192) 45.0 -> 35.5 on 64, (384, 4096, 4096) 35.1 -> 30.1 on 64; over the projections of Llama-3-8B and
// 1B as planned at M 130-5000 (224 shapes) 0.94-1.96 times as fast, 1.055 in the mean, the worst qkv of 1B at M 1500 31.6 ->
// 33.6.
int gemm_mid_groups(int M, int N, int K) {
  const int spx = cu_count() / 8, tm = (M + 127) / 128, tn = N / 256;
  if (M <= 0 || tn <= 0 || K < 64 || tm > spx) return 0;
  const int whole = 8 * (spx / tm), all = whole + 8 * (spx % tm) / tm;
  int groups = mid_us(M, N, K, all) < 0.97 * mid_us(M, N, K, whole) || (long)tn * (K / 64) <= whole ? all : whole;
  double least = 0.94 * mid_us(M, N, K, groups);
  for (int g = 8; K >= 768 && g < whole; g += 8) {
    const double us = mid_us(M, N, K, g);
    if (us < least) {
      least = us;
      groups = g;
    }
  }
  return groups;
}

// Estimated us of a product on `groups` groups of the kernel with tiles of 256 or 192 rows (all XCDs').  A pair of K-steps takes
// 1.83 us, from some 70 working workgroups on 1.64 + 0.0027 a workgroup and 0.0048 more for each past 192, or the weights' way
// from memory; the ends 10.4 for whole tiles and, with partial tiles of 256 KB, 0.027 a workgroup and 2.48 a part besides.
// (256 rows: fitted to 12,900 launches of M 128-4096 at 11 sizes of N 2048-28,672, K 1024-14,336: half of them within 2.7 %,
// nine of ten within 7.5 %; the groups taken by it cost 0.9 % more than the best in the mean.  192 rows: to 520 launches of M
// 400-3700 at nine of those sizes, on another card: 3.2 and 8.2 %, the groups 0.6 %.)
struct WideTime {
  double step, base, per, over, whole, equal, uneven, part, wgs, further;
};
constexpr WideTime kWide256 = {1.83, 1.64, 0.0027, 0.0048, 10.4, 11.4, 12.5, 2.48, 0.027, 7.0};
constexpr WideTime kWide192 = {1.445, 1.586, 0.0022, 0.0041, 7.2, 6.4, 5.9, 2.16, 0.039, 5.2};

static double wide_us(int M, int N, int K, int groups, int rows) {
  const WideTime& f = rows == 192 ? kWide192 : kWide256;
  const int tm = (M + rows - 1) / rows, tn = N / 256, kt = K / 128;
  const double iters = (double)tn * kt, q = iters / groups, wgs = (groups < iters ? groups : iters) * tm;
  const double step = fmax(f.step, f.base + f.per * wgs) + f.over * fmax(0., wgs - 192.);
  const double weights = (double)tn * 512 * K / 5.0e6;
  double ends = f.whole, steps = q * step;
  if (tn % groups) {
    const bool equal = groups % tn == 0 && kt % (groups / tn) == 0;
    const double parts = equal ? (double)(groups / tn) : groups > tn ? ceil(kt / fmax(q, 1.)) : 1.;
    ends = (equal ? f.equal : f.uneven) + f.part * parts + f.wgs * wgs;
    if (!equal) steps = ceil(q) * step;
  }
  if (tn > groups) ends += f.further * ((double)tn / groups - 1.);
  return ends + fmax(steps, weights);
}

// Groups of that kernel and the estimate of its time on them; 0 groups where it is not measured (K below 1024) or
// does not take the sizes (each XCD as many column tiles).  From three row tiles on: with fewer, weights that take longer from
// memory than the products are slower ((391, 10240, 8192) 0.81 times as fast), and others gain nothing over gemm256.
static int wide_groups(int M, int N, int K, int min_tm, int rows, double* us) {
  const int spx = cu_count() / 8, tm = (M + rows - 1) / rows, tn = N / 256;
  *us = __builtin_huge_val();
  if (M <= 0 || tn <= 0 || K < 1024 || K % 128 || tn % 8 || tm < min_tm || tm > spx) return 0;
  int groups = 0;
  for (int gn = 8; gn <= 8 * (spx / tm); gn += 8) {
    const double t = wide_us(M, N, K, gn, rows);
    if (t < *us) {
      *us = t;
      groups = gn;
    }
  }
  return groups;
}

// Which kernel a product takes: the 256-row one where the estimates say 13 % less (527 of the 1,156 sizes of that sweep with
// three row tiles and more, 1.26 times as fast in the mean, none slower, the least 1.024; at 6.5 % less 656, 9 of them slower,
// (1001, 4096, 14336) 0.95).  Between those lines a call has nothing or 1-2 % of it, too little for sums of K in another order:
// prefill of Llama-3-8B, us of a call, 128 rows -> 256, and the ratio of the estimates of down: 660 tokens 11,902 -> 11,713
// (0.907), 900 13,256 -> 13,249 and 1,000 13,691 -> 13,738 (0.892), 1,093 16,175 -> 15,940, 15,942 -> 15,562 and 15,971 -> 15,877 on other
// cards (0.933), 1,350 18,905 -> 18,663 (0.892); below it 1,200 17,210 -> 16,636 (0.825), 1,280 17,578 -> 16,998, 1,500 19,876
// -> 19,585 (0.821), 1,700 22,519 -> 21,606 (0.782), 2,000 24,336 -> 23,693 (0.806).  us of a launch, 128 rows -> 256:
// Llama-3-8B's down at M 1500 168 -> 148, 2000 198 -> 172, 3000 322 -> 265, Llama-3.2-1B's down at 3400 115 -> 97; but o of
// Llama-3-8B at M 1093 51 -> 54, qkv at 640 41 -> 53: partial tiles of 256 KB a workgroup are 64 MB to write and read, some 25
// us of a full launch.
static int mid_pick(int M, int N, int K, bool* wide, double* us) {
  const int groups = gemm_mid_groups(M, N, K);
  *us = groups ? mid_us(M, N, K, groups) : __builtin_huge_val();
  double w_us;
  const int w_groups = groups ? wide_groups(M, N, K, 3, 256, &w_us) : 0;
  *wide = w_groups && w_us < 0.87 * *us;
  if (!*wide) return groups;
  *us = 1.1 * w_us;  // (beside gemm256: the step of Llama-3-8B at 3,000 tokens 34,732 us with it, 35,015 on this)
  return w_groups;
}

// Groups on which the 256-row kernel runs a product, 0: it does not; forced: where the rule would leave it to the other one, too.
int gemm_mid_wide_groups(int M, int N, int K, int forced) {
  bool wide;
  double us;
  if (forced) return wide_groups(M, N, K, 1, 256, &us);
  const int groups = mid_pick(M, N, K, &wide, &us);
  return wide ? groups : 0;
}

// Estimated us of the launch, infinite where the kernels do not take M.
double gemm_mid_us(int M, int N, int K) {
  bool wide;
  double us;
  if (mid_pick(M, N, K, &wide, &us)) return us;
  return M <= 0 || N < 256 ? 0. : __builtin_huge_val();
}

// ... of the kernel with tiles of 192 rows, which the caller asks for by the variant of that name: in front of the other two
// where fewer rows of its tiles lie past the prompt's end.
double gemm_mid_192_us(int M, int N, int K) {
  double us;
  return gemm_mid_groups(M, N, K) && wide_groups(M, N, K, 3, 192, &us) ? us : __builtin_huge_val();
}

// Workspace the launcher needs: partial slabs and behind them the counts of ended workgroups (bytes), and ready flags
// and counts (ints).
static long slabs_end() { return (long)cu_count() * 2 * kSlabFloats * 4; }
long gemm_mid_slab_bytes() { return slabs_end() + 8 * 128; }
// ready flags of the 256-row kernel's workgroups, and behind them the 128-row kernel's counts, one per (row tile, group)
int gemm_mid_counters(int M, int N) {
  (void)M;
  (void)N;
  return 2 * (cu_count() & ~7);
}

// epilogue 0: C = A B^T (+ residual, bf16 add after rounding); 4 / 6: SwiGLU / tanh-GELU GLU over 8-row [gate | up] groups
// (C has N / 2 columns; residual: null, or their fp32 bias [gate | up]).  slabs: gemm_mid_slab_bytes() bytes, the last 1024
// zero on first use; cnt: >= gemm_mid_counters() ints, zero on first use (the launch leaves them zero).  spin_limit: looks
// at a count before an owner hands its tile over (256 rows: at a flag, before it gives up and writes NaN), -1: the kernel's
// own.  variant: 0 default (by the estimates), 192 tiles of 192 rows (as the 128-row kernel where those do not take the sizes);
// A/B harness only: 32 / 64 the 128-row kernel with that K-step, 256 the 256-row kernel, + 1000 = DIAG 1 (split tiles not
// combined: timing only). BK 32 (6-stage ring) measured 5-20 % slower than BK 64 on every mid shape, with LDS bank conflicts on
// its 64-B A rows (profiles/gemm_mid_r6.md): kept as an A/B arm only.
int gemm_mid(const void* A, long lda, const void* B, void* C, long ldc, const void* residual, long ldr, int M, int N,
             int K, int epilogue, void* slabs, long slab_bytes, int* cnt, int n_cnt, hipStream_t s, int variant,
             int b_group, long spin_limit) {
  if (!gemm_mid_ok(M, N, K, lda)) return hipErrorInvalidValue;
  if (b_group != 1 && b_group != 8) return hipErrorInvalidValue;
  if (epilogue != MID_NONE && !glu8_epilogue(epilogue)) return hipErrorInvalidValue;
  if (!slabs || !cnt || slab_bytes < gemm_mid_slab_bytes() || n_cnt < gemm_mid_counters(M, N) ||
      slab_bytes >= (1L << 32))
    return hipErrorInvalidValue;
  bool wide;
  double us;
  int groups = mid_pick(M, N, K, &wide, &us);
  if (variant == 256 || variant == 192) {
    wide = true;
    groups = wide_groups(M, N, K, 1, variant, &us);
  } else if (variant) {
    wide = false;
  }
  // (its buffer descriptors span 256 rows of the operands, of C and of the residual in 32 bits)
  const bool spans = (255L * lda + K) * 2 < (1L << 31) && 512L * ldc < (1L << 32) && (!residual || 512L * ldr < (1L << 32));
  if (!groups || (wide && !spans)) {
    if (variant == 256) return hipErrorInvalidValue;
    wide = false;
  }
  const int rows = !wide ? 128 : variant == 192 ? 192 : 256;
  if (!wide) groups = gemm_mid_groups(M, N, K);
  const bool diag = variant >= 1000;
  const int bk = (variant % 1000) == 32 ? 32 : 64;
  GMid p{};
  p.A = (const bf16*)A;
  p.B = (const bf16*)B;
  p.C = (bf16*)C;
  p.residual = (const bf16*)residual;
  p.slabs = (float*)slabs;
  p.cnt = cnt;
  p.M = M;
  p.N = N;
  p.K = K;
  p.lda = lda;
  p.ldc = ldc;
  p.ldr = ldr;
  p.tiles_m = (M + rows - 1) / rows;
  p.tiles_n = N / 256;
  p.kt = K / (wide ? 128 : bk);
  const int grid = cu_count() & ~7;
  p.ended = (unsigned*)((char*)slabs + slabs_end());
  p.spin_limit = spin_limit >= 0 ? spin_limit : wide ? 1L << 22 : 128;
  p.spx = grid / 8;
  p.gn = groups;
  if (wide) p.tiles_n /= 8;  // an XCD's
  p.gpx = min(p.spx / p.tiles_m, p.gn / 8);  // (with fewer groups the other slots' workgroups end at once)
  const int iters = p.tiles_n * p.kt, shares = wide ? p.gn / 8 : p.gn;
  p.q = iters / shares;
  p.r = iters % shares;
  p.b_bytes = (unsigned)((long)N * K * 2);
  p.slab_bytes = (unsigned)slab_bytes;
  p.bgrp = b_group;
#define MID_LAUNCH(E, R, BKV, D) hipLaunchKernelGGL((gemm_mid_kernel<E, R, BKV, D>), dim3(grid), dim3(512), 0, s, p)
#define MID_BK(E, R)                       \
  do {                                     \
    if (diag) {                            \
      if (bk == 64) MID_LAUNCH(E, R, 64, 1); \
      else MID_LAUNCH(E, R, 32, 1);        \
    } else if (bk == 64) {                 \
      MID_LAUNCH(E, R, 64, 0);             \
    } else {                               \
      MID_LAUNCH(E, R, 32, 0);             \
    }                                      \
  } while (0)
#define WIDE_LAUNCH(E, R)                                                                            \
  do {                                                                                               \
    if (rows == 192) hipLaunchKernelGGL((gemm_wide_kernel<E, R, 192>), dim3(grid), dim3(512), 0, s, p); \
    else hipLaunchKernelGGL((gemm_wide_kernel<E, R, 256>), dim3(grid), dim3(512), 0, s, p);            \
  } while (0)
  if (wide) {
    if (epilogue == MID_SWIGLU8 && residual) WIDE_LAUNCH(MID_SWIGLU8, true);
    else if (epilogue == MID_GEGLU8 && residual) WIDE_LAUNCH(MID_GEGLU8, true);
    else if (epilogue == MID_SWIGLU8) WIDE_LAUNCH(MID_SWIGLU8, false);
    else if (epilogue == MID_GEGLU8) WIDE_LAUNCH(MID_GEGLU8, false);
    else if (epilogue == MID_REGLU8 && residual) WIDE_LAUNCH(MID_REGLU8, true);
    else if (epilogue == MID_REGLU8) WIDE_LAUNCH(MID_REGLU8, false);
    else if (residual) WIDE_LAUNCH(MID_NONE, true);
    else WIDE_LAUNCH(MID_NONE, false);
  } else if (epilogue == MID_SWIGLU8 && residual) MID_BK(MID_SWIGLU8, true);
  else if (epilogue == MID_GEGLU8 && residual) MID_BK(MID_GEGLU8, true);
  else if (epilogue == MID_SWIGLU8) MID_BK(MID_SWIGLU8, false);
  else if (epilogue == MID_GEGLU8) MID_BK(MID_GEGLU8, false);
  else if (epilogue == MID_REGLU8 && residual) MID_BK(MID_REGLU8, true);
  else if (epilogue == MID_REGLU8) MID_BK(MID_REGLU8, false);
  else if (residual) MID_BK(MID_NONE, true);
  else MID_BK(MID_NONE, false);
#undef MID_BK
#undef WIDE_LAUNCH
#undef MID_LAUNCH
  return hipGetLastError();
}

}  // namespace dab
