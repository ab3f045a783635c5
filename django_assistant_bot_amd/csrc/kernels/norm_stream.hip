// Decode projections of a few rows with the RMS norm in front of them:  C[M, N] = RMSNorm(x + residual) . W[N, K]^T, the
// norm's input being the split-K slabs of the projection before it (or plain rows).  M <= 4 (complete rows: 8), weights in the shuffle_weights
// layout, K <= 4096, M K_slice <= 32768.
//
// A decode layer of a few sequences is a chain of launches; the two norms of a layer are one small workgroup a row between
// two weight streams, 3.2 us each for 40 KB of work, most of it launch, round trip and drain.  Here every workgroup of the
// consuming projection normalises the rows itself: eight waves sum the slabs, add the residual and write the normalised
// slice of K to LDS (the same roundings as rmsnorm_slab_kernel), while the other four have their whole weight ring on its
// way, whose first loads take longer from HBM than the norm.  Every workgroup reads all slabs and the residual from L2 or
// the Infinity Cache, 40 KB a row and CU; 8 / M waves share a row, so that up to 4 rows come in one round trip.  Workgroup 0
// writes the new residual.
//
// us, norm launch and stream_gemm -> here, 4 slabs of K 4096 / 8 of K 2048: (1, 6144, 4096) 14.1 -> 12.0, 4 rows 14.6 ->
// 12.9; gated (1, 28672, 4096) 43.0 -> 40.1, 4 rows 43.8 -> 41.8; (1, 3072, 2048) 7.9 -> 6.3, 4 rows 8.2 -> 7.0; gated (1,
// 16384, 2048) 16.9 -> 15.5, 4 rows 16.9 -> 16.3.  5-8 rows, a wave each: (5, 3072, 2048) 8.2 -> 9.5, not taken of slabs.
// Complete rows (norm_rows; rows_stream.hip leaves them), up to 8, are one read each: 6 rows, norm launch and stream_gemm ->
// here, gated (28672, 4096) 42.4 -> 36.3, (6144, 4096) 16.4 -> 10.6, gated (16384, 2048) 18.5 -> 14.2, (3072, 2048) 10.5 -> 4.4.
//
// Weights: wave w of the tile's NWC compute waves holds RT 16-row blocks; a chunk is 32 k of them, 1 KB a block, MFMA A
// fragments straight to registers through a ring of DEP chunks (128 KB in flight a CU).  The rows are the B operand, in
// LDS for all of the slice, 16-B piece c of row m at c ^ m (reads of 16 rows: distinct banks); lanes past the last row read
// it again.  No barrier in the K loop: the waves run free.
#include <type_traits>

#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

struct NormStream {
  const void* slabs;  // [S][M][K]
  int S;
  long slab_stride;
  const bf16* residual;  // [M][K] or null
  const bf16* gain;      // [K]
  bf16* residual_out;    // [M][K] or null
  float eps;
  const bf16* W;
  void* out;  // [SO][M][N] slabs (SO > 1), or rows
  long ldo;
  int M, N, K, SO, kc;
  int glu;      // SwiGLU over 8-row [gate | up] groups
  int slab_f32; // SO > 1: the slabs in 32 bits
  int wgrp;     // row blocks per group of the weight copy
};

constexpr int kNormWaves = 8;
constexpr int kNormRows = 4;
constexpr int kNormX = 65536;  // bytes of the rows' slice

}  // namespace

// WPR: norm waves a row (8 / WPR rows); VPL: 8-column pieces a lane holds of its row (K <= 512 WPR VPL); U: slabs whose loads
// are in flight together
template <int RT, int NWC, int DEP, int WPR, int VPL, int U, typename ST>
__global__ __launch_bounds__(64 * (NWC + kNormWaves), 1) void norm_stream_kernel(NormStream p) {
  constexpr int BN = 16 * RT * NWC;
  __shared__ __attribute__((aligned(16))) char xs[kNormX + kNormWaves * 4];
  float* const red = reinterpret_cast<float*>(xs + kNormX);  // [norm wave]
  const int tile = blockIdx.x / p.SO, slice = blockIdx.x % p.SO;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k_begin = slice * p.kc, n0 = tile * BN;
  const int row_bytes = p.kc * 2;

  if (w >= NWC) {
    // ------------------------------------------------------------------ norm waves
    const int nw = w - NWC, nvec = p.K / 8;
    const int m = min(nw / WPR, p.M - 1);  // (waves past the last row repeat it and write nothing)
    const bool mine = nw / WPR < p.M;
    int iv[VPL];
    bool ok[VPL];
    u32x4 gain[VPL], h[VPL];  // h: the row (with the residual), bf16
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      const int i = (nw % WPR + k * WPR) * 64 + lane;
      ok[k] = mine && i < nvec;
      iv[k] = min(i, nvec - 1);
    }
    if constexpr (U == 0) {
#pragma unroll
      for (int k = 0; k < VPL; ++k) h[k] = reinterpret_cast<const u32x4*>((const bf16*)p.slabs + (size_t)m * p.K)[iv[k]];
#pragma unroll
      for (int k = 0; k < VPL; ++k) gain[k] = reinterpret_cast<const u32x4*>(p.gain)[iv[k]];
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();  // (the weights' loads start behind these, as below)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        float f[8];
        unpack8(h[k], f);
        if (ok[k]) {
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += f[j] * f[j];
        }
      }
    } else {
      u32x4 r[VPL];
      float v[VPL][8];
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        if (p.residual) r[k] = reinterpret_cast<const u32x4*>(p.residual + (size_t)m * p.K)[iv[k]];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[k][j] = 0.f;
      }
      const ST* base = (const ST*)p.slabs + (size_t)m * p.K;
      for (int s0 = 0; s0 < p.S; s0 += U) {
        SlabVec8<ST> a[VPL][U];
#pragma unroll
        for (int k = 0; k < VPL; ++k)
#pragma unroll
          for (int u = 0; u < U; ++u) a[k][u].load(base + (size_t)min(s0 + u, p.S - 1) * p.slab_stride + (size_t)iv[k] * 8);
        if (s0 == 0) {
#pragma unroll
          for (int k = 0; k < VPL; ++k) gain[k] = reinterpret_cast<const u32x4*>(p.gain)[iv[k]];
          __builtin_amdgcn_sched_barrier(0);
          // the weights' loads start behind these: queued behind 128 KB of them the rows came 1.5 us later
          __builtin_amdgcn_s_barrier();
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (s0 + u < p.S) {  // uniform
#pragma unroll
            for (int k = 0; k < VPL; ++k) a[k][u].add_to(v[k]);
          }
      }
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[k][j] = bf2f(f2bf(v[k][j]));
        if (p.residual) {
          float f[8];
          unpack8(r[k], f);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[k][j] = bf2f(f2bf(v[k][j] + f[j]));
        }
        h[k] = pack8(v[k]);
        if (ok[k]) {
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += v[k][j] * v[k][j];
        }
      }
    }
    ss = wave_sum_valu(ss);
    if (lane == 0) red[nw] = ss;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < WPR; ++q) t += red[nw / WPR * WPR + q];
    const float inv = rsqrtf(t / (float)p.K + p.eps);
    const int p0 = k_begin / 8, p1 = p0 + p.kc / 8;  // pieces of the slice
#pragma unroll
    for (int k = 0; k < VPL; ++k) {
      if (!ok[k] || iv[k] < p0 || iv[k] >= p1) continue;
      float x[8], f[8];
      unpack8(h[k], x);
      unpack8(gain[k], f);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = x[j] * inv * f[j];
      *reinterpret_cast<u32x4*>(xs + m * row_bytes + 16 * ((iv[k] - p0) ^ m)) = pack8(x);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (blockIdx.x == 0 && p.residual_out)
#pragma unroll
      for (int k = 0; k < VPL; ++k)
        if (ok[k]) reinterpret_cast<u32x4*>(p.residual_out + (size_t)m * p.K)[iv[k]] = h[k];
    return;
  }

  // -------------------------------------------------------------------- compute waves
  const int nch = p.kc / 32;
  const int cstride = p.wgrp * 1024;  // bytes from one chunk of a block to the next
  __amdgpu_buffer_rsrc_t rs[RT];
#pragma unroll
  for (int a = 0; a < RT; ++a) {
    const int b = n0 / 16 + RT * w + a;  // row block: fragment (b, c) at ((b / G) K/32 + c) G + b % G KB
    const size_t at = ((size_t)(b / p.wgrp) * (p.K / 32) + k_begin / 32) * p.wgrp + b % p.wgrp;
    // (a chunk past the slice reads zeros without traffic)
    rs[a] = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p.W) + at * 512, (short)0, (nch - 1) * cstride + 1024, 0x00020000);
  }
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 wr[DEP][RT];
  auto load = [&](int slot, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < RT; ++a)
      wr[slot][a] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs[a], lane * 16, c * cstride, 2));
  };
#pragma unroll
  for (int j = 0; j < DEP; ++j) load(j, j);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  f32x4 acc[RT][2];  // even and odd chunks: two chains of MFMAs
#pragma unroll
  for (int a = 0; a < RT; ++a) acc[a][0] = acc[a][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int m = min(li, p.M - 1);
  const char* xr = xs + m * row_bytes;
  auto step = [&](int j, int c) __attribute__((always_inline)) {
    const bf16x8 x = *reinterpret_cast<const bf16x8*>(xr + 16 * ((4 * c + g) ^ m));
#pragma unroll
    for (int a = 0; a < RT; ++a) acc[a][j & 1] = mfma16(wr[j][a], x, acc[a][j & 1]);
  };
  int c0 = 0;
  for (; c0 + DEP < nch; c0 += DEP) {
#pragma unroll
    for (int j = 0; j < DEP; ++j) {
      step(j, c0 + j);
      load(j, c0 + j + DEP);  // right behind its MFMAs
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int j = 0; j < DEP; ++j)
    if (c0 + j < nch) step(j, c0 + j);

  // acc[a]: weight rows 16 (RT w + a) + 4 g + r of column (row of X) li
  const bool live = li < p.M;
#pragma unroll
  for (int a = 0; a < RT; ++a) {
    const f32x4 v = acc[a][0] + acc[a][1];
    const int n = n0 + 16 * (RT * w + a) + 4 * g;
    if (p.glu) {
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {  // lanes 0..31: rows 0-7 (gate) and, from lane + 32, 8-15 (up)
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[r]), __float_as_uint(v[r]), false, false);
        o[r] = silu_f(__uint_as_float(s[0])) * __uint_as_float(s[1]);
      }
      if (live && g < 2)
        *reinterpret_cast<u32x2*>((bf16*)p.out + (size_t)li * p.ldo + (n0 + 16 * (RT * w + a)) / 2 + 4 * g) =
            u32x2{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
    } else if (p.SO > 1) {
      // (write-through: the slab lines leave this L2 as they are written, not at the kernel's end)
      const size_t at = ((size_t)slice * p.M + li) * p.N + n;
      const auto so = __builtin_amdgcn_make_buffer_rsrc(p.out, (short)0, p.SO * p.M * p.N * (p.slab_f32 ? 4 : 2), 0x00020000);
      if (live) {
        if (p.slab_f32)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), so, (unsigned)(at * 4), 0, 16);
        else
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])}, so, (unsigned)(at * 2), 0, 16);
      }
    } else if (live) {
      *reinterpret_cast<u32x2*>((bf16*)p.out + (size_t)li * p.ldo + n) = u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
    }
  }
}

// Whether the kernel takes M rows of K in SO slices, bn weight rows a workgroup (64 or 128)
int norm_stream_ok(int M, int N, int K, int SO, int bn) {
  if (M < 1 || M > kNormRows || K < 256 || K % 8 || K > 4096) return 0;
  if (SO < 1 || K % (32 * SO) || (long)M * (K / SO) * 2 > kNormX) return 0;
  if ((bn != 64 && bn != 128) || N <= 0 || N % bn || (long)SO * M * N * 4 >= (1L << 31) || (long)N * K * 2 >= (1L << 31)) return 0;
  return 1;
}

// slabs: S of fp32 (slabs_f32) or bf16 [M][K]; residual, residual_out: both or neither.  glu: 8-row groups, SO 1.
int norm_stream(const void* slabs, int S, int slabs_f32, const void* residual, const void* gain, void* residual_out, float eps,
                const void* W, void* out, long ldo, int M, int N, int K, int SO, int out_f32, int glu, int w_group, int bn,
                hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (!norm_stream_ok(M, N, K, SO, bn) || S < 1 || (glu && SO > 1) || ldo % 4 || (!residual) != (!residual_out)) return hipErrorInvalidValue;
  if (w_group < 1 || N % (16 * w_group)) return hipErrorInvalidValue;
  const NormStream p = {slabs, S, (long)M * K, (const bf16*)residual, (const bf16*)gain, (bf16*)residual_out, eps, (const bf16*)W,
                        out, ldo, M, N, K, SO, K / SO, glu, out_f32, w_group};
  const dim3 grid(N / bn * SO), block(64 * (4 + kNormWaves));
#define NS_LAUNCH(RT, DEP, WPR, VPL, U, ST) \
  hipLaunchKernelGGL((norm_stream_kernel<RT, 4, DEP, WPR, VPL, U, ST>), grid, block, 0, s, p)
#define NS_TILE(WPR, VPL, U, ST)                      \
  do {                                                \
    if (bn == 64) NS_LAUNCH(1, 32, WPR, VPL, U, ST);  \
    else NS_LAUNCH(2, 16, WPR, VPL, U, ST);           \
  } while (0)
#define NS_SLABS(WPR, VPL)                                                             \
  do {                                                                                 \
    constexpr int u = VPL > 2 ? 4 : 8; /* (what 168 registers hold) */                 \
    if (slabs_f32) NS_TILE(WPR, VPL, u / 2, float);                                    \
    else if (S <= 4) NS_TILE(WPR, VPL, 4, bf16);                                       \
    else NS_TILE(WPR, VPL, u, bf16);                                                   \
  } while (0)
#define NS_ROWS(WPR)                               \
  do {                                             \
    if (K <= 2048) NS_SLABS(WPR, (4 + WPR - 1) / WPR); \
    else NS_SLABS(WPR, 8 / WPR);                   \
  } while (0)
  if (M == 1) NS_ROWS(8);
  else if (M == 2) NS_ROWS(4);
  else NS_ROWS(2);
#undef NS_SLABS
#undef NS_TILE
#undef NS_ROWS
#undef NS_LAUNCH
  return hipGetLastError();
}

// ... of up to 8 complete rows (no slabs, no residual); with more than 4 a norm wave each.  Slices of whole eights of 16-B
// pieces, in which the rows are permuted.  bn: 48, 64 or 128 weight rows a workgroup, a compute wave for 16.
//
// With the rows read once the ring need not cover the norm's reads of slabs, and short ones are quicker; 48 rows find 256 CUs
// work where 64 find 192.  us, 6 rows, 4 waves with rings of 32 or, gated, 16 chunks of two blocks -> rings of 8: (6144, 4096) in
// two slices 12.3 -> 11.4 on 64 rows, 10.7 on 48, (3072, 2048) in four 5.9 -> 5.0, 4.4; gated (28672, 4096) 37.3 -> 36.4, (16384,
// 2048) 15.0 -> 14.4 (one row 15.7 -> 13.7).  Gated on 64 rows 41.2 and 16.3.
int norm_rows_ok(int M, int N, int K, int SO, int bn) {
  return M >= 1 && M <= kNormWaves && (bn == 48 || bn == 64 || bn == 128) && N > 0 && N % bn == 0 && K >= 256 && K <= 4096 && SO >= 1 &&
         K % (64 * SO) == 0 && (long)M * (K / SO) * 2 <= kNormX && (long)SO * M * N * 4 < (1L << 31) && (long)N * K * 2 < (1L << 31);
}

int norm_rows(const void* x, const void* gain, float eps, const void* W, void* out, long ldo, int M, int N, int K, int SO, int out_f32,
              int glu, int w_group, int bn, hipStream_t s) {
  if (!norm_rows_ok(M, N, K, SO, bn) || (glu && SO > 1) || ldo % 4) return hipErrorInvalidValue;
  if (w_group < 1 || N % (16 * w_group)) return hipErrorInvalidValue;
  const NormStream p = {x, 1, (long)M * K, nullptr, (const bf16*)gain, nullptr, eps, (const bf16*)W,
                        out, ldo, M, N, K, SO, K / SO, glu, out_f32, w_group};
  const dim3 grid(N / bn * SO);
#define NS_LAUNCH(NWC, WPR)                                                                                        \
  do {                                                                                                             \
    constexpr int few = (4 + WPR - 1) / WPR, more = 8 / WPR;                                                       \
    const dim3 block(64 * (NWC + kNormWaves));                                                                     \
    if (K <= 2048) hipLaunchKernelGGL((norm_stream_kernel<1, NWC, 8, WPR, few, 0, bf16>), grid, block, 0, s, p);   \
    else hipLaunchKernelGGL((norm_stream_kernel<1, NWC, 8, WPR, more, 0, bf16>), grid, block, 0, s, p);            \
  } while (0)
#define NS_ROWS(WPR)                       \
  do {                                     \
    if (bn == 48) NS_LAUNCH(3, WPR);       \
    else if (bn == 64) NS_LAUNCH(4, WPR);  \
    else NS_LAUNCH(8, WPR);                \
  } while (0)
  if (M == 1) NS_ROWS(8);
  else if (M == 2) NS_ROWS(4);
  else if (M <= 4) NS_ROWS(2);
  else NS_ROWS(1);
#undef NS_ROWS
#undef NS_LAUNCH
  return hipGetLastError();
}

}  // namespace dab
