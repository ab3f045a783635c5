// bf16 GEMM C[M,N] = A[M,K] . B[N,K]^T (+ residual, or a GLU over 8-row [gate | up] groups) for prompts of some 100 to 2,000
// tokens, B in the ops.shuffle_weights fragment layout: the projections whose tiles of 128 x 256 and more are fewer than the
// CUs.  gemm_mid cuts those along K, and its owners add the parts: 8 us and more a launch, whatever the product.  Here tiles
// of 32 x 64 to 128 x 256 as the sizes ask for, each a workgroup that walks the whole K (or, in front of a norm that sums
// them, a K-slice that it leaves as an fp32 slab), with no exchange between workgroups.
//
// What bounds it, by copies, reads and products measured apart (a K-tile is 64 deep): a CU takes some 120 GB/s of operands
// out of its L2 but 60-70 of what comes from memory, as layer after layer of weights does: 80-100 KB in flight over 1.3 us.
// So tiles load as many bytes as fit LDS ahead of their products, and the larger ones run as fast with weights from L2
// (192 x 128: 0.57 us a K-tile) as from memory (0.57-0.6).  Asking the L2 for later K-tiles is no gain, as a CU's loads return
// in order (64 x 128: 52 -> 62 us at (256, 2048, 8192)), nor are fragments straight into registers, or read a K-tile ahead.
//   * Small tiles: the waves form KG groups that take the K-tiles in turn, each with a ring of its own, and meet in LDS at the
//     end: two to four waves a SIMD whose reads and products overlap (64 x 64: 0.30 -> 0.17 us a K-tile out of L2, from
//     memory 0.24; 96 x 64: 0.38 -> 0.22 and 0.28).
//   * The copies of a later K-tile go out one at a time between the products: all of them in front hold the waves up until
//     the last is accepted (192 x 128: 0.65 -> 0.57 us a K-tile, 128 x 256 0.80 -> 0.77).
//
// us, cold weights, gemm_mid / gemm256 -> here: (260, 2048, 2048) 19.4 -> 9.7, (515, 3072, 2048) 22.2 -> 13.6, (260, 6144,
// 4096) 35 -> 26, (800, 6144, 4096) 55 -> 48, (140, 28672, 4096) GLU 75 -> 60; with a residual (300, 4096, 4096) 29 -> 21, (1200, 4096,
// 4096) 57 -> 47.  Launches alone are quicker here, too, where the estimates, which know no epilogue, lie within the plan's 7 % and
// gemm_mid keeps the product: (600, 4096, 4096) with a residual 37.6 / 34.7, (1093, 4096, 4096) 51 / 45, (1093, 6144, 4096) 62.5 / 58.
#include <cmath>
#include <type_traits>

#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

struct FragParams {
  const bf16* A;
  const bf16* B;  // shuffle_weights layout, [N][K]
  bf16* C;
  const bf16* residual;
  const float* glu_bias;  // fp32 [gate N / 2 | up N / 2]
  float* slabs;           // [slices][M][N] fp32 instead of C
  int M, N, K;
  int lda, ldc, ldr;
  int slices;
  int bgrp;
  int act;  // GLU epilogue: 4, 6 or 7
};

enum { FRAG_PLAIN = 0, FRAG_GLU = 1, FRAG_SLAB = 2 };

typedef __attribute__((address_space(3))) void frag_lds;

template <int N>
__device__ __forceinline__ void frag_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t frag_rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

}  // namespace

// BM x BN tiles by KG groups of WM x WN waves, each group over a ring of NS K-tiles in LDS, filled by LDS-DMA NS - 1 ahead with
// counted waits and one barrier a K-tile.
template <int BM, int BN, int WM, int WN, int KG, int NS, int EPI>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_frag_kernel(FragParams p) {
  constexpr int W = WM * WN, MI = BM / (16 * WM), NI = BN / (16 * WN);  // 16 x 16 tiles of a wave
  constexpr int kA = BM * 128, kStage = (BM + BN) * 128, kDma = (BM + BN) / 8 / W;
  constexpr int UN = MI * NI / 2;  // units of the epilogue: two neighbouring column blocks of a row block
  static_assert((BM + BN) % (8 * W) == 0 && BM % (16 * WM) == 0 && BN % (32 * WN) == 0, "whole copies and pairs of tiles a wave");
  static_assert(NS == 3 || NS == 4, "waits for up to two K-tiles ahead");
  static_assert(BM * BN * 4 * (KG - 1) <= KG * NS * kStage, "the groups' sums meet in the ring");
  __shared__ __attribute__((aligned(16))) char smem[KG * NS * kStage];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wv / W, w = wv % W, wm = w / WN, wn = w % WN;

  // neighbouring ids on one XCD: the row tiles of a column block read its weights from one L2
  const int tiles_m = (p.M + BM - 1) / BM, nwg = gridDim.x, xcd = blockIdx.x % 8, q8 = nwg / 8, r8 = nwg % 8;
  const int id0 = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + blockIdx.x / 8;
  const int tiles = EPI == FRAG_SLAB ? tiles_m * ((p.N + BN - 1) / BN) : 1;
  const int slice = EPI == FRAG_SLAB ? id0 / tiles : 0, id = id0 - slice * tiles;
  const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;

  // copies of 1 KB: 8 rows of A (16-B chunk c of row r at c ^ ((r >> 1) & 7), swizzled at the source; rows past the matrix
  // read the last one), or a 16 x 32 fragment of B in lane order (blocks past the matrix read the last one)
  const __amdgpu_buffer_rsrc_t ra = frag_rsrc(p.A, (unsigned)(((size_t)(p.M - 1) * p.lda + p.K) * 2));
  const __amdgpu_buffer_rsrc_t rb = frag_rsrc(p.B, (unsigned)((size_t)p.N * p.K * 2));
  const unsigned cb = (unsigned)p.bgrp * 1024u, kblk = (unsigned)(p.K / 32) * 1024u;
  unsigned at[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int c = i * W + w;
    if (c < BM / 8) {
      const int r = 8 * c + (lane >> 3);
      at[i] = (unsigned)((min(m0 + r, p.M - 1) * p.lda + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2);
    } else {
      const int f = c - BM / 8, rb_ = min(n0 / 16 + f / 2, p.N / 16 - 1);
      at[i] = (unsigned)(rb_ / p.bgrp) * p.bgrp * kblk + (unsigned)(rb_ % p.bgrp) * 1024u + (unsigned)(f & 1) * cb + lane * 16;
    }
  }
  const int kt = p.K / 64;
  const int k0 = EPI == FRAG_SLAB ? kt * slice / p.slices : 0, nk = (EPI == FRAG_SLAB ? kt * (slice + 1) / p.slices : kt) - k0;
  // K-tiles kg, kg + KG, ... are group kg's
  const int steps = (nk + KG - 1) / KG, mine = (nk - kg + KG - 1) / KG;
  char* const ring = smem + kg * NS * kStage;
  auto stage1 = [&](int i, char* dst, unsigned sa, unsigned sb) __attribute__((always_inline)) {
    // (which operand: known here but for the copies of a step that holds both)
    if (i * W + W <= BM / 8 || (i * W < BM / 8 && i * W + w < BM / 8))
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (frag_lds*)(dst + i * W * 1024), 16, (unsigned)at[i], sa, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (frag_lds*)(dst + i * W * 1024), 16, (unsigned)at[i], sb, 0, 0);
  };
  auto stage = [&](int buf, int t) __attribute__((always_inline)) {
    const unsigned k = (unsigned)(k0 + kg + KG * t);
#pragma unroll
    for (int i = 0; i < kDma; ++i) stage1(i, ring + buf * kStage + w * 1024, k * 128u, k * 2u * cb);
  };
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < mine) stage(t, t);

  const int sw = (li >> 1) & 7;
  int rdA[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) rdA[ks] = wm * (BM / WM) * 128 + li * 128 + 16 * ((4 * ks + g) ^ sw);
  const int rdB = kA + wn * (BN / WN) * 128 + lane * 16;
  f32x4 acc[MI][NI];
#pragma unroll
  for (int j = 0; j < MI; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  auto step = [&](int t, auto more) __attribute__((always_inline)) {
    constexpr bool kMore = decltype(more)::value;
    if (kMore) frag_wait<(NS - 2) * kDma>();
    else if (NS == 4 && mine - 1 - t >= 2) frag_wait<2 * kDma>();
    else if (NS >= 3 && mine - 1 - t >= 1) frag_wait<kDma>();
    else frag_wait<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last K-tile's reads: its buffer is filled next
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const char* s = ring + buf * kStage;
    char* const dst = ring + (buf == 0 ? NS - 1 : buf - 1) * kStage + w * 1024;
    const unsigned k = (unsigned)(k0 + kg + KG * (t + NS - 1)), sa = k * 128u, sb = k * 2u * cb;
    if (kMore || KG == 1 || t < mine) {
      bf16x8 af[MI][2], bfr[NI][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int j = 0; j < MI; ++j) af[j][ks] = *reinterpret_cast<const bf16x8*>(s + j * 2048 + rdA[ks]);
#pragma unroll
        for (int i = 0; i < NI; ++i) bfr[i][ks] = *reinterpret_cast<const bf16x8*>(s + rdB + i * 2048 + ks * 1024);
      }
      __builtin_amdgcn_s_setprio(1);
      constexpr int kMul = 2 * MI * NI;
#pragma unroll
      for (int x = 0; x < kMul; ++x) {
        if constexpr (kMore) {
#pragma unroll
          for (int d = 0; d < kDma; ++d)
            if (d * kMul / kDma == x) {
              __builtin_amdgcn_sched_barrier(0);
              stage1(d, dst, sa, sb);
              __builtin_amdgcn_sched_barrier(0);
            }
        }
        const int ks = x / (MI * NI), j = x / NI % MI, i = x % NI;
        acc[j][i] = mfma16(bfr[i][ks], af[j][ks], acc[j][i]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    buf = buf == NS - 1 ? 0 : buf + 1;
  };
  int t = 0;
  for (; t + NS - 1 < mine; ++t) step(t, std::true_type());
  for (; t < steps; ++t) step(t, std::false_type());

  // the groups' sums: unit u is finished by group u % KG, which adds the others' from LDS
  if constexpr (KG > 1) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int x = kg - u % KG - 1 + (kg <= u % KG ? KG : 0);  // 0 .. KG - 2 behind the owner; the owner: KG - 1
      if (x != KG - 1) {
        char* dst = smem + ((u * (KG - 1) + x) * W + w) * 2048 + lane * 16;
        *reinterpret_cast<f32x4*>(dst) = acc[u / (NI / 2)][2 * (u % (NI / 2))];
        *reinterpret_cast<f32x4*>(dst + 1024) = acc[u / (NI / 2)][2 * (u % (NI / 2)) + 1];
      }
    }
    __syncthreads();
  }

  // acc[j][i][r] = C[m0 + wm BM / WM + 16 j + li][n0 + wn BN / WN + 16 i + 4 g + r]
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    if (KG > 1 && kg != u % KG) continue;
    const int j = u / (NI / 2), i = 2 * (u % (NI / 2));
    f32x4 a = acc[j][i], b = acc[j][i + 1];
#pragma unroll
    for (int x = 0; x < KG - 1; ++x) {
      const char* src = smem + ((u * (KG - 1) + x) * W + w) * 2048 + lane * 16;
      a += *reinterpret_cast<const f32x4*>(src);
      b += *reinterpret_cast<const f32x4*>(src + 1024);
    }
    const int m = m0 + wm * (BM / WM) + 16 * j + li, n = n0 + wn * (BN / WN) + 16 * i;
    if (m >= p.M || n >= p.N) continue;
    if constexpr (EPI == FRAG_SLAB) {
      float* dst = p.slabs + ((size_t)slice * p.M + m) * p.N + n + 4 * g;
      *reinterpret_cast<f32x4*>(dst) = a;
      *reinterpret_cast<f32x4*>(dst + 16) = b;
    } else if constexpr (EPI == FRAG_GLU) {
      // 8-row [gate | up] groups inside each block: lanes 0-31 take block i's, lanes 32-63 block i + 1's
      f32x4 bg = {0.f, 0.f, 0.f, 0.f}, bu = {0.f, 0.f, 0.f, 0.f};
      if (p.glu_bias) {
        const float* fb = p.glu_bias + n / 2 + 4 * g;
        bg = *reinterpret_cast<const f32x4*>(fb);
        bu = *reinterpret_cast<const f32x4*>(fb + p.N / 2);
      }
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[r]), __float_as_uint(b[r]), false, false);
        const float gate = __uint_as_float(s[0]) + bg[r], up = __uint_as_float(s[1]) + bu[r];
        o[r] = (p.act == 4 ? glu_act<GLU_SILU>(gate) : p.act == 6 ? glu_act<GLU_GELU>(gate) : glu_act<GLU_RELU>(gate)) * up;
      }
      *reinterpret_cast<u32x2*>(p.C + (size_t)m * p.ldc + n / 2 + 4 * g) = u32x2{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
    } else {
      // 8 columns a lane
      const int nc = n + 16 * (g & 1) + 8 * (g >> 1);
      float o[8];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[r]), __float_as_uint(b[r]), false, false);
        o[r] = __uint_as_float(s[0]);
        o[4 + r] = __uint_as_float(s[1]);
      }
      if (p.residual) {
        const u32x4 rw = *reinterpret_cast<const u32x4*>(p.residual + (size_t)m * p.ldr + nc);
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // round like a bf16 GEMM output, then the bf16 add (HF)
          o[2 * q] = bf2f(f2bf(o[2 * q])) + __uint_as_float(rw[q] << 16);
          o[2 * q + 1] = bf2f(f2bf(o[2 * q + 1])) + __uint_as_float(rw[q] & 0xffff0000u);
        }
      }
      u32x4 v;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = pack2bf(o[2 * q], o[2 * q + 1]);
      *reinterpret_cast<u32x4*>(p.C + (size_t)m * p.ldc + nc) = v;
    }
  }
}

namespace {

// The tiles, and what their times were fitted with: us = start + round c + c K-tiles (step + busy b) + out M N / 10^6, c tiles
// on the busiest of 256 CUs, b the share of them that work; or the weights' way from memory (5.6 TB/s and 3 us), whichever is
// longer.  The second five: as slabs, `out` for each of them.  (2,100 launches of M 96-2300, 19 pairs of N 1024-28,672 and K
// 1024-14,336, and 4,800 of K-slices: half of them within 5 %, nine of ten within 14 %; the tile chosen by it is 0.1 % slower
// than the best in the mean.)
struct FragTime {
  float start, round, step, busy, out;
};
struct FragTile {
  int bm, bn;
  FragTime whole, slab;
};
constexpr FragTile kFrag[] = {
    {32, 64, {1.79f, 0.f, 0.157f, 0.019f, 2.16f}, {1.45f, 1.60f, 0.133f, 0.041f, 1.70f}},
    {64, 64, {1.15f, 0.f, 0.224f, 0.023f, 1.14f}, {1.43f, 1.43f, 0.184f, 0.064f, 0.80f}},
    {96, 64, {0.96f, 0.01f, 0.282f, 0.f, 1.52f}, {1.80f, 1.28f, 0.286f, 0.f, 0.99f}},
    {64, 128, {1.07f, 0.f, 0.360f, 0.f, 1.16f}, {1.78f, 2.13f, 0.341f, 0.035f, 0.67f}},
    {128, 128, {1.55f, 0.77f, 0.447f, 0.034f, 1.06f}, {2.19f, 2.31f, 0.440f, 0.084f, 0.61f}},
    {192, 128, {1.93f, 1.26f, 0.560f, 0.062f, 0.82f}, {2.52f, 2.91f, 0.578f, 0.087f, 0.54f}},
    {128, 256, {0.64f, 2.34f, 0.725f, 0.052f, 0.85f}, {3.18f, 3.80f, 0.712f, 0.122f, 0.46f}}};
constexpr int kFrags = sizeof(kFrag) / sizeof(kFrag[0]);

float frag_tile_us(const FragTile& t, int M, int N, int K, int slices) {
  const FragTime& f = slices > 1 ? t.slab : t.whole;
  const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * slices, c = (tiles + 255) / 256;
  const float busy = (tiles < 256 ? tiles : 256) / 256.f;
  const float us = f.start + f.round * c + K / 64 / slices * c * (f.step + f.busy * busy) + f.out * 1e-6f * slices * M * N;
  return fmaxf(us, 2.f * N * K / 5.6e6f + 3.f);
}

}  // namespace

// The tile with the least estimate for a product in so many K-slices (1: whole).
static int frag_tile(int M, int N, int K, int slices) {
  int best = 0;
  for (int i = 1; i < kFrags; ++i)
    if (frag_tile_us(kFrag[i], M, N, K, slices) < frag_tile_us(kFrag[best], M, N, K, slices)) best = i;
  return best;
}

// Its time in us, infinite outside the sizes that were measured.
double frag_us(int M, int N, int K, int slices) {
  if (M <= 64 || M > 4096 || N < 1024 || K < 1024 || K % 64 || N % 32 || slices < 1 || K / 64 < slices) return __builtin_huge_val();
  return frag_tile_us(kFrag[frag_tile(M, N, K, slices)], M, N, K, slices);
}

// Shapes the kernel takes: whole K-tiles and pairs of weight blocks, 31-bit offsets into A, 32-bit ones into B.
int gemm_frag_ok(long M, long N, long K, long lda) {
  return M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 32 == 0 && lda % 8 == 0 && lda >= K && (M * lda + K) * 2 < (1L << 31) &&
         N * K * 2 < (1L << 32);
}

// epilogue 0: C = A B^T (+ residual, bf16 add after rounding); 4 / 6 / 7: SwiGLU / tanh-GELU / ReLU GLU over 8-row [gate | up]
// groups (C has N / 2 columns; glu_bias: null, or fp32 [gate | up]).  slabs: [slices][M][N] fp32 sums instead of C.
// tile: -1 by the estimate.
int gemm_frag(const void* A, long lda, const void* B, void* C, long ldc, const void* residual, long ldr, const void* glu_bias,
              void* slabs, int slices, int M, int N, int K, int epilogue, int b_group, int tile, hipStream_t s) {
  if (!gemm_frag_ok(M, N, K, lda) || (b_group != 1 && b_group != 8) || N % (16 * b_group)) return hipErrorInvalidValue;
  if (slabs ? slices < 1 || slices > K / 64 || epilogue || residual || glu_bias
            : !C || ldc % 8 || ldc < 0 || ldr % 8 || ldr < 0 || ldc >= (1L << 31) || ldr >= (1L << 31))
    return hipErrorInvalidValue;
  if (epilogue ? !glu8_epilogue(epilogue) || residual != nullptr : glu_bias != nullptr) return hipErrorInvalidValue;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C | (uintptr_t)residual | (uintptr_t)glu_bias | (uintptr_t)slabs) % 16)
    return hipErrorInvalidValue;
  const FragParams p = {(const bf16*)A, (const bf16*)B, (bf16*)C, (const bf16*)residual, (const float*)glu_bias, (float*)slabs,
                        M, N, K, (int)lda, (int)ldc, (int)ldr, slices, b_group, epilogue};
#define FRAG_AS(T, WM, WN, KG, NS)                                                                                          \
  case T: {                                                                                                                \
    constexpr int BM = kFrag[T].bm, BN = kFrag[T].bn;                                                                       \
    const dim3 grid(((M + BM - 1) / BM) * ((N + BN - 1) / BN) * (slabs ? slices : 1)), block(64 * WM * WN * KG);            \
    if (slabs) hipLaunchKernelGGL((gemm_frag_kernel<BM, BN, WM, WN, KG, NS, FRAG_SLAB>), grid, block, 0, s, p);             \
    else if (epilogue) hipLaunchKernelGGL((gemm_frag_kernel<BM, BN, WM, WN, KG, NS, FRAG_GLU>), grid, block, 0, s, p);      \
    else hipLaunchKernelGGL((gemm_frag_kernel<BM, BN, WM, WN, KG, NS, FRAG_PLAIN>), grid, block, 0, s, p);                  \
    break;                                                                                                                 \
  }
  switch (tile >= 0 ? tile : frag_tile(M, N, K, slabs ? slices : 1)) {
    FRAG_AS(0, 2, 2, 4, 3)
    FRAG_AS(1, 2, 2, 2, 3)
    FRAG_AS(2, 2, 2, 2, 3)
    FRAG_AS(3, 2, 4, 2, 3)
    FRAG_AS(4, 2, 4, 1, 4)
    FRAG_AS(5, 4, 2, 1, 3)
    FRAG_AS(6, 4, 4, 1, 3)
    default: return hipErrorInvalidValue;
  }
#undef FRAG_AS
  return hipGetLastError();
}

}  // namespace dab
