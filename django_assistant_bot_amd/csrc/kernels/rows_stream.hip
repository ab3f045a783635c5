// Decode projections of up to 8 rows that end in the residual stream:  C[M, N] = X[M, K] . W[N, K]^T + residual, W in the
// shuffle_weights layout (o and down of a decoder layer).
//
// A split-K stream leaves slabs, which either a norm launch sums (4.5-4.8 us between two weight streams) or every workgroup of
// the next projection.  Here a workgroup has 16 weight rows (or 8) over the whole K, so the rows leave complete and the next
// projection normalises them itself (norm_rows in norm_stream.hip).  What bounds it: the weights from memory, the launch and two
// round trips, and, with more rows, the reads of X, all of which every workgroup takes out of L2:
//   * a lane takes 16 B of X; 8 lanes take 128 B of a row, 64 k: the pieces of one chunk of 32 k go to columns 0-7 of the MFMA's
//     second operand, those of the next chunk to columns 8-15, and each chunk's product is kept in sums of its own, of which half
//     the columns count.  A load for two chunks, of whole lines: (4096, 14336) at 6 rows 24 -> 20 us, (4096, 4096) 9.5 -> 7.3 (a
//     load a chunk of 16 rows' 64 B, with rings of 16 chunks).
//   * pairs of chunks w, w + NW, ... are wave w's, so that a workgroup reads 16 or 32 KB in a row; weights and X straight to
//     registers through a ring of DEP pairs, no LDS and no barrier until the waves' sums meet.  Deeper rings are slower (24 chunks
//     8.9 us, 16 9.5, 8 7.3-8.2 at (4096, 4096)).
//
// us, split-K stream with bf16 slabs / that and the norm -> here, 6 rows, weights of many copies in turn: (2048, 2048) 4.8 / 7.6 ->
// 3.9, (2048, 8192) 8.9 / 11.7 -> 8.3, (4096, 4096) 8.9 / 11.7 -> 7.3, (4096, 14336) 20.5 / 23.4 -> 19.7, (3072, 3072) 6.2 / 8.9 ->
// 5.8; not better (5120, 13824) 25.0 / 29.3 -> 30.5, which no model with a norm in the projection has (K up to 4096 there).
#include <type_traits>

#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

struct RowsStream {
  const bf16* X;  // [M][K], rows ldx apart
  const bf16* W;
  const bf16* residual;  // [M][N]
  bf16* out;             // [M][N]
  int M, N, K, ldx;
  int wgrp;  // row blocks per group of the weight copy
};

}  // namespace

// NW waves, rings of DEP pairs of chunks, ROWS weight rows a workgroup (8: the other half of a block's lanes repeats them)
template <int NW, int DEP, int ROWS>
__global__ __launch_bounds__(64 * NW, 1) void rows_stream_kernel(RowsStream p) {
  __shared__ __attribute__((aligned(16))) f32x4 sums[NW - 1][64];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, li = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x * ROWS / 16, n = ROWS * blockIdx.x + 4 * g, m = min(li & 7, p.M - 1);
  const int pairs = p.K / 64, np = (pairs - w + NW - 1) / NW;  // pairs w, w + NW, ... of chunks
  const int cs = p.wgrp * 1024, stride = NW * 2 * cs;          // bytes from one chunk of a block to the next, from one pair of the wave
  // fragment (b, c) at ((b / G) K/32 + c) G + b % G KB; pairs past K read zeros without traffic
  const size_t at = ((size_t)(b / p.wgrp) * 2 * pairs + 2 * w) * p.wgrp + b % p.wgrp;
  const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p.W) + at * 512, (short)0, np > 0 ? (np - 1) * stride + cs + 1024 : 0, 0x00020000);
  const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p.X), (short)0, ((p.M - 1) * p.ldx + p.K) * 2, 0x00020000);
  const int vw = ROWS == 16 ? lane * 16 : (lane & ~8) * 16 + 128 * (blockIdx.x & 1);
  const int vx = (m * p.ldx + 32 * (li >> 3) + 8 * g) * 2;
  bf16x8 wf[DEP][2], xf[DEP];
  auto load = [&](int slot, int c) __attribute__((always_inline)) {
    wf[slot][0] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, vw, c * stride, 2));
    wf[slot][1] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, vw, c * stride + cs, 2));
    xf[slot] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rx, vx, (w + NW * c) * 128, 0));
  };
#pragma unroll
  for (int j = 0; j < DEP; ++j) load(j, j);
  __builtin_amdgcn_sched_barrier(0);
  u32x2 res = {0u, 0u};
  if (w == 0 && 4 * g < ROWS) res = *reinterpret_cast<const u32x2*>(p.residual + (size_t)m * p.N + n);
  f32x4 even = {0.f, 0.f, 0.f, 0.f}, odd = {0.f, 0.f, 0.f, 0.f};  // sums of the pairs' first chunks (columns 0-7) and second (8-15)
  auto step = [&](int j) __attribute__((always_inline)) {
    even = mfma16(wf[j][0], xf[j], even);
    odd = mfma16(wf[j][1], xf[j], odd);
  };
  int c0 = 0;
  for (; c0 + DEP < np; c0 += DEP) {  // (as many pairs as the ring holds: none but its own loads)
#pragma unroll
    for (int j = 0; j < DEP; ++j) {
      step(j);
      load(j, c0 + j + DEP);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int j = 0; j < DEP; ++j)
    if (c0 + j < np) step(j);
  f32x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = even[r] + __shfl_xor(odd[r], 8, 64);
  if (w) sums[w - 1][lane] = v;
  __syncthreads();
  if (w) return;
#pragma unroll
  for (int i = 0; i < NW - 1; ++i) v += sums[i][lane];
  if (li >= p.M || 4 * g >= ROWS) return;
  // v[r] = C[li][n + r]; rounded like a bf16 GEMM output, then the bf16 add
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = bf2f(f2bf(v[r])) + bf2f((uint16_t)(res[r >> 1] >> (16 * (r & 1))));
  *reinterpret_cast<u32x2*>(p.out + (size_t)li * p.N + n) = u32x2{pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
}

// Whether the kernel takes the sizes: up to 8 rows, whole pairs of chunks, 31-bit offsets.
int rows_stream_ok(int M, int N, int K, long ldx, int w_group) {
  return M > 0 && M <= 8 && N > 0 && w_group > 0 && N % (16 * w_group) == 0 && K >= 256 && K % 64 == 0 && ldx >= K && ldx % 8 == 0 &&
         (M * ldx + K) * 2 < (1L << 31) && (long)w_group * (K / 32) * 1024 < (1L << 31);
}

int rows_stream(const void* X, long ldx, const void* W, const void* residual, void* out, int M, int N, int K, int w_group,
                hipStream_t s, int tile) {
  if (!rows_stream_ok(M, N, K, ldx, w_group) || !residual || !out) return hipErrorInvalidValue;
  if (((uintptr_t)X | (uintptr_t)W) % 16 || ((uintptr_t)residual | (uintptr_t)out) % 8) return hipErrorInvalidValue;
  const RowsStream p = {(const bf16*)X, (const bf16*)W, (const bf16*)residual, (bf16*)out, M, N, K, (int)ldx, w_group};
  // 8 weight rows a workgroup where 16 leave CUs without one (us of 16 / 8 rows, 6 rows of X: (2048, 8192) 9.5 / 8.3, (2048,
  // 2048) 4.2 / 3.9, (2048, 5632) 7.4 / 6.6, (3072, 3072) 5.8 / 7.4); with a long K 16 waves ((4096, 14336) 20.1 -> 19.7, (4096,
  // 4096) 7.3 -> 7.8)
  if (tile < 0) tile = N < 3072 ? 1 : K > 8192 ? 2 : 0;
  switch (tile) {
    case 0: hipLaunchKernelGGL((rows_stream_kernel<8, 4, 16>), dim3(N / 16), dim3(512), 0, s, p); break;
    case 1: hipLaunchKernelGGL((rows_stream_kernel<8, 4, 8>), dim3(N / 8), dim3(512), 0, s, p); break;
    case 2: hipLaunchKernelGGL((rows_stream_kernel<16, 3, 16>), dim3(N / 16), dim3(1024), 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace dab
