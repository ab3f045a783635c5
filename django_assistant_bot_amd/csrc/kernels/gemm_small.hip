// bf16 MFMA GEMMs  C[M,N] = A[M,K] . B[N,K]^T (+bias) (+GELU) (+residual), both operands row-major, for the encoder's
// projections below the sizes that fill gemm256: one question, a few dozen short texts, a few thousand tokens.
//
// gemm_small_kernel, as long as tiles of 16 x 16 to 32 x 64 (64 x 64 where K is long) are no more than the CUs.  At M =
// 19 a projection is 1-5 MB of weights and a chain of round trips, so what counts is how many workgroups ask for the
// weights at once and how much of K a wave walks alone.  The 128 x 128 tiles of gemm.hip make N / 128 workgroups (6 at N
// = 768) that step through K one 64-wide tile and one drained queue at a time.  Here N = 768 makes 48 workgroups a row
// tile; their 8 waves split K, each with an LDS ring of its own: no barrier until the sums meet.  What bounds it is a
// CU's share of the operands from past its L2, 60 GB/s; so the tile grows with M only as far as the CUs stay full.
//   * LDS-DMA of 8 rows x 128 B, not fragments straight into registers: a load of 16 rows x 64 B runs at 38 GB/s a CU
//     even out of L2, whole 128-B lines at 120-150 (us at (19, 768, 3072): 7.8 -> 5.2, (19, 768, 768): 4.1 -> 3.0);
//   * two pieces in flight a wave for the 16-wide tiles, one for the larger ones (the eight waves are 64-128 KB in
//     flight already; a second piece measured the same and took the second workgroup's LDS).
//
// gemm_ring_kernel above that: tiles of 32 x 64 to 128 x 256 over an LDS ring, one barrier a K-tile and counted waits, so
// the loads of the next K-tiles stay in flight (gemm.hip drains its queue every K-tile).  A K-tile takes 0.26-0.66 us, with
// the tile's size, not with what is left of the ring (4 and 6 buffers, fragments read a K-tile ahead and K rotated by column
// block measured the same), so what counts is how many tiles the busiest CU has and how large they are: ring_tile.
//
// us at (M, N, K), cold weights: gemm.hip's 128 x 128 (from M = 1024 gemm256) -> tiles of 64 x 64 -> here:
//     19, 768, 768   11.9 -> 3.0     19, 2304, 768  12.0 -> 3.4     19, 3072, 768  15.9 -> 4.0     19, 768, 3072  44.2 -> 5.2
//    256, 768, 768   13.9 -> 3.9    256, 2304, 768  14.3 -> 6.4    256, 3072, 768  14.9 -> 8.1    256, 768, 3072  34.8 -> 8.6
//    930, 768, 768   16.1 -> 7.2 -> 6.5     930, 2304, 768  16.8 -> 11.0 -> 9.5    930, 3072, 768  20.8 -> 12.0 -> 10.6
//   1700, 768, 768    8.7 -> 8.0           1700, 2304, 768  14.3 -> 11.8          1700, 3072, 768  25.5 (gemm256) -> 16.7
//   2900, 768, 768   12.7 -> 11.1          2900, 768, 3072 (128 x 128, with the norm behind it) 40.3 -> 30.0
// Epilogues round as gemm.hip does.
#include <type_traits>

#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

struct SmallParams {
  const bf16* A;
  const bf16* B;
  bf16* C;
  const bf16* bias;
  const bf16* residual;
  int M, N, K;
  int lda, ldb, ldc, ldr;
  int work;  // AHEAD: workgroups with a tile; those behind them read the next launch's weights
  float* slabs;  // SLAB: the slices' fp32 sums [slices][M][N] instead of C
  int slices;
  Upcoming next;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const bf16* base, int rows, int ld, int K) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(base), (short)0, (int)(((size_t)(rows - 1) * ld + K) * 2), 0x00020000);
}

}  // namespace

// The epilogue of the split-K tiles: thread e < BM BN / 4 sums 4 columns of a row over the waves' partial tiles.  Its bias
// and residual are loaded at the kernel's start: behind the barrier they were one more round trip of the chain.
template <int E>
struct SmallTail {
  u32x2 bias[E], residual[E];
};

// element i of the thread: row r, columns c .. c + 3 of the tile
template <int BN, int NT>
__device__ __forceinline__ void small_at(int i, int& r, int& c) {
  const int e = threadIdx.x + NT * i;
  r = e / (BN / 4);
  c = 4 * (e % (BN / 4));
}

template <int BM, int BN, int NT, int E>
__device__ __forceinline__ SmallTail<E> small_tail(const SmallParams& p, int m0, int n0) {
  SmallTail<E> t;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    int r, c;
    small_at<BN, NT>(i, r, c);
    const bool live = r < BM && m0 + r < p.M && n0 + c < p.N;  // N % 4 == 0 (launcher)
    t.bias[i] = t.residual[i] = u32x2{0u, 0u};
    if (live && p.bias) t.bias[i] = *reinterpret_cast<const u32x2*>(p.bias + n0 + c);
    if (live && p.residual) t.residual[i] = *reinterpret_cast<const u32x2*>(p.residual + (size_t)(m0 + r) * p.ldr + n0 + c);
  }
  return t;
}

template <int BM, int BN, int LDN, int W, bool GELU, int E>
__device__ __forceinline__ void small_finish(const SmallParams& p, const SmallTail<E>& t, const float (*part)[BM * LDN], int m0,
                                             int n0) {
#pragma unroll
  for (int i = 0; i < E; ++i) {
    int r, c;
    small_at<BN, 64 * W>(i, r, c);
    if (r >= BM || m0 + r >= p.M || n0 + c >= p.N) continue;
    const int at = r * LDN + c;
    f32x4 s = *reinterpret_cast<const f32x4*>(&part[0][at]);
#pragma unroll
    for (int k = 1; k < W; ++k) s += *reinterpret_cast<const f32x4*>(&part[k][at]);
    if (p.bias) {
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] += bf2f((uint16_t)(t.bias[i][q >> 1] >> (16 * (q & 1))));
    }
    if constexpr (GELU) {
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] = gelu_erf(s[q]);
    }
    if (p.residual) {
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] = bf2f(f2bf(s[q])) + bf2f((uint16_t)(t.residual[i][q >> 1] >> (16 * (q & 1))));
    }
    *reinterpret_cast<u32x2*>(p.C + (size_t)(m0 + r) * p.ldc + n0 + c) = u32x2{pack2bf(s[0], s[1]), pack2bf(s[2], s[3])};
  }
}

// neighbouring ids on one XCD: the row tiles of a column block read its weights from one L2
__device__ __forceinline__ int small_id(int nwg) {
  const int xcd = blockIdx.x % 8, q8 = nwg / 8, r8 = nwg % 8;
  return (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + blockIdx.x / 8;
}

// The arguments in one round of scalar loads, ahead of the branch on `work` (a second round behind it: 0.15 us a launch)
__device__ __forceinline__ void small_args(const SmallParams& p) {
  asm volatile("" ::"s"(p.A), "s"(p.B), "s"(p.C), "s"(p.bias), "s"(p.residual), "s"(p.M), "s"(p.N), "s"(p.K), "s"(p.lda), "s"(p.ldb),
               "s"(p.ldc), "s"(p.ldr), "s"(p.work));
}

typedef __attribute__((address_space(3))) void small_lds;

template <int N>
__device__ __forceinline__ void small_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// K-pieces of 64 go round the W waves: piece w + W j is wave w's, through a ring of D pieces of its own in LDS.
template <int MT, int NT, int W, int D, bool GELU, bool AHEAD = false>
__global__ __launch_bounds__(64 * W) void gemm_small_kernel(SmallParams p) {
  if (AHEAD) small_args(p);
  if (AHEAD && __builtin_expect((int)blockIdx.x >= p.work, 0)) return read_upcoming<512>(p.next, p.work);
  constexpr int BM = 16 * MT, BN = 16 * NT, LDN = BN + 4;  // LDN: fp32 row of a partial tile, off the bank period
  constexpr int kA = BM * 128, kPiece = kA + BN * 128, kDma = 2 * MT + 2 * NT;
  constexpr int kRing = W * D * kPiece, kPart = W * BM * LDN * 4;
  constexpr bool kOver = kRing + kPart > 80 * 1024;  // the sums over the ring: one more barrier, less LDS
  constexpr int E = (BM * BN / 4 + 64 * W - 1) / (64 * W);
  // one array: with two the compiler knows which of them the copies write, and waits for all copies before each read
  __shared__ __attribute__((aligned(16))) char smem[kOver ? (kRing > kPart ? kRing : kPart) : kRing + kPart];
  float(*part)[BM * LDN] = reinterpret_cast<float(*)[BM * LDN]>(smem + (kOver ? 0 : kRing));
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (p.M + BM - 1) / BM, id = small_id(AHEAD ? p.work : (int)gridDim.x);
  const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;
  const SmallTail<E> tail = small_tail<BM, BN, 64 * W, E>(p, m0, n0);

  // rows past the matrix read the last one (their results are not stored); byte offsets fit 31 bits (launcher)
  const __amdgpu_buffer_rsrc_t ra = rows_rsrc(p.A, p.M, p.lda, p.K), rb = rows_rsrc(p.B, p.N, p.ldb, p.K);
  unsigned va[2 * MT], vb[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int r = 8 * i + (lane >> 3);
    va[i] = (unsigned)((min(m0 + r, p.M - 1) * p.lda + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2);
  }
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) {
    const int r = 8 * i + (lane >> 3);
    vb[i] = (unsigned)((min(n0 + r, p.N - 1) * p.ldb + 8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2);
  }
  char* const ring = smem + w * (D * kPiece);
  const int pieces = p.K / 64, mine = (pieces - w + W - 1) / W;  // <= 0: none
  auto load = [&](int slot, int j) __attribute__((always_inline)) {
    char* dst = ring + slot * kPiece;
    const unsigned so = (unsigned)(w + W * j) * 128u;
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (small_lds*)(dst + kA + i * 1024), 16, (unsigned)vb[i], so, 0, 0);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (small_lds*)(dst + i * 1024), 16, (unsigned)va[i], so, 0, 0);
  };
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < mine) load(d, d);
  const int sw = (li >> 1) & 7;
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  for (int j = 0; j < mine; ++j) {
    const int ahead = min(D, mine - j) - 1;  // pieces after j in flight
    static_assert(D <= 3, "waits for up to two pieces ahead");
    if (ahead >= 2) small_wait<2 * kDma>();
    else if (ahead == 1) small_wait<kDma>();
    else small_wait<0>();
    const char* src = ring + slot * kPiece + li * 128;
    bf16x8 fb[2][NT], fa[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = 16 * ((4 * h + g) ^ sw);
#pragma unroll
      for (int i = 0; i < NT; ++i) fb[h][i] = *reinterpret_cast<const bf16x8*>(src + kA + i * 2048 + at);
#pragma unroll
      for (int t = 0; t < MT; ++t) fa[h][t] = *reinterpret_cast<const bf16x8*>(src + t * 2048 + at);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read: the slot is filled again
    if (j + D < mine) load(slot, j + D);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[i][t] = mfma16(fb[h][i], fa[h][t], acc[i][t]);
    slot = slot == D - 1 ? 0 : slot + 1;
  }

  if constexpr (kOver) __syncthreads();
  // acc[i][j][r] = C[m0 + 16 j + li][n0 + 16 i + 4 g + r]
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) *reinterpret_cast<f32x4*>(&part[w][(16 * j + li) * LDN + 16 * i + 4 * g]) = acc[i][j];
  __syncthreads();
  small_finish<BM, BN, LDN, W, GELU, E>(p, tail, part, m0, n0);
}

// The same split-K tiles with the LayerNorm of their input in front: A = LayerNorm(X) gain + offset of the rows of X, K = 256
// S wide; the column block at 0 writes the normalised rows to `normed` (the next residual).  A LayerNorm launch between
// two projections is 3.2 us, all of it a launch and two round trips; here every workgroup normalises its rows itself (a
// wave 2 MT of them, in the lane order and with the sums of layernorm_rows_kernel: the same bits) while its weights,
// asked for before, are on their way.  LayerNorm + projection at (19, 2304, 768): 3.2 + 4.9 us -> 4.8; (19, 3072, 768): 3.2 +
// 5.4 -> 5.4; the encoder's forward of one question 437 -> 344 us.
struct SmallNorm {
  const bf16* gain;
  const bf16* offset;
  bf16* normed;
  float eps;
};

template <int MT, int S, bool GELU>
__global__ __launch_bounds__(512) void gemm_ln_kernel(SmallParams p, SmallNorm nm) {
  small_args(p);
  asm volatile("" ::"s"(nm.gain), "s"(nm.offset), "s"(nm.normed), "s"(nm.eps));
  if (__builtin_expect((int)blockIdx.x >= p.work, 0)) return read_upcoming<512>(p.next, p.work);
  constexpr int BM = 16 * MT, BN = 16, LDN = BN + 4, W = 8, K = 256 * S, LDA = 2 * K + 16;  // bytes of an LDS row
  __shared__ __attribute__((aligned(16))) float part[W][BM * LDN];
  __shared__ __attribute__((aligned(16))) char rows[BM * LDA];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (p.M + BM - 1) / BM, id = small_id(p.work);
  const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;

  u32x2 xv[2 * MT][S], gv[S], ov[S];
#pragma unroll
  for (int r = 0; r < 2 * MT; ++r) {
    if (m0 + w + 8 * r >= p.M) break;  // wave-uniform
    const u32x2* xr = reinterpret_cast<const u32x2*>(p.A + (size_t)(m0 + w + 8 * r) * p.lda);
#pragma unroll
    for (int c = 0; c < S; ++c) xv[r][c] = xr[c * 64 + lane];
  }
#pragma unroll
  for (int c = 0; c < S; ++c) {
    gv[c] = reinterpret_cast<const u32x2*>(nm.gain)[c * 64 + lane];
    ov[c] = reinterpret_cast<const u32x2*>(nm.offset)[c * 64 + lane];
  }
  const bf16* wr = p.B + (size_t)min(n0 + li, p.N - 1) * p.ldb + 8 * g;
  bf16x8 fb[2][2];  // K-pieces w and w + 8, as in gemm_small_kernel
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (64 * (w + W * i) < K)
#pragma unroll
      for (int h = 0; h < 2; ++h) fb[i][h] = *reinterpret_cast<const bf16x8*>(wr + 64 * (w + W * i) + 32 * h);
  constexpr int E = (BM * BN / 4 + 64 * W - 1) / (64 * W);
  const SmallTail<E> tail = small_tail<BM, BN, 64 * W, E>(p, m0, n0);
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int r = 0; r < 2 * MT; ++r) {
    const int m = m0 + w + 8 * r;
    if (m >= p.M) break;  // the LDS row keeps what it held: it meets only results that are not stored
    float v[S][4];
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < S; ++c) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        v[c][2 * j] = __uint_as_float(xv[r][c][j] << 16);
        v[c][2 * j + 1] = __uint_as_float(xv[r][c][j] & 0xffff0000u);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) s += v[c][j];
    }
    s = wave_sum_valu(s);
    const float mean = s / (float)K;
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < S; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float d = v[c][j] - mean;
        sq += d * d;
      }
    sq = wave_sum_valu(sq);
    const float inv = rsqrtf(sq / (float)K + nm.eps);
#pragma unroll
    for (int c = 0; c < S; ++c) {
      float o[4];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        o[2 * j] = (v[c][2 * j] - mean) * inv * __uint_as_float(gv[c][j] << 16) + __uint_as_float(ov[c][j] << 16);
        o[2 * j + 1] = (v[c][2 * j + 1] - mean) * inv * __uint_as_float(gv[c][j] & 0xffff0000u) +
                       __uint_as_float(ov[c][j] & 0xffff0000u);
      }
      const u32x2 y = {pack2bf(o[0], o[1]), pack2bf(o[2], o[3])};
      *reinterpret_cast<u32x2*>(rows + (w + 8 * r) * LDA + (c * 64 + lane) * 8) = y;
      if (n0 == 0) reinterpret_cast<u32x2*>(nm.normed + (size_t)m * K)[c * 64 + lane] = y;
    }
  }
  __syncthreads();
  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (64 * (w + W * i) < K)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[j] = mfma16(fb[i][h], *reinterpret_cast<const bf16x8*>(rows + (16 * j + li) * LDA + 128 * (w + W * i) + 64 * h + 16 * g), acc[j]);
#pragma unroll
  for (int j = 0; j < MT; ++j) *reinterpret_cast<f32x4*>(&part[w][(16 * j + li) * LDN + 4 * g]) = acc[j];
  __syncthreads();
  small_finish<BM, BN, LDN, W, GELU, E>(p, tail, part, m0, n0);
}

// Attention over a few packed tokens with the output projection behind it: y = attention(qkv) w^T + b + residual, T <= 32
// KB, heads of D = 32 or 64.  Apart these are two launches that wait for each other, and the first is a dozen workgroups on
// 256 CUs.  Here a wave of the projection's split-K tile (its K-pieces w and w + 8 are one head of 64 or two of 32)
// computes the attention of those heads for the tile's 16 rows itself, from qkv out of the L2, and feeds it to its MFMAs
// from registers: the accumulators of O^T = V^T P^T are the projection's operand once its weights come in the same order of
// columns (two runs of 4 for one of 8).  Every column block repeats the attention, 12 MFMAs and 8 exponentials a lane
// and head.  What bounds it is the chain qkv -> scores -> row maximum -> V -> projection, and a CU's reads of qkv: whole
// lines, through LDS (fragments of 16 rows x 64 B straight into registers: 6.1 us against 4.9 at 19 tokens, H 768).  K
// and V share their rows in LDS.  One question of 19 tokens, 12 layers of 768: 298 -> 257 us; weights
// from HBM 305 -> 282.
// Arithmetic as in flash_kernel (attention.hip) and gemm_small_kernel: scores and sums fp32, P and O rounded to bf16.
struct SmallAttention {
  const bf16* qkv;  // [M, 3 K]
  const int* cu;
  int batch;
  float scale_log2;
};

template <int D, int KB>
__global__ __launch_bounds__(512) void gemm_attn_kernel(SmallParams p, SmallAttention at) {
  small_args(p);
  asm volatile("" ::"s"(at.qkv), "s"(at.cu), "s"(at.batch), "s"(at.scale_log2));
  if (__builtin_expect((int)blockIdx.x >= p.work, 0)) return read_upcoming<512>(p.next, p.work);
  constexpr int W = 8, LDN = 20, KT = 2 * KB, ND = D / 32, HP = 64 / D;  // HP: heads of a 64-wide piece
  // a wave's rows of 128 B: 16 of Q, 16 of the weights, 32 KB of K and, once the scores are there, of V
  constexpr int kW = 2048, kKV = 4096, kWave = kKV + KB * 4096;
  constexpr float kMasked = -__builtin_huge_valf();
  __shared__ __attribute__((aligned(16))) float part[W][16 * LDN];
  __shared__ __attribute__((aligned(16))) char rows[W * kWave];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_m = (p.M + 15) / 16, id = small_id(p.work);
  const int m0 = (id % tiles_m) * 16, n0 = (id / tiles_m) * 16;
  const SmallTail<1> tail = small_tail<16, 16, 64 * W, 1>(p, m0, n0);
  const int H = p.K, last = p.M - 1, ld = 3 * H;
  const int query = min(m0 + li, last);
  char* const ws = rows + w * kWave;

  // whole lines: a load is 8 rows of 128 B
  const int r8 = lane >> 3, c8 = lane & 7;
  bf16x8 q[2][2], k[2][4 * KB], v[2][4 * KB], wt[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c0 = 64 * (w + W * i);
    if (c0 >= H) break;  // wave-uniform
    const bf16* base = at.qkv + c0 + 8 * c8;
#pragma unroll
    for (int t = 0; t < 2; ++t) q[i][t] = *reinterpret_cast<const bf16x8*>(base + (size_t)min(m0 + 8 * t + r8, last) * ld);
#pragma unroll
    for (int t = 0; t < 4 * KB; ++t) k[i][t] = *reinterpret_cast<const bf16x8*>(base + H + (size_t)min(8 * t + r8, last) * ld);
#pragma unroll
    for (int t = 0; t < 4 * KB; ++t) v[i][t] = *reinterpret_cast<const bf16x8*>(base + 2 * H + (size_t)min(8 * t + r8, last) * ld);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      wt[i][t] = *reinterpret_cast<const bf16x8*>(p.B + (size_t)min(n0 + 8 * t + r8, p.N - 1) * p.ldb + c0 + 8 * c8);
  }
  // the query's sequence: the last start at or before it, the first one after it
  int lo = 0, hi = p.M;
  for (int b0 = 0; b0 <= at.batch; b0 += 64) {
    const int starts = at.cu[min(b0 + lane, at.batch)], n = min(64, at.batch + 1 - b0);
    for (int b = 0; b < n; ++b) {
      const int c = __builtin_amdgcn_readlane(starts, b);
      lo = c <= query ? c : lo;
      hi = c > query ? min(hi, c) : hi;
    }
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (64 * (w + W * i) >= H) break;
    // 16-B chunk c of row r at c ^ ((r / 2) & 7); of V, whose reads transpose pairs of chunks, at c ^ (2 (r / 2) & 7)
    auto put = [&](int at_, int r, int sw, const bf16x8& x) __attribute__((always_inline)) {
      *reinterpret_cast<bf16x8*>(ws + at_ + r * 128 + 16 * (c8 ^ (sw & 7))) = x;
    };
#pragma unroll
    for (int t = 0; t < 2; ++t) put(0, 8 * t + r8, (8 * t + r8) >> 1, q[i][t]);
#pragma unroll
    for (int t = 0; t < 4 * KB; ++t) put(kKV, 8 * t + r8, (8 * t + r8) >> 1, k[i][t]);
#pragma unroll
    for (int t = 0; t < 2; ++t) put(kW, 8 * t + r8, (8 * t + r8) >> 1, wt[i][t]);
    const int sw = (li >> 1) & 7;
    f32x4 s[HP][KT];
    float mx[HP];
#pragma unroll
    for (int hd = 0; hd < HP; ++hd) {
      mx[hd] = kMasked;
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        s[hd][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < ND; ++c) {
          const int off = li * 128 + 16 * ((4 * (ND * hd + c) + g) ^ sw);
          s[hd][t] = mfma16(*reinterpret_cast<const bf16x8*>(ws + kKV + t * 2048 + off), *reinterpret_cast<const bf16x8*>(ws + off), s[hd][t]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = 16 * t + 4 * g + r;
          s[hd][t][r] = (key >= lo) & (key < hi) ? s[hd][t][r] * at.scale_log2 : kMasked;
          mx[hd] = fmaxf(mx[hd], s[hd][t][r]);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 4 * KB; ++t) put(kKV, 8 * t + r8, 2 * ((8 * t + r8) >> 1), v[i][t]);
#pragma unroll
    for (int hd = 0; hd < HP; ++hd) {
      mx[hd] = fmaxf(mx[hd], __shfl_xor(mx[hd], 16, 64));
      mx[hd] = fmaxf(mx[hd], __shfl_xor(mx[hd], 32, 64));
      float l = 0.f;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[hd][t][r] = __builtin_amdgcn_exp2f(s[hd][t][r] - mx[hd]);
          l += s[hd][t][r];
        }
      l += __shfl_xor(l, 16, 64);
      l += __shfl_xor(l, 32, 64);
      bf16x8 pb[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const f32x4 x = s[hd][2 * kb], y = s[hd][2 * kb + 1];
        pb[kb] = __builtin_bit_cast(bf16x8, u32x4{pack2bf(x[0], x[1]), pack2bf(x[2], x[3]), pack2bf(y[0], y[1]), pack2bf(y[2], y[3])});
      }
      f32x4 o[2 * ND];
#pragma unroll
      for (int t = 0; t < 2 * ND; ++t) {
        o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const int r = 32 * kb + 4 * g + (li >> 2), ch = 2 * (t + 2 * ND * hd) + ((li & 3) >> 1);
          const char* src = ws + kKV + r * 128 + 16 * (ch ^ ((2 * (r >> 1)) & 7)) + 8 * (li & 1);
          const bf16x4 a = ds_read_tr16(src), b = ds_read_tr16(src + 16 * 128);
          o[t] = mfma16(bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}, pb[kb], o[t]);
        }
      }
      const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
      for (int c = 0; c < ND; ++c) {  // 32 columns of the head: their slots (g, e) are columns 4 g + (e & 3) + 16 (e >> 2)
        const u32x4 a = {pack2bf(o[2 * c][0] * inv, o[2 * c][1] * inv), pack2bf(o[2 * c][2] * inv, o[2 * c][3] * inv),
                         pack2bf(o[2 * c + 1][0] * inv, o[2 * c + 1][1] * inv), pack2bf(o[2 * c + 1][2] * inv, o[2 * c + 1][3] * inv)};
        const int ch = 4 * (ND * hd + c) + (g >> 1);
        const char* wrow = ws + kW + li * 128 + 8 * (g & 1);
        const u32x2 f0 = *reinterpret_cast<const u32x2*>(wrow + 16 * (ch ^ sw)), f1 = *reinterpret_cast<const u32x2*>(wrow + 16 * ((ch + 2) ^ sw));
        acc = mfma16(__builtin_bit_cast(bf16x8, u32x4{f0[0], f0[1], f1[0], f1[1]}), __builtin_bit_cast(bf16x8, a), acc);
      }
    }
  }
  *reinterpret_cast<f32x4*>(&part[w][li * LDN + 4 * g]) = acc;
  __syncthreads();
  small_finish<16, 16, LDN, W, false, 1>(p, tail, part, m0, n0);
}

// BM x BN tiles by WM x WN waves over a ring of NS K-tiles (64 wide) in LDS, filled by LDS-DMA NS - 1 tiles ahead with
// counted waits: one barrier a K-tile and no drained queue.  LDS rows of 128 B, 16-B chunk c of row r at
// c ^ ((r >> 1) & 7) (the swizzle goes on the source address, LDS-DMA writes lane-linearly); a copy is 8 rows, and copy q of a
// K-tile's A and B rows, one behind the other, is wave q mod the waves'.  The copies go out one at a time between the products:
// all in front of the fragment reads, they hold the waves up until the last is accepted, which is as long as the products take
// (24 texts of 8-64 tokens 628 -> 596 us, 10 of 200 920 -> 908; fragments read a K-tile ahead besides: the same).  Bias and
// residual are asked for at the start: at the end they were one more round trip (0.2-0.7 us).
constexpr int ring_occupancy(int rows, int waves, int ns) {  // waves a SIMD that the ring leaves room for
  const int n = 163840 / (rows * 128 * ns) * waves / 4;
  return n < 1 ? 1 : n > 8 ? 8 : n;
}

template <int BM, int BN, int WM, int WN, int NS, bool GELU, bool SLAB = false>
__global__ __launch_bounds__(64 * WM * WN, ring_occupancy(BM + BN, WM * WN, NS)) void gemm_ring_kernel(SmallParams p) {
  constexpr int W = WM * WN, MI = BM / (16 * WM), NI = BN / (16 * WN);  // 16 x 16 tiles of a wave
  constexpr int kA = BM * 128, kStage = (BM + BN) * 128, kDma = (BM + BN) / 8 / W;
  static_assert((BM + BN) % (8 * W) == 0 && BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "whole copies and tiles a wave");
  static_assert(NS == 3 || NS == 4, "waits for up to two K-tiles ahead");
  __shared__ __attribute__((aligned(16))) char smem[NS * kStage];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;
  // SLAB: the tiles of a K-slice have neighbouring ids, so an XCD reads one or two slices of A and a few columns' weights
  const int tiles_m = (p.M + BM - 1) / BM, tiles = SLAB ? tiles_m * ((p.N + BN - 1) / BN) : 1, id0 = small_id(gridDim.x);
  const int slice = SLAB ? id0 / tiles : 0, id = id0 - slice * tiles;
  const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;

  const __amdgpu_buffer_rsrc_t ra = rows_rsrc(p.A, p.M, p.lda, p.K), rb = rows_rsrc(p.B, p.N, p.ldb, p.K);
  unsigned at[kDma];  // rows past the matrix read the last one
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = 8 * (i * W + w) + (lane >> 3), c = 8 * ((lane & 7) ^ ((r >> 1) & 7));
    at[i] = (unsigned)((r < BM ? min(m0 + r, p.M - 1) * p.lda + c : min(n0 + r - BM, p.N - 1) * p.ldb + c) * 2);
  }
  auto copy = [&](int i, char* dst, unsigned so) __attribute__((always_inline)) {
    // (which operand: known here but for the copies of a step that holds rows of both)
    if (8 * (i * W + W) <= BM || (8 * i * W < BM && 8 * (i * W + w) < BM))
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (small_lds*)(dst + i * W * 1024), 16, (unsigned)at[i], so, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (small_lds*)(dst + i * W * 1024), 16, (unsigned)at[i], so, 0, 0);
  };
  auto stage = [&](int buf, int kt) {
#pragma unroll
    for (int i = 0; i < kDma; ++i) copy(i, smem + buf * kStage + w * 1024, (unsigned)kt * 128u);
  };
  const int k0 = SLAB ? p.K / 64 * slice / p.slices : 0, nk = (SLAB ? p.K / 64 * (slice + 1) / p.slices : p.K / 64) - k0;
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nk) stage(t, k0 + t);
  u32x2 bias[NI], res[NI][MI];
  if constexpr (!SLAB) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = n0 + wn * (BN / WN) + 16 * i + 4 * g;
      bias[i] = p.bias && n < p.N ? *reinterpret_cast<const u32x2*>(p.bias + n) : u32x2{0u, 0u};
#pragma unroll
      for (int j = 0; j < MI; ++j) {
        const int m = m0 + wm * (BM / WM) + 16 * j + li;
        res[i][j] = p.residual && n < p.N && m < p.M ? *reinterpret_cast<const u32x2*>(p.residual + (size_t)m * p.ldr + n) : u32x2{0u, 0u};
      }
    }
  }
  const int sw = (li >> 1) & 7;
  int rd[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) rd[ks] = li * 128 + 16 * ((4 * ks + g) ^ sw);

  f32x4 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  auto step = [&](int t, auto more) __attribute__((always_inline)) {
    constexpr bool kMore = decltype(more)::value;  // a K-tile is left to be copied
    const int ahead = kMore ? NS - 2 : min(NS - 2, nk - 1 - t);  // K-tiles after t that may stay in flight
    if (ahead >= 2) small_wait<2 * kDma>();
    else if (ahead == 1) small_wait<kDma>();
    else small_wait<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last K-tile's reads: its buffer is filled next
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    char* const dst = smem + (buf == 0 ? NS - 1 : buf - 1) * kStage + w * 1024;
    const unsigned so = (unsigned)(k0 + t + NS - 1) * 128u;
    const char* sa = smem + buf * kStage + wm * (BM / WM) * 128;
    const char* sb = smem + buf * kStage + kA + wn * (BN / WN) * 128;
    bf16x8 af[MI][2], bfr[NI][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int j = 0; j < MI; ++j) af[j][ks] = *reinterpret_cast<const bf16x8*>(sa + j * 2048 + rd[ks]);
#pragma unroll
      for (int i = 0; i < NI; ++i) bfr[i][ks] = *reinterpret_cast<const bf16x8*>(sb + i * 2048 + rd[ks]);
    }
    __builtin_amdgcn_s_setprio(1);
    constexpr int kMul = 2 * NI * MI;
#pragma unroll
    for (int x = 0; x < kMul; ++x) {
      if constexpr (kMore) {
#pragma unroll
        for (int c = 0; c < kDma; ++c)
          if (c * kMul / kDma == x) {
            __builtin_amdgcn_sched_barrier(0);
            copy(c, dst, so);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
      const int ks = x / (NI * MI), i = x / MI % NI, j = x % MI;
      acc[i][j] = mfma16(bfr[i][ks], af[j][ks], acc[i][j]);
    }
    __builtin_amdgcn_s_setprio(0);
    buf = buf == NS - 1 ? 0 : buf + 1;
  };
  int t = 0;
  for (; t + NS - 1 < nk; ++t) step(t, std::true_type());
  for (; t < nk; ++t) step(t, std::false_type());
  // acc[i][j][r] = C[m0 + wm BM / WM + 16 j + li][n0 + wn BN / WN + 16 i + 4 g + r]
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int n = n0 + wn * (BN / WN) + 16 * i + 4 * g;
    if (n >= p.N) continue;
#pragma unroll
    for (int j = 0; j < MI; ++j) {
      const int m = m0 + wm * (BM / WM) + 16 * j + li;
      if (m >= p.M) continue;
      if constexpr (SLAB) {
        *reinterpret_cast<f32x4*>(p.slabs + ((size_t)slice * p.M + m) * p.N + n) = acc[i][j];
        continue;
      }
      f32x4 s = acc[i][j];
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] += bf2f((uint16_t)(bias[i][q >> 1] >> (16 * (q & 1))));
      if constexpr (GELU) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = gelu_erf(s[q]);
      }
      if (p.residual) {
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = bf2f(f2bf(s[q])) + bf2f((uint16_t)(res[i][j][q >> 1] >> (16 * (q & 1))));
      }
      *reinterpret_cast<u32x2*>(p.C + (size_t)m * p.ldc + n) = u32x2{pack2bf(s[0], s[1]), pack2bf(s[2], s[3])};
    }
  }
}

// The ring's tiles, and what their time was fitted with: us = start + round (rounds - 1) + tile c + K-tiles max(step rounds,
// share c), c tiles on the busiest of 256 CUs, `fit` of them at a time; a GELU 50 ns more for 1000 elements of a tile.
struct RingTile {
  int bm, bn, fit;
  float start, round, tile, step, share;
};
constexpr RingTile kRing[] = {{32, 64, 3, 2.28f, 0.f, 0.46f, 0.209f, 0.132f},    {64, 64, 3, 2.52f, 0.89f, 0.42f, 0.256f, 0.201f},
                              {96, 64, 2, 3.09f, 2.81f, 0.45f, 0.309f, 0.245f},  {96, 96, 2, 3.46f, 3.76f, 0.91f, 0.381f, 0.289f},
                              {64, 128, 2, 3.15f, 1.72f, 0.92f, 0.316f, 0.264f}, {64, 192, 1, 3.50f, 2.25f, 1.67f, 0.392f, 0.150f},
                              {128, 192, 1, 4.69f, 4.32f, 2.92f, 0.578f, 0.150f}, {128, 256, 1, 5.34f, 4.64f, 3.36f, 0.660f, 0.157f}};
constexpr int kRings = sizeof(kRing) / sizeof(kRing[0]);

static float ring_us(const RingTile& t, int M, int N, int K, int gelu, int slices = 1) {
  const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * slices;
  const long c = (tiles + 255) / 256, rounds = (c + t.fit - 1) / t.fit;
  const float steps = K / 64 / slices, step = t.step * rounds, share = t.share * c;
  return t.start + t.round * (rounds - 1) + (t.tile + (gelu ? 5e-5f * t.bm * t.bn : 0.f)) * c + steps * (step > share ? step : share);
}

// The tile of the ring with the least estimate.  All of them sum K in one order: the choice changes no bits.  Fitted to 4,300
// launches (M 200-6400, the projections of encoders of 384, 768 and 1024): half of the estimates within 5 %, nine of ten
// within 15 %.  Over those shapes 9 % faster than tiles of 64 x 64 (128 x 128 with a long K) and gemm256 as they were chosen
// before, up to 69 % ((4000, 1024, 1024) 27.6 -> 16.4 us), 0.95 at worst ((560, 1024, 4096) in three slices 16.2 -> 17.0).  Calls of the
// encoder: bge-base 24 texts of 8-64 tokens 748 -> 716, 1300 tokens 854 -> 766, 2200 1186 -> 1045, 7000 2509 -> 2027; MiniLM
// 4000 473 -> 404; bge-large 1000 1907 -> 1719, 5000 5604 -> 4609.
// (All of that with the copies of a K-tile in front of its products and the former GELU.  As both are now the estimates are 7 % too long
// in the middle, 15 % too short to 25 % too long for eight of ten of 60 sizes, and the tile taken by them is 2 % slower than the
// best in the mean; the most (3100, 768, 768) 12.5 us on 96 x 64, 9.6 on 64 x 192, and (6000, 768, 3072) 48 on 96 x 96, 37 on 128 x
// 192.)
int ring_tile(int M, int N, int K, int gelu, int slices) {
  int best = 0;
  for (int i = 1; i < kRings; ++i)
    if (ring_us(kRing[i], M, N, K, gelu, slices) < ring_us(kRing[best], M, N, K, gelu, slices)) best = i;
  return best;
}

// Whether the ring beats gemm256 (row-major weights), or the 128 x 128 kernel where that does not take the shape, at a size
// that small_tile leaves to them: by a tenth of the estimate of gemm256, waves of 256 tiles of 256 x 256, each with its
// epilogue, and by 1.44 times that.  Where the 128 x 128 kernel has no more than the two tiles a CU that run side by side, its
// own estimate decides, too (the product and the result's way to memory, half of them within 3 %; the ring's with a residual's
// reads in it).  (By that estimate alone, whatever the tiles, also qkv of MiniLM from 9,100 tokens on: a call of 21,000 tokens
// 1,291 -> 1,227 us, but of 11,900 830 -> 839.)  Over 1,113 sizes (24 pairs of N and K, M 400-30,000) 8 % faster than without
// the ring, over 716 others (22 pairs, M 600-30,000) 10 %; 8 of them are more than 2 % slower in their sweep, and in both only
// (8000, 1024, 256) 11.9 -> 12.4 and (30000, 256, 256) 11.8 -> 12.2  us, before -> ring: (6400, 768, 768) 24.3 -> 17.2, (5300,
// 1152, 384) 15.8 -> 11.2, (17500, 1000, 768) 61 -> 45.  Left where they were, us there / on the ring: (3200, 3072, 768) 26.1 /
// 28.4, (4600, 2304, 768) 21.9 / 32, (17500, 384, 1536) 34.3 / 37.3, (11000, 640, 1280) 31.0 / 32.4.
bool ring_wins(int M, int N, int K, int gelu, int residual) {
  if (M <= 0 || N <= 0 || K < 64) return false;
  const bool large = gemm256_wins(M, N) && gemm256_ok(M, N, K, K, K);
  const float ring = ring_us(kRing[ring_tile(M, N, K, gelu, 1)], M, N, K, gelu);
  const long waves = ((long)((M + 255) / 256) * ((N + 255) / 256) + 255) / 256;
  if (ring >= (large ? 0.9f : 1.44f) * (2.1f + waves * (0.0146f * K + 7.f + (gelu ? 5.7f : 0.f) + (residual ? 3.9f : 0.f)))) return false;
  const long c = ((long)((M + 127) / 128) * ((N + 127) / 128) + 255) / 256;  // tiles of 128 x 128 on the busiest CU
  if (large || c > 2) return true;
  const float mn = 1e-6f * M * N, other = 5.3f + 0.0151f * K + 0.81f * mn + c * (gelu ? 1.26f : residual ? 2.1f : 0.f);
  return 1.18f * ring + 1.7f + (residual ? -0.12f : -0.53f) * mn < 0.97f * other;
}

// Rows of a projection that go to gemm256, all or whole waves of 256 tiles: the few rows behind those, for which a last wave
// would run as long as a full one, go to the ring, where its estimate and 4 us are under 0.85 of that wave's.  The sums of K have one
// order in both: no bits change.  Past twelve waves nothing is gained: the power limit holds the clock, and the workgroups have
// drifted apart until the last wave.  Over 422 sizes (the projections of encoders of 384, 768 and 1024, M 5,000-112,000) it takes
// 247, 1.11 times as fast in the mean, two of them 0.98.  us, gemm256 -> with the ring: (24291, 768, 3072) 139 -> 111, (70055, 768,
// 3072) 313 -> 296, (10885, 3072, 768) GELU 72 -> 58, (29177, 2304, 768) 109 -> 100; left whole (98339, 3072, 768) GELU 513 / 518,
// (12292, 2304, 768) 47 / 60.
int gemm256_rows(int M, int N, int K, int gelu, int residual) {
  if (M <= 0 || N < 256 || N % 256 || K < 64 || (gelu && residual)) return M;
  const long tn = N / 256, waves = ((M + 255) / 256) * tn / 256;
  const int rows = (int)(waves * 256 / tn * 256);
  if (waves < 1 || waves > 12 || rows <= 0 || rows >= M) return M;
  if (!gelu && !residual && gemm256_far_a(M, K) && !gemm256_far_a(rows, K)) return M;  // (its tile order is worth more)
  const float ring = ring_us(kRing[ring_tile(M - rows, N, K, gelu, 1)], M - rows, N, K, gelu);
  return ring + 4.f < 0.85f * (0.0146f * K + 7.f + (gelu ? 5.7f : 0.f) + (residual ? 3.9f : 0.f)) ? rows : M;
}

template <int I, int WM, int WN, int NS>
static void ring_launch(const SmallParams& p, int gelu, hipStream_t s) {
  constexpr RingTile t = kRing[I];
  static_assert(t.fit == 163840 / ((t.bm + t.bn) * 128 * NS), "as many tiles at a time as a CU's LDS has rings for");
  const int slices = p.slabs ? p.slices : 1;
  const dim3 grid(((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn) * slices), block(64 * WM * WN);
  if (p.slabs) hipLaunchKernelGGL((gemm_ring_kernel<t.bm, t.bn, WM, WN, NS, false, true>), grid, block, 0, s, p);
  else if (gelu) hipLaunchKernelGGL((gemm_ring_kernel<t.bm, t.bn, WM, WN, NS, true>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((gemm_ring_kernel<t.bm, t.bn, WM, WN, NS, false>), grid, block, 0, s, p);
}

// tile: that one (tests), -1: by the estimate
static void gemm_ring(const SmallParams& p, int gelu, hipStream_t s, int tile = -1) {
  switch (tile >= 0 ? tile : ring_tile(p.M, p.N, p.K, gelu, p.slabs ? p.slices : 1)) {
    case 0: return ring_launch<0, 2, 2, 4>(p, gelu, s);
    case 1: return ring_launch<1, 2, 4, 3>(p, gelu, s);
    case 2: return ring_launch<2, 2, 2, 3>(p, gelu, s);
    case 3: return ring_launch<3, 2, 2, 3>(p, gelu, s);
    case 4: return ring_launch<4, 2, 4, 3>(p, gelu, s);
    case 5: return ring_launch<5, 2, 4, 4>(p, gelu, s);
    case 6: return ring_launch<6, 4, 2, 3>(p, gelu, s);
    default: return ring_launch<7, 4, 4, 3>(p, gelu, s);
  }
}

// Shapes and alignments the kernel takes (8-B bias / residual / output vectors, 16-B operand vectors, 31-bit offsets).
int gemm_small_ok(long M, long N, long K, long lda, long ldb, long ldc, long ldr) {
  return M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 4 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 4 == 0 && ldr % 4 == 0 &&
         lda >= 0 && ldb >= 0 && ldc >= 0 && ldr >= 0 && (M * lda + K) * 2 < (1L << 31) && (N * ldb + K) * 2 < (1L << 31) &&
         ldc < (1L << 31) && ldr < (1L << 31);
}

// Workgroups behind `grid` of 512 that read the next launch's weights: as few as do it in 16 loads a thread, on CUs that have no
// workgroup with a tile.  us a forward of 19 / 6 tokens of bge-base and 19 of bge-large, weights of three copies in turn: without
// 284 / 259 / 626, 8 loads a thread 267 / 237 / 610, 16 265 / 237 / 600, 24 279 / 276 / 596; up to 320 workgroups 278 / 251 /
// 664; as 2 to 8 loads a thread of the workgroups with a tile, waited for at their end, 295 / 274 / 650.  40 tokens 360 -> 347 with the
// tiles of 16 x 16 alone, 329 with the other split-K tiles; 120 417 -> 402, 240 486 -> 479.
static int next_blocks(const Upcoming& next, int grid) {
  if (!next.w || next.bytes < 128 || next.bytes % 128 || (uintptr_t)next.w % 16) return 0;
  const int room = (256 - grid) & ~7, want = (int)(((long)next.bytes / 8 + 16 * 8192 - 1) / (16 * 8192) * 8);
  return room < 8 ? 0 : min(want, room);
}

// tile: as small_tile says; kRingTile + 16 + i: tile i of the ring, whatever its estimate (tests).
int gemm_small(const void* A, long lda, const void* B, long ldb, void* C, long ldc, const void* bias, const void* residual,
               long ldr, int M, int N, int K, int gelu, int tile, hipStream_t s, Upcoming next) {
  if (M <= 0 || N <= 0) return 0;
  if (!gemm_small_ok(M, N, K, lda, ldb, ldc, residual ? ldr : 0)) return hipErrorInvalidValue;
  if (((uintptr_t)A | (uintptr_t)B) % 16 || ((uintptr_t)C | (uintptr_t)bias | (uintptr_t)residual) % 8) return hipErrorInvalidValue;
  SmallParams p = {(const bf16*)A, (const bf16*)B, (bf16*)C, (const bf16*)bias, (const bf16*)residual, M, N, K,
                         (int)lda, (int)ldb, (int)ldc, (int)ldr};
  p.next = next;
#define SMALL_AS(MT_, NT_, W_, D_, A_)                                                                                  \
  do {                                                                                                                \
    if (gelu) hipLaunchKernelGGL((gemm_small_kernel<MT_, NT_, W_, D_, true, A_>), grid, dim3(64 * W_), 0, s, p);       \
    else hipLaunchKernelGGL((gemm_small_kernel<MT_, NT_, W_, D_, false, A_>), grid, dim3(64 * W_), 0, s, p);           \
  } while (0)
#define SMALL(T, MT_, NT_, W_, D_)                                                                                    \
  case T: {                                                                                                           \
    p.work = ((M + 16 * MT_ - 1) / (16 * MT_)) * ((N + 16 * NT_ - 1) / (16 * NT_));                                   \
    const int more = next_blocks(next, p.work);                                                                       \
    const dim3 grid(p.work + more);                                                                                   \
    if (more) SMALL_AS(MT_, NT_, W_, D_, true);                                                                       \
    else SMALL_AS(MT_, NT_, W_, D_, false);                                                                           \
    break;                                                                                                            \
  }
  switch (tile) {
    SMALL(0, 1, 1, 8, 2)
    SMALL(1, 2, 1, 8, 2)
    case kRingTile: gemm_ring(p, gelu, s); break;
    case kRingTile + 16 ... kRingTile + 16 + kRings - 1: gemm_ring(p, gelu, s, tile - kRingTile - 16); break;
    SMALL(6, 2, 2, 8, 1)
    SMALL(7, 2, 4, 8, 1)
    SMALL(8, 4, 4, 8, 1)
    default: return hipErrorInvalidValue;
  }
#undef SMALL
#undef SMALL_AS
  return hipGetLastError();
}

// K-slices that a long-K projection in front of a LayerNorm (which sums them: layernorm_slabs) is cut into, 0: none.  The
// widths are those of layernorm_slab_kernel's instances.  Its tiles alone leave CUs idle or one workgroup each, whose share
// of the operands from past L2 is what takes the time; in slices they fill the chip.  The slabs cost 8 bytes an element and
// slice there and back, which a short K or few rows do not pay for.
//
// The bands were measured when a slice ran on tiles of 64 x 64 (up to 256 of them) or 128 x 128 (from 64 of them on) alone
// and are counted in those; the launch takes the tile that ring_tile estimates for the slices.  With these eight tiles the
// bands are a little wrong on both sides: (560, 1024, 4096) in three slices 16.2 -> 17.0 us against the 64 x 64 tile, and by
// ring_us two slices would be the quicker for bge-base at 961-1,300 tokens and bge-large at 641-1,024, which run whole.  us
// of product and LayerNorm, one launch -> slices: (rows, H, K) (832, 768, 3072) 16.9 -> 14.8, (600, 1024, 4096) 19.0 ->
// 15.9, (2200, 384, 1536) 14.2 -> 13.2; with 128 x 128 (1500, 768, 3072) 22.7 -> 21.2, (2200, 768, 3072) 29.4 -> 26.2,
// (1100, 1024, 4096) 27.0 -> 25.1, (3200, 384, 1536) 19.8 -> 16.9; not taken (600, 768, 3072) 13.5 -> 13.9, (1500, 384,
// 1536) 12.0 -> 12.3 in three slices of 512, (4600, 768, 3072) 41.8 -> 48.3, (832, 768, 768) 9.5 -> 10.3.  Whole calls of
// the encoder, weights of three copies in turn: bge-base 800 tokens 703 -> 676, 900 735 -> 708, 1400 964 -> 922, 1650 1091
// -> 1021, 2500 1293 -> 1207; MiniLM 1850 275 -> 269, 2650 330 -> 321, 3200 391 -> 368, 5000 493 -> 469; not taken bge-base
// in two slices of 1536, 1000 765 -> 776, 1150 818 -> 832, 1300 847 -> 861 (with the weights on the die 773 -> 751 at 1180),
// 1300 in three of 128 x 128 847 -> 869; bge-large 765 in two of 2048 1757 -> 1788.
int slab_slices(int M, int N, int K) {
  if (M <= 0 || K < 1536 || K % 64 || (N != 384 && N != 768 && N != 1024)) return 0;
  const long t64 = ((M + 63) / 64) * (long)(N / 64), t128 = ((M + 127) / 128) * (long)(N / 128);
  if (t64 >= 139 && t64 <= 170 && K >= 3 * 768) return 3;
  if (t64 >= 171 && t64 <= (K <= 2048 ? 256 : 180) && K < 4096) return 2;
  if (t64 <= 256) return 0;
  if (t128 >= 64 && t128 <= 85) return 3;
  if (t128 >= 96 && t128 <= 128) return 2;
  return 0;
}

// slabs [slices][M][N] fp32 = the K-slices' sums of A w^T, as slab_slices says; tile: as gemm_ring's
int gemm_slab(const void* A, const void* B, void* slabs, int M, int N, int K, hipStream_t s, int tile) {
  const int slices = slab_slices(M, N, K);
  if (tile >= kRings || !slices || !gemm_small_ok(M, N, K, K, K, N, 0)) return hipErrorInvalidValue;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)slabs) % 16) return hipErrorInvalidValue;
  const SmallParams p = {(const bf16*)A, (const bf16*)B, nullptr, nullptr, nullptr, M, N, K, K, K, N, 0, 0, (float*)slabs, slices};
  gemm_ring(p, 0, s, tile);
  return hipGetLastError();
}

// C = LayerNorm(x) w^T + b (GELU) for the projections that take tile 0 or 1 and the widths of layernorm_rows_kernel;
// normed [M, K] receives the normalised rows (not x itself: other workgroups still read it).
int gemm_ln_ok(int M, int N, int K, int tile) {
  return (K == 768 || K == 1024) && (tile == 0 || tile == 1) && gemm_small_ok(M, N, K, K, K, N, N);
}

int gemm_ln(const void* x, const void* gain, const void* offset, float eps, void* normed, const void* w, const void* b, void* C,
            int M, int N, int K, int gelu, int tile, hipStream_t s, Upcoming next) {
  if (!gemm_ln_ok(M, N, K, tile) || normed == x) return hipErrorInvalidValue;
  if (((uintptr_t)w) % 16 || ((uintptr_t)x | (uintptr_t)gain | (uintptr_t)offset | (uintptr_t)normed | (uintptr_t)C | (uintptr_t)b) % 8)
    return hipErrorInvalidValue;
  SmallParams p = {(const bf16*)x, (const bf16*)w, (bf16*)C, (const bf16*)b, nullptr, M, N, K, K, K, N, N};
  const SmallNorm nm = {(const bf16*)gain, (const bf16*)offset, (bf16*)normed, eps};
  const int mt = tile + 1, work = ((M + 16 * mt - 1) / (16 * mt)) * ((N + 15) / 16), grid = work + next_blocks(next, work);
  p.work = work;
  p.next = next;
#define LN_GEMM(MT_, S_)                                                                                               \
  if (mt == MT_ && K == 256 * S_) {                                                                                    \
    if (gelu) hipLaunchKernelGGL((gemm_ln_kernel<MT_, S_, true>), dim3(grid), dim3(512), 0, s, p, nm);                  \
    else hipLaunchKernelGGL((gemm_ln_kernel<MT_, S_, false>), dim3(grid), dim3(512), 0, s, p, nm);                      \
  }
  LN_GEMM(1, 3)
  LN_GEMM(2, 3)
  LN_GEMM(1, 4)
  LN_GEMM(2, 4)
#undef LN_GEMM
  return hipGetLastError();
}

// y = attention(qkv) w^T + b + residual of a few packed tokens (qkv [T, 3 H], cu [batch + 1]): up to 32, and up to 64 where
// a wave's two pieces are not yet more than the two launches (us a layer, two launches -> one, one text or four of T / 4: H 384
// at T 6-32 5.6 -> 4.0, 33-64 5.7-5.9 -> 5.0-5.1; H 768 at 6-32 6.5-6.7 -> 4.7-5.0, 33-64 6.8-7.0 -> 6.4-6.7, eight of 8
// 7.0 -> 7.05; H 1024 at 6-32 7.2-7.5 -> 5.9-6.3, 33-64 7.5-7.7 -> 8.1-8.9).
int gemm_attn_ok(int T, int H, int D, int batch) {
  return T > 0 && T <= (H <= 768 ? 64 : 32) && batch > 0 && (D == 32 || D == 64) && H % 64 == 0 && H > 0 && H <= 1024;
}

int gemm_attn(const void* qkv, const int* cu, int batch, int D, float scale, const void* w, const void* b, const void* residual,
              void* y, int T, int H, hipStream_t s, Upcoming next) {
  if (!gemm_attn_ok(T, H, D, batch)) return hipErrorInvalidValue;
  if (((uintptr_t)qkv | (uintptr_t)w) % 16 || ((uintptr_t)b | (uintptr_t)residual | (uintptr_t)y) % 8 || (uintptr_t)cu % 4)
    return hipErrorInvalidValue;
  SmallParams p = {nullptr, (const bf16*)w, (bf16*)y, (const bf16*)b, (const bf16*)residual, T, H, H, H, H, H, H};
  p.work = ((T + 15) / 16) * (H / 16);
  p.next = next;
  const SmallAttention at = {(const bf16*)qkv, cu, batch, scale * 1.44269504088896340736f};
  const dim3 grid(p.work + next_blocks(next, p.work));
  if (D == 64 && T <= 32) hipLaunchKernelGGL((gemm_attn_kernel<64, 1>), grid, dim3(512), 0, s, p, at);
  else if (D == 64) hipLaunchKernelGGL((gemm_attn_kernel<64, 2>), grid, dim3(512), 0, s, p, at);
  else if (T <= 32) hipLaunchKernelGGL((gemm_attn_kernel<32, 1>), grid, dim3(512), 0, s, p, at);
  else hipLaunchKernelGGL((gemm_attn_kernel<32, 2>), grid, dim3(512), 0, s, p, at);
  return hipGetLastError();
}

}  // namespace dab
