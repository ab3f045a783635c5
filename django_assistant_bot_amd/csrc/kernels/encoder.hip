// The sentence encoder's forward as one call: every launch of its layers enqueued from native code.
//
// For one question the GPU works 0.26 ms on 52 launches (0.45 ms on 87 with the LayerNorms and the attention apart), and
// issuing those from Python took 1.06 ms (11.6 us a launch: wrapper, checks, a tensor for each result).  Here a
// launch costs the runtime's own 1-2 us; the five activation buffers are the caller's, shared by all layers.  (The
// reference runs one text a call through an eager model: ai/embedders/transformers.py:15-29.)
#include "common.h"
#include "launchers.h"

namespace dab {

// Which kernel of gemm_small a projection with row-major weights takes: 0, 1, 6, 7, 8 a tile of the split-K kernel, kRingTile
// (3) the barrier-stepped ring, whose tile ring_tile (gemm_small.hip) picks, -1 the 128 x 128 / 256 x 256 kernels unless ring_wins.
//
// The smallest tile that still gives each CU about one workgroup: K split over a workgroup's waves up to 256 tiles of
// 16 x 16, 32 x 16, 32 x 32, 32 x 64, and 64 x 64 where K is long (K of 384 and more: every other kernel sums K in one
// order, so that results there do not depend on M); then the ring, up to 1200 tiles of 64 x 64 (1000 where M is over 3 N: each
// XCD streams the rows again for every column block), with a long K up to 256 of 128 x 128.  Both sides of each line, us (us of the
// tile before -> of the tile after it): 192 tiles of 16 x 16 at (64, 768, 768) 3.1 /
// 3.4, 288 at (19, 2304, 768) 3.6 / 3.4; 192 of 32 x 16 at (128, 768, 768) 3.4 / 3.8, 288 at (64, 2304, 768) 5.3 / 4.1;
// 192 of 32 x 32 at (256, 768, 768) 3.9 / 4.6, 288 at (128, 2304, 768) 5.3 / 4.8; 192 of 32 x 64 at (512, 768, 768) 5.1
// / 5.5 (ring of 64 x 64, as below), with K 3072 11.4 / 14.7, 288 at (256, 2304, 768) 7.9 / 6.4; 224 of 64 x 64 at (870, 1024,
// 4096) 17.6 / 20.6, 288 at (1500, 768, 3072) 26.5 / 19.6, but with the short K 168 at (870, 768, 768) 7.0 / 6.7.  The ring's end
// was measured when it had no tiles but 64 x 64 and, with a long K, 128 x 128: ring / gemm256 with 1152 tiles at (2048, 2304, 768)
// 20.2 / 25.4, 1692 at (3000, 2304, 768) 29.3 / 26.7, 1008 at (5333, 768, 768) 18.0 / 18.4, 1104 at (5866, 768, 768) 20.3 / 18.5, at (4400,
// 1024, 1024) 23.9 / 22.0; 192 of 128 x 128 at (4096, 768, 3072) 37.7 / 64.4, 282 at (6000, 768, 3072) 71.3 / 64.0.  The tiles that it
// has now only make it faster: up to there it is taken without a look at the estimates, behind them where ring_wins says so.
int small_tile(int M, int N, int K) {
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (K >= 384) {
    if (tiles(16, 16) <= 256) return 0;
    if (tiles(32, 16) <= 256) return 1;
    if (tiles(32, 32) <= 256) return 6;
    if (tiles(32, 64) <= 256) return 7;
    if (K > 1024 && tiles(64, 64) <= 256) return 8;
  }
  const bool ring = K <= 1024 ? tiles(64, 64) <= (M > 3L * N ? 1000 : 1200) : tiles(128, 128) <= 256;
  return ring ? kRingTile : -1;
}

// y[M, N] = x[M, K] w[N, K]^T + b (GELU) (+ residual), everything contiguous: ops.gemm_bt's choice of kernel.
static int projection(const bf16* x, const void* w, const void* b, const bf16* residual, bf16* y, int M, int N, int K, int gelu,
                      hipStream_t s, Upcoming next = {}) {
  int tile = small_tile(M, N, K);
  if (tile < 0 && ring_wins(M, N, K, gelu, residual != nullptr)) tile = kRingTile;
  const bool small = gemm_small_ok(M, N, K, K, K, N, N) &&
                     !(((uintptr_t)x | (uintptr_t)w) % 16 || ((uintptr_t)y | (uintptr_t)b | (uintptr_t)residual) % 8);
  if (tile >= 0 && small) return gemm_small(x, K, w, K, y, N, b, residual, N, M, N, K, gelu, tile, s, next);
  if (gemm256_wins(M, N) && gemm256_ok(M, N, K, K, K)) {
    const int rows = small ? gemm256_rows(M, N, K, gelu, residual != nullptr) : M;
    const int rc = gemm256(x, K, w, K, y, N, b, residual, N, rows, N, K, gelu, s, 0, 1);
    if (rc || rows == M) return rc;
    const long o = (long)rows * N;
    return gemm_small(x + (long)rows * K, K, w, K, y + o, N, b, residual ? residual + o : nullptr, N, M - rows, N, K, gelu, kRingTile, s);
  }
  return gemm_bt(x, K, w, K, y, N, b, residual, N, M, N, K, gelu, 0, nullptr, nullptr, nullptr, 0, s, 0, 1);
}

// Packed token ids [T] -> hidden states x [T, H].  `layers`: per layer qkv, o, ln1, i, d, ln2 as (weight, bias) or (gain,
// offset) pairs.  Up to 32 or 64 tokens the attention runs inside the output projection (gemm_attn_ok).  Buffers: x, y, att
// [T, H], qkv [T, 3 H], ffn [T, F], slabs [slices, T, H] fp32 where the down projection is cut into K-slices that the
// LayerNorm behind it sums (slab_slices), or null.
int encoder_forward(const int* ids, const int* pos, const int* cu, int T, int batch, int max_len, int H, int heads, int F,
                    int n_layers, float eps, const void* word, const void* pos_table, const void* type, const void* gain,
                    const void* offset, const uintptr_t* layers, void* x_, void* y_, void* att_, void* qkv_, void* ffn_,
                    void* slabs, hipStream_t s) {
  if (T <= 0 || batch <= 0 || max_len <= 0) return 0;
  if (H <= 0 || heads <= 0 || H % heads || H % 64 || F % 64 || F <= 0) return hipErrorInvalidValue;
  const int D = H / heads;
  if (D != 32 && D != 64 && D != 128) return hipErrorInvalidValue;
  bf16 *x = (bf16*)x_, *y = (bf16*)y_, *att = (bf16*)att_, *qkv = (bf16*)qkv_, *ffn = (bf16*)ffn_;
  int rc = bert_embed(x, ids, pos, nullptr, word, pos_table, type, gain, offset, T, H, eps, s);
  const float scale = 1.f / sqrtf((float)D);
  // The weights that launches read ahead: each the next launch's, a LayerNorm also those of the projection behind the next,
  // where that one's tiles leave no room for readers.  us a forward, weights of three copies in turn, without the latter -> with:
  // bge-base 240 tokens 481 -> 468, 816 632 -> 609, 1500 820 -> 798, 3000 1,209 -> 1,210; bge-large 180 1,040 -> 981, 600 1,428 ->
  // 1,369, 1200 1,937 -> 1,837, 1800 2,239 -> 2,222; where the next launch has readers too 120 405 -> 414.
  auto reads_next = [](int tile) { return tile >= 0 && tile != kRingTile; };
  // x = LayerNorm(y), then out = x w^T + b: one launch where the projection takes a split-K tile (one or two row tiles, so
  // that a row is normalised by as many workgroups as read it anyway), two where its rows outgrow that
  auto norm_projection = [&](const uintptr_t* ln, const void* w, const void* b, bf16* out, int N, int gelu, Upcoming next) {
    const int tile = small_tile(T, N, H);
    if (gemm_ln_ok(T, N, H, tile) && !(((uintptr_t)w) % 16 || (ln[0] | ln[1] | (uintptr_t)b) % 8))
      return gemm_ln(y, (const void*)ln[0], (const void*)ln[1], eps, x, w, b, out, T, N, H, gelu, tile, s, next);
    const int e = layernorm(x, y, nullptr, (const void*)ln[0], (const void*)ln[1], T, H, eps, s, {w, (unsigned)((long)N * H * 2)},
                            reads_next(tile) ? Upcoming{} : next);
    return e ? e : projection(x, w, b, nullptr, out, T, N, H, gelu, s, next);
  };
  const int slices = slabs ? slab_slices(T, H, F) : 0;
  const uintptr_t* ln = nullptr;  // the layer's own norm of y, applied in front of the next projection
  for (int l = 0; l < n_layers && !rc; ++l) {
    const uintptr_t* w = layers + 12 * l;
    auto W = [&](int i) { return (const void*)w[i]; };
    auto ahead = [&](const void* m, long n, long k) { return Upcoming{m, (unsigned)(n * k * 2)}; };
    const Upcoming o = ahead(W(2), H, H), up = ahead(W(6), F, H), down = ahead(W(8), H, F);
    const Upcoming qkv_next = l + 1 < n_layers ? ahead((const void*)w[12], 3 * H, H) : Upcoming{};
    const Upcoming o_next = l + 1 < n_layers && !reads_next(small_tile(T, 3 * H, H)) ? ahead((const void*)w[14], H, H) : Upcoming{};
    rc = ln ? norm_projection(ln, W(0), W(1), qkv, 3 * H, 0, o) : projection(x, W(0), W(1), nullptr, qkv, T, 3 * H, H, 0, s, o);
    // (33-64 tokens of 768, weights of several copies in turn, us a call apart -> inside: one text of 40 370 -> 360, of 56 379 -> 370,
    // four of 15 379 -> 377, eight of 8 381 -> 383, twenty of 3 378 -> 384: up to four texts)
    const bool attn_o = gemm_attn_ok(T, H, D, batch) && (T <= 32 || H <= 384 || batch <= 4) && !(w[2] % 16 || w[3] % 8);
    if (!rc && attn_o) rc = gemm_attn(qkv, cu, batch, D, scale, W(2), W(3), x, y, T, H, s, up);
    if (!rc && !attn_o)
      rc = flash_attention(qkv, 3 * H, D, qkv + H, qkv + 2 * H, 3 * H, D, nullptr, nullptr, nullptr, 0, 0, att, H, D, cu, cu,
                           nullptr, batch, max_len, heads, heads, D, 0, 0, scale, s);
    if (!rc && !attn_o) rc = projection(att, W(2), W(3), x, y, T, H, H, 0, s, up);
    if (!rc) rc = norm_projection(w + 4, W(6), W(7), ffn, F, 1, down);
    if (slices && !(w[8] % 16 || (w[9] | w[10] | w[11]) % 4)) {
      if (!rc) rc = gemm_slab(ffn, W(8), slabs, T, H, F, s);
      if (!rc) rc = layernorm_slabs(x, slabs, slices, W(9), x, W(10), W(11), T, H, eps, s, qkv_next, o_next);
      ln = nullptr;
      continue;
    }
    if (!rc) rc = projection(ffn, W(8), W(9), x, y, T, H, F, 0, s, qkv_next);
    ln = w + 10;
  }
  if (!rc && ln) rc = layernorm(x, y, nullptr, (const void*)ln[0], (const void*)ln[1], T, H, eps, s);
  return rc;
}

}  // namespace dab
