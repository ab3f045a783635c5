// Bidirectional attention over packed sequences, heads of 64 (the bge / BERT encoders): the form for long texts and for
// many of them.  (Reference: HF BertSelfAttention, ai/embedders/transformers.py:18-22.)
//
// What bounds it: the softmax.  A score costs an exponential (16 cycles a wave) and about three more vector
// instructions against 8 cycles of MFMA, so everything else has to run beside them.  The 16 x 16 form of attention.hip
// staged K and V through registers with two barriers a tile and spread a query's keys over four lane groups: 623 us
// a layer for 400 chunks of 32-512 tokens (12 heads), 188 TFLOP/s.  Here:
//   * 32 x 32 x 16 MFMAs, S^T = K Q^T: a lane owns one query and half of its keys, so a row maximum is 31 maxima in
//     registers and one exchange, and P leaves in the order in which O^T = V^T P^T takes it (V's rows are read in the
//     same order, transposed by the LDS read);
//   * 128 queries a workgroup (4 waves), two LDS buffers of 64 keys of K and V, filled by LDS-DMA a tile ahead: one
//     barrier a tile, nothing passes through registers.  32 KB and 108 registers keep 4 workgroups on a CU, which hides
//     a tile's chain better than a third buffer (3 workgroups: 310 us against 298);
//   * waves whose queries lie past the sequence only stage.
// 400 chunks 519 -> 285 us (the same launch of the 16 x 16 form measured beside it), 200 x 512 tokens 324 -> 236 us (683
// TFLOP/s); about 960 cycles of vector issue and 512 of MFMA a wave and tile, so the sum of both is what remains.
#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

struct PackedParams {
  const bf16* q;
  const bf16* k;
  const bf16* v;
  bf16* out;
  long q_tok, q_head, kv_tok, kv_head, o_tok, o_head;
  const int* cu;
  int group;  // query heads per key head
  int heads, units, nqb;  // (sequence, head) pairs, query blocks of the longest sequence
  float scale_log2;
  // PAGED: k and v are caches [blocks][key heads][block_size][64]; the queries are the last of ctx[b] tokens
  const int* tables;
  const int* ctx;
  int max_blocks, block_size;
};

typedef __attribute__((address_space(3))) void pk_lds;

constexpr int kPkTile = 8192;  // 64 rows of 64 bf16
constexpr int kPkStages = 2;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pk_rsrc(const bf16* base, long tok, int rows) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(base), (short)0, (int)(((rows - 1) * tok + 64) * 2), 0x00020000);
}

__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}

// The transposed V reads of two 16-key blocks (2 KB apart; lower and upper keys 1 KB apart) for d 0-31 (a0) and 32-63
// (a1), waited in the same statement.  As an intrinsic the read makes hipcc drain every LDS-DMA in flight first.
__device__ __forceinline__ void pk_read_tr8(unsigned a0, unsigned a1, u32x2 (&v)[8]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:1024\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:1024\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:2048\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:3072\n\t"
      "ds_read_b64_tr_b16 %6, %9 offset:2048\n\t"
      "ds_read_b64_tr_b16 %7, %9 offset:3072\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(a0), "v"(a1)
      : "memory");
}

}  // namespace

// 16-B chunk c of row r of a tile lies at chunk c ^ (2 (r / 2) & 7): conflict-free for the row reads of K and the
// transposed reads of V (pairs of chunks stay together)
//
// PAGED: the same for causal prompts over a paged cache (Llama-3.2-1B's prefill), whose 64-key tiles each lie in one cache
// block.  The blocks of the most keys start first, over all heads of an XCD; the heads of a key head are on one where the
// key heads divide.  us, the 16 x 16 form -> here, 32 heads on 8: 1 x 400 tokens 11.9 -> 10.8, 1093 28.1 -> 23.8, 2000 61.3 ->
// 37.7, 4 x 700 29.5 -> 21.3, 16 x 250 24.5 -> 18.7, 3 x 64 behind 3000 58.3 -> 50.5; 60 tokens 5.0 -> 5.2.
template <bool PAGED>
__global__ __launch_bounds__(256, 4) void flash_packed64_kernel(PackedParams p) {
  __shared__ __attribute__((aligned(16))) char smem[kPkStages * 2 * kPkTile];
  // a (sequence, head)'s query blocks on one XCD, whose L2 serves their re-reads of its K / V; consecutive (sequence,
  // head) pairs on different ones (batches come sorted by length: contiguous shares gave one XCD all the long texts)
  const int per = PAGED ? (p.units + 7) / 8 : 1, at = (int)(blockIdx.x / 8);
  const int unit = (PAGED ? at % per : at / p.nqb) * 8 + (int)(blockIdx.x % 8);
  if (unit >= p.units) return;
  int hq = unit % p.heads;
  const int b = unit / p.heads;
  if (PAGED && p.heads / p.group % 8 == 0) hq = (hq / (8 * p.group) * 8 + hq % 8) * p.group + hq / 8 % p.group;
  const int start = p.cu[b], nq = p.cu[b + 1] - start;
  const int len = PAGED ? p.ctx[b] : nq, past = len - nq;
  const int q0 = (PAGED ? (nq + 127) / 128 - 1 - at / per : at % p.nqb) * 128;
  if (PAGED ? q0 < 0 : q0 >= nq) return;  // whole workgroup
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles = ((PAGED ? min(len, past + q0 + 128) : len) + 63) / 64;
  const bool work = q0 + 32 * w < nq;  // wave-uniform

  // ---- staging: instruction i of a tile copies rows 8 i .. 8 i + 7; wave w does i = w and w + 4 of K and of V.  Rows
  // past the sequence read its last one (finite; masked below)
  const long head = PAGED ? 0 : (long)(hq / p.group) * p.kv_head + (long)start * p.kv_tok;
  __amdgpu_buffer_rsrc_t rk, rv;
  if constexpr (!PAGED) rk = pk_rsrc(p.k + head, p.kv_tok, len), rv = pk_rsrc(p.v + head, p.kv_tok, len);
  // PAGED: the block ids of the first 128 tiles, two a lane
  const int* const table = PAGED ? p.tables + (size_t)b * p.max_blocks : nullptr;
  const int tpb = PAGED ? p.block_size / 64 : 1;
  const int bt0 = PAGED && lane / tpb < p.max_blocks ? table[lane / tpb] : 0;
  const int bt1 = PAGED && (64 + lane) / tpb < p.max_blocks ? table[(64 + lane) / tpb] : 0;
  const int srow = 8 * w + (lane >> 3);
  const unsigned sch = 16u * (unsigned)((lane & 7) ^ ((2 * (srow >> 1)) & 7));  // (rows 32 apart share it)
  const unsigned kvb = PAGED ? 128u : (unsigned)p.kv_tok * 2u;
  auto stage = [&](int buf, int kt) {
    char* dst = smem + buf * 2 * kPkTile + w * 1024;
    int first = 64 * kt;
    if constexpr (PAGED) {
      const int blk = kt < 64 ? __builtin_amdgcn_readlane(bt0, kt) : kt < 128 ? __builtin_amdgcn_readlane(bt1, kt - 64)
                                                                    : __builtin_amdgcn_readfirstlane(((volatile const int*)table)[kt / tpb]);
      const size_t base = (((size_t)blk * (p.heads / p.group) + hq / p.group) * p.block_size + kt % tpb * 64) * 64;
      rk = pk_rsrc(p.k + base, 64, 64), rv = pk_rsrc(p.v + base, 64, 64);
      first = 0;
    }
    const int end = len - 1 - 64 * kt + first;
    const unsigned r0 = (unsigned)min(first + srow, end), r1 = (unsigned)min(first + 32 + srow, end);
    const unsigned v0 = r0 * kvb + sch, v1 = r1 * kvb + sch;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (pk_lds*)dst, 16, v0, 0u, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (pk_lds*)(dst + 4096), 16, v1, 0u, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (pk_lds*)(dst + kPkTile), 16, v0, 0u, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (pk_lds*)(dst + kPkTile + 4096), 16, v1, 0u, 0, 0);
  };

  // ---- this lane's query: B operand of K Q^T, k = 16 c + 8 h ..
  const int my_q = q0 + 32 * w + r;
  bf16x8 qf[4];
  {
    const bf16* row = p.q + (long)(start + min(my_q, nq - 1)) * p.q_tok + (long)hq * p.q_head + 8 * h;
#pragma unroll
    for (int c = 0; c < 4; ++c) qf[c] = *reinterpret_cast<const bf16x8*>(row + 16 * c);
  }
  // the query loads retire here (the statement uses them), so that every later wait counts only DMA
  asm volatile("" : "+v"(qf[0]), "+v"(qf[1]), "+v"(qf[2]), "+v"(qf[3])::"memory");
  if (!PAGED || tiles > 0) stage(0, 0);

  const int ksw = (r >> 1) & 3;
  int kof[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) kof[c] = r * 128 + 16 * (2 * (c ^ ksw) + h);
  // transposed V reads: lane 4 q + p of a 16-lane group names row q, columns 4 p .. of its 16 columns
  const int vq = (lane >> 2) & 3, vp = lane & 3, vsw = 2 * ((2 * h + (vq >> 1)) & 3);
  int vof[2];
#pragma unroll
  for (int d = 0; d < 2; ++d)
    vof[d] = (4 * h + vq) * 128 + 16 * ((4 * d + 2 * ((lane >> 4) & 1) + (vp >> 1)) ^ vsw) + 8 * (vp & 1);

  f32x16 o[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) o[0][i] = o[1][i] = 0.f;
  float m_run = -1e30f, l_run = 0.f;

  int buf = 0;
  for (int kt = 0; kt < tiles; ++kt) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last tile's reads: its buffer is filled next
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + 1 < tiles) stage(buf ^ 1, kt + 1);
    const char* ks = smem + buf * 2 * kPkTile;
    const char* vs = ks + kPkTile;
    buf ^= 1;
    if (!work || (PAGED && 64 * kt > past + q0 + 32 * w + 31)) continue;  // (PAGED: keys behind all of the wave's queries)

    f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        s[kb] = mfma32(*reinterpret_cast<const bf16x8*>(ks + kb * 4096 + kof[c]), qf[c], s[kb]);
    }
    // s[kb][i]: key 64 kt + 32 kb + (i & 3) + 8 (i >> 2) + 4 h of this lane's query
    if (64 * kt + 64 > len || (PAGED && 64 * kt + 63 > past + q0 + 32 * w)) {
      const int left = (PAGED ? min(len, past + my_q + 1) : len) - 64 * kt - 4 * h;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (32 * kb + (i & 3) + 8 * (i >> 2) >= left) s[kb][i] = -__builtin_huge_valf();
    }
    float mx = max32(s[0], s[1]) * p.scale_log2;  // scale > 0 (launcher)
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // the running maximum is kept until a row's maximum grows by more than 2^8 (P stays <= 2^8): the rescale of O and l
    // is skipped on most tiles
    const bool keep = __all(mx - m_run <= 8.f);
    const float m_new = keep ? m_run : fmaxf(m_run, mx);
    float ls = 0.f;
    bf16x8 pb[4];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int g2 = 0; g2 < 2; ++g2) {
        u32x4 pk;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e0 = __builtin_amdgcn_exp2f(fmaf(s[kb][8 * g2 + 2 * j], p.scale_log2, -m_new));
          const float e1 = __builtin_amdgcn_exp2f(fmaf(s[kb][8 * g2 + 2 * j + 1], p.scale_log2, -m_new));
          ls += e0 + e1;
          pk[j] = pack2bf(e0, e1);
        }
        pb[2 * kb + g2] = __builtin_bit_cast(bf16x8, pk);
      }
    if (keep) {
      l_run += ls;
    } else {
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run = l_run * alpha + ls;
      m_run = m_new;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        o[0][i] *= alpha;
        o[1][i] *= alpha;
      }
    }
    // slot j of lane half h in 16-key block kb: key 16 kb + 4 h + j (j < 4) or 16 kb + 8 + 4 h + j - 4
#pragma unroll
    for (int kp = 0; kp < 2; ++kp) {
      u32x2 v[8];  // [16-key block of the pair][d][lower / upper keys]
      pk_read_tr8(lds_addr(vs) + kp * 4096 + vof[0], lds_addr(vs) + kp * 4096 + vof[1], v);
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const u32x2 lo = v[4 * k2 + 2 * d], hi = v[4 * k2 + 2 * d + 1];
          o[d] = mfma32(__builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]}), pb[2 * kp + k2], o[d]);
        }
    }
  }
  if (!work) return;
  const float l = l_run + __shfl_xor(l_run, 32, 64);
  if (my_q >= nq) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bf16* row = p.out + (long)(start + my_q) * p.o_tok + (long)hq * p.o_head + 4 * h;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x2*>(row + 32 * d + 8 * i) =
          u32x2{pack2bf(o[d][4 * i] * inv, o[d][4 * i + 1] * inv), pack2bf(o[d][4 * i + 2] * inv, o[d][4 * i + 3] * inv)};
}

// Whether the 32 x 32 form is the faster one for `units` (sequence, head) pairs of up to max_len tokens.  Texts of one
// 64-query block are a chain of one tile either way.  Up to 256 tokens the 16 x 16 form's workgroups of 64 queries start
// quicker as long as each of them has a CU.  us, 16 x 16 form / this one, 12 heads: 1 text of 112 tokens 4.8 / 5.2, 8 of
// 128 5.2 / 5.4, 12 of 128 5.9 / 5.5, 1 of 192 5.9 / 6.0, 6 of 256 8.4 / 7.4, 1 of 512 11.2 / 10.8, 3 of 512 13.6 / 11.1.
bool flash_packed64_wins(long units, int max_len) {
  return max_len > 256 || (max_len > 64 && units * ((max_len + 63) / 64) > 256);
}

int flash_packed64(const void* q, long q_tok, long q_head, const void* k, const void* v, long kv_tok, long kv_head, void* out,
                   long o_tok, long o_head, const int* cu, int batch, int max_len, int Hq, int Hkv, float scale, hipStream_t s) {
  if (batch <= 0 || max_len <= 0) return 0;
  if (Hkv <= 0 || Hq % Hkv || !(scale > 0.f) || kv_tok <= 0 || (long)max_len * kv_tok * 2 >= (1L << 31) ||
      ((long)batch * Hq + 8) * ((max_len + 127) / 128) >= (1L << 31))
    return hipErrorInvalidValue;
  const PackedParams p = {(const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, q_tok, q_head, kv_tok, kv_head, o_tok,
                          o_head, cu, Hq / Hkv, Hq, batch * Hq, (max_len + 127) / 128, scale * 1.4426950408889634f, nullptr, nullptr, 0, 0};
  hipLaunchKernelGGL(flash_packed64_kernel<false>, dim3((unsigned)((p.units + 7) / 8 * 8 * p.nqb)), dim3(256), 0, s, p);
  return hipGetLastError();
}

// Causal attention of packed queries [T, Hq, 64] over a paged cache.
int flash_paged64(const void* q, long q_tok, long q_head, const void* k_cache, const void* v_cache, const int* tables,
                  int max_blocks, int block_size, void* out, long o_tok, long o_head, const int* cu, const int* ctx, int batch, int max_q, int Hq,
                  int Hkv, float scale, hipStream_t s) {
  if (batch <= 0 || max_q <= 0) return 0;
  if (Hkv <= 0 || Hq % Hkv || !(scale > 0.f) || block_size <= 0 || block_size % 64 ||
      ((long)batch * Hq + 8) * ((max_q + 127) / 128) >= (1L << 31))
    return hipErrorInvalidValue;
  const PackedParams p = {(const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, (bf16*)out, q_tok, q_head, 0, 0, o_tok,
                          o_head, cu, Hq / Hkv, Hq, batch * Hq, (max_q + 127) / 128, scale * 1.4426950408889634f, tables, ctx,
                          max_blocks, block_size};
  hipLaunchKernelGGL(flash_packed64_kernel<true>, dim3((unsigned)((p.units + 7) / 8 * 8 * p.nqb)), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace dab
