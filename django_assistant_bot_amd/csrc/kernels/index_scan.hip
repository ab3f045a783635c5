// Persistent exact-cosine scan of the in-HBM index (the threshold-candidate pass of VectorIndex search; the pgvector
// CosineDistance ORDER BY it replaces: reference rag/services/search_service.py:185-196).
//
// The scan is an HBM stream (1.5 GB for 1M x 768 rows; 128 queries x 1M rows are 0.2 TFLOP, half of the stream's time on
// the matrix cores).  The GEMM kernels stage the queries again for every output tile (as many L2 bytes as the rows they
// scan); here they are read ONCE per workgroup and a persistent grid streams the rows.  Two kernels:
//   * index_scan_kernel: row-major rows, 1-96 queries in LDS, rows in a VGPR ring;
//   * index_scan_reg_kernel: rows of a shuffle_weights copy (each 16-row x 32-k A fragment is 1 KB contiguous in lane
//     order), 1-256 queries in registers, rows in an LDS ring.
//
// index_scan_kernel:
//   * MT 16-query tiles (M <= 16 MT): MT 1-2 -> 4-wave workgroups, 2 per CU; MT 3-6 -> 8-wave
//     workgroups, 1 per CU (up to 144 KB of queries in LDS: MT 5-6 need K <= 768);
//   * persistent grid, tile = 32 rows per wave (two 16-row MFMA A tiles),
//     row-major 16-B loads (lane = row li, k 8g..8g+7 of a 32-k chunk) with the tile's base in the
//     buffer descriptor, whose range clamps the last partial tile to zeros;
//   * the ring runs across tile boundaries (a flat stream of 32-k chunks), so the next tile's loads
//     are in flight under the current tile's epilogue;
//   * queries [16 MT, K] in LDS with chunk c of row r at c ^ (r & 15): conflict-free ds_read_b128
//     B fragments (one fragment feeds both A tiles' MFMAs; one A fragment feeds MT MFMAs);
//   * epilogue straight from the accumulators: a score >= thr[query] (rare) takes a slot in the
//     wave's LDS list; flushing the list applies the row / query group filters and appends to the
//     query's global list with one returning atomic per hit (gemm.hip EPI_CANDIDATES) -- a wait
//     that in the tile loop would drain the wave's whole load ring.
#include "common.h"
#include "launchers.h"

namespace dab {

namespace {

struct ScanParams {
  const bf16* X;  // queries [M, K]
  long ldx;
  const bf16* W;  // index rows [N, K]
  long ldw;
  int M, N, K;
  const int* row_group;
  const int* q_group;
  const float* thr;
  int* cnt;
  float* cand_val;
  int* cand_idx;
  int cap;
  float* scores;  // SCORES: [M][N]
  const uint32_t* allow;  // SCORES: [M][ceil(N / 32)] row bitmask or null
  uint32_t* parts;        // SCORES: [M][ldp] the greatest ordered bits (float_key) of every 16 rows, or null
  int ldp;
};

constexpr int kScanKMax = 1024;
constexpr int kScanMaxM = 96;
// widest rows the queries of MT 16-query tiles may have (LDS: 16 MT KMax 2 B <= 144 KB)
constexpr int scan_kmax(int mt) { return mt <= 4 ? kScanKMax : 768; }
constexpr int kScanRT = 2;     // 16-row A tiles per wave
constexpr int kScanNWIN = 8;   // chunks (of 32 k) in flight per wave
constexpr int kScanListW = 160;  // candidate list entries per wave (12 B each)

}  // namespace

template <int MT, int NW>
__global__ __launch_bounds__(64 * NW, 8 / NW) void index_scan_kernel(ScanParams p) {
  constexpr int RT = kScanRT, NWIN = kScanNWIN, TR = 32 * NW;  // rows per workgroup tile
  constexpr int XS = 16 * MT * scan_kmax(MT) * 2;
  __shared__ __attribute__((aligned(16))) char xs[XS + 64 + NW * kScanListW * 12];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cpr = p.K / 8;  // 16-B chunks per query row
  const int RB = p.K * 2;

  // ---- per-wave candidate lists (after the queries): a hit takes an LDS slot; the group filters
  // and the global append (a returning atomic, whose wait would drain this wave's whole load ring)
  // run when the list is flushed -- at a high-water mark and at the end
  int* const lcnt = reinterpret_cast<int*>(xs + XS);
  int* const l_n = lcnt + 16 + w * kScanListW;
  int* const l_m = lcnt + 16 + NW * kScanListW + w * kScanListW;
  float* const l_v = reinterpret_cast<float*>(lcnt + 16 + 2 * NW * kScanListW + w * kScanListW);
  auto cand_global = [&](int m, int n, float v) {
    const int rg = p.row_group ? p.row_group[n] : 0;
    const int qgm = p.q_group ? p.q_group[m] : -1;
    if (rg >= 0 && (qgm < 0 || rg == qgm)) {
      const int slot = atomicAdd(p.cnt + m, 1);
      if (slot < p.cap) {
        p.cand_val[(size_t)m * p.cap + slot] = v;
        p.cand_idx[(size_t)m * p.cap + slot] = n;
      }
    }
  };
  auto list_count = [&]() {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(lcnt + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  };
  auto cand_flush = [&]() {  // wave-uniform
    const int c = list_count();
    for (int e = lane; e < c; e += 64) cand_global(l_m[e], l_n[e], l_v[e]);
    if (lane == 0) __hip_atomic_store(lcnt + w, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    // retire the flush's own memory ops here, so the code after it (and the hit test of every tile,
    // which the compiler merges with this path) inherits no pending store or load to wait for
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  };
  if (tid < NW) lcnt[tid] = 0;

  // ---- queries -> LDS once (rows >= M repeat row M - 1; their scores are never appended)
  for (int e = tid; e < 16 * MT * cpr; e += 64 * NW) {
    const int r = e / cpr, c = e % cpr;
    const u32x4 v = *reinterpret_cast<const u32x4*>(p.X + (size_t)min(r, p.M - 1) * p.ldx + 8 * c);
    *reinterpret_cast<u32x4*>(xs + r * RB + 16 * (c ^ (r & 15))) = v;
  }
  float thr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = 16 * t + li;
    thr[t] = m < p.M ? p.thr[m] : __builtin_nanf("");
  }
  __syncthreads();

  // ---- flat chunk stream over this wave's tiles: tile i of the wave = rows
  // (blockIdx.x + i * gridDim.x) * TR + 32 w .. + 31; chunk = 32 k of both 16-row A tiles
  const int nck = p.K / 32;  // chunks per tile (a multiple of NWIN: checked by the launcher)
  const int tiles = (p.N + TR - 1) / TR;
  const int my_tiles = blockIdx.x < tiles ? (tiles - 1 - blockIdx.x) / gridDim.x + 1 : 0;
  if (my_tiles == 0) return;
  auto tile_row0 = [&](int i) { return (blockIdx.x + i * gridDim.x) * TR + 32 * w; };
  // descriptor of tile i (rows past N read zeros); past the wave's last tile or wholly past N: empty
  // range (the ring's loads return zeros without memory traffic)
  auto rsrc_of = [&](int i) {
    const int r0 = tile_row0(i);
    const bool live = i < my_tiles && r0 < p.N;
    const int rows = live ? min(32, p.N - r0) : 0;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(p.W + (size_t)min(r0, p.N - 1) * p.ldw), (short)0,
                                             (int)(rows * p.ldw * 2), 0x00020000);
  };
  const int voff = (int)((li * p.ldw + 8 * g) * 2);
  const int astr = (int)(16 * p.ldw * 2);  // next 16-row block
  constexpr int CSTR = 64;                 // next 32-k chunk

  bf16x8 wr[NWIN][RT];
  int ld_tile = 0, ld_c = 0;  // next chunk to load (wave-uniform)
  auto ld_rs = rsrc_of(0);
  auto load = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < RT; ++a)
      wr[slot][a] = __builtin_bit_cast(
          bf16x8, __builtin_amdgcn_raw_buffer_load_b128(ld_rs, voff + a * astr, ld_c * CSTR, 2));  // nt: read once
    if (++ld_c == nck) {
      ld_c = 0;
      ld_rs = rsrc_of(++ld_tile);
    }
  };
#pragma unroll
  for (int s = 0; s < NWIN; ++s) load(s);

  f32x4 acc[RT][MT];
  for (int i = 0; i < my_tiles; ++i) {
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[a][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < nck; c0 += NWIN) {
#pragma unroll
      for (int s = 0; s < NWIN; ++s) {
        const int c = c0 + s;
        bf16x8 bx[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t)
          bx[t] = *reinterpret_cast<const bf16x8*>(xs + (16 * t + li) * RB + 16 * ((4 * c + g) ^ li));
#pragma unroll
        for (int a = 0; a < RT; ++a)
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[a][t] = mfma16(wr[s][a], bx[t], acc[a][t]);
        load(s);  // refill the slot right behind its MFMAs (NWIN chunks ahead)
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // ---- candidates: acc[a][t] lane (li, g) = scores of query 16 t + li against rows 16 a + 4 g + r
    const int r0 = tile_row0(i);
    if (r0 >= p.N) continue;  // wave-uniform
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = r0 + 16 * a + 4 * g + r;
          const float v = acc[a][t][r];
          const bool hit = v >= thr[t] && n < p.N;
          // the list holds <= kScanListW - 64 entries here, so the <= 64 hits of one step fit
          if (__builtin_amdgcn_ballot_w64(hit)) {
            if (hit) {
              const int slot = __hip_atomic_fetch_add(lcnt + w, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              l_n[slot] = n;
              l_m[slot] = 16 * t + li;
              l_v[slot] = v;
            }
            if (list_count() > kScanListW - 64) cand_flush();
          }
        }
  }
  cand_flush();
}

// The scan of a shuffle_weights copy: the queries stay in REGISTERS, the rows pass through LDS.
//   * 8 waves = QG query groups of MT 16-query tiles x 8 / QG row halves; a wave holds its queries' fragments for the
//     whole launch (4 VGPRs per 16 queries x 32 k: MT 2 at K 768 = 192), so its product needs one LDS read per row
//     fragment and nothing else;
//   * a stage = 32 rows x half of K (all of it at K 256), copied by LDS-DMA (the layout is lane order already: no
//     swizzle, no conflicts), NS stages in a ring (128-144 KB), all but the one in use in flight: HBM latency is covered
//     by the ring, not by waves;
//   * one barrier a stage (1 us of HBM time at K 768);
//   * LDS reads: QG x the row bytes.  1M rows of 768: 24 MB a CU with 4 groups (80 us), 48 MB with 8 (160 us), below the
//     stream's 236 us at 6.5 TB/s.
// Hits (a score >= thr[query]; some 1500 a query) are listed in LDS, the slot from the ballot (an LDS atomic would make the
// compiler drain the ring).  Their append to the query's global list was what bounded the scan next: an atomic per hit,
// and counters of 32 queries share a cache line (K 256, 1M rows, 128 queries: 238 us against 81 us for one query), and a
// wave that flushes holds up the others at the barrier.  So the workgroup flushes together (a long list of one wave raises
// a flag) with one global atomic per query that has hits.
// SCORES: every score is stored instead, -inf where the group filters or the row mask drop the row, and on request the
// greatest of every 16 rows (what the selection of the best k reads first: search.hip).  The filters of a tile travel with
// its rows, one 4-B copy a lane, and every wave issues the same stores for every tile (masked lanes past the buffer's
// end), so that the counted wait knows what is younger than the stage it waits for; a load of the filters where they are
// used, or a wait for the stores, would empty the ring once a tile.  us, rows of 768 (gemm_bt's scores): 4 queries of 60,001
// rows 17.6 (21.0), 10 of 142,939 41 (51), 42 of 31,098 14.9 (20.8), 1 of 1,000,003 234 (6.6 TB/s).
// 1M rows of 768, us (floor 236), against queries in LDS / gemm256's candidate epilogue above 96: 1 query 226 (242), 16:
// 226 (245), 64: 234 (291), 96: 232 (301), 128: 248 (400), 192: 347 (444), 256: 378 (467); of 1024: 1: 300 (315), 128: 333
// (470); of 256: 1: 81 (83), 128: 124 (257).  20k rows of 768: 1: 21 (23), 128: 27 (36).
constexpr int kRegList = 184;  // hits a wave lists (10 B each)

template <int NCK, int MT, int QG, bool SCORES>
__global__ __launch_bounds__(512, 2) void index_scan_reg_kernel(ScanParams p) {
  constexpr int RW = 8 / QG, RB = 2 / RW;  // row halves, 16-row blocks of a wave
  constexpr int H = NCK > 8 ? 2 : 1, HALF = NCK / H;  // stages of a tile, 32-k chunks of a stage
  constexpr int kStage = 2 * HALF * 1024, kDma = kStage / 8192;
  constexpr int NS = NCK <= 16 ? 8 : NCK == 24 ? 6 : 4;
  constexpr int TS = NS / H + 2;  // SCORES: tiles whose filters are held (256 B a wave: 32 row groups, 32 mask words)
  constexpr int kQ = 16 * MT * QG, kTail = SCORES ? TS * 8 * 256 + 4 * kQ : 64 + 4 * kQ + 8 * kRegList * 10;
  static_assert(RW * RB == 2 && kQ <= 512 && NCK % 8 == 0 && NS * kStage + kTail <= 160 * 1024, "LDS");
  // entries of a wave's memory queue younger than a stage's rows: those of the NS - 2 stages behind it, and the stores
  // of the tiles that ended since (SCORES)
  constexpr int kYoung = (NS - 2) * kDma + (SCORES ? 2 * ((NS - 2) / H) : 0), kStores = SCORES ? 2 * RB * MT : 0;
  static_assert(kYoung <= 63 && (NS - 2) % H == 0, "vmcnt range");
  typedef __attribute__((address_space(3))) void scan_lds;
  // one array: with two the compiler knows which of them the copies write, and waits for all copies before each read
  __shared__ __attribute__((aligned(16))) char ring[NS * kStage + kTail];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qg = w % QG, rw = w / QG, q0 = 16 * MT * qg;
  const bool live = q0 < p.M;  // wave-uniform: a group without queries only copies
  // [tile & 1]: a list grew long in that tile; read in the next one (between two barriers that keep its writers away)
  int* const flag = reinterpret_cast<int*>(ring + NS * kStage);
  int* const qcnt = reinterpret_cast<int*>(ring + NS * kStage + 64);               // [kQ]
  int* const l_n = qcnt + kQ + w * kRegList;
  float* const l_v = reinterpret_cast<float*>(qcnt + kQ + 8 * kRegList) + w * kRegList;
  uint16_t* const l_m = reinterpret_cast<uint16_t*>(qcnt + kQ + 16 * kRegList) + w * kRegList;  // query of the group
  int listed = 0;  // wave-uniform

  auto passes = [&](int e) {  // the group filters of hit e
    const int rg = p.row_group ? p.row_group[l_n[e]] : 0;
    const int qgm = p.q_group ? p.q_group[q0 + l_m[e]] : -1;
    return rg >= 0 && (qgm < 0 || rg == qgm);
  };
  auto put = [&](int e, int m, int slot) {
    if (slot >= p.cap) return;
    const size_t at = (size_t)(q0 + m) * p.cap + slot;
    p.cand_val[at] = l_v[e];
    p.cand_idx[at] = l_n[e];
  };
  auto drained = [] { __builtin_amdgcn_s_waitcnt(0x0f70); };  // vmcnt(0): the counted waits start from an empty queue
  // all waves: the hits of a query take their slots with one global atomic of the workgroup
  auto flush_all = [&]() {
    if (tid < kQ) qcnt[tid] = 0;
    __syncthreads();
    if (tid < 2) flag[tid] = 0;
    for (int e = lane; e < listed; e += 64)  // l_m: query and rank among the workgroup's hits of the query (< 2 kRegList)
      l_m[e] = passes(e) ? l_m[e] | atomicAdd(qcnt + q0 + l_m[e], 1) << 5 : 0xffff;
    __syncthreads();
    if (tid < kQ && qcnt[tid]) qcnt[tid] = atomicAdd(p.cnt + tid, qcnt[tid]);
    __syncthreads();
    for (int e = lane; e < listed; e += 64)
      if (l_m[e] != 0xffff) put(e, l_m[e] & 31, qcnt[q0 + (l_m[e] & 31)] + (l_m[e] >> 5));
    listed = 0;
    drained();
  };
  // this wave alone, inside a tile with more hits than the list has room for
  auto flush_own = [&]() {
    for (int e = lane; e < listed; e += 64)
      if (passes(e)) put(e, l_m[e], atomicAdd(p.cnt + q0 + l_m[e], 1));
    listed = 0;
    drained();
  };
  int* const groups = reinterpret_cast<int*>(ring + NS * kStage + TS * 8 * 256);  // SCORES: of the queries (negative: any)
  if (SCORES) {
    if (tid < kQ) groups[tid] = p.row_group && p.q_group ? p.q_group[min(tid, p.M - 1)] : -1;
  } else if (tid < 2) {
    flag[tid] = 0;
  }  // read behind the first stage's barrier

  // queries -> registers (rows past the last repeat it; no score reaches their NaN threshold)
  bf16x8 qf[MT][NCK];
  float thr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = q0 + 16 * t + li;
    const bf16* x = p.X + (size_t)min(m, p.M - 1) * p.ldx + 8 * g;
#pragma unroll
    for (int c = 0; c < NCK; ++c) qf[t][c] = *reinterpret_cast<const bf16x8*>(x + 32 * c);
    thr[t] = !SCORES && m < p.M ? p.thr[m] : __builtin_nanf("");
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int c = 0; c < NCK; ++c) asm volatile("" : "+v"(qf[t][c]));  // loaded: the waits below count copies only
    asm volatile("" : "+v"(thr[t]));
  }

  const int tiles = (p.N + 31) / 32;
  const int steps = H * ((tiles - 1 - (int)blockIdx.x) / (int)gridDim.x + 1);  // grid <= tiles
  unsigned dma_off[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int d = w + 8 * i;
    dma_off[i] = (unsigned)(((d / HALF) * NCK + d % HALF) * 1024 + lane * 16);
  }
  // SCORES: a tile's filters, by lanes 0..31: the rows' groups, and behind them the mask words of the wave's queries
  const int words = (p.N + 31) / 32;
  const __amdgpu_buffer_rsrc_t rs_group =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(p.row_group), (short)0, SCORES && p.row_group ? p.N * 4 : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_allow = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(p.allow), (short)0, SCORES && p.allow ? (int)((unsigned)p.M * (unsigned)words * 4u) : 0, 0x00020000);
  const uint32_t no_mask = p.allow ? 0u : ~0u;
  const unsigned allow_off = SCORES ? (unsigned)(q0 + min(lane, 16 * MT - 1)) * (unsigned)words * 4u : 0u;
  auto filters = [&](int st) {
    const unsigned tile = st < steps ? blockIdx.x + (unsigned)(st / H) * gridDim.x : 0u;
    char* dst = ring + NS * kStage + (((unsigned)(st / H) % TS) * 8 + w) * 256;
    if (lane < 32) {  // (past the end: zeros)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_group, (scan_lds*)dst, 4, 4u * lane, 128u * tile, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_allow, (scan_lds*)(dst + 128), 4, allow_off, 4u * tile, 0, 0);
    }
  };
  // a stage past the last reads an empty range (zeros, no traffic): every step adds the same copies to the queue
  // (first: it starts a tile)
  auto stage = [&](int buf, int st, bool first) {
    if (SCORES && first) filters(st);
    const size_t tile = blockIdx.x + (size_t)(st / H) * gridDim.x;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p.W + (st < steps ? tile : 0) * (2 * NCK * 512)), (short)0,
                                          st < steps ? 2 * NCK * 1024 : 0, 0x00020000);
    const unsigned so = (unsigned)(st % H) * (unsigned)(HALF * 1024);
    char* dst = ring + buf * kStage + w * 1024;
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (scan_lds*)(dst + i * 8192), 16, (unsigned)dma_off[i], so, 0, 2);
  };
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) stage(st, st, st % H == 0);
  // buffers of the scores and the parts' maxima: a lane without one stores past their end, where it is dropped
  const __amdgpu_buffer_rsrc_t rs_scores =
      __builtin_amdgcn_make_buffer_rsrc(p.scores, (short)0, SCORES ? (int)((unsigned)p.M * (unsigned)p.N * 4u) : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_parts =
      __builtin_amdgcn_make_buffer_rsrc(p.parts, (short)0, p.parts ? (int)((unsigned)p.M * (unsigned)p.ldp * 4u) : 0, 0x00020000);
  int buf = 0;
  for (int st = 0; st < steps; st += H) {
    f32x4 acc[RB][MT];
#pragma unroll
    for (int a = 0; a < RB; ++a)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[a][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < H; ++h) {
      // the stores of tile j are younger than stage s where H j + H + NS - 2 >= s: those of the last tiles before this one
      constexpr int kEnded = (NS - 1) / H, kMost = kYoung + kEnded * kStores;  // (one more tile at the first of two stages)
      if (SCORES && live && st / H > kEnded)
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kMost < 63 ? kMost : 63) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kYoung) : "memory");
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last stage's reads: its buffer is filled next
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      stage(buf == 0 ? NS - 1 : buf - 1, st + h + NS - 1, (h + NS - 1) % H == 0);
      if (live) {
        const char* src = ring + buf * kStage + rw * (HALF * 1024) + lane * 16;
        constexpr int PF = 4 / RB;  // fragments read ahead
        bf16x8 rf[PF][RB];
#pragma unroll
        for (int c = 0; c < PF; ++c)
#pragma unroll
          for (int a = 0; a < RB; ++a) rf[c][a] = *reinterpret_cast<const bf16x8*>(src + (a * HALF + c) * 1024);
#pragma unroll
        for (int c = 0; c < HALF; ++c) {
#pragma unroll
          for (int a = 0; a < RB; ++a)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[a][t] = mfma16(rf[c % PF][a], qf[t][h * HALF + c], acc[a][t]);
          if (c + PF < HALF)
#pragma unroll
            for (int a = 0; a < RB; ++a)
              rf[c % PF][a] = *reinterpret_cast<const bf16x8*>(src + (a * HALF + c + PF) * 1024);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      buf = buf == NS - 1 ? 0 : buf + 1;
      if (!SCORES && h == 0) {
        int full;
        asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                     : "=v"(full) : "v"((unsigned)(uintptr_t)(scan_lds*)(flag + ((st / H + 1) & 1))) : "memory");
        if (__builtin_amdgcn_readfirstlane(full)) flush_all();
      }
    }
    if (!live) continue;
    const int r0 = (blockIdx.x + st / H * gridDim.x) * 32 + 16 * RB * rw;
    if constexpr (SCORES) {
      const unsigned at = (unsigned)(uintptr_t)(scan_lds*)(ring + NS * kStage + (((unsigned)(st / H) % TS) * 8 + w) * 256);
#pragma unroll
      for (int a = 0; a < RB; ++a) {
        const int n = r0 + 16 * a + 4 * g, in = n & 31;  // (N % 4 == 0: four rows are there or none of them)
        int4 group;  // (read by asm statements: before an ordinary read hipcc may drain the copies in flight)
        asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(group) : "v"(at + 4u * in) : "memory");
        const int rg[4] = {group.x, group.y, group.z, group.w};
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const int m = q0 + 16 * t + li;
          uint32_t seen;
          int q_group;
          asm volatile("ds_read_b32 %0, %2\n\tds_read_b32 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(seen), "=&v"(q_group)
                       : "v"(at + 128u + 4u * (16 * t + li)), "v"((unsigned)(uintptr_t)(scan_lds*)(groups + m)) : "memory");
          seen = (seen | no_mask) >> in;
          f32x4 v;  // (without branches: hipcc lost a lane's -inf behind those of && on vector elements)
          uint32_t best = 0;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool pass = (rg[r] >= 0) & ((q_group < 0) | (rg[r] == q_group)) & ((seen >> r & 1u) != 0u) & (n < p.N);
            const float x = pass ? acc[a][t][r] : -__builtin_huge_valf();
            best = max(best, float_key(x));
            v[r] = x;
          }
          const bool there = m < p.M && n < p.N;
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs_scores,
                                                 there ? ((unsigned)m * (unsigned)p.N + (unsigned)n) * 4u : 0xffffff00u, 0, 0);
          const auto s32 = __builtin_amdgcn_permlane32_swap(best, best, false, false);  // over the 16 rows
          best = max(s32[0], s32[1]);
          const auto s16 = __builtin_amdgcn_permlane16_swap(best, best, false, false);
          best = max(s16[0], s16[1]);
          __builtin_amdgcn_raw_buffer_store_b32(best, rs_parts,
                                                there && g == 0 ? ((unsigned)m * (unsigned)p.ldp + (unsigned)(n >> 4)) * 4u : 0xffffff00u,
                                                0, 0);
        }
      }
      continue;
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int a = 0; a < RB; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = r0 + 16 * a + 4 * g + r;
          const float v = acc[a][t][r];
          const bool hit = v >= thr[t] && n < p.N;
          const unsigned long long hits = __builtin_amdgcn_ballot_w64(hit);
          if (hits) {  // the list holds <= kRegList - 64 entries here
            if (hit) {
              const int slot = listed + __builtin_amdgcn_mbcnt_hi((unsigned)(hits >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)hits, 0));
              l_n[slot] = n;
              l_m[slot] = 16 * t + li;
              l_v[slot] = v;
            }
            listed += __builtin_popcountll(hits);
            if (listed > kRegList - 64) flush_own();
          }
        }
    if (listed > kRegList - 72 && lane == 0) flag[st / H & 1] = 1;
  }
  if constexpr (SCORES) drained();
  else flush_all();
}

// row-major rows
int index_scan_candidates(const void* X, long ldx, const void* W, long ldw, int M, int N, int K, const int* row_group,
                          const int* q_group, const float* thr, int* cnt, float* cand_val, int* cand_idx, int cap,
                          hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (M > kScanMaxM || K > scan_kmax((M + 15) / 16) || K % (32 * kScanNWIN) || ldx % 8 || ldw % 8 || cap <= 0)
    return hipErrorInvalidValue;
  if (32L * ldw * 2 >= (1L << 31)) return hipErrorInvalidValue;
  ScanParams p;
  p.X = (const bf16*)X;
  p.ldx = ldx;
  p.W = (const bf16*)W;
  p.ldw = ldw;
  p.M = M;
  p.N = N;
  p.K = K;
  p.row_group = row_group;
  p.q_group = q_group;
  p.thr = thr;
  p.cnt = cnt;
  p.cand_val = cand_val;
  p.cand_idx = cand_idx;
  p.cap = cap;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const int mt = (M + 15) / 16;
  const int nw = mt <= 2 ? 4 : 8, per_cu = 8 / nw;
  const long tiles = (N + 32L * nw - 1) / (32L * nw);
  const int grid = (int)(tiles < (long)per_cu * cus ? tiles : (long)per_cu * cus);
  switch (mt) {
    case 1: hipLaunchKernelGGL((index_scan_kernel<1, 4>), dim3(grid), dim3(256), 0, s, p); break;
    case 2: hipLaunchKernelGGL((index_scan_kernel<2, 4>), dim3(grid), dim3(256), 0, s, p); break;
    case 3: hipLaunchKernelGGL((index_scan_kernel<3, 8>), dim3(grid), dim3(512), 0, s, p); break;
    case 4: hipLaunchKernelGGL((index_scan_kernel<4, 8>), dim3(grid), dim3(512), 0, s, p); break;
    case 5: hipLaunchKernelGGL((index_scan_kernel<5, 8>), dim3(grid), dim3(512), 0, s, p); break;
    default: hipLaunchKernelGGL((index_scan_kernel<6, 8>), dim3(grid), dim3(512), 0, s, p); break;
  }
  return hipGetLastError();
}

// Query groups of index_scan_reg_kernel and their 16-query tiles for M queries of K; 0: not taken.  What the registers
// hold: 2 tiles a wave up to K 768, 1 at K 1024.  Four groups (two waves a group, each with half of the rows) as long as
// they suffice: half the LDS reads.
static int scan_groups(int M, int K, int* mt) {
  if (M <= 0 || K <= 0 || K % 256 || K > kScanKMax) return 0;
  const int most = K > 768 ? 1 : 2;
  for (int qg = 4; qg <= 8; qg += 4)
    for (*mt = 1; *mt <= most; ++*mt)
      if (M <= 16 * qg * *mt) return qg;
  return 0;
}

int index_scan_takes(int M, int K) {
  int mt;
  return scan_groups(M, K, &mt) != 0;
}

template <bool SCORES>
static int scan_reg_launch(const ScanParams& p, hipStream_t s) {
  int mt, dev = 0, cus = 256;
  const int qg = scan_groups(p.M, p.K, &mt);
  if (!qg || p.ldx % 8) return hipErrorInvalidValue;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const int grid = (int)min((long)cus, (p.N + 31L) / 32);
#define SCAN_REG(NCK_, MT_, QG_)                  \
  if (p.K == 32 * NCK_ && mt == MT_ && qg == QG_) \
    hipLaunchKernelGGL((index_scan_reg_kernel<NCK_, MT_, QG_, SCORES>), dim3(grid), dim3(512), 0, s, p)
#define SCAN_REG_K(NCK_)   \
  SCAN_REG(NCK_, 1, 4);    \
  SCAN_REG(NCK_, 2, 4);    \
  SCAN_REG(NCK_, 1, 8);    \
  SCAN_REG(NCK_, 2, 8)
  SCAN_REG_K(8);
  SCAN_REG_K(16);
  SCAN_REG_K(24);
  SCAN_REG(32, 1, 4);
  SCAN_REG(32, 1, 8);
#undef SCAN_REG_K
#undef SCAN_REG
  return hipGetLastError();
}

// W: the rows in the shuffle_weights layout, with at least round_up(N, 32) rows
int index_scan_candidates_shuf(const void* X, long ldx, const void* W, int M, int N, int K, const int* row_group,
                               const int* q_group, const float* thr, int* cnt, float* cand_val, int* cand_idx,
                               int cap, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (cap <= 0) return hipErrorInvalidValue;
  const ScanParams p = {(const bf16*)X, ldx, (const bf16*)W, K, M, N, K, row_group, q_group, thr, cnt, cand_val, cand_idx, cap, nullptr, nullptr, nullptr, 0};
  return scan_reg_launch<false>(p, s);
}

// ... their scores [M][N], N % 4 == 0, -inf where the groups or the row mask drop a row; parts (or null): the greatest
// ordered bits of every 16 rows, [M][ldp]
int index_scan_scores_shuf(const void* X, long ldx, const void* W, int M, int N, int K, const int* row_group,
                           const int* q_group, const void* allow, float* scores, void* parts, int ldp, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 4 || ((uintptr_t)scores | (uintptr_t)row_group) % 16 || (parts && ldp < (N + 15) / 16)) return hipErrorInvalidValue;
  if ((long)M * N * 4 > 0xffffff00L || (parts && (long)M * ldp * 4 > 0xffffff00L)) return hipErrorInvalidValue;  // buffer range
  const ScanParams p = {(const bf16*)X, ldx, (const bf16*)W, K, M, N, K, row_group, q_group, nullptr, nullptr, nullptr, nullptr, 0,
                        scores, (const uint32_t*)allow, (uint32_t*)parts, ldp};
  return scan_reg_launch<true>(p, s);
}

}  // namespace dab
