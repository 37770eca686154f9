// Dense causal prefill over the paged cache, gfx950 MFMA (fp16 in, fp32 acc).
//
// Replaces BatchPrefillWithPagedKVCacheKernel (kernels/aoa_kv/kernels/include/
// prefill/prefill.cuh:688-870) for one sequence: o = softmax(q k^T / sqrt(d)) v
// with query i (position L - qo_len + i) attending keys 0 .. L - qo_len + i.
//
// Formulation: each wave owns 32 queries and computes the transposed scores
// S^T = K Q^T with v_mfma_f32_32x32x16_f16 (keys on the MFMA rows, queries on
// the columns).  In the 32x32 accumulator lane l holds column l%32, so every
// lane holds the scores of ONE query -- its own -- for 16 of the tile's 32
// keys (the other 16 sit in lane l^32).  The softmax row statistics are
// therefore per lane (plus one exchange with lane l^32), and the fp16
// probabilities already sit in the B-operand layout of O^T += V^T P^T, so P
// never goes through LDS.  Lane layouts (checked on the hardware):
//   A: lane l -> row l%32, 8 k-values;  B: lane l -> column l%32, 8 k-values,
//   A and B elements with the same (l/32, j) share a k;
//   C: register i of lane l -> row 8*(i/4) + 4*(l/32) + i%4, column l%32.
//
// Block = 4 waves = 128 queries of one head.  K and V tiles of 64 keys go
// from the paged cache straight into LDS (global_load_lds_dwordx4, no
// register staging), double-buffered so tile i+1 loads while tile i is
// computed.  Rows are 256 bytes (one key, 128 dims) with their 16-byte
// chunks permuted per row (k_swz / v_swz below), so the K reads of a wave
// and the V transpose reads hit distinct banks (no LDS bank conflicts,
// measured with SQ_LDS_BANK_CONFLICT).  Each wave
// loads 16 rows per tile: one page of 16 tokens, half a page of 32 or two
// pages of 8, so its page ids are one or two scalar loads; with pages of 1,
// 2 or 4 tokens, each lane loads the id of the page of its rows (one vector
// load per load instruction).  Either way fetched a tile ahead.  The V^T operand of O^T += V^T P^T is read from the
// row-major V tile with ds_read_b64_tr_b16: in each 16-lane group, output
// lane 4a+b receives element b of the 8-byte blocks addressed by lanes a,
// a+4, a+8, a+12 (checked on the hardware), so four lanes pointing at four
// consecutive key rows give each lane one dim of four keys.
#include "kernels.hpp"

namespace aoakv {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4;
typedef __attribute__((address_space(3))) char lds_char;

constexpr int kPfThreads = 256;
constexpr int kPfQueriesPerWave = 32;
constexpr int kPfQueriesPerBlock = 128;
constexpr int kPfTileKeys = 64;
constexpr float kLog2e = 1.4426950408889634f;

__device__ inline floatx16 mfma32(const half8& a, const half8& b, const floatx16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// This lane's value and lane l^32's, combined: v_permlane32_swap exchanges
// the two halves of the wave in registers, where __shfl_xor would go through
// the LDS unit (ds_bpermute) and queue behind the tile reads.
__device__ inline float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// row of accumulator register i for lane group g
__device__ inline int crow(int i, int g) { return 8 * (i / 4) + 4 * g + (i % 4); }

// Chunk swizzles (16-byte chunk j of key row r sits at chunk j ^ swz(r));
// a row of D dims has CH = D / 8 chunks.  K is read as one chunk of 32
// consecutive rows per instruction: XOR with r % CH spreads them over all
// chunk positions.  V is read with the transpose read: a 16-lane group takes
// 2 adjacent chunks of 4 consecutive rows (the other group of the half-wave
// the next 2 chunks), so XOR with (CH / 4) * (r % 4) gives those chunks
// distinct positions (D = 128: 16 chunks, conflict-free as measured).
template <int CH>
__device__ inline int k_swz(int r) { return r & (CH - 1); }
template <int CH>
__device__ inline int v_swz(int r) { return (CH / 4) * (r & 3); }

// One 16-byte global -> LDS copy per lane (the lane lands at byte 16 * lane
// of `lds`).  A plain function: the builtin's operands inside the kernel
// template would be value-dependent, and the host pass then drops the
// kernel's launch stub.
__device__ inline void load_lds16(const f16* g, char* lds) {
  __builtin_amdgcn_global_load_lds(g, lds, 16, 0, 0);
}

// byte offset of 16-byte chunk j of key row r in a K tile of D-dim rows
template <int D>
__device__ inline int tile_off(int r, int j) { return r * (2 * D) + 16 * (j ^ k_swz<D / 8>(r)); }

// Tile geometry of a D-dim head (namespace-scope constants: the kernel's
// lambdas use them without capturing anything).
template <int D>
struct PfShape {
  static constexpr int kRowBytes = D * 2;                        // one key row
  static constexpr int kTileBytes = kPfTileKeys * kRowBytes;     // 16 KB at D = 128
  static constexpr int kCh = kRowBytes / 16;                     // 16-byte chunks per row
  static constexpr int kRPI = 1024 / kRowBytes;                  // rows per load instruction
  static constexpr int kKS = D / 16;                             // k-steps of the score MFMAs
  static constexpr int kDB = D / 32;                             // dim blocks of O
};

// Workgroups per CU: two at head dims 64 and 128 (64 KB of LDS and at most
// 256 registers per lane each); one at 256, whose tiles take 128 KB and whose
// O accumulators alone 128 registers (one wave per SIMD, up to 512).
template <int D>
constexpr int pf_blocks_per_cu() { return D == 256 ? 1 : 2; }

// Running max before a query's first visible key: below every score, and
// finite, so a tile (or a whole chunk) with no visible key leaves
// probabilities of 2^-inf = 0 and no inf - inf.
constexpr float kPfNoMax = -1e30f;

// Key tiles of query tile qt, and the chunks they are split into.
__host__ __device__ inline uint32_t pf_tiles(uint32_t L, uint32_t Lq, uint32_t causal,
                                             uint32_t qt) {
  uint32_t qend = (qt + 1u) * kPfQueriesPerBlock;
  qend = qend < Lq ? qend : Lq;
  const uint32_t kend = causal ? L - Lq + qend : L;
  return (kend + kPfTileKeys - 1) / kPfTileKeys;
}
// ceil(n / chunk) for n <= 2^25 tiles: chunk_rcp = floor(2^32 / chunk) + 1
// rounds n - 1 tiles down exactly while n * chunk < 2^32.
__host__ __device__ inline uint32_t pf_chunks(uint32_t n, uint32_t chunk_rcp) {
  return (uint32_t)(((uint64_t)(n - 1u) * chunk_rcp) >> 32) + 1u;
}
// floats of one item's partial: O [D / 4][128 queries][4], m [128], l [128]
__host__ __device__ constexpr size_t pf_partial_floats(int D) {
  return (size_t)kPfQueriesPerBlock * (D + 2);
}

// S: tokens per page (1, 2, 4, 8, 16 or 32); D: head dim (64, 128 or 256).
template <int S, int D>
__global__ __launch_bounds__(kPfThreads, pf_blocks_per_cu<D>()) void prefill_kernel(PrefillArgs a) {
  static_assert(S == 1 || S == 2 || S == 4 || S == 8 || S == 16 || S == 32,
                "a wave's 16 rows: 16 / S pages, or half of one");
  static_assert(D == 64 || D == 128 || D == 256, "head dims of the MFMA prefill");
  using Sh = PfShape<D>;

  // two buffers of [K | V] tiles, separate objects so the compiler sees that
  // the loads into one never alias the reads of the other (no wait on them)
  __shared__ __attribute__((aligned(16))) char s_buf0[2 * Sh::kTileBytes];
  __shared__ __attribute__((aligned(16))) char s_buf1[2 * Sh::kTileBytes];
  const int tid = threadIdx.x;
  const int lane = (int)__lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int g = lane / 32;      // lane group
  const int c = lane % 32;      // query column of this lane
  const uint32_t L = a.L, Lq = a.Lq;
  const uint32_t nqt = (Lq + kPfQueriesPerBlock - 1) / kPfQueriesPerBlock;
  // XCD-aware work order.  Workgroup b runs on XCD b % 8, and each XCD has
  // its own L2.  Items go heaviest query tile first over all heads, head
  // fastest, so with a multiple of 8 heads XCD x has the heads of x alone:
  // its Hq / 8 consecutive ones (sharing kv heads with GQA), whose K/V its L2
  // then holds for the query tiles in flight.  The lightest tiles of every
  // head come last and fill the CUs' ends.  (Other counts spread a head over 2
  // to 8 XCDs, and are still faster than head by head on one: 8192 tokens, 12
  // heads 258 -> 239 us, 20 435 -> 374, 28 514 -> 500, 6 183 -> 152.)
  const uint32_t per_head = a.chunk_rcp != 0u ? a.per_head : nqt;  // items
  const uint32_t hs = blockIdx.x % a.Hq;
  const uint32_t h = a.Hq % kXcds == 0u ? hs % kXcds * (a.Hq / kXcds) + hs / kXcds : hs;
  const uint32_t hkv = h / (a.Hq / a.H);   // its kv head (GQA groups share K/V)
  uint32_t qt = nqt - 1u, rank = blockIdx.x / a.Hq;
  const uint32_t item = h * per_head + rank;  // its partial's place
  uint32_t ntiles = 0u, nchunks = 1u;
  if (a.chunk_rcp != 0u) {
    for (;; --qt) {
      ntiles = pf_tiles(L, Lq, a.causal, qt);
      nchunks = pf_chunks(ntiles, a.chunk_rcp);
      if (rank < nchunks || qt == 0u) break;
      rank -= nchunks;
    }
  } else {
    qt -= rank;
    rank = 0u;
    ntiles = pf_tiles(L, Lq, a.causal, qt);
  }
  // this item's key tiles
  const uint32_t t0 = rank * ntiles / nchunks, t1 = (rank + 1u) * ntiles / nchunks;
  const uint32_t off = L - Lq;                 // position of query 0
  const uint32_t npages = (L + S - 1) / S;

  const uint32_t q = qt * kPfQueriesPerBlock + wave * kPfQueriesPerWave + c;
  const bool q_live = q < Lq;
  const uint32_t qpos = q_live ? off + q : L - 1u;  // last key this query sees
  // keys this wave needs (waves above the diagonal skip tiles; a wave with no
  // live query skips them all)
  const uint32_t wq_first = qt * kPfQueriesPerBlock + wave * kPfQueriesPerWave;
  uint32_t wq_last = wq_first + kPfQueriesPerWave - 1u;
  if (wq_last >= Lq) wq_last = Lq - 1u;
  const uint32_t wave_kend = wq_first >= Lq ? 0u : a.causal ? off + wq_last + 1u : L;

  // ---- this lane's query, dims 16*s + 8*g .. +8 for s < D / 16
  half8 qreg[Sh::kKS];
#pragma unroll
  for (int s = 0; s < Sh::kKS; ++s)
    qreg[s] = q_live ? *reinterpret_cast<const half8*>(a.q + ((size_t)q * a.Hq + h) * D +
                                                          16 * s + 8 * g)
                     : half8{};

  // ---- tile loader: wave w fills rows 16w .. 16w+15 of K and V (keys
  // 64 t + 16 w ..), 1 KB (Sh::kRPI rows) per instruction; lane l lands at byte
  // 16*l of its instruction's rows, i.e. row l/Sh::kCh, chunk slot l%Sh::kCh -> it
  // fetches the global chunk (l%Sh::kCh) ^ swz(row).  The page of load
  // instruction i's rows: S >= 8, id[i] (rows 0..7 of the wave one page,
  // rows 8..15 the same or, S = 8, the next); S < 8, each lane's own row's
  // page.  A page past the sequence reads the last page (its keys are
  // masked).  With S >= 8 the page table is read through the constant
  // address space: the kernel never writes it, and a scalar load keeps it
  // off the vector memory counter that the K/V tile loads are waited on with.
  constexpr int kNI = 16 / Sh::kRPI;  // load instructions per wave and tile
  struct PageIds {
    uint32_t id[kNI];
  };
  const __attribute__((address_space(4))) int32_t* kv_idx =
      (const __attribute__((address_space(4))) int32_t*)a.kv_indices;
  const int lrow = lane / Sh::kCh, lslot = lane % Sh::kCh;
  auto page_of = [&](uint32_t tile) -> PageIds {
    const uint32_t key0 = tile * kPfTileKeys + 16u * (uint32_t)wave;  // the wave's first row
    PageIds ph;
    if constexpr (S >= 8) {
      uint32_t p0 = key0 / S, p1 = (key0 + 8u) / S;
      p0 = p0 < npages ? p0 : npages - 1u;
      p1 = p1 < npages ? p1 : npages - 1u;
      const uint32_t x = (uint32_t)kv_idx[p0];
      const uint32_t y = S == 8 ? (uint32_t)kv_idx[p1] : x;
#pragma unroll
      for (int i = 0; i < kNI; ++i) ph.id[i] = Sh::kRPI * i < 8 ? x : y;
    } else {
#pragma unroll
      for (int i = 0; i < kNI; ++i) {
        uint32_t p = (key0 + (uint32_t)(Sh::kRPI * i + lrow)) / S;
        p = p < npages ? p : npages - 1u;
        ph.id[i] = (uint32_t)a.kv_indices[p];
      }
    }
    return ph;
  };
  // token slot of the wave's row 0 in its page
  const uint32_t slot0 = S == 32 ? 16u * ((uint32_t)wave % 2u) : 0u;
  auto load_tile = [&](char* buf, const PageIds& phys) {
#pragma unroll
    for (int i = 0; i < kNI; ++i) {
      const int r = 16 * wave + Sh::kRPI * i + lrow;  // row in the tile; r % 16 = Sh::kRPI i + lrow
      const uint32_t pg = phys.id[i];
      const size_t e = elem_off(a.g, pg, 0, hkv, (slot0 + (uint32_t)(r & 15)) % S);
      load_lds16(a.kv + e + 8 * (lslot ^ k_swz<Sh::kCh>(r)),
                 buf + (16 * wave + Sh::kRPI * i) * Sh::kRowBytes);
      load_lds16(a.kv + e + a.g.kv + 8 * (lslot ^ v_swz<Sh::kCh>(r)),
                 buf + Sh::kTileBytes + (16 * wave + Sh::kRPI * i) * Sh::kRowBytes);
    }
  };

  // ---- per-lane LDS offsets.  K operand (S^T = K Q^T): row ks*32 + c,
  // chunk 2s + g.  V^T operand via the transpose read: in 16-lane group G,
  // lane r = 4m + a addresses key row key0 + m, dims 32t + 16*(G%2) + 4a.
  const int vm = (lane % 16) / 4, va4 = lane % 4, vG = lane / 16;
  auto v_off = [&](int t, int key0) {
    const int row = key0 + vm;
    const int dim = 32 * t + 16 * (vG % 2) + 4 * va4;
    return row * Sh::kRowBytes + 16 * ((dim / 8) ^ v_swz<Sh::kCh>(row)) + 2 * (dim % 8);
  };

  // lane-constant byte offsets inside a tile (the loop adds the buffer base)
  int k_off[Sh::kKS], v_lo[Sh::kDB], v_hi[Sh::kDB];
#pragma unroll
  for (int s8 = 0; s8 < Sh::kKS; ++s8) k_off[s8] = tile_off<D>(c, 2 * s8 + g);  // + ks * 32 rows below
#pragma unroll
  for (int t = 0; t < Sh::kDB; ++t) {  // key0 = 4g (+ ks*32 + 16*hf below) and key0 + 8
    v_lo[t] = v_off(t, 4 * g);
    v_hi[t] = v_off(t, 4 * g + 8);
  }
  // adding whole multiples of 16 rows keeps both swizzles: offsets step by
  // 16 rows
  constexpr int kRow16 = 16 * Sh::kRowBytes;

  floatx16 acc_o[Sh::kDB];
#pragma unroll
  for (int t = 0; t < Sh::kDB; ++t) acc_o[t] = floatx16{};
  float m_run = kPfNoMax, l_run = 0.f;  // running max of the unscaled scores
  const float scale = a.sm_scale * kLog2e;
  // smallest query position of this wave: tiles with every key at or below
  // it (and below L) need no mask
  const uint32_t wave_q0 = off + qt * kPfQueriesPerBlock + wave * kPfQueriesPerWave;

  // one 64-key tile from LDS buffer `tile_base`
  auto tile = [&](const lds_char* tile_base, uint32_t k0) {
    const lds_char* sK = tile_base;
    const lds_char* sV = tile_base + Sh::kTileBytes;
    // ---- S^T = K Q^T for two 32-key sub-tiles.  All K fragments of a
    // sub-tile are read before its MFMAs, and the second sub-tile's reads
    // go out before the first sub-tile's MFMAs, so no MFMA waits on a
    // just-issued LDS read.  At D = 256 (16 fragments per sub-tile) they go
    // in batches of 8, each read while the previous batch's MFMAs run, to
    // keep the registers of one wave per SIMD.
    floatx16 acc_s[2];
    if constexpr (Sh::kKS <= 8) {
      half8 kf0[Sh::kKS], kf1[Sh::kKS];
#pragma unroll
      for (int s8 = 0; s8 < Sh::kKS; ++s8)
        kf0[s8] = *reinterpret_cast<const __attribute__((address_space(3))) half8*>(sK + k_off[s8]);
#pragma unroll
      for (int s8 = 0; s8 < Sh::kKS; ++s8)
        kf1[s8] = *reinterpret_cast<const __attribute__((address_space(3))) half8*>(
            sK + k_off[s8] + 2 * kRow16);
      __builtin_amdgcn_sched_barrier(0);
      acc_s[0] = floatx16{};
#pragma unroll
      for (int s8 = 0; s8 < Sh::kKS; ++s8) acc_s[0] = mfma32(kf0[s8], qreg[s8], acc_s[0]);
      acc_s[1] = floatx16{};
#pragma unroll
      for (int s8 = 0; s8 < Sh::kKS; ++s8) acc_s[1] = mfma32(kf1[s8], qreg[s8], acc_s[1]);
    } else {
      constexpr int kB = 8;                      // fragments per batch
      constexpr int kNB = 2 * Sh::kKS / kB;      // batches per tile (both sub-tiles)
      auto kread = [&](int bt, half8 (&kf)[kB]) {  // batch bt: sub-tile bt / (kNB / 2)
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int s8 = (bt % (kNB / 2)) * kB + j;
          kf[j] = *reinterpret_cast<const __attribute__((address_space(3))) half8*>(
              sK + k_off[s8] + (bt / (kNB / 2)) * 2 * kRow16);
        }
      };
      half8 kfa[kB], kfb[kB];
      acc_s[0] = floatx16{};
      acc_s[1] = floatx16{};
      kread(0, kfa);
#pragma unroll
      for (int bt = 0; bt < kNB; bt += 2) {
        kread(bt + 1, kfb);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int s8 = (bt % (kNB / 2)) * kB + j;
          acc_s[bt / (kNB / 2)] = mfma32(kfa[j], qreg[s8], acc_s[bt / (kNB / 2)]);
        }
        if (bt + 2 < kNB) kread(bt + 2, kfa);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int s8 = ((bt + 1) % (kNB / 2)) * kB + j;
          acc_s[(bt + 1) / (kNB / 2)] = mfma32(kfb[j], qreg[s8], acc_s[(bt + 1) / (kNB / 2)]);
        }
      }
    }
    // ---- causal / length mask (only where a key can be past L or past
    // some query of the wave), running max of this query
    const bool full = k0 + kPfTileKeys <= L && (!a.causal || k0 + kPfTileKeys - 1u <= wave_q0);
    if (!full) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const uint32_t key = k0 + ks * 32 + crow(i, g);
          const bool ok = key < L && (!a.causal || key <= qpos);
          acc_s[ks][i] = ok ? acc_s[ks][i] : -INFINITY;
        }
    }
    float mt = acc_s[0][0];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 16; ++i) mt = fmaxf(mt, acc_s[ks][i]);
    mt = pair_max(mt);
    // Lazy rescaling: the reference max m_run moves only when some query's
    // tile max exceeds it by more than 2^8 in probability (the first tile
    // with a visible key always moves it).  Otherwise
    // probabilities stay <= 256, exact in fp16 relative terms, and the
    // final o = O / l divides both by the same reference.
    const bool move = __builtin_amdgcn_ballot_w64((mt - m_run) * scale > 8.f) != 0;
    const float m_new = move ? fmaxf(m_run, mt) : m_run;
    const float neg_m = -m_new * scale;
    float lt = 0.f;
    half8 pb[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        // 2^((s - m) * scale); a masked score (-inf) gives 0
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(acc_s[ks][i], scale, neg_m));
        lt += p;
        pb[ks][i / 8][i % 8] = (f16)p;
      }
    }
    lt = pair_sum(lt);
    if (move) {  // the reference moved for some query: rescale
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale);  // m_run = kPfNoMax: 0
      l_run = l_run * alpha;
#pragma unroll
      for (int t = 0; t < Sh::kDB; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc_o[t][i] *= alpha;
    }
    l_run = l_run + lt;
    m_run = m_new;

    // ---- O^T += V^T P^T.  B element j of half hf of sub-tile ks is the
    // probability of key ks*32 + 16*hf + 8*(j/4) + 4*g + j%4, so the A
    // operand of lane l is dim 32t + l%32 of keys key0 .. key0+3 (j < 4)
    // and key0+8 .. key0+11 (j >= 4), key0 = ks*32 + 16*hf + 4*g.
    // the 4 fragments (8 transpose reads) of dim block t+1 are read while
    // dim block t's MFMAs run
    auto vfrags = [&](int t, half8 (&vf)[4]) {
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {  // kk = 2*ks + hf
        const int rows = kk * kRow16;
        const half4 lo = __builtin_bit_cast(
            half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(sV + v_lo[t] + rows)));
        const half4 hi = __builtin_bit_cast(
            half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(sV + v_hi[t] + rows)));
        vf[kk] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
    };
    half8 vfa[4], vfb[4];
    vfrags(0, vfa);
#pragma unroll
    for (int t = 0; t < Sh::kDB; t += 2) {
      vfrags(t + 1, vfb);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc_o[t] = mfma32(vfa[kk], pb[kk / 2][kk % 2], acc_o[t]);
      if (t + 2 < Sh::kDB) vfrags(t + 2, vfa);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) acc_o[t + 1] = mfma32(vfb[kk], pb[kk / 2][kk % 2], acc_o[t + 1]);
    }
  };

  load_tile(s_buf0, page_of(t0));
  PageIds phys_next = page_of(t0 + 1u);
  // two tiles per trip: even tiles in buffer 0, odd tiles in buffer 1
  for (uint32_t it = t0; it < t1; it += 2) {
#pragma unroll
    for (uint32_t u = 0; u < 2; ++u) {
      const uint32_t ti = it + u;
      if (ti >= t1) break;  // uniform
      // tile ti has landed in LDS (this wave's loads: vmcnt; the others':
      // the barrier), and every wave is done with the other buffer
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (ti + 1 < t1) {  // in flight during this tile's MFMAs
        load_tile(u == 0u ? s_buf1 : s_buf0, phys_next);
        phys_next = page_of(ti + 2u);
      }
      if ((ti + 1u) * kPfTileKeys > L) {  // uniform: the tile holding the sequence's end
        // rows of keys at or past L hold whatever the cache held there (the
        // last page's unwritten slots, or the last page read again): their
        // probability is exactly 0, but 0 * NaN is NaN in the MFMA, so their
        // V rows are zeroed before any wave reads them
        char* vbuf = (u == 0u ? s_buf0 : s_buf1) + Sh::kTileBytes;
        const uint32_t first_dead = L - ti * kPfTileKeys;  // < kPfTileKeys
        for (uint32_t i = first_dead * (Sh::kRowBytes / 16u) + threadIdx.x;
             i < (uint32_t)kPfTileKeys * (Sh::kRowBytes / 16u); i += kPfThreads)
          reinterpret_cast<uint4*>(vbuf)[i] = uint4{0u, 0u, 0u, 0u};
        __syncthreads();
      }
      if (ti * kPfTileKeys < wave_kend)  // wave-uniform: skip tiles above this wave's queries
        tile((const lds_char*)(u == 0u ? s_buf0 : s_buf1), ti * kPfTileKeys);
    }
  }

  if (nchunks > 1u) {  // ---- a chunk's partial, for prefill_merge_kernel
    float* part = a.partial + (size_t)item * pf_partial_floats(D);
    float4* po = reinterpret_cast<float4*>(part) + wave * kPfQueriesPerWave + c;
#pragma unroll
    for (int j = 0; j < Sh::kDB * 4; ++j) {
      const floatx16& x = acc_o[j / 4];
      const int i0 = 4 * (j % 4);
      // dims 32 (j / 4) + crow(i0, g) .. + 3
      po[(8 * (j / 4) + 2 * (j % 4) + g) * kPfQueriesPerBlock] =
          float4{x[i0], x[i0 + 1], x[i0 + 2], x[i0 + 3]};
    }
    if (g == 0) {
      float* pm = part + kPfQueriesPerBlock * D + wave * kPfQueriesPerWave + c;
      pm[0] = m_run;
      pm[kPfQueriesPerBlock] = l_run;
    }
    return;
  }

  // ---- o = O / l: lane holds its query's dims t*32 + crow(i, g)
  if (!q_live) return;
  const float inv_l = 1.f / l_run;
  f16* orow = a.o + ((size_t)q * a.Hq + h) * D;
#pragma unroll
  for (int t = 0; t < Sh::kDB; ++t) {
#pragma unroll
    for (int i0 = 0; i0 < 16; i0 += 4) {
      half4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (f16)(acc_o[t][i0 + r] * inv_l);
      *reinterpret_cast<half4*>(orow + t * 32 + crow(i0, g)) = v;
    }
  }
}

// Joins the chunks' partials of split query tiles: one workgroup per (query
// head, query tile, 32 queries); thread t takes query t % 32 and D / 8 dims.
template <int D>
__global__ __launch_bounds__(kPfThreads) void prefill_merge_kernel(PrefillArgs a) {
  const uint32_t nqt = (a.Lq + kPfQueriesPerBlock - 1) / kPfQueriesPerBlock;
  const uint32_t sub = blockIdx.x % 4u, x = blockIdx.x / 4u;
  const uint32_t h = x / nqt, qt = x % nqt;
  const uint32_t nchunks = pf_chunks(pf_tiles(a.L, a.Lq, a.causal, qt), a.chunk_rcp);
  const uint32_t row = sub * 32u + threadIdx.x % 32u, j0 = threadIdx.x / 32u;
  const uint32_t q = qt * kPfQueriesPerBlock + row;
  if (nchunks == 1u || q >= a.Lq) return;
  uint32_t item = h * a.per_head;  // the tile's first
  for (uint32_t y = nqt - 1u; y > qt; --y)
    item += pf_chunks(pf_tiles(a.L, a.Lq, a.causal, y), a.chunk_rcp);
  const float scale = a.sm_scale * kLog2e;
  const float* part = a.partial + (size_t)item * pf_partial_floats(D);
  float m = kPfNoMax, l = 0.f;
  for (uint32_t s = 0; s < nchunks; ++s)
    m = fmaxf(m, part[s * pf_partial_floats(D) + kPfQueriesPerBlock * D + row]);
  constexpr int kV = D / 32;  // 4-dim vectors per thread
  float4 acc[kV] = {};
  for (uint32_t s = 0; s < nchunks; ++s) {
    const float* p = part + s * pf_partial_floats(D);
    const float* pm = p + kPfQueriesPerBlock * D + row;
    const float w = __builtin_amdgcn_exp2f((pm[0] - m) * scale);
    l += pm[kPfQueriesPerBlock] * w;
#pragma unroll
    for (int v = 0; v < kV; ++v) {
      const float4 y = reinterpret_cast<const float4*>(p)[(kV * j0 + v) * kPfQueriesPerBlock + row];
      acc[v].x += y.x * w;
      acc[v].y += y.y * w;
      acc[v].z += y.z * w;
      acc[v].w += y.w * w;
    }
  }
  const float inv_l = 1.f / l;
  f16* orow = a.o + ((size_t)q * a.Hq + h) * D + 4 * kV * j0;
#pragma unroll
  for (int v = 0; v < kV; ++v)
    *reinterpret_cast<half4*>(orow + 4 * v) =
        half4{(f16)(acc[v].x * inv_l), (f16)(acc[v].y * inv_l), (f16)(acc[v].z * inv_l),
              (f16)(acc[v].w * inv_l)};
}

// The calls that are split, and into chunks of how many key tiles.  One item
// (128 queries of a head) walks its key tiles one after the other, so few
// items over a long context leave most CUs idle: 500 queries x 32 heads over
// 16384 keys are 128 items of 256 tiles, 334 us (396 TFLOP/s); as 512 items
// of 64 tiles, 151 us (878).  100 queries over 8192 keys: 165 -> 39 us; 300
// over 16000 at 16 heads of dim 256: 641 -> 155.  A split costs its partials
// (fp32, written and read once) and a second launch, so a call whose items
// fill the chip is faster whole (3001 x 3001, 32 heads: 90 us, in chunks of
// 32 tiles 110; 8192 x 8192: 585, in chunks of 64 659).  Measured step times decide: a CU
// with k items resident takes t[k] us per tile of each (d64 0.92, 1.25, 1.8;
// d128 1.3, 2.05; d256 2.56), the partials move at 4 TB/s, the joining launch
// takes 5 us.  Against measured calls of 16 to 1536 items the estimate is
// within 15%, and picks the best split or one within 10% of it.
PrefillPlan prefill_plan(uint32_t L, uint32_t Lq, uint32_t causal, uint32_t Hq,
                         uint32_t head_dim) {
  constexpr uint32_t kCus = 256u;
  constexpr float kStep[3][3] = {{0.92f, 1.25f, 1.8f}, {1.3f, 2.05f, 2.05f}, {2.56f, 2.56f, 2.56f}};
  const float* step = kStep[head_dim == 64u ? 0 : head_dim == 128u ? 1 : 2];
  const uint32_t occ = head_dim == 64u ? 3u : head_dim == 128u ? 2u : 1u;  // items per CU
  const uint32_t slots = kCus * occ;
  PrefillPlan best{};
  const uint32_t nqt = (Lq + kPfQueriesPerBlock - 1) / kPfQueriesPerBlock;
  const uint32_t nmax = pf_tiles(L, Lq, causal, nqt - 1u);
  if ((uint64_t)nqt * Hq >= 2u * slots || nmax < 8u || nmax > 65535u) return best;
  float best_us = 0.f;
  // chunks of 2 / s of the longest item's tiles
  for (uint32_t s : {2u, 3u, 4u, 6u, 8u, 10u, 12u, 16u, 20u, 24u, 32u, 40u, 48u, 64u, 96u, 128u}) {
    const uint32_t chunk = (2u * nmax + s - 1u) / s;
    if (chunk < 4u) break;
    const uint32_t rcp = (uint32_t)((1ull << 32) / chunk) + 1u;
    uint64_t items = 0u, partials = 0u, tiles = 0u;
    for (uint32_t qt = 0; qt < nqt; ++qt) {
      const uint32_t t = pf_tiles(L, Lq, causal, qt), c = pf_chunks(t, rcp);
      items += c;
      tiles += t;
      partials += c > 1u ? c : 0u;
    }
    const uint32_t per_head = (uint32_t)items;
    items *= Hq;
    if (s > 2u && items > 4u * slots) break;
    // all resident at once: the longest; else the CUs' rate, and half of the
    // longest at the end
    float us = items <= slots
                   ? (float)chunk * step[(items + kCus - 1u) / kCus - 1u]
                   : (float)(tiles * Hq) * step[occ - 1u] / (float)slots + 0.5f * chunk * step[0];
    if (s > 2u)
      us += 5.f + (float)(partials * Hq * pf_partial_floats((int)head_dim)) * 8.f / 4e6f;
    if (s == 2u) {
      best_us = 0.95f * us;  // a split has to be worth its launch
    } else if (us < best_us) {
      best_us = us;
      best.chunk_rcp = rcp;
      best.per_head = per_head;
      best.workspace_bytes = items * pf_partial_floats((int)head_dim) * sizeof(float);
    }
  }
  return best;
}

template <int D>
static hipError_t launch_pf(const PrefillArgs& a, uint32_t page_size, hipStream_t s) {
  const uint32_t nqt = (a.Lq + kPfQueriesPerBlock - 1) / kPfQueriesPerBlock;
  const uint32_t items = (a.chunk_rcp != 0u ? a.per_head : nqt) * a.Hq;
  const dim3 grid(items), block(kPfThreads);
  switch (page_size) {
    case 1: hipLaunchKernelGGL((prefill_kernel<1, D>), grid, block, 0, s, a); break;
    case 2: hipLaunchKernelGGL((prefill_kernel<2, D>), grid, block, 0, s, a); break;
    case 4: hipLaunchKernelGGL((prefill_kernel<4, D>), grid, block, 0, s, a); break;
    case 8: hipLaunchKernelGGL((prefill_kernel<8, D>), grid, block, 0, s, a); break;
    case 16: hipLaunchKernelGGL((prefill_kernel<16, D>), grid, block, 0, s, a); break;
    case 32: hipLaunchKernelGGL((prefill_kernel<32, D>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  if (hipError_t e = hipGetLastError(); e != hipSuccess || a.chunk_rcp == 0u) return e;
  hipLaunchKernelGGL(prefill_merge_kernel<D>, dim3(a.Hq * nqt * 4u), block, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_prefill(const PrefillArgs& args, uint32_t page_size, uint32_t head_dim,
                          void* workspace, size_t workspace_bytes, hipStream_t s) {
  PrefillArgs a = args;
  const PrefillPlan p = prefill_plan(a.L, a.Lq, a.causal, a.Hq, head_dim);
  if (p.chunk_rcp != 0u && workspace != nullptr && workspace_bytes >= p.workspace_bytes) {
    a.chunk_rcp = p.chunk_rcp;
    a.per_head = p.per_head;
    a.partial = static_cast<float*>(workspace);
  }
  switch (head_dim) {
    case 64: return launch_pf<64>(a, page_size, s);
    case 128: return launch_pf<128>(a, page_size, s);
    case 256: return launch_pf<256>(a, page_size, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace aoakv
