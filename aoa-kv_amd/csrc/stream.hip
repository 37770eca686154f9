// Decode attention as a stream over a list of pages (gfx950): every page of a
// sequence (dense decode, any shape), and the selected pages of the head dims
// and page sizes that decode.hip's kernels do not take (64, 128, 256 with
// pages of 1..32 tokens).
//
// Replaces BatchDecodeWithPagedKVCacheKernel + VariableLengthMergeStates
// (decode_attn.cuh:482-688, 1004-1044) for those calls; logits fp16(q.k), then
// fp16(. / sqrt(d)) (quest_attention.py:265-268), softmax and sums in fp32.
//
// A D-dim fp16 vector is held by D / 8 lanes (a lane group), 8 dims each, so a
// wave-wide 16-byte load takes 512 / D tokens.  A workgroup's tokens are cut
// into batches of 4 such loads of K and of V; wave w takes batches w, w + 4,
// ..., with kAhead of them in flight.  Each lane group keeps an online softmax
// of its own tokens: nothing crosses groups until the end.
//
// Bound by HBM for long lists, else by the chain of a workgroup's round trips
// (page table, ids, K/V, partials, merge).  Two layers, with a workgroup per 8
// pages and now: 16384 tokens x 32 heads 121 -> 91 us (5.9 TB/s; a plain read
// of 1 GiB runs at 6.05), 1000 tokens 14.7 -> 14.3, 32 / 8 heads at 24000 117
// -> 60, head dim 64 at 20000 151 -> 61, 256 (16 heads) at 8000 92 -> 54; one
// selected layer of 128 pages x 16 heads of dim 256 (decode alone) 16.2 ->
// 13.3.
#include "kernels.hpp"
#include "topk.hpp"

namespace aoakv {
namespace {

constexpr uint32_t kStThreads = kThreads;
constexpr uint32_t kStWaves = kStThreads / kWave;
constexpr uint32_t kStListPages = 512;  // pages whose ids are staged at a time
constexpr uint32_t kStSelfWorkgroups = 1024;  // 4 per CU (36 KB of LDS each)
constexpr int kU = 4;                   // loads of K (and of V) per batch
constexpr float kNoMax = -1e30f;        // running max before the first token: finite

// x of the quad's lane U in all four lanes (DPP quad_perm)
template <int U>
__device__ inline float quad_bcast(float x) {
  return dpp<U * 0x55>(x);
}

// the values of lanes l and l ^ 16 (or l ^ 32), combined in both
__device__ inline float swap16_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline float swap16_max(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float swap32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline float swap32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
constexpr int kRowRor8 = 0x128;  // lane l of a row reads lane l ^ 8

// sum over the D / 8 lanes of a group, in every lane of it
template <int D>
__device__ inline float lanes_sum(float x) {
  x = x + dpp<kQuadSwap1>(x);
  x = x + dpp<kQuadSwap2>(x);
  x = x + dpp<kRowHalfMirror>(x);
  if constexpr (D >= 128) x = x + dpp<kRowMirror>(x);
  if constexpr (D == 256) x = swap16_sum(x);
  return x;
}
// sum / max over the groups of a wave (lanes of the same dims)
template <int D>
__device__ inline float groups_sum(float x) {
  if constexpr (D == 64) x = x + dpp<kRowRor8>(x);
  if constexpr (D <= 128) x = swap16_sum(x);
  return swap32_sum(x);
}
template <int D>
__device__ inline float groups_max(float x) {
  if constexpr (D == 64) x = fmaxf(x, dpp<kRowRor8>(x));
  if constexpr (D <= 128) x = swap16_max(x);
  return swap32_max(x);
}

// fp16(x / sqrt(D)) of an fp16 value, as an fp32 division rounds it (sqrt(64)
// and sqrt(256) are powers of two: the product is exact)
template <int D>
__device__ inline float logit_f16(float x) {
  if constexpr (D == 128) return (float)r16(div_sqrt_head_dim_f16(x));
  return (float)r16(x * (D == 64 ? 0.125f : 0.0625f));
}

// Which pages a kernel attends: all (dense), the call's selection rows, or (for
// a layer) the selection it makes itself from the scores.
enum Pages { kAll, kListed, kSelf };

// A call and its split.
struct StreamArgs : DecodeArgs {
  uint32_t page_rcp;  // the factor that divides by the page size (0: pages of one token)
  // kAll: the chunks the call's pages are cut into (per head, over all its
  // sequences), below and from long_pages pages of all sequences on, and the
  // factors that divide by these numbers (0: by one)
  uint32_t batch;
  uint32_t split, split_rcp, long_split, long_rcp;
  uint32_t long_pages;
  // kSelf: the rows the selection is made from (complete), and where it goes
  const float* scores;
  uint32_t score_stride;
  uint32_t select_flags;
  int32_t* sel_out;
};

// ceil(n / d) for 1 <= n, rcp = floor(2^32 / d) + 1 (0: d = 1); from n * d = 2^32
// on it may be more
__device__ inline uint32_t div_up(uint32_t n, uint32_t rcp) {
  return rcp == 0u ? n : (uint32_t)(((uint64_t)(n - 1u) * rcp) >> 32) + 1u;
}

// Where a workgroup of a dense call works: sequence b's chunk `chunk` of `per`
// pages, with b's place in the page table.
struct Place {
  uint32_t b, chunk, per, pbeg, pages, last_len;
};

// Pages per chunk of a call of `total` pages.  (The bound matters only for more
// than 64 sequences with page tables past it, which `total` counts whole.)
__device__ inline uint32_t chunk_pages(const StreamArgs& a, uint32_t total) {
  const bool is_long =
      total >= a.long_pages && (uint64_t)a.max_pages * a.batch >= a.long_pages;
  const uint32_t per = is_long ? div_up(total, a.long_rcp) : div_up(total, a.split_rcp);
  return per < kGenChunkPages ? kGenChunkPages : per;
}

// The item-th chunk of the call: sequences in order, each one's chunks in order.
// No pages: there is none.
__device__ inline Place find_item(const StreamArgs& a, uint32_t item) {
  const uint32_t lane = __lane_id();
  if (a.batch == 1u) {
    const uint32_t beg = (uint32_t)a.kv_indptr[0], n = (uint32_t)a.kv_indptr[1] - beg;
    const uint32_t len = (uint32_t)a.kv_last_page_len[0];
    const uint32_t P = n < a.max_pages ? n : a.max_pages;
    return Place{0u, item, chunk_pages(a, P != 0u ? P : 1u), beg, n, len};
  }
  auto of = [](uint32_t x, uint32_t j) {
    return (uint32_t)__builtin_amdgcn_readlane((int)x, (int)j);
  };
  if (a.batch <= (uint32_t)kWave) {  // a lane per sequence, their chunks counted
    const uint32_t i = lane < a.batch ? lane : a.batch - 1u;
    const uint32_t beg = (uint32_t)a.kv_indptr[i], end = (uint32_t)a.kv_indptr[i + 1u];
    const uint32_t len = (uint32_t)a.kv_last_page_len[i];
    uint32_t P = end - beg < a.max_pages ? end - beg : a.max_pages;
    if (lane >= a.batch) P = 0u;
    const uint32_t total = of(wave_incl_scan(P), kWave - 1u);
    if (total == 0u) return Place{};
    const uint32_t per = chunk_pages(a, total);
    const uint32_t n = (P + per - 1u) / per;
    const uint32_t incl = wave_incl_scan(n);
    const uint64_t past = __builtin_amdgcn_ballot_w64(item < incl);
    if (past == 0u) return Place{};
    const uint32_t j = (uint32_t)__builtin_ctzll(past);
    return Place{j, item - (of(incl, j) - of(n, j)), per, of(beg, j), of(end, j) - of(beg, j),
                 of(len, j)};
  }
  // more: sequence b's items start at floor(pages before it / per) + b, room
  // for its chunks whatever the lengths, so only its own place is needed; 64
  // sequences are tried at a time
  const uint32_t first = (uint32_t)a.kv_indptr[0];
  const uint32_t total = (uint32_t)a.kv_indptr[a.batch] - first;
  if (total == 0u) return Place{};
  const uint32_t per = chunk_pages(a, total);
  uint32_t lo = 0u, n = a.batch;
  for (;;) {
    const uint32_t stride = (n + kWave - 1u) / kWave;
    const bool in = lane * stride < n;
    const uint32_t i = in ? lo + lane * stride : lo;
    const uint32_t beg = (uint32_t)a.kv_indptr[i], end = (uint32_t)a.kv_indptr[i + 1u];
    const uint32_t len = (uint32_t)a.kv_last_page_len[i];
    const uint32_t off = (beg - first) / per + i;
    const uint64_t le = __builtin_amdgcn_ballot_w64(in && off <= item);
    if (le == 0u) return Place{};  // malformed page table
    const uint32_t j = 63u - (uint32_t)__builtin_clzll(le);
    if (stride == 1u)
      return Place{lo + j, item - of(off, j), per, of(beg, j), of(end, j) - of(beg, j),
                   of(len, j)};
    const uint32_t left = n - j * stride;
    n = left < stride ? left : stride;
    lo += j * stride;
  }
}

// One workgroup per (chunk of the page list, G query heads of a kv head).  G:
// 1, or the whole GQA group, whose K/V is then loaded once.
// kAll: the pages of all sequences are cut into as many chunks per head as
// fill the chip (each sequence into chunks of that many pages, at least
// kGenChunkPages), a count made here from the page table: what a call gives
// depends on its sequences alone, not on the page count it was sized for, nor on
// G.  Selected pages are cut into chunks of kGenChunkPages.  The last chunk of a
// sequence to arrive at the head's counter merges the partials in chunk
// order and clears them.
// NT: no other workgroup reads these pages: non-temporal loads.
// kSelf: there are no selection rows yet; every workgroup of a kv head runs the
// head's top-k on the scores the previous launch wrote, takes its chunk's
// entries and writes them out (as decode.hip's two-launch layer).
template <int D, int G, bool NT, Pages PAGES>
__global__ __launch_bounds__(kStThreads) void stream_decode_kernel(StreamArgs a) {
  constexpr bool SELF = PAGES == kSelf;
  constexpr uint32_t N = D / 8, GPW = kWave / N;  // lanes per group, groups per wave
  constexpr uint32_t kBatch = kU * GPW;           // tokens
  // two batches in flight; three were slower at every shape measured (16
  // sequences' d64 layer 43.0 against 38.5 us, pages of 8 127.8 against
  // 115.1 per 4 layers).  Registers, and waves per SIMD: selected pages 128
  // and 4, every page 140 and 3; groups of 2, 4 and 8 heads 146, 188 and 256
  // (with 16 spilled to AGPRs), and 3, 2 and 1
  constexpr int kAhead = 2;
  constexpr uint32_t kStride = (uint32_t)D + 4u;  // partial: o[D], m, l, pad
  struct Shared {
    float o[kStWaves][G][D];
    float ml[kStWaves][G][2];
  };
  struct Empty {};
  __shared__ uint32_t s_page[SELF ? kGenChunkPages : kStListPages];
  __shared__ union {
    typename std::conditional<SELF, TopkShared, Empty>::type tk;
    Shared d;
  } sm;
  __shared__ uint32_t s_last;
  auto& s_o = sm.d.o;
  auto& s_ml = sm.d.ml;
  const uint32_t lane = __lane_id();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t l = lane % N, v = lane / N;
  const bool quest = PAGES != kAll && (a.flags & kFlagQuestKernel) != 0u;
  const uint32_t S = a.S;
  uint32_t chunk, hq0, hkv, per = kGenChunkPages;
  Place at;
  if constexpr (PAGES == kAll) {
    // heads fastest, so the workgroups in flight read whole pages
    // (neighbouring heads are neighbours in HBM)
    uint32_t item = blockIdx.y + gridDim.y * blockIdx.z;
    if constexpr (G > 1 || NT) {
      hkv = blockIdx.x;
      hq0 = hkv * G;
    } else {
      // the heads of a GQA group on one XCD (workgroup x runs on x % 8), which
      // reads their K/V from HBM once: 32 / 8 heads, two layers at 2000 tokens
      // 23.7 -> 15.2 us
      const uint32_t group = a.Hq / a.Hkv, x = blockIdx.x + a.Hq * item;
      const uint32_t u = x / (kXcds * group) * kXcds + x % kXcds;
      hkv = u % a.Hkv;
      hq0 = hkv * group + x / kXcds % group;
      item = u / a.Hkv;
    }
    at = find_item(a, item);
    per = at.per;
    chunk = at.chunk;
  } else {
    chunk = blockIdx.x;
    hq0 = blockIdx.y * G;
    hkv = hq0 / (a.Hq / a.Hkv);
    const uint32_t b = blockIdx.z, beg = (uint32_t)a.kv_indptr[b];
    at = Place{b, chunk, per, beg, (uint32_t)a.kv_indptr[b + 1u] - beg,
               (uint32_t)a.kv_last_page_len[b]};
  }
  const uint32_t b = at.b, pbeg = at.pbeg, lpl = at.last_len;
  const uint32_t P = at.pages < a.max_pages ? at.pages : a.max_pages;
  if (P != at.pages && chunk == 0u && threadIdx.x == 0u) flag_error(a.error, kErrTruncated);
  if (P == 0u || lpl == 0u || lpl > S) return;  // malformed page table
  uint32_t npages = P, budget = 0u;
  if constexpr (PAGES != kAll) {
    budget = a.token_budgets ? (uint32_t)a.token_budgets[b] : a.token_budget;
    npages = num_selected_pages((P - 1u) * S + lpl, budget, S, P, quest ? kFlagQuestKernel : 0u);
    const uint32_t row_cap = a.sel_stride + (quest ? 1u : 0u);
    if (npages > row_cap) npages = row_cap;
  }
  // the workspace holds max_chunks chunks of 8 pages per head
  if (npages > a.max_chunks * kGenChunkPages) {
    npages = a.max_chunks * kGenChunkPages;
    if (chunk == 0u && threadIdx.x == 0u) flag_error(a.error, kErrTruncated);
  }
  if (chunk * per >= npages) return;  // uniform per block
  const uint32_t nsel = quest ? npages - 1u : npages;
  const int32_t* sel_row =
      PAGES == kListed ? a.sel + ((size_t)b * a.Hkv + hkv) * a.sel_stride : nullptr;
  const uint32_t last_phys = (uint32_t)a.kv_indices[pbeg + P - 1u];
  const size_t bh0 = (size_t)b * a.Hq + hq0;
  H8 q[G];
#pragma unroll
  for (int g = 0; g < G; ++g) q[g] = ld16(a.q + (bh0 + g) * D + l * kVec);

  float m[G], lsum[G], o[G][kVec];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = kNoMax;
    lsum[g] = 0.f;
#pragma unroll
    for (int j = 0; j < kVec; ++j) o[g][j] = 0.f;
  }
  const uint32_t i0 = chunk * per, i1 = i0 + per < npages ? i0 + per : npages;
  if constexpr (SELF) {
    static_assert(G == 1, "a query head per workgroup");
    // candidates: every scored page (quest_kernel: but the last); the
    // selection's first nout entries, in page order
    const uint32_t row = P < a.score_stride + (quest ? 1u : 0u) ? P
                                                               : a.score_stride + (quest ? 1u : 0u);
    const uint32_t cand = quest ? row - 1u : row;
    uint32_t k = num_selected_pages((row - 1u) * S + lpl, budget, S, row, a.select_flags);
    if (quest) k -= 1u;
    if (k > a.sel_stride) k = a.sel_stride;
    const int32_t* ids = a.kv_indices + pbeg;
    const bool pick = k != 0u && k < cand;
    if (pick)
      topk_staged<true>(a.scores + ((size_t)b * a.Hkv + hkv) * a.score_stride, cand, k,
                        (a.select_flags & kFlagFixed) != 0u, ids, nullptr, sm.tk);
    const uint32_t nout = pick ? k : (k == 0u ? 0u : cand);
    // this chunk's entries, here and in the selection output (whose end the
    // last chunk writes); an entry the top-k did not yield means the shapes
    // disagree
    int32_t* out = a.sel_out + ((size_t)b * a.Hkv + hkv) * a.sel_stride;
    auto entry = [&](uint32_t i) { return pick ? sm.tk.key[i] : (uint32_t)ids[i]; };
    if (threadIdx.x < per) {  // per = kGenChunkPages
      const uint32_t i = i0 + threadIdx.x;
      if (i < nsel && i >= nout) flag_error(a.error, kErrTruncated);
      s_page[threadIdx.x] = i >= nsel ? last_phys : i < nout ? entry(i) : last_phys;
    }
    const uint32_t o_end = i1 == npages || i0 + per > nout ? nout : i0 + per;
    for (uint32_t i = i0 + threadIdx.x; i < o_end; i += kStThreads) out[i] = (int32_t)entry(i);
    __syncthreads();  // (the top-k's memory is the softmax's from here)
  }
  for (uint32_t ib = i0; ib < i1; ib += kStListPages) {
    // ---- the ids of up to kStListPages pages of the list
    const uint32_t np = i1 - ib < kStListPages ? i1 - ib : kStListPages;
    if constexpr (!SELF) {
      if (ib != i0) __syncthreads();  // the ids before were read
      for (uint32_t i = threadIdx.x; i < np; i += kStThreads)
        s_page[i] = PAGES == kAll    ? (uint32_t)a.kv_indices[pbeg + ib + i]
                    : ib + i < nsel ? (uint32_t)sel_row[ib + i]
                                    : last_phys;
      __syncthreads();
    }
    const uint32_t T = np * S;  // token slots
    const uint32_t nb = (T + kBatch - 1u) / kBatch;
    // loads of batch i (clamped: a slot past the end reads the last one), and
    // which of this lane's group's tokens exist
    H8 kk[kAhead][kU], vv[kAhead][kU];
    uint32_t ok[kAhead];
    auto load = [&](uint32_t i, int s) {
      ok[s] = 0u;
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t t = i * kBatch + (uint32_t)u * GPW + v;
        const uint32_t tc = t < T ? t : T - 1u;
        // tc / S (exact: tc < 2^14, S <= 32)
        const uint32_t e = a.page_rcp != 0u ? (uint32_t)(((uint64_t)tc * a.page_rcp) >> 32) : tc;
        const uint32_t slot = tc - e * S, phys = s_page[e];
        const f16* kp = a.kv + elem_off(a.g, phys, 0, hkv, slot) + l * kVec;
        const f16* vp = kp + a.g.kv;
        kk[s][u] = NT ? ld16_nt(kp) : ld16(kp);
        vv[s][u] = NT ? ld16_nt(vp) : ld16(vp);
        if (t < T && (phys != last_phys || slot < lpl)) ok[s] |= 1u << u;
      }
    };
    auto attend = [&](int s) {
      // slots without a token hold whatever the cache held: 0 * NaN is NaN
      if (__builtin_amdgcn_ballot_w64(ok[s] != (1u << kU) - 1u) != 0u) {
#pragma unroll
        for (int u = 0; u < kU; ++u)
          if (!((ok[s] >> u) & 1u)) vv[s][u] = H8{};
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float x[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          float acc = 0.f;
#pragma unroll
          for (int p = 0; p < kVec / 2; ++p)
            acc = __builtin_amdgcn_fdot2(half_pair(q[g], p), half_pair(kk[s][u], p), acc, false);
          x[u] = lanes_sum<D>(acc);
        }
        // lane l % 4 rounds and exponentiates token l % 4
        const uint32_t um = lane % 4u;
        float pick = x[0];
#pragma unroll
        for (int u = 1; u < kU; ++u) pick = um == (uint32_t)u ? x[u] : pick;
        float xm = logit_f16<D>((float)r16(pick));
        xm = (ok[s] >> um) & 1u ? xm : -INFINITY;
        float mt = fmaxf(xm, dpp<kQuadSwap1>(xm));
        mt = fmaxf(mt, dpp<kQuadSwap2>(mt));
        const float mn = fmaxf(m[g], mt);
        const float c = __expf(m[g] - mn), p = __expf(xm - mn);
        m[g] = mn;
        float ps = p + dpp<kQuadSwap1>(p);
        ps = ps + dpp<kQuadSwap2>(ps);
        lsum[g] = lsum[g] * c + ps;
        const float pv[kU] = {quad_bcast<0>(p), quad_bcast<1>(p), quad_bcast<2>(p),
                              quad_bcast<3>(p)};
#pragma unroll
        for (int j = 0; j < kVec; ++j) {
          float acc = o[g][j] * c;
#pragma unroll
          for (int u = 0; u < kU; ++u)
            acc = __builtin_fmaf(pv[u], (float)vv[s][u].v[j], acc);
          o[g][j] = acc;
        }
      }
    };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) load(wave + (uint32_t)s * kStWaves, s);
    uint32_t i = wave;
    if constexpr (PAGES == kAll && G == 1) {
      // no load past the list's end, for which a short list would wait at its
      // own (two layers of 32 heads, 500 tokens 13.3 -> 11.2 us); three waves per
      // SIMD instead of four, no slower on long lists
      static_assert(kAhead == 2, "the loop's exits");
      for (; i < nb; i += 2u * kStWaves) {
        attend(0);
        if (i + 2u * kStWaves >= nb) {
          if (i + kStWaves < nb) attend(1);
          break;
        }
        load(i + 2u * kStWaves, 0);
        attend(1);
        if (i + 3u * kStWaves >= nb) {
          attend(0);
          break;
        }
        load(i + 3u * kStWaves, 1);
      }
    } else {
      for (; i < nb; i += kAhead * kStWaves) {
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
          if (i + (uint32_t)s * kStWaves >= nb) break;  // wave-uniform
          attend(s);
          load(i + (uint32_t)(s + kAhead) * kStWaves, s);
        }
      }
    }
  }
  const uint32_t nch = (npages + per - 1u) / per;

  // ---- the wave's groups, then the workgroup's waves
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float mw = groups_max<D>(m[g]);
    const float w = __expf(m[g] - mw);
    const float lw = groups_sum<D>(lsum[g] * w);
    float ow[kVec];
#pragma unroll
    for (int j = 0; j < kVec; ++j) ow[j] = groups_sum<D>(o[g][j] * w);
    if (v == 0u) {
#pragma unroll
      for (int j = 0; j < kVec; ++j) s_o[wave][g][l * kVec + j] = ow[j];
      if (l == 0u) {
        s_ml[wave][g][0] = mw;
        s_ml[wave][g][1] = lw;
      }
    }
  }
  __syncthreads();
  for (uint32_t x = threadIdx.x; x < (uint32_t)(G * D); x += kStThreads) {
    const uint32_t g = x / D, d = x % D;
    float M = s_ml[0][g][0];
#pragma unroll
    for (uint32_t w = 1; w < kStWaves; ++w) M = fmaxf(M, s_ml[w][g][0]);
    float acc = 0.f, Ls = 0.f;
#pragma unroll
    for (uint32_t w = 0; w < kStWaves; ++w) {
      const float sc = __expf(s_ml[w][g][0] - M);
      acc = acc + sc * s_o[w][g][d];
      Ls = Ls + sc * s_ml[w][g][1];
    }
    if (nch == 1u) {
      a.o[(bh0 + g) * D + d] = r16(acc / Ls);
    } else {
      float* part = a.partial + ((bh0 + g) * a.max_chunks + chunk) * kStride;
      st_agent(part + d, acc);
      if (d == 0u) {
        st_agent(part + D, M);
        st_agent(part + D + 1u, Ls);
      }
    }
  }
  if (nch == 1u) return;
  if (!arrive_last(&a.counters[bh0 * kCounterStride], nch, &s_last)) return;
  // the last chunk to arrive merges: in groups of kC chunks, every load of a
  // group issued before any is used, folded in chunk order
  auto merge = [&](auto group) {
    constexpr uint32_t kC = decltype(group)::value;
    for (uint32_t x = threadIdx.x; x < (uint32_t)(G * D); x += kStThreads) {
      const uint32_t g = x / D, d = x % D;
      const float* base = a.partial + (bh0 + g) * a.max_chunks * kStride;
      float M = kNoMax, Ls = 0.f, acc = 0.f;
      for (uint32_t c0 = 0; c0 < nch; c0 += kC) {
        float mc[kC], lc[kC], oc[kC];
#pragma unroll
        for (uint32_t u = 0; u < kC; ++u) {
          const float* part = base + (c0 + u < nch ? c0 + u : nch - 1u) * kStride;
          mc[u] = ld_agent(part + D);
          lc[u] = ld_agent(part + D + 1u);
          oc[u] = ld_agent(part + d);
        }
        float Mn = M;
#pragma unroll
        for (uint32_t u = 0; u < kC; ++u) Mn = fmaxf(Mn, mc[u]);
        const float keep = __expf(M - Mn);
        Ls = Ls * keep;
        acc = acc * keep;
#pragma unroll
        for (uint32_t u = 0; u < kC; ++u) {
          const float w = c0 + u < nch ? __expf(mc[u] - Mn) : 0.f;
          Ls = Ls + w * lc[u];
          acc = acc + w * oc[u];
        }
        M = Mn;
      }
      a.o[(bh0 + g) * D + d] = r16(acc / Ls);
    }
  };
  if (nch <= 8u) merge(std::integral_constant<uint32_t, 8u>{});
  else merge(std::integral_constant<uint32_t, 16u>{});
  __syncthreads();  // every thread has read the partials
  for (uint32_t g = 0; g < (uint32_t)G; ++g) {
    uint32_t* pw = reinterpret_cast<uint32_t*>(a.partial + (bh0 + g) * a.max_chunks * kStride);
    for (uint32_t i = threadIdx.x; i < nch * kStride; i += kStThreads) st_agent_u32(pw + i, 0u);
  }
}

template <int D>
hipError_t launch_d(const StreamArgs& a, uint32_t G, dim3 grid, hipStream_t s) {
  const dim3 block(kStThreads);
  const bool mha = a.Hq == a.Hkv;
#define AOAKV_ST(G_, NT_, PAGES_) \
  hipLaunchKernelGGL((stream_decode_kernel<D, G_, NT_, PAGES_>), grid, block, 0, s, a)
  if (a.scores != nullptr) {
    if (mha) AOAKV_ST(1, true, kSelf);
    else AOAKV_ST(1, false, kSelf);
  } else if (a.sel != nullptr) {
    if (mha) AOAKV_ST(1, true, kListed);
    else AOAKV_ST(1, false, kListed);
  } else {
    // K/V of one reader: no GQA group, or a whole group per workgroup
    switch (G) {
      case 1:
        if (mha) AOAKV_ST(1, true, kAll);
        else AOAKV_ST(1, false, kAll);
        break;
      case 2: AOAKV_ST(2, true, kAll); break;
      case 4: AOAKV_ST(4, true, kAll); break;
      case 8: AOAKV_ST(8, true, kAll); break;
      default: return hipErrorInvalidValue;
    }
  }
#undef AOAKV_ST
  return hipGetLastError();
}

}  // namespace

// Dense calls are cut into 512 workgroups (2 per CU, and no fewer than 8 pages
// each), which stream 32 heads of 16384 tokens at 5.9 TB/s; more of them cost
// more partials (1024: 25.5 -> 32 us at 3000 tokens, 92 -> 96 at 16384).  The
// heads of a GQA group read their K/V through one XCD's L2, at 12 to 17 TB/s
// whatever the group.  A workgroup for the whole group reads it at HBM's 6
// TB/s, but takes its heads one after the other (one workgroup per CU, 256 in
// all), 11 to 34 us before that shows.  So a call is long, and read by
// groups, from 256 MiB of L2 reads on (more where fewer than 8 kv heads make
// more and shorter chunks).  Two layers, a head and a group per workgroup:
// 32 / 8 heads at 5000 tokens 21 and 33 us, 12000 36 and 43, 24000 60 and 59,
// 65536 153 and 114; 32 / 16 at 10000 37 and 40, 20000 72 and 66; 32 / 4 at
// 40000 88 and 106, 65536 133 and 130; head dim 64, 32 / 8 at 30000 42 and 42;
// 256, 16 / 8 at 20000 74 and 74.
// The chunks come from the tokens there are.  Made from the call's bound and
// its batch, one sequence of 65536 tokens among 15 of 1000 (32 heads) took 1770
// us, now 423, and among 31 (32 / 8 heads) 2545, now 161.
// Pages of all sequences from which a call is long:
static uint32_t dense_long_pages(const DecodeArgs& a, uint32_t head_dim) {
  if (a.Hq == a.Hkv) return ~0u;
  const uint64_t bytes = (uint64_t)(256u << 20) * (a.Hkv < 8u ? 8u / a.Hkv : 1u);
  const uint64_t page = 4ull * head_dim * a.Hq * a.S;
  return (uint32_t)((bytes + page - 1u) / page);
}

// The layers whose decode selects for itself: rows the top-k stages, and no
// more workgroups than are resident at once (each repeats its head's top-k,
// which spares the launch of its own, 5.9 us).  Four layers: head dim 256,
// 20011 tokens, 256 workgroups 118 -> 108 us; 64 x 32 heads, 32768 tokens, 512
// workgroups 82 -> 75; with 2048 workgroups (pages of 8, budget 4096) 187 and
// selecting for themselves 222.
bool stream_selects(const DecodeArgs& a, uint32_t batch, uint32_t max_pages) {
  return max_pages <= kStageMaxPages && (uint64_t)a.max_chunks * a.Hq * batch <= kStSelfWorkgroups;
}

hipError_t launch_stream_decode(const DecodeArgs& args, uint32_t batch, uint32_t head_dim,
                                hipStream_t s, const EstimateArgs* self) {
  StreamArgs a{};
  static_cast<DecodeArgs&>(a) = args;
  if (self != nullptr) {
    a.scores = self->scores;
    a.score_stride = self->score_stride;
    a.select_flags = self->flags;
    a.sel_out = self->sel;
  }
  auto rcp = [](uint32_t d) { return d > 1u ? (uint32_t)((1ull << 32) / d) + 1u : 0u; };
  a.page_rcp = rcp(a.S);
  uint32_t G = 1u;
  dim3 grid(a.max_chunks, a.Hq, batch);
  if (a.sel == nullptr) {
    a.batch = batch;
    a.long_pages = dense_long_pages(a, head_dim);
    a.split = 512u / a.Hq > 1u ? 512u / a.Hq : 1u;
    // (every sequence of a few may end in a chunk of its own: still 512 in all)
    if (batch > 1u && 4u * batch <= a.split) a.split -= batch;
    a.long_split = 256u / a.Hkv > 1u ? 256u / a.Hkv : 1u;
    a.split_rcp = rcp(a.split);
    a.long_rcp = rcp(a.long_split);
    const bool may_be_long = (uint64_t)a.max_pages * batch >= a.long_pages;
    if (may_be_long || a.heads_per_item > 1u) G = a.Hq / a.Hkv;
    const uint32_t split = may_be_long && a.long_split > a.split ? a.long_split : a.split;
    // a sequence takes at most one item more than its share of the chunks
    uint32_t items = batch > 1u ? split + batch : split < a.max_chunks ? split : a.max_chunks;
    // (per-head workgroups of a group: whole sets of one per XCD)
    if (G != a.Hq / a.Hkv)
      while (items * a.Hkv % kXcds != 0u) ++items;
    constexpr uint32_t kRows = 32768u;
    grid = dim3(a.Hq / G, items < kRows ? items : kRows, (items + kRows - 1u) / kRows);
  }
  switch (head_dim) {
    case 64: return launch_d<64>(a, G, grid, s);
    case 128: return launch_d<128>(a, G, grid, s);
    case 256: return launch_d<256>(a, G, grid, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace aoakv
