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
// (page table, ids, K/V, partials, merge).  Two layers, before (a workgroup
// per 8 pages) and now: 16384 tokens x 32 heads 121 -> 98 us (5.5 TB/s; a
// plain read of 1 GiB runs at 6.05), 32 / 8 heads at 24000 118 -> 62, head
// dim 64 at 20000 153 -> 63, 256 (16 heads) at 8000 95 -> 58; one selected
// layer of 128 pages x 16 heads of dim 256 (decode alone) 16.2 -> 13.3.
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

// A call, and its split: chunks the grid holds per head (<= max_chunks), and
// the factor that divides by the page size (0: pages of one token).
struct StreamArgs : DecodeArgs {
  uint32_t grid_chunks;
  uint32_t page_rcp;
  // SELF: the rows the selection is made from (complete), and where it goes
  const float* scores;
  uint32_t score_stride;
  uint32_t select_flags;
  int32_t* sel_out;
};

// One workgroup per (chunk of the page list, G query heads of a kv head,
// sequence).  G: 1, or the whole GQA group, whose K/V is then loaded once.
// The list is split over a.grid_chunks chunks (of at least kGenChunkPages
// pages); the last to arrive at the head's counter merges their partials in
// chunk order and clears them.
// NT: no other workgroup reads these pages: non-temporal loads.
// SELF: there are no selection rows yet; every workgroup of a kv head runs the
// head's top-k on the scores the previous launch wrote, takes its chunk's
// entries and writes them out (as decode.hip's two-launch layer).
template <int D, int G, bool NT, bool SELF = false>
__global__ __launch_bounds__(kStThreads) void stream_decode_kernel(StreamArgs a) {
  constexpr uint32_t N = D / 8, GPW = kWave / N;  // lanes per group, groups per wave
  constexpr uint32_t kBatch = kU * GPW;           // tokens
  // two batches in flight: 128 registers, four waves per SIMD; three (168)
  // were slower at every shape measured (16 sequences' d64 layer 43.0
  // against 38.5 us, pages of 8 127.8 against 115.1 per 4 layers)
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
  // dense: heads fastest, so the workgroups in flight read whole pages
  // (neighbouring heads are neighbours in HBM); else chunks fastest
  const uint32_t chunk = a.sel == nullptr ? blockIdx.y : blockIdx.x;
  const uint32_t hq0 = (a.sel == nullptr ? blockIdx.x : blockIdx.y) * G, b = blockIdx.z;
  const uint32_t hkv = hq0 / (a.Hq / a.Hkv);
  const bool quest = (a.flags & kFlagQuestKernel) != 0u;
  const uint32_t S = a.S;
  const uint32_t pbeg = (uint32_t)a.kv_indptr[b];
  const uint32_t P_table = (uint32_t)a.kv_indptr[b + 1] - pbeg;
  const uint32_t P = P_table < a.max_pages ? P_table : a.max_pages;
  if (P != P_table && chunk == 0u && threadIdx.x == 0u) flag_error(a.error, kErrTruncated);
  const uint32_t lpl = (uint32_t)a.kv_last_page_len[b];
  if (P == 0u || lpl == 0u || lpl > S) return;  // malformed page table
  const uint32_t budget = a.token_budgets ? (uint32_t)a.token_budgets[b] : a.token_budget;
  uint32_t npages = P;
  if (a.sel != nullptr) {
    npages = num_selected_pages((P - 1u) * S + lpl, budget, S, P, quest ? kFlagQuestKernel : 0u);
    const uint32_t row_cap = a.sel_stride + (quest ? 1u : 0u);
    if (npages > row_cap) npages = row_cap;
  }
  // the workspace holds max_chunks chunks of 8 pages per head
  if (npages > a.max_chunks * kGenChunkPages) {
    npages = a.max_chunks * kGenChunkPages;
    if (chunk == 0u && threadIdx.x == 0u) flag_error(a.error, kErrTruncated);
  }
  uint32_t per = (npages + a.grid_chunks - 1u) / a.grid_chunks;  // pages per chunk
  if (per < kGenChunkPages) per = kGenChunkPages;
  const uint32_t nch = (npages + per - 1u) / per;
  if (chunk >= nch) return;  // uniform per block
  const uint32_t nsel = (quest && a.sel != nullptr) ? npages - 1u : npages;
  const int32_t* sel_row = a.sel ? a.sel + ((size_t)b * a.Hkv + hkv) * a.sel_stride : nullptr;
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
    const uint32_t o_end = chunk == nch - 1u || i0 + per > nout ? nout : i0 + per;
    for (uint32_t i = i0 + threadIdx.x; i < o_end; i += kStThreads) out[i] = (int32_t)entry(i);
    __syncthreads();  // (the top-k's memory is the softmax's from here)
  }
  for (uint32_t ib = i0; ib < i1; ib += kStListPages) {
    // ---- the ids of up to kStListPages pages of the list
    const uint32_t np = i1 - ib < kStListPages ? i1 - ib : kStListPages;
    if constexpr (!SELF) {
      if (ib != i0) __syncthreads();  // the ids before were read
      for (uint32_t i = threadIdx.x; i < np; i += kStThreads)
        s_page[i] = sel_row == nullptr ? (uint32_t)a.kv_indices[pbeg + ib + i]
                    : ib + i < nsel    ? (uint32_t)sel_row[ib + i]
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
#pragma unroll
    for (int s = 0; s < kAhead; ++s) load(wave + (uint32_t)s * kStWaves, s);
    for (uint32_t i = wave; i < nb; i += kAhead * kStWaves) {
#pragma unroll
      for (int s = 0; s < kAhead; ++s) {
        if (i + (uint32_t)s * kStWaves >= nb) break;  // wave-uniform
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
        load(i + (uint32_t)(s + kAhead) * kStWaves, s);
      }
    }
  }

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
  // the last chunk to arrive merges: in groups of 16 chunks, every load of a
  // group issued before any is used, folded in chunk order
  for (uint32_t x = threadIdx.x; x < (uint32_t)(G * D); x += kStThreads) {
    const uint32_t g = x / D, d = x % D;
    const float* base = a.partial + (bh0 + g) * a.max_chunks * kStride;
    float M = kNoMax, Ls = 0.f, acc = 0.f;
    for (uint32_t c0 = 0; c0 < nch; c0 += 16u) {
      float mc[16], lc[16], oc[16];
#pragma unroll
      for (uint32_t u = 0; u < 16u; ++u) {
        const float* part = base + (c0 + u < nch ? c0 + u : nch - 1u) * kStride;
        mc[u] = ld_agent(part + D);
        lc[u] = ld_agent(part + D + 1u);
        oc[u] = ld_agent(part + d);
      }
      float Mn = M;
#pragma unroll
      for (uint32_t u = 0; u < 16u; ++u) Mn = fmaxf(Mn, mc[u]);
      const float keep = __expf(M - Mn);
      Ls = Ls * keep;
      acc = acc * keep;
#pragma unroll
      for (uint32_t u = 0; u < 16u; ++u) {
        const float w = c0 + u < nch ? __expf(mc[u] - Mn) : 0.f;
        Ls = Ls + w * lc[u];
        acc = acc + w * oc[u];
      }
      M = Mn;
    }
    a.o[(bh0 + g) * D + d] = r16(acc / Ls);
  }
  __syncthreads();  // every thread has read the partials
  for (uint32_t g = 0; g < (uint32_t)G; ++g) {
    uint32_t* pw = reinterpret_cast<uint32_t*>(a.partial + (bh0 + g) * a.max_chunks * kStride);
    for (uint32_t i = threadIdx.x; i < nch * kStride; i += kStThreads) st_agent_u32(pw + i, 0u);
  }
}

template <int D>
hipError_t launch_d(const StreamArgs& a, uint32_t G, dim3 grid, hipStream_t s) {
  const dim3 block(kStThreads);
  if (a.scores != nullptr) {
    if (a.Hq == a.Hkv)
      hipLaunchKernelGGL((stream_decode_kernel<D, 1, true, true>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((stream_decode_kernel<D, 1, false, true>), grid, block, 0, s, a);
    return hipGetLastError();
  }
  // K/V of one reader: no GQA group, or a whole group per workgroup
  if (G > 1u || a.Hq == a.Hkv) {
    switch (G) {
      case 1: hipLaunchKernelGGL((stream_decode_kernel<D, 1, true>), grid, block, 0, s, a); break;
      case 2: hipLaunchKernelGGL((stream_decode_kernel<D, 2, true>), grid, block, 0, s, a); break;
      case 4: hipLaunchKernelGGL((stream_decode_kernel<D, 4, true>), grid, block, 0, s, a); break;
      case 8: hipLaunchKernelGGL((stream_decode_kernel<D, 8, true>), grid, block, 0, s, a); break;
      default: return hipErrorInvalidValue;
    }
  } else {
    hipLaunchKernelGGL((stream_decode_kernel<D, 1, false>), grid, block, 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace

// Query heads per workgroup of a dense call: the whole GQA group, whose K/V is
// then read once, when that still gives the chip 512 workgroups of 8 pages;
// below, a head each (their partials are merged in parallel).  32 / 8 heads,
// two layers: 12000 tokens 82 us a head each (decode.hip's kernel), 45
// grouped; 5000 tokens 27 and 35.
static uint32_t dense_group(const DecodeArgs& a, uint32_t batch) {
  return (uint64_t)a.max_chunks * a.Hkv * batch >= 512u ? a.Hq / a.Hkv : 1u;
}

// The dense calls of the tuned shape that stream: without GQA from 1024
// workgroups of 8 pages on.  Two layers of 32 heads: 3000 tokens (752) 28.0
// us streamed, 27.9 by decode.hip's kernel, 5000 (1280) 38.6 and 44.6, 16384
// 98 and 122 (5.5 and 4.4 TB/s), 24000 137 and 181.
bool stream_dense(const DecodeArgs& a, uint32_t batch) {
  return dense_group(a, batch) > 1u ||
         (a.Hq == a.Hkv && (uint64_t)a.max_chunks * a.Hq * batch >= 1024u);
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
  a.page_rcp = a.S > 1u ? (uint32_t)((1ull << 32) / a.S) + 1u : 0u;
  const bool dense = a.sel == nullptr;
  const uint32_t G = dense ? dense_group(a, batch) : 1u, heads = a.Hq / G;
  a.grid_chunks = a.max_chunks;
  if (dense) {
    // a workgroup per CU (two without GQA), each a long stream: the partials
    // and their merge shrink with the chunks (32 / 8 heads, 24000 tokens: 89
    // us with 768 workgroups, 72 with 512, 62 with 256)
    const uint64_t want = (G > 1u ? 256u : 512u) / ((uint64_t)heads * batch);
    a.grid_chunks = want < 1u ? 1u : want < a.max_chunks ? (uint32_t)want : a.max_chunks;
  }
  const dim3 grid = dense ? dim3(heads, a.grid_chunks, batch) : dim3(a.grid_chunks, heads, batch);
  switch (head_dim) {
    case 64: return launch_d<64>(a, G, grid, s);
    case 128: return launch_d<128>(a, G, grid, s);
    case 256: return launch_d<256>(a, G, grid, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace aoakv
