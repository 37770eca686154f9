// Per-head top-k selection by one 256-thread workgroup (gfx950): the radix
// select over order keys, and the handoff words it may read. Shared by
// decode.hip and stream.hip. Functions note phase times with TL where the
// including file defines it (decode.hip's profiling build).
#pragma once

#include <type_traits>

#include "kernels.hpp"

#ifndef TL
#define TL(ev) \
  do {         \
  } while (0)
#endif

namespace aoakv {

constexpr int kThreads = 256;

// ======================================================================
// block-wide helpers (256 threads = 4 waves)
// ======================================================================

// Inclusive prefix sum over the 64 lanes of a wave: DPP row_shr steps inside
// each 16-lane row, then the totals of the rows below through readlane.
__device__ inline uint32_t wave_incl_scan(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
  const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
  const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
  const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
  const uint32_t row = __lane_id() / kLanesPerRow;
  return v + (row > 0u ? r0 : 0u) + (row > 1u ? r1 : 0u) + (row > 2u ? r2 : 0u);
}

// min / max of a uint32 over the wave (DPP inside rows, readlane across)
template <bool MAX>
__device__ inline uint32_t wave_reduce_u32(uint32_t v) {
  auto op = [](uint32_t x, uint32_t y) { return MAX ? (x > y ? x : y) : (x < y ? x : y); };
  v = op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kQuadSwap1, 0xf, 0xf, true));
  v = op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kQuadSwap2, 0xf, 0xf, true));
  v = op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kRowHalfMirror, 0xf, 0xf, true));
  v = op(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kRowMirror, 0xf, 0xf, true));
  const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
  const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
  const uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
  return op(op(a, b), op(c, d));
}

// ======================================================================
// top-k selection for one (sequence, kv head), one 256-thread block
// ======================================================================

// Bound on polls of a handoff word before a wait gives up (it then sets the
// error flag and goes on with stand-in data, so every wave still exits).
constexpr uint32_t kSpinLimit = 1u << 18;

// Sleeps until `ps` picoseconds of wall time have passed since t0, a reading
// of s_memrealtime: a 100 MHz counter of its own, so the wait does not scale
// with the core clock (1.3-2.6 GHz with load and temperature).  The counter
// is read a few times per wait, not polled: between reads the wave sleeps
// for a bound on the time left (one `s_sleep 1` lasts 64 core cycles, at
// most 5 ticks at 1.3 GHz), so each read finds at most the time left and
// the reads converge on the end.  Polling a clock (s_memrealtime or
// s_memtime) in every waiting wave slowed the whole layer by 0.4-1 us.
__device__ inline void sleep_until(uint64_t t0, uint64_t ps) {
  const uint64_t end = t0 + ps / 10000u;
  for (uint64_t now = __builtin_amdgcn_s_memrealtime(); now < end;
       now = __builtin_amdgcn_s_memrealtime()) {
    for (uint32_t n = (uint32_t)((end - now) / 5u) + 1u; n != 0u; --n) __builtin_amdgcn_s_sleep(1);
  }
}

// Polls an agent-coherent handoff word until it is written (non-zero);
// returns the value - 1, or 0 after kSpinLimit polls with *error set.
__device__ inline uint32_t wait_word(const uint32_t* p, uint32_t* error) {
  uint32_t v, it = 0u;
  while ((v = ld_agent_u32(p)) == 0u) {
    __builtin_amdgcn_s_sleep(1);
    if (++it > kSpinLimit) {
      flag_error(error, kErrWait);
      return 0u;
    }
  }
  return v - 1u;
}

// A float as a handoff word: bits + 1, never 0 (the all-ones NaN pattern,
// which arithmetic never produces, is stored as the canonical NaN).
__device__ inline uint32_t to_word(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  return (u == 0xFFFFFFFFu ? 0x7FC00000u : u) + 1u;
}

// Pages whose scores and page ids are staged in LDS (16 per thread); longer
// rows are read straight from global memory.
constexpr uint32_t kStageMaxPages = 16u * kThreads;

struct TopkShared {
  alignas(16) uint32_t hist[3][kThreads];  // radix histograms, rotating over 3 buffers
  alignas(16) uint32_t key[kStageMaxPages];  // staged order keys, then the output
  int32_t id[kStageMaxPages];                // staged page ids
  uint32_t red[8];
  uint32_t s4[4];
};

struct RadixResult {
  uint32_t hmask;    // bits of (key - kmin) that decide the bucket (~0u << hi)
  uint32_t thr;      // the bucket of the k-th key: (key - kmin) & hmask == thr
  uint32_t kr;       // keys still to take from that bucket
  bool take_bucket;  // the bucket is taken whole (else: hi == 0, equal keys)
};

// Finds the bucket holding the kr-th largest free key (free_mask bit j: key[j]
// takes part) by a radix select over key - kmin, 8-bit digits from the top
// set bit of kmax - kmin down (one head's scores span a narrow range, so the
// first digit already spreads the keys); it stops as soon as the bucket of
// the kr-th key is taken whole.  One barrier per pass: the histogram is
// scanned by every wave, and buffers rotate over three, so the buffer cleared
// in pass i was last read in pass i-2, before the barrier of pass i-1.
// hist[0] must be zero on entry.
template <int KPT, typename Mask>
__device__ __forceinline__ RadixResult radix_select(const uint32_t (&rel)[KPT], Mask free_mask,
                                                    uint32_t range, uint32_t kr, TopkShared& sh) {
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = __lane_id();
  uint32_t prefix = 0u;
  int hi = range == 0u ? 0 : 32 - __builtin_clz(range);
  bool take_bucket = false;
  uint32_t buf = 0;
  while (hi > 0) {
    const int w = hi < 8 ? hi : 8;
    const int sft = hi - w;
    const uint32_t hmask = hi >= 32 ? 0u : ~0u << hi;
    // every key adds 1 to its bin if it takes part, else 0: no per-key
    // branch (keys that do not take part land on scattered bins)
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      const bool part = ((free_mask >> j) & (Mask)1) && ((rel[j] ^ prefix) & hmask) == 0u;
      atomicAdd(&sh.hist[buf][(rel[j] >> sft) & ((1u << w) - 1u)], part ? 1u : 0u);
    }
    const uint32_t nxt = buf == 2u ? 0u : buf + 1u;
    sh.hist[nxt][tid] = 0u;
    __syncthreads();
    // lane L holds bins 255-4L .. 252-4L (descending)
    const uint4 h = *reinterpret_cast<const uint4*>(&sh.hist[buf][252u - 4u * lane]);
    const uint32_t s4 = (h.x + h.y) + (h.z + h.w);
    const uint32_t incl = wave_incl_scan(s4);
    const uint32_t excl = incl - s4;
    const bool hit = excl < kr && kr <= incl;  // exactly one lane
    const uint32_t c0 = excl + h.w, c1 = c0 + h.z, c2 = c1 + h.y;
    const uint32_t j = kr <= c0 ? 0u : kr <= c1 ? 1u : kr <= c2 ? 2u : 3u;
    const uint32_t above_l = j == 0u ? excl : j == 1u ? c0 : j == 2u ? c1 : c2;
    const uint32_t count_l = j == 0u ? h.w : j == 1u ? h.z : j == 2u ? h.y : h.x;
    const uint32_t src = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(hit));
    const uint32_t jj = (uint32_t)__builtin_amdgcn_readlane((int)j, (int)src);
    const uint32_t above = (uint32_t)__builtin_amdgcn_readlane((int)above_l, (int)src);
    const uint32_t count = (uint32_t)__builtin_amdgcn_readlane((int)count_l, (int)src);
    prefix |= (255u - 4u * src - jj) << sft;
    kr -= above;
    hi = sft;
    buf = nxt;
    TL(kTlPass1);
    if (count == kr) {  // every key of the bucket is selected
      take_bucket = true;
      break;
    }
  }
  const uint32_t hmask = hi >= 32 ? 0u : ~0u << hi;
  return RadixResult{hmask, prefix & hmask, kr, take_bucket};
}

// Selects k of P pages from fp32 `scores` (filter_util.py:373-380): with
// `fixed`, pages 0 and P-1 always; the rest by descending score, ties to the
// lower page index.  Writes kv_ids[page] of the selected pages to out[] in
// ascending page order (agent-coherent stores).
//
// Thread t owns pages [t*kpt, t*kpt + kpt) as register keys, kpt <= KPT and
// P <= 256 * KPT.  With KPT <= 16 scores and ids are first copied to LDS
// with coalesced loads and the output is compacted in LDS and stored
// coalesced; with KPT = 64 (rows up to 16384 pages) keys are read and the
// output written per thread.
//
// SELF (one-launch layer): every decode workgroup of the kv head (of each
// query head of its group) runs this same selection on the same score words.
// The words are only read (a merging workgroup clears them), their
// wait starts with one sentinel word per scoring chunk, and the output stays
// in sh.key[0, k) for the caller (nothing is stored).
template <int KPT, bool SELF = false>
__device__ __forceinline__ void topk_block(const float* __restrict__ scores, uint32_t P, uint32_t k,
                                           bool fixed, const int32_t* __restrict__ kv_ids,
                                           int32_t* __restrict__ out, TopkShared& sh,
                                           uint32_t* hout, uint32_t hstride, uint32_t hcopies,
                                           uint32_t* hwords = nullptr, uint32_t* error = nullptr) {
  // page i of the output, also as id + 1 into the hcopies handoff rows
  auto put = [&](uint32_t i, int32_t id) {
    st_agent_i32(out + i, id);
    if (hout != nullptr)
      for (uint32_t c = 0; c < hcopies; ++c) st_agent_u32(hout + c * hstride + i, (uint32_t)id + 1u);
  };
  constexpr bool kStaged = KPT <= 16;
  static_assert(KPT % 4 == 0 && (KPT <= 16 || KPT == 64), "keys per thread");
  using Mask = typename std::conditional<(KPT > 32), uint64_t, uint32_t>::type;
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = __lane_id();
  const uint32_t wave = tid / kWave;
  if (!SELF && hwords != nullptr && (k == 0u || k >= P)) {
    // the scores are not needed, but their handoff words must be consumed
    for (uint32_t i = tid; i < P; i += kThreads) {
      uint32_t it = 0u;
      for (; ld_agent_u32(hwords + i) == 0u && it < kSpinLimit; ++it) __builtin_amdgcn_s_sleep(1);
      // a word written after this gave up would be left set
      if (it >= kSpinLimit) flag_error(error, kErrWait);
      st_agent_u32(hwords + i, 0u);
    }
  }
  if (k == 0u) return;  // (quest_kernel convention with a budget of one page)
  if (k >= P) {  // everything selected
    for (uint32_t i = tid; i < P; i += kThreads) put(i, kv_ids[i]);
    return;
  }
  // kpt rounded up to 4 so staged keys are read as 16-byte LDS vectors
  const uint32_t kpt = kStaged ? (((P + kThreads - 1) / kThreads + 3u) & ~3u)
                               : (P + kThreads - 1) / kThreads;
  const uint32_t i0 = tid * kpt;
  const uint32_t nforced = fixed ? (P == 1u ? 1u : 2u) : 0u;
  auto is_free = [&](uint32_t i) { return !(fixed && (i == 0u || i == P - 1u)); };
  sh.hist[0][tid] = 0u;

  uint32_t key[KPT];
  uint32_t kmin = 0xFFFFFFFFu, kmax = 0u;
  if constexpr (kStaged) {
    // coalesced copy: all loads issued before any is used
    float sv[KPT];
    int32_t iv[KPT];
    if (hwords == nullptr) {
#pragma unroll
      for (int m = 0; m < KPT; ++m) {  // unconditional loads of clamped indices
        uint32_t i = tid + (uint32_t)m * kThreads;
        i = i < P ? i : P - 1u;
        sv[m] = ld_agent(scores + i);
        iv[m] = kv_ids[i];
      }
#ifdef AOAKV_TIMELINE
      // (noted once the loads have returned)
      if (__builtin_bit_cast(uint32_t, sv[KPT - 1]) != 0x7FBADBADu) TL(kTlRowLoaded);
#endif
    } else {
      // page ids first, then this thread's score words, polled until the
      // scoring items have written them, then cleared for the next launch
      // (only the thread owning a word clears it; clamped reads of another
      // thread's word are not used)
      uint32_t w[KPT];
#pragma unroll
      for (int m = 0; m < KPT; ++m) {
        uint32_t i = tid + (uint32_t)m * kThreads;
        i = i < P ? i : P - 1u;
        iv[m] = kv_ids[i];
      }
      if constexpr (SELF) {
        // first the head's last score word alone, so that the workgroups
        // waiting for a head poll one cache line each, not the whole row
        // (512 workgroups polling every word, or one word per scoring chunk,
        // cost 1.2 or 0.2 us per layer in memory traffic at config 2)
        if (wave == 0u) {
          const uint32_t* sw = hwords + (P - 1u);
          uint32_t it = 0u;
          for (; it < kSpinLimit; ++it) {
            if (__builtin_amdgcn_ballot_w64(ld_agent_u32(sw) == 0u) == 0u) break;
            __builtin_amdgcn_s_sleep(1);
          }
          if (it >= kSpinLimit && lane == 0u) flag_error(error, kErrWait);
        }
        __syncthreads();
        TL(kTlScoresSeen);
      }
      auto load_words = [&]() {
#pragma unroll
        for (int m = 0; m < KPT; ++m) {
          uint32_t i = tid + (uint32_t)m * kThreads;
          i = i < P ? i : P - 1u;
          w[m] = ld_agent_u32(hwords + i);
        }
      };
      auto missing = [&]() {
        bool z = false;
#pragma unroll
        for (int m = 0; m < KPT; ++m) z |= tid + (uint32_t)m * kThreads < P && w[m] == 0u;
        return z;
      };
      load_words();
      uint32_t it = 0u;
      for (; missing(); ++it) {
        if (it >= kSpinLimit) break;  // stand-in scores
        __builtin_amdgcn_s_sleep(1);
        load_words();
      }
      // a wait that gave up is flagged here, outside the poll loop (an atomic
      // inside it made this loop's code 0.4 us per layer slower): words
      // written after it are left set, and the next launch must not run on
      // them
      if (it >= kSpinLimit) flag_error(error, kErrWait);
      TL(kTlRowLoaded);
#pragma unroll
      for (int m = 0; m < KPT; ++m) {
        const uint32_t i = tid + (uint32_t)m * kThreads;
        if (!SELF && i < P) st_agent_u32(hwords + i, 0u);
        sv[m] = __builtin_bit_cast(float, w[m] - 1u);
      }
    }
    // no per-key branch: entries past P (inside the staging arrays, which
    // hold 256 * KPT) are written too and never read as valid keys
#pragma unroll
    for (int m = 0; m < KPT; ++m) {
      const uint32_t i = tid + (uint32_t)m * kThreads;
      const uint32_t kk = order_key(sv[m]);
      sh.key[i] = kk;
      sh.id[i] = iv[m];
      const bool use = i < P && is_free(i);
      kmin = use && kk < kmin ? kk : kmin;
      kmax = use && kk > kmax ? kk : kmax;
    }
  } else {
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      const uint32_t i = i0 + j;
      const bool valid = (uint32_t)j < kpt && i < P;
      key[j] = order_key(ld_agent(scores + (valid ? i : P - 1u)));
      if (valid && is_free(i)) {
        kmin = key[j] < kmin ? key[j] : kmin;
        kmax = key[j] > kmax ? key[j] : kmax;
      }
    }
  }
  kmin = wave_reduce_u32<false>(kmin);
  kmax = wave_reduce_u32<true>(kmax);
  if (lane == 0) {
    sh.red[wave] = kmin;
    sh.red[4 + wave] = kmax;
  }
  __syncthreads();
  TL(kTlStaged);
  kmin = sh.red[0];
  kmax = sh.red[4];
#pragma unroll
  for (int w4 = 1; w4 < 4; ++w4) {
    kmin = sh.red[w4] < kmin ? sh.red[w4] : kmin;
    kmax = sh.red[4 + w4] > kmax ? sh.red[4 + w4] : kmax;
  }
  if constexpr (kStaged) {
#pragma unroll
    for (int c = 0; c < KPT / 4; ++c) {
      const uint4 v = *reinterpret_cast<const uint4*>(&sh.key[i0 + 4u * c]);
      key[4 * c + 0] = v.x;
      key[4 * c + 1] = v.y;
      key[4 * c + 2] = v.z;
      key[4 * c + 3] = v.w;
    }
  }
  Mask free_mask = 0, valid_mask = 0;  // bit j: page i0+j exists / is not forced
  uint32_t rel[KPT];
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const uint32_t i = i0 + j;
    rel[j] = key[j] - kmin;
    const bool v = (uint32_t)j < kpt && i < P;
    valid_mask |= (Mask)v << j;
    free_mask |= (Mask)(v && is_free(i)) << j;
  }
  // >= 1: k == 0 returned above, and with fixed forcing k >= 3 > nforced
  const RadixResult rr = radix_select<KPT, Mask>(rel, free_mask, kmax - kmin, k - nforced, sh);
  TL(kTlSelected);

  // selection classes at the final resolution:
  //   above:  forced, or (rel & hmask) > thr  -- selected
  //   bucket: (rel & hmask) == thr            -- rr.kr of them selected: all when
  //           take_bucket, else (equal keys) the lowest pages first
  Mask above_m = 0, eq_m = 0;
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const bool v = (valid_mask >> j) & 1u, f = (free_mask >> j) & 1u;
    const uint32_t r = rel[j] & rr.hmask;
    above_m |= (Mask)(v && (!f || r > rr.thr)) << j;
    eq_m |= (Mask)(v && f && r == rr.thr) << j;
  }
  // one scan of (pages above, bucket pages) packed in 16-bit halves gives the
  // output position: selected pages before mine = above before + min(bucket
  // pages before, kr)
  const uint32_t na = (uint32_t)__builtin_popcountll((uint64_t)above_m);
  const uint32_t ne = (uint32_t)__builtin_popcountll((uint64_t)eq_m);
  const uint32_t packed = na | (ne << 16);
  // this thread's page ids, read before the barrier below (after it, the id
  // array takes the discarded writes of the compaction)
  int32_t myid[kStaged ? KPT : 1];
  if constexpr (kStaged) {
#pragma unroll
    for (int c = 0; c < KPT / 4; ++c) {
      const int4 v = *reinterpret_cast<const int4*>(&sh.id[i0 + 4u * c]);
      myid[4 * c + 0] = v.x;
      myid[4 * c + 1] = v.y;
      myid[4 * c + 2] = v.z;
      myid[4 * c + 3] = v.w;
    }
  }
  const uint32_t incl = wave_incl_scan(packed);
  if (lane == kWave - 1) sh.s4[wave] = incl;
  __syncthreads();
  uint32_t before = incl - packed;
#pragma unroll
  for (uint32_t w4 = 0; w4 < 4; ++w4) before += w4 < wave ? sh.s4[w4] : 0u;
  const uint32_t eq_before = before >> 16;
  uint32_t pos = (before & 0xFFFFu) + (eq_before < rr.kr ? eq_before : rr.kr);
  uint32_t eq_rank = eq_before;
  if constexpr (kStaged) {
    // every key and id read from LDS finished before the barrier above, so
    // sh.key takes the compacted output and sh.id[tid] the discarded writes
    // (every key writes somewhere: no per-key branch)
    uint32_t* s_out = sh.key;
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      const bool eq = (eq_m >> j) & 1u;
      const bool take = ((above_m >> j) & 1u) || (eq && (rr.take_bucket || eq_rank < rr.kr));
      eq_rank += eq ? 1u : 0u;
      uint32_t* dst = take ? &s_out[pos] : reinterpret_cast<uint32_t*>(&sh.id[tid]);
      *dst = (uint32_t)myid[j];
      pos += take ? 1u : 0u;
    }
    __syncthreads();
    if (!SELF)
      for (uint32_t i = tid; i < k; i += kThreads) put(i, (int32_t)s_out[i]);
    TL(kTlOutput);
  } else {
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      bool take = (above_m >> j) & 1u;
      if ((eq_m >> j) & 1u) take = rr.take_bucket || eq_rank++ < rr.kr;
      if (take) put(pos++, kv_ids[i0 + j]);
    }
  }
}

// top-k of a row of P <= kStageMaxPages pages with the fewest keys per thread
template <bool SELF = false>
__device__ __forceinline__ void topk_staged(const float* __restrict__ scores, uint32_t P, uint32_t k,
                                            bool fixed, const int32_t* __restrict__ kv_ids,
                                            int32_t* __restrict__ out, TopkShared& sh,
                                            uint32_t* hout = nullptr, uint32_t hstride = 0u,
                                            uint32_t hcopies = 0u, uint32_t* hwords = nullptr,
                                            uint32_t* error = nullptr) {
  if (P <= 4u * kThreads)
    topk_block<4, SELF>(scores, P, k, fixed, kv_ids, out, sh, hout, hstride, hcopies, hwords,
                          error);
  else if (P <= 8u * kThreads)
    topk_block<8, SELF>(scores, P, k, fixed, kv_ids, out, sh, hout, hstride, hcopies, hwords,
                          error);
  else
    topk_block<16, SELF>(scores, P, k, fixed, kv_ids, out, sh, hout, hstride, hcopies, hwords,
                          error);
}

}  // namespace aoakv
