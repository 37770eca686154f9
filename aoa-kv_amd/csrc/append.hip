// Paged KV append with AOA-KV metadata maintenance (gfx950).
//
// Replaces the reference's AppendPagedKVCachePrefillKernel and
// AppendPagedKVCacheDecodeKernel (kernels/aoa_kv/kernels/include/decode/
// decode_page.cuh:398-692) with the simulation's semantics
// (filtering/filter_util.py:555-638, 669-716, 758-834):
//   * per page and head: Kmax / Kmin (exact fp16 min/max),
//   * V̄ = page mean of V (fp32 sum in token order, one rounding) for a page
//     filled from empty, the fp16 running mean for tokens added to a page
//     that already holds tokens,
//   * log-norm of V̄ for EVERY page, the partial last page included (the
//     reference kernel only writes full pages and reads them at the wrong
//     index, decode_attn.cuh:185-190).
//
// Work mapping: a workgroup of 4 waves covers one page x 16 heads; each
// wave covers 4 heads, one 16-lane DPP row per head, 8 dims per lane.  A
// wave's 16-byte loads of one token read 4 consecutive heads = 1 KB
// contiguous from the NHD input.
#include "kernels.hpp"

namespace aoakv {

constexpr int kHeadsPerWave = 4;
constexpr int kHeadsPerBlock = 16;


// With ROPE the block rows of grid.y past the kv heads' rotate q in place, and
// k is rotated (in place, and as stored): RoPE and append of a prompt in one
// pass, where the two launches read k twice.  Bound by HBM: 16000 tokens, 32
// heads, 944 MB needed: 229 us in two launches (rope_kernel 104, append 118),
// 187 in one (5.05 TB/s; a 1 GiB copy runs at 5.2).  Small prompts save the
// launch: 333 tokens 16.7 -> 13.2 us.
template <bool ROPE>
__global__ __launch_bounds__(256) void append_prefill_kernel(AppendPrefillArgs a) {
  const uint32_t lane = __lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t row = lane / kLanesPerRow;
  const uint32_t l16 = lane % kLanesPerRow;
  const uint32_t kv_blocks = (a.H + kHeadsPerBlock - 1) / kHeadsPerBlock;
  const bool q_block = ROPE && blockIdx.y >= kv_blocks;  // uniform per block
  const uint32_t h = (q_block ? blockIdx.y - kv_blocks : blockIdx.y) * kHeadsPerBlock +
                     wave * kHeadsPerWave + row;
  const uint32_t p = a.first_page + blockIdx.x;

  const uint32_t S = a.S;
  const uint32_t L = (a.num_pages - 1u) * S + a.last_page_len;
  const uint32_t start = L - a.N;  // first appended position
  const uint32_t e0 = start > p * S ? start - p * S : 0u;
  const uint32_t e1 = (L - p * S) < S ? (L - p * S) : S;
  const uint32_t n = e1 - e0;
  const uint32_t d0 = l16 * kVec;
  const uint32_t tok0 = p * S + e0 - start;  // row of the page's first token in k, v, q

  // cos / sin of the page's tokens for the 64 frequencies, once per block
  // (the whole 16 heads of each token read them)
  __shared__ float s_rope[ROPE ? kPageSize : 1][2][kHeadDim / 2];
  if constexpr (ROPE) {
    const uint32_t i = threadIdx.x % (kHeadDim / 2);
    const float f = a.rope_f.f[i];
    for (uint32_t t = threadIdx.x / (kHeadDim / 2); t < n; t += 256u / (kHeadDim / 2))
      sincosf((float)(p * S + e0 + t) * f, &s_rope[t][1][i], &s_rope[t][0][i]);
    __syncthreads();
  }
  auto table = [&](uint32_t t) {
    RopeTable rt;
    const uint32_t i = d0 % (kHeadDim / 2);
#pragma unroll
    for (int j = 0; j < kVec; ++j) {
      rt.c[j] = s_rope[t][0][i + j];
      rt.s[j] = s_rope[t][1][i + j];
    }
    return rt;
  };
  // tokens in flight (with RoPE at 16000 tokens: 2 201 us, 4 194, 8 187, 16
  // 187; without, 4 and 8 alike)
  constexpr uint32_t kB = ROPE ? 8 : 4;
  if constexpr (ROPE) {
    if (q_block) {
      if (h >= a.Hq) return;
      const size_t q_row = (size_t)a.Hq * kHeadDim;
      f16* q = a.q + tok0 * q_row + (size_t)h * kHeadDim + d0;
      for (uint32_t i0 = 0; i0 < n; i0 += kB) {
        H8 x[kB];
#pragma unroll
        for (uint32_t u = 0; u < kB; ++u) x[u] = ld16(q + (i0 + u < n ? i0 + u : n - 1u) * q_row);
#pragma unroll
        for (uint32_t u = 0; u < kB; ++u)
          if (i0 + u < n) st16(q + (i0 + u) * q_row, rope_row(x[u], table(i0 + u), l16));
      }
      return;
    }
  }
  if (h >= a.H) return;  // whole rows exit together

  const uint32_t phys = (uint32_t)a.kv_indices[p];
  const uint32_t mpage = (uint32_t)a.meta_indices[p / S];
  const uint32_t ment = p % S;

  f16* kmax_p = a.meta + elem_off(a.g, mpage, 0, h, ment) + d0;
  f16* kmin_p = a.meta + elem_off(a.g, mpage, 1, h, ment) + d0;
  f16* vbar_p = a.v_mean + ((size_t)phys * a.H + h) * kHeadDim + d0;

  H8 kmax, kmin, vbar;
  float vsum[kVec];
#pragma unroll
  for (int j = 0; j < kVec; ++j) vsum[j] = 0.f;
  if (e0 > 0u) {
    kmax = ld16(kmax_p);
    kmin = ld16(kmin_p);
    vbar = ld16(vbar_p);
  } else {
#pragma unroll
    for (int j = 0; j < kVec; ++j) {
      kmax.v[j] = (f16)-65504.0f;
      kmin.v[j] = (f16)65504.0f;
    }
  }

  const size_t in_row = (size_t)a.H * kHeadDim;
  f16* kin = a.k + tok0 * in_row + (size_t)h * kHeadDim + d0;
  const f16* vin = a.v + tok0 * in_row + (size_t)h * kHeadDim + d0;
  f16* kout = a.kv + elem_off(a.g, phys, 0, h, e0) + d0;
  f16* vout = a.kv + elem_off(a.g, phys, 1, h, e0) + d0;

  // kB tokens' loads go out together (the in-place stores of k would
  // otherwise hold back the next token's loads)
  for (uint32_t i0 = 0; i0 < n; i0 += kB) {
    H8 kk[kB], vv[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      const uint32_t i = i0 + u < n ? i0 + u : n - 1u;
      kk[u] = ld16(kin + i * in_row);
      vv[u] = ld16(vin + i * in_row);
    }
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      const uint32_t i = i0 + u;
      if (i >= n) break;
      if constexpr (ROPE) {
        kk[u] = rope_row(kk[u], table(i), l16);
        st16(kin + i * in_row, kk[u]);
      }
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
        kmax.v[j] = kk[u].v[j] > kmax.v[j] ? kk[u].v[j] : kmax.v[j];
        kmin.v[j] = kk[u].v[j] < kmin.v[j] ? kk[u].v[j] : kmin.v[j];
      }
      if (e0 == 0u) {
        // page filled from empty: V̄ = mean over its tokens (compute_page_v_mean)
#pragma unroll
        for (int j = 0; j < kVec; ++j) vsum[j] = vsum[j] + (float)vv[u].v[j];
      } else {
        // tokens added to a page that already holds e0 tokens: running mean
#pragma unroll
        for (int j = 0; j < kVec; ++j)
          vbar.v[j] = running_mean(vbar.v[j], vv[u].v[j], e0 + i);
      }
      st16(kout + (size_t)i * a.g.tok, kk[u]);
      st16(vout + (size_t)i * a.g.tok, vv[u]);
    }
  }
  if (e0 == 0u) {
#pragma unroll
    for (int j = 0; j < kVec; ++j) vbar.v[j] = r16(vsum[j] / (float)n);
  }
  st16(kmax_p, kmax);
  st16(kmin_p, kmin);
  st16(vbar_p, vbar);
  f16 lvn = log_norm_row(vbar);
  if (l16 == 0u) a.v_log_norm[(size_t)phys * a.H + h] = lvn;
}


// One new token per sequence (update_page_filters / update_mean_page_filters,
// filter_util.py:681-716, 758-795).  With ROPE the block rows of grid.y past
// the kv heads' rotate q in place, and k is rotated (in place, and as stored)
// before the append: RoPE + append + metadata in one launch, the reference's
// apply_rope_in_place then append_kv_cache_decode (QuestAttention.py:98-111).
// The new token sits at position L - 1 of its sequence (L counts it).
// Bound by its chain of round trips and by the rotation's sines: q / k and v are
// loaded beside the page table and the page's metadata flies during the
// rotation; with the log-norm's chain in registers, 32 heads 5.7 -> 5.05 us.
template <bool ROPE>
__global__ __launch_bounds__(256) void append_decode_kernel(AppendDecodeArgs a) {
  const uint32_t lane = __lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t row = lane / kLanesPerRow;
  const uint32_t l16 = lane % kLanesPerRow;
  const uint32_t b = blockIdx.x;
  const uint32_t kv_blocks = (a.H + kHeadsPerBlock - 1) / kHeadsPerBlock;
  const bool q_block = ROPE && blockIdx.y >= kv_blocks;  // uniform per block
  const uint32_t h = (q_block ? blockIdx.y - kv_blocks : blockIdx.y) * kHeadsPerBlock +
                     wave * kHeadsPerWave + row;
  if (h >= (q_block ? a.Hq : a.H)) return;

  const uint32_t S = a.S;
  const uint32_t d0 = l16 * kVec;
  // q or k, and v, need no earlier load: they go out beside the page table's
  f16* const x_p = (q_block ? a.q + ((size_t)b * a.Hq + h) * kHeadDim
                            : a.k + ((size_t)b * a.H + h) * kHeadDim) + d0;
  const H8 x = ld16(x_p);
  const H8 vv = ld16(a.v + ((size_t)b * a.H + (q_block ? 0u : h)) * kHeadDim + d0);
  const uint32_t pbeg = (uint32_t)a.kv_indptr[b];
  const uint32_t P = (uint32_t)a.kv_indptr[b + 1] - pbeg;
  const uint32_t lpl = (uint32_t)a.kv_last_page_len[b];
  if (P == 0u || lpl == 0u || lpl > S) return;  // malformed page table: nothing to do
  const uint32_t pos = (P - 1u) * S + lpl - 1u;
  if constexpr (ROPE) {
    if (q_block) {
      st16(x_p, rope_row(x, rope_table(pos, l16, a.rope_f.f), l16));
      return;
    }
  }
  const uint32_t e = lpl - 1u;  // entry of the new token
  const uint32_t p = P - 1u;
  const uint32_t phys = (uint32_t)a.kv_indices[pbeg + p];
  const uint32_t mpage = (uint32_t)a.meta_indices[(uint32_t)a.meta_indptr[b] + p / S];
  const uint32_t ment = p % S;

  f16* kmax_p = a.meta + elem_off(a.g, mpage, 0, h, ment) + d0;
  f16* kmin_p = a.meta + elem_off(a.g, mpage, 1, h, ment) + d0;
  f16* vbar_p = a.v_mean + ((size_t)phys * a.H + h) * kHeadDim + d0;

  H8 kk = x, kmax{}, kmin{}, vbar{};
  if (e != 0u) {  // (in flight during the rotation)
    kmax = ld16(kmax_p);
    kmin = ld16(kmin_p);
    vbar = ld16(vbar_p);
  }
  if constexpr (ROPE) {
    kk = rope_row(x, rope_table(pos, l16, a.rope_f.f), l16);
    st16(x_p, kk);
  }
  if (e == 0u) {  // new page: max = min = k, V̄ = v
    kmax = kk;
    kmin = kk;
    vbar = vv;
  } else {
#pragma unroll
    for (int j = 0; j < kVec; ++j) {
      kmax.v[j] = kk.v[j] > kmax.v[j] ? kk.v[j] : kmax.v[j];
      kmin.v[j] = kk.v[j] < kmin.v[j] ? kk.v[j] : kmin.v[j];
      vbar.v[j] = running_mean(vbar.v[j], vv.v[j], e);
    }
  }
  st16(a.kv + elem_off(a.g, phys, 0, h, e) + d0, kk);
  st16(a.kv + elem_off(a.g, phys, 1, h, e) + d0, vv);
  st16(kmax_p, kmax);
  st16(kmin_p, kmin);
  st16(vbar_p, vbar);
  f16 lvn = log_norm_row(vbar);
  if (l16 == 0u) a.v_log_norm[(size_t)phys * a.H + h] = lvn;
}

hipError_t launch_append_prefill(const AppendPrefillArgs& a, hipStream_t s) {
  const uint32_t L = (a.num_pages - 1u) * a.S + a.last_page_len;
  const uint32_t first_page = (L - a.N) / a.S;
  AppendPrefillArgs b = a;
  b.first_page = first_page;
  const uint32_t kv_blocks = (a.H + kHeadsPerBlock - 1) / kHeadsPerBlock;
  dim3 grid(a.num_pages - first_page, kv_blocks);
  if (a.q != nullptr) {
    grid.y += (a.Hq + kHeadsPerBlock - 1) / kHeadsPerBlock;
    hipLaunchKernelGGL(append_prefill_kernel<true>, grid, dim3(256), 0, s, b);
  } else {
    hipLaunchKernelGGL(append_prefill_kernel<false>, grid, dim3(256), 0, s, b);
  }
  return hipGetLastError();
}

hipError_t launch_append_decode(const AppendDecodeArgs& a, uint32_t batch, hipStream_t s) {
  const uint32_t kv_blocks = (a.H + kHeadsPerBlock - 1) / kHeadsPerBlock;
  if (a.rope) {
    const uint32_t q_blocks = (a.Hq + kHeadsPerBlock - 1) / kHeadsPerBlock;
    hipLaunchKernelGGL(append_decode_kernel<true>, dim3(batch, kv_blocks + q_blocks), dim3(256),
                       0, s, a);
  } else {
    hipLaunchKernelGGL(append_decode_kernel<false>, dim3(batch, kv_blocks), dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

// In-place RoPE of q [N, Hq, D] and k [N, Hkv, D], token n at position
// past + n (apply_rope_in_place, page.cu:224-265).  A block takes one token:
// each lane computes the cos / sin of its 8 dims once and its row rotates
// heads row, row + 16, ... of q then k.
__global__ __launch_bounds__(256) void rope_kernel(RopeArgs a) {
  const uint32_t lane = __lane_id();
  const uint32_t l16 = lane % kLanesPerRow;
  const uint32_t r = threadIdx.x / kLanesPerRow;  // 16 rows per block
  const uint32_t n = blockIdx.x;
  const RopeTable rt = rope_table(a.past + n, l16, a.rope_f.f);
  for (uint32_t h = r; h < a.Hq + a.Hkv; h += 16u) {
    f16* p = h < a.Hq ? a.q + ((size_t)n * a.Hq + h) * kHeadDim
                      : a.k + ((size_t)n * a.Hkv + (h - a.Hq)) * kHeadDim;
    p += l16 * kVec;
    st16(p, rope_row(ld16(p), rt, l16));
  }
}

hipError_t launch_rope(const RopeArgs& a, hipStream_t s) {
  if (a.N == 0u) return hipSuccess;
  hipLaunchKernelGGL(rope_kernel, dim3(a.N), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace aoakv
