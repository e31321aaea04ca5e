// The dW split-K reduce (experts.hip's dw_reduce_kernel; also run inside combine_dx's
// launch, router_grad.hip): the fp32 partials of the multi-chunk groups summed in chunk
// order into dW.  The workgroup's index is an argument, so the body runs in any launch whose
// workgroups have NT threads.
#pragma once

#include "experts_common.h"

namespace nsmoe {

struct DwReduceArgs {
  ExpParams p_in, p_out;  // dW_in and dW_out: pointers and partials
  int wgs;                // workgroups (0: no reduce to run)
};

// Blocks of NT threads x 4 elements in one group's dW.
__host__ __device__ __forceinline__ int dw_reduce_blocks(int64_t mn) {
  return (int)((mn + 4 * NT - 1) / (4 * NT));
}

// Block b of the `nch` partials at `src` (mn elements each) into dst: each thread 4
// consecutive elements, up to DEPTH chunks' 16-byte loads in flight at once; the additions
// are in chunk order for every element, whatever the launch shape.
template <int DT>
__device__ __forceinline__ void dw_reduce_block(const float* src, int64_t mn, int nch, int b,
                                                typename Elem<DT>::T* dst) {
  const int64_t i = ((int64_t)b * NT + threadIdx.x) * 4;
  if (i >= mn) return;
  if (mn % 4 == 0) {  // every partial is 16-byte aligned
    constexpr int DEPTH = 16;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < nch; c0 += DEPTH) {
      f32x4 a[DEPTH];
#pragma unroll
      for (int u = 0; u < DEPTH; ++u)
        if (c0 + u < nch) a[u] = *(const f32x4*)(src + (int64_t)(c0 + u) * mn + i);
#pragma unroll
      for (int u = 0; u < DEPTH; ++u)
        if (c0 + u < nch) acc += a[u];
    }
    if (DT != DT_F32 && ((uintptr_t)dst & 7) == 0) {  // one 8-byte store
      *(uint2*)(dst + i) = make_uint2(pack2<DT>(acc[0], acc[1]), pack2<DT>(acc[2], acc[3]));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[i + e] = Elem<DT>::from_f(acc[e]);
    }
  } else {
    for (int e = 0; e < 4 && i + e < mn; ++e) {
      float acc = 0.0f;
      for (int c = 0; c < nch; ++c) acc += src[(int64_t)c * mn + i + e];
      dst[i + e] = Elem<DT>::from_f(acc);
    }
  }
}

// Workgroup wg of r.wgs.  The multi-chunk groups and their first partials are listed in LDS
// (up to NT groups a round, shared groups first, as the partials lie), then the (group, mode,
// block) items of the list are dealt over the workgroups: no barrier between items, so the
// loads of one overlap the stores of the last.
template <int DT>
__device__ __forceinline__ void dw_reduce_wg(const DwReduceArgs& r, int wg) {
  using T = typename Elem<DT>::T;
  __shared__ int s_g[NT], s_base[NT], s_sum[NT / 64], s_cnt[NT / 64];
  const ExpParams& p = r.p_in;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int64_t mn_in = (int64_t)p.d * 2 * p.H, mn_out = (int64_t)p.H * p.d;
  const int b_in = dw_reduce_blocks(mn_in), nb = b_in + dw_reduce_blocks(mn_out);
  int base = 0;
  for (int v0 = 0; v0 < p.E + p.S; v0 += NT) {
    const int v = v0 + tid;
    const int g = v < p.S ? p.E + v : v - p.S;
    int c = v < p.E + p.S ? dw_chunks(rows_of(p, g), p.dw_rc) : 0;
    if (c <= 1) c = 0;
    const int incl = wave_scan_incl(c);
    const unsigned long long hit = __ballot(c > 0);
    if (lane == 63) {
      s_sum[wave] = incl;
      s_cnt[wave] = __popcll(hit);
    }
    __syncthreads();
    int at = __popcll(hit & ((1ull << lane) - 1)), n = 0, first = base + incl - c;
    for (int w = 0; w < NT / 64; ++w) {
      if (w < wave) {
        at += s_cnt[w];
        first += s_sum[w];
      }
      n += s_cnt[w];
      base += s_sum[w];
    }
    if (c) {
      s_g[at] = g;
      s_base[at] = first;
    }
    __syncthreads();
    for (int64_t it = wg; it < (int64_t)n * nb; it += r.wgs) {
      const int li = (int)(it / nb), b = (int)(it % nb);
      const int gg = s_g[li], nch = dw_chunks(rows_of(p, gg), p.dw_rc);
      const bool in = b < b_in;
      const ExpParams& q = in ? r.p_in : r.p_out;
      const int64_t mn = in ? mn_in : mn_out;
      T* dst = gg < p.E ? (T*)q.dw_a + (int64_t)gg * mn : (T*)q.dw_sh + (int64_t)(gg - p.E) * mn;
      dw_reduce_block<DT>(q.partial + (int64_t)s_base[li] * mn, mn, nch, in ? b : b - b_in, dst);
    }
    __syncthreads();  // the list is read before the next round rewrites it
  }
}

}  // namespace nsmoe
