// The chain over a row's segments shared by the segmented state recurrence (state_bwd.hip) and the
// segmented forward scan (recompute.hip).
#pragma once
#include "common.hpp"

namespace rewy {

// Segmented forms, step 2: per (row, head, 8 state columns), walk the row's segments.  REV (the
// reverse recurrence): from the last to the first, X (the state at the segment's end; dht or zero
// for the last) is written to xbuf[segment], then X <- P X + Q, the state at the segment's start;
// after the first segment X is the row's dh0.  Else (the forward scan) from the first to the last,
// X the state at the segment's start (h0 or zero for the first), at the end the row's final state:
// read `dht` as the initial and `dh0` as the final state.  fp32 throughout.  P is staged in
// LDS transposed (coalesced global reads, fetched one segment ahead into registers;
// lane r then reads P[r][k] from consecutive banks), X in LDS; thread (r, half) owns
// state row r and 4 of the 8 columns.  Narrow column blocks give B*H*16 work-groups:
// the chain's length is the number of segments, each step a 128 x 128 x 8 product.
constexpr int COMB_COLS = 8;
template <bool REV>
__global__ __launch_bounds__(256) void state_combine_kernel(const float* __restrict__ pbuf,
                                                            const float* __restrict__ qbuf,
                                                            const float* __restrict__ dht, float* __restrict__ xbuf,
                                                            float* __restrict__ dh0, int segs, int H, int vf) {
  __shared__ float pt[KD][KD + 1];      // P^T of the current segment (odd pitch: transposed writes spread over banks)
  __shared__ f32x4 xs[KD][COMB_COLS / 4];
  const int bh = blockIdx.x, row = bh / H, h = bh % H;
  const int tid = threadIdx.x, r = tid >> 1, hc = tid & 1;
  const int col = COMB_COLS * blockIdx.y + 4 * hc;
  // dht / dh0 are [K,V] or (vf, state_v_first) [V,K] per (row, head)
  f32x4 x = zero4();
  if (dht) {
    const float* d = dht + (size_t)bh * KD * VD;
    if (vf) {
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = d[(col + e) * KD + r];
    } else {
      x = *reinterpret_cast<const f32x4u*>(d + r * VD + col);
    }
  }
  f32x4 pre[KD * KD / 4 / 256];
  auto fetch = [&](int sg) {
    const float* P = pbuf + (((size_t)row * segs + sg) * H + h) * KD * KD;
#pragma unroll
    for (int i = 0; i < KD * KD / 4 / 256; ++i) {     // lanes along rows of P
      const int p4 = tid + 256 * i;
      pre[i] = *reinterpret_cast<const f32x4*>(P + (size_t)(p4 >> 5) * KD + 4 * (p4 & 31));
    }
  };
  fetch(REV ? segs - 1 : 0);
  for (int i = 0; i < segs; ++i) {
    const int sg = REV ? segs - 1 - i : i;
    const size_t seg = ((size_t)row * segs + sg) * H + h;
    const size_t xo = (seg * KD + r) * VD + col;
    f32x4 acc = *reinterpret_cast<const f32x4*>(qbuf + xo);
#pragma unroll
    for (int i = 0; i < KD * KD / 4 / 256; ++i) {
      const int p4 = tid + 256 * i, pr = p4 >> 5, pc = 4 * (p4 & 31);
#pragma unroll
      for (int e = 0; e < 4; ++e) pt[pc + e][pr] = pre[i][e];
    }
    xs[r][hc] = x;
    *reinterpret_cast<f32x4*>(xbuf + xo) = x;
    __syncthreads();
    if (i + 1 < segs) fetch(REV ? sg - 1 : sg + 1);
#pragma unroll 16
    for (int kk = 0; kk < KD; ++kk) {
      const float p = pt[kk][r];
      const f32x4 xv = xs[kk][hc];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(p, xv[e], acc[e]);
    }
    __syncthreads();
    x = acc;
  }
  if (dh0) {
    float* d = dh0 + (size_t)bh * KD * VD;
    if (vf) {
#pragma unroll
      for (int e = 0; e < 4; ++e) d[(col + e) * KD + r] = x[e];
    } else {
      *reinterpret_cast<f32x4u*>(d + r * VD + col) = x;
    }
  }
}

}  // namespace rewy
