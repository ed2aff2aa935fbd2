// The forward state scan with the output formed in it, for a forward whose backward does not read
// the states (recompute policy, inference): fdr_fwd_h and fdr_fwd_o in one sweep over operands that
// fdr_fwd_prepare_scan writes in the order it reads them (sop, scan_body.hpp).
//
// Replaces, with fdr_fwd_prepare_scan before it, FLA's recompute_w_u_fwd,
// chunk_gated_delta_rule_fwd_h and chunk_fwd_o (reference _compat/gdn.py:33-123,
// _compat/kda.py:89-113).  Per (batch, head, value tile) and for chunk c = 0 .. NT-1, with h the
// fp32 state in accumulators and h_c its bf16 rounding:
//
//   v_new_c = u_c - w_c h_c                                  (bf16)
//   o_c     = scale (q 2^gc) h_c + Aqk v_new_c               (bf16)
//   h       = diag(lambda_c) h + kg_c^T v_new_c
//
// h_c and v_new_c never leave the chip.
//
// SPLIT: v_new enters the state's update as bf16 hi + lo (16-bit mantissa) instead of one bf16, the precision
// of the affine-step form, whose kg^T u goes into the state in fp32 (affine.hip).  It serves the calls that
// form would take (few heads).  Final state against fp64, one bf16 / hi + lo / affine-step: DeltaNet B=1
// T=2048 H=4 3.77e-3 / 3.11e-3 / 3.30e-3, KDA 3.26e-3 / 2.83e-3 / 2.83e-3; whole forward, us, one bf16 / hi + lo:
// 45.8 / 47.9 and 55.4 / 58.7, KDA T=65536 H=16 1403 / 1473.  Of a segment's map only Q takes the split (P's
// columns too: 1516 us, the same errors).
#include "rewy_amd.h"

#include "scan_body.hpp"
#include "segment_combine.hpp"

namespace rewy {

template <int BV, bool SPLIT>
struct ScanOSmem {
  static constexpr int LDK = KD + 8;
  static constexpr int LDT = C + 8;
  bf16 k[2][C * KD];              // kg tile by chunk parity: read after a step's last barrier
  bf16 hT[BV][LDK];               // h^T
  bf16 vT[BV][LDT];               // v_new^T
  bf16 vlT[SPLIT ? BV : 1][LDT];  // and its rest
};

// Eight waves own 16 state rows each; beside that waves 0-3 form v_new and waves 4-7 o, each for one
// 16-token tile and all BV columns, so that a token tile's w, q and Aqk fragments feed one wave and
// need no LDS.  Each role runs a loop of its own: its loads and stores are the same every step and
// the compiler's wait counts exact.  A step is bound by its chain h -> v_new -> h (two barriers) and
// by what a CU loads per step (78 KiB): 1.1 us on idle CUs, 1.5-2 us with all of them busy.
// Against fdr_fwd_h then fdr_fwd_o: KDA B=8 T=4096 H=16 206 us (64-wide tiles) against 382, GDN 177
// against 338; GDN2 B=2 T=8192 H=32 253 (32-wide) against 432; KDA B=1 T=8192 H=32 196 (16-wide)
// against 299, H=8 142 against 159.  All operands staged through LDS instead took 260, 396 and 314
// (first, third and fourth); two chunks of prefetch instead of one 206, 265 and 207.
template <int BV, bool VEC, bool MAP, bool SPLIT>
__global__ __launch_bounds__(512) void fwd_scan_o_kernel(const char* __restrict__ ops, const float* __restrict__ h0,
                                                         bf16* __restrict__ o_out, float* __restrict__ ht_out, int T,
                                                         int H, float scale, const int* __restrict__ chunk_off,
                                                         int vf, const int* __restrict__ cu, int N, int segs,
                                                         const float* __restrict__ xseg,
                                                         const float* __restrict__ xlast) {
  using S = ScanOSmem<BV, SPLIT>;
  __shared__ __attribute__((aligned(16))) S sm;
  constexpr int NVT = VD / BV;
  constexpr int NCT = BV / 16;
  const int logical = chunk_off ? packed_logical(chunk_off, N, H, NVT) : xcd_logical_block();
  if (logical < 0) return;
  const int vt = logical % NVT;
  const int bh = logical / NVT;
  const int b = bh / H, h = bh % H;
  // chunks [c0, c0 + NT): row b of T tokens, or sequence b of a packed batch (as fwd_h_kernel)
  // or (segs > 1) segment sg of row rb, from its own start state
  const int rb = chunk_off ? b : b / segs, sg = b - rb * segs, NTr = T / C;
  const int c0 = chunk_off ? min(max(chunk_off[b], 0), NTr) : rb * NTr + sg * NTr / segs;
  const int NT = chunk_off ? max(min(chunk_off[b + 1], NTr) - c0, 0) : rb * NTr + (sg + 1) * NTr / segs - c0;
  const size_t sbh = chunk_off ? bh : rb * H + h;     // the states' index
  const int tid = threadIdx.x, l = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_id());
  const int lc = l & 15, lg = l >> 4;
  const int v_base = vt * BV;
  const size_t rsv = (size_t)H * VD;
  const int drow = wv & 3, trow = 16 * drow + lc;     // this wave's token tile, this lane's operand row

  // state rows [16 wv, 16 wv + 16)
  f32x4 st[NCT];
  const float* src = h0 ? h0 + sbh * KD * VD : nullptr;     // [K,V] or, state_v_first (vf), [V,K]
  int svf = vf;
  if (!chunk_off && sg > 0) {
    if (sg < segs - 1) {
      src = xseg + ((size_t)(rb * (segs - 1) + sg) * H + h) * KD * VD;
      svf = 0;
    } else {
      src = xlast + sbh * KD * VD;
    }
  }
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    f32x4 a = zero4();
    if (src) {
      const int col = v_base + 16 * ct + lc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kr = 16 * wv + 4 * lg + r;
        a[r] = src[svf ? col * KD + kr : kr * VD + col];
      }
    }
    st[ct] = a;
  }
  auto chunk_ops = [&](int c) { return ops + ((size_t)(c0 + c) * H + h) * sop::BYTES; };

  // ---- both roles: kg and lambda of a chunk, one step ahead in registers ----
  u32x4 rk[2];
  f32x4 rlam;
  auto load_common = [&](const char* p) {
#pragma unroll
    for (int i = 0; i < 2; ++i) rk[i] = *reinterpret_cast<const u32x4*>(p + sop::K + 16 * (tid + 512 * i));
    rlam = *reinterpret_cast<const f32x4*>(p + sop::LAM + 4 * (16 * wv + 4 * lg));
  };
  auto settle_common = [&]() {
    settle(rk[0]);
    settle(rk[1]);
    settle(rlam);
  };
  auto stage_common = [&](int db) {
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(sm.k[db] + 8 * (tid + 512 * i)) = rk[i];
  };
  // h_c -> LDS (transposed, bf16)
  auto write_h = [&]() {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      bf16x4 v4;
#pragma unroll
      for (int r = 0; r < 4; ++r) v4[r] = to_bf16(st[ct][r]);
      *reinterpret_cast<bf16x4*>(&sm.hT[16 * ct + lc][16 * wv + 4 * lg]) = v4;
    }
  };
  // h <- lambda h + kg^T v_new
  auto update = [&](int db, f32x4 lam) {
    const bf16x8 k0 = frag_tr<16>(sm.k[db], 0, 16 * wv), k1 = frag_tr<16>(sm.k[db], 32, 16 * wv);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      f32x4 a = st[ct] * lam;
      a = mfma(k0, frag(&sm.vT[16 * ct][0], S::LDT), a);
      a = mfma(k1, frag(&sm.vT[16 * ct][32], S::LDT), a);
      if constexpr (SPLIT) {
        a = mfma(k0, frag(&sm.vlT[16 * ct][0], S::LDT), a);
        a = mfma(k1, frag(&sm.vlT[16 * ct][32], S::LDT), a);
      }
      st[ct] = a;
    }
  };
  // A step needs no barrier at its start: h^T and v_new^T were last read before the previous step's
  // last barrier or this step's first, and kg has a buffer per chunk parity.

  if (wv < 4) {
    // ---- v_new = u - w h (rows t, column v) ----
    u32x4 wn[4];
    bf16x4 un[NCT];
    auto load = [&](const char* p) {
      load_common(p);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        wn[ks] = *reinterpret_cast<const u32x4*>(p + sop::W + ((drow * 4 + ks) * 64 + l) * 16);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
        un[ct] = *reinterpret_cast<const bf16x4*>(p + sop::U + ((drow * 8 + vt * NCT + ct) * 64 + l) * 8);
    };
    auto settle_all = [&]() {
      settle_common();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) settle(wn[ks]);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) settle(un[ct]);
    };
    if (NT > 0) {
      load(chunk_ops(0));
      settle_all();
    }
    for (int c = 0; c < NT; ++c) {
      const int db = c & 1;
      stage_common(db);
      bf16x8 wf[4];
      f32x4 a[NCT];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) wf[ks] = __builtin_bit_cast(bf16x8, wn[ks]);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) a[ct][r] = -to_f32(un[ct][r]);
      const f32x4 lam = rlam;
      load(chunk_ops(c + 1 < NT ? c + 1 : c));   // (the last chunk re-fetches itself: no branch)
      write_h();
      lds_barrier();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) a[ct] = mfma(wf[ks], frag(&sm.hT[16 * ct][32 * ks], S::LDK), a[ct]);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        bf16x4 lo;
        const bf16x4 hi = split_hi4(-a[ct], lo);
        *reinterpret_cast<bf16x4*>(&sm.vT[16 * ct + lc][16 * drow + 4 * lg]) = hi;
        if constexpr (SPLIT) *reinterpret_cast<bf16x4*>(&sm.vlT[16 * ct + lc][16 * drow + 4 * lg]) = lo;
      }
      lds_barrier();
      update(db, lam);
      settle_all();          // the next chunk's operands
    }
  } else {
    // ---- o^T = scale h^T (q 2^gc)^T + v_new^T Aqk^T (rows v, column t) ----
    u32x4 qn[4], qln[VEC ? 4 : 1], an[4];
    float fqn = 0.f;
    auto load = [&](const char* p) {
      load_common(p);
      if constexpr (!VEC) fqn = *reinterpret_cast<const float*>(p + sop::FQ + 4 * trow);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        qn[ks] = *reinterpret_cast<const u32x4*>(p + sop::Q + ((drow * 4 + ks) * 64 + l) * 16);
        if constexpr (VEC) qln[ks] = *reinterpret_cast<const u32x4*>(p + sop::QL + ((drow * 4 + ks) * 64 + l) * 16);
      }
      // hi, lo of columns 0-31, then of 32-63 (tokens 32-63 only: above the diagonal for the
      // others, whose waves re-read the first and skip its products)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        an[j] = *reinterpret_cast<const u32x4*>(p + sop::A + ((drow * 4 + (drow < 2 ? j & 1 : j)) * 64 + l) * 16);
    };
    auto settle_all = [&]() {
      settle_common();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        settle(qn[ks]);
        if constexpr (VEC) settle(qln[ks]);
        settle(an[ks]);
      }
      settle(fqn);
    };
    if (NT > 0) {
      load(chunk_ops(0));
      settle_all();
    }
    for (int c = 0; c < NT; ++c) {
      const int db = c & 1;
      stage_common(db);
      bf16x8 qf[4], qlf[VEC ? 4 : 1], af[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        qf[ks] = __builtin_bit_cast(bf16x8, qn[ks]);
        if constexpr (VEC) qlf[ks] = __builtin_bit_cast(bf16x8, qln[ks]);
        af[ks] = __builtin_bit_cast(bf16x8, an[ks]);
      }
      const float f = VEC ? scale : fqn;
      const f32x4 lam = rlam;
      load(chunk_ops(c + 1 < NT ? c + 1 : c));
      write_h();
      lds_barrier();
      f32x4 oa[NCT], ob[NCT];
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) oa[ct] = ob[ct] = zero4();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
          const bf16x8 hf = frag(&sm.hT[16 * ct][32 * ks], S::LDK);
          oa[ct] = mfma(hf, qf[ks], oa[ct]);
          if constexpr (VEC) ob[ct] = mfma(hf, qlf[ks], ob[ct]);
        }
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) oa[ct] = (VEC ? oa[ct] + ob[ct] : oa[ct]) * f;
      lds_barrier();
      update(db, lam);
      const Rows<MAP> rs_ = seq_chunk_rows<MAP>(cu, b, c, c0 + c);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const bf16x8 v0 = frag(&sm.vT[16 * ct][0], S::LDT);
        f32x4 a = mfma(v0, af[0], oa[ct]);
        a = mfma(v0, af[1], a);
        if (drow >= 2) {                             // wave-uniform
          const bf16x8 v1 = frag(&sm.vT[16 * ct][32], S::LDT);
          a = mfma(v1, af[2], a);
          a = mfma(v1, af[3], a);
        }
        bf16x4 o4;
#pragma unroll
        for (int r = 0; r < 4; ++r) o4[r] = to_bf16(a[r]);
        *reinterpret_cast<bf16x4*>(
            rs_.dst(o_out + (rs_.tok0 + trow) * rsv + (size_t)h * VD + v_base + 16 * ct + 4 * lg, trow)) = o4;
      }
      settle_all();
    }
  }
  if (ht_out && (chunk_off || sg == segs - 1)) {
    float* dst = ht_out + sbh * KD * VD;
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kr = 16 * wv + 4 * lg + r, col = v_base + 16 * ct + lc;
        dst[vf ? col * KD + kr : kr * VD + col] = st[ct][r];
      }
  }
}

// Segmented rows, step 1: the map X -> P X + Q of every segment of a row but the last, as
// fwd_xfer_kernel (recompute.hip) forms it -- 64 columns of P and of Q to a work-group, per-chunk
// arithmetic the scan's -- but over the scan's operands: w and u go straight to registers, kg's LDS
// image is copied.  P to pbuf [N (segs - 1), H, K, K], Q to qbuf likewise.  Bound by the step's chain as
// the scan (2.1 us a chunk).  With the combine and the segments' scans (KDA, us, one scan / in segments):
// H=16 1024 chunks 1434 / 705, 256 chunks 359 / 204, H=8 256 chunks 262 / 145, H=4 128 chunks 134 / 92.
template <bool SPLIT>
struct ScanXferSmem {
  static constexpr int LDK = KD + 8;
  static constexpr int LDT = C + 8;
  bf16 k[2][C * KD];       // by chunk parity
  bf16 hT[128][LDK];       // state^T: columns 0-63 of P's half, 64-127 of Q's
  bf16 vT[128][LDT];       // [-w P | u - w Q]^T
  bf16 vlT[SPLIT ? 64 : 1][LDT];   // the rest of Q's columns
};

template <bool SPLIT>
__global__ __launch_bounds__(512) void scan_xfer_kernel(const char* __restrict__ ops, float* __restrict__ pbuf,
                                                        float* __restrict__ qbuf, int T, int H, int segs) {
  using S = ScanXferSmem<SPLIT>;
  __shared__ __attribute__((aligned(16))) S sm;
  const int logical = xcd_logical_block();
  const int half = logical & 1;
  const int bh = logical >> 1;
  const int b = bh / H, h = bh % H;
  const int row = b / (segs - 1), sg = b % (segs - 1), NTr = T / C;
  const int c0 = row * NTr + sg * NTr / segs;
  const int NT = row * NTr + (sg + 1) * NTr / segs - c0;
  const int base = 64 * half;
  const int tid = threadIdx.x, l = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_id());
  const int lc = l & 15, lg = l >> 4;
  f32x4 st[8];                          // state rows [16 wv, 16 wv + 16)
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) st[j][r] = (j < 4 && 16 * wv + 4 * lg + r == base + 16 * j + lc) ? 1.f : 0.f;
  const int drow = wv & 3, dct0 = 4 * (wv >> 2);    // v: waves 0-3 P's columns, 4-7 Q's
  const bool q_half = wv >= 4;
  u32x4 rk[2], wn[4];
  bf16x4 un[4];
  f32x4 rlam;
  auto load_chunk = [&](int c) {
    const char* p = ops + ((size_t)(c0 + c) * H + h) * sop::BYTES;
#pragma unroll
    for (int i = 0; i < 2; ++i) rk[i] = *reinterpret_cast<const u32x4*>(p + sop::K + 16 * (tid + 512 * i));
    rlam = *reinterpret_cast<const f32x4*>(p + sop::LAM + 4 * (16 * wv + 4 * lg));
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      wn[ks] = *reinterpret_cast<const u32x4*>(p + sop::W + ((drow * 4 + ks) * 64 + l) * 16);
    // (P's waves load u too and drop it: the loads of every wave the same)
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
      un[cc] = *reinterpret_cast<const bf16x4*>(p + sop::U + ((drow * 8 + 4 * half + cc) * 64 + l) * 8);
  };
  auto settle_chunk = [&]() {
    settle(rk[0]);
    settle(rk[1]);
    settle(rlam);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      settle(wn[ks]);
      settle(un[ks]);
    }
  };
  if (NT > 0) {
    load_chunk(0);
    settle_chunk();
  }
  for (int c = 0; c < NT; ++c) {
    // no barrier at a step's start: as fwd_scan_o_kernel
    const int db = c & 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(sm.k[db] + 8 * (tid + 512 * i)) = rk[i];
    bf16x8 wf[4];
    f32x4 a[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) wf[ks] = __builtin_bit_cast(bf16x8, wn[ks]);
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
      for (int r = 0; r < 4; ++r) a[cc][r] = q_half ? -to_f32(un[cc][r]) : 0.f;
    const f32x4 lam = rlam;
    load_chunk(c + 1 < NT ? c + 1 : c);    // (the last chunk re-fetches itself: no branch)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      bf16x4 v4;
#pragma unroll
      for (int r = 0; r < 4; ++r) v4[r] = to_bf16(st[j][r]);
      *reinterpret_cast<bf16x4*>(&sm.hT[16 * j + lc][16 * wv + 4 * lg]) = v4;
    }
    lds_barrier();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int cc = 0; cc < 4; ++cc)
        a[cc] = mfma(wf[ks], frag(&sm.hT[16 * (dct0 + cc)][32 * ks], S::LDK), a[cc]);
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      bf16x4 lo;
      const bf16x4 hi = split_hi4(-a[cc], lo);
      *reinterpret_cast<bf16x4*>(&sm.vT[16 * (dct0 + cc) + lc][16 * drow + 4 * lg]) = hi;
      if (SPLIT && q_half) *reinterpret_cast<bf16x4*>(&sm.vlT[16 * cc + lc][16 * drow + 4 * lg]) = lo;
    }
    lds_barrier();
    const bf16x8 k0 = frag_tr<16>(sm.k[db], 0, 16 * wv), k1 = frag_tr<16>(sm.k[db], 32, 16 * wv);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f32x4 x = st[j] * lam;
      x = mfma(k0, frag(&sm.vT[16 * j][0], S::LDT), x);
      x = mfma(k1, frag(&sm.vT[16 * j][32], S::LDT), x);
      if constexpr (SPLIT) {
        if (j >= 4) {
          x = mfma(k0, frag(&sm.vlT[16 * (j - 4)][0], S::LDT), x);
          x = mfma(k1, frag(&sm.vlT[16 * (j - 4)][32], S::LDT), x);
        }
      }
      st[j] = x;
    }
    settle_chunk();
  }
  float* pdst = pbuf + (size_t)bh * KD * KD;
  float* qdst = qbuf + (size_t)bh * KD * VD;
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      (j < 4 ? pdst : qdst)[(16 * wv + 4 * lg + r) * KD + base + 16 * (j & 3) + lc] = st[j][r];
}

template <int BV>
static hipError_t launch_scan_o(const void* ops, bool vec, const float* h0, void* o, float* ht, int N, int T, int H,
                                float scale, const int* co, int vf, const int* cu, int segs, float* ws, bool split,
                                hipStream_t s) {
  const int grid = co ? packed_grid(N, H, VD / BV) : N * segs * H * (VD / BV);
  const float *xseg = nullptr, *xlast = nullptr;
  if (segs > 1) {
    const size_t maps = (size_t)N * (segs - 1) * H * KD * VD;
    float *pbuf = ws, *qbuf = ws + maps, *xb = ws + 2 * maps, *xl = ws + 3 * maps;
    hipLaunchKernelGGL(split ? scan_xfer_kernel<true> : scan_xfer_kernel<false>, dim3(N * (segs - 1) * H * 2), dim3(512),
                       0, s, (const char*)ops, pbuf, qbuf, T, H, segs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(state_combine_kernel<false>, dim3(N * H, VD / COMB_COLS), dim3(256), 0, s, pbuf, qbuf, h0, xb, xl,
                       segs - 1, H, vf);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    xseg = xb;
    xlast = xl;
  }
#define SO_LAUNCH(VEC, MAP, SPLIT)                                                                              \
  hipLaunchKernelGGL((fwd_scan_o_kernel<BV, VEC, MAP, SPLIT>), dim3(grid), dim3(512), 0, s, (const char*)ops, h0,   \
                     (bf16*)o, ht, T, H, scale, co, vf, cu, N, segs, xseg, xlast)
  if (split) {                                       // dense rows
    if (vec) SO_LAUNCH(true, false, true);
    else SO_LAUNCH(false, false, true);
  } else if (vec) {
    if (cu) SO_LAUNCH(true, true, false);
    else SO_LAUNCH(true, false, false);
  } else {
    if (cu) SO_LAUNCH(false, true, false);
    else SO_LAUNCH(false, false, false);
  }
#undef SO_LAUNCH
  return hipGetLastError();
}

}  // namespace rewy

using namespace rewy;

// Value-tile width: the narrowest tile with at most 256 work-groups, as the other scans' (us at 16 /
// 32 / 64: B*H = 32 196 / 235 / 342, 64 393 / 253 / 355, 128 400 / 263 / 206).
static int scan_o_bv(int N, int H) {
  const int bh = N * H;
  if (bh * 8 <= 256) return 16;
  if (bh * 4 <= 256) return 32;
  return 64;
}

extern "C" size_t fdr_scan_workspace_bytes(int N, int H, int segments) {
  if (N <= 0 || H <= 0 || segments <= 1) return 0;
  return (size_t)N * H * (3 * (size_t)(segments - 1) + 1) * KD * VD * sizeof(float);
}

static hipError_t scan_o_dispatch(const void* operands, int gate_mode, const float* h0, void* o, float* ht,
                                  int state_v_first, const int* chunk_offsets, const int* cu_seqlens, int N,
                                  int T, int H, int K, int V, int chunk, float scale, int value_block, int segments,
                                  void* workspace, bool split, hipStream_t stream) {
  if (K != KD || V != VD || chunk != C || T <= 0 || T % C || N <= 0 || H <= 0) return hipErrorInvalidValue;
  if (!operands || !o || gate_mode < RG_NONE || gate_mode > RG_VECTOR) return hipErrorInvalidValue;
  if (cu_seqlens && !chunk_offsets) return hipErrorInvalidValue;
  if (split && chunk_offsets) return hipErrorInvalidValue;
  if (!aligned16(operands) || !aligned16(workspace)) return hipErrorInvalidValue;
  if (segments < 1 || segments > T / C || (segments > 1 && (chunk_offsets || !workspace))) return hipErrorInvalidValue;
  const int bv = value_block > 0 ? value_block : scan_o_bv(N * segments, H);
#define SO_ARGS operands, gate_mode == RG_VECTOR, h0, o, ht, N, T, H, scale, chunk_offsets, state_v_first ? 1 : 0, \
                cu_seqlens, segments, (float*)workspace, split, stream
  switch (bv) {
    case 16: return launch_scan_o<16>(SO_ARGS);
    case 32: return launch_scan_o<32>(SO_ARGS);
    case 64: return launch_scan_o<64>(SO_ARGS);
    default: return hipErrorInvalidValue;
  }
#undef SO_ARGS
}

extern "C" hipError_t fdr_fwd_scan_o(const void* operands, int gate_mode, const float* h0, void* o, float* ht,
                                     int state_v_first, const int* chunk_offsets, const int* cu_seqlens, int N,
                                     int T, int H, int K, int V, int chunk, float scale, int value_block, int segments,
                                     void* workspace, hipStream_t stream) {
  return scan_o_dispatch(operands, gate_mode, h0, o, ht, state_v_first, chunk_offsets, cu_seqlens, N, T, H, K, V, chunk,
                         scale, value_block, segments, workspace, false, stream);
}

// The two launches as one host call: a short forward is bound by the host, and a foreign-function
// call with its argument checks costs it ~8 us.
static hipError_t forward_scan_dispatch(const void* q, const void* k, const void* v, const void* g, int gate_mode,
                                        int raw_gate, const float* A_log, const float* dt_bias, int has_lower_bound,
                                        float lower_bound, const void* beta, const void* b_gate, const void* w_gate,
                                        float norm_eps, int raw_beta, float beta_scale, void* q_norm, void* k_norm,
                                        float* q_rnorm, float* k_rnorm, float* beta_out, float* gc, float* Aqk,
                                        float* Akk, void* operands, const float* h0, void* o, float* ht,
                                        int state_v_first, const int* chunk_offsets, const int* cu_seqlens,
                                        const int* chunk_indices, int B, int T, int N, int H, int qk_heads, int K,
                                        int V, int chunk, float scale, int value_block, int segments, void* workspace,
                                        bool split, hipStream_t stream) {
  // what only fdr_fwd_scan_o would refuse, before the first launch (T here: as fdr_fwd_prepare_scan's)
  if (!o || N <= 0 || (!chunk_offsets && N != B) || (cu_seqlens && !chunk_offsets) || (chunk_offsets && B != 1) ||
      (value_block != 0 && value_block != 16 && value_block != 32 && value_block != 64) ||
      segments < 1 || segments > T / C || (segments > 1 && (chunk_offsets || !workspace)) || (split && chunk_offsets) ||
      !aligned16(workspace))
    return hipErrorInvalidValue;
  const hipError_t st =
      fdr_fwd_prepare_scan(q, k, v, g, gate_mode, raw_gate, A_log, dt_bias, has_lower_bound, lower_bound, beta, b_gate,
                           w_gate, norm_eps, raw_beta, beta_scale, q_norm, k_norm, q_rnorm, k_rnorm, beta_out, gc, Aqk,
                           Akk, operands, cu_seqlens, chunk_indices, B, T, H, qk_heads, K, V, chunk,
                           scale, stream);
  if (st != hipSuccess) return st;
  return scan_o_dispatch(operands, gate_mode, h0, o, ht, state_v_first, chunk_offsets, cu_seqlens, N, T, H, K, V, chunk,
                         scale, value_block, segments, workspace, split, stream);
}

extern "C" hipError_t fdr_forward_scan(const void* q, const void* k, const void* v, const void* g, int gate_mode,
                                       int raw_gate, const float* A_log, const float* dt_bias, int has_lower_bound,
                                       float lower_bound, const void* beta, const void* b_gate, const void* w_gate,
                                       float norm_eps, int raw_beta, float beta_scale, void* q_norm, void* k_norm,
                                       float* q_rnorm, float* k_rnorm, float* beta_out, float* gc, float* Aqk,
                                       float* Akk, void* operands, const float* h0, void* o, float* ht,
                                       int state_v_first, const int* chunk_offsets, const int* cu_seqlens,
                                       const int* chunk_indices, int B, int T, int N, int H, int qk_heads, int K,
                                       int V, int chunk, float scale, int value_block, int segments, void* workspace,
                                       hipStream_t stream) {
  return forward_scan_dispatch(q, k, v, g, gate_mode, raw_gate, A_log, dt_bias, has_lower_bound, lower_bound, beta,
                               b_gate, w_gate, norm_eps, raw_beta, beta_scale, q_norm, k_norm, q_rnorm, k_rnorm,
                               beta_out, gc, Aqk, Akk, operands, h0, o, ht, state_v_first, chunk_offsets, cu_seqlens,
                               chunk_indices, B, T, N, H, qk_heads, K, V, chunk, scale, value_block, segments,
                               workspace, false, stream);
}

extern "C" hipError_t fdr_forward_scan_split(const void* q, const void* k, const void* v, const void* g, int gate_mode,
                                             int raw_gate, const float* A_log, const float* dt_bias,
                                             int has_lower_bound, float lower_bound, const void* beta,
                                             const void* b_gate, const void* w_gate, float norm_eps, int raw_beta,
                                             float beta_scale, void* q_norm, void* k_norm, float* q_rnorm,
                                             float* k_rnorm, float* beta_out, float* gc, float* Aqk, float* Akk,
                                             void* operands, const float* h0, void* o, float* ht, int state_v_first,
                                             const int* chunk_offsets, const int* cu_seqlens, const int* chunk_indices,
                                             int B, int T, int N, int H, int qk_heads, int K, int V, int chunk,
                                             float scale, int value_block, int segments, void* workspace,
                                             hipStream_t stream) {
  return forward_scan_dispatch(q, k, v, g, gate_mode, raw_gate, A_log, dt_bias, has_lower_bound, lower_bound, beta,
                               b_gate, w_gate, norm_eps, raw_beta, beta_scale, q_norm, k_norm, q_rnorm, k_rnorm,
                               beta_out, gc, Aqk, Akk, operands, h0, o, ht, state_v_first, chunk_offsets, cu_seqlens,
                               chunk_indices, B, T, N, H, qk_heads, K, V, chunk, scale, value_block, segments,
                               workspace, true, stream);
}
