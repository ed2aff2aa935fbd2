// Chunk-parallel pieces of the delta-rule forward.
//
// Replace, per chunk-head, the parts of FLA's chunk_kda_fwd / chunk_gdn2_fwd /
// chunk_gated_delta_rule_fwd / chunk_delta_rule_fwd (reference
// _compat/kda.py:89-113, _compat/gdn.py:33-123, _compat/gdn2.py:87-108) that
// are not the state scan:
//
//   fdr_fwd_prepare, fdr_fwd_prepare_wu, fdr_fwd_prepare_scan (one work-group per chunk-head):
//     gc  = chunk-local cumsum of the raw (natural-log) gate, times 1/ln 2   (FLA chunk_local_cumsum)
//     Aqk = scale tril(q k^T 2^(g_i - g_s))                                 (diagonal included)
//     Akk = (I + strict_tril((b k) k^T 2^(g_i - g_s)))^-1                  (FLA chunk_*_fwd_intra + solve_tril)
//     and (fdr_fwd_prepare_wu) w = Akk (b k 2^g), u = Akk (w_gate v), qg, kg as fdr_prepare_wu
//   fdr_fwd_o (one work-group per chunk-head):
//     o   = scale (q 2^g) h_c + Aqk v_new                                   (FLA chunk_fwd_o)
//
// The state scan between them is fdr_fwd_h (recompute.hip); fdr_fwd_scan_o (fwd_scan.hip) is the scan
// and the output in one.
//
// Gate products.  A scalar gate's 2^(g_i - g_s) multiplies the finished fp32 tile.  A vector
// gate's: for rows i of 16-row block I and rows s of block J <= I the
// per-channel factor 2^(g_i - g_s) is split at the anchor n = 16 I (the first
// row of block I): q 2^(g_i - g_n) <= 1 and k 2^(g_n - g_s) (<= 1 for J < I),
// both split into bf16 hi + lo so each 16 x 16 tile is three MFMAs per 32-wide
// slice of K (16-bit operand mantissas, the lo x lo term dropped).  A diagonal block whose gate span reaches 100 in
// log2 units (where the k-side factor could overflow) is evaluated pairwise in
// fp32 instead.
#include "rewy_amd.h"

#include "scan_body.hpp"

namespace rewy {

enum GateModeF { FG_NONE = 0, FG_SCALAR = 1, FG_VECTOR = 2 };

namespace fwd {
constexpr int LDM = C + 4;      // fp32 pitch of the 64 x 64 matrices
constexpr float RCP_LN2 = 1.4426950408889634f;
constexpr float WIDE = 100.f;   // diagonal-block gate span that takes the pairwise path
}  // namespace fwd

// LDS of fwd_prepare.  Three lives of the same bytes: the staged rows and gates (dead once the
// 16 x 16 tiles and E are formed), the inverse's matrices with E and Z beside them, and A's hi / lo
// rows over M and T for the WY products.  73 KiB at most, so two work-groups share a CU.
template <int GATE, bool VEC_B, bool WY>
struct PrepareSmem {
  static constexpr bool VEC = GATE == FG_VECTOR;
  struct In {
    bf16 k[C * KD];                    // rows, swizzled (tr_off<16>)
    bf16 b[VEC_B ? C * KD : 8];
    float g[VEC ? C * KD : 4];         // log2 cumsum rows (gx_off)
    float tot[VEC ? 8 * KD : 4];       // sums of each wave's 8 rows
  };
  struct Inv {
    float M[C][fwd::LDM];    // strict_tril(b k k^T 2^(g_i-g_s)), the lower tiles
    float T[32][36];         // products of the block inverse
    float X[C][fwd::LDM];    // (I + M)^-1
    bf16 e[WY ? C * KD : 8]; // E = b k 2^g rows (swizzled)
    bf16 z[WY ? C * VD : 8]; // Z = w_gate v rows (swizzled)
  };
  struct Wy {
    bf16 ah[C][C + 8];       // Akk rows, bf16 hi and lo
    bf16 al[C][C + 8];
  };
  static_assert(sizeof(Wy) <= sizeof(float) * (C * fwd::LDM + 32 * 36), "A's rows lie over M and T");
  union {
    In in;
    Inv inv;
    Wy wy;
  };
  float gs[C];               // scalar gate (log2 cumsum) per row
  float beta[C];
};

// element offset in the fp32 gate tile [64][128]: 16-byte chunk c of row r at chunk c ^ (r & 15),
// so the same chunk of 16 rows, which one fragment read touches, lies in 16 distinct bank groups
__device__ __forceinline__ int gx_off(int r, int col) { return r * KD + ((((col >> 2) ^ (r & 15))) << 2) + (col & 3); }

// WU: 0 the intra matrices only (fdr_fwd_prepare); 1 also w, u and, for a vector gate, kg; 2 also qg
// (fdr_fwd_prepare_wu); 3 the operands of fdr_fwd_scan_o in its own layout (sop) in place of w, u and
// kg, gc / Aqk / Akk where asked for (fdr_fwd_prepare_scan; B=8 T=4096 H=16 KDA 410 us with all
// three, 350 without, against 357 for WU = 1, whose scan and output passes then cost 176 us more).
//
// Bound by HBM traffic and by the chain load -> cumsum -> tiles -> inverse -> WY products of a
// work-group; two work-groups a CU overlap their chains.  Forming w / u here, from the inverse while
// it is in LDS, drops prepare_wu's launch and its re-reads of k, g and Akk: at B=8 T=4096 H=16 KDA
// (no qg) 360 us, 4.4 TB/s, against 268 + 264 us for the two; GDN 226 against 146 + 150; GDN2
// B=2 T=8192 H=32 397 against 276 + 308 (its fwd_prepare had taken 453 at one work-group a CU).
//
// RAW (KDA with WU): graw is the raw gate input (1 fp32, 2 bf16), activated here (act), so the
// activated gate never goes to HBM (KDA prefill B=1 T=8192 H=32, bf16 gate: 688 -> 552 us, of which
// the activation pass alone had taken 146 us).
struct GateAct {
  const float* A_log;      // [H], null in mode 2
  const float* dt_bias;    // [H*K] or null
  float lower_bound;
  int mode;                // kda_gate_act's
};

// WU = 3 also takes q / k before their L2 normalisation and beta before its sigmoid (InputAct): the
// normalisation and the sigmoid then ride on the loads, in fdr_l2norm_fwd's and fdr_beta_sigmoid_fwd's
// arithmetic, instead of in passes of their own over q and k (two reads, two writes and three launches).
// The kernel is bound by its loads' latency at two work-groups a CU, so the sums hide; with nothing saved
// the passes' traffic goes altogether, else the normalised rows are still written for the backward.
// Whole calls (us, passes of their own / on load): KDA prefill T=8192 H=32 437 / 397, GDN prompt of 301
// tokens H=16 114 / 94, forward + backward of KDA B=4 T=4096 H=16 1123 / 1119, of packed GDN T=9226 H=16
// 614 / 600.
struct InputAct {
  float norm_eps;          // > 0: q, k raw
  bf16 *qn, *kn;           // normalised q, k [B,T,HQ,K] and their 1 / norm [B,T,HQ] for the backward, or null
  float *rq, *rk;
  int raw_beta;            // 1 fp32, 2 bf16: beta = beta_scale sigmoid(raw)
  float beta_scale;
  float* beta_out;         // activated beta for the backward, or null
};

template <int GATE, bool VEC_B, bool MAP, int WU, int RAW = 0>
__global__ __launch_bounds__(512, 4) void fwd_prepare_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k, const bf16* __restrict__ v,
    const void* __restrict__ graw_, const float* __restrict__ beta, const bf16* __restrict__ bgate,
    const bf16* __restrict__ wgate, float* __restrict__ gc_out, float* __restrict__ aqk_out,
    float* __restrict__ akk_out, bf16* __restrict__ w_out, bf16* __restrict__ u_out, bf16* __restrict__ qg_out,
    bf16* __restrict__ kg_out, char* __restrict__ sop_out, int T, int H, int HQ, float scale, const int* __restrict__ cu,
    const int* __restrict__ ci, GateAct act, InputAct in) {
  static_assert(!RAW || (GATE == FG_VECTOR && !VEC_B && WU), "the raw gate is KDA's, in the one-pass form");
  const float* __restrict__ graw = reinterpret_cast<const float*>(graw_);
  constexpr bool VEC = GATE == FG_VECTOR, WY = WU > 0, SOP = WU == 3;
  using fwd::LDM;
  using SM = PrepareSmem<GATE, VEC_B, WY>;
  __shared__ __attribute__((aligned(16))) SM sm;
  bf16* sk = sm.in.k;
  bf16* sb = sm.in.b;
  float* sg = sm.in.g;
  auto& sgs = sm.gs;
  auto& sbeta = sm.beta;
  auto& sM = sm.inv.M;
  auto& sX = sm.inv.X;
  auto& sT = sm.inv.T;

  const int blk = blockIdx.x;
  const int NT = T / C;
  // heads run fastest: work-groups in flight together read neighbouring heads of
  // the same tokens, i.e. contiguous HBM rows
  const int h = blk % H;
  const int c = (blk / H) % NT;
  const int b = blk / (H * NT);
  const int tid = threadIdx.x, l = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_id());
  const int lc = l & 15, lg = l >> 4;
  const Rows<MAP> rw = chunk_rows<MAP>(cu, ci, b, c, T);
  const size_t tok0 = rw.tok0;
  const size_t rsk = (size_t)H * KD;
  const size_t kofs = tok0 * rsk + (size_t)h * KD;
  const size_t mofs = (tok0 * H + h) * C;      // [t][64] matrices of this chunk-head
  const size_t rsm = (size_t)H * C;
  const QKRows qr = qk_rows(tok0, h, H, HQ);   // q / k rows (grouped value heads: HQ < H)
  char* const sop = SOP ? sop_out + (size_t)blk * sop::BYTES : nullptr;

  // Tiles (I, J), J <= I, over the waves: wave -> (row block I, first column block J0, tile
  // count); the two waves with two tiles form the row operands of block I once for both.
  const int I = wv == 0 || wv == 2 || wv == 3 ? 3 : wv == 1 || wv == 4 ? 2 : wv == 7 ? 0 : 1;
  const int J0 = wv == 2 ? 2 : wv == 3 ? 3 : wv == 4 ? 2 : wv == 6 ? 1 : 0;
  const int NJ = wv < 2 ? 2 : 1;

  // ---- loads first, all in flight together ----
  float2 gv[8];                                // vector gate: columns 2 (tid & 63), rows 8 wv ..
  const int gcol = 2 * l;
  uint32_t gb[8];                              // (RAW 2: two bf16)
  float2 gbias = {0.f, 0.f};
  float ga_log = 0.f;
  if constexpr (RAW == 2) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      gb[r] = *reinterpret_cast<const uint32_t*>(
          rw.src(reinterpret_cast<const bf16*>(graw_) + kofs + (size_t)(8 * wv + r) * rsk + gcol, 8 * wv + r));
  }
  if constexpr (RAW != 0) {
    if (act.dt_bias) gbias = load2(act.dt_bias + h * KD + gcol);
    if (act.A_log) ga_log = act.A_log[h];
  }
  if constexpr (VEC && RAW != 2) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      gv[r] = load2(rw.src(graw + kofs + (size_t)(8 * wv + r) * rsk + gcol, 8 * wv + r));
  }
  float gx = 0.f;
  if constexpr (GATE == FG_SCALAR) gx = *rw.src(graw + (tok0 + l) * H + h, l);
  u32x4 rk[2], rb[2], rv[2], rwg[2];
  float rbt[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = tid + 512 * i, t = p >> 4, c8 = (p & 15) * 8;
    rk[i] = *reinterpret_cast<const u32x4*>(rw.src(k + qr.ofs + (size_t)t * qr.rs + c8, t));
    if constexpr (VEC_B) rb[i] = *reinterpret_cast<const u32x4*>(rw.src(bgate + kofs + (size_t)t * rsk + c8, t));
    else if (SOP && in.raw_beta == 2)
      rbt[i] = to_f32(*rw.src(reinterpret_cast<const bf16*>(beta) + (tok0 + t) * H + h, t));
    else rbt[i] = *rw.src(beta + (tok0 + t) * H + h, t);
  }
  // q's operand rows straight from HBM (each read by the one to three waves of its row block)
  bf16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    qf[ks] = *reinterpret_cast<const bf16x8*>(
        rw.src(q + qr.ofs + (size_t)(16 * I + lc) * qr.rs + 32 * ks + 8 * lg, 16 * I + lc));
  if constexpr (WY) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + 512 * i, t = p >> 4, c8 = (p & 15) * 8;
      rv[i] = *reinterpret_cast<const u32x4*>(rw.src(v + kofs + (size_t)t * rsk + c8, t));
      if constexpr (VEC_B) rwg[i] = *reinterpret_cast<const u32x4*>(rw.src(wgate + kofs + (size_t)t * rsk + c8, t));
    }
  }

  const int HG = H / HQ;                       // value heads a q / k head serves; the first stores for it
  float rq_ = 1.f;                             // 1 / norm of this lane's operand row of q
  if constexpr (SOP) {
    if (!VEC_B && in.raw_beta) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int p = tid + 512 * i, t = p >> 4;
        rbt[i] = rw.ok(t) ? in.beta_scale * sigmoid_y(exp_f(rbt[i])) : 0.f;
        if (in.beta_out && (p & 15) == 0) *rw.dst(in.beta_out + (tok0 + t) * H + h, t) = rbt[i];
      }
    }
    if (in.norm_eps > 0.f) {
      const bool first = h % HG == 0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {            // k: a row's 16 pieces in 16 lanes
        const int p = tid + 512 * i, t = p >> 4;
        bf16x8 x = __builtin_bit_cast(bf16x8, rk[i]);
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) s += to_f32(x[j]) * to_f32(x[j]);
        s = sum_row16(s);
        const float r = 1.f / sqrtf(s + in.norm_eps);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = to_bf16(to_f32(x[j]) * r);
        rk[i] = __builtin_bit_cast(u32x4, x);
        if (in.kn && first) {
          *reinterpret_cast<u32x4*>(rw.dst(in.kn + qr.ofs + (size_t)t * qr.rs + 8 * (p & 15), t)) = rk[i];
          if ((p & 15) == 0) *rw.dst(in.rk + (tok0 + t) * HQ + h / HG, t) = r;
        }
      }
      float s = 0.f;                           // q: a row's operand slices in the lanes lc + 16 lg
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int j = 0; j < 8; ++j) s += to_f32(qf[ks][j]) * to_f32(qf[ks][j]);
      s = sum_lane_groups(s);
      rq_ = 1.f / sqrtf(s + in.norm_eps);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[ks][j] = to_bf16(to_f32(qf[ks][j]) * rq_);
    }
  }

  // ---- gate cumsum (log2 units); k (, b) rows into LDS ----
  if constexpr (VEC) {
    if constexpr (RAW != 0) {
      const float a = act.mode == 2 ? 1.f : expf(ga_log);
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        if constexpr (RAW == 2)
          gv[r] = {__builtin_bit_cast(float, gb[r] << 16), __builtin_bit_cast(float, gb[r] & 0xffff0000u)};
        // (a missing row's gate is zero, not the activation of zero)
        gv[r].x = rw.ok(8 * wv + r) ? kda_gate_act(act.mode, gv[r].x + gbias.x, a, act.lower_bound) : 0.f;
        gv[r].y = rw.ok(8 * wv + r) ? kda_gate_act(act.mode, gv[r].y + gbias.y, a, act.lower_bound) : 0.f;
      }
    }
    // wave wv sums its 8 rows, the carries come from the waves before it
#pragma unroll
    for (int r = 1; r < 8; ++r) {
      gv[r].x += gv[r - 1].x;
      gv[r].y += gv[r - 1].y;
    }
    *reinterpret_cast<float2*>(sm.in.tot + wv * KD + gcol) = gv[7];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = tid + 512 * i, t = p >> 4;
    store_tr_chunk<16>(sk, t, p & 15, rk[i]);
    if constexpr (VEC_B) store_tr_chunk<16>(sb, t, p & 15, rb[i]);
    else if ((p & 15) == 0) sbeta[t] = rbt[i];
  }
  if constexpr (VEC) {
    lds_barrier();
    float2 carry = {0.f, 0.f};
    for (int pp = 0; pp < wv; ++pp) {
      const float2 s = *reinterpret_cast<const float2*>(sm.in.tot + pp * KD + gcol);
      carry.x += s.x;
      carry.y += s.y;
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int t = 8 * wv + r;
      const float2 x = {(gv[r].x + carry.x) * fwd::RCP_LN2, (gv[r].y + carry.y) * fwd::RCP_LN2};
      *reinterpret_cast<float2*>(sg + gx_off(t, gcol)) = x;
      if (!SOP || gc_out) *reinterpret_cast<f32x2u*>(rw.dst(gc_out + kofs + (size_t)t * rsk + gcol, t)) = f32x2u{x.x, x.y};
      if (SOP && t == C - 1)
        *reinterpret_cast<float2*>(sop + sop::LAM + 4 * gcol) = float2{fast_exp2(x.x), fast_exp2(x.y)};
    }
  } else if constexpr (GATE == FG_SCALAR) {
    if (wv == 0) {
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const float y = __shfl_up(gx, d);
        if (l >= d) gx += y;
      }
      gx *= fwd::RCP_LN2;
      sgs[l] = gx;
      if (!SOP || gc_out) *rw.dst(gc_out + (tok0 + l) * H + h, l) = gx;
    }
  }
  // Z = w_gate v (bf16), held until the staged rows' LDS is free
  bf16x8 zh[2];
  if constexpr (WY) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bf16x8 vx = __builtin_bit_cast(bf16x8, rv[i]);
      bf16x8 wx = {};
      if constexpr (VEC_B) wx = __builtin_bit_cast(bf16x8, rwg[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) zh[i][j] = to_bf16((VEC_B ? to_f32(wx[j]) : rbt[i]) * to_f32(vx[j]));
    }
  }
  lds_barrier();

  // 8 consecutive gate values of a row (two 16-byte reads)
  auto gate8 = [&](int t, int k0, float (&x)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(sg + gx_off(t, k0));
    const f32x4 d = *reinterpret_cast<const f32x4*>(sg + gx_off(t, k0 + 4));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[j] = a[j];
      x[j + 4] = d[j];
    }
  };

  // ---- 16 x 16 tiles (I, J), J <= I: Aqk and M, formed transposed: lane: row i = 16 I + lc,
  // four consecutive columns s = 16 J + 4 lg + r ----
  f32x4 mkk[2] = {zero4(), zero4()};
  f32x4 aqk[2] = {zero4(), zero4()};
  if constexpr (!VEC) {
    // The scalar gate's factor leaves the product: exact bf16 products, one MFMA a slice, and
    // scale 2^(g_i - g_s), beta_i 2^(g_i - g_s) (exponents <= 0) on the fp32 results.
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8 ka = frag_row<16>(sk, 16 * I, 32 * ks);
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        if (jj >= NJ) break;                  // wave-uniform
        const bf16x8 kb = frag_row<16>(sk, 16 * (J0 + jj), 32 * ks);
        aqk[jj] = mfma(kb, qf[ks], aqk[jj]);
        mkk[jj] = mfma(kb, ka, mkk[jj]);
      }
    }
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      if (jj >= NJ) break;
      const int i = 16 * I + lc;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int s = 16 * (J0 + jj) + 4 * lg + r;
        float f = 1.f;
        if constexpr (GATE == FG_SCALAR) f = fast_exp2(sgs[i] - sgs[s]);
        aqk[jj][r] *= f;
        mkk[jj][r] *= sbeta[i] * f;
      }
    }
  } else {
    const int n = 16 * I;                       // anchor row
    // a diagonal block whose gate span (first row - last row: the gates are cumsums of log decays)
    // reaches WIDE over some channel goes pairwise; its one wave decides
    bool pairwise = false;
    if (NJ == 1 && J0 == I) {
      const float2 a = *reinterpret_cast<const float2*>(sg + gx_off(n, gcol));
      const float2 d = *reinterpret_cast<const float2*>(sg + gx_off(n + 15, gcol));
      pairwise = __any(fmaxf(a.x - d.x, a.y - d.y) >= fwd::WIDE);
    }
    if (!pairwise) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int k0 = 32 * ks + 8 * lg;
        const int ia = 16 * I + lc;             // A rows (i)
        bf16x8 qh, ql, bh_, bl;
        float gn[8];
        gate8(n, k0, gn);
        {
          float ga[8];
          gate8(ia, k0, ga);
          const bf16x8 ka = frag_row<16>(sk, 16 * I, 32 * ks);
          bf16x8 ba = {};
          if constexpr (VEC_B) ba = frag_row<16>(sb, 16 * I, 32 * ks);
          const float be = VEC_B ? 0.f : sbeta[ia];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float fa = fast_exp2(ga[j] - gn[j]);                  // <= 1
            bf16 hh, ll;
            split_bf16(to_f32(qf[ks][j]) * fa, hh, ll);
            qh[j] = hh;
            ql[j] = ll;
            split_bf16((VEC_B ? to_f32(ba[j]) : be) * to_f32(ka[j]) * fa, hh, ll);
            bh_[j] = hh;
            bl[j] = ll;
          }
        }
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
          if (jj >= NJ) break;                  // wave-uniform
          float gs_[8];
          gate8(16 * (J0 + jj) + lc, k0, gs_);  // B columns (s)
          const bf16x8 kb = frag_row<16>(sk, 16 * (J0 + jj), 32 * ks);
          bf16x8 kh, kl;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            bf16 hh, ll;
            split_bf16(to_f32(kb[j]) * fast_exp2(gn[j] - gs_[j]), hh, ll);   // factor <= 1 off the diagonal
            kh[j] = hh;
            kl[j] = ll;
          }
          aqk[jj] = mfma(kh, qh, aqk[jj]);
          aqk[jj] = mfma(kl, qh, aqk[jj]);
          aqk[jj] = mfma(kh, ql, aqk[jj]);
          mkk[jj] = mfma(kh, bh_, mkk[jj]);
          mkk[jj] = mfma(kl, bh_, mkk[jj]);
          mkk[jj] = mfma(kh, bl, mkk[jj]);
        }
      }
    } else {
      // exact pairwise diagonal: lane (lg, lc) owns row 16 I + lc, columns s = 16 I + 4 lg + r
      const int i = 16 * I + lc;
#pragma unroll 1
      for (int r = 0; r < 4; ++r) {
        const int s = 16 * I + 4 * lg + r;
        float a = 0.f, m = 0.f;
        if (s <= i) {
#pragma unroll 4
          for (int kc = 0; kc < KD; ++kc) {
            const float f = fast_exp2(sg[gx_off(i, kc)] - sg[gx_off(s, kc)]);
            const float ks_ = to_f32(sk[tr_off<16>(s, kc)]);
            float qi = to_f32(*rw.src(q + qr.ofs + (size_t)i * qr.rs + kc, i));
            if (SOP && in.norm_eps > 0.f) qi = to_f32(to_bf16(qi * rq_));
            a += qi * ks_ * f;
            const float bi = VEC_B ? to_f32(sb[tr_off<16>(i, kc)]) : sbeta[i];
            m += bi * to_f32(sk[tr_off<16>(i, kc)]) * ks_ * f;
          }
        }
        aqk[0][r] = a;
        mkk[0][r] = m;
      }
    }
  }
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    if (jj >= NJ) break;
    const int i = 16 * I + lc, s0 = 16 * (J0 + jj) + 4 * lg;
    f32x4 a;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = s0 + r <= i ? scale * aqk[jj][r] : 0.f;
    if (!SOP || aqk_out) *reinterpret_cast<f32x4*>(rw.dst(aqk_out + mofs + (size_t)i * rsm + s0, i)) = a;
    if constexpr (SOP) {
      bf16x4 lo;
      const bf16x4 hi = split_hi4(a, lo);
      bf16* fa = reinterpret_cast<bf16*>(sop + sop::A) + sop::frag_off(i, 2 * (s0 & 32) + (s0 & 31), 4);
      *reinterpret_cast<bf16x4*>(fa) = hi;
      *reinterpret_cast<bf16x4*>(fa + 64 * 8) = lo;
    }
  }
  // zero upper tiles of Aqk (J > I): 6 tiles of 64 16-byte pieces; of the operand fragments the two
  // that lie in a slice the scan reads
  if (tid < 384) {
    const int tix = tid >> 6, e = tid & 63;
    const int I_ = tix < 3 ? 0 : tix < 5 ? 1 : 2;
    const int J_ = I_ + 1 + (tix - (I_ == 0 ? 0 : I_ == 1 ? 3 : 5));
    const int i = 16 * I_ + (e >> 2), s0 = 16 * J_ + 4 * (e & 3);
    if (!SOP || aqk_out) *reinterpret_cast<f32x4*>(rw.dst(aqk_out + mofs + (size_t)i * rsm + s0, i)) = zero4();
    if constexpr (SOP) {
      if (J_ == (I_ | 1)) {
        bf16* fa = reinterpret_cast<bf16*>(sop + sop::A) + sop::frag_off(i, 2 * (s0 & 32) + (s0 & 31), 4);
        *reinterpret_cast<bf16x4*>(fa) = bf16x4{};
        *reinterpret_cast<bf16x4*>(fa + 64 * 8) = bf16x4{};
      }
    }
  }
  if constexpr (SOP) {
    // q's operand fragments from the rows this wave holds: each (row block, slice) once, the waves
    // with two tiles spared
    constexpr uint32_t SLICES = 0xFC3EC310u;    // four bits a wave
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (!((SLICES >> (4 * wv + ks)) & 1)) continue;      // wave-uniform
      bf16* fq_ = reinterpret_cast<bf16*>(sop + sop::Q) + ((I * 4 + ks) * 64 + l) * 8;
      if (in.qn && h % HG == 0) {
        const int t = 16 * I + lc;
        *reinterpret_cast<bf16x8*>(rw.dst(in.qn + qr.ofs + (size_t)t * qr.rs + 32 * ks + 8 * lg, t)) = qf[ks];
        if (ks == 1 && lg == 0) *rw.dst(in.rq + (tok0 + t) * HQ + h / HG, t) = rq_;   // (one wave a row block has slice 1)
      }
      if constexpr (VEC) {
        float ga[8];
        gate8(16 * I + lc, 32 * ks + 8 * lg, ga);
        bf16x8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          bf16 hh, ll;
          split_bf16(to_f32(qf[ks][j]) * fast_exp2(ga[j]), hh, ll);
          hi[j] = hh;
          lo[j] = ll;
        }
        *reinterpret_cast<bf16x8*>(fq_) = hi;
        *reinterpret_cast<bf16x8*>(fq_ + (sop::QL - sop::Q) / 2) = lo;
      } else {
        *reinterpret_cast<bf16x8*>(fq_) = qf[ks];
      }
    }
    if constexpr (!VEC) {
      if (tid < C)
        reinterpret_cast<float*>(sop + sop::FQ)[tid] = GATE == FG_SCALAR ? scale * fast_exp2(sgs[tid]) : scale;
      else if (tid < C + KD)
        reinterpret_cast<float*>(sop + sop::LAM)[tid - C] = GATE == FG_SCALAR ? fast_exp2(sgs[rw.clamp(C - 1)]) : 1.f;
    }
  }
  // E = b k 2^g (bf16), and kg = k 2^(g_last - g), qg = q 2^g to HBM (vector gates)
  bf16x8 eh[2];
  if constexpr (WY) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + 512 * i, t = p >> 4, ch = p & 15;
      const bf16x8 kx = *reinterpret_cast<const bf16x8*>(sk + tr_off<16>(t, 8 * ch));
      if constexpr (VEC) {
        float gt[8], gl[8];
        gate8(t, 8 * ch, gt);
        gate8(C - 1, 8 * ch, gl);
        bf16x8 bx = {}, ok;
        if constexpr (VEC_B) bx = *reinterpret_cast<const bf16x8*>(sb + tr_off<16>(t, 8 * ch));
        const float be = VEC_B ? 0.f : sbeta[t];
        float ge[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          ge[j] = fast_exp2(gt[j]);
          eh[i][j] = to_bf16((VEC_B ? to_f32(bx[j]) : be) * to_f32(kx[j]) * ge[j]);
          ok[j] = to_bf16(to_f32(kx[j]) * fast_exp2(gl[j] - gt[j]));
        }
        if constexpr (SOP)
          *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16*>(sop + sop::K) + tr_off<16>(t, 8 * ch)) = ok;
        else
          *reinterpret_cast<bf16x8*>(rw.dst(kg_out + kofs + (size_t)t * rsk + 8 * ch, t)) = ok;
        if constexpr (WU == 2) {
          const bf16x8 qx = __builtin_bit_cast(
              bf16x8, *reinterpret_cast<const u32x4*>(rw.src(q + qr.ofs + (size_t)t * qr.rs + 8 * ch, t)));
          bf16x8 oq;
#pragma unroll
          for (int j = 0; j < 8; ++j) oq[j] = to_bf16(to_f32(qx[j]) * ge[j]);
          *reinterpret_cast<bf16x8*>(rw.dst(qg_out + kofs + (size_t)t * rsk + 8 * ch, t)) = oq;
        }
      } else {
        const float ge = GATE == FG_SCALAR ? fast_exp2(sgs[t]) : 1.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) eh[i][j] = to_bf16(sbeta[t] * to_f32(kx[j]) * ge);
        if constexpr (SOP) {
          // kg = k 2^(g_last - g), rounded as the other scans round it
          const u32x4 kr = __builtin_bit_cast(u32x4, kx);
          *reinterpret_cast<u32x4*>(reinterpret_cast<bf16*>(sop + sop::K) + tr_off<16>(t, 8 * ch)) =
              GATE == FG_SCALAR ? scale_bf16x8(kr, fast_exp2(sgs[rw.clamp(C - 1)] - sgs[t])) : kr;
        }
      }
    }
  }
  lds_barrier();                                // staged rows and gates dead: M, X, E and Z take their LDS
  // M tiles from the accumulators.  The inverse reads nothing of M on or above the diagonal.
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    if (jj >= NJ) break;
    *reinterpret_cast<f32x4*>(&sM[16 * I + lc][16 * (J0 + jj) + 4 * lg]) = mkk[jj];
  }
  if constexpr (WY) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + 512 * i;
      store_tr_chunk<16>(sm.inv.e, p >> 4, p & 15, __builtin_bit_cast(u32x4, eh[i]));
      store_tr_chunk<16>(sm.inv.z, p >> 4, p & 15, __builtin_bit_cast(u32x4, zh[i]));
    }
  }
  // the two upper blocks of the inverse that the block products read, zero
  if (tid < 128) {
    const int e = tid & 63, o = 32 * (tid >> 6);
    *reinterpret_cast<f32x4*>(&sX[o + (e >> 2)][o + 16 + 4 * (e & 3)]) = zero4();
  }
  lds_barrier();

  // ---- inverse of the unit lower-triangular I + M (fp32) ----
  // diagonal 16 x 16 blocks by forward substitution: wave 0, lane = (block, column)
  if (wv == 0) {
    const int B4 = lg, j = lc, base = 16 * B4;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float acc = (i == j) ? 1.f : 0.f;
#pragma unroll
      for (int m = 0; m < i; ++m) acc -= sM[base + i][base + m] * x[m];
      x[i] = acc;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sX[base + i][base + j] = x[i];
  }
  lds_barrier();
  // Off-diagonal blocks by doubling, [[A, 0], [C, D]]^-1 = [[A^-1, 0], [-D^-1 C A^-1, D^-1]]:
  // first inside the two 32 x 32 diagonal blocks, then for the 64 x 64 whole (C = M off the
  // diagonal).  Each product is spread over all 512 threads (one or two outputs each),
  // with fixed trip counts (the zero upper parts of X and M are summed as zeros) and
  // 16-byte reads of the row operand.
  auto rowdot = [&](const float* row, const float* col, int pitch, int n) -> float {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int m = 0; m < 32; m += 4) {
      if (m >= n) break;
      const f32x4 r4 = *reinterpret_cast<const f32x4*>(row + m);
      a0 += r4[0] * col[(m + 0) * pitch];
      a1 += r4[1] * col[(m + 1) * pitch];
      a0 += r4[2] * col[(m + 2) * pitch];
      a1 += r4[3] * col[(m + 3) * pitch];
    }
    return a0 + a1;
  };
  {
    // P = M_{r,r-1} X_{r-1,r-1}, r = 1, 3
    const int q2 = tid >> 8, e = tid & 255, i = e >> 4, j = e & 15;
    const int cb = 32 * q2, rb_ = cb + 16;
    sT[16 * q2 + i][j] = rowdot(&sM[rb_ + i][cb], &sX[cb][cb + j], LDM, 16);
  }
  lds_barrier();
  {
    // X_{r,r-1} = -X_{r,r} P
    const int q2 = tid >> 8, e = tid & 255, i = e >> 4, j = e & 15;
    const int rb_ = 32 * q2 + 16;
    sX[rb_ + i][rb_ - 16 + j] = -rowdot(&sX[rb_ + i][rb_], &sT[16 * q2][j], 36, 16);
  }
  lds_barrier();
  // T = M_BL X_TL (rows 32..63, columns 0..31)
#pragma unroll
  for (int k2 = 0; k2 < 2; ++k2) {
    const int o = tid + 512 * k2, i = o >> 5, j = o & 31;
    sT[i][j] = rowdot(&sM[32 + i][0], &sX[0][j], LDM, 32);
  }
  lds_barrier();
  // X_BL = -X_BR T
#pragma unroll
  for (int k2 = 0; k2 < 2; ++k2) {
    const int o = tid + 512 * k2, i = o >> 5, j = o & 31;
    sX[32 + i][j] = -rowdot(&sX[32 + i][32], &sT[0][j], 36, 32);
  }
  lds_barrier();
  // ---- Akk rows -> HBM, and their bf16 hi / lo over M and T ----
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = tid + 512 * i;
    const int t = p >> 4, ch = p & 15;
    const f32x4 a = 4 * ch <= t ? tril_piece(*reinterpret_cast<const f32x4*>(&sX[t][4 * ch]), t, ch) : zero4();
    if (!SOP || akk_out) *reinterpret_cast<f32x4*>(rw.dst(akk_out + mofs + (size_t)t * rsm + 4 * ch, t)) = a;
    if constexpr (WY) {
      bf16x4 lo;
      const bf16x4 hi = split_hi4(a, lo);
      *reinterpret_cast<bf16x4*>(&sm.wy.ah[t][4 * ch]) = hi;
      *reinterpret_cast<bf16x4*>(&sm.wy.al[t][4 * ch]) = lo;
    }
  }
  if constexpr (WY) {
    lds_barrier();
    // ---- w^T = E^T A^T, u^T = Z^T A^T: wave wv the k (v) rows [16 wv, 16 wv + 16), all tokens ----
    // prepare_wu_kernel's products in its order (the zero upper half of A skipped): the same bits
    constexpr int LDA = C + 8;
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      const bf16* src = which == 0 ? sm.inv.e : sm.inv.z;
      bf16* dst = SOP ? nullptr : (which == 0 ? w_out : u_out) + kofs;
      const bf16x8 x0 = frag_tr<16>(src, 0, 16 * wv);
      const bf16x8 x1 = frag_tr<16>(src, 32, 16 * wv);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        // SOP: u itself (rows t, column v), the accumulator order of the scan's u - w h
        const bool swap = SOP && which == 1;
        f32x4 acc = zero4();
        auto mm = [&](bf16x8 x, const bf16* a) {
          acc = swap ? mfma(frag(a, LDA), x, acc) : mfma(x, frag(a, LDA), acc);
        };
        mm(x0, &sm.wy.ah[16 * tt][0]);
        mm(x0, &sm.wy.al[16 * tt][0]);
        if (tt >= 2) {
          mm(x1, &sm.wy.ah[16 * tt][32]);
          mm(x1, &sm.wy.al[16 * tt][32]);
        }
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = to_bf16(acc[r]);
        if constexpr (SOP) {
          bf16* p = which == 0
                        ? reinterpret_cast<bf16*>(sop + sop::W) + sop::frag_off(16 * tt + lc, 16 * wv + 4 * lg, 4)
                        : reinterpret_cast<bf16*>(sop + sop::U) + ((tt * 8 + wv) * 64 + l) * 4;
          *reinterpret_cast<bf16x4*>(p) = o;
        } else {
          // lane: token t = 16 tt + lc, columns 16 wv + 4 lg .. +3
          *reinterpret_cast<bf16x4*>(rw.dst(dst + (size_t)(16 * tt + lc) * rsk + 16 * wv + 4 * lg, 16 * tt + lc)) = o;
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------------
// fdr_fwd_o:  o = scale (q 2^g) h_c + Aqk v_new
// ------------------------------------------------------------------------------------------
template <int GATE, bool MAP>
__global__ __launch_bounds__(512) void fwd_o_kernel(const bf16* __restrict__ q, const float* __restrict__ gc,
                                                     const float* __restrict__ aqk, const bf16* __restrict__ hst,
                                                     const bf16* __restrict__ vnew, bf16* __restrict__ o_out,
                                                     int T, int H, int HQ, float scale,
                                                     const int* __restrict__ cu, const int* __restrict__ ci) {
  // swizzled, unpadded tiles (80 KiB in all, so two work-groups share a CU)
  __shared__ __attribute__((aligned(16))) bf16 sqg[C * KD];       // scale q 2^g rows [i][k], hi
  __shared__ __attribute__((aligned(16))) bf16 sqgl[C * KD];      // lo
  __shared__ __attribute__((aligned(16))) bf16 sah[C * C];        // Aqk rows [i][s], hi
  __shared__ __attribute__((aligned(16))) bf16 sal[C * C];        // lo
  __shared__ __attribute__((aligned(16))) bf16 sv[C * VD];        // v_new rows (swizzled)
  __shared__ __attribute__((aligned(16))) bf16 shT[C * KD];       // 64 rows of h [k][v] (swizzled)
  // (q h) contracts over K = the rows of h, read transposed; h is staged in two halves.
  const int blk = blockIdx.x;
  const int NT = T / C;
  // heads run fastest: work-groups in flight together read neighbouring heads of
  // the same tokens, i.e. contiguous HBM rows
  const int h = blk % H;
  const int c = (blk / H) % NT;
  const int b = blk / (H * NT);
  const int tid = threadIdx.x, l = lane_id(), wv = wave_id();
  const int lc = l & 15, lg = l >> 4;
  const Rows<MAP> rw = chunk_rows<MAP>(cu, ci, b, c, T);
  const size_t tok0 = rw.tok0;
  const size_t rsk = (size_t)H * KD;
  const size_t kofs = tok0 * rsk + (size_t)h * KD;
  const size_t mofs = (tok0 * H + h) * C;
  const size_t rsm = (size_t)H * C;
  const size_t hoff = (((size_t)b * NT + c) * H + h) * KD * VD;

  // stage scale * q 2^g (hi/lo), Aqk (hi/lo), v_new
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = tid + 512 * i;
    const int t = p >> 4, c8 = (p & 15) * 8;
    const QKRows qr = qk_rows(tok0, h, H, HQ);
    const bf16x8 qx =
        __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(rw.src(q + qr.ofs + (size_t)t * qr.rs + c8, t)));
    bf16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float f = scale;
      if constexpr (GATE == FG_VECTOR) f *= fast_exp2(gc[kofs + (size_t)rw.clamp(t) * rsk + c8 + j]);
      else if constexpr (GATE == FG_SCALAR) f *= fast_exp2(gc[(tok0 + rw.clamp(t)) * H + h]);
      bf16 hh, ll;
      split_bf16(to_f32(qx[j]) * f, hh, ll);
      hi[j] = hh;
      lo[j] = ll;
    }
    store_tr_chunk<16>(sqg, t, p & 15, __builtin_bit_cast(u32x4, hi));
    store_tr_chunk<16>(sqgl, t, p & 15, __builtin_bit_cast(u32x4, lo));
    store_tr_chunk<16>(sv, t, p & 15, *reinterpret_cast<const u32x4*>(rw.src(vnew + kofs + (size_t)t * rsk + c8, t)));
    const int c4 = (p & 15) * 4;
    // causal: pieces above the diagonal are not fetched, elements above it are zero
    f32x4 a = *reinterpret_cast<const f32x4*>(tril_src(rw.src(aqk + mofs + (size_t)t * rsm + c4, t), t, p & 15));
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = tril_elem(a[r], t, c4 + r);
    bf16x4 alo;
    const bf16x4 ahi = split_hi4(a, alo);
    *reinterpret_cast<bf16x4*>(sah + tr_off<8>(t, c4)) = ahi;
    *reinterpret_cast<bf16x4*>(sal + tr_off<8>(t, c4)) = alo;
  }
  // wave w: output rows 16 (w & 3) .. +16, columns 64 (w >> 2) .. +64 (4 tiles)
  const int I = wv & 3, cb = 64 * (wv >> 2);
  f32x4 acc[4] = {zero4(), zero4(), zero4(), zero4()};
  for (int half = 0; half < 2; ++half) {
    lds_barrier();
    // h rows [64 half .. 64 half + 64)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + 512 * i;
      const int r = p >> 4, c8 = (p & 15) * 8;
      store_tr_chunk<16>(shT, r, p & 15, *reinterpret_cast<const u32x4*>(hst + hoff + (size_t)(64 * half + r) * VD + c8));
    }
    lds_barrier();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8 ah = frag_row<16>(sqg, 16 * I, 64 * half + 32 * ks);
      const bf16x8 al = frag_row<16>(sqgl, 16 * I, 64 * half + 32 * ks);
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        const bf16x8 bh_ = frag_tr<16>(shT, 32 * ks, cb + 16 * ct);   // h rows over K, columns v
        acc[ct] = mfma(ah, bh_, acc[ct]);
        acc[ct] = mfma(al, bh_, acc[ct]);
      }
    }
  }
  // Aqk v_new: A = Aqk rows i (s-contiguous), B = v_new rows read transposed
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const bf16x8 ah = frag_row<8>(sah, 16 * I, 32 * ks);
    const bf16x8 al = frag_row<8>(sal, 16 * I, 32 * ks);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const bf16x8 bv = frag_tr<16>(sv, 32 * ks, cb + 16 * ct);
      acc[ct] = mfma(ah, bv, acc[ct]);
      acc[ct] = mfma(al, bv, acc[ct]);
    }
  }
  // lane: rows 16 I + 4 lg + r, column cb + 16 ct + lc
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *rw.dst(o_out + kofs + (size_t)(16 * I + 4 * lg + r) * rsk + cb + 16 * ct + lc, 16 * I + 4 * lg + r) =
          to_bf16(acc[ct][r]);
}

}  // namespace rewy

using namespace rewy;

// B rows of T tokens (cu == nullptr), or (cu, ci) a packed batch of NC chunks, T = NC * 64.
// w != nullptr: w, u (and kg, optionally qg, for a vector gate) too.  raw_gate: g is KDA's raw gate
// (1 fp32, 2 bf16), activated as act says.
template <bool MAP>
static hipError_t fwd_prepare_launch(const void* q, const void* k, const void* v, const void* g, int gate_mode,
                                     const float* beta, const void* b_gate, const void* w_gate, float* gc, float* Aqk,
                                     float* Akk, void* w, void* u, void* qg, void* kg, int B, int T, int H,
                                     int qk_heads, float scale, hipStream_t stream, const int* cu, const int* ci,
                                     int raw_gate = 0, GateAct act = {}, void* sop = nullptr, InputAct in = {}) {
  const int HQ = qk_heads > 0 ? qk_heads : H;
  if (H % HQ || (b_gate && HQ != H)) return hipErrorInvalidValue;
  if (!q || !k || (!sop && (!Aqk || !Akk))) return hipErrorInvalidValue;
  if (gate_mode != FG_NONE && (!g || (!sop && !gc))) return hipErrorInvalidValue;
  const bool vec_b = b_gate != nullptr, vec = gate_mode == FG_VECTOR;
  if (vec_b && !vec) return hipErrorInvalidValue;
  if (!vec_b && !beta) return hipErrorInvalidValue;
  if (sop && (w || !v || (vec_b && !w_gate))) return hipErrorInvalidValue;
  if (w && (!v || !u || vec != (kg != nullptr) || (vec_b && !w_gate))) return hipErrorInvalidValue;
  if (qg && (!w || !vec)) return hipErrorInvalidValue;
  if (raw_gate && ((!w && !sop) || !vec || vec_b || raw_gate < 0 || raw_gate > 2)) return hipErrorInvalidValue;
  if (raw_gate && act.mode != 2 && !act.A_log) return hipErrorInvalidValue;
  const dim3 grid(B * H * (T / C)), block(512);
#define FDR_PREP_R(G, VB, WU, RAW)                                                                              \
  hipLaunchKernelGGL((fwd_prepare_kernel<G, VB, MAP, WU, RAW>), grid, block, 0, stream, (const bf16*)q,         \
                     (const bf16*)k, (const bf16*)v, g, beta, (const bf16*)b_gate, (const bf16*)w_gate, gc, Aqk, \
                     Akk, (bf16*)w, (bf16*)u, (bf16*)qg, (bf16*)kg, (char*)sop, T, H, HQ, scale, cu, ci, act, in)
#define FDR_PREP(G, VB, WU) FDR_PREP_R(G, VB, WU, 0)
#define FDR_PREP_V(VB)                          \
  if (!w) FDR_PREP(FG_VECTOR, VB, 0);           \
  else if (!qg) FDR_PREP(FG_VECTOR, VB, 1);     \
  else FDR_PREP(FG_VECTOR, VB, 2)
  if (sop) {
    if (raw_gate == 1) FDR_PREP_R(FG_VECTOR, false, 3, 1);
    else if (raw_gate == 2) FDR_PREP_R(FG_VECTOR, false, 3, 2);
    else if (vec_b) FDR_PREP(FG_VECTOR, true, 3);
    else if (vec) FDR_PREP(FG_VECTOR, false, 3);
    else if (gate_mode == FG_SCALAR) FDR_PREP(FG_SCALAR, false, 3);
    else if (gate_mode == FG_NONE) FDR_PREP(FG_NONE, false, 3);
    else return hipErrorInvalidValue;
  } else if (raw_gate == 1) {
    if (qg) FDR_PREP_R(FG_VECTOR, false, 2, 1);
    else FDR_PREP_R(FG_VECTOR, false, 1, 1);
  } else if (raw_gate == 2) {
    if (qg) FDR_PREP_R(FG_VECTOR, false, 2, 2);
    else FDR_PREP_R(FG_VECTOR, false, 1, 2);
  } else if (vec_b) {
    FDR_PREP_V(true);
  } else if (vec) {
    FDR_PREP_V(false);
  } else if (gate_mode == FG_SCALAR) {
    if (w) FDR_PREP(FG_SCALAR, false, 1);
    else FDR_PREP(FG_SCALAR, false, 0);
  } else if (gate_mode == FG_NONE) {
    if (w) FDR_PREP(FG_NONE, false, 1);
    else FDR_PREP(FG_NONE, false, 0);
  } else {
    return hipErrorInvalidValue;
  }
#undef FDR_PREP_V
#undef FDR_PREP
#undef FDR_PREP_R
  return hipGetLastError();
}

template <bool MAP>
static hipError_t fwd_o_launch(const void* q, const float* gc, int gate_mode, const float* Aqk, const void* h,
                               const void* v_new, void* o, int B, int T, int H, int qk_heads, float scale,
                               hipStream_t stream, const int* cu, const int* ci) {
  const int HQ = qk_heads > 0 ? qk_heads : H;
  if (H % HQ) return hipErrorInvalidValue;
  if (!q || !Aqk || !h || !v_new || !o) return hipErrorInvalidValue;
  if (gate_mode != FG_NONE && !gc) return hipErrorInvalidValue;
  const dim3 grid(B * H * (T / C)), block(512);
#define FDR_O(G)                                                                                           \
  hipLaunchKernelGGL((fwd_o_kernel<G, MAP>), grid, block, 0, stream, (const bf16*)q, gc, Aqk, (const bf16*)h, \
                     (const bf16*)v_new, (bf16*)o, T, H, HQ, scale, cu, ci)
  if (gate_mode == FG_VECTOR) FDR_O(FG_VECTOR);
  else if (gate_mode == FG_SCALAR) FDR_O(FG_SCALAR);
  else if (gate_mode == FG_NONE) FDR_O(FG_NONE);
  else return hipErrorInvalidValue;
#undef FDR_O
  return hipGetLastError();
}

extern "C" hipError_t fdr_fwd_prepare(const void* q, const void* k, const float* g, int gate_mode,
                                      const float* beta, const void* b_gate, float* gc, float* Aqk, float* Akk,
                                      int B, int T, int H, int qk_heads, int K, int chunk, float scale,
                                      hipStream_t stream) {
  if (K != KD || chunk != C || T <= 0 || T % C || B <= 0 || H <= 0) return hipErrorInvalidValue;
  return fwd_prepare_launch<false>(q, k, nullptr, g, gate_mode, beta, b_gate, nullptr, gc, Aqk, Akk, nullptr, nullptr,
                                   nullptr, nullptr, B, T, H, qk_heads, scale, stream, nullptr, nullptr);
}

extern "C" hipError_t fdr_fwd_prepare_varlen(const void* q, const void* k, const float* g, int gate_mode,
                                             const float* beta, const void* b_gate, float* gc, float* Aqk,
                                             float* Akk, const int* cu_seqlens, const int* chunk_indices,
                                             int num_chunks, int H, int qk_heads, int K, int chunk, float scale,
                                             hipStream_t stream) {
  if (K != KD || chunk != C || num_chunks <= 0 || H <= 0 || !cu_seqlens || !chunk_indices)
    return hipErrorInvalidValue;
  return fwd_prepare_launch<true>(q, k, nullptr, g, gate_mode, beta, b_gate, nullptr, gc, Aqk, Akk, nullptr, nullptr,
                                  nullptr, nullptr, 1, num_chunks * C, H, qk_heads, scale, stream, cu_seqlens,
                                  chunk_indices);
}

extern "C" hipError_t fdr_fwd_prepare_wu(const void* q, const void* k, const void* v, const void* g, int gate_mode,
                                         int raw_gate, const float* A_log, const float* dt_bias,
                                         int has_lower_bound, float lower_bound, const float* beta,
                                         const void* b_gate, const void* w_gate, float* gc, float* Aqk, float* Akk,
                                         void* w, void* u, void* qg, void* kg, const int* cu_seqlens,
                                         const int* chunk_indices, int B, int T, int H, int qk_heads, int K, int V,
                                         int chunk, float scale, hipStream_t stream) {
  if (K != KD || V != VD || chunk != C || T <= 0 || T % C || B <= 0 || H <= 0 || !w) return hipErrorInvalidValue;
  if ((cu_seqlens == nullptr) != (chunk_indices == nullptr) || (cu_seqlens && B != 1)) return hipErrorInvalidValue;
  const GateAct act{A_log, dt_bias, lower_bound, has_lower_bound ? (A_log ? 1 : 2) : 0};
  if (cu_seqlens)
    return fwd_prepare_launch<true>(q, k, v, g, gate_mode, beta, b_gate, w_gate, gc, Aqk, Akk, w, u, qg, kg, 1, T, H,
                                    qk_heads, scale, stream, cu_seqlens, chunk_indices, raw_gate, act);
  return fwd_prepare_launch<false>(q, k, v, g, gate_mode, beta, b_gate, w_gate, gc, Aqk, Akk, w, u, qg, kg, B, T, H,
                                   qk_heads, scale, stream, nullptr, nullptr, raw_gate, act);
}

extern "C" size_t fdr_scan_operands_bytes(int num_chunks, int H) { return (size_t)num_chunks * H * sop::BYTES; }

extern "C" hipError_t fdr_fwd_prepare_scan(const void* q, const void* k, const void* v, const void* g, int gate_mode,
                                           int raw_gate, const float* A_log, const float* dt_bias,
                                           int has_lower_bound, float lower_bound, const void* beta,
                                           const void* b_gate, const void* w_gate, float norm_eps, int raw_beta,
                                           float beta_scale, void* q_norm, void* k_norm, float* q_rnorm,
                                           float* k_rnorm, float* beta_out, float* gc, float* Aqk, float* Akk,
                                           void* operands, const int* cu_seqlens, const int* chunk_indices, int B,
                                           int T, int H, int qk_heads, int K, int V, int chunk, float scale,
                                           hipStream_t stream) {
  if (!(norm_eps >= 0.f) || raw_beta < 0 || raw_beta > 2 || (raw_beta && b_gate)) return hipErrorInvalidValue;
  const bool qk_out = q_norm != nullptr;
  if ((k_norm != nullptr) != qk_out || (q_rnorm != nullptr) != qk_out || (k_rnorm != nullptr) != qk_out ||
      (qk_out && norm_eps == 0.f) || (beta_out && !raw_beta))
    return hipErrorInvalidValue;
  const InputAct in{norm_eps, (bf16*)q_norm, (bf16*)k_norm, q_rnorm, k_rnorm, raw_beta, beta_scale, beta_out};
  if (K != KD || V != VD || chunk != C || T <= 0 || T % C || B <= 0 || H <= 0 || !operands)
    return hipErrorInvalidValue;
  if (!aligned16(operands)) return hipErrorInvalidValue;
  if ((cu_seqlens == nullptr) != (chunk_indices == nullptr) || (cu_seqlens && B != 1)) return hipErrorInvalidValue;
  const GateAct act{A_log, dt_bias, lower_bound, has_lower_bound ? (A_log ? 1 : 2) : 0};
  if (cu_seqlens)
    return fwd_prepare_launch<true>(q, k, v, g, gate_mode, (const float*)beta, b_gate, w_gate, gc, Aqk, Akk, nullptr,
                                    nullptr, nullptr, nullptr, 1, T, H, qk_heads, scale, stream, cu_seqlens, chunk_indices,
                                    raw_gate, act, operands, in);
  return fwd_prepare_launch<false>(q, k, v, g, gate_mode, (const float*)beta, b_gate, w_gate, gc, Aqk, Akk, nullptr,
                                   nullptr, nullptr, nullptr, B, T, H, qk_heads, scale, stream, nullptr, nullptr,
                                   raw_gate, act, operands, in);
}

extern "C" hipError_t fdr_fwd_o(const void* q, const float* gc, int gate_mode, const float* Aqk, const void* h,
                                const void* v_new, void* o, int B, int T, int H, int qk_heads, int K, int V,
                                int chunk, float scale, hipStream_t stream) {
  if (K != KD || V != VD || chunk != C || T <= 0 || T % C || B <= 0 || H <= 0) return hipErrorInvalidValue;
  return fwd_o_launch<false>(q, gc, gate_mode, Aqk, h, v_new, o, B, T, H, qk_heads, scale, stream, nullptr, nullptr);
}

extern "C" hipError_t fdr_fwd_o_varlen(const void* q, const float* gc, int gate_mode, const float* Aqk,
                                       const void* h, const void* v_new, void* o, const int* cu_seqlens,
                                       const int* chunk_indices, int num_chunks, int H, int qk_heads, int K, int V,
                                       int chunk, float scale, hipStream_t stream) {
  if (K != KD || V != VD || chunk != C || num_chunks <= 0 || H <= 0 || !cu_seqlens || !chunk_indices)
    return hipErrorInvalidValue;
  return fwd_o_launch<true>(q, gc, gate_mode, Aqk, h, v_new, o, 1, num_chunks * C, H, qk_heads, scale, stream,
                            cu_seqlens, chunk_indices);
}
