"""The chunked forward on the gfx950 kernels (the optimized backend's forward).

Stands where the reference calls FLA's ``chunk_kda_fwd`` / ``chunk_gdn2_fwd`` /
``chunk_gated_delta_rule_fwd`` / ``chunk_delta_rule_fwd`` (reference
``_compat/kda.py:89-113``, ``_compat/gdn.py:33-123``, ``_compat/gdn2.py:87-108``)
and returns the same (o, final_state, saved) as ``rewy_amd.forward.chunk_forward``
(its PyTorch restatement, used by the original backend and on the CPU):

  1. ``fdr_fwd_prepare_wu`` -- gc (log2 chunk-local cumsum), Aqk, Akk = (I + M)^-1, w, u
     (and kg, qg for vector gates);
  2. ``fdr_fwd_h``          -- per-chunk states h, v_new and the final state;
  3. ``fdr_fwd_o``          -- o = scale (q 2^gc) h + Aqk v_new.

Where no backward reads the states (recompute policy, inference) two launches instead:
``fdr_fwd_prepare_scan`` (step 1 with the scan's operands in the scan's order) and
``fdr_fwd_scan_o`` (steps 2-3 in one sweep, the states kept on the chip), made by one library
call (``fdr_forward_scan``).

No fallback: a missing HIP library raises.
"""
from __future__ import annotations

import torch

from . import ops

GATE_MODE = {"delta": ops.GATE_NONE, "gdn": ops.GATE_SCALAR, "kda": ops.GATE_VECTOR, "gdn2": ops.GATE_VECTOR}


def _as(x, dtype):
    if x.dtype is dtype and x.is_contiguous():      # (the common case, without a call into torch)
        return x
    return x.to(dtype).contiguous()


STATES_MIN_CHUNKS = 64


def _states_form(N, H, HQ, NT, keep, act):
    """The state scan's form where a forward that keeps no states is still faster with the scan's own
    pass and ``fwd_o``, or None: the affine-step form, for inference (``keep`` None) without activations
    (``act``) on the short rows of one to four heads that ``ops.scan_segments`` does not split.  The form's
    several library calls are host time, its steps shorter.  Whole eager calls (us, affine-step / the scan that
    forms the output): DeltaNet H=4 48 chunks 74 / 65, 64 chunks 74 / 81, 95 chunks 99 / 114; KDA H=1 48 chunks
    80 / 75, 64 chunks 80 / 94, 95 chunks 96 / 130; with raw q, k and beta KDA H=2 64 chunks 112 / 89, 95 chunks
    113 / 121 (waited for after each call 193 / 165); forward and backward KDA H=2 64 chunks 365 / 312, 95 chunks
    368 / 318, DeltaNet H=4 95 chunks 269 / 241."""
    if keep is None and not act and HQ == H and N * H <= 4 and NT >= STATES_MIN_CHUNKS \
            and ops.scan_segments(N, H, NT) == 1:
        return "affine"
    return None


def chunk_forward_hip(op, q, k, v, g=None, beta=None, b=None, w=None, initial_state=None, scale=None,
                      output_final_state=False, varlen=None, state_v_first=False, fuse_scan=False, want_qg=True,
                      gate=None, keep="all", norm=False, beta_act=None):
    """``varlen`` (an ``ops.Varlen``): B = 1 holds sequences packed along T, starting
    anywhere (FLA's cu_seqlens); initial / final states are per sequence, and every stage
    takes the batch's chunk map (a sequence's last chunk may be partial).  ``state_v_first``:
    initial / final states are [N,H,V,K] (read and written so by ``fwd_h``); the saved
    per-chunk h stays [B,NT,H,K,V].  ``fuse_scan`` (``keep`` "all"): w / u in the scan (``fdr_fwd_h_wy``,
    the same bits, u not materialized: saved ``u`` is None).  No operator asks for it: step 1 forms w / u at a
    third of ``fdr_prepare_wu``'s cost, which leaves the sweep nothing for a vector gate (KDA B=8 T=4096 H=16
    738 us, with the sweep 827), and the other families' forward keeps no states.
    ``gate`` (KDA) = (lower_bound, A_log, dt_bias): g is the raw gate, activated inside step 1.
    ``want_qg=False``: saved ``qg`` is None (only a backward that recomputes nothing reads it).

    ``keep``: "all" saves every intermediate; "matrices" only gc, Akk and, for a vector gate,
    Aqk (a backward that recomputes the rest), None nothing (no backward) -- then the states never leave the chip and
    the output is formed in the scan (``ops.forward_scan``).

    ``norm``: q and k (bf16) are raw and L2-normalised first, ``beta_act`` = s: beta is the raw input of
    s * sigmoid(beta) -- on load in step 1 where the states stay on the chip, else by passes of their
    own.  Saved then also hold what the backward reads: the normalised q, k with their rows' 1 / norm
    rq, rk, and the activated beta."""
    if fuse_scan and keep != "all":
        raise ValueError('fuse_scan: the sweep keeps the states (keep="all")')
    B, T, HQ, K = q.shape
    scale = K ** -0.5 if scale is None else scale
    gm = GATE_MODE[op]
    bf, f32 = torch.bfloat16, torch.float32
    q, k, v = _as(q, bf), _as(k, bf), _as(v, bf)
    g = None if gm == ops.GATE_NONE else _as(g, g.dtype if gate is not None else f32)
    vb = op == "gdn2"
    beta = None if vb else _as(beta, beta.dtype if beta_act and beta.dtype is bf else f32)
    b = _as(b, bf) if vb else None
    w = _as(w, bf) if vb else None
    h0 = None if initial_state is None else _as(initial_state, f32)
    vec = gm == ops.GATE_VECTOR
    N, H = (B if varlen is None else varlen.N), v.shape[2]
    form = "auto" if varlen is None else "direct"
    split = varlen is None and ops.split_pays(N, H, T // ops.CHUNK)
    if keep != "all" and varlen is None:
        form = _states_form(N, H, HQ, T // ops.CHUNK, keep, norm or beta_act)
    if keep != "all" and (varlen is not None or form is None):
        o, final, saved = ops.forward_scan(q, k, v, g, gm, beta=beta, b=b, w=w, scale=scale, h0=h0,
                                           want_final=output_final_state, state_v_first=state_v_first, varlen=varlen,
                                           gate=gate, want_saved=keep is not None, norm=norm, beta_act=beta_act,
                                           split=split)
        saved["scale"] = scale
        return o, final, saved
    rq = rk = None
    if norm:
        from .norm import l2norm_fwd
        (q, rq), (k, rk) = l2norm_fwd(q), l2norm_fwd(k)
    if beta_act:
        from .gates import beta_sigmoid
        beta = beta_sigmoid(beta, beta_act, native=True)
    if fuse_scan:
        if gate is not None:
            from .gates import kda_gate
            g = kda_gate(g, gate[1], gate[2], gate[0], native=True)
        gc, Aqk, Akk = ops.fwd_prepare(q, k, g, gm, beta=beta, b=b, scale=scale, varlen=varlen)
        wu = ops.fwd_h_wy(k, v, Akk, gc, gm, beta=beta, q=q if vec else None, b=b, w=w, h0=h0,
                          want_final=output_final_state, varlen=varlen, state_v_first=state_v_first)
        wu["u"] = None
        h, v_new, final = wu["h"], wu["v_new"], wu["final"]
    else:
        gc, Aqk, Akk, wu = ops.fwd_prepare_wu(q, k, v, g, gm, beta=beta, b=b, w=w, scale=scale, varlen=varlen,
                                              want_qg=vec and want_qg, gate=gate)
        h, v_new, final = ops.fwd_h(wu["kg"] if vec else k, wu["w"], wu["u"], gc, gm, h0=h0,
                                    want_final=output_final_state, varlen=varlen,
                                    method=form, state_v_first=state_v_first, split=split)
    o = ops.fwd_o(q, gc, gm, Aqk, h, v_new, scale, varlen=varlen)
    saved = dict(gc=gc, Aqk=Aqk, Akk=Akk, w=wu["w"], u=wu["u"], qg=wu["qg"], kg=wu["kg"], v_new=v_new, h=h,
                 scale=scale)
    if norm:
        saved.update(q=q, k=k, rq=rq, rk=rk)
    if beta_act:
        saved["beta"] = beta
    return o, final, saved
