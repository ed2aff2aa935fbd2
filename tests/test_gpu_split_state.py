"""v_new taken into the state as bf16 hi + lo (fdr_fwd_h_split, fdr_forward_scan_split) where the affine-step
form would otherwise run: the two forms' bits against each other, and the precision of the public forward's
final state against the affine-step form's.

That form adds kg^T u to the state in fp32; one bf16 rounding of v_new in its place is an error of 2^-9 of
v_new's part of the state, 12 to 18 % on top of the final state's 2.8e-3 to 3.3e-3 against fp64.  Two forms
without it differ by the sampling of their roundings, below 1 % over the 32768 values and more of a state."""
import pytest
import torch

from oracle import delta_oracle as O
from tests._inputs import make_inputs

pytestmark = pytest.mark.gpu

GATE = {"delta": 0, "gdn": 1, "kda": 2, "gdn2": 2}


@pytest.mark.parametrize("op,B,NT,H,groups,vf,h0", [
    ("delta", 1, 3, 2, 1, False, True), ("gdn", 2, 5, 4, 2, True, True), ("kda", 1, 4, 3, 1, True, False),
    ("kda", 1, 1, 2, 2, False, True), ("gdn2", 2, 7, 1, 1, False, False)])
def test_split_forms_agree(op, B, NT, H, groups, vf, h0):
    from rewy_amd import ops
    print(f"\n[split] {op} B={B} NT={NT} H={H} groups={groups} vf={vf}", flush=True)
    T, gm = 64 * NT, GATE[op]
    xs, _ = make_inputs(op, B, T, H, seed=81, gate="mild")
    xs = {n: x.cuda() for n, x in xs.items()}
    q, k = (xs[n][:, :, :H // groups].contiguous() for n in ("q", "k"))
    side = dict(beta=xs.get("beta"), b=xs.get("b"), w=xs.get("w"), scale=0.088)
    s0 = xs["initial_state"] * 10 if h0 else None
    gc, _, _, wu = ops.fwd_prepare_wu(q, k, xs["v"], xs.get("g"), gm, **side)
    scan = lambda **kw: ops.fwd_h(wu["kg"] if gm == 2 else k, wu["w"], wu["u"], gc, gm, h0=s0,  # noqa: E731
                                  want_final=True, state_v_first=vf, split=True, **kw)
    whole = lambda **kw: ops.forward_scan(q, k, xs["v"], xs.get("g"), gm, h0=s0, want_final=True,  # noqa: E731
                                          state_v_first=vf, split=True, **side, **kw)
    h, v_new, final = scan(method="direct")
    plain = ops.fwd_h(wu["kg"] if gm == 2 else k, wu["w"], wu["u"], gc, gm, h0=s0, want_final=True, state_v_first=vf,
                      method="direct")
    torch.cuda.synchronize()
    rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())  # noqa: E731
    assert torch.equal(h[:, 0], plain[0][:, 0]) and torch.equal(v_new[:, :64], plain[1][:, :64])
    assert 0 < rel(final, plain[2]) <= 4e-3           # one bf16 rounding of v_new apart
    for vb in (16, 32, 64):
        for a, r in zip(scan(method="direct", value_block=vb), (h, v_new, final)):
            assert torch.equal(a, r), vb
        o, ht, _ = whole(value_block=vb, segments=1)
        assert torch.equal(ht, final), vb
        for segs in {2, NT} - set(range(NT + 1, 3)):
            o2, ht2, _ = whole(value_block=vb, segments=segs)
            assert torch.equal(o2[:, :64 * (NT // segs)], o[:, :64 * (NT // segs)])
            a = scan(method="segmented", segments=segs, value_block=vb)
            assert torch.equal(a[0][:, :NT // segs], h[:, :NT // segs])
            assert max(rel(ht2, final), rel(a[2], final), rel(o2, o), rel(a[1], v_new)) <= 8e-3, (vb, segs)


@pytest.mark.parametrize("op,T,H,keep", [
    ("delta", 512, 2, None), ("gdn", 512, 2, "matrices"), ("kda", 512, 2, None), ("gdn2", 1024, 3, "matrices"),
    ("kda", 1024, 16, "all"), ("gdn2", 576, 9, "all"), ("gdn", 64 * 64, 4, None), ("delta", 64 * 96, 2, None),
    ("kda", 64 * 128, 4, "all")])
def test_final_state_is_as_precise_as_the_affine_step_form(op, T, H, keep):
    from rewy_amd import ops
    from rewy_amd.hip_forward import chunk_forward_hip
    print(f"\n[split] precision {op} T={T} H={H} keep={keep}", flush=True)
    gm = GATE[op]
    xs, _ = make_inputs(op, 1, T, H, seed=83, gate="mild")
    xs = {n: x.cuda() for n, x in xs.items()}
    h0 = xs["initial_state"]
    side = dict(beta=xs.get("beta"), b=xs.get("b"), w=xs.get("w"))
    _, final, _ = chunk_forward_hip(op, xs["q"], xs["k"], xs["v"], g=xs.get("g"), initial_state=h0,
                                    output_final_state=True, keep=keep, **side)
    gc, _, _, wu = ops.fwd_prepare_wu(xs["q"], xs["k"], xs["v"], xs.get("g"), gm, **side)
    affine = ops.fwd_h(wu["kg"] if gm == 2 else xs["k"], wu["w"], wu["u"], gc, gm, h0=h0, want_final=True,
                       method="affine")[2]
    with torch.no_grad():
        want = O.torch_token_recurrence(op, {n: x.double() for n, x in xs.items()})[1]
    rel = lambda a: float((a.double() - want).norm() / want.norm())  # noqa: E731
    print(f"{rel(final):.3e} affine {rel(affine):.3e}", flush=True)
    assert rel(final) <= 1.02 * rel(affine)


def test_split_takes_dense_rows():
    from rewy_amd import ops
    xs, _ = make_inputs("kda", 1, 128, 1, seed=3)
    q, k, v, g, beta = (xs[n].cuda() for n in ("q", "k", "v", "g", "beta"))
    vl = ops.Varlen([0, 64, 128], q.device)
    with pytest.raises(ValueError):
        ops.forward_scan(q, k, v, g, 2, beta=beta, varlen=vl, split=True)
    with pytest.raises(ValueError):
        ops.fwd_h(k, k, v, g, 2, varlen=vl, split=True)
