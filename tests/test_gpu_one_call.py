"""The one-call forms against the calls they make, bit for bit: fdr_forward_scan (fdr_fwd_prepare_scan +
fdr_fwd_scan_o; dense, packed aligned, packed with partial chunks, V-first states) and
fdr_scalar_bwd_affine (the affine-step backward of GDN / DeltaNet); and the packed tables' copy behind other work."""
import pytest
import torch

from tests._inputs import make_inputs

pytestmark = pytest.mark.gpu

GATE = {"delta": 0, "gdn": 1, "kda": 2, "gdn2": 2}


@pytest.mark.parametrize("op", list(GATE))
@pytest.mark.parametrize("lens", [None, (64, 128), (65, 1, 62)])
def test_forward_call(op, lens):
    from rewy_amd import ops
    B, T, H = (2, 128, 2) if lens is None else (1, sum(lens), 2)
    print(f"\n[forward call] {op} lens={lens}", flush=True)
    xs, _ = make_inputs(op, B, T, H, seed=71)
    xs = {n: x.cuda() for n, x in xs.items()}
    vl = None if lens is None else ops.Varlen([0, *torch.tensor(lens).cumsum(0).tolist()], xs["q"].device)
    N, gm = B if lens is None else len(lens), GATE[op]
    h0 = torch.randn(N, H, 128, 128, generator=torch.Generator().manual_seed(2)).cuda()
    kw = dict(beta=xs.get("beta"), b=xs.get("b"), w=xs.get("w"), scale=0.088, varlen=vl)
    gc, Aqk, Akk, operands = ops.fwd_prepare_scan(xs["q"], xs["k"], xs["v"], xs.get("g"), gm, **kw)
    want = ops.fwd_scan_o(operands, gm, B, T, H, 0.088, h0=h0, want_final=True, state_v_first=True, varlen=vl)
    got = ops.forward_scan(xs["q"], xs["k"], xs["v"], xs.get("g"), gm, h0=h0, want_final=True, state_v_first=True, **kw)
    torch.cuda.synchronize()
    sv = got[2]
    for a, r in zip((*got[:2], sv["gc"], sv["Aqk"], sv["Akk"]), (*want, gc, Aqk, Akk)):
        assert (a is None and r is None) or torch.equal(a, r)


def test_forward_call_takes_the_tile_it_is_given(monkeypatch):
    """value_block on a packed batch is the caller's, the rule's only without one; other widths are refused."""
    from rewy_amd import ops
    xs, _ = make_inputs("kda", 1, 130, 2, seed=71)
    xs = {n: x.cuda() for n, x in xs.items() if n != "initial_state"}
    vl = ops.Varlen([0, 65, 130], xs["q"].device)
    run = lambda **kw: ops.forward_scan(xs["q"], xs["k"], xs["v"], xs["g"], 2, beta=xs["beta"], **kw)  # noqa: E731
    asked = []
    real = ops.packed_tile
    monkeypatch.setattr(ops, "packed_tile", lambda *a: (asked.append(a), real(*a))[1])
    want = run(varlen=vl)[0]
    assert len(asked) == 1
    for vb in (16, 32, 64):
        assert torch.equal(run(varlen=vl, value_block=vb)[0], want)
    assert len(asked) == 1
    xd = {n: x[:, :128].contiguous() for n, x in xs.items()}
    for x, batch in ((xs, vl), (xd, None)):
        for vb in (8, 48, -16):
            with pytest.raises(ValueError):
                ops.forward_scan(x["q"], x["k"], x["v"], x["g"], 2, beta=x["beta"], varlen=batch, value_block=vb)


@pytest.mark.parametrize("op", ["delta", "gdn"])
@pytest.mark.parametrize("vf,states", [(False, True), (True, True), (False, False)])
def test_affine_backward_call(op, vf, states, monkeypatch):
    from rewy_amd import ops
    from rewy_amd.backends import backward as bw
    from rewy_amd.hip_forward import chunk_forward_hip
    B, T, H = 2, 64 * 11, 2
    print(f"\n[affine call] {op} vf={vf} states={states}", flush=True)
    xs, dO = make_inputs(op, B, T, H, seed=73)
    xs = {n: x.cuda() for n, x in xs.items()}
    h0 = xs["initial_state"] if states else None
    dht = torch.randn(B, H, 128, 128, generator=torch.Generator().manual_seed(4)).cuda() if states else None
    _, _, sv = chunk_forward_hip(op, xs["q"], xs["k"], xs["v"], g=xs.get("g"), beta=xs["beta"], initial_state=h0,
                                 state_v_first=vf, keep="matrices")
    kw = dict(q=xs["q"], k=xs["k"], v=xs["v"], beta=xs["beta"], A=sv["Akk"], scale=sv["scale"], initial_state=h0,
              do=dO.cuda(), dht=dht, state_v_first=vf, beta_sigmoid=1.0)
    run = (lambda: bw.gdn_backward(g=sv["gc"], **kw)) if op == "gdn" else (lambda: bw.delta_backward(**kw))
    calls = []
    real = ops.scalar_bwd_affine
    monkeypatch.setattr(ops, "scalar_bwd_affine", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    got = run()
    assert calls, "the one-call form did not run"
    monkeypatch.setattr(ops, "SCALAR_ONE_CALL", False)
    want = run()
    torch.cuda.synchronize()
    for i, (a, r) in enumerate(zip(got, want)):
        assert (a is None and r is None) or torch.equal(a, r), i


def test_packed_tables_behind_other_work():
    """Without ``wait`` the tables' copy waits for nothing and nothing overwrites its source before it ran:
    many batches enqueued behind a long kernel each hold their own tables."""
    from rewy_amd import ops
    dev = torch.device("cuda")
    x = torch.randn(4096, 4096, device=dev)
    for _ in range(20):
        x = x @ x * 1e-2
    tables = [ops.Varlen([0, 10 + i, 200 + 3 * i], dev, wait=False) for i in range(50)]
    torch.cuda.synchronize()
    for i, t in enumerate(tables):
        cu = [0, 10 + i, 200 + 3 * i]
        nch = [-(-(b - a) // 64) for a, b in zip(cu, cu[1:])]
        assert t.cu_seqlens.tolist() == cu and t.chunk_offsets.tolist() == [0, nch[0], sum(nch)]
        assert t.chunk_indices.tolist() == [[n, j] for n, m in enumerate(nch) for j in range(m)]


def test_packed_tables_are_ready_for_any_stream():
    """A Varlen made behind a long kernel on one stream is read on another without a wait between them."""
    from rewy_amd import ops
    dev = torch.device("cuda")
    side = torch.cuda.Stream()
    cu = [0, 100, 164, 300]
    want = [[0, 0], [0, 1], [1, 0], [2, 0], [2, 1], [2, 2]]
    stale = torch.full((64,), -1, device=dev, dtype=torch.int32)     # what a table not yet copied would show
    torch.cuda.synchronize()
    del stale
    torch.cuda._sleep(100_000_000)
    vl = ops.Varlen(cu, dev)
    with torch.cuda.stream(side):
        got = [x.clone() for x in (vl.cu_seqlens, vl.chunk_offsets, vl.chunk_indices)]
    side.synchronize()
    assert got[0].tolist() == cu and got[1].tolist() == [0, 2, 3, 6] and got[2].tolist() == want
    torch.cuda.synchronize()
