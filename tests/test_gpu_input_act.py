"""q / k normalised and beta activated on the prepare kernel's loads (fdr_forward_scan with norm / beta_act)
against the separate kernels (fdr_l2norm_fwd, fdr_beta_sigmoid_fwd) in front of it, and fdr_qk_norm_bwd
against two fdr_l2norm_bwd.

k and beta go through the same arithmetic in the same order: the same bits.  q's row sum is taken in the
operand's order: 128 fp32 terms, so its 1 / norm within 2^-17 of the other and its bf16 rows within one
rounding step (2^-7 of the value at most).  What the scan forms from q is linear in it: o, Aqk within
2^-7 of each product's factor, over 128 terms of either sign at most sqrt(128) 2^-8 of the largest, and o's
own bf16 rounding."""
import pytest
import torch

from tests._inputs import make_inputs

pytestmark = pytest.mark.gpu

GATE = {"delta": 0, "gdn": 1, "kda": 2, "gdn2": 2}
CASES = [(op, 1, 64, 1, 1, "default", None, torch.float32) for op in GATE]
CASES += [(op, 2, 192, 4, 2, "default", None, torch.bfloat16) for op in ("delta", "gdn", "kda")]
CASES += [(op, 1, 193, 2, 1, "default", (1, 65, 0, 127), torch.bfloat16) for op in GATE]
CASES += [("kda", 1, 128, 2, 2, "wide", None, torch.float32), ("kda", 1, 97, 2, 1, "wide", (34, 63), torch.float32)]


def _raw(x, seed):
    s = torch.rand(*x.shape[:-1], 1, generator=torch.Generator().manual_seed(seed)) * 3
    s.view(-1)[5] = 0.0                                   # a zero row
    return (x.float() * s).bfloat16()


@pytest.mark.parametrize("op,B,T,H,groups,gate,lens,dt", CASES)
def test_inputs_on_load(op, B, T, H, groups, gate, lens, dt):
    from rewy_amd import ops
    from rewy_amd.gates import beta_sigmoid
    from rewy_amd.norm import l2norm_fwd
    print(f"\n[input act] {op} B={B} T={T} H={H} groups={groups} gate={gate} lens={lens} {dt}", flush=True)
    xs, _ = make_inputs(op, B, T, H, seed=91, gate=gate)
    q, k = (_raw(xs[n][:, :, :H // groups], i).cuda().contiguous() for i, n in enumerate(("q", "k")))
    v, g, b, w = (None if xs.get(n) is None else xs[n].cuda() for n in ("v", "g", "b", "w"))
    act = None if op == "gdn2" else 2.0
    raw = None if act is None else torch.randn(B, T, H, generator=torch.Generator().manual_seed(6)).to(dt).cuda()
    gm = GATE[op]
    vl = None if lens is None else ops.Varlen([0, *torch.tensor(lens).cumsum(0).tolist()], q.device)
    N = B if lens is None else len(lens)
    h0 = torch.randn(N, H, 128, 128, generator=torch.Generator().manual_seed(2)).cuda() * 0.05
    kw = dict(b=b, w=w, scale=0.088, h0=h0, want_final=True, varlen=vl)
    (qn, rq), (kn, rk) = l2norm_fwd(q), l2norm_fwd(k)
    beta = None if act is None else beta_sigmoid(raw, act, native=True)
    ro, rht, rsv = ops.forward_scan(qn, kn, v, g, gm, beta=beta, **kw)
    for saved in (True, False):
        o, ht, sv = ops.forward_scan(q, k, v, g, gm, beta=raw, norm=True, beta_act=act, want_saved=saved, **kw)
        torch.cuda.synchronize()
        assert torch.equal(ht, rht)                       # q has no part in the state
        tol = 128 ** 0.5 * 2.0 ** -8 + 2.0 ** -8
        assert float((o.float() - ro.float()).abs().max()) <= tol * float(ro.float().abs().max()) + 1e-30
        if not saved:
            assert all(x is None for x in sv.values())
            continue
        assert torch.equal(sv["k"], kn) and torch.equal(sv["rk"], rk) and torch.equal(sv["Akk"], rsv["Akk"])
        assert act is None or torch.equal(sv["beta"], beta)
        assert torch.allclose(sv["rq"], rq, rtol=2.0 ** -17, atol=0)
        assert float(((sv["q"].float() - qn.float()).abs() - 2.0 ** -7 * qn.float().abs()).max()) <= 0
        if sv["Aqk"] is not None:
            d = (sv["Aqk"] - rsv["Aqk"]).abs().max()
            assert float(d) <= 128 ** 0.5 * 2.0 ** -8 * float(rsv["Aqk"].abs().max())


def test_inputs_on_load_refusals():
    from rewy_amd import ops
    xs, _ = make_inputs("gdn", 1, 64, 2, seed=1)
    xs = {n: x.cuda() for n, x in xs.items()}
    with pytest.raises((TypeError, ValueError)):          # an activated beta is fp32
        ops.forward_scan(xs["q"], xs["k"], xs["v"], xs["g"], 1, beta=xs["beta"].bfloat16())
    with pytest.raises((TypeError, ValueError)):
        ops.forward_scan(xs["q"], xs["k"], xs["v"], xs["g"], 1, beta=xs["beta"].half(), beta_act=1.0)


@pytest.mark.parametrize("shape,group", [((1, 1, 1), 1), ((1, 65, 3), 1), ((2, 2048, 4), 1), ((1, 63, 2), 4)])
def test_both_norm_backwards_in_one_launch(shape, group):
    """group = 1: the bits of fdr_l2norm_bwd.  Else dy is the fp32 sum of the group's rows: the same formula
    in fp64 on the CPU, within one bf16 rounding and the fp32 sums (128 + group terms)."""
    from rewy_amd import _lib
    from rewy_amd.norm import l2norm_fwd, qk_norm_bwd
    g_ = torch.Generator().manual_seed(8)
    q, k = (torch.randn(*shape, 128, generator=g_).bfloat16().cuda() for _ in range(2))
    dq, dk = (torch.randn(*shape[:2], shape[2] * group, 128, generator=g_).bfloat16().cuda() for _ in range(2))
    (_, rq), (_, rk) = l2norm_fwd(q), l2norm_fwd(k)
    got = qk_norm_bwd(q, rq, dq, k, rk, dk)
    P = _lib.ptr
    for x, r, d, a in ((q, rq, dq, got[0]), (k, rk, dk, got[1])):
        if group > 1:
            xd, rd = x.cpu().double(), r.cpu().double().unsqueeze(-1)
            dy = d.cpu().double().view(*shape, group, 128).sum(3)
            y = xd * rd
            want = rd * (dy - y * (y * dy).sum(-1, keepdim=True))
            tol = 2.0 ** -8 * want.abs() + (128 + group) * 2.0 ** -23 * (rd * dy.abs()).amax(-1, keepdim=True) * 2
            assert bool(((a.cpu().double() - want).abs() <= tol).all())
            continue
        want = torch.empty_like(x)
        _lib.check(_lib.load().fdr_l2norm_bwd(P(x), 1, P(r), P(d), P(want), x.numel() // 128, 128,
                                              _lib.stream_handle(x.device)), "fdr_l2norm_bwd")
        torch.cuda.synchronize()
        assert torch.equal(a, want)


@pytest.mark.parametrize("op,lens,fold", [("kda", None, False), ("kda", (1, 65, 62), False), ("kda", None, True),
                                          ("kda", (130,), True), ("gdn2", None, False), ("gdn2", (63, 65), False)])
def test_norm_backward_in_the_chunk_kernel(op, lens, fold):
    """fdr_chunk_bwd_qk_norm against fdr_chunk_bwd (or _gate_fold): everything but dq, dk the same bits; dq, dk
    the formula r (dy - y (y . dy)) of the other's dq, dk, whose bf16 rounding (2^-9 of dy) goes through
    the projection (at most twice that of dy's norm) before this one's own rounding."""
    from rewy_amd import ops
    from rewy_amd.norm import l2norm_fwd
    print(f"\n[chunk norm] {op} lens={lens} fold={fold}", flush=True)
    B, T, H = (2, 128, 3) if lens is None else (1, sum(lens), 3)
    xs, dO = make_inputs(op, B, T, H, seed=17)
    xs = {n: x.cuda() for n, x in xs.items()}
    vl = None if lens is None else ops.Varlen([0, *torch.tensor(lens).cumsum(0).tolist()], xs["q"].device)
    NC = B * T // 64 if vl is None else vl.NC
    (q, rq), (k, rk) = (l2norm_fwd(_raw(xs[n].cpu(), i).cuda()) for i, n in enumerate(("q", "k")))
    g_ = torch.Generator().manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g_).cuda()  # noqa: E731
    shape = (B, NC // B, H, 128, 128)
    h, dh = (rnd(*shape).bfloat16() * 0.1 for _ in range(2))
    v_new, dR = (rnd(B, T, H, 128).bfloat16() for _ in range(2))
    gc, _, Akk = ops.fwd_prepare(q, k, xs["g"], 2, beta=xs.get("beta"), b=xs.get("b"), scale=0.088, varlen=vl)
    kw = dict(beta=xs.get("beta"), b=xs.get("b"), w=xs.get("w"), varlen=vl)
    if fold:
        kw["gate_fold"] = dict(g_raw=rnd(B, T, H, 128).bfloat16(), A_log=rnd(H), dt_bias=rnd(H * 128), lower_bound=None)
    args = (q, k, xs["v"], v_new, dO.cuda(), dR, gc, 2, Akk, h, dh, 0.088)
    want, got = ops.chunk_bwd(*args, **kw), ops.chunk_bwd(*args, qk_rnorm=(rq, rk), **kw)
    torch.cuda.synchronize()
    for n, a in got.items():
        if n not in ("dq", "dk"):
            assert (a is None and want[n] is None) or torch.equal(a, want[n]), n
    for n, y, r in (("dq", q, rq), ("dk", k, rk)):
        dy, yd, rd = want[n].double(), y.double(), r.double().unsqueeze(-1)
        ref = rd * (dy - yd * (yd * dy).sum(-1, keepdim=True))
        tol = rd * dy.norm(dim=-1, keepdim=True) * 2.0 ** -8 + 2.0 ** -8 * ref.abs()
        assert bool(((got[n].double() - ref).abs() <= tol).all()), n


def test_norm_backward_refusals():
    from rewy_amd import ops
    xs, dO = make_inputs("gdn", 1, 64, 2, seed=1)
    xs = {n: x.cuda() for n, x in xs.items()}
    z = torch.zeros(1, 1, 2, 128, 128, device="cuda", dtype=torch.bfloat16)
    r = torch.ones(1, 64, 2, device="cuda")
    with pytest.raises(ValueError):                       # the vector-gate families'
        ops.chunk_bwd(xs["q"], xs["k"], xs["v"], xs["v"], dO.cuda(), dO.cuda(), xs["g"], 1,
                      torch.zeros(1, 64, 2, 64, device="cuda"), z, z, 0.088, beta=xs["beta"], qk_rnorm=(r, r))


@pytest.mark.parametrize("op,lens", [("kda", None), ("gdn", None), ("gdn", (65, 63))])
def test_strided_rows_are_copied_once(op, lens, monkeypatch):
    """q and k as slices of one projection: the contiguous copies that the forward reads are the ones saved for
    the backward, and the result is the contiguous rows'."""
    import rewy_amd as fdr
    from rewy_amd import ops
    xs, dO = make_inputs(op, 1, 128, 2, seed=19, h0=False)
    xs = {n: x.cuda() for n, x in xs.items()}
    qkv = torch.cat([xs[n] for n in ("q", "k", "v")], -1)
    read, saved = [], []
    real = ops.forward_scan
    monkeypatch.setattr(ops, "forward_scan", lambda q, k, *a, **kw: (read.append((q, k)),      # (kept alive)
                                                                      real(q, k, *a, **kw))[1])
    kw = dict(use_qk_l2norm_in_kernel=True)
    if lens:
        kw["cu_seqlens"] = torch.tensor([0, *lens]).cumsum(0).cuda()

    def run(q, k):
        ys = [x.detach().requires_grad_() for x in (q, k)]
        with fdr.use_backend("optimized"), torch.autograd.graph.saved_tensors_hooks(
                lambda x: (saved.append(x.data_ptr()), x)[1], lambda x: x):
            o, _ = {"kda": fdr.chunk_kda, "gdn": fdr.chunk_gated_delta_rule}[op](
                *ys, xs["v"], xs["g"], xs["beta"], **kw)
        return (o, *torch.autograd.grad(o, ys, dO.cuda()))
    got = run(qkv[..., :128], qkv[..., 128:256])
    assert len(read) == 1 and {x.data_ptr() for x in read[0]} <= set(saved)
    want = run(xs["q"], xs["k"])
    torch.cuda.synchronize()
    for a, r in zip(got, want):
        assert torch.equal(a, r)


@pytest.mark.parametrize("NT,raw", [(3, False), (3, True), (96, False)])
def test_fp32_inputs_start_at_any_float(NT, raw):
    """Gate, dt_bias and initial state as slices of flat buffers that start one float in (96 chunks: the state
    goes through the segments' chain): the aligned tensors' bits."""
    import rewy_amd as fdr
    from rewy_amd import ops
    assert (ops.scan_segments(1, 2, NT) > 1) == (NT == 96)
    xs, _ = make_inputs("kda", 1, 64 * NT, 2, seed=23, gate="mild")
    xs = {n: x.cuda() for n, x in xs.items()}
    kw = {}
    if raw:
        xs["g"] = _raw(xs["g"].cpu(), 3).float().cuda()
        kw = dict(use_gate_in_kernel=True, A_log=torch.zeros(2, device="cuda"),
                  dt_bias=torch.linspace(-1, 1, 256, device="cuda"))

    def shifted(x):
        flat = torch.empty(x.numel() + 1, device=x.device, dtype=x.dtype)
        y = flat[1:].view(x.shape)
        y.copy_(x)
        assert y.is_contiguous() and y.data_ptr() % 8 == 4
        return y

    def run(f):
        a = {n: f(x) if n in ("g", "initial_state") else x for n, x in xs.items()}
        b = {n: f(x) if n == "dt_bias" else x for n, x in kw.items() if n != "use_gate_in_kernel"}
        with fdr.use_backend("optimized"), torch.no_grad():
            return fdr.chunk_kda(**a, **b, use_gate_in_kernel=raw, output_final_state=True)
    got, want = run(shifted), run(lambda x: x)
    torch.cuda.synchronize()
    for a, r in zip(got, want):
        assert torch.equal(a, r)
