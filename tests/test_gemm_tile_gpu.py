"""q3_gemm: ragged sizes, K-major operands, pieces and K splits against fp64 products, and the fused
epilogues bit for bit against the plain product followed by the separate kernel."""
import pytest
import torch

from _util import max_rel, randn, seeded
from test_gemm_plan import KINDS, SHAPES as PLANNED, pieces, planned

from qwen3_triton import _hip as H
from qwen3_triton.kernels import _ops
from qwen3_triton.kernels.linear import gemm, matmul

pytestmark = pytest.mark.gpu
# one rounding of the fp32 sum to the storage type: half an ulp of the largest value, 2^-9 (bf16) / 2^-12 (fp16)
TOL = {torch.bfloat16: 4e-3, torch.float16: 5e-4}


def guarded(m, n, dtype):
    """An [m, n] output inside a larger buffer of sevens: what lies outside must stay."""
    buf = torch.full((m + 3, n + 16), 7.0, device="cuda", dtype=dtype)
    return buf, buf[:m, :n]


def untouched(buf, m, n):
    return bool((buf[m:] == 7).all()) and bool((buf[:, n:] == 7).all())


# edges of the 32 / 64 / 128 / 256 tiles and of the 64-wide k-tile, single rows, long k (splits), many tiles
SHAPES = [(1, 8, 8), (17, 64, 72), (33, 136, 64), (65, 4096, 4096), (128, 1024, 1032), (257, 264, 200),
          (333, 4096, 1024), (2050, 4104, 328), (40, 512, 12288)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("layout", ["NT", "NN", "TN"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_layouts(m, n, k, layout, dtype):
    if layout == "TN":   # the weight gradient's shape: features x features over a ragged token count
        m, k = -(-k // 8) * 8, m
    print(f"q3_gemm {layout} {m}x{n}x{k} {dtype}", flush=True)
    gen = seeded(m + 3 * n + k)
    a, b = randn(m, k, gen=gen, dtype=dtype).cuda(), randn(n, k, gen=gen, dtype=dtype).cuda()
    buf, c = guarded(m, n, dtype)
    ao = a.t().contiguous() if layout == "TN" else a
    bo = b if layout == "NT" else b.t().contiguous()
    gemm([ao], [bo], [c], m, n, k, kmajor=(layout == "TN", layout != "NT"))
    assert max_rel(c, a.double() @ b.double().t()) < TOL[dtype]
    assert untouched(buf, m, n)


@pytest.mark.parametrize("kind,m,n,k", [(kind, *s) for kind in KINDS for s in PLANNED[kind]])
def test_every_tile(kind, m, n, k):
    """Every tile, K split and second launch of the plan in every form: against fp64 (a residual sum rounds twice,
    the SwiGLU backward from another rounding of dY), the fused norm and SwiGLU against their kernels."""
    layout, axis, epilogue = KINDS[kind]
    launches = planned(kind, m, n, k)
    dt = torch.float16 if (m + n // 8 + k) % 4 == 0 else torch.bfloat16
    print(f"q3_gemm {kind} {m}x{n}x{k} {dt} {launches}", flush=True)
    gen = torch.Generator("cuda").manual_seed(m + 3 * n + k)

    def rnd(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dt)

    def close(a, e, tol):
        return float((a.double() - e).abs().max() / e.abs().max()) <= tol
    parts = pieces(kind, m, n, k)
    ms, ns, ks = (parts if axis == ax else (size,) for ax, size in ((3, m), (2, n), (1, k)))
    a, b = (rnd(k, m) if layout == "TN" else rnd(m, k)), (rnd(n, k) if layout == "NT" else rnd(k, n))
    # the pieces are matrices of their own, the outputs lie in guarded buffers
    al = [t.contiguous() for t in (a.split(ms, 1) if axis == 3 else a.split(ks, 1) if axis == 1 else [a])]
    bl = [t.contiguous() for t in (b.split(ns, 0) if axis == 2 else b.split(ks, 0) if axis == 1 else [b])]
    e = (a.double().t() if layout == "TN" else a.double()) @ (b.double().t() if layout == "NT" else b.double())
    args = dict(kmajor=(layout == "TN", layout != "NT"), axis=axis, epilogue=epilogue)
    if epilogue in (H.GEMM_PLAIN, H.GEMM_RESIDUAL):
        outs = [guarded(mm, nn, dt) for mm in ms for nn in ns]
        if epilogue == H.GEMM_RESIDUAL:   # in place
            res = rnd(m, n)
            outs[0][1].copy_(res)
            args["res"], e = outs[0][1], res.double() + e
        gemm(al, bl, [c for _, c in outs], m, n, k, **args)
        es = e.split(ms, 0) if axis == 3 else e.split(ns, 1)
        for (buf, c), r in zip(outs, es):
            assert close(c, r, TOL[dt] * (2 if epilogue else 1)) and untouched(buf, *c.shape)
    elif epilogue == H.GEMM_RESIDUAL_NORM:
        res, nw = rnd(m, n), rnd(n)
        c, h = res.clone(), torch.empty_like(res)
        gemm(al, bl, [c], m, n, k, res=c, norm=(nw, 1e-6, h), **args)
        assert close(c, res.double() + e, 2 * TOL[dt])
        eh = _ops.rmsnorm_fwd(c, nw, 1e-6)
        if launches[0][4] == 1:
            assert torch.equal(h, eh)
        else:   # the combining pass sums the squares in another order: a few values one rounding step apart
            assert (h != eh).float().mean().item() < 0.01 and close(h, eh.double(), 2 * TOL[dt])
    elif epilogue == H.GEMM_GATE_UP:
        w2 = rnd(n, k)
        g, u, y, y2 = (torch.empty(m, n, device="cuda", dtype=dt) for _ in range(4))
        gemm([a], [b, w2], [y], m, n, k, g=g, u=u, **args)
        assert close(g, e, TOL[dt]) and close(u, a.double() @ w2.double().t(), TOL[dt])
        assert torch.equal(y, _ops.swiglu_fwd(g, u))
        gemm([a], [b, w2], [y2], m, n, k, **args)
        assert torch.equal(y2, y)
    else:
        g, u = rnd(m, n), rnd(m, n)
        dg, du = torch.empty_like(g), torch.empty_like(g)
        gemm([a], [b], [dg, du], m, n, k, g=g, u=u, **args)
        for c, r in zip((dg, du), _ops.swiglu_bwd(g, u, e.to(dt))):
            assert close(c, r.double(), 4 * TOL[dt])


@pytest.mark.parametrize("m,n,k", [(1, 1, 8), (40, 77, 136), (333, 1001, 520), (2050, 513, 200)])
def test_columns_off_the_chunk_grid(m, n, k):
    """Output columns that are no whole 16-byte chunks: scalar stores, with and without the residual."""
    print(f"q3_gemm columns {m}x{n}x{k}", flush=True)
    gen = seeded(m + n)
    dt = torch.bfloat16
    x, w, res = (randn(*s, gen=gen, dtype=dt).cuda() for s in ((m, k), (n, k), (m, n)))
    e = x.double() @ w.double().t()
    buf, c = guarded(m, n, dt)
    gemm([x], [w], [c], m, n, k)
    assert max_rel(c, e) < TOL[dt] and untouched(buf, m, n)
    y = c.clone()
    c.copy_(res)
    gemm([x], [w], [c], m, n, k, epilogue=H.GEMM_RESIDUAL, res=c)
    assert torch.equal(c, _ops.add(res, y)) and untouched(buf, m, n)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_benchmark_layer_products(dtype):
    """The twelve products of an 8192-token decoder layer as the modules launch them (hidden 4096, intermediate
    12288, q/k/v of 4096 + 1024 + 1024): sampled rows against fp64."""
    t, hid, inter, qkv = 8192, 4096, 12288, (4096, 1024, 1024)
    gen = torch.Generator("cuda").manual_seed(8)
    tol = TOL[dtype]

    def rnd(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype)

    def new(*shape):
        return torch.empty(shape, device="cuda", dtype=dtype)

    def check(what, c, a, b, tol=tol, res=None):
        """c's sampled rows against a's (one row of the product per row of a) times b, plus res."""
        rows = torch.arange(7, c.shape[0], c.shape[0] // 61, device="cuda")
        e = a(rows).double() @ b.double() + (0 if res is None else res[rows].double())
        assert float((c[rows].double() - e).abs().max() / e.abs().max()) <= tol, what
    x, res, wo, wd = rnd(t, hid), rnd(t, hid), rnd(hid, hid, scale=0.02), rnd(hid, inter, scale=0.02)
    ws = [rnd(n, hid, scale=0.02) for n in qkv]
    wg, wu = rnd(inter, hid, scale=0.02), rnd(inter, hid, scale=0.02)
    print(f"layer products {dtype}: forward", flush=True)
    ys = [new(t, n) for n in qkv]
    gemm([x], ws, ys, t, sum(qkv), hid, axis=2)
    for y, w in zip(ys, ws):
        check("q/k/v", y, lambda r: x[r], w.t())
    o, g, u, y, out = new(t, hid), new(t, inter), new(t, inter), new(t, inter), new(t, hid)
    gemm([x], [wo], [o], t, hid, hid, epilogue=H.GEMM_RESIDUAL, res=res)
    check("o", o, lambda r: x[r], wo.t(), 2 * tol, res)
    gemm([x], [wg, wu], [y], t, inter, hid, epilogue=H.GEMM_GATE_UP, g=g, u=u)
    check("gate", g, lambda r: x[r], wg.t())
    check("up", u, lambda r: x[r], wu.t())
    assert torch.equal(y, _ops.swiglu_fwd(g, u))
    gemm([y], [wd], [out], t, hid, inter, epilogue=H.GEMM_RESIDUAL, res=res)
    check("down", out, lambda r: y[r], wd.t(), 2 * tol, res)
    print(f"layer products {dtype}: backward", flush=True)
    dy = rnd(t, hid)
    dwd, dg, du = new(hid, inter), new(t, inter), new(t, inter)
    gemm([dy], [y], [dwd], hid, inter, t, kmajor=(True, True))
    check("dW down", dwd, lambda r: dy[:, r].t(), y)
    gemm([dy], [wd], [dg, du], t, inter, hid, kmajor=(False, True), epilogue=H.GEMM_SWIGLU_BWD, g=g, u=u)
    rows = torch.arange(7, t, t // 61, device="cuda")
    for c, e in zip((dg, du), _ops.swiglu_bwd(g[rows], u[rows], (dy[rows].double() @ wd.double()).to(dtype))):
        assert max_rel(c[rows], e) <= 4 * tol   # dY rounds from fp32 and from fp64
    dx, dwg, dwu = new(t, hid), new(inter, hid), new(inter, hid)
    gemm([dg, du], [wg, wu], [dx], t, hid, 2 * inter, kmajor=(False, True), axis=1)
    check("dX gate/up", dx, lambda r: torch.cat([dg[r], du[r]], 1), torch.cat([wg, wu]))
    gemm([dg, du], [x], [dwg, dwu], 2 * inter, hid, t, kmajor=(True, True), axis=3)
    check("dW gate", dwg, lambda r: dg[:, r].t(), x)
    check("dW up", dwu, lambda r: du[:, r].t(), x)
    dwo, dxo = new(hid, hid), new(t, hid)
    gemm([dy], [x], [dwo], hid, hid, t, kmajor=(True, True))
    check("dW o", dwo, lambda r: dy[:, r].t(), x)
    gemm([dy], [wo], [dxo], t, hid, hid, kmajor=(False, True))
    check("dX o", dxo, lambda r: dy[r], wo)
    gemm(ys, ws, [dx], t, hid, sum(qkv), kmajor=(False, True), axis=1)
    check("dX q/k/v", dx, lambda r: torch.cat([c[r] for c in ys], 1), torch.cat(ws))
    dws = [new(n, hid) for n in qkv]
    gemm(ys, [x], dws, sum(qkv), hid, t, kmajor=(True, True), axis=3)
    for c, d in zip(dws, ys):
        check("dW q/k/v", c, lambda r: d[:, r].t(), x)


def test_operands_in_place():
    """Row-strided operands (column blocks of wider matrices) and NaN / infinity around them: nothing outside
    the operand enters a product."""
    gen = seeded(3)
    m, n, k = 70, 40, 88
    for kmajor in ((False, False), (False, True), (True, True)):
        mm = 72 if kmajor[0] else m
        a = torch.full((200, 160), float("nan")).bfloat16()
        b = torch.full((200, 160), float("inf")).bfloat16()
        ra, rb = (k, mm) if kmajor[0] else (mm, k), (k, n) if kmajor[1] else (n, k)
        a[:ra[0], 8:8 + ra[1]] = randn(*ra, gen=gen, dtype=torch.bfloat16)
        b[:rb[0], 16:16 + rb[1]] = randn(*rb, gen=gen, dtype=torch.bfloat16)
        av, bv = a.cuda()[:ra[0], 8:8 + ra[1]], b.cuda()[:rb[0], 16:16 + rb[1]]
        c = torch.empty(mm, n, device="cuda", dtype=torch.bfloat16)
        gemm([av], [bv], [c], mm, n, k, kmajor=kmajor)
        e = (av.double().t() if kmajor[0] else av.double()) @ (bv.double() if kmajor[1] else bv.double().t())
        assert max_rel(c, e) < TOL[torch.bfloat16], kmajor


@pytest.mark.parametrize("m,ns,k", [(65, (4096, 1024, 1024), 4096), (333, (256, 64, 72), 512), (9, (40, 8), 104)])
def test_pieces(m, ns, k):
    """q/k/v-style pieces along n, k and m against fp64."""
    gen = seeded(sum(ns) + m)
    dt = torch.bfloat16
    x = randn(m, k, gen=gen, dtype=dt).cuda()
    ws = [randn(n, k, gen=gen, dtype=dt).cuda() for n in ns]
    dys = [randn(m, n, gen=gen, dtype=dt).cuda() for n in ns]
    bufs = [guarded(m, n, dt) for n in ns]
    print(f"q3_gemm pieces {m} {ns} {k}", flush=True)
    gemm([x], ws, [c for _, c in bufs], m, sum(ns), k, axis=2)
    for (buf, c), w, n in zip(bufs, ws, ns):
        assert max_rel(c, x.double() @ w.double().t()) < TOL[dt] and untouched(buf, m, n)
    dx = torch.empty(m, k, device="cuda", dtype=dt)
    gemm(dys, ws, [dx], m, k, sum(ns), kmajor=(False, True), axis=1)
    assert max_rel(dx, sum(d.double() @ w.double() for d, w in zip(dys, ws))) < TOL[dt]
    bufs = [guarded(n, k, dt) for n in ns]
    gemm(dys, [x], [c for _, c in bufs], sum(ns), k, m, kmajor=(True, True), axis=3)
    for (buf, c), d, n in zip(bufs, dys, ns):
        assert max_rel(c, d.double().t() @ x.double()) < TOL[dt] and untouched(buf, n, k)


@pytest.mark.parametrize("m,n,k", [(65, 4096, 4096), (20, 264, 4096), (333, 4096, 1024), (600, 256, 64), (3, 8, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_epilogues(m, n, k, dtype):
    """Residual (in place too), residual + norm, gate/up and the SwiGLU backward: bit-equal to the plain product
    followed by the add / norm / SwiGLU kernels (the fused norm sums its squares in another order)."""
    print(f"q3_gemm epilogues {m}x{n}x{k} {dtype}", flush=True)
    gen = seeded(m + n + 5 * k)
    x = randn(m, k, gen=gen, dtype=dtype).cuda()
    w, w2 = (randn(n, k, gen=gen, dtype=dtype, scale=0.05).cuda() for _ in range(2))
    res, nw = randn(m, n, gen=gen, dtype=dtype).cuda(), randn(n, gen=gen, dtype=dtype).cuda()
    y = torch.empty(m, n, device="cuda", dtype=dtype)
    gemm([x], [w], [y], m, n, k)
    e = _ops.add(res, y)
    out = torch.empty_like(y)
    gemm([x], [w], [out], m, n, k, epilogue=H.GEMM_RESIDUAL, res=res)
    assert torch.equal(out, e)
    c, h = res.clone(), torch.empty_like(y)
    gemm([x], [w], [c], m, n, k, epilogue=H.GEMM_RESIDUAL_NORM, res=c, norm=(nw, 1e-6, h))
    eh = _ops.rmsnorm_fwd(e, nw, 1e-6)
    assert torch.equal(c, e)
    # 1 / rms may differ in its last fp32 bit: a few values one rounding step (2^-8 / 2^-11 of the value) apart
    assert (h != eh).float().mean().item() < 0.01 and max_rel(h, eh) <= (8e-3 if dtype == torch.bfloat16 else 1e-3)
    g, u, sy, sy2 = (torch.empty_like(y) for _ in range(4))
    gemm([x], [w, w2], [sy], m, n, k, epilogue=H.GEMM_GATE_UP, g=g, u=u)
    assert torch.equal(sy, _ops.swiglu_fwd(g, u))
    assert max_rel(g, x.double() @ w.double().t()) < TOL[dtype] and max_rel(u, x.double() @ w2.double().t()) < TOL[dtype]
    gemm([x], [w, w2], [sy2], m, n, k, epilogue=H.GEMM_GATE_UP)
    assert torch.equal(sy2, sy)
    wk = w.t().contiguous()   # [k, n]: K-major
    dy, dg, du = (torch.empty_like(y) for _ in range(3))
    gemm([x], [wk], [dg, du], m, n, k, kmajor=(False, True), epilogue=H.GEMM_SWIGLU_BWD, g=g, u=u)
    eg, eu = _ops.swiglu_bwd(g, u, (x.double() @ w.double().t()).to(dtype))
    assert max_rel(dg, eg) <= 4 * TOL[dtype] and max_rel(du, eu) <= 4 * TOL[dtype]   # dY rounds from fp32 and from fp64
    if k < 1024:   # unsplit plain product: the same fp32 sums
        gemm([x], [wk], [dy], m, n, k, kmajor=(False, True))
        eg, eu = _ops.swiglu_bwd(g, u, dy)
        assert torch.equal(dg, eg) and torch.equal(du, eu)


@pytest.mark.parametrize("m,n,k", [(6145, 4096, 4096), (9300, 4096, 512), (4700, 8192, 512), (12800, 2048, 512)])
def test_residual_in_place_over_two_launches(m, n, k):
    """Row counts that q3_gemm forms in two launches, the second on 192-row tiles: with the residual in place no
    row takes the product twice, and the norm is that of the same sum."""
    print(f"q3_gemm residual in place {m}x{n}x{k}", flush=True)
    gen = torch.Generator("cuda").manual_seed(m)
    dt = torch.bfloat16
    x, w, res = (torch.randn(s, generator=gen, device="cuda").to(dt) for s in ((m, k), (n, k), (m, n)))
    nw = torch.randn(n, generator=gen, device="cuda").to(dt)
    y, c = torch.empty_like(res), res.clone()
    gemm([x], [w], [y], m, n, k)
    e = _ops.add(res, y)
    gemm([x], [w], [c], m, n, k, epilogue=H.GEMM_RESIDUAL, res=c)
    assert torch.equal(c, e)
    c, h = res.clone(), torch.empty_like(res)
    gemm([x], [w], [c], m, n, k, epilogue=H.GEMM_RESIDUAL_NORM, res=c, norm=(nw, 1e-6, h))
    assert torch.equal(c, e) and torch.equal(h, _ops.rmsnorm_fwd(e, nw, 1e-6))


def test_refusals():
    x = torch.zeros(16, 64, device="cuda", dtype=torch.bfloat16)
    c = torch.zeros(16, 16, device="cuda", dtype=torch.bfloat16)
    for a, b, kw in ((x[:, 4:60], x[:, 4:60], {}),                     # 8-byte aligned rows
                     (x, x, dict(kmajor=(True, False))),               # K-major A with a k-contiguous B
                     (x, x, dict(epilogue=H.GEMM_RESIDUAL_NORM)),      # no residual, norm weight or output
                     (x, x, dict(epilogue=H.GEMM_GATE_UP))):           # one weight only
        with pytest.raises(RuntimeError):
            gemm([a], [b], [c], 16, 16, a.shape[1], **kw)
    big = torch.zeros(65, 4096, device="cuda", dtype=torch.bfloat16)
    d = H.GemmDesc()
    d.dtype, d.pieces, d.m, d.n, d.k = H.BF16, 1, 65, 65, 4096
    for f in ("a", "b"):
        getattr(d, f)[0], getattr(d, "ld" + f)[0] = big.data_ptr(), 4096
    out = torch.zeros(65, 72, device="cuda", dtype=torch.bfloat16)
    d.c[0], d.ldc[0], d.n = out.data_ptr(), 72, 64
    import ctypes
    need = H.query("q3_gemm_workspace_bytes", ctypes.addressof(d))
    assert need > 0
    ws = torch.empty(need, device="cuda", dtype=torch.uint8)
    with pytest.raises(RuntimeError):   # a workspace below the stated size is refused before any launch
        H.call("q3_gemm", ctypes.addressof(d), ws.data_ptr(), need - 16, H.stream())


def test_fused_layers_refuse_what_the_layers_refuse():
    """A feature vector without a token axis and weights that are no matrices: the errors of ``linear`` and
    ``gate_up_swiglu``."""
    from qwen3_triton.kernels.linear import shared_input_projections
    from qwen3_triton.kernels.mlp_precision import mlp_block
    x = torch.zeros(2, 64, device="cuda", dtype=torch.bfloat16)
    w = torch.zeros(64, 64, device="cuda", dtype=torch.bfloat16)
    for xs, ws in ((x[0], [w, w]), (x, [w[0]]), (x, [w, w[..., None]])):
        with pytest.raises(ValueError, match="Expected"):
            shared_input_projections(xs, ws)
    assert shared_input_projections(x, []) == []
    for xs, ws in ((x[0], (w, w, w)), (x, (w[0], w[0], w)), (x, (w[..., None], w[..., None], w)), (x, (w, w, w[0]))):
        with pytest.raises(ValueError, match="Expected"):
            mlp_block(xs, *ws)


@pytest.mark.parametrize("b,s,h,v", [(1, 2, 64, 8), (1, 129, 64, 264), (3, 67, 128, 1000), (1, 257, 64, 520)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_lm_head_ragged(b, s, h, v, dtype):
    """The fused LM head + loss at token counts off the tile grid: loss and gradients against fp64, a second
    backward through the same graph equal to the first."""
    from qwen3_triton.kernels.lm_head_ce import lm_head_cross_entropy
    print(f"lm_head {b}x{s} {h} -> {v} {dtype}", flush=True)
    gen = seeded(b * s + v)
    x0, w0 = randn(b, s, h, gen=gen, dtype=dtype), randn(v, h, gen=gen, dtype=dtype, scale=0.1)
    labels = torch.randint(0, v, (b, s), generator=gen)
    labels[0, s // 2:s // 2 + s // 8] = -100
    x, w = x0.cuda().requires_grad_(), w0.cuda().requires_grad_()
    loss = lm_head_cross_entropy(x, w, labels.cuda())
    first = torch.autograd.grad(loss, [x, w], retain_graph=True)
    second = torch.autograd.grad(loss, [x, w])
    xr, wr = x0.double().requires_grad_(), w0.double().requires_grad_()
    z = xr @ wr.t()
    e = torch.nn.functional.cross_entropy(z[:, :-1].reshape(-1, v), labels[:, 1:].reshape(-1), ignore_index=-100)
    grads = torch.autograd.grad(e, [xr, wr])
    assert abs(float(loss.detach()) - float(e)) <= 1e-3 * abs(float(e))
    # the logits stay fp32; dz rounds once to the storage type, and the gradient once (2^-9 / 2^-12 of each value)
    for a, c, g in zip(first, second, grads):
        assert torch.equal(a, c)
        assert max_rel(a, g) <= 2 * TOL[dtype]


def test_operands_past_2_34_elements():
    """K-major operands whose rows span more than 2^34 elements (34 GB): the same products as from dense ones."""
    print("q3_gemm wide operands", flush=True)
    k, ld, m, n = 8200, 1 << 21, 72, 136
    buf = torch.empty(k * ld, device="cuda", dtype=torch.bfloat16)
    a, b = buf.as_strided((k, m), (ld, 1), 0), buf.as_strided((k, n), (ld, 1), 1024)
    gen = seeded(34)
    a0, b0 = randn(k, m, gen=gen, dtype=torch.bfloat16).cuda(), randn(k, n, gen=gen, dtype=torch.bfloat16).cuda()
    a.copy_(a0), b.copy_(b0)
    assert torch.equal(matmul(a.t(), b), matmul(a0.t(), b0))          # both K-major
    x0 = randn(m, k, gen=gen, dtype=torch.bfloat16).cuda()
    assert torch.equal(matmul(x0, b), matmul(x0, b0))                 # a k-contiguous, b K-major
    assert max_rel(matmul(x0, b0), x0.double() @ b0.double()) < TOL[torch.bfloat16]


def test_lm_head_logits_past_2_34_elements():
    """LM-head training above 2^34 logits (113080 tokens of a 151936-word vocabulary): sampled rows of both
    gradients against fp64 (logits of deviation 1: bf16 logits leave 2^-9 of a probability)."""
    from qwen3_triton.kernels.lm_head_ce import lm_head_cross_entropy
    t, h, v = 113080, 64, 151936
    print(f"lm_head {t} x {h} -> {v}", flush=True)
    gen = torch.Generator("cuda").manual_seed(1)
    x = torch.randn(1, t, h, generator=gen, device="cuda").bfloat16().requires_grad_()
    w = (torch.randn(v, h, generator=gen, device="cuda") * h ** -0.5).bfloat16().requires_grad_()
    y = torch.randint(0, v, (1, t), generator=gen, device="cuda")
    dx, dw = torch.autograd.grad(lm_head_cross_entropy(x, w, y), (x, w))
    xs, ws = x.detach()[0].float(), w.detach().float()
    lse = torch.cat([(xs[i:i + 4096] @ ws.t()).logsumexp(1) for i in range(0, t, 4096)]).double()
    tgt = torch.full((t,), -1, device="cuda")
    tgt[:-1] = y[0, 1:]
    valid = (tgt >= 0).double() / (t - 1)
    rows, cols = torch.tensor([0, 1, 4097, t - 9, t - 2], device="cuda"), torch.tensor([0, 7, 75000, v - 1], device="cuda")
    xd, wd = xs.double(), ws.double()
    dz = (xd[rows] @ wd.t() - lse[rows, None]).exp()
    dz[torch.arange(len(rows)), tgt[rows]] -= 1
    assert max_rel(dx[0, rows], (dz * valid[rows, None]) @ wd) <= 2e-2
    dz = (xd @ wd[cols].t() - lse[:, None]).exp() - (tgt[:, None] == cols).double()
    assert max_rel(dw[cols], (dz * valid[:, None]).t() @ xd) <= 2e-2
