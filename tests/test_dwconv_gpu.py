"""Depthwise conv7 + SiLU on (B, L, C) (libissm_hip.so) against torch's Conv1d + SiLU in fp64 on the CPU
(the formulation of models/dest_module.py:400-423).  fp32: rel. error <= 1e-5 forward, 1e-4 gradients;
bf16: <= 1e-2 / 3e-2 (the convolution output is rounded to bf16 before SiLU, as a bf16 Conv1d module's is)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _ref(u, ws, bs):
    C = u.shape[-1]
    return [F.silu(F.conv1d(u.transpose(1, 2), w.reshape(C, 1, 7), b, padding=3, groups=C)).transpose(1, 2)
            for w, b in zip(ws, bs)]


def _rel(a, b):
    return ((a.double().cpu() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


CASES = [
    # B, L, C, nsets, dtype, strided input
    (2, 100, 290, 2, torch.float32, True),
    (1, 5, 33, 1, torch.float32, False),
    (3, 16, 64, 2, torch.float32, False),
    (2, 1, 8, 2, torch.float32, False),
    (2, 257, 290, 2, torch.bfloat16, True),
    (1, 40, 130, 1, torch.bfloat16, False),
    (2, 1030, 520, 1, torch.bfloat16, False),   # 8 and 16 tokens a thread (few tokens, as above: 4)
    (2, 2051, 520, 2, torch.float32, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_L%d_C%d_S%d_%s_%s" % (*c[:4], str(c[4])[6:], "view" if c[5] else "dense"))
def test_dwconv_silu_matches_fp64(case):
    from dest3d_amd.dwconv import dwconv_silu
    B, L, C, S, dtype, strided = case
    g = torch.Generator().manual_seed(77 + L + C)
    full = torch.randn(B, L, C + 24, generator=g).to(dtype)
    base = full.cuda().requires_grad_()
    u = base[..., 8:8 + C] if strided else base[..., :C].contiguous()
    ws = [(0.4 * torch.randn(C, 1, 7, generator=g)).cuda().requires_grad_() for _ in range(S)]
    bs = [(0.2 * torch.randn(C, generator=g)).cuda().requires_grad_() for _ in range(S)]
    ys = dwconv_silu(u, ws, bs)
    u64 = (full[..., 8:8 + C] if strided else full[..., :C]).double().requires_grad_()
    w64 = [w.detach().double().cpu().requires_grad_() for w in ws]
    b64 = [b.detach().double().cpu().requires_grad_() for b in bs]
    refs = _ref(u64, w64, b64)
    ftol, gtol = (1e-5, 1e-4) if dtype == torch.float32 else (1e-2, 3e-2)
    assert len(ys) == S
    for y, r in zip(ys, refs):
        assert y.shape == (B, L, C) and y.dtype == dtype
        assert _rel(y, r) <= ftol
    gy = [torch.randn(B, L, C, generator=g).to(dtype) for _ in range(S)]
    torch.autograd.backward(list(ys), [t.cuda() for t in gy])
    torch.autograd.backward(refs, [t.double() for t in gy])
    got_du = base.grad[..., 8:8 + C] if strided else base.grad[..., :C]
    assert _rel(got_du, u64.grad) <= gtol
    for s in range(S):
        assert ws[s].grad.shape == (C, 1, 7)
        assert _rel(ws[s].grad, w64[s].grad) <= gtol
        assert _rel(bs[s].grad, b64[s].grad) <= gtol


CHAIN_CASES = [
    # B, L, C, dtype, strided input
    (2, 100, 290, torch.float32, True),
    (3, 16, 64, torch.float32, False),
    (2, 1, 8, torch.float32, False),
    (1, 5, 33, torch.float32, False),
    (1, 23, 40, torch.float32, False),
    (2, 257, 290, torch.bfloat16, True),
    (2, 1030, 520, torch.float32, False),
    (2, 2051, 520, torch.bfloat16, True),
]


@pytest.mark.parametrize("case", CHAIN_CASES, ids=lambda c: "B%d_L%d_C%d_%s_%s" % (*c[:3], str(c[3])[6:], "view" if c[4] else "dense"))
def test_dwconv_chain_matches_fp64(case):
    """chain=True: the second set convolves the first set's result (models/dest_module.py:530,534), forward and every
    gradient -- du and the first set's weight gradient collect what flows back through the second convolution."""
    from dest3d_amd.dwconv import dwconv_silu
    B, L, C, dtype, strided = case
    print(f"[case] dwconv chain B={B} L={L} C={C} {dtype}", flush=True)
    g = torch.Generator().manual_seed(91 + L + C)
    full = torch.randn(B, L, C + 24, generator=g).to(dtype)
    base = full.cuda().requires_grad_()
    u = base[..., 8:8 + C] if strided else base[..., :C].contiguous()
    ws = [(0.4 * torch.randn(C, 1, 7, generator=g)).cuda().requires_grad_() for _ in range(2)]
    bs = [(0.2 * torch.randn(C, generator=g)).cuda().requires_grad_() for _ in range(2)]
    ys = dwconv_silu(u, ws, bs, chain=True)
    u64 = (full[..., 8:8 + C] if strided else full[..., :C]).double().requires_grad_()
    w64 = [w.detach().double().cpu().requires_grad_() for w in ws]
    b64 = [b.detach().double().cpu().requires_grad_() for b in bs]
    r0 = _ref(u64, w64[:1], b64[:1])[0]
    r1 = _ref(r0, w64[1:], b64[1:])[0]
    ftol, gtol = (1e-5, 1e-4) if dtype == torch.float32 else (1.5e-2, 4e-2)
    for y, r in zip(ys, (r0, r1)):
        assert y.shape == (B, L, C) and y.dtype == dtype
        assert _rel(y, r) <= ftol
    gy = [torch.randn(B, L, C, generator=g).to(dtype) for _ in range(2)]
    torch.autograd.backward(list(ys), [t.cuda() for t in gy])
    torch.autograd.backward([r0, r1], [t.double() for t in gy])
    got_du = base.grad[..., 8:8 + C] if strided else base.grad[..., :C]
    assert _rel(got_du, u64.grad) <= gtol
    for s in range(2):
        assert _rel(ws[s].grad, w64[s].grad) <= gtol
        assert _rel(bs[s].grad, b64[s].grad) <= gtol


def test_dwconv_chain_only_second_gradient():
    """Only the second output has a gradient: it still reaches u and the first set's parameters through the chain."""
    from dest3d_amd.dwconv import dwconv_silu
    g = torch.Generator().manual_seed(6)
    u = torch.randn(2, 50, 40, generator=g).cuda().requires_grad_()
    ws = [(0.4 * torch.randn(40, 7, generator=g)).cuda().requires_grad_() for _ in range(2)]
    bs = [(0.2 * torch.randn(40, generator=g)).cuda().requires_grad_() for _ in range(2)]
    _, y1 = dwconv_silu(u, ws, bs, chain=True)
    y1.sum().backward()
    u64 = u.detach().double().cpu().requires_grad_()
    w64 = [w.detach().double().cpu().requires_grad_() for w in ws]
    b64 = [b.detach().double().cpu().requires_grad_() for b in bs]
    r1 = _ref(_ref(u64, w64[:1], b64[:1])[0], w64[1:], b64[1:])[0]
    r1.sum().backward()
    assert _rel(u.grad, u64.grad) <= 1e-4
    assert _rel(ws[0].grad, w64[0].grad.reshape(40, 7)) <= 1e-4 and _rel(bs[0].grad, b64[0].grad) <= 1e-4


def test_dwconv_one_absent_gradient():
    from dest3d_amd.dwconv import dwconv_silu
    g = torch.Generator().manual_seed(5)
    u = torch.randn(2, 50, 40, generator=g).cuda().requires_grad_()
    ws = [torch.randn(40, 7, generator=g).cuda().requires_grad_() for _ in range(2)]
    bs = [torch.randn(40, generator=g).cuda().requires_grad_() for _ in range(2)]
    y0, y1 = dwconv_silu(u, ws, bs)
    y0.sum().backward()
    assert ws[1].grad.abs().max().item() == 0.0 and bs[1].grad.abs().max().item() == 0.0
    u64 = u.detach().double().cpu().requires_grad_()
    r = _ref(u64, [ws[0].detach().double().cpu()], [bs[0].detach().double().cpu()])[0]
    r.sum().backward()
    assert _rel(u.grad, u64.grad) <= 1e-4


def test_dwconv_rejects_unbuilt_shapes():
    import ctypes as C
    from dest3d_amd import _lib as L
    lib = L.load()
    a = L.DwConvArgs()
    a.batch, a.seqlen, a.channels, a.nsets, a.taps = 1, 8, 8, 1, 5
    assert lib.issm_dwconv_silu_fwd(C.byref(a)) == -5
    a.taps, a.nsets = 7, 3
    assert lib.issm_dwconv_silu_fwd(C.byref(a)) == -5
    a.nsets = 1
    assert lib.issm_dwconv_silu_fwd(C.byref(a)) == -1
    a.chain = 1                               # a chain needs two sets
    assert lib.issm_dwconv_silu_fwd(C.byref(a)) == -2


def test_dwconv_split_outputs_equal_the_slices():
    """With `split` the forward writes channels [0, split) and [split, C) as two dense tensors and the backward
    takes the gradient in the same two pieces: identical to slicing / concatenating around the unsplit call."""
    import ctypes as C
    from dest3d_amd import _lib as L
    from dest3d_amd import dwconv as D
    lib = L.load()
    g = torch.Generator().manual_seed(3)
    B, Ln, Cn, split = 2, 45, 38, 32
    u = torch.randn(B, Ln, Cn, generator=g).cuda()
    w = torch.randn(2, Cn, 7, generator=g).cuda()
    b = torch.randn(2, Cn, generator=g).cuda()
    dy = torch.randn(2, B, Ln, Cn, generator=g).cuda()

    def run(split_at):
        y = torch.empty(2, B, Ln, Cn if not split_at else split_at, device="cuda")
        tail = torch.empty(2, B, Ln, Cn - split_at, device="cuda") if split_at else None
        pre = torch.empty(2, B, Ln, Cn, device="cuda")
        a = D._args(u, 2)
        a.w, a.bias, a.y, a.pre = w.data_ptr(), b.data_ptr(), y.data_ptr(), pre.data_ptr()
        keep = []
        if split_at:
            a.split, a.y_tail = split_at, tail.data_ptr()
        L.check(lib.issm_dwconv_silu_fwd(C.byref(a)), "fwd")
        du = torch.empty(B, Ln, Cn, device="cuda")
        part = torch.empty(lib.issm_dwconv_partial_rows(B, Ln), 2, 8, Cn, device="cuda")
        dw, db = torch.empty(2, Cn, 7, device="cuda"), torch.empty(2, Cn, device="cuda")
        a.du, a.partial, a.dw, a.dbias = du.data_ptr(), part.data_ptr(), dw.data_ptr(), db.data_ptr()
        for s in range(2):
            if split_at:
                keep += [dy[s, ..., :split_at].contiguous(), dy[s, ..., split_at:].contiguous()]
                a.dy[s], a.dy_tail[s] = keep[-2].data_ptr(), keep[-1].data_ptr()
            else:
                a.dy[s] = dy[s].data_ptr()
        L.check(lib.issm_dwconv_silu_bwd(C.byref(a)), "bwd")
        torch.cuda.synchronize()
        return y, tail, du, dw, db

    y0, _, du0, dw0, db0 = run(0)
    y1, t1, du1, dw1, db1 = run(split)
    assert torch.equal(y1, y0[..., :split]) and torch.equal(t1, y0[..., split:])
    assert torch.equal(du1, du0) and torch.equal(dw1, dw0) and torch.equal(db1, db0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Ln,Cn,split,absent,far", [(2, 64, 34, 32, None, False), (1, 65, 97, 33, None, False), (2, 129, 32, 0, 0, False),
                                                      (1, 63, 7, 5, 1, False), (3, 192, 70, 64, None, False), (1, 3, 40, 38, None, True)])
def test_chain_backward_in_its_tiles(dtype, B, Ln, Cn, split, absent, far):
    """Tiles of 64 tokens and of 32 channels on either side of the split, a set without a gradient, tokens 2^22 elements apart, NaN around
    every tensor; the parts that issm_dwconv_silu_bwd_part leaves add up to the sums."""
    import ctypes as C
    from dest3d_amd import _lib as L
    from dest3d_amd import dwconv as D
    lib = L.load()
    g = torch.Generator().manual_seed(Ln + Cn)
    rnd = lambda *s: torch.randn(*s, generator=g)
    nan = lambda n: torch.full((n,), float("nan"), dtype=dtype, device="cuda")

    def framed(t):   # the same values between NaN
        t = t.to(dtype).cuda().contiguous()
        return torch.cat([nan(640), t.flatten(), nan(640)])[640:-640].view(t.shape)
    rows = (1 << 22) + 64 if far else Cn + 6
    u = nan(B * Ln * rows).view(B, Ln, rows)[..., :Cn]
    u.copy_(rnd(B, Ln, Cn))
    w, b = (0.4 * rnd(2, Cn, 7)).cuda(), rnd(2, Cn).cuda()
    pre, dy = framed(rnd(2, B, Ln, Cn)), [None if s == absent else rnd(B, Ln, Cn).to(dtype) for s in range(2)]
    pieces = [[] if t is None else [framed(p) for p in ((t[..., :split], t[..., split:]) if split else (t,))] for t in dy]
    du = torch.full((B, Ln, rows), 3.0, dtype=dtype, device="cuda")
    nr = lib.issm_dwconv_part_rows(B, Ln)
    assert 0 < nr <= lib.issm_dwconv_partial_rows(B, Ln)
    part, dw, db = torch.full((nr + 1, 2, 8, Cn), 3.0, device="cuda"), torch.zeros(2, Cn, 7, device="cuda"), torch.zeros(2, Cn, device="cuda")
    a = D._args(u, 2)
    a.w, a.bias, a.pre, a.chain, a.split, a.partial = w.data_ptr(), b.data_ptr(), pre.data_ptr(), 1, split, part.data_ptr()
    a.du, a.du_batch_stride, a.du_token_stride = du.data_ptr(), Ln * rows, rows
    for s in range(2):
        for field, t in zip((a.dy, a.dy_tail), pieces[s]):
            field[s] = t.data_ptr()
    L.check(lib.issm_dwconv_silu_bwd_part(C.byref(a)), "part")
    torch.cuda.synchronize()
    assert (part[nr] == 3.0).all() and (du[..., Cn:] == 3.0).all()
    first = du.clone()
    a.dw, a.dbias = dw.data_ptr(), db.data_ptr()
    L.check(lib.issm_dwconv_silu_bwd(C.byref(a)), "bwd")
    torch.cuda.synchronize()
    assert torch.equal(first, du)
    sums = part[:nr].double().sum(0)
    close = lambda got, want, tol: ((got.double().cpu() - want.double().cpu()).norm() <= tol * want.double().norm().cpu() + 1e-30)
    assert close(dw, sums[:, :7].transpose(1, 2), 1e-6) and close(db, sums[:, 7], 1e-6)
    # fp64: dpre[1], what flows back through the second convolution, dpre[0]
    p64, u64, w64 = pre.double().cpu(), u.double().cpu(), w.double().cpu()
    silu_grad = lambda x: torch.sigmoid(x) * (1 + x * (1 - torch.sigmoid(x)))
    d64 = [torch.zeros(B, Ln, Cn, dtype=torch.double) if t is None else t.double() for t in dy]
    y0 = F.silu(p64[0]).to(dtype).double()

    def back(d, wt, x):   # input and weight gradient of a depthwise convolution
        x = x.clone().requires_grad_()
        wt = wt.reshape(Cn, 1, 7).clone().requires_grad_()
        F.conv1d(x.transpose(1, 2), wt, padding=3, groups=Cn).backward(d.transpose(1, 2))
        return x.grad, wt.grad.reshape(Cn, 7)
    e1 = d64[1] * silu_grad(p64[1])
    through, gw1 = back(e1, w64[1], y0)
    e0 = (d64[0] + through) * silu_grad(p64[0])
    want, gw0 = back(e0, w64[0], u64)
    assert close(du[..., :Cn], want, 1e-5 if dtype == torch.float32 else 3e-3)
    assert close(dw, torch.stack([gw0, gw1]), 1e-5) and close(db, torch.stack([e0.sum((0, 1)), e1.sum((0, 1))]), 1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Ln,Cn,split", [(1, 16, 34, 32), (2, 17, 33, 0), (1, 35, 7, 5), (1, 3, 40, 38), (40, 65, 770, 768)])
def test_chain_forward_in_its_tiles(dtype, B, Ln, Cn, split):
    """Tiles of 16 and of 64 tokens and the rows too far apart for either (2^22 elements): the same bits, and nothing written beside them."""
    import ctypes as C
    from dest3d_amd import _lib as L
    from dest3d_amd import dwconv as D
    lib = L.load()
    g = torch.Generator().manual_seed(Ln + Cn)
    near = torch.full((B, Ln, Cn + 6), float("nan"), dtype=dtype, device="cuda")[..., :Cn]
    near.copy_(torch.randn(B, Ln, Cn, generator=g))
    w, b = (0.4 * torch.randn(2, Cn, 7, generator=g)).cuda(), torch.randn(2, Cn, generator=g).cuda()

    def run(u, seqs):
        y = torch.full((2 * seqs * Ln * Cn + 1,), 3.0, dtype=dtype, device="cuda")
        pre = torch.full((2 * seqs * Ln * Cn + 1,), 3.0, dtype=dtype, device="cuda")
        a = D._args(u, 2)
        a.w, a.bias, a.pre, a.chain, a.split = w.data_ptr(), b.data_ptr(), pre.data_ptr(), 1, split
        a.y, a.y_tail = y.data_ptr(), y.data_ptr() + 2 * seqs * Ln * split * y.element_size()
        L.check(lib.issm_dwconv_silu_fwd(C.byref(a)), "fwd")
        torch.cuda.synchronize()
        assert y[-1] == 3.0 and pre[-1] == 3.0
        pieces = y[:-1].split([2 * seqs * Ln * split, 2 * seqs * Ln * (Cn - split)])
        return torch.cat([t.view(2, seqs, Ln, -1) for t in pieces if t.numel()], -1), pre[:-1].view(2, seqs, Ln, Cn)
    y, pre = run(near, B)
    ref = _ref(near.double().cpu(), [w[0].double().cpu()], [b[0].double().cpu()])[0]
    assert _rel(y[0], ref) <= (1e-5 if dtype == torch.float32 else 1e-2)
    ref = _ref(y[0].double().cpu(), [w[1].double().cpu()], [b[1].double().cpu()])[0]
    assert _rel(y[1], ref) <= (1e-5 if dtype == torch.float32 else 1e-2)
    rows = 1 << 22
    apart = torch.full((min(Ln, 36) * rows,), float("nan"), dtype=dtype, device="cuda").view(1, -1, rows)[..., :Cn]
    apart.copy_(near[:1, :36])
    if Ln <= 36:
        far_y, far_pre = run(apart, 1)
        assert torch.equal(far_y[:, 0], y[:, 0]) and torch.equal(far_pre[:, 0], pre[:, 0])
    one_y, one_pre = run(near[-1:], 1)   # (of many sequences 64 tokens a tile, of one 16)
    assert torch.equal(one_y[:, 0], y[:, -1]) and torch.equal(one_pre[:, 0], pre[:, -1])


@pytest.mark.parametrize("dtype,Ln", [(torch.float32, 15503), (torch.bfloat16, 31001)])
def test_chain_beyond_the_last_cache(dtype, Ln):
    """More rows than 256 MB hold: the forms that take them, against the first and the last tokens in calls of their own (their inner edge left out):
    the same bits of both outputs and what is kept for the backward."""
    import ctypes as C
    from dest3d_amd import _lib as L
    lib, B, Cn, split, few = L.load(), 3, 290, 288, 300
    g = torch.Generator(device="cuda").manual_seed(Ln)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    u, w, b = rnd(B, Ln, Cn).to(dtype), 0.4 * rnd(2, Cn, 7), 0.2 * rnd(2, Cn)

    def run(u):
        n = u.shape[1]
        y, tail, pre = (torch.full((2, B, n, c), 3.0, dtype=dtype, device="cuda") for c in (split, Cn - split, Cn))
        a = L.DwConvArgs(batch=B, seqlen=n, channels=Cn, nsets=2, taps=7, dtype=L.dtype_code(dtype), u=u.data_ptr(), u_batch_stride=n * Cn,
                         u_token_stride=Cn, w=w.data_ptr(), bias=b.data_ptr(), y=y.data_ptr(), y_tail=tail.data_ptr(), pre=pre.data_ptr(), split=split,
                         chain=1, stream=L.current_stream_ptr(u.device))
        assert lib.issm_dwconv_silu_fwd(C.byref(a)) == 0
        torch.cuda.synchronize()
        return y, tail, pre
    whole, first, last = run(u), run(u[:, :few].contiguous()), run(u[:, -few:].contiguous())
    for t, f, l in zip(whole, first, last):
        assert torch.equal(t[:, :, :few - 6], f[:, :, :few - 6]) and torch.equal(t[:, :, 6 - few:], l[:, :, 6:])
        assert t.isfinite().all() and (t[:, :, few:-few] != 3.0).any(-1).all()
