"""issm_linear_fwd (libissm_hip.so) and the projections that take it: y = x w^T against an fp64 product of the same bf16
operands."""
import ctypes as C

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from dest3d_amd import _lib as L

pytestmark = pytest.mark.gpu


def _operands(tokens, nin, nout, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(tokens, nin, generator=g).bfloat16()
    w = (torch.randn(nout, nin, generator=g) * nin ** -0.5).bfloat16()
    return x, w, x.double() @ w.double().t()


def _close(y, x, w, ref):
    """One bf16 rounding of the result, and nin additions of 2^-24 of the products' magnitudes."""
    size = x.double().abs() @ w.double().abs().t()
    bound = 2.0 ** -8 * ref.abs() + x.shape[1] * 2.0 ** -24 * size
    assert ((y.double().cpu() - ref).abs() <= bound).all()


class Job(C.Structure):
    _fields_ = [("x", C.c_void_p), ("w", C.c_void_p), ("y", C.c_void_p), ("tokens", C.c_int64), ("nin", C.c_int32),
                ("nout", C.c_int32), ("turn", C.c_int32)]


class Args(C.Structure):
    _fields_ = [("job", Job * 2), ("njobs", C.c_int32), ("dtype", C.c_int32), ("stream", C.c_void_p)]


@pytest.mark.parametrize("shapes", [[(1, 32, 1)], [(64, 288, 32)], [(65, 288, 33), (16, 288, 586)], [(17, 256, 31), (130, 544, 35)],
                                    [(1023, 320, 64)], [(3, 96, 7), (0, 32, 5)], [(64, 288, 33), (512, 288, 288, 256)],
                                    [(15, 64, 5, 5), (130, 96, 35, 13)], [(70, 32, 17, 70), (66, 32, 3, 1)]])
def test_linear_at_its_remainders(shapes):
    """Rows, outputs and steps that fill no tile, batch of fragments or aligned store; one and two products a launch; results
    transposed within every fourth number of tokens."""
    lib = L.load()
    a, kept = Args(), []
    for i, (t, nin, nout, *turn) in enumerate(shapes):
        x, w, ref = _operands(t, nin, nout, 7 * i + t)
        xd, wd = x.cuda(), w.cuda()
        y = torch.full((t + 1, nout), 3.0, dtype=torch.bfloat16, device="cuda")     # a row behind the result
        a.job[i] = Job(xd.data_ptr(), wd.data_ptr(), y.data_ptr(), t, nin, nout, *turn)
        kept.append((x, w, ref, xd, wd, y, turn))
    a.njobs, a.dtype, a.stream = len(shapes), L.ISSM_BF16, L.current_stream_ptr(torch.device("cuda", 0))
    assert lib.issm_linear_fwd(C.byref(a)) == 0
    torch.cuda.synchronize()
    for x, w, ref, _, _, y, turn in kept:
        got = y[:-1]
        if turn:
            got = got.reshape(-1, y.shape[1], turn[0]).transpose(1, 2).reshape(got.shape)
        _close(got, x, w, ref)
        assert (y[-1] == 3.0).all()


@pytest.mark.parametrize("shapes", [[(8192, 288, 586), (2048, 288, 288)], [(16400, 96, 200)], [(11000, 288, 97)], [(4097, 320, 289), (8193, 64, 610)],
                                    [(64, 32, 160000)], [(64, 96, 96)], [(3700, 288, 96), (65, 864, 100)]])
def test_many_tokens_at_their_remainders(shapes):
    """Products in tiles (from 64 tokens and 96 outputs on, for odd multiples of 288 from more than 256 workgroups of linear.hip on): tokens, outputs
    and contractions that fill no tile or step, rows of odd length."""
    test_linear_at_its_remainders(shapes)


@pytest.mark.parametrize("shapes", [[(8192, 288, 586), (33, 288, 288)], [(63, 320, 320), (300, 320, 650)], [(1000, 192, 95), (70, 192, 200)],
                                    [(700, 320, 161), (66, 320, 97, 33)], [(1024, 288, 512), (1, 288, 5)], [(1024, 288, 480), (64, 288, 1024)],
                                    [(2048, 288, 257), (0, 288, 288)]])
def test_products_of_a_launch_in_a_form_each(shapes):
    """One product in tiles beside one that is not (few tokens, few outputs, turned), in either order, and both sides of the 256 workgroups up to which
    odd multiples of 288 features go without; every product as by itself."""
    test_linear_at_its_remainders(shapes)
    lib = L.load()
    a, kept = Args(), []
    for i, (t, nin, nout, *turn) in enumerate(shapes):
        x, w, _ = _operands(max(t, 1), nin, nout, i)
        y, alone = (torch.full((max(t, 1), nout), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        kept.append((x.cuda(), w.cuda(), y, alone))
        a.job[0], a.njobs, a.dtype = Job(kept[i][0].data_ptr(), kept[i][1].data_ptr(), alone.data_ptr(), t, nin, nout, *turn), 1, L.ISSM_BF16
        a.stream = L.current_stream_ptr(alone.device)
        assert lib.issm_linear_fwd(C.byref(a)) == 0
    for i, (t, nin, nout, *turn) in enumerate(shapes):
        a.job[i] = Job(*(v.data_ptr() for v in kept[i][:3]), t, nin, nout, *turn)
    a.njobs = 2
    assert lib.issm_linear_fwd(C.byref(a)) == 0
    torch.cuda.synchronize()
    for *_, y, alone in kept:
        assert torch.equal(y, alone)


@pytest.mark.parametrize("shapes", [[(64, 2, 96)], [(65, 586, 288), (64, 288, 288)], [(1000, 98, 130)], [(130, 94, 98), (4099, 610, 320)]])
def test_gradient_to_the_tokens_at_its_remainders(shapes):
    """issm_linear_dx: y = x w with w (in, out); contractions that end within a piece of eight, a row of which the next begins with what is
    no number."""
    lib = L.load()
    a, kept = Args(), []
    for i, (t, nin, nout) in enumerate(shapes):
        g = torch.Generator().manual_seed(3 * i + t)
        x, w = torch.randn(t, nin, generator=g).bfloat16(), (torch.randn(nin, nout, generator=g) * nin ** -0.5).bfloat16()
        x[t // 2 :: 7, 0] = float("nan")
        xd, wd = x.cuda(), w.cuda()
        y = torch.full((t + 1, nout), 3.0, dtype=torch.bfloat16, device="cuda")
        a.job[i] = Job(xd.data_ptr(), wd.data_ptr(), y.data_ptr(), t, nin, nout, 0)
        kept.append((x, w, xd, wd, y))
    a.njobs, a.dtype, a.stream = len(shapes), L.ISSM_BF16, L.current_stream_ptr(torch.device("cuda", 0))
    assert lib.issm_linear_dx(C.byref(a)) == 0
    torch.cuda.synchronize()
    for x, w, _, _, y in kept:
        ok = ~x[:, 0].isnan()
        assert y[:-1].cpu()[~ok].isnan().all()
        _close(y[:-1][ok.cuda()], x[ok], w.t(), x[ok].double() @ w.double())
        assert (y[-1] == 3.0).all()
    for t, nin, nout in ((63, 96, 96), (64, 96, 95), (64, 97, 96), (64, 96, 97)):
        a.njobs, a.job[0].tokens, a.job[0].nin, a.job[0].nout = 1, t, nin, nout
        assert lib.issm_linear_dx(C.byref(a)) != 0


def test_linear_refuses_what_it_does_not_take():
    lib = L.load()
    x = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda")
    good = (x.data_ptr(), x.data_ptr(), x.data_ptr(), 8, 32, 8)
    for job, n, dtype in ((good, 3, L.ISSM_BF16), (good, 1, L.ISSM_F32), ((*good[:4], 33, 8), 1, L.ISSM_BF16), ((*good[:4], 0, 8), 1, L.ISSM_BF16),
                          ((x.data_ptr() + 2, *good[1:]), 1, L.ISSM_BF16), ((None, *good[1:]), 1, L.ISSM_BF16), ((*good[:3], -1, 32, 8), 1, L.ISSM_BF16),
                          ((*good, 3), 1, L.ISSM_BF16), ((*good, -1), 1, L.ISSM_BF16)):
        a = Args()
        a.job[0] = Job(*job)
        a.njobs, a.dtype = n, dtype
        assert lib.issm_linear_fwd(C.byref(a)) != 0
    assert lib.issm_linear_fwd(None) != 0


@pytest.mark.parametrize("kind", ["contiguous", "every second row", "columns of a wider tensor", "odd features", "one row", "no rows",
                                  "unaligned", "transposed weight"])
def test_projections_of_every_form(kind):
    """The layer's projections accept what nn.Linear accepts: forms the kernel does not take go to the library's product."""
    from dest3d_amd.scan_module import _LinearTokens
    nin = 90 if kind == "odd features" else 96
    x, w, _ = _operands(0 if kind == "no rows" else 1 if kind == "one row" else 40, nin, 50, 3)
    x, w = x.cuda(), w.cuda()
    if kind == "every second row":
        x = x.repeat_interleave(2, 0)[::2]
    elif kind == "columns of a wider tensor":
        x = torch.cat([x, x], dim=1)[:, :nin]
    elif kind == "unaligned":
        x = torch.cat([x.new_zeros(1), x.flatten()])[1:].view(-1, nin)
    elif kind == "transposed weight":
        w = w.t().contiguous().t()
    x.requires_grad_()
    w.requires_grad_()
    y = _LinearTokens.apply(x, w)
    assert y.shape == (x.shape[0], 50)
    ref = x.detach().double().cpu() @ w.detach().double().cpu().t()
    _close(y.detach(), x.detach().cpu(), w.detach().cpu(), ref)
    dy = torch.ones_like(y)
    y.backward(dy)
    want = torch.ones(y.shape, dtype=torch.double) @ w.detach().double().cpu()
    assert ((x.grad.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()


def test_projections_under_transforms():
    """functorch's transforms are refused, as they are by the autograd function the kernel is reached through."""
    from dest3d_amd.scan_module import _LinearTokens
    x, w, _ = _operands(40, 96, 50, 4)
    x, w = x.cuda(), w.cuda()
    with torch.no_grad(), pytest.raises(RuntimeError):
        torch.vmap(lambda t: _LinearTokens.apply(t, w))(x.view(4, 10, 96))


class Products(TorchDispatchMode):
    """Multiply-adds of the matrix products it sees."""

    def __init__(self):
        super().__init__()
        self.seen = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func in (torch.ops.aten.mm.default, torch.ops.aten.bmm.default, torch.ops.aten.addmm.default):
            a, b = args[-2:]
            self.seen += a.numel() * b.shape[-1]
        return func(*args, **(kwargs or {}))


def test_a_dispatch_mode_sees_the_projections():
    """A mode that counts operations sees the four projections, and their gradients, of a layer as the library's products."""
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(5)
    B, Ln, K, D = 2, 70, 40, 288
    layer = MultiHeadISSMScan(d_model=D, d_state=K, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16()
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    x = [bf(B, Ln, D).requires_grad_(), bf(B, K, D).requires_grad_(), bf(B, Ln, K, 16)]
    size = B * (Ln * D * (layer.key_proj.out_features + D) + K * 2 * D * D)
    with torch.no_grad(), Products() as forward:
        got = layer(*x, None, None)
    assert forward.seen == size
    with torch.no_grad():
        for a, b in zip(got, layer(*x, None, None)):
            assert ((a - b).float().norm() <= 2.0 ** -7 * b.float().norm())
    with Products() as training:
        out = layer(*x, None, None)
        torch.autograd.backward(out, [torch.ones_like(t) for t in out])
    assert training.seen == 3 * size


class DwArgs(C.Structure):
    _fields_ = [("dy", C.c_void_p), ("x", C.c_void_p), ("dw", C.c_void_p), ("tokens", C.c_int64), ("nin", C.c_int32),
                ("nout", C.c_int32), ("dtype", C.c_int32), ("scratch", C.c_void_p), ("bytes", C.c_size_t), ("stream", C.c_void_p)]


@pytest.mark.parametrize("tokens,nin,nout", [(1, 6, 4), (33, 7, 5), (64, 96, 64), (257, 98, 65), (1000, 288, 586), (8200, 97, 130)])
def test_weight_gradient_at_its_remainders(tokens, nin, nout):
    """Rows that fill no step, columns that fill no tile, one part and many; what is behind the operands is NaN, the scratch
    starts as NaN.  One bf16 rounding of the result and an fp32 sum over the tokens."""
    lib = L.load()
    g = torch.Generator().manual_seed(tokens)
    x, dy = torch.randn(tokens, nin, generator=g).bfloat16(), torch.randn(tokens, nout, generator=g).bfloat16()
    pad = lambda t: torch.cat([t, torch.full_like(t[:1], float("nan"))]).cuda()
    xd, dyd = pad(x), pad(dy)
    dw = torch.full((nout + 1, nin), 3.0, dtype=torch.bfloat16, device="cuda")
    size = lib.issm_linear_dw_scratch_bytes(tokens, nin, nout)
    scratch = torch.full((size // 4 + 1,), float("nan"), device="cuda")
    a = DwArgs(dyd.data_ptr(), xd.data_ptr(), dw.data_ptr(), tokens, nin, nout, L.ISSM_BF16, scratch.data_ptr(), size,
               L.current_stream_ptr(torch.device("cuda", 0)))
    assert lib.issm_linear_dw(C.byref(a)) == 0
    torch.cuda.synchronize()
    ref, mag = dy.double().t() @ x.double(), dy.double().abs().t() @ x.double().abs()
    assert ((dw[:-1].double().cpu() - ref).abs() <= 2.0 ** -8 * ref.abs() + tokens * 2.0 ** -24 * mag).all()
    assert (dw[-1] == 3.0).all() and scratch[-1].isnan()
    for field, bad in (("bytes", size - 1), ("dtype", L.ISSM_F32), ("nin", 5), ("nout", 3), ("tokens", 0), ("scratch", None)):
        was = getattr(a, field)
        setattr(a, field, bad)
        assert lib.issm_linear_dw(C.byref(a)) != 0, field
        setattr(a, field, was)


@pytest.mark.parametrize("shapes", [[(1000, 288, 586), (64, 288, 288)], [(33, 7, 5), (8200, 97, 130)]])
def test_two_weight_gradients_in_a_launch(shapes):
    """The same bits as one at a time."""
    lib = L.load()
    args, kept = [], []
    for t, nin, nout in shapes:
        x, dy = torch.randn(t, nin).bfloat16().cuda(), torch.randn(t, nout).bfloat16().cuda()
        alone, pair = (torch.full((nout, nin), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        size = lib.issm_linear_dw_scratch_bytes(t, nin, nout)
        scratch = torch.full((size // 4,), float("nan"), device="cuda")
        a = DwArgs(dy.data_ptr(), x.data_ptr(), alone.data_ptr(), t, nin, nout, L.ISSM_BF16, scratch.data_ptr(), size,
                   L.current_stream_ptr(torch.device("cuda", 0)))
        assert lib.issm_linear_dw(C.byref(a)) == 0
        a.dw = pair.data_ptr()
        args.append(a)
        kept.append((x, dy, scratch, alone, pair))
    assert lib.issm_linear_dw_pair(C.byref(args[0]), C.byref(args[1])) == 0
    torch.cuda.synchronize()
    for *_, alone, pair in kept:
        assert torch.equal(alone, pair)
    args[1].bytes -= 1
    assert lib.issm_linear_dw_pair(C.byref(args[0]), C.byref(args[1])) != 0
    assert lib.issm_linear_dw_pair(C.byref(args[0]), None) != 0


@pytest.mark.parametrize("K", [40, 130])
def test_projections_beside_each_other(K):
    """An output that no loss reads gives its projection no gradient and leaves the others' as they are; frozen sides stay without one."""
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(7)
    B, Ln, D = 2, 70, 288
    layer = MultiHeadISSMScan(d_model=D, d_state=K, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16()
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    key, query, dist, dkey, dquery = bf(B, Ln, D), bf(B, K, D), bf(B, Ln, K, 16), bf(B, Ln, D), bf(B, K, D)
    grads = lambda: {n: p.grad for n, p in layer.named_parameters() if p.grad is not None}
    out = layer(key, query, dist, None, None)
    torch.autograd.backward(out[:1], [dkey])
    alone = grads()
    assert "out_key_proj.weight" in alone and "out_query_proj.weight" not in alone and "query_norm.weight" not in alone
    layer.zero_grad(set_to_none=True)
    out = layer(key, query, dist, None, None)
    torch.autograd.backward(out, [dkey, torch.zeros_like(dquery)])
    both = grads()
    for n, g in alone.items():
        assert torch.equal(g, both[n]), n
    for p in layer.parameters():
        p.requires_grad_(False)
    layer.out_query_proj.weight.requires_grad_()
    out = layer(key, query, dist, None, None)
    assert not out[0].requires_grad and out[1].requires_grad


@pytest.mark.parametrize("form", ["plain", "rows apart", "expanded gradient", "wide"])
def test_weight_gradient_of_every_form(form):
    from dest3d_amd.scan_module import _LinearTokens
    nin, nout = (512, 512) if form == "wide" else (96, 50)
    x, w, _ = _operands(300, nin, nout, 6)
    x, w = x.cuda(), w.cuda().requires_grad_()
    if form == "rows apart":
        x = torch.cat([x, x], dim=1)[:, :nin]
    dy = torch.randn(300, nout).cuda().bfloat16()
    if form == "expanded gradient":
        dy = dy[:1].expand(300, nout)
    _LinearTokens.apply(x, w).backward(dy)
    x, dy = x.double().cpu(), dy.double().cpu()
    ref, mag = dy.t() @ x, dy.abs().t() @ x.abs()
    # (the library may add in bf16 pieces: a rounding of the result each, four at most)
    assert ((w.grad.double().cpu() - ref).abs() <= 2.0 ** -7 * ref.abs() + 2.0 ** -9 * mag.sqrt() + 300 * 2.0 ** -24 * mag).all()


def test_backward_passes_of_either_output():
    """One pass after the other through a layer's two outputs, without retain_graph, to what only that output was made with: the gradients of one
    pass for both."""
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(8)
    B, Ln, K, D = 2, 70, 40, 288
    layer = MultiHeadISSMScan(d_model=D, d_state=K, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16()
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    key, query, dist, dkey, dquery = bf(B, Ln, D), bf(B, K, D), bf(B, Ln, K, 16), bf(B, Ln, D), bf(B, K, D)
    of_key, of_query = [layer.out_key_proj.weight], [layer.out_query_proj.weight, layer.query_norm.weight, layer.query_norm.bias]
    want = torch.autograd.grad(layer(key, query, dist, None, None), of_key + of_query, (dkey, dquery))
    out = layer(key, query, dist, None, None)
    got = torch.autograd.grad(out[0], of_key, dkey) + torch.autograd.grad(out[1], of_query, dquery)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    # (and where nothing else has a gradient)
    for p in layer.parameters():
        p.requires_grad_(False)
    layer.out_key_proj.weight.requires_grad_()
    layer.out_query_proj.weight.requires_grad_()
    out = layer(key, query, dist, None, None)
    out[1].backward(dquery)
    out[0].backward(dkey)
    assert torch.equal(layer.out_key_proj.weight.grad, want[0]) and torch.equal(layer.out_query_proj.weight.grad, want[1])


@pytest.mark.parametrize("form", ["few", "many", "odd", "expanded gradient", "unaligned gradient", "wide", "again"])
def test_gradient_to_the_tokens_of_every_form(form):
    """Both routes of the projections and of their gradients to the tokens, and the forms that stay the library's."""
    from dest3d_amd.scan_module import _LinearTokens
    t, nin, nout = {"many": (2049, 288, 610), "odd": (130, 96, 51), "wide": (100, 96, 1300)}.get(form, (130, 96, 202))
    x, w, ref = _operands(t, nin, nout, 9)
    x, w = x.cuda().requires_grad_(), w.cuda()
    dy = torch.randn(t, nout).cuda().bfloat16()
    if form == "expanded gradient":
        dy = dy[:1].expand(t, nout)
    elif form == "unaligned gradient":
        dy = torch.cat([dy.new_zeros(1), dy.flatten()])[1:].view(t, nout)
    y = _LinearTokens.apply(x, w)
    _close(y.detach(), x.detach().cpu(), w.cpu(), ref)
    if form == "again":
        dy.requires_grad_()
        dx, = torch.autograd.grad(y, x, dy, create_graph=True)
        got, = torch.autograd.grad(dx, dy, x.detach())
        _close(got, x.detach().cpu(), w.cpu(), ref)
    else:
        y.backward(dy)
        dx = x.grad
    _close(dx.detach(), dy.detach().cpu(), w.cpu().t(), dy.detach().double().cpu() @ w.double().cpu())


def test_weight_gradient_differentiated_again():
    """d/d dy of sum(dW * v) = x v^T: a backward pass under create_graph stays differentiable."""
    from dest3d_amd.scan_module import _LinearTokens
    x, w, _ = _operands(40, 96, 50, 8)
    x, w = x.cuda(), w.cuda().requires_grad_()
    dy = torch.randn(40, 50).cuda().bfloat16().requires_grad_()
    v = torch.randn(50, 96).cuda().bfloat16()
    dw, = torch.autograd.grad(_LinearTokens.apply(x, w), w, dy, create_graph=True)
    got, = torch.autograd.grad(dw, dy, v)
    _close(got, x.cpu(), v.cpu(), x.double().cpu() @ v.double().cpu().t())


class OutArgs(C.Structure):
    _fields_ = [("batch", C.c_int32), ("seqlen", C.c_int32), ("queries", C.c_int32), ("d_inner", C.c_int32), ("dtype", C.c_int32),
                ("y", C.c_void_p * 2), ("z", C.c_void_p), ("z_row_stride", C.c_int64), ("key_weight", C.c_void_p),
                ("key_eps", C.c_float), ("key", C.c_void_p), ("last", C.c_void_p * 2), ("query_weight", C.c_void_p),
                ("query_bias", C.c_void_p), ("query_eps", C.c_float), ("query", C.c_void_p), ("stream", C.c_void_p)]


@pytest.mark.parametrize("B,Ln,K,di,affine", [(1, 1, 1, 4, True), (2, 5, 9, 256, False), (3, 7, 16, 288, True), (1, 3, 7, 516, True),
                                              (2, 0, 3, 1024, False), (2, 6, 0, 260, True)])
def test_behind_the_scan(B, Ln, K, di, affine):
    """Rows, queries and features that fill no workgroup, wave or vector, against fp64 on the sums and averages rounded to bf16.
    Bound: the rounding of the result to 8 bits, and 2^-20 of the magnitudes for fp32 statistics and the fast exponential."""
    g = torch.Generator().manual_seed(di + K)
    r = lambda *s: torch.randn(*s, generator=g)
    bf = lambda t: t.bfloat16().cuda()
    y, zx, kw = [bf(r(B, Ln, di)) for _ in range(2)], bf(r(B, Ln, di + 3)), bf(r(di))
    last, qw, qb = [r(B, di, K).cuda() for _ in range(2)], bf(r(di)), bf(r(di))
    key, query = bf(torch.zeros(B * Ln + 1, di)), bf(torch.zeros(B * K + 1, di))
    ptr = lambda t: t.data_ptr() if t.numel() else None
    a = OutArgs(B, Ln, K, di, L.ISSM_BF16, (C.c_void_p * 2)(*map(ptr, y)), ptr(zx), di + 3, kw.data_ptr(), 4e-5, key.data_ptr(),
                (C.c_void_p * 2)(*map(ptr, last)), qw.data_ptr() if affine else None, qb.data_ptr() if affine else None, 1e-5,
                query.data_ptr(), L.current_stream_ptr(torch.device("cuda", 0)))
    assert L.load().issm_layer_out(C.byref(a)) == 0
    torch.cuda.synchronize()
    c = lambda t: t.double().cpu()
    z = c(zx)[..., :di]
    v = c((y[0].float() + y[1].float()).bfloat16()) * z * torch.sigmoid(z)
    v = (v * (v.pow(2).mean(-1, keepdim=True) + 4e-5).rsqrt() * c(kw)).reshape(-1, di)
    assert ((c(key[:-1]) - v).abs() <= 2.0 ** -8 * v.abs() + 2.0 ** -20).all() and (key[-1] == 0).all()
    s = c(((last[0] + last[1]) * 0.5).bfloat16()).transpose(1, 2).reshape(-1, di)
    s = (s - s.mean(-1, keepdim=True)) * (s.var(-1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    size = s.abs()
    if affine:
        s, size = s * c(qw) + c(qb), size * c(qw).abs() + c(qb).abs()
    assert ((c(query[:-1]) - s).abs() <= 2.0 ** -8 * s.abs() + 2.0 ** -20 * (1 + size)).all() and (query[-1] == 0).all()
    for field, bad in (("dtype", L.ISSM_F32), ("d_inner", 2), ("d_inner", 1028), ("batch", -1), ("z_row_stride", 1)):
        if field == "z_row_stride" and B * Ln == 0:
            continue
        was = getattr(a, field)
        setattr(a, field, bad)
        assert L.load().issm_layer_out(C.byref(a)) != 0, field
        setattr(a, field, was)


@pytest.mark.parametrize("B,Ln,K,di,outs", [(1, 1, 1, 32, (1, 1)), (2, 9, 19, 288, (288, 288)), (1, 40, 33, 320, (130, 97)),
                                            (3, 7, 16, 512, (33, 129)), (1, 20, 17, 1024, (128, 5)), (1, 3, 2, 576, (260, 260)),
                                            (2, 0, 3, 288, (9, 9)), (2, 6, 0, 64, (70, 70)), (1, 17, 5, 96, (0, 31))])
def test_norms_and_projections_behind_the_scan(B, Ln, K, di, outs):
    """issm_layer_end against fp64 on the sums and averages rounded to bf16: rows that fill no tile, outputs that fill no wave or
    vector, one set of fragments and several.  Bound: the norm's rounding to 8 bits in each term, and the result's own."""
    g = torch.Generator().manual_seed(di + K)
    r = lambda *s: torch.randn(*s, generator=g)
    bf = lambda t: t.bfloat16().cuda()
    y, zx, kw = [bf(r(B, Ln, di)) for _ in range(2)], bf(r(B, Ln, di + 3)), bf(r(di))
    last, qw, qb = [r(B, di, K).cuda() for _ in range(2)], bf(r(di)), bf(r(di))
    w, rows = [bf(r(o, di)) for o in outs], (B * Ln, B * K)
    got = [bf(torch.full((n + 1, o), 3.0)) for n, o in zip(rows, outs)]
    ptr = lambda t: t.data_ptr() if t.numel() else None
    a = OutArgs(B, Ln, K, di, L.ISSM_BF16, (C.c_void_p * 2)(*map(ptr, y)), ptr(zx), di + 3, kw.data_ptr(), 4e-5, None,
                (C.c_void_p * 2)(*map(ptr, last)), qw.data_ptr(), qb.data_ptr(), 1e-5, None,
                L.current_stream_ptr(torch.device("cuda", 0)))
    q = Args((Job * 2)(*[Job(None, ptr(w[i]), ptr(got[i]), rows[i], di, outs[i], 0) for i in range(2)]), 2, L.ISSM_BF16, None)
    lib = L.load()
    assert lib.issm_layer_end(C.byref(a), C.byref(q)) == 0
    torch.cuda.synchronize()
    c = lambda t: t.double().cpu()
    z = c(zx)[..., :di]
    v = c((y[0].float() + y[1].float()).bfloat16()) * z * torch.sigmoid(z)
    v = (v * (v.pow(2).mean(-1, keepdim=True) + 4e-5).rsqrt() * c(kw)).reshape(-1, di)
    s = c(((last[0] + last[1]) * 0.5).bfloat16()).transpose(1, 2).reshape(-1, di)
    s = (s - s.mean(-1, keepdim=True)) * (s.var(-1, unbiased=False, keepdim=True) + 1e-5).rsqrt() * c(qw) + c(qb)
    for t, x, m in zip(got, (v, s), w):
        ref, mag = x @ c(m).t(), x.abs() @ c(m).abs().t()
        assert ((c(t[:-1]) - ref).abs() <= 2.0 ** -8 * (ref.abs() + mag) + 2.0 ** -18 * (1 + mag)).all() and (t[-1] == 3.0).all()
    for who, field, bad in ((a, "dtype", L.ISSM_F32), (a, "d_inner", di + 4), (q, "njobs", 1), (q.job[0], "tokens", rows[0] + 1),
                            (q.job[1], "turn", 1), (q.job[1], "nin", di + 32)):
        was = getattr(who, field)
        setattr(who, field, bad)
        assert lib.issm_layer_end(C.byref(a), C.byref(q)) != 0, field
        setattr(who, field, was)


@pytest.mark.parametrize("B,Ln,K", [(1, 130, 40), (2, 64, 256), (3, 1, 1)])
@pytest.mark.parametrize("mask", [None, "weights", "drop"])
def test_layer_without_a_gradient(B, Ln, K, mask):
    """The layer's shorter chain against the one that is differentiated: up to the output projections the same kernels on the
    same operands, except for the two norms, whose results may round to the neighbouring bf16 number; through the projection that
    is 2^-7 of its terms' magnitudes (8 bits, and the result's own rounding)."""
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(B * Ln + K)
    layer = MultiHeadISSMScan(d_model=288, d_state=K, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16()
    key, query = torch.randn(B, Ln, 288).cuda().bfloat16(), torch.randn(B, K, 288).cuda().bfloat16()
    dist = torch.randn(B, Ln, K, 16).cuda().bfloat16()
    m = None if mask is None else torch.rand(B, Ln, K).cuda() if mask == "weights" else torch.rand(B, Ln, K).cuda() < 0.3
    want = layer(key, query, dist, None, m)
    with torch.no_grad():
        got = layer(key, query, dist, None, m)
    assert want[0].requires_grad and not got[0].requires_grad
    with torch.no_grad():
        for a, b, w in zip(got, want, (layer.out_key_proj.weight, layer.out_query_proj.weight)):
            assert a.shape == b.shape and torch.isfinite(a).all()
            # rows of the normed operand have unit mean square (times the norm's weight, 1 at initialisation)
            size = w.float().abs().sum(1) * 1.0
            assert ((a - b).float().abs() <= 2.0 ** -7 * size + 2.0 ** -7 * b.float().abs()).all()
    layer.requires_grad_(False)
    frozen = layer(key, query, dist, None, m)
    assert all(torch.equal(a, b) for a, b in zip(frozen, got))


@pytest.mark.parametrize("D,H,G,per_head_d,B,Ln,K,mask", [(288, 8, 1, True, 1, 130, 40, "weights"), (288, 8, 1, False, 2, 70, 33, None),
                                                          (64, 4, 2, False, 3, 65, 20, "drop"), (96, 6, 3, True, 2, 1, 1, None),
                                                          (160, 8, 2, False, 1, 200, 64, "weights"), (512, 8, 1, True, 1, 77, 130, None)])
def test_layer_without_a_gradient_against_fp64(D, H, G, per_head_d, B, Ln, K, mask):
    """The layer's shorter chain, row by row of its results, against an fp64 evaluation on the same bf16 parameters and inputs:
    several widths, groups and forms of D, norms whose eps counts.  A rounding to bf16 is 2^-8 / sqrt 12 of a value on average; a
    dozen to sixteen of them lie on the way from an input to a result (projection, two convolutions, dt, B, C, the scan's operands,
    its two outputs and their sum, the norm, the result), together 3.9e-3 to 4.5e-3 of a row (measured: 3.0e-3 to 4.9e-3, single
    rows of 64 features up to 1.5e-2).  A quarter of an eps, another head's D or A, another norm's eps move the rows by 0.05 to 1.
    """
    from dest3d_amd.scan_module import MultiHeadISSMScan
    from oracle.module_ref import multi_head_issm_scan_ref
    torch.manual_seed(D + Ln)
    layer = MultiHeadISSMScan(d_model=D, d_state=K, d_dist=16, chunk_size=256, nheads=H, ngroups=G, expand=1)
    if not per_head_d:
        layer.D = torch.nn.Parameter(torch.empty(H, D // H))
    with torch.no_grad():
        layer.D.normal_()
        for p in (layer.key_norm.weight, layer.query_norm.weight, layer.query_norm.bias):
            p.add_(0.3 * torch.randn_like(p))
    layer.key_norm.eps, layer.query_norm.eps = 0.02, 0.1
    layer = layer.cuda().bfloat16()
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    x = bf(B, Ln, D), bf(B, K, D), 0.5 * bf(B, Ln, K, 16)
    m = None if mask is None else torch.rand(B, Ln, K).cuda() if mask == "weights" else torch.rand(B, Ln, K).cuda() < 0.3
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    with torch.no_grad():
        before = count()
        got = layer(*x, None, m)
        assert count() - before <= (5 if mask == "drop" else 3)     # one buffer between inputs and outputs: this is the shorter chain
    want = layer(*x, None, m)
    sd = {k: v.detach().double().cpu() for k, v in layer.state_dict().items()}
    cfg = dict(nheads=H, ngroups=G, d_inner=D, d_state=K, use_biscan=True, key_eps=0.02, query_eps=0.1)
    ref = multi_head_issm_scan_ref(sd, cfg, *(t.double().cpu() for t in x), None if m is None else m.cpu())
    for out in (got, want):
        for a, r in zip(out, ref):
            off = (a.detach().double().cpu() - r).norm(dim=-1) / r.norm(dim=-1)
            assert off.mean() <= 2.0 ** -7 and off.max() <= 2.0 ** -5


def test_layer_without_a_gradient_in_a_graph():
    """The shorter chain recorded into a HIP graph: every replay, with eager work and other inputs between, gives the eager result."""
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(3)
    layer = MultiHeadISSMScan(d_model=288, d_state=64, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16()
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    x = [bf(1, 200, 288), bf(1, 64, 288), bf(1, 200, 64, 16)]
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(*x, None, None)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(*x, None, None)
        for _ in range(4):
            for t in x:
                t.copy_(bf(*t.shape))
            want = layer(*x, None, None)
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(out, want))


@pytest.mark.parametrize("reentrant", [True, False])
def test_checkpointed_layers(reentrant):
    """A layer under reentrant checkpointing runs without gradients first and with them afterwards, one under the other kind with
    them twice: the same kernels, hence the outputs and gradients of the layers that are not checkpointed, bit for bit.  Steps long
    enough for chunks out of a tile's range, where the kernels for either case round differently."""
    from torch.utils.checkpoint import checkpoint
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(9)
    layers = [MultiHeadISSMScan(d_model=288, d_state=40, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16() for _ in range(3)]
    for layer in layers:
        layer.dt_bias.data += 6.0
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    key, query, dist, dkey, dquery = bf(2, 130, 288), bf(2, 40, 288), bf(2, 130, 40, 16), bf(2, 130, 288), bf(2, 40, 288)

    def step(run):
        k, q = key.clone().requires_grad_(), query.clone().requires_grad_()
        hk, hq = k, q
        for layer in layers:
            layer.zero_grad(set_to_none=True)
            ok, oq = run(layer, hk, hq)
            hk, hq = hk + ok, hq + oq
        torch.autograd.backward((hk, hq), (dkey, dquery))
        return hk, hq, k.grad, q.grad, *(p.grad for layer in layers for p in layer.parameters())

    want = step(lambda layer, k, q: layer(k, q, dist, None))
    got = step(lambda layer, k, q: checkpoint(layer, k, q, dist, None, use_reentrant=reentrant))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("B,Ln,K", [(2, 130, 40), (4, 1000, 40)])
def test_checkpointed_segments_of_several_layers(B, Ln, K):
    """Segments of two layers under reentrant checkpointing, one scene's products and several scenes': only a segment's own inputs want a
    gradient in its first run, and the layers behind the first take training's kernels in it all the same."""
    from torch.utils.checkpoint import checkpoint
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(9)
    layers = [MultiHeadISSMScan(d_model=288, d_state=K, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16() for _ in range(4)]
    for layer in layers:
        layer.dt_bias.data += 6.0   # steps long enough for chunks out of a tile's range
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    key, query, dist, dkey, dquery = bf(B, Ln, 288), bf(B, K, 288), bf(B, Ln, K, 16), bf(B, Ln, 288), bf(B, K, 288)

    def segment(first):
        def run(k, q):
            for layer in layers[first:first + 2]:
                ok, oq = layer(k, q, dist, None)
                k, q = k + ok, q + oq
            return k, q
        return run

    def step(wrap):
        k, q = key.clone().requires_grad_(), query.clone().requires_grad_()
        for layer in layers:
            layer.zero_grad(set_to_none=True)
        out = wrap(segment(2), *wrap(segment(0), k, q))
        torch.autograd.backward(out, (dkey, dquery))
        return *out, k.grad, q.grad, *(p.grad for layer in layers for p in layer.parameters())

    want = step(lambda f, *x: f(*x))
    got = step(lambda f, *x: checkpoint(f, *x, use_reentrant=True))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    with torch.no_grad():
        plain = segment(0)(key, query)
    with torch.inference_mode():   # no backward can follow there, although forward-mode derivatives are off as in an autograd function
        assert all(torch.equal(a, b) for a, b in zip(segment(0)(key, query), plain))


@pytest.mark.parametrize("reentrant", [True, False])
def test_both_runs_of_a_segment_with_a_frozen_layer(reentrant):
    """A layer that nothing is differentiated through, in a segment that is run twice."""
    from torch.utils.checkpoint import checkpoint
    from dest3d_amd.scan_module import MultiHeadISSMScan
    torch.manual_seed(9)
    layer = MultiHeadISSMScan(d_model=288, d_state=40, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16().requires_grad_(False)
    layer.dt_bias.data += 6.0
    bf = lambda *s: torch.randn(*s).cuda().bfloat16()
    key, query, dist, scale, seen = bf(2, 130, 288), bf(2, 40, 288), bf(2, 130, 40, 16), bf(2, 130, 288).requires_grad_(), []

    def segment(s):
        seen.append(layer(key, query, dist, None))
        return seen[-1][0] * s

    checkpoint(segment, scale, use_reentrant=reentrant).sum().backward()
    assert len(seen) == 2 and all(torch.equal(a, b) for a, b in zip(*seen)) and torch.equal(scale.grad, seen[0][0])


@pytest.mark.parametrize("B,Ln,K", [(3, 1000, 40), (8, 1024, 64), (8, 1024, 160), (8, 1024, 77)])
def test_layer_without_a_gradient_of_several_scenes(B, Ln, K):
    """Beyond the sizes whose single products the layer's own kernel takes, up to the chain's limit, the convolutions and the generation in
    one launch and, with an even and an odd number of queries, in two; bounds as above."""
    test_layer_without_a_gradient(B, Ln, K, "weights")


@pytest.mark.parametrize("D,B,short", [(32, 110, True), (64, 60, True), (64, 61, False), (128, 31, True), (128, 32, False), (288, 8, True), (288, 9, False), (320, 4, True), (320, 5, False),
                                       (384, 3, True), (384, 4, False)])
def test_layer_without_a_gradient_takes_the_shorter_chain_where_it_is_the_faster(D, B, short):
    """Scenes of 1024 tokens, told by the number of allocations."""
    from dest3d_amd.scan_module import MultiHeadISSMScan
    layer = MultiHeadISSMScan(d_model=D, d_state=8, d_dist=16, chunk_size=256, nheads=8, expand=1).cuda().bfloat16()
    x = [torch.zeros(s, device="cuda", dtype=torch.bfloat16) for s in ((B, 1024, D), (B, 8, D), (B, 1024, 8, 16))]
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    with torch.no_grad():
        before = count()
        layer(*x, None, None)
        assert (count() - before <= 3) == short


@pytest.mark.parametrize("D,H,Ln", [(512, 8, 1000), (640, 10, 300)])
def test_wide_layer_without_a_gradient_against_fp64(D, H, Ln):
    test_layer_without_a_gradient_against_fp64(D, H, 1, True, 1, Ln, 33, "weights")
