"""issm_linear_fwd (libissm_hip.so) and the projections that take it: y = x w^T against an fp64 product of the same bf16
operands."""
import ctypes as C

import pytest
import torch

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
                ("nout", C.c_int32)]


class Args(C.Structure):
    _fields_ = [("job", Job * 2), ("njobs", C.c_int32), ("dtype", C.c_int32), ("stream", C.c_void_p)]


@pytest.mark.parametrize("shapes", [[(1, 32, 1)], [(64, 288, 32)], [(65, 288, 33), (16, 288, 586)], [(17, 256, 31), (130, 544, 35)],
                                    [(1023, 320, 64)], [(3, 96, 7), (0, 32, 5)]])
def test_linear_at_its_remainders(shapes):
    """Rows, outputs and steps that fill no tile, batch of fragments or aligned store; one and two products a launch."""
    lib = L.load()
    a, kept = Args(), []
    for i, (t, nin, nout) in enumerate(shapes):
        x, w, ref = _operands(t, nin, nout, 7 * i + t)
        xd, wd = x.cuda(), w.cuda()
        y = torch.full((t + 1, nout), 3.0, dtype=torch.bfloat16, device="cuda")     # a row behind the result
        a.job[i] = Job(xd.data_ptr(), wd.data_ptr(), y.data_ptr(), t, nin, nout)
        kept.append((x, w, ref, xd, wd, y))
    a.njobs, a.dtype, a.stream = len(shapes), L.ISSM_BF16, L.current_stream_ptr(torch.device("cuda", 0))
    assert lib.issm_linear_fwd(C.byref(a)) == 0
    torch.cuda.synchronize()
    for x, w, ref, _, _, y in kept:
        _close(y[:-1], x, w, ref)
        assert (y[-1] == 3.0).all()


def test_linear_refuses_what_it_does_not_take():
    lib = L.load()
    x = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda")
    good = (x.data_ptr(), x.data_ptr(), x.data_ptr(), 8, 32, 8)
    for job, n, dtype in ((good, 3, L.ISSM_BF16), (good, 1, L.ISSM_F32), ((*good[:4], 33, 8), 1, L.ISSM_BF16), ((*good[:4], 0, 8), 1, L.ISSM_BF16),
                          ((x.data_ptr() + 2, *good[1:]), 1, L.ISSM_BF16), ((None, *good[1:]), 1, L.ISSM_BF16), ((*good[:3], -1, 32, 8), 1, L.ISSM_BF16)):
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
