"""issm_layer_grads (libissm_hip.so): the gradients of a layer's small parameters from the parts that the backwards leave, against fp64
sums, and the parts themselves against the entry points that sum them."""
import ctypes as C

import pytest
import torch

from dest3d_amd import _lib as L

pytestmark = pytest.mark.gpu


class Args(C.Structure):
    _fields_ = [("conv", C.c_void_p), ("gen", C.c_void_p), ("norm", C.c_void_p), ("conv_rows", C.c_int32), ("gen_rows", C.c_int32),
                ("norm_rows", C.c_int32), ("C", C.c_int32), ("H", C.c_int32), ("G", C.c_int32), ("di", C.c_int32), ("K", C.c_int32),
                ("dA", C.c_void_p), ("A", C.c_void_p), ("dD", C.c_void_p), ("nD", C.c_int32), ("dtype", C.c_int32),
                ("out", C.c_void_p), ("stream", C.c_void_p)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,Cc,H,G,di,K,nD,batch", [
    ((128, 256, 2048), 290, 8, 1, 288, 256, 8, 2), ((1, 1, 1), 3, 1, 1, 1, 1, 1, 1), ((17, 33, 65), 36, 10, 1, 32, 65, 320, 3),
    ((0, 0, 0), 34, 4, 4, 30, 63, 30, 1), ((31, 16, 31), 7, 2, 3, 5, 130, 300, 0), ((33, 512, 513), 130, 8, 2, 128, 0, 8, 1)])
def test_sums_of_the_parts(dtype, rows, Cc, H, G, di, K, nD, batch):
    lib = L.load()
    g = torch.Generator().manual_seed(Cc + K)
    rnd = lambda *s: torch.randn(*s, generator=g)
    R0 = H + 2 * G
    conv, gen, bias, norm = rnd(rows[0], 2, 8, Cc), rnd(rows[1], R0, 16), rnd(rows[1], R0), rnd(rows[2], di)
    dA, A, dD, dh0 = rnd(H, K), -torch.rand(H, 1, generator=g).expand(H, K).contiguous(), rnd(nD), rnd(max(batch, 1), di, max(K, 1))

    def laid(f):   # the results one behind the other, f applied to each part before its sum
        c, s = f(conv.double()).sum(0), f(gen.double()).sum(0)
        parts = [t for d in range(2) for t in (c[d, :7].t(), c[d, 7])]
        parts += [s[:H], s[H:], f(bias.double()).sum(0)[:H], f(dA.double()).sum(1) * (f(A.double())[:, 0] if K else 0)]
        return torch.cat([t.reshape(-1) for t in parts] + [f(dD.double()), f(norm.double()).sum(0)])
    dev = [t.cuda() for t in (conv, torch.cat([gen.flatten(), bias.flatten()]), norm, dA, A, dD, dh0)]
    n = 16 * Cc + 16 * R0 + 2 * H + nD + di
    out = torch.full((n + 1,), 3.0, dtype=dtype, device="cuda")
    turned = torch.full((dh0.numel() + 1,), 3.0, dtype=dtype, device="cuda")
    code = L.ISSM_BF16 if dtype == torch.bfloat16 else L.ISSM_F32
    stream = L.current_stream_ptr(torch.device("cuda", 0))
    a = Args(*(t.data_ptr() for t in dev[:3]), *rows, Cc, H, G, di, K, *(t.data_ptr() for t in dev[3:6]), nD, code, out.data_ptr(), stream)
    t = L.TransposeArgs()
    t.batch, t.rows, t.cols, t.in_dtype, t.out_dtype, t.alpha = batch, di, K, L.ISSM_F32, code, 1.0
    t.in0, t.out, t.stream = dev[6].data_ptr(), turned.data_ptr(), stream
    assert lib.issm_layer_grads(C.byref(a), C.byref(t)) == 0
    torch.cuda.synchronize()
    ref, size = laid(lambda v: v), laid(torch.abs)
    # additions of 2^-24 of the magnitudes, and one rounding to the result's type
    bound = 2.0 ** -24 * (max(*rows, K) + 2) * size + (2.0 ** -8 if code == L.ISSM_BF16 else 2.0 ** -24) * ref.abs()
    assert ((out[:-1].double().cpu() - ref).abs() <= bound).all() and out[-1] == 3.0
    if batch and K:
        assert torch.equal(turned[:-1].view(batch, K, di).cpu(), dh0.transpose(1, 2).to(dtype))
    assert turned[-1] == 3.0 and (batch and K or (turned == 3.0).all())
    a.H = 0
    assert lib.issm_layer_grads(C.byref(a), None) != 0
    assert lib.issm_layer_grads(None, None) != 0


class Producers(C.Structure):
    _fields_ = [("dtok", C.c_void_p), ("stride", C.c_int64), ("dtail", C.c_void_p)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens,K,H,G,weighted", [(1, 64, 8, 1, True), (37, 128, 10, 1, False), (130, 33, 4, 4, True), (9, 64, 2, 2, True)])
def test_parts_of_the_generation(dtype, tokens, K, H, G, weighted):
    """issm_param_gen_bwd_part writes what issm_param_gen_bwd does, its sums undone and its bias gradients in two places."""
    lib = L.load()
    code = L.ISSM_BF16 if dtype == torch.bfloat16 else L.ISSM_F32
    gen = torch.Generator().manual_seed(tokens)
    io = lambda *s: torch.randn(*s, generator=gen).to(dtype).cuda()
    R0, R = H + 2 * G, H + 4 * G
    dist, W, ddt = io(tokens, K, 16), torch.randn(R0, 16, generator=gen).cuda(), io(tokens, H, K)
    grads, raw, w = [io(tokens, G, K) for _ in range(4)], io(tokens, H, K), torch.rand(tokens, K, generator=gen).cuda()
    blocks = lib.issm_param_gen_bwd_blocks(tokens)
    f32 = lambda *s: torch.full(s, 3.0, device="cuda")

    def args(ddist):
        a = L.PGenArgs()
        a.tokens, a.K, a.M, a.H, a.G, a.dtype, a.has_back = tokens, K, 16, H, G, code, 1
        a.dist, a.W, a.ddt, a.ddist = dist.data_ptr(), W.data_ptr(), ddt.data_ptr(), ddist.data_ptr()
        a.dBm, a.dCm, a.dBm_back, a.dCm_back = (t.data_ptr() for t in grads)
        if weighted:
            a.weights, a.dt_raw = w.data_ptr(), raw.data_ptr()
        a.stream = L.current_stream_ptr(torch.device("cuda", 0))
        return a
    whole, part = torch.empty_like(dist), torch.empty_like(dist)
    a, dbias, total, dW, scratch = args(whole), f32(tokens, R), f32(R), f32(R0, 16), f32(blocks, R0, 16)
    a.dbias, a.dbias_sum, a.dW, a.dw_partial = dbias.data_ptr(), total.data_ptr(), dW.data_ptr(), scratch.data_ptr()
    assert lib.issm_param_gen_bwd(C.byref(a)) == 0
    b, parts = args(part), f32(blocks * R0 * 17 + 1)
    tok, tail = torch.full((tokens, H + 3), 3.0, dtype=dtype, device="cuda"), torch.full((2, tokens, 2 * G), 3.0, dtype=dtype, device="cuda")
    b.dw_partial = parts.data_ptr()
    to = Producers(tok.data_ptr(), H + 3, tail.data_ptr())
    assert lib.issm_param_gen_bwd_part(C.byref(b), C.byref(to)) == 0
    torch.cuda.synchronize()
    assert torch.equal(whole, part) and torch.equal(scratch.flatten(), parts[:blocks * R0 * 16])
    assert torch.equal(tok[:, :H], dbias[:, :H].to(dtype)) and (tok[:, H:] == 3.0).all() and parts[-1] == 3.0
    assert torch.equal(tail[0], dbias[:, H:R0].to(dtype)) and torch.equal(tail[1], dbias[:, R0:].to(dtype))
    sums = parts[blocks * R0 * 16:-1].view(blocks, R0).double().sum(0)
    assert ((sums - dbias[:, :R0].double().sum(0)).abs() <= 2.0 ** -22 * dbias[:, :R0].double().abs().sum(0)).all()
    to.stride = H - 1
    assert lib.issm_param_gen_bwd_part(C.byref(b), C.byref(to)) != 0
    assert lib.issm_param_gen_bwd_part(C.byref(b), None) != 0


def _turn(src, other, alpha, out):
    code = lambda t: L.ISSM_BF16 if t.dtype == torch.bfloat16 else L.ISSM_F32
    t = L.TransposeArgs()
    t.batch, t.rows, t.cols, t.in_dtype, t.out_dtype, t.alpha = *src.shape, code(src), code(out), alpha
    t.in0, t.in1, t.out, t.stream = src.data_ptr(), None if other is None else other.data_ptr(), out.data_ptr(), L.current_stream_ptr(src.device)
    return t


@pytest.mark.parametrize("dtype,to", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("rows,cols,B,R,Cc", [(1, 4, 1, 1, 1), (5, 256, 2, 65, 64), (130, 288, 0, 3, 5), (7, 260, 1, 64, 130), (33, 1024, 3, 70, 33)])
def test_behind_the_scan_with_gradients(dtype, to, rows, cols, B, R, Cc):
    """The norm of a sum and the turned average in one launch: the bits of the sum, the norm and the transposition on their own."""
    lib = L.load()
    g = torch.Generator().manual_seed(rows + cols)
    x, x2, z = (torch.randn(rows, cols, generator=g).to(dtype).cuda() for _ in range(3))
    w = torch.randn(cols, generator=g).to(dtype).cuda()
    s0, s1 = (torch.randn(B, R, Cc, generator=g).cuda() for _ in range(2))
    full = lambda *s, dt=dtype: torch.full(s, 3.0, dtype=dt, device="cuda")
    from dest3d_amd.layernorm_gated import _norm_args
    want, y, ssum = full(rows, cols), full(rows + 1, cols), full(rows + 1, cols)
    rstd, rstd2, turned, alone = full(rows, dt=torch.float32), full(rows, dt=torch.float32), full(B, Cc, R, dt=to), full(B, Cc, R, dt=to)
    total = x + x2
    a = _norm_args(total, z, w, 1e-5, None, False)
    a.y, a.y_row_stride, a.rstd = want.data_ptr(), cols, rstd.data_ptr()
    assert lib.issm_gated_rmsnorm_fwd(C.byref(a)) == 0
    assert lib.issm_transpose_states(C.byref(_turn(s0, s1, 0.5, alone))) == 0
    a.x, a.y, a.rstd = x.data_ptr(), y.data_ptr(), rstd2.data_ptr()
    t = _turn(s0, s1, 0.5, turned)
    assert lib.issm_layer_behind(C.byref(a), C.c_void_p(x2.data_ptr()), C.c_void_p(ssum.data_ptr()), C.byref(t)) == 0
    torch.cuda.synchronize()
    assert torch.equal(ssum[:rows], total) and torch.equal(y[:rows], want) and torch.equal(rstd, rstd2) and torch.equal(turned, alone)
    assert (ssum[rows] == 3.0).all() and (y[rows] == 3.0).all()
    assert lib.issm_layer_behind(C.byref(a), None, C.c_void_p(ssum.data_ptr()), C.byref(t)) != 0
    a.layer_norm, a.mean = 1, rstd.data_ptr()
    assert lib.issm_layer_behind(C.byref(a), C.c_void_p(x2.data_ptr()), C.c_void_p(ssum.data_ptr()), C.byref(t)) != 0


class LayerParams(C.Structure):
    _fields_ = [("src", C.c_void_p * 9), ("n", C.c_int32 * 9), ("dtype", C.c_int32 * 9), ("a_log", C.c_int32), ("K", C.c_int32),
                ("out", C.c_void_p), ("A", C.c_void_p), ("stream", C.c_void_p)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sizes,K,B,R,Cc", [((3, 0, 1, 500, 2, 7, 8, 8, 1), 33, 2, 65, 70), ((0,) * 9, 4, 1, 64, 64), ((9,) * 9, 0, 0, 1, 1)])
def test_begin_of_a_layer(dtype, sizes, K, B, R, Cc):
    """The small parameters and the turned queries in one launch: the bits of either on its own."""
    lib = L.load()
    g = torch.Generator().manual_seed(K)
    arrays, q = [torch.randn(n, generator=g).to(dtype).cuda() for n in sizes], torch.randn(B, R, Cc, generator=g).to(dtype).cuda()
    out, A, out2, A2 = (torch.full((n + 1,), 3.0, device="cuda") for n in 2 * (sum(sizes), sizes[7] * K))
    turned = torch.full((B, Cc, R), 3.0, dtype=dtype, device="cuda")
    p = LayerParams()
    for i, t in enumerate(arrays):
        p.src[i], p.n[i], p.dtype[i] = t.data_ptr(), t.numel(), L.ISSM_BF16 if dtype == torch.bfloat16 else L.ISSM_F32
    p.a_log, p.K, p.out, p.A, p.stream = 7, K, out.data_ptr(), A.data_ptr(), L.current_stream_ptr(q.device)
    assert lib.issm_layer_params(C.byref(p)) == 0
    p.out, p.A = out2.data_ptr(), A2.data_ptr()
    assert lib.issm_layer_begin(C.byref(p), C.byref(_turn(q, None, 1.0, turned))) == 0
    torch.cuda.synchronize()
    assert torch.equal(out, out2) and torch.equal(A, A2) and torch.equal(turned, q.transpose(1, 2))
    assert lib.issm_layer_begin(C.byref(p), None) != 0
