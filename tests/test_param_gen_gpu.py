"""Generation of dt / B / C from the distance encoding (libissm_hip.so) against an fp64 evaluation of the
reference's formulas (models/dest_module.py:541-553): two Linear layers over dist, transposes, broadcast
biases.  fp32: rel. error <= 1e-5 forward, 1e-4 gradients; bf16: <= 1e-2 / 2e-2 (outputs are rounded to
bf16; sums run in fp32)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(dist, W, bias, H, G, has_back):
    base = torch.einsum("rm,blkm->blrk", W, dist)
    R0 = H + 2 * G
    main = base + bias[..., :R0].unsqueeze(-1)
    outs = [main[:, :, :H], main[:, :, H:H + G], main[:, :, H + G:]]
    if has_back:
        outs.append(base[:, :, H:H + G] + bias[..., R0:R0 + G].unsqueeze(-1))
        outs.append(base[:, :, H + G:] + bias[..., R0 + G:].unsqueeze(-1))
    return outs


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


CASES = [
    # B, L, K, H, G, back, dtype
    (2, 37, 256, 8, 1, True, torch.float32),
    (1, 16, 256, 8, 2, True, torch.float32),
    (3, 5, 100, 4, 1, False, torch.float32),
    (1, 33, 300, 2, 2, True, torch.float32),
    (2, 64, 256, 8, 1, True, torch.bfloat16),
    (1, 19, 77, 3, 1, False, torch.bfloat16),
    (1, 11, 50, 3, 1, True, torch.bfloat16),     # K even, not a multiple of 4
    (2, 6, 77, 2, 1, False, torch.float32),      # K odd
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_L%d_K%d_H%d_G%d_back%d_%s" % (*c[:5], int(c[5]), str(c[6])[6:]))
def test_scan_params_match_fp64(case):
    from dest3d_amd.param_gen import scan_params
    B, L, K, H, G, back, dtype = case
    g = torch.Generator().manual_seed(1234 + L + K)
    M, R0 = 16, H + 2 * G
    R = R0 + (2 * G if back else 0)
    dist = torch.randn(B, L, K, M, generator=g).to(dtype).cuda().requires_grad_()
    W = (0.3 * torch.randn(R0, M, generator=g)).cuda().requires_grad_()
    bias = torch.randn(B, L, R, generator=g).cuda().requires_grad_()
    outs = scan_params(dist, W, bias, H, G, back)
    d64, W64, b64 = (t.detach().double().requires_grad_() for t in (dist, W, bias))
    refs = _ref(d64, W64, b64, H, G, back)
    assert len(outs) == len(refs)
    ftol, gtol = (1e-5, 1e-4) if dtype == torch.float32 else (1e-2, 2e-2)
    for o, r in zip(outs, refs):
        assert o.shape == r.shape and o.dtype == dtype and o.is_contiguous()
        assert _rel(o, r) <= ftol
    # the last output gets no gradient: absent gradients count as zero
    gouts = [torch.randn(o.shape, generator=g).to(dtype).cuda() for o in outs[:-1]]
    torch.autograd.backward(list(outs[:-1]), gouts)
    torch.autograd.backward(refs[:-1], [t.double() for t in gouts])
    assert _rel(dist.grad, d64.grad) <= gtol
    assert _rel(W.grad, W64.grad) <= gtol
    assert _rel(bias.grad, b64.grad) <= gtol
    if back:
        assert bias.grad[..., -G:].abs().max().item() == 0.0


WCASES = [
    (2, 21, 256, 8, 1, True, torch.float32),
    (1, 9, 100, 4, 2, False, torch.float32),
    (2, 33, 128, 8, 1, True, torch.bfloat16),
    (1, 7, 52, 3, 1, True, torch.bfloat16),
    (1, 5, 50, 2, 1, True, torch.bfloat16),
    (1, 4, 33, 2, 1, False, torch.float32),
]


@pytest.mark.parametrize("case", WCASES, ids=lambda c: "B%d_L%d_K%d_H%d_G%d_back%d_%s" % (*c[:5], int(c[5]), str(c[6])[6:]))
def test_scan_params_with_locality_weights(case):
    """dt = softplus(raw) * weights (models/dest_module.py:553-557), gradients of dist, W, bias and weights."""
    import torch.nn.functional as F
    from dest3d_amd.param_gen import scan_params
    B, L, K, H, G, back, dtype = case
    g = torch.Generator().manual_seed(99 + L + K)
    M, R0 = 16, H + 2 * G
    R = R0 + (2 * G if back else 0)
    dist = torch.randn(B, L, K, M, generator=g).to(dtype).cuda().requires_grad_()
    W = (0.6 * torch.randn(R0, M, generator=g)).cuda().requires_grad_()
    bias = (2.0 * torch.randn(B, L, R, generator=g)).cuda().requires_grad_()
    bias.data[0, 0, 0] = 40.0   # softplus above torch's threshold
    wts = torch.rand(B, L, K, generator=g)
    wts[0, :, ::7] = 0.0        # dropped entries
    wts = wts.cuda().requires_grad_()
    outs = scan_params(dist, W, bias, H, G, back, weights=wts)
    d64, W64, b64, w64 = (t.detach().double().requires_grad_() for t in (dist, W, bias, wts))
    refs = _ref(d64, W64, b64, H, G, back)
    raw = refs[0]
    if dtype == torch.bfloat16:   # the saved raw value is rounded to the I/O dtype before softplus, as a bf16 module's is
        raw = raw + (raw.detach().float().bfloat16().double() - raw.detach())
    refs[0] = F.softplus(raw) * w64.unsqueeze(2)
    ftol, gtol = (1e-5, 2e-4) if dtype == torch.float32 else (1e-2, 3e-2)
    for o, r in zip(outs, refs):
        assert o.shape == r.shape and o.dtype == dtype
        assert _rel(o, r) <= ftol
    gouts = [torch.randn(o.shape, generator=g).to(dtype).cuda() for o in outs]
    torch.autograd.backward(list(outs), gouts)
    torch.autograd.backward(refs, [t.double() for t in gouts])
    assert _rel(dist.grad, d64.grad) <= gtol
    assert _rel(W.grad, W64.grad) <= gtol
    assert _rel(bias.grad, b64.grad) <= gtol
    assert _rel(wts.grad, w64.grad) <= gtol


def test_scan_params_rejects_unbuilt_shapes():
    from dest3d_amd import _lib as L
    import ctypes as C
    lib = L.load()
    a = L.PGenArgs()
    a.tokens, a.K, a.M, a.H, a.G = 4, 8, 8, 2, 1
    assert lib.issm_param_gen_fwd(C.byref(a)) == -5
    a.M, a.H = 16, 12
    assert lib.issm_param_gen_fwd(C.byref(a)) == -5
    a.H = 2
    assert lib.issm_param_gen_fwd(C.byref(a)) == -1


@pytest.mark.parametrize("B,L,K,H,G,di,weighted", [(1, 1, 1, 1, 1, 2, True), (2, 9, 50, 8, 1, 288, True), (1, 37, 77, 3, 2, 36, False),
                                                   (2, 1030, 6, 2, 1, 512, True), (1, 2051, 3, 2, 1, 520, False), (3, 5, 700, 4, 4, 64, True)])
def test_generation_and_convolutions_in_one_launch(B, L, K, H, G, di, weighted):
    """issm_conv_param_gen_fwd against the two launches it stands for: the same operations in the same order, so the same bits.
    Tokens that fill no thread, workgroups of several tokens and of a part of one, 4, 8 and 16 tokens a thread of the convolutions."""
    import ctypes as C
    from dest3d_amd import _lib as LB
    lib, dev, bf = LB.load(), "cuda", torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(L + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    Cc, W = di + 2 * G, 2 * di + 2 * G + H
    zx, w, bias = rnd(B, L, W).to(bf), rnd(2, Cc, 7), rnd(2, Cc)
    dist, pw, add, wts = rnd(B, L, K, 16).to(bf), 0.3 * rnd(H + 2 * G, 16), rnd(H), torch.rand(B, L, K, generator=g, device=dev)
    stream = LB.current_stream_ptr(torch.device("cuda", 0))

    def run(joined):
        o = [torch.full(s, 7.0, device=dev, dtype=bf) for s in ((2, B, L, di), (2, B, L, 2 * G), (2, B, L, Cc), (B, L, H, K),
                                                                *[(B, L, G, K)] * 4)]
        c = LB.DwConvArgs(batch=B, seqlen=L, channels=Cc, nsets=2, taps=7, dtype=LB.ISSM_BF16, u=zx.data_ptr() + 2 * di,
                          u_batch_stride=L * W, u_token_stride=W, w=w.data_ptr(), bias=bias.data_ptr(), y=o[0].data_ptr(),
                          pre=None if joined else o[2].data_ptr(), stream=stream, split=di,
                          y_tail=None if joined else o[1].data_ptr(), chain=1)
        p = LB.PGenArgs(tokens=B * L, K=K, M=16, H=H, G=G, dtype=LB.ISSM_BF16, has_back=1, dist=dist.data_ptr(), W=pw.data_ptr(),
                        dt=o[3].data_ptr(), Bm=o[4].data_ptr(), Cm=o[5].data_ptr(), Bm_back=o[6].data_ptr(),
                        Cm_back=o[7].data_ptr(), weights=wts.data_ptr() if weighted else None, stream=stream,
                        tok=zx.data_ptr() + 2 * (di + Cc), tok_stride=W, tok_add=add.data_ptr(),
                        tail=None if joined else o[1].data_ptr())
        if joined:
            LB.check(lib.issm_conv_param_gen_fwd(C.byref(c), C.byref(p)), "joined")
            for who, field, bad in ((c, "chain", 0), (c, "split", di - 1), (c, "dtype", LB.ISSM_F32), (p, "tokens", B * L + 1), (p, "has_back", 0)):
                was = getattr(who, field)
                setattr(who, field, bad)
                assert lib.issm_conv_param_gen_fwd(C.byref(c), C.byref(p)) != 0, field
                setattr(who, field, was)
        else:
            LB.check(lib.issm_dwconv_silu_fwd(C.byref(c)), "conv")
            LB.check(lib.issm_param_gen_fwd_only(C.byref(p)), "generation")
        torch.cuda.synchronize()
        return [o[i] for i in (0, 3, 4, 5, 6, 7)]

    for got, want in zip(run(True), run(False)):
        assert torch.equal(got, want)


def test_rows_beyond_32_bit_offsets():
    """A token with so many queries that its rows are not within 31-bit byte offsets: the kernels with 64-bit places, against the same
    queries in a call of their own."""
    import ctypes as C
    from dest3d_amd import _lib as L
    lib = L.load()
    K, H, G, few = 53_700_001, 10, 1, 777
    torch.manual_seed(4)
    W, bias = torch.randn(H + 2 * G, 16).cuda(), torch.randn(1, H + 2 * G).cuda()
    dist = torch.zeros(1, K, 16, dtype=torch.bfloat16, device="cuda")
    dist[:, -few:] = torch.randn(1, few, 16).bfloat16().cuda()

    def run(d):
        k = d.shape[1]
        dt, Bm, Cm = (torch.full((1, n, k), 3.0, dtype=torch.bfloat16, device="cuda") for n in (H, G, G))
        a = L.PGenArgs()
        a.tokens, a.K, a.M, a.H, a.G, a.dtype, a.has_back = 1, k, 16, H, G, L.ISSM_BF16, 0
        a.dist, a.W, a.bias, a.dt, a.Bm, a.Cm = (t.data_ptr() for t in (d, W, bias, dt, Bm, Cm))
        a.stream = L.current_stream_ptr(d.device)
        assert lib.issm_param_gen_fwd(C.byref(a)) == 0
        torch.cuda.synchronize()
        return dt, Bm, Cm
    for far, near in zip(run(dist), run(dist[:, -few:].contiguous())):
        assert torch.equal(far[..., -few:], near)
        assert torch.equal(far[..., :5], far[..., K // 2:K // 2 + 5]) and (far[..., 0] != 3.0).all()


@pytest.mark.parametrize("form,K", [("bias", 26_900_001), ("bias weights raw", 53_700_002), ("tok", 53_700_002), ("tok weights raw", 26_900_001),
                                    ("tok weights", 53_700_001), ("joined", 53_700_002)])
def test_forms_beyond_32_bit_offsets(form, K):
    """The other forms of the kernels with 64-bit places -- fp32 and bf16, gathered biases and the producers' own, with a reversed pair, weights with and
    without raw dt, and the one with the convolutions in its launch -- against the last queries in a call of their own: the same bits."""
    import ctypes as C
    from dest3d_amd import _lib as L
    lib, H, G, few, di = L.load(), 10, 1, 777, 34
    dtype = torch.float32 if K < 50_000_000 else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    R0, Cc = H + 2 * G, di + 2 * G
    W, add, bias = 0.3 * rnd(R0, 16), rnd(H), rnd(1, H + 4 * G)
    row, tail = rnd(1, 2 * di + 2 * G + H).to(dtype), rnd(2, 1, 2 * G).to(dtype)
    cw, cb = rnd(2, Cc, 7), rnd(2, Cc)
    dist = torch.zeros(1, K, 16, dtype=dtype, device="cuda")
    dist[:, -few:] = rnd(1, few, 16).to(dtype)
    weights = torch.ones(1, K, device="cuda")
    weights[:, -few:] = torch.rand(1, few, generator=g, device="cuda")
    stream = L.current_stream_ptr(torch.device("cuda", 0))

    def run(d, w):
        k = d.shape[1]
        out = [torch.full((1, n, k), 3.0, dtype=dtype, device="cuda") for n in (H, G, G, G, G) + ((H,) if "raw" in form else ())]
        a = L.PGenArgs(tokens=1, K=k, M=16, H=H, G=G, dtype=L.dtype_code(dtype), has_back=1, dist=d.data_ptr(), W=W.data_ptr(), stream=stream)
        a.dt, a.Bm, a.Cm, a.Bm_back, a.Cm_back = (t.data_ptr() for t in out[:5])
        if "raw" in form:
            a.dt_raw = out[5].data_ptr()
        if "weights" in form or form == "joined":
            a.weights = w.data_ptr()
        if "bias" in form:
            a.bias = bias.data_ptr()
        else:
            a.tok, a.tok_stride, a.tok_add = row[:, di + Cc:].data_ptr(), row.shape[1], add.data_ptr()
            if form != "joined":
                a.tail = tail.data_ptr()
        if form == "joined":
            y = torch.full((2, 1, 1, di), 3.0, dtype=dtype, device="cuda")
            c = L.DwConvArgs(batch=1, seqlen=1, channels=Cc, nsets=2, taps=7, dtype=L.ISSM_BF16, u=row[:, di:].data_ptr(), u_batch_stride=row.shape[1],
                             u_token_stride=row.shape[1], w=cw.data_ptr(), bias=cb.data_ptr(), y=y.data_ptr(), stream=stream, split=di, chain=1)
            L.check(lib.issm_conv_param_gen_fwd(C.byref(c), C.byref(a)), "joined")
            out.append(y)
        else:
            # (raw dt is the training form's: without it, and with weights, only the form that no backward follows takes the call)
            L.check((lib.issm_param_gen_fwd if "raw" in form or "weights" not in form else lib.issm_param_gen_fwd_only)(C.byref(a)), form)
        torch.cuda.synchronize()
        return out
    far, near = run(dist, weights), run(dist[:, -few:].contiguous(), weights[:, -few:].contiguous())
    for f, n in zip(far, near):
        assert torch.equal(f[..., -n.shape[-1]:], n)
        if n.shape[-1] == few:
            assert torch.equal(f[..., :5], f[..., K // 2:K // 2 + 5]) and (f[..., 0] != 3.0).all()


@pytest.mark.parametrize("K", [(1 << 24) - 64, 1 << 24])
def test_backward_at_the_last_offsets_of_its_pieces(K):
    """Both sides of the number of queries up to which a token's ddist lies behind a buffer, against the queries that have a gradient in a call of
    their own: fp32 sums of the same values, in other blocks."""
    import ctypes as C
    from dest3d_amd import _lib as L
    lib, H, G, few, dtype = L.load(), 1, 1, 128, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(1)
    W = torch.randn(H + 2 * G, 16, generator=g, device="cuda")
    full = [torch.zeros(1, *s, dtype=dtype, device="cuda") for s in ((K, 16), (H, K), (G, K), (G, K))]
    full[0][:, -few:] = torch.randn(1, few, 16, generator=g, device="cuda").to(dtype)
    for t in full[1:]:
        t[..., -few:] = torch.randn(*t.shape[:2], few, generator=g, device="cuda").to(dtype)

    def run(d, *grads):
        dd, dbias, dW = torch.full_like(d, 3.0), torch.empty(1, H + 2 * G, device="cuda"), torch.empty(H + 2 * G, 16, device="cuda")
        scratch = torch.empty(lib.issm_param_gen_bwd_blocks(1), H + 2 * G, 16, device="cuda")
        a = L.PGenArgs(tokens=1, K=d.shape[1], M=16, H=H, G=G, dtype=L.ISSM_BF16, has_back=0, dist=d.data_ptr(), W=W.data_ptr(),
                       dw_partial=scratch.data_ptr(), dW=dW.data_ptr(), dbias=dbias.data_ptr(), ddist=dd.data_ptr(),
                       stream=L.current_stream_ptr(d.device))
        a.ddt, a.dBm, a.dCm = (t.data_ptr() for t in grads)
        assert lib.issm_param_gen_bwd(C.byref(a)) == 0
        torch.cuda.synchronize()
        return dd, dbias, dW
    want = run(full[0][:, -few:].contiguous(), *(t[..., -few:].contiguous() for t in full[1:]))
    dd, dbias, dW = run(*full)
    assert _rel(dd[:, -few:], want[0]) <= 2.0 ** -8 and (dd[:, :-few] == 0).all()
    assert _rel(dbias, want[1]) <= 1e-5 and _rel(dW, want[2]) <= 1e-5


@pytest.mark.parametrize("operands,ddist", [(1, 0), (2, 2), (4, 8), (0, 1), (3, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_backward_of_operands_at_any_element(dtype, operands, ddist):
    """Gradients, dt and dist that begin `operands` elements behind an aligned address, ddist `ddist` elements: as from aligned ones.  (A ddist at
    an odd bf16 element takes the form with a bound on k: the same rows' sums in blocks of 16, another order of the sums over k.)"""
    import ctypes as C
    from dest3d_amd import _lib as L
    lib = L.load()
    tokens, K, H, G = 21, 128, 8, 1
    R0, R = H + 2 * G, H + 4 * G
    gen = torch.Generator().manual_seed(3)
    W, w = torch.randn(R0, 16, generator=gen).cuda(), torch.rand(tokens, K, generator=gen).cuda()
    tensors = [torch.randn(tokens, *s, generator=gen).to(dtype) for s in ((K, 16), (H, K), (G, K), (G, K), (G, K), (G, K), (H, K))]

    def run(shift, dshift):
        behind = lambda t, n: torch.cat([t.new_zeros(n), t.flatten()]).cuda()
        kept = [behind(t, shift) for t in tensors]
        dd = torch.full((dshift + tokens * K * 16 + 1,), 3.0, dtype=dtype, device="cuda")
        f32 = lambda *s: torch.empty(*s, device="cuda")
        sums = f32(tokens, K), f32(tokens, R), f32(R), f32(R0, 16)
        scratch = f32(lib.issm_param_gen_bwd_blocks(tokens), R0, 16)
        a = L.PGenArgs()
        a.tokens, a.K, a.M, a.H, a.G, a.dtype, a.has_back = tokens, K, 16, H, G, L.dtype_code(dtype), 1
        a.W, a.weights, a.dw_partial = W.data_ptr(), w.data_ptr(), scratch.data_ptr()
        a.dist, a.ddt, a.dBm, a.dCm, a.dBm_back, a.dCm_back, a.dt_raw = (t[shift:].data_ptr() for t in kept)
        a.ddist = dd[dshift:].data_ptr()
        a.dweights, a.dbias, a.dbias_sum, a.dW = (t.data_ptr() for t in sums)
        a.stream = L.current_stream_ptr(dd.device)
        assert lib.issm_param_gen_bwd(C.byref(a)) == 0
        torch.cuda.synchronize()
        assert (dd[:dshift] == 3.0).all() and dd[-1] == 3.0
        return dd[dshift:-1], *sums
    same = dtype == torch.float32 or ddist % 2 == 0
    for got, want in zip(run(operands, ddist), run(0, 0)):
        if same:
            assert torch.equal(got, want)
        else:   # fp32 sums in another order; ddist and bf16 roundings of it
            assert _rel(got, want) <= (2.0 ** -8 if got.dtype == torch.bfloat16 else 1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_backward_without_queries(dtype):
    """No query: sums of nothing, and nothing read or written where a query would be."""
    import ctypes as C
    from dest3d_amd import _lib as L
    lib = L.load()
    tokens, H, G = 9, 4, 1
    R0, R = H + 2 * G, H + 4 * G
    W, buf = torch.randn(R0, 16).cuda(), torch.full((64,), 3.0, dtype=dtype, device="cuda")
    out = [torch.full(s, 3.0, device="cuda") for s in ((tokens, R), (R,), (R0, 16), (lib.issm_param_gen_bwd_blocks(tokens), R0, 16))]
    a = L.PGenArgs()
    a.tokens, a.K, a.M, a.H, a.G, a.dtype, a.has_back = tokens, 0, 16, H, G, L.dtype_code(dtype), 1
    a.W = W.data_ptr()
    a.dist = a.ddt = a.dBm = a.dCm = a.dBm_back = a.dCm_back = a.ddist = buf.data_ptr()
    a.dbias, a.dbias_sum, a.dW, a.dw_partial = (t.data_ptr() for t in out)
    a.stream = L.current_stream_ptr(buf.device)
    assert lib.issm_param_gen_bwd(C.byref(a)) == 0
    torch.cuda.synchronize()
    assert all((t == 0.0).all() for t in out[:3]) and (buf == 3.0).all()
