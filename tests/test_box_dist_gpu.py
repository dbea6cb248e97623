"""Box distance encoding + locality weight (libissm_hip.so) against the fp64 numpy oracle (itself pinned by torch's
grid_sample, tests/test_oracle_boxdist.py).  fp32: rel. error <= 1e-4 forward and table gradient (the sampling
position goes through a hardware log2; the table gradient is summed with LDS atomics); bf16 output: <= 1e-2."""
import numpy as np
import pytest
import torch

from oracle import boxdist_ref as R

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a = np.asarray(a, np.float64)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


def _inputs(B, nP, nQ, seed, angles):
    rng = np.random.default_rng(seed)
    key = rng.uniform(-4, 4, size=(B, nP, 3)).astype(np.float32)
    qxyz = rng.uniform(-4, 4, size=(B, nQ, 3)).astype(np.float32)
    qsize = rng.uniform(0.1, 2.5, size=(B, nQ, 3)).astype(np.float32)
    ang = (rng.uniform(-3, 3, size=(B, nQ)) if angles else np.zeros((B, nQ))).astype(np.float32)
    return key, qxyz, qsize, ang


# the table gradient scatters with LDS atomics below 65536 (point, box) pairs and sorts by window above: both sizes
CASES = [(2, 37, 256, False, (10, 10, 10)), (1, 5, 300, True, (10, 10, 10)), (2, 64, 19, True, (4, 6, 7)),
         (1, 1, 1, False, (10, 10, 10)), (2, 160, 256, False, (10, 10, 10)), (1, 230, 300, True, (10, 10, 10)),
         (1, 1100, 64, True, (4, 6, 7)), (1, 1500, 43, True, (10, 10, 10)),   # two point segments, ragged box group
         (1, 4200, 16, True, (5, 4, 3)), (3, 1400, 16, False, (1, 30, 30))]     # four workgroups a CU in the gradient, 3072 bins


def test_box_dist_forward_does_not_depend_on_the_segments():
    """Enough boxes for the longest segments, the last pair of which has a short one and an empty one, against the same
    points in calls of few points (shortest segments): the same bits."""
    from dest3d_amd.box_dist import box_dist, box_parametrization_to_corners
    key, qxyz, qsize, ang = (torch.from_numpy(x).cuda() for x in _inputs(1, 1030, 2041, 5, True))
    table = torch.randn(16, 10, 10, 10, generator=torch.Generator().manual_seed(1)).cuda()
    corners = box_parametrization_to_corners(qxyz, qsize, ang)
    whole = box_dist(table, key, corners)
    for lo, hi in ((0, 65), (448, 577), (1000, 1030)):
        part = box_dist(table, key[:, lo:hi].contiguous(), corners[:, 1980:].contiguous())
        assert torch.equal(part, whole[:, lo:hi, 1980:])


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_P%d_Q%d_ang%d_%dx%dx%d" % (*c[:3], int(c[3]), *c[4]))
def test_box_dist_forward_and_table_gradient(case):
    from dest3d_amd.box_dist import box_dist, box_parametrization_to_corners
    B, nP, nQ, angles, dims = case
    key, qxyz, qsize, ang = _inputs(B, nP, nQ, 11 + nP + nQ, angles)
    rng = np.random.default_rng(3)
    table = rng.standard_normal((16, *dims)).astype(np.float32)
    t = torch.from_numpy(table).cuda().requires_grad_()
    tk, tq, ts, ta = (torch.from_numpy(x).cuda() for x in (key, qxyz, qsize, ang))
    corners = box_parametrization_to_corners(tq, ts, ta)
    assert np.abs(corners.cpu().numpy() - R.box_corners(qxyz, qsize, ang)).max() < 1e-5
    dist = box_dist(t, tk, corners, ta if angles else None)
    ref = R.box_dist(key, qxyz, qsize, ang, table)
    assert dist.shape == (B, nP, nQ, 16) and dist.is_contiguous()
    e_fwd = _rel(dist.detach().cpu().numpy(), ref)
    assert e_fwd <= 2e-5
    g = rng.standard_normal(ref.shape).astype(np.float32)
    dist.backward(torch.from_numpy(g).cuda())
    gref = R.box_dist_table_grad(key, qxyz, qsize, ang, table.shape, g)
    e_bwd = _rel(t.grad.cpu().numpy(), gref)
    print(f"    pairs {B * nP * nQ}: dist err {e_fwd:.2e}, table gradient err {e_bwd:.2e}", flush=True)
    assert e_bwd <= 2e-5
    # bf16 output
    dist_bf = box_dist(t.detach(), tk, corners, ta if angles else None, out_dtype=torch.bfloat16)
    assert dist_bf.dtype == torch.bfloat16
    assert _rel(dist_bf.float().cpu().numpy(), ref) <= 1e-2


@pytest.mark.parametrize("nP,nQ,dims,spread", [(65, 9, (10, 10, 10), 4.0), (1100, 64, (4, 6, 7), 4.0), (3, 300, (5, 4, 3), 0.2), (200, 16, (1, 30, 30), 2.0),
                                               (130, 8, (10, 10, 10), 200.0), (1, 1, (2, 2, 2), 0.0)])
def test_boxes_along_the_axes_without_a_gradient(nP, nQ, dims, spread):
    """Calls that no backward follows: boxes along the axes are summed axis by axis.  Positions of an axis in the same cell, in
    neighbouring ones, apart and outside the table, a quarter of the boxes turned, against the fp64 oracle (bound as above)."""
    from dest3d_amd.box_dist import BoxDistFn, box_parametrization_to_corners
    run = lambda t, k, c, only: BoxDistFn.apply(t, k, c, None, None, None, 0.0, 512.0, 4.0, torch.float32, True, False, only)[0]
    key, qxyz, qsize, ang = _inputs(2, nP, nQ, 5 + nP + nQ, True)
    key, qxyz = (key * np.float32(spread / 4) for key in (key, qxyz))
    qsize[:, ::3] *= np.float32(1e-3)
    heading = ang * (np.arange(nQ) % 4 == 1)
    table = np.random.default_rng(4).standard_normal((16, *dims)).astype(np.float32)
    t, tk, tq, ts, th = (torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda() for x in (table, key, qxyz, qsize, heading))
    corners = box_parametrization_to_corners(tq, ts, th)
    whole, dist = run(t, tk, corners, False), run(t, tk, corners, True)
    # the oracle takes one angle for the corners and the rotation: the boxes that are not turned
    plain = np.arange(nQ) % 4 != 1
    ref = R.box_dist(key, qxyz, qsize, np.zeros_like(ang), table)
    assert _rel(dist.cpu().numpy()[:, :, plain], ref[:, :, plain]) <= 2e-5
    assert torch.equal(dist[:, :, ~plain], whole[:, :, ~plain])
    assert (dist - whole).norm() <= 2e-5 * whole.norm()
    # values that are not finite: of the table, of a point, of a box
    odd = t.clone()
    odd[3, 0, 0, 0], odd[5, -1, -1, -1] = float("nan"), float("inf")
    kodd, codd = tk.clone(), corners.clone()
    kodd[0, nP // 2, 1], codd[1, nQ // 2, 2, 0] = float("inf"), float("nan")
    for tt, kk, cc in ((odd, tk, corners), (t, kodd, codd)):
        got, want = run(tt, kk, cc, True), run(tt, kk, cc, False)
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        ok = want.isfinite()
        assert (got[ok] - want[ok]).norm() <= 2e-5 * want[ok].norm() + 1e-30


@pytest.mark.parametrize("nP,nQ,dims,spread", [(33, 65, (10, 10, 10), 4.0), (1100, 64, (4, 6, 7), 4.0), (700, 100, (5, 4, 3), 0.2),
                                               (520, 130, (10, 10, 10), 200.0), (4200, 16, (1, 30, 30), 2.0)])
def test_boxes_along_the_axes_in_training(nP, nQ, dims, spread):
    """Encoding and table gradient of boxes along the axes, which find windows and weights axis by axis, against the same boxes with one corner moved
    by a unit in the last place, which take the form by corners: 3e-7 of a position of up to 4, which the logarithm stretches by at most 300
    nodes next to a point (1e-4 of a node) and by a few elsewhere; 2e-5 of the norm, as against the oracle.  Small and large calls (the gradient in
    LDS and by sorted windows); a point and a box that are not finite come out in the same places."""
    from dest3d_amd.box_dist import box_dist, box_parametrization_to_corners
    key, qxyz, qsize, ang = _inputs(2, nP, nQ, 3 + nP + nQ, False)
    key, qxyz = (v * np.float32(spread / 4) for v in (key, qxyz))
    qsize[:, ::3] *= np.float32(1e-3)
    tk, tq, ts, ta = (torch.from_numpy(v).cuda() for v in (key, qxyz, qsize, ang))
    g = torch.Generator().manual_seed(2)
    table, dout = torch.randn(16, *dims, generator=g).cuda(), torch.randn(2, nP, nQ, 16, generator=g).cuda()
    corners = box_parametrization_to_corners(tq, ts, ta)
    moved = corners.clone()
    moved[:, :, 5, 0] = torch.nextafter(moved[:, :, 5, 0], torch.full_like(moved[:, :, 5, 0], 1e9))

    def run(k, c):
        t = table.clone().requires_grad_()
        dist = box_dist(t, k, c)
        dist.backward(dout)
        return dist.detach(), t.grad

    for got, want in zip(run(tk, corners), run(tk, moved)):
        assert (got - want).norm() <= 2e-5 * want.norm()
    tk[0, nP // 2, 1], corners[1, nQ // 2, 2, 0], moved[1, nQ // 2, 2, 0] = float("inf"), float("nan"), float("nan")
    got, want = run(tk, corners)[0], run(tk, moved)[0]
    assert torch.equal(got.isfinite(), want.isfinite())
    ok = want.isfinite()
    assert (got[ok] - want[ok]).norm() <= 2e-5 * want[ok].norm()


def test_local_weight_and_fused_module_call():
    from dest3d_amd.box_dist import BoxDistFun, local_weight
    B, nP, nQ = 2, 50, 256
    key, qxyz, qsize, ang = _inputs(B, nP, nQ, 5, False)
    qpos = np.concatenate([qxyz, qsize], -1)
    tk, tpos = torch.from_numpy(key).cuda(), torch.from_numpy(qpos).cuda()
    w = local_weight(tk, tpos, 15.0)
    wref = R.local_weight(key, qpos, 15.0)
    assert w.shape == (B, nP, nQ) and w.dtype == torch.float32
    assert np.abs(w.cpu().numpy() - wref).max() <= 1e-4      # values in [0, 1]; exp of up to -15 * 10
    torch.manual_seed(0)
    m = BoxDistFun(out_dim=16).cuda()
    assert set(m.state_dict()) == {"relative_coords_table", "cpb_mlps.0.weight", "cpb_mlps.0.bias", "cpb_mlps.2.weight"}
    dist, w2 = m(tk, tpos[..., :3], tpos[..., 3:], torch.zeros(B, nQ, device="cuda"), weight_query_pos=tpos)
    table = m.rpe_table().detach().double().cpu().numpy()
    ref = R.box_dist(key, qxyz, qsize, ang, table)
    assert _rel(dist.detach().cpu().numpy(), ref) <= 1e-4
    # the fused call derives centre and radius from the boxes inside the kernel: equal up to the rounding of the radius
    assert torch.allclose(w2, w, rtol=2e-4, atol=1e-7)
    dist.square().sum().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in m.parameters())
    # gradient of the MLP through the table: against autograd of the same MLP fed the oracle's table gradient
    gtab = R.box_dist_table_grad(key, qxyz, qsize, ang, table.shape, 2 * ref)
    m2 = BoxDistFun(out_dim=16).double()
    m2.load_state_dict({k: v.double().cpu() for k, v in m.state_dict().items()})
    (m2.rpe_table() * torch.from_numpy(gtab)).sum().backward()
    for (n, p), p2 in zip(m.named_parameters(), m2.parameters()):
        assert _rel(p.grad.cpu().numpy(), p2.grad.numpy()) <= 2e-3, n


def test_table_gradient_is_bit_reproducible():
    """The gradient is accumulated in 64-bit fixed point: the order of the adds cannot change it."""
    from dest3d_amd.box_dist import box_dist, box_parametrization_to_corners
    key, qxyz, qsize, ang = _inputs(2, 200, 256, 21, False)
    tk, tq, ts, ta = (torch.from_numpy(x).cuda() for x in (key, qxyz, qsize, ang))
    corners = box_parametrization_to_corners(tq, ts, ta)
    g = torch.randn(2, 200, 256, 16, generator=torch.Generator().manual_seed(1)).cuda()
    grads = []
    for _ in range(3):
        t = torch.randn(16, 10, 10, 10, generator=torch.Generator().manual_seed(2)).cuda().requires_grad_()
        box_dist(t, tk, corners).backward(g)
        grads.append(t.grad.clone())
    assert torch.equal(grads[0], grads[1]) and torch.equal(grads[0], grads[2])
    # a zero upstream gradient gives an exactly zero table gradient
    t = torch.randn(16, 10, 10, 10, generator=torch.Generator().manual_seed(2)).cuda().requires_grad_()
    box_dist(t, tk, corners).backward(torch.zeros_like(g))
    assert t.grad.abs().max().item() == 0.0
    # the fixed point is scaled to max|ddist|: upstream gradients of any magnitude give the same relative result,
    # vanishing ones a finite (zero) one; both sides of the 65536-pair switch between the two accumulation paths
    for npts in (200, 20):
        gs = g[:, :npts].contiguous()
        ref = None
        for scale in (1.0, 1e30, 1e-25, 1e-37):
            t = torch.randn(16, 10, 10, 10, generator=torch.Generator().manual_seed(2)).cuda().requires_grad_()
            box_dist(t, tk[:, :npts].contiguous(), corners).backward(gs * scale)
            assert torch.isfinite(t.grad).all()
            if ref is None:
                ref = t.grad.double()
            elif scale > 1e-30:
                assert _rel((t.grad.double() / scale).cpu().numpy(), ref.cpu().numpy()) <= 1e-6, (npts, scale)
            else:
                assert t.grad.abs().max().item() <= 1e-30


@pytest.mark.parametrize("quant,rpe_dim", [("bilinear_4_10", 128), ("bilinear_4_3", 7), ("bilinear_2_1", 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_table_without_a_gradient(quant, rpe_dim, dtype):
    """One kernel for the table's MLP, at node and hidden counts that fill no workgroup, against fp64 with the roundings of the
    modules: coordinates, hidden values, results.  A hidden value may round the other way (2^-8 of it, through |W2|); sums of
    hidden products in fp32.  What the kernel is not for goes through the modules: wide MLPs, hooks, gradients."""
    from dest3d_amd.box_dist import BoxDistFun
    torch.manual_seed(rpe_dim)
    m = BoxDistFun(out_dim=16, rpe_quant=quant, rpe_dim=rpe_dim).cuda().to(dtype)
    assert m._plain_table() is None                      # parameters that want a gradient
    with torch.no_grad():
        got = m._plain_table()
        hook = m.cpb_mlps[1].register_forward_hook(lambda *_: None)
        assert m._plain_table() is None
        hook.remove()
        assert BoxDistFun(out_dim=16, rpe_dim=257).cuda()._plain_table() is None
        want = m.rpe_table()
    lin1, _, lin2 = m.cpb_mlps
    h = (m.relative_coords_table.to(dtype).double() @ lin1.weight.double().t() + lin1.bias.double()).to(dtype).double().relu()
    ref, mag = (f(h) @ f(lin2.weight.double()).t() for f in (lambda t: t, torch.abs))
    ref, mag = (t[0].permute(3, 0, 1, 2).cpu() for t in (ref, mag))
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20
    assert got.shape == want.shape and got.dtype == torch.float32 and got.is_contiguous()
    assert ((got.double().cpu() - ref).abs() <= u * (mag + ref.abs())).all()


@pytest.mark.parametrize("quant,rpe_dim", [("bilinear_4_10", 128), ("bilinear_4_3", 7), ("bilinear_2_1", 256)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("again", [False, True])
def test_gradients_of_the_tables_mlp(quant, rpe_dim, dtype, again):
    """One kernel for the MLP's backward, against fp64 from hidden values rounded as the modules round them (each may round the other way,
    2^-8 of it); the forward is the modules'.  A backward that is to be differentiated again goes through operations."""
    from dest3d_amd.box_dist import BoxDistFun, BoxTableFn
    torch.manual_seed(rpe_dim)
    m = BoxDistFun(out_dim=16, rpe_quant=quant, rpe_dim=rpe_dim).cuda().to(dtype)
    mlp = m._plain_mlp()
    table = BoxTableFn.apply(m, *mlp)
    assert table.dtype == torch.float32 and torch.equal(table, m.rpe_table().float())
    g = torch.randn(table.shape, device="cuda").to(dtype).float()
    grads = torch.autograd.grad(table, mlp[:3], g, create_graph=again)
    w1, b1, w2, x = (t.detach().double() for t in mlp)
    x = m.relative_coords_table.to(dtype).double().reshape(-1, 3)
    h = (x @ w1.t() + b1).to(dtype).double().relu()
    gd = g.double().reshape(16, -1)
    dh = (gd.t() @ w2) * (h > 0)
    near = (gd.t() @ w2).abs() * ((x @ w1.t() + b1).abs() <= 2.0 ** -18 * ((x.abs() @ w1.abs().t()) + b1.abs()))   # either side of zero
    u = (2.0 ** -5 if again else 2.0 ** -8) if dtype == torch.bfloat16 else 2.0 ** -18
    for got, want, mag, edge in ((grads[0], dh.t() @ x, dh.abs().t() @ x.abs(), near.t() @ x.abs()), (grads[1], dh.sum(0), dh.abs().sum(0), near.sum(0)),
                                 (grads[2], gd @ h, gd.abs() @ h, 0.0)):
        assert got.dtype == dtype and ((got.double() - want).abs() <= u * (mag + want.abs()) + edge + 1e-12).all()
    if again:
        torch.autograd.grad(grads[2].float().square().sum(), mlp[0])
    hook = m.cpb_mlps[1].register_forward_hook(lambda *_: None)
    assert m._plain_mlp() is None
    hook.remove()


@pytest.mark.parametrize("again", [False, True])
def test_tables_mlp_after_its_first_layer_has_changed(again):
    """The encoding's first weights and its bias changed in place between forward and backward: the gradients of the values that the forward used,
    as from the modules, which do not keep them; the second weights are kept, and say so."""
    from dest3d_amd.box_dist import BoxDistFun, BoxTableFn
    torch.manual_seed(5)
    m = BoxDistFun(out_dim=16).cuda()
    mlp = m._plain_mlp()
    g = torch.randn(16, 10, 10, 10, device="cuda")
    run = lambda t: torch.autograd.grad(t, mlp[:3], g, create_graph=again)
    of_modules = lambda: m.rpe_table().float().contiguous()
    want, kept = run(of_modules()), run(BoxTableFn.apply(m, *mlp))
    for make in (of_modules, lambda: BoxTableFn.apply(m, *mlp)):
        table = make()
        before = [p.detach().clone() for p in mlp[:3]]
        with torch.no_grad():
            mlp[0].neg_()
            mlp[1].add_(1.0)
        for a, b, c in zip(run(table), want, kept):
            assert (a - b).norm() <= 1e-5 * b.norm() and (torch.equal(a, c) or make is of_modules)
        with torch.no_grad():
            mlp[0].copy_(before[0])
            mlp[1].copy_(before[1])
    if again:   # differentiated twice: d / dw1 of a function of dw2
        a, = torch.autograd.grad(want[2].square().sum(), mlp[0])
        b, = torch.autograd.grad(kept[2].square().sum(), mlp[0])
        assert (a - b).norm() <= 1e-5 * a.norm()
    table = BoxTableFn.apply(m, *mlp)
    with torch.no_grad():
        mlp[2].add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        run(table)



def test_modes_see_the_tables_mlp():
    """Who counts or records operations or functions sees the two products of the table's MLP; a default device does not ask."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._device import DeviceContext
    from torch.utils._python_dispatch import TorchDispatchMode
    from dest3d_amd.box_dist import BoxDistFun
    m = BoxDistFun(out_dim=16).cuda()
    seen = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func is torch.nn.functional.linear)
            return func(*args, **(kwargs or {}))

    class Operations(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func in (torch.ops.aten.mm.default, torch.ops.aten.addmm.default))
            return func(*args, **(kwargs or {}))

    args = (torch.rand(1, 5, 3).cuda(), torch.rand(1, 3, 3).cuda(), torch.rand(1, 3, 3).cuda(), torch.zeros(1, 3).cuda())
    with torch.no_grad():
        want = m(*args)
        with DeviceContext("cuda"):
            assert m._plain_table() is not None
        for mode in (Functions, Operations):
            seen.clear()
            with mode():
                got = m(*args)
            assert sum(seen) == 2
            assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)
        compiled = torch.compile(m.rpe_table, backend="eager")()
        assert torch.allclose(compiled, m._plain_table(), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("shape", [(4, 4, 4, 3), (2, 4, 4, 4, 3), (1, 4, 4, 4, 6), (1, 2, 4, 4, 4, 3)])
def test_table_of_a_replaced_lattice(shape):
    """Without a gradient a lattice of another form does what it does with one: the modules take it or refuse it."""
    from dest3d_amd.box_dist import BoxDistFun
    m = BoxDistFun(out_dim=16).cuda()
    m.relative_coords_table = torch.randn(shape, device="cuda")
    args = (torch.rand(1, 5, 3).cuda(), torch.rand(1, 3, 3).cuda(), torch.rand(1, 3, 3).cuda(), torch.zeros(1, 3).cuda())

    def call():
        try:
            return m(*args)
        except RuntimeError:
            return None

    want = call()
    assert (want is not None) == (shape == (2, 4, 4, 4, 3))
    with torch.no_grad():
        assert m._plain_table() is None
        got = call()
    assert want is None and got is None or torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_encoding_in_a_checkpointed_segment(dtype):
    """Reentrant checkpointing runs a segment without gradients first: the encoding's sums and its table are training's in that run too, so
    that outputs and gradients are those of the segment that is not checkpointed."""
    from torch.utils.checkpoint import checkpoint
    from dest3d_amd.box_dist import BoxDistFun
    torch.manual_seed(2)
    m = BoxDistFun(out_dim=16).cuda().to(dtype)
    key, qxyz, qsize, ang = (torch.from_numpy(x).cuda() for x in _inputs(2, 300, 64, 8, False))
    boxes, scale, dout = torch.cat([qxyz, qsize], dim=-1), torch.rand(2, 300, 64, 16).cuda().to(dtype), torch.randn(2, 300, 64, 16).cuda().to(dtype)

    def segment(s):
        dist, weights = m(key, boxes[..., :3], boxes[..., 3:], ang, weight_query_pos=boxes)
        return dist * s, weights

    def step(run):
        s = scale.clone().requires_grad_()
        m.zero_grad(set_to_none=True)
        out, weights = run(s)
        out.backward(dout)
        return out, weights, s.grad, *(p.grad for p in m.parameters())

    want, got = step(segment), step(lambda s: checkpoint(segment, s, use_reentrant=True))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_operands_of_another_size_or_device_are_refused():
    """Refused before a kernel is given their address."""
    from dest3d_amd.box_dist import box_dist, box_parametrization_to_corners, local_weight
    from dest3d_amd.dwconv import dwconv_silu
    from dest3d_amd.param_gen import scan_params
    key, qxyz, qsize, ang = (torch.from_numpy(x).cuda() for x in _inputs(2, 9, 5, 1, True))
    table = torch.randn(16, 4, 4, 4).cuda()
    corners, query = box_parametrization_to_corners(qxyz, qsize, ang), torch.cat([qxyz, qsize], -1)
    box_dist(table, key, corners, ang)
    for args in ((table, key, corners[:1], ang), (table, key, corners, ang[:1]), (table, key[..., :2], corners, ang),
                 (table.cpu(), key, corners, ang), (table, key, corners.cpu(), ang), (table, key, corners, ang.cpu())):
        with pytest.raises((RuntimeError, ValueError)):
            box_dist(*args)
    for bad in (query[:1], query.cpu()):
        with pytest.raises((RuntimeError, ValueError)):
            local_weight(key, bad)
    u, w, b = torch.randn(1, 9, 4).cuda(), torch.randn(4, 1, 7).cuda(), torch.randn(4).cuda()
    dwconv_silu(u, [w], [b])
    for ww, bb in ((w.cpu(), b), (w, b.cpu()), (w, b[:3]), (w[:3], b)):
        with pytest.raises((RuntimeError, ValueError)):
            dwconv_silu(u, [ww], [bb])
    d, W, bias, wts = torch.randn(1, 9, 5, 16).cuda(), torch.randn(4, 16).cuda(), torch.randn(1, 9, 4).cuda(), torch.rand(1, 9, 5).cuda()
    scan_params(d, W, bias, 2, 1, weights=wts)
    for args in ((W.cpu(), bias, wts), (W, bias.cpu(), wts), (W, bias, wts.cpu())):
        with pytest.raises(RuntimeError):
            scan_params(d, *args[:2], 2, 1, weights=args[2])


def test_box_dist_rejects_unbuilt_shapes():
    import ctypes as C
    from dest3d_amd import _lib as L
    lib = L.load()
    a = L.BoxDistArgs()
    a.batch, a.seqlen, a.nquery, a.D, a.H, a.W = 1, 4, 4, 11, 10, 10
    assert lib.issm_box_dist_fwd(C.byref(a)) == -5
    a.D = 10
    assert lib.issm_box_dist_fwd(C.byref(a)) == -1
