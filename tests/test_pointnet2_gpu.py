"""Point-set operators (libissm_hip.so, issm_pn2_*) against the numpy oracle: indices exactly, values to fp32
rounding (the gradients are float-atomic sums: 1e-5 relative)."""
import numpy as np
import pytest
import torch

from oracle import pointnet2_ref as R

pytestmark = pytest.mark.gpu


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("shape", [(2, 700, 64), (1, 5000, 256), (3, 37, 37), (1, 1, 1)])
def test_furthest_point_sampling(shape):
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    B, N, npoint = shape
    rng = np.random.default_rng(N)
    xyz = rng.uniform(-4, 4, size=(B, N, 3)).astype(np.float32)
    if N > 10:
        xyz[0, 3] = 0.0            # padding point at the origin: never drawn
        xyz[0, 7] = xyz[0, 5]      # a duplicate
    idx = furthest_point_sample(_cuda(xyz), npoint)
    assert idx.dtype == torch.int32 and idx.shape == (B, npoint)
    assert (idx.cpu().numpy() == R.furthest_point_sampling(xyz, npoint)).all()


def test_furthest_point_sampling_beyond_the_register_path():
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    rng = np.random.default_rng(9)
    xyz = rng.uniform(-4, 4, size=(1, 50000, 3)).astype(np.float32)
    idx = furthest_point_sample(_cuda(xyz), 48).cpu().numpy()
    assert (idx == R.furthest_point_sampling(xyz, 48)).all()


@pytest.mark.parametrize("n", [63, 64, 65, 2048, 2049, 4096, 4097, 8193, 12289, 16385, 20481, 24576, 24577])
def test_furthest_point_sampling_at_the_edges_of_its_variants(n):
    """Group and slot remainders of every register variant, and the first size beyond them; sample 1 is clustered (a flat
    sheet, duplicates, one far point), sample 2 all padding but one point, sample 3 one point repeated."""
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    rng = np.random.default_rng(n)
    xyz = rng.uniform(-4, 4, size=(4, n, 3)).astype(np.float32)
    xyz[1, :, 2] = 1.0
    xyz[1, n // 2:] = xyz[1, :n - n // 2]
    xyz[1, 11] = (300.0, -20.0, 5.0)
    xyz[2] = 0.0
    xyz[2, n // 3] = 2.0
    xyz[3] = xyz[3, 5]
    npoint = min(n, 80)
    idx = furthest_point_sample(_cuda(xyz), npoint).cpu().numpy()
    assert (idx == R.furthest_point_sampling(xyz, npoint)).all()


@pytest.mark.parametrize("n,npoint", [(700, 300), (4096, 512)])
def test_furthest_point_sampling_on_a_voxelized_cloud(n, npoint):
    """Coordinates on a quarter-metre grid: most running distances tie, within groups, waves and the workgroup."""
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    xyz = (np.random.default_rng(n).integers(1, 17, size=(2, n, 3)) * 0.25).astype(np.float32)
    idx = furthest_point_sample(_cuda(xyz), npoint).cpu().numpy()
    assert (idx == R.furthest_point_sampling(xyz, npoint)).all()


@pytest.mark.parametrize("n", [65, 2048, 8193])
@pytest.mark.parametrize("every", [2, 3, 20, 1000])
def test_furthest_point_sampling_where_some_points_lie_far_from_most(n, every):
    """Points of either sorting grid, and on their limits: sample 1 has more than half of its points in one place."""
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 8, size=(2, n, 3)).astype(np.float32)
    xyz[:, every // 2::every] = rng.uniform(-900, 900, size=xyz[:, every // 2::every].shape)
    xyz[1, n // 3:] = xyz[1, n // 3]
    idx = furthest_point_sample(_cuda(xyz), min(n, 200)).cpu().numpy()
    assert (idx == R.furthest_point_sampling(xyz, min(n, 200))).all()


@pytest.mark.parametrize("n", [64, 700, 5000, 24576])
@pytest.mark.parametrize("kind", ["extent 1e6", "metres on a map", "infinite points", "first point no number"])
def test_furthest_point_sampling_where_running_distances_never_come_below_their_start(n, kind):
    """Squared distances of 1e10 and more leave every running distance at its start of 1e10: the smallest index is next, also
    of a group of points that no draw comes near."""
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    rng = np.random.default_rng(n)
    xyz = rng.uniform(-4, 4, size=(2, n, 3)).astype(np.float32)
    if kind == "extent 1e6":
        xyz *= np.float32(2e5)
    elif kind == "metres on a map":
        xyz = (xyz * 100 + np.array([5e5, 4.2e6, 100.0])).astype(np.float32)
        xyz[:, 0] = 0.0                     # a padding point first
    elif kind == "infinite points":
        xyz[0, n // 3:n // 3 + 9] = np.inf
        xyz[1, n // 2:, 0] = -np.inf
    else:
        xyz[0, 0] = np.nan
        xyz.view(np.uint32)[1, 0] = 0xffffffff
    npoint = min(n, 64)
    idx = furthest_point_sample(_cuda(xyz), npoint).cpu().numpy()
    with np.errstate(invalid="ignore"):
        assert (idx == R.furthest_point_sampling(xyz, npoint)).all()


@pytest.mark.parametrize("seed,npoint", [(3, 1024), (8, 1024), (54, 1024)])
def test_furthest_point_sampling_near_ties_go_the_way_of_plain_fp32_steps(seed, npoint):
    """Clouds in which two candidates' running minimum distances come within one unit in the last place of each other
    (draws 960, 885 and 874 of these seeds): a squared distance evaluated with a fused multiply-add, fma(dz, dz,
    fma(dy, dy, dx dx)), rounds the other way there and draws another point from then on.  The kernel evaluates
    (dx dx + dy dy) + dz dz with every operation rounded, like the oracle."""
    from dest3d_amd.pointnet2_utils import furthest_point_sample
    xyz = np.random.default_rng(seed).uniform(-2, 2, size=(1, 4096, 3)).astype(np.float32)
    idx = furthest_point_sample(_cuda(xyz), npoint).cpu().numpy()
    assert (idx == R.furthest_point_sampling(xyz, npoint)).all()


@pytest.mark.parametrize("shape", [(2, 3000, 128, 0.6, 16), (1, 100, 7, 0.3, 64), (2, 65, 5, 10.0, 3), (1, 40, 4, 1e-3, 8)])
def test_ball_query(shape):
    from dest3d_amd.pointnet2_utils import ball_query
    B, N, M, radius, nsample = shape
    rng = np.random.default_rng(N + M)
    xyz = rng.uniform(-2, 2, size=(B, N, 3)).astype(np.float32)
    q = xyz[:, rng.integers(0, N, size=M)] + rng.normal(0, 0.05, size=(B, M, 3)).astype(np.float32)
    q[0, 0] = 100.0
    idx = ball_query(radius, nsample, _cuda(xyz), _cuda(q.astype(np.float32)))
    assert idx.dtype == torch.int32
    assert (idx.cpu().numpy() == R.ball_query(radius, nsample, xyz, q.astype(np.float32))).all()


@pytest.mark.parametrize("b,n,m", [(1, 1025, 17), (2, 5121, 40), (1, 9300, 64), (5, 1500, 3300)])
@pytest.mark.parametrize("kind", ["spread", "in order along an axis", "heaps", "no numbers"])
def test_ball_query_looks_in_order_and_masks(b, n, m, kind):
    """Behind the first 1024 points a centre either goes on looking in order or takes the masks, leaves them when it has enough,
    or overflows its list in the middle of a chunk of 4096 points; one and four centres a wave, more slots than a list holds."""
    from dest3d_amd.pointnet2_utils import ball_query
    rng = np.random.default_rng(n + m)
    xyz = rng.uniform(0, 8, size=(b, n, 3)).astype(np.float32)
    if kind == "in order along an axis":
        xyz[..., 1].sort(axis=1)
    elif kind == "heaps":                  # 300 points in one place, behind the first chunk where there is one
        at = max(n - 300, 1024)
        xyz[:, at:at + 300] = xyz[:, 5:6] + rng.normal(0, 0.01, size=xyz[:, at:at + 300].shape).astype(np.float32)
    q = xyz[:, rng.integers(0, n, size=m)] + rng.normal(0, 0.05, size=(b, m, 3)).astype(np.float32)
    q[:, 0] = xyz[:, 5]
    if kind == "no numbers":
        xyz[:, n // 2, 0] = np.nan
        xyz[:, n // 3] = np.inf
        q[0, 1, 2] = np.nan
        q[-1, 2, 1] = -np.inf
    for radius, nsample in ((0.3, 16), (0.8, 64), (1.1, 200), (-0.5, 3), (0.0, 4), (30.0, 5)):
        idx = ball_query(radius, nsample, _cuda(xyz), _cuda(q)).cpu().numpy()
        with np.errstate(invalid="ignore"):
            assert (idx == R.ball_query(radius, nsample, xyz, q)).all(), (radius, nsample)


def test_three_nn_and_interpolate():
    from dest3d_amd.pointnet2_utils import three_interpolate, three_nn
    rng = np.random.default_rng(5)
    B, n, m, c = 2, 777, 300, 19
    u = rng.uniform(-2, 2, size=(B, n, 3)).astype(np.float32)
    k = rng.uniform(-2, 2, size=(B, m, 3)).astype(np.float32)
    dist, idx = three_nn(_cuda(u), _cuda(k))
    d2_ref, idx_ref = R.three_nn(u, k)
    assert (idx.cpu().numpy() == idx_ref).all()
    assert np.allclose(dist.cpu().numpy(), np.sqrt(d2_ref), rtol=1e-6, atol=0)
    feats = rng.standard_normal((B, c, m)).astype(np.float32)
    w = (1.0 / (np.sqrt(d2_ref) + 1e-8))
    w = (w / w.sum(-1, keepdims=True)).astype(np.float32)
    f = _cuda(feats).requires_grad_()
    y = three_interpolate(f, idx, _cuda(w))
    ref = R.three_interpolate(feats, idx_ref, w)
    assert np.abs(y.detach().cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    gy = rng.standard_normal(ref.shape).astype(np.float32)
    y.backward(_cuda(gy))
    gref = R.three_interpolate_grad(gy, idx_ref, w, m)
    assert np.abs(f.grad.cpu().numpy() - gref).max() <= 1e-5 * np.abs(gref).max()
    # fewer than three known points
    dist, idx = three_nn(_cuda(u[:, :5]), _cuda(k[:, :2]))
    assert torch.isinf(dist[..., 2]).all() and (idx[..., 2] == 0).all()


def test_group_and_gather_with_gradients():
    from dest3d_amd.pointnet2_utils import gather_operation, grouping_operation
    rng = np.random.default_rng(6)
    B, C, N, M, S = 2, 13, 500, 60, 16
    pts = rng.standard_normal((B, C, N)).astype(np.float32)
    idx = rng.integers(0, N, size=(B, M, S)).astype(np.int32)
    idx[0, 0, :] = 7                                  # many duplicates: the gradient accumulates
    f = _cuda(pts).requires_grad_()
    g = grouping_operation(f, _cuda(idx))
    assert (g.detach().cpu().numpy() == R.group_points(pts, idx)).all()
    gy = rng.standard_normal(g.shape).astype(np.float32)
    g.backward(_cuda(gy))
    gref = R.group_points_grad(gy, idx, N)
    assert np.abs(f.grad.cpu().numpy() - gref).max() <= 1e-5 * np.abs(gref).max()
    f2 = _cuda(pts).requires_grad_()
    y = gather_operation(f2, _cuda(idx[:, :, 0].copy()))
    assert (y.detach().cpu().numpy() == R.gather_points(pts, idx[:, :, 0])).all()
    gy1 = rng.standard_normal(y.shape).astype(np.float32)
    y.backward(_cuda(gy1))
    g1 = R.gather_points_grad(gy1, idx[:, :, 0], N)
    assert np.abs(f2.grad.cpu().numpy() - g1).max() <= 1e-5 * np.abs(g1).max()


def test_reference_layout_gradient_entry_points():
    """issm_pn2_group_points_grad / issm_pn2_three_interpolate_grad write the (b, c, n) layout directly (the Python
    wrappers use the channel-last variants): called here through the C ABI."""
    from dest3d_amd import _lib as L
    lib = L.load()
    rng = np.random.default_rng(12)
    B, C, N, M, S, n3 = 2, 70, 90, 11, 5, 33
    idx = rng.integers(0, N, size=(B, M, S)).astype(np.int32)
    gy = rng.standard_normal((B, C, M, S)).astype(np.float32)
    tg, ti = _cuda(gy), _cuda(idx)
    out = torch.zeros(B, C, N, device="cuda")
    st = L.current_stream_ptr(out.device)
    L.check(lib.issm_pn2_group_points_grad(B, C, N, M, S, tg.data_ptr(), ti.data_ptr(), out.data_ptr(), st), "group grad")
    ref = R.group_points_grad(gy, idx, N)
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    out_cl = torch.zeros(B, N, C, device="cuda")
    L.check(lib.issm_pn2_group_points_grad_cl(B, C, N, M, S, tg.data_ptr(), ti.data_ptr(), out_cl.data_ptr(), st), "group grad cl")
    assert np.abs(out_cl.transpose(1, 2).cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    i3 = rng.integers(0, N, size=(B, n3, 3)).astype(np.int32)
    w3 = rng.uniform(0, 1, size=(B, n3, 3)).astype(np.float32)
    g3 = rng.standard_normal((B, C, n3)).astype(np.float32)
    out3 = torch.zeros(B, C, N, device="cuda")
    tg3, ti3, tw3 = _cuda(g3), _cuda(i3), _cuda(w3)     # kept alive until the kernel has run
    L.check(lib.issm_pn2_three_interpolate_grad(B, C, n3, N, tg3.data_ptr(), ti3.data_ptr(), tw3.data_ptr(),
                                                out3.data_ptr(), st), "interp grad")
    torch.cuda.synchronize()
    ref3 = R.three_interpolate_grad(g3, i3, w3, N)
    assert np.abs(out3.cpu().numpy() - ref3).max() <= 1e-5 * np.abs(ref3).max()


def test_query_and_group_module():
    from dest3d_amd.pointnet2_utils import GroupAll, QueryAndGroup, furthest_point_sample, gather_operation
    rng = np.random.default_rng(8)
    B, N, C, M, S = 2, 400, 5, 32, 8
    xyz = rng.uniform(-1, 1, size=(B, N, 3)).astype(np.float32)
    feats = rng.standard_normal((B, C, N)).astype(np.float32)
    txyz, tf = _cuda(xyz), _cuda(feats)
    fps = furthest_point_sample(txyz, M)
    new_xyz = gather_operation(txyz.transpose(1, 2).contiguous(), fps).transpose(1, 2).contiguous()
    out, gxyz = QueryAndGroup(0.4, S, use_xyz=True, ret_grouped_xyz=True, normalize_xyz=True)(txyz, new_xyz, tf)
    assert out.shape == (B, 3 + C, M, S) and gxyz.shape == (B, 3, M, S)
    idx = R.ball_query(0.4, S, xyz, new_xyz.cpu().numpy())
    want_xyz = (R.group_points(xyz.transpose(0, 2, 1), idx) - new_xyz.cpu().numpy().transpose(0, 2, 1)[..., None]) / 0.4
    assert np.allclose(gxyz.cpu().numpy(), want_xyz, atol=1e-6)
    assert (out[:, 3:].cpu().numpy() == R.group_points(feats, idx)).all()
    assert GroupAll()(txyz, None, tf).shape == (B, 3 + C, 1, N)


@pytest.mark.parametrize("B,C,N,M,S", [(1, 1, 1, 1, 1), (2, 3, 63, 16, 4), (1, 2, 257, 300, 7), (2, 5, 1023, 511, 9),
                                       (1, 3, 4099, 640, 32), (1, 2, 5120, 700, 16), (2, 3, 5121, 800, 16), (1, 1, 40960, 5200, 16),
                                       (1, 1, 40961, 5200, 16)])
def test_grouped_rows_and_their_gradient(B, C, N, M, S):
    """Row remainders, sums in doubles and in floats, entries cut over several workgroups (few channels, many entries), the longest row in LDS and the first
    beyond it; index runs of every length, within a lane's four entries, across lanes and across the rows of a wave."""
    from dest3d_amd.pointnet2_utils import QueryAndGroup, grouping_operation
    rng = np.random.default_rng(N + M)
    idx = np.repeat(rng.integers(0, N, size=B * M * S), rng.integers(1, 90, size=B * M * S))[:B * M * S]
    idx = idx.astype(np.int32).reshape(B, M, S)
    idx[0, M // 2:] = rng.integers(0, N, size=(M - M // 2, S))
    feats = rng.standard_normal((B, C, N)).astype(np.float32)
    f = _cuda(feats).requires_grad_()
    g = grouping_operation(f, _cuda(idx))
    assert (g.detach().cpu().numpy() == R.group_points(feats, idx)).all()
    gy = rng.standard_normal(g.shape).astype(np.float32)
    g.backward(_cuda(gy))
    ref = R.group_points_grad(gy, idx, N)
    assert np.abs(f.grad.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    # coordinates and features in one pass: bit for bit what the separate operators give, and the same gradient
    xyz = rng.uniform(-1, 1, size=(B, N, 3)).astype(np.float32)
    x, q = _cuda(xyz), _cuda(xyz[:, rng.integers(0, N, size=M)])
    one = QueryAndGroup(0.3, S, normalize_xyz=True)
    parts = QueryAndGroup(0.3, S, normalize_xyz=True, ret_grouped_xyz=True)
    f1, f2 = f.detach().clone().requires_grad_(), f.detach().clone().requires_grad_()
    a, (b, _) = one(x, q, f1), parts(x, q, f2)
    assert torch.equal(a, b)
    w = _cuda(rng.standard_normal(a.shape).astype(np.float32))
    a.backward(w)
    b.backward(w)
    assert (f1.grad - f2.grad).abs().max() <= 1e-5 * f2.grad.abs().max()


@pytest.mark.parametrize("N", [300, 5121])
@pytest.mark.parametrize("few", [2, 16, 256])
def test_grouping_gradient_where_many_entries_meet_in_few_points(N, few):
    """Neighbouring entries go to different points, all to the same few: the additions of a wave and of the waves collide."""
    from dest3d_amd.pointnet2_utils import grouping_operation
    rng = np.random.default_rng(few)
    idx = (np.arange(2 * 500 * 32) % 2 if few == 2 else rng.integers(0, few, size=2 * 500 * 32)).astype(np.int32).reshape(2, 500, 32)
    f = torch.zeros(2, 7, N, device="cuda", requires_grad=True)
    gy = rng.integers(-8, 9, size=(2, 7, 500, 32)).astype(np.float32)       # sums are whole numbers: exact in any order
    gy[0, 0, 3, 5] = np.nan
    g, = torch.autograd.grad(grouping_operation(f, _cuda(idx)), f, _cuda(gy))
    want = np.zeros((2, 7, N))
    for b in range(2):
        for c in range(7):
            np.add.at(want[b, c], idx[b].ravel(), gy[b, c].ravel().astype(np.float64))
    assert np.array_equal(g.cpu().numpy(), want.astype(np.float32), equal_nan=True)


def test_grouping_up_to_the_largest_sample():
    """2^31 - 1024 entries in a sample: counts of entries that step past the end of a row stay right.  Forward (features, and
    coordinates relative to the centres) and gradient (ones: how often a point is grouped, exact in fp32)."""
    from dest3d_amd.pointnet2_utils import _GroupXyzPoints, grouping_operation
    N, M, S = 5000, (1 << 21) - 1, 1024
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of free memory")
    idx = torch.arange(M * S, dtype=torch.int32, device="cuda").remainder_(N).view(1, M, S)
    feats = torch.randn(1, 1, N, device="cuda").requires_grad_()
    out = grouping_operation(feats, idx)
    step = 1 << 28
    for at in range(0, M * S, step):
        part = idx.flatten()[at:at + step]
        assert torch.equal(out.detach().flatten()[at:at + step], feats.detach().flatten()[part.long()])
    count, = torch.autograd.grad(out, feats, torch.ones((), device="cuda").expand_as(out))
    want = torch.full((N,), M * S // N, dtype=torch.float32, device="cuda")
    want[:M * S % N] += 1
    assert torch.equal(count.flatten(), want)
    del out
    xyz, centres = torch.randn(1, N, 3, device="cuda"), torch.randn(1, M, 3, device="cuda")
    out = _GroupXyzPoints.apply(None, xyz, centres, idx, 2.0)
    for lo, hi in ((0, 3), (M // 2, M // 2 + 5), (M - 9, M)):
        want = (xyz[0, idx[0, lo:hi].long()] - centres[0, lo:hi, None]) * 2.0
        assert torch.equal(out[0, :, lo:hi], want.permute(2, 0, 1))


@pytest.mark.parametrize("c,m,n", [(1, 1, 3), (3, 5, 700), (9, 2560, 2600), (8, 2561, 2700), (5, 10240, 10300), (2, 10241, 10300),
                                   (2, 40, 20000), (512, 30, 1023), (700, 3, 5121), (3, 1000, 40960), (1, 900, 40961)])
def test_interpolation_rows(c, m, n):
    from dest3d_amd.pointnet2_utils import three_interpolate
    rng = np.random.default_rng(m)
    feats = rng.standard_normal((2, c, m)).astype(np.float32)
    idx = rng.integers(0, m, size=(2, n, 3)).astype(np.int32)
    w = rng.uniform(0, 1, size=(2, n, 3)).astype(np.float32)
    f = _cuda(feats).requires_grad_()
    y = three_interpolate(f, _cuda(idx), _cuda(w))
    ref = R.three_interpolate(feats, idx, w)
    assert np.abs(y.detach().cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    gy = rng.standard_normal(ref.shape).astype(np.float32)
    y.backward(_cuda(gy))
    gref = R.three_interpolate_grad(gy, idx, w, m)
    assert np.abs(f.grad.cpu().numpy() - gref).max() <= 1e-5 * np.abs(gref).max()


@pytest.mark.parametrize("b,c", [(1, 1), (2, 5), (2, 515), (3, 1027)])
@pytest.mark.parametrize("n,m,kind", [(1, 1, "any"), (21, 4, "eights"), (22, 70, "any"), (171, 1, "any"), (1366, 3, "sorted"),
                                      (1366, 300, "one has most"), (4000, 900, "eights"), (9000, 4000, "any")])
def test_interpolation_gradient_lists(b, c, n, m, kind):
    """The sorted lists at their remainders, one, two and four rows a workgroup (the last one short): points whose entries
    fill blocks of eight, fill several waves' shares, or are none; called through the C ABI at every size.  A point's sum of
    k products carries at most k + 1 roundings of 2^-24 of the sum of their magnitudes."""
    from dest3d_amd import _lib as L
    lib = L.load()
    rng = np.random.default_rng(n + c)
    idx = rng.integers(0, m, size=(b, n * 3))
    if kind == "eights":
        idx = np.repeat(rng.integers(0, m, size=(b, n)), 8, axis=1)[:, :n * 3]
    elif kind == "one has most":
        idx[:, 20:n * 3 - 20] = m // 2
    elif kind == "sorted":
        idx.sort(axis=1)
    idx = idx.reshape(b, n, 3).astype(np.int32)
    w = rng.uniform(0, 1, size=(b, n, 3)).astype(np.float32)
    gy = rng.standard_normal((b, c, n)).astype(np.float32)
    tg, ti, tw = _cuda(gy), _cuda(idx), _cuda(w)
    ws = torch.empty(lib.issm_pn2_three_interpolate_grad_rows_workspace(b, n, m), dtype=torch.uint8, device="cuda")
    out = torch.full((b, c, m), float("nan"), device="cuda")
    L.check(lib.issm_pn2_three_interpolate_grad_rows(b, c, n, m, tg.data_ptr(), ti.data_ptr(), tw.data_ptr(), ws.data_ptr(),
                                                     out.data_ptr(), L.current_stream_ptr(out.device)), "interp grad rows")
    got = out.cpu().numpy()
    for i in range(b):
        ref, size = np.zeros((m, c)), np.zeros((m, c))
        for k in range(3):
            term = gy[i].T.astype(np.float64) * w[i, :, k:k + 1]
            np.add.at(ref, idx[i, :, k], term)
            np.add.at(size, idx[i, :, k], np.abs(term))
        count = np.bincount(idx[i].ravel(), minlength=m)[:, None]
        assert (np.abs(got[i].T - ref) <= (count + 1) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("b,c,n,m", [(3, 343, 5123, 700), (2, 301, 10243, 40), (2, 151, 20483, 2048), (1, 259, 40960, 3000)])
def test_interpolation_gradient_of_rows_that_fill_the_lds(b, c, n, m):
    """Four, two, one row a set, and one without the zero behind it, more sets than CUs: a workgroup takes several, some of them of
    two samples, and the last workgroup fewer."""
    test_interpolation_gradient_lists(b, c, n, m, "any")


@pytest.mark.parametrize("c,m,n", [(300, 50, 3501), (700, 3, 5121), (220, 900, 9999), (60, 1000, 40960)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_interpolation_rows_keep_a_target_without_a_number_to_its_points(c, m, n, value):
    """Target 0's gradient is no number (ordinary under loss scaling): its own three points get it, the others nothing of it.
    Four, two and one row per workgroup, and list lengths that fill no workgroup's share."""
    from dest3d_amd.pointnet2_utils import three_interpolate
    rng = np.random.default_rng(n)
    idx = rng.integers(0, m, size=(2, n, 3)).astype(np.int32)
    idx[:, 0] = m - 1
    idx[:, 1:][idx[:, 1:] == m - 1] = 0
    w = rng.uniform(0.1, 1, size=(2, n, 3)).astype(np.float32)
    f = _cuda(rng.standard_normal((2, c, m)).astype(np.float32)).requires_grad_()
    y = three_interpolate(f, _cuda(idx), _cuda(w))
    gy = rng.standard_normal(y.shape).astype(np.float32)
    gy[:, :, 0] = value
    y.backward(_cuda(gy))
    g = f.grad.cpu().numpy()
    assert (np.isnan(g[..., m - 1]) if np.isnan(value) else np.isposinf(g[..., m - 1])).all()
    gy[:, :, 0] = 0.0
    ref = R.three_interpolate_grad(gy, idx, w, m)[..., :m - 1]
    assert np.abs(g[..., :m - 1] - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("b,n,m", [(1, 1, 256), (1, 129, 2048), (2, 1025, 2049), (3, 700, 4096), (1, 33000, 4097), (300, 3, 300), (2, 1024, 8192), (1, 262145, 257),
                                   (86, 2049, 256), (129, 1025, 2047), (17, 16385, 4063), (17, 16385, 4064), (257, 1024, 300), (257, 1025, 300),
                                   (257, 1537, 1519), (257, 1536, 1520), (171, 2561, 256), (513, 3, 1025)])
def test_three_nn_shares(b, n, m):
    """Targets shared by workgroups at the edges of their shares, known points at those of a thread's: the pass over all points by index."""
    from dest3d_amd.pointnet2_utils import three_nn
    g = torch.Generator().manual_seed(n + m)
    u, k = torch.rand(b, n, 3, generator=g).cuda(), torch.rand(b, m, 3, generator=g).cuda()
    k[:, 1::7] = k[:, :1]     # some in one place: ties go to the smaller index
    dist, idx = three_nn(u, k)
    at = torch.unique(torch.tensor([0, n // 3, n // 2, n - 1] + [min(x, n - 1) for x in range(0, n, 127)])).cuda()
    d = (u[:, at, None].cpu().double() - k[:, None].cpu().double()).pow(2).sum(-1)
    near = torch.sort(d, dim=-1, stable=True).values[..., :3]
    got = torch.gather(d, 2, idx[:, at].cpu().long())
    assert ((got - near).abs() <= 1e-6 * near + 1e-12).all() and ((dist[:, at].cpu().double().pow(2) - near).abs() <= 1e-5 * near + 1e-12).all()
    assert (idx[:, at, 0] != idx[:, at, 1]).all() and (idx[:, at, 1] != idx[:, at, 2]).all()


@pytest.mark.parametrize("m", [255, 256, 257, 2048, 8192, 8193])
def test_three_nn_grid(m):
    """Both sides of the grid's range; sample 1: a flat sheet with duplicates (ties go to the smaller index), clusters and far
    points, unknown points far outside; sample 2: one place; sample 3: coordinates the grid cannot hold."""
    from dest3d_amd.pointnet2_utils import three_nn
    rng = np.random.default_rng(m)
    k = rng.uniform(-2, 2, size=(4, m, 3)).astype(np.float32)
    u = rng.uniform(-2, 2, size=(4, 700, 3)).astype(np.float32)
    k[1, :, 1] = 0.5
    k[1, m // 2:] = k[1, :m - m // 2]
    k[1, m // 4:m // 3] *= 0.01
    k[1, 7] = (1e4, 3.0, -1e5)
    u[1, :50] *= 1e3
    u[1, 50:60] = k[1, :10]
    k[2] = k[2, 0]
    k[3, 5, 0] = np.inf
    dist, idx = three_nn(_cuda(u), _cuda(k))
    d2_ref, idx_ref = R.three_nn(u, k)
    assert (idx.cpu().numpy() == idx_ref).all()
    assert np.allclose(dist.cpu().numpy(), np.sqrt(d2_ref), rtol=1e-6, atol=0)


def test_error_codes():
    from dest3d_amd import _lib as L
    lib = L.load()
    assert lib.issm_pn2_furthest_point_sampling(1, 10, 4, None, None, None, None) == -1
    assert lib.issm_pn2_furthest_point_sampling(1, 0, 4, None, None, None, None) == -2
    assert lib.issm_pn2_ball_query(-1, 10, 4, 0.5, 8, None, None, None, None) == -2
    assert lib.issm_pn2_group_points(1, 2, 0, 4, 4, None, None, None, None) == -2
    assert lib.issm_pn2_three_nn(0, 5, 5, None, None, None, None, None) == 0


def test_operands_of_another_batch_or_device_are_refused():
    """Refused before a kernel is given their address: a batch smaller than the first operand's, and tensors on the host."""
    from dest3d_amd import pointnet2_utils as P
    xyz, feat, centres = torch.rand(2, 40, 3).cuda(), torch.rand(2, 5, 40).cuda(), torch.rand(2, 8, 3).cuda()
    idx, idx3 = torch.zeros(2, 8, 4, dtype=torch.int32).cuda(), torch.zeros(2, 30, 3, dtype=torch.int32).cuda()
    weight = torch.rand(2, 30, 3).cuda()
    calls = [(P.furthest_point_sample, (torch.rand(2, 40, 2).cuda(), 8), ()), (P.gather_operation, (feat, idx[:, :, 0]), (1,)),
             (P.three_nn, (xyz, centres), (1,)), (P.three_interpolate, (feat, idx3, weight), (1, 2)),
             (P.grouping_operation, (feat, idx), (1,)), (P.ball_query, (0.3, 4, xyz, centres), (3,)),
             (P.QueryAndGroup(0.3, 4), (xyz, centres, feat), (1, 2))]
    for call, args, at in calls:
        if not at:
            with pytest.raises(ValueError):
                call(*args)
            continue
        call(*args)
        for i in at:
            for bad, error in ((args[i][:1], (ValueError, RuntimeError)), (args[i].cpu(), RuntimeError)):
                with pytest.raises(error):
                    call(*(bad if j == i else t for j, t in enumerate(args)))
