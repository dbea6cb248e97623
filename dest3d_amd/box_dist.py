"""Box-to-point distance encoding (``BoxDistFun``) and locality weight of DEST's decoder layer, on MI355X.

Mirrors models/dest_module.py:147-195 (``BoxDistFun``: same constructor arguments, buffer and parameter names, so
a reference ``state_dict`` loads unchanged) and :240-249 (``local_weight``).  The per-(point, box) work -- corner
deltas, rotation, signed-log compression, trilinear sampling of the learned table, the sum over 8 corners, and the
exponential weight -- runs in one kernel of libissm_hip.so with the table in LDS; ``dist`` comes out contiguous as
(B, nP, nQ, C), the layout the scan's parameter generation reads.  Only the table (hence the small MLP that
produces it) receives a gradient: the reference detaches the corners, and point positions and angles are inputs.
There is no fallback path."""
from __future__ import annotations

import ctypes as C
from typing import Optional

import torch
import torch.nn as nn

import torch.autograd.forward_ad as _forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import _lib as L
from .scan_module import _hooked

CHANNELS = 16      # table channels the kernels are built for (DEST's decoder: BoxDistFun(out_dim=16))
MAX_NODES = 1024   # table nodes that fit the LDS copy


def box_parametrization_to_corners(center, size, angle):
    """The 8 corners (..., 8, 3) of boxes given centre (..., 3), size (..., 3) = (l, w, h) and heading (...),
    in the frame of the inputs; corner order of dest_module.py:62-70 after the camera/lidar axis changes of
    :26-38 are composed: x = cx + sx l/2 cos + sz w/2 sin, y = cy - sx l/2 sin + sz w/2 cos, z = cz - sy h/2."""
    sx = center.new_tensor([1, 1, -1, -1, 1, 1, -1, -1])
    sy = center.new_tensor([1, 1, 1, 1, -1, -1, -1, -1])
    sz = center.new_tensor([1, -1, -1, 1, 1, -1, -1, 1])
    lx = size[..., 0:1] / 2 * sx
    hy = size[..., 2:3] / 2 * sy
    wz = size[..., 1:2] / 2 * sz
    c, s = torch.cos(angle).unsqueeze(-1), torch.sin(angle).unsqueeze(-1)
    x = center[..., 0:1] + lx * c + wz * s
    y = center[..., 1:2] - lx * s + wz * c
    z = center[..., 2:3] - hy
    return torch.stack([x, y, z], dim=-1)


def _f32c(t: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    return None if t is None else t.detach().float().contiguous()


def _lattice(coords: torch.Tensor) -> Optional[tuple]:
    """(n0, n1, n2) of a (1, n0, n1, n2, 3) table of coordinates; None for any other shape.  (The kernel writes 16 values for
    every three of the coordinates, so their number has to be that of the table's nodes.)"""
    return tuple(coords.shape[1:4]) if coords.dim() == 5 and coords.shape[0] == 1 and coords.shape[4] == 3 else None


def _watched() -> bool:
    """Whether a dispatch or function mode, a tracer or a compiler sees the operations that are called here.  (A default device
    is a function mode as well, and asks for nothing but new tensors.)"""
    return bool(torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack()
                or any(type(m) is not DeviceContext for m in _get_current_function_mode_stack()))


class _HiddenFn(torch.autograd.Function):
    """The hidden values of the table's MLP, from copies of their weights, as values that w1 and b1 get a gradient through."""

    @staticmethod
    def forward(ctx, w1, b1, x, first):
        h = torch.relu(nn.functional.linear(x, first[:w1.numel()].view(w1.shape), first[w1.numel():]))
        ctx.save_for_backward(x, h)
        return h

    @staticmethod
    def backward(ctx, dh):
        x, h = ctx.saved_tensors
        dh = dh * (h > 0)
        return dh.t() @ x, dh.sum(0), None, None


class BoxTableFn(torch.autograd.Function):
    """The table of ``BoxDistFun`` with gradients: its modules' products forward, one kernel backward.  The modules keep neither w1 nor b1 for
    their backward, and both may be changed in place before it: what the kernel computes the hidden values from again are copies."""

    @staticmethod
    def forward(ctx, module, w1, b1, w2, coords):
        ctx.first = (w1, b1)   # (whose gradient it is; not their values)
        ctx.save_for_backward(torch.cat((w1.reshape(-1), b1)), w2, coords.to(w1.dtype))
        return module.rpe_table().float().contiguous()

    @staticmethod
    def backward(ctx, dtable):
        first, w2, coords = ctx.saved_tensors
        w1, b1 = ctx.first
        if torch.is_grad_enabled():   # to be differentiated again: as operations that autograd records
            x, g = coords.reshape(-1, 3), dtable.reshape(CHANNELS, -1).to(w1.dtype)
            h = _HiddenFn.apply(w1, b1, x, first)
            dh = (g.t() @ w2) * (h > 0)
            return None, dh.t() @ x, dh.sum(0), g @ h, None
        a, g = _table_args(first[:w1.numel()].view(w1.shape), first[w1.numel():], w2, coords), _f32c(dtable)
        grads = [torch.empty_like(t) for t in (w1, b1, w2)]
        with torch.cuda.device(w1.device):
            L.check(L.load().issm_box_table_bwd(C.byref(a), g.data_ptr(), *(t.data_ptr() for t in grads)), "issm_box_table_bwd")
        return None, *grads, None


def _table_args(w1, b1, w2, coords):
    a = L.BoxTableArgs()
    a.nodes, a.hidden = coords.numel() // 3, w1.shape[0]
    a.dtype, a.coords_dtype = L.dtype_code(w1.dtype), L.dtype_code(coords.dtype)
    a.coords, a.w1, a.b1, a.w2 = coords.data_ptr(), w1.data_ptr(), b1.data_ptr(), w2.data_ptr()
    a.stream = L.current_stream_ptr(w1.device)
    return a


def _wants_gradient(mlp) -> bool:
    return torch.is_grad_enabled() and any(p.requires_grad for p in mlp)


class BoxDistFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, table, key_xyz, corners, angle, qcenter, radius, weight_dist, log_scale, max_value, out_dtype,
                want_dist, want_weights, only=False):
        L.require_gpu(key_xyz, "key_xyz")
        lib = L.load()
        Bsz, nP = key_xyz.shape[:2]
        nQ = corners.shape[1]
        key, cor, ang = _f32c(key_xyz), _f32c(corners), _f32c(angle)
        as_boxes = cor.dim() == 3          # (B, nQ, 7) boxes instead of (B, nQ, 8, 3) corners
        assert cor.shape[2:] == ((7,) if as_boxes else (8, 3))
        L.require_operand(key, "key_xyz", key, Bsz, nP, 3)
        L.require_operand(cor, "the boxes", key, Bsz, nQ, *cor.shape[2:])
        L.require_operand(ang, "angle", key, Bsz, nQ)
        a = L.BoxDistArgs()
        a.batch, a.seqlen, a.nquery = Bsz, nP, nQ
        a.dtype = L.dtype_code(out_dtype)
        a.key = key.data_ptr()
        if as_boxes:
            a.boxes, a.min_radius = cor.data_ptr(), 0.64
        else:
            a.corners = cor.data_ptr()
        a.angle = None if ang is None else ang.data_ptr()
        a.log_scale, a.max_value = float(log_scale), float(max_value)
        a.stream = L.current_stream_ptr(key.device)
        a.D = a.H = a.W = 1
        dist = weights = tab = qc = rad = None
        with torch.cuda.device(key.device):
            if want_dist:
                assert table.dim() == 4 and table.shape[0] == CHANNELS, "table must be (16, D, H, W)"
                tab = _f32c(table)
                L.require_operand(tab, "table", key)
                a.D, a.H, a.W = tab.shape[1:]
                a.table = tab.data_ptr()
                dist = torch.empty((Bsz, nP, nQ, CHANNELS), dtype=out_dtype, device=key.device)
                a.dist = dist.data_ptr()
            if want_weights:
                weights = torch.empty((Bsz, nP, nQ), dtype=torch.float32, device=key.device)
                a.weight_dist = float(weight_dist)
                if qcenter is not None:
                    qc, rad = _f32c(qcenter), _f32c(radius)
                    L.require_operand(qc, "the weights' centres", key, Bsz, nQ, 3)
                    L.require_operand(rad, "the weights' radii", key, Bsz, nQ)
                    a.qcenter, a.radius = qc.data_ptr(), rad.data_ptr()
                else:
                    assert as_boxes, "weights need (qcenter, radius) or boxes"
                a.weights = weights.data_ptr()
            run = lib.issm_box_dist_fwd_only if only else lib.issm_box_dist_fwd   # only: no backward follows
            L.check(run(C.byref(a)), "issm_box_dist_fwd")
        ctx.save_for_backward(key, cor, ang)
        ctx.meta = (None if table is None else (tuple(table.shape), table.dtype), log_scale, max_value, out_dtype)
        ctx.mark_non_differentiable(*[t for t in (weights,) if t is not None])
        return dist, weights

    @staticmethod
    def backward(ctx, ddist, _dweights):
        key, cor, ang = ctx.saved_tensors
        tmeta, log_scale, max_value, out_dtype = ctx.meta
        dtable = None
        if ddist is not None and tmeta is not None and ctx.needs_input_grad[0]:
            lib = L.load()
            (Cn, D, H, W), tdt = tmeta
            Bsz, nP = key.shape[:2]
            nQ = cor.shape[1]
            g = ddist.to(out_dtype).contiguous()
            with torch.cuda.device(key.device):
                a = L.BoxDistArgs()
                a.batch, a.seqlen, a.nquery, a.D, a.H, a.W = Bsz, nP, nQ, D, H, W
                a.dtype = L.dtype_code(out_dtype)
                a.key = key.data_ptr()
                if cor.dim() == 3:
                    a.boxes, a.min_radius = cor.data_ptr(), 0.64
                else:
                    a.corners = cor.data_ptr()
                a.angle = None if ang is None else ang.data_ptr()
                a.log_scale, a.max_value = float(log_scale), float(max_value)
                nbytes = lib.issm_box_dist_bwd_scratch_bytes(Bsz, nP, nQ, D, H, W)
                partial = torch.empty(nbytes // 8, dtype=torch.int64, device=key.device)
                out = torch.zeros((Cn, D, H, W), dtype=torch.float32, device=key.device)
                a.ddist, a.partial, a.dtable = g.data_ptr(), partial.data_ptr(), out.data_ptr()
                a.stream = L.current_stream_ptr(key.device)
                L.check(lib.issm_box_dist_bwd(C.byref(a)), "issm_box_dist_bwd")
            dtable = out.to(tdt)
        return (dtable,) + (None,) * 12


def box_dist(table, key_xyz, corners, angle=None, log_scale=512.0, max_value=4.0, out_dtype=None):
    """table (16, D, H, W), key_xyz (B, nP, 3), corners (B, nQ, 8, 3), angle (B, nQ) or None -> (B, nP, nQ, 16)."""
    out_dtype = out_dtype or (table.dtype if table.dtype in (torch.float32, torch.bfloat16) else torch.float32)
    return BoxDistFn.apply(table, key_xyz, corners, angle, None, None, 0.0, log_scale, max_value, out_dtype,
                           True, False)[0]


def local_weight(key_xyz, query_pos, weight_dist=15.0, min_radius=0.64):
    """exp(weight_dist * min(radius - |key - centre|, 0)), radius = max(|size|, min_radius); query_pos (B, nQ, 6)
    = centre + size -> (B, nP, nQ) fp32   (dest_module.py:240-249)."""
    radius = query_pos[..., 3:].float().square().sum(-1).sqrt().clamp_min(min_radius)
    corners = query_pos.new_zeros((*query_pos.shape[:2], 8, 3))
    return BoxDistFn.apply(None, key_xyz, corners, None, query_pos[..., :3], radius, float(weight_dist), 512.0, 4.0,
                           torch.float32, False, True)[1]


class BoxDistFun(nn.Module):
    """Learned relative-position encoding between key points and query boxes (dest_module.py:147-195)."""

    def __init__(self, log_scale: int = 512, rpe_quant: str = "bilinear_4_10", out_dim: int = 4, rpe_dim: int = 128):
        super().__init__()
        self.log_scale = log_scale
        self.interp_method, max_value, num_points = rpe_quant.split("_")
        max_value, num_points = float(max_value), int(num_points)
        if self.interp_method != "bilinear":
            raise NotImplementedError("the HIP kernel samples the table trilinearly ('bilinear' grid_sample mode)")
        if out_dim != CHANNELS or num_points ** 3 > MAX_NODES:
            raise NotImplementedError(f"built for out_dim == {CHANNELS} and at most {MAX_NODES} table nodes")
        lin = torch.linspace(-max_value, max_value, num_points, dtype=torch.float32)
        table = torch.stack(torch.meshgrid(lin, lin, lin, indexing="ij"), dim=-1).unsqueeze(0)
        self.register_buffer("relative_coords_table", table)
        self.max_value = max_value
        self.cpb_mlps = nn.Sequential(nn.Linear(3, rpe_dim, bias=True), nn.ReLU(inplace=False),
                                      nn.Linear(rpe_dim, out_dim, bias=False))

    def rpe_table(self) -> torch.Tensor:
        """(out_dim, n, n, n): the MLP evaluated on the coordinate lattice (dest_module.py:191)."""
        return self.cpb_mlps(self.relative_coords_table.to(self.cpb_mlps[0].weight.dtype))[0].permute(3, 0, 1, 2)

    def _plain_mlp(self):
        """(w1, b1, w2, coords) of the table where the kernels take them and the modules are what this class made them (calling them would
        do nothing else, and nobody watches); None otherwise."""
        if _watched():
            return None
        if type(self.cpb_mlps) is not nn.Sequential or len(self.cpb_mlps) != 3:
            return None
        lin1, act, lin2 = self.cpb_mlps
        if type(lin1) is not nn.Linear or type(act) is not nn.ReLU or type(lin2) is not nn.Linear:
            return None
        ps, coords = (lin1.weight, lin1.bias, lin2.weight), self.relative_coords_table
        w = ps[0]
        if type(self).rpe_table is not BoxDistFun.rpe_table or "rpe_table" in self.__dict__ or lin2.bias is not None or \
                lin1.bias is None or any(_hooked(m) for m in (self.cpb_mlps, lin1, act, lin2)):
            return None
        if torch.is_autocast_enabled("cuda") or _forward_ad._current_level >= 0 or not w.is_cuda or \
                w.dtype not in (torch.float32, torch.bfloat16) or type(coords) is not torch.Tensor or \
                coords.dtype not in (torch.float32, torch.bfloat16) or \
                w.shape[0] > 256 or w.shape != (w.shape[0], 3) or ps[1].shape != w.shape[:1] or \
                ps[2].shape != (CHANNELS, w.shape[0]) or not coords.is_contiguous() or coords.device != w.device or \
                (torch.is_grad_enabled() and coords.requires_grad) or \
                any(p.dtype != w.dtype or p.device != w.device or not p.is_contiguous() or
                    type(p) not in (nn.Parameter, torch.Tensor) for p in ps) or _lattice(coords) is None:
            return None
        return (*ps, coords)

    def _plain_table(self, mlp=None):
        """The same table, (out_dim, n, n, n) fp32, from one kernel where nothing is to be differentiated; None otherwise."""
        mlp = self._plain_mlp() if mlp is None else mlp
        # (a checkpointed segment's run: both of them take the sums of one with gradients)
        if mlp is None or _wants_gradient(mlp) or L.host().runs_twice():
            return None
        w = mlp[0]
        table = torch.empty((CHANNELS, *_lattice(mlp[3])), dtype=torch.float32, device=w.device)
        a = _table_args(*mlp)
        a.table = table.data_ptr()
        with torch.cuda.device(w.device):
            L.check(L.load().issm_box_table(C.byref(a)), "issm_box_table")
        return table

    def forward(self, key_xyz, query_xyz, query_size, query_angle, weight_query_pos=None, weight_dist=15.0):
        """-> dist (B, nP, nQ, out_dim).  With ``weight_query_pos`` (B, nQ, 6) the locality weights (B, nP, nQ)
        of ``local_weight`` are computed in the same pass and returned as a second value."""
        # the kernel derives the corners (and, for the weights, centre and radius) from the boxes themselves
        boxes = torch.cat([query_xyz, query_size, query_angle.unsqueeze(-1)], dim=-1).detach()
        mlp = self._plain_mlp()
        table = None if mlp is None else self._plain_table(mlp)
        plain = table is not None
        if mlp is not None and _wants_gradient(mlp):
            table = BoxTableFn.apply(self, *mlp)
        elif not plain:
            mlp, table = None, self.rpe_table()
        out_dtype = self.cpb_mlps[0].weight.dtype if mlp is not None else table.dtype if table.dtype in (torch.float32, torch.bfloat16) else torch.float32
        if weight_query_pos is None:
            return BoxDistFn.apply(table, key_xyz, boxes, query_angle, None, None, 0.0, self.log_scale, self.max_value,
                                   out_dtype, True, False, plain)[0]
        same_boxes = (weight_query_pos.shape[-1] == 6 and query_xyz.data_ptr() == weight_query_pos.data_ptr()
                      and query_size.data_ptr() == weight_query_pos[..., 3:].data_ptr()
                      and query_xyz.stride() == weight_query_pos[..., :3].stride())
        if same_boxes:        # query_pos[..., :3] / query_pos[..., 3:], as the decoder layer calls it
            qc = rad = None   # the weight's boxes are the encoding's: centre and radius come from `boxes`
        else:
            qc = weight_query_pos[..., :3]
            rad = weight_query_pos[..., 3:].float().square().sum(-1).sqrt().clamp_min(0.64)
        return BoxDistFn.apply(table, key_xyz, boxes, query_angle, qc, rad, float(weight_dist), self.log_scale,
                               self.max_value, out_dtype, True, True, plain)
