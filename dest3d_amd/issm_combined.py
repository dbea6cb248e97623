"""Operator API of the interactive-SSM chunked scan on MI355X.

Same Python surface as the reference's issm_triton/issm_combined.py:
``ISSM_chunk_scan_combined(x, dt, A, B, C, chunk_size, D=None, z=None, dt_bias=None,
initial_states=None, seq_idx=None, dt_softplus=False, dt_limit=(0, inf),
return_final_states=False)`` (issm_combined.py:16-34) backed by
``ISSMChunkScanCombinedFn`` (issm_combined.py:37-54) with the same 14 backward slots.
Checks, argument blocks, allocation and the autograd nodes are compiled (csrc/host_ops.cpp);
all arithmetic runs in libissm_hip.so.

``ISSM_biscan_combined`` additionally runs the bidirectional pair of scans that
MultiHeadISSMScan issues (models/dest_module.py:565-575) in one call, reading the shared
dt backwards for the second direction instead of materialising flipped copies.
"""
from __future__ import annotations

import ctypes as C

import torch

from . import _lib as L

INF = float("inf")


class _Problem:
    """Kernel-ready argument block of one call (1 or 2 directions) for callers of the C ABI from Python (the stage entry
    points, preallocated buffers): checks, conversions and the block itself are those of the operators below."""

    def __init__(self, xs, dt, A, Bs, Cs, chunk_size, D, zs, dt_bias, h0, seq_idx, dt_softplus, dt_limit):
        _chunk_size(chunk_size)
        if seq_idx is not None and len(xs) != 1:
            raise NotImplementedError("seq_idx with the fused bidirectional scan")
        two = lambda v: (v[0], v[1] if len(v) > 1 else None)
        self.device = xs[0].device
        self._block, self._tensors = L.host().scan_args(
            *two(xs), dt, A, *two(Bs), *two(Cs), D, *two(zs), dt_bias, h0, seq_idx, bool(dt_softplus), float(dt_limit[0]),
            float(dt_limit[1]))

    def args(self) -> L.ScanArgs:
        a = L.ScanArgs.from_buffer_copy(self._block)
        a.stream = L.current_stream_ptr(self.device)
        return a

    def workspace(self, a: L.ScanArgs, bwd: bool) -> torch.Tensor:
        lib = L.load()
        n = C.c_size_t(0)
        fn = lib.issm_bwd_workspace_bytes if bwd else lib.issm_fwd_workspace_bytes
        L.check(fn(C.byref(a), C.byref(n)), "workspace query")
        return torch.empty(max(n.value, 256), dtype=torch.uint8, device=self.device)


def _chunk_size(chunk_size):
    if not (isinstance(chunk_size, int) and chunk_size > 0):
        raise ValueError(f"chunk_size must be a positive int, got {chunk_size!r}")


class ISSMChunkScanCombinedFn:
    """Autograd contract of issm_combined.py:37-54: gradients for x, dt, A, B, C, D, z, dt_bias, initial_states, none for
    chunk_size, seq_idx, dt_softplus, dt_limit, return_final_states.  The node itself is compiled."""

    @staticmethod
    def apply(x, dt, A, B, C, chunk_size, D=None, z=None, dt_bias=None, initial_states=None, seq_idx=None,
              dt_softplus=False, dt_limit=(0.0, INF), return_final_states=False):
        _chunk_size(chunk_size)
        res = L.host().scan(x, dt, A, B, C, D, z, dt_bias, initial_states, seq_idx, bool(dt_softplus), float(dt_limit[0]),
                            float(dt_limit[1]), bool(return_final_states))
        return (res[0], res[1]) if return_final_states else res[0]


def ISSM_chunk_scan_combined(x, dt, A, B, C, chunk_size, D=None, z=None, dt_bias=None, initial_states=None,
                             seq_idx=None, dt_softplus=False, dt_limit=(0.0, INF), return_final_states=False):
    """
    Argument:
        x: (batch, seqlen, nheads, headdim)
        dt: (batch, seqlen, nheads, dstate)
        A: (nheads, dstate)
        B: (batch, seqlen, ngroups, dstate)
        C: (batch, seqlen, ngroups, dstate)
        chunk_size: int (accepted for parity; the result does not depend on it)
        D: (nheads, headdim) or (nheads,)
        z: (batch, seqlen, nheads, headdim)
        dt_bias: (nheads, dstate)
        initial_states: (batch, nheads, headdim, dstate)
        seq_idx: (batch, seqlen) integer ids of the sequences packed into a row, or None.  The ids of a row must
            not decrease.  initial_states count as id 0 (issm_chunk_scan.py:123): they feed the first sequence of a
            row whose ids start at 0 and nothing in a row whose ids start higher.  Every change of id is a cut
            (the reference's equality masks would reconnect a repeated id inside a chunk only; not reproduced).
        dt_softplus: whether to apply softplus to dt (+ dt_bias)
    Return:
        out: (batch, seqlen, nheads, headdim)  [, final_states (batch, nheads, headdim, dstate) fp32]
    """
    s = _head_split(x.shape[-1]) if x.dim() == 4 else 1
    if s > 1:
        x, dt, A, D, z, dt_bias, initial_states = _split_heads(s, x, dt, A, D, z, dt_bias, initial_states)
    res = ISSMChunkScanCombinedFn.apply(x, dt, A, B, C, chunk_size, D, z, dt_bias, initial_states, seq_idx,
                                        dt_softplus, dt_limit, return_final_states)
    if s == 1:
        return res
    if return_final_states:
        return _merge_heads(s, res[0]), _merge_heads(s, res[1], state=True)
    return _merge_heads(s, res)


MAX_HEADDIM = 64   # what one workgroup's tiles are built for (ISSM_E_UNSUPPORTED above it)


def _head_split(headdim: int) -> int:
    """The scan is independent across the head dimension, so a head wider than the kernels' 64 runs as `s` heads of
    headdim / s that share the head's dt, A and dt_bias (the reference has no such limit, issm_combined.py:58-83):
    the smallest s that divides headdim with headdim / s <= 64."""
    if headdim <= MAX_HEADDIM:
        return 1
    return next(s for s in range(2, headdim + 1) if headdim % s == 0 and headdim // s <= MAX_HEADDIM)


def _split_heads(s, x, dt, A, D, z, dt_bias, h0):
    """Views / repeats that turn (H, P) into (H s, P / s), head h -> heads h s .. h s + s - 1 (same group as h).
    Plain differentiable tensor operations: autograd sums the gradients of the repeated dt, A, dt_bias, D."""
    b, l, h, p = x.shape
    q = p // s
    rep = lambda t, dim: None if t is None else t.repeat_interleave(s, dim=dim)
    heads = lambda t: None if t is None else t.reshape(b, l, h * s, q)
    if D is not None:
        D = D.reshape(h * s, q) if D.dim() == 2 else D.repeat_interleave(s, dim=0)
    h0 = None if h0 is None else h0.reshape(b, h * s, q, h0.shape[-1])
    return heads(x), rep(dt, 2), rep(A, 0), D, heads(z), rep(dt_bias, 0), h0


def _merge_heads(s, t, state=False):
    if state:   # (B, H s, P / s, N) -> (B, H, P, N)
        return t.reshape(t.shape[0], t.shape[1] // s, t.shape[2] * s, t.shape[3])
    return t.reshape(t.shape[0], t.shape[1], t.shape[2] // s, t.shape[3] * s)


class ISSMBiScanFn:
    """ISSM_biscan_combined for heads of up to 64; gradients for all tensor arguments.  The node itself is compiled."""

    @staticmethod
    def apply(x_f, x_b, dt, A, B_f, B_b, C_f, C_b, chunk_size, D, dt_bias, initial_states, dt_softplus, dt_limit):
        _chunk_size(chunk_size)
        return tuple(L.host().biscan(x_f, x_b, dt, A, B_f, B_b, C_f, C_b, D, dt_bias, initial_states, bool(dt_softplus),
                                     float(dt_limit[0]), float(dt_limit[1])))


def ISSM_biscan_combined(x_f, x_b, dt, A, B_f, B_b, C_f, C_b, chunk_size, D=None, dt_bias=None,
                         initial_states=None, dt_softplus=False, dt_limit=(0.0, INF)):
    """Both directions of MultiHeadISSMScan's bidirectional scan in one operator call -> (y_f, y_b, last_f, last_b).
    Inputs and outputs are in natural time order; direction "b" is scanned from the last token to the first (what
    dest_module.py:568-573 obtains with four flips and a second operator call)."""
    s = _head_split(x_f.shape[-1]) if x_f.dim() == 4 else 1
    if s > 1:
        x_b = x_b.reshape(x_b.shape[0], x_b.shape[1], x_b.shape[2] * s, x_b.shape[3] // s)
        x_f, dt, A, D, _, dt_bias, initial_states = _split_heads(s, x_f, dt, A, D, None, dt_bias, initial_states)
    res = ISSMBiScanFn.apply(x_f, x_b, dt, A, B_f, B_b, C_f, C_b, chunk_size, D, dt_bias, initial_states, dt_softplus, dt_limit)
    if s == 1:
        return res
    return (_merge_heads(s, res[0]), _merge_heads(s, res[1]), _merge_heads(s, res[2], state=True),
            _merge_heads(s, res[3], state=True))
