"""Gated RMSNorm / LayerNorm on MI355X with the Python surface of the reference's
issm_triton/layernorm_gated.py: ``RMSNorm`` and ``LayerNorm`` modules (layernorm_gated.py:378-427),
``rmsnorm_fn`` / ``layernorm_fn`` (:370-375) and the autograd function behind them (``LayerNormFn``,
:328-367).  Arithmetic runs in libissm_hip.so."""
from __future__ import annotations

import torch

from . import _lib as L


def _norm_args(x2, z2, w, eps, group_size, norm_before_gate, bias=None, layer_norm=False) -> L.NormArgs:
    """The C ABI's argument block for callers from Python (preallocated buffers, graph capture), as the operator fills it."""
    return L.NormArgs.from_buffer_copy(L.host().norm_args(x2, z2, w, bias, float(eps), 0 if group_size is None else int(group_size),
                                                          bool(norm_before_gate), bool(layer_norm)))


class LayerNormFn:
    """layernorm_gated.py:328-367: same arguments, same four gradients (x, weight, bias, z); the node itself is compiled."""

    @staticmethod
    def apply(x, weight, bias, z=None, eps=1e-6, group_size=None, norm_before_gate=True, is_rms_norm=False):
        return L.host().norm(x, weight, bias, z, float(eps), 0 if group_size is None else int(group_size), bool(norm_before_gate),
                             bool(is_rms_norm))


def layernorm_fn(x, weight, bias, z=None, eps=1e-6, group_size=None, norm_before_gate=True, is_rms_norm=False):
    """layernorm_gated.py:370-371."""
    return LayerNormFn.apply(x, weight, bias, z, eps, group_size, norm_before_gate, is_rms_norm)


def rmsnorm_fn(x, weight, bias, z=None, eps=1e-6, group_size=None, norm_before_gate=True):
    """layernorm_gated.py:374-375."""
    return LayerNormFn.apply(x, weight, bias, z, eps, group_size, norm_before_gate, True)


class LayerNorm(torch.nn.Module):
    """Drop-in for issm_triton.layernorm_gated.LayerNorm (layernorm_gated.py:378-403)."""

    def __init__(self, hidden_size, eps=1e-5, group_size=None, norm_before_gate=True, device=None, dtype=None):
        """If group_size is not None, each group of group_size features is normalised on its own.
        group_size=None means a single group."""
        factory_kwargs = {"device": device, "dtype": dtype}
        super().__init__()
        self.eps = eps
        self.weight = torch.nn.Parameter(torch.empty(hidden_size, **factory_kwargs))
        self.bias = torch.nn.Parameter(torch.empty(hidden_size, **factory_kwargs))
        self.group_size = group_size
        self.norm_before_gate = norm_before_gate
        self.reset_parameters()

    def reset_parameters(self):
        torch.nn.init.ones_(self.weight)
        torch.nn.init.zeros_(self.bias)

    def forward(self, x, z=None):
        """norm(x) * silu(z) if norm_before_gate, else norm(x * silu(z)); z optional."""
        return layernorm_fn(x, self.weight, self.bias, z=z, group_size=self.group_size, eps=self.eps,
                            norm_before_gate=self.norm_before_gate)


class RMSNorm(torch.nn.Module):
    """Drop-in for issm_triton.layernorm_gated.RMSNorm (layernorm_gated.py:405-427)."""

    def __init__(self, hidden_size, eps=1e-5, group_size=None, norm_before_gate=True, device=None, dtype=None):
        """If group_size is not None, each group of group_size features is normalised on its own.
        group_size=None means a single group."""
        factory_kwargs = {"device": device, "dtype": dtype}
        super().__init__()
        self.eps = eps
        self.weight = torch.nn.Parameter(torch.empty(hidden_size, **factory_kwargs))
        self.register_parameter("bias", None)
        self.group_size = group_size
        self.norm_before_gate = norm_before_gate
        self.reset_parameters()

    def reset_parameters(self):
        torch.nn.init.ones_(self.weight)

    def forward(self, x, z=None):
        """norm(x) * silu(z) if norm_before_gate, else norm(x * silu(z)); z optional."""
        return rmsnorm_fn(x, self.weight, self.bias, z=z, eps=self.eps, group_size=self.group_size,
                          norm_before_gate=self.norm_before_gate)
