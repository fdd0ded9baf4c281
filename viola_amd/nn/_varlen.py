"""Variable-group (MoE-expert style) FP8 linear: `groups` independent Linear(scaling="grouped")
problems that share in/out features and differ in how many rows each owns.

The reference has no such operator (its "grouped" means group-scaled quantization); the semantics
here are "a Python loop of per-group viola.nn.Linear(scaling='grouped')": rows are quantized with
(1, 32) tiles, weights with (32, 32) blocks per group, and the weight gradient of a group uses the
transposed (1, 32) quantization of that group's own rows (32-token tiles counted from the group's
first row). One launch covers all groups; empty groups yield no rows and a zero dW.
"""

import functools
import math

import torch
from torch import nn

from .. import _lib
from . import _grouped_kernels as kernels
from ..precision import settings

_FORMATS = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
GW = (32, 32)


@functools.lru_cache(maxsize=None)
def _recipe(forward_dtype, backward_dtype):
    """The recipe of the native host path (csrc/host.cpp), which runs forward and backward."""
    forward, backward = _FORMATS[forward_dtype], _FORMATS[backward_dtype]
    return _lib.host().Recipe({"grouped": True, "native": False, "fp8_weight": True, "cache_transpose": False,
                               "fwd": _lib.code(forward), "bwd": _lib.code(backward), "fwd_limit": torch.finfo(forward).max,
                               "bwd_limit": torch.finfo(backward).max, "in": 0, "out": 0})


def _offsets(counts, device):
    """Row offsets of the groups and offsets on the padded token axis (whole tiles of 32 per group, 128 in all), on the host and
    as the native host path puts them on the device."""
    counts = [int(c) for c in (counts.tolist() if isinstance(counts, torch.Tensor) else counts)]
    table = _lib.host().segment_offsets(counts, torch.device(device)).view(torch.int64)[:2 * (len(counts) + 1)].view(2, -1)
    offsets, padded = table.tolist()
    return offsets, padded, table[0], table[1]


def quantize_transposed_segmented(x, dtype, offsets_dev, padded_dev, groups, t_total, *, rowwise=False):
    """Per-group quantized transpose of x [M, C]: codes [C, t_total], scales [C, t_total/32]. With rowwise, also the
    plain (1, 32) row-wise codes and scales of x, from the same read where the kernel takes the shape: returns (qt, st, q, s).
    The quantizer of the native host path's forward and backward, as an operator."""
    name = {fp8: key for key, fp8 in _FORMATS.items()}[dtype]
    return tuple(_lib.host().quantize_segments(x, _recipe(name, name), offsets_dev, padded_dev, int(groups), int(t_total), bool(rowwise)))


def grouped_linear(x, weight, weight_scale, counts, *, forward_dtype="e4m3", backward_dtype="e4m3", grad_dtype=None):
    """y[rows of group g] = x[rows of group g] @ dequant(weight[g]).T for every group, one launch.

    weight [G, N, K] FP8 codes, weight_scale [G, ceil(N/32), ceil(K/32)] fp32, counts: rows per group
    (host list or CPU tensor, sum == x.shape[0])."""
    assert x.is_cuda and x.dim() == 2
    grad_dtype = grad_dtype or weight.grad_dtype or torch.float32
    counts = counts.tolist() if isinstance(counts, torch.Tensor) else counts
    return _lib.host().experts(x, weight, weight_scale, [int(c) for c in counts], _recipe(forward_dtype, backward_dtype), grad_dtype)


class GroupedExperts(nn.Module):
    """`groups` expert weight matrices [out, in] stored as FP8 codes with (32, 32) block scales."""

    def __init__(self, groups, in_features, out_features, *, forward_dtype="e4m3", backward_dtype="e4m3",
                 device=None, dtype=None):
        super().__init__()
        self.groups, self.in_features, self.out_features = groups, in_features, out_features
        self.forward_dtype, self.backward_dtype = forward_dtype, backward_dtype
        policy = settings()
        shape = (groups, out_features, in_features)
        self._initial_weight = torch.empty(shape, device=device, dtype=policy["master_weight_dtype"] or torch.float32)
        self.weight = nn.Parameter(torch.empty(shape, device=device, dtype=_FORMATS[forward_dtype]))
        self.weight.grad_dtype = policy["gradient_dtype"] or torch.float32
        self.register_buffer("weight_scale", torch.ones((groups, *kernels.scale_shape(shape[1:], GW)), device=device,
                                                        dtype=torch.float32))
        self.reset_parameters()

    @torch.no_grad()
    def reset_parameters(self):
        for g in range(self.groups):
            nn.init.kaiming_uniform_(self._initial_weight[g], a=math.sqrt(5))
        self.refresh_weight(self._initial_weight)

    @torch.no_grad()
    def refresh_weight(self, master):
        assert master.is_cuda, "viola_amd kernels run on the GPU only: construct GroupedExperts on the GPU"
        for g in range(self.groups):
            kernels.quantize(master[g], self.weight.dtype, GW, out=self.weight[g], scale_out=self.weight_scale[g])

    def dequantize_weight(self):
        return torch.stack([kernels.dequantize(self.weight[g], self.weight_scale[g], GW) for g in range(self.groups)])

    def forward(self, x, counts):
        assert x.is_cuda, "viola_amd kernels run on the GPU only"
        return grouped_linear(x, self.weight, self.weight_scale, counts, forward_dtype=self.forward_dtype,
                              backward_dtype=self.backward_dtype, grad_dtype=self.weight.grad_dtype)
