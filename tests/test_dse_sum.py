"""The reduction of dscale_embed's partials alone (dsqg_bwd_params): its float32 rounding against a
64-bit sum, over partial counts around its groups and deep ones.

A rounding is uniform within half an ulp, at most 2^-24 / sqrt(3) of the value (rms), and the errors of
L additions, each of sums that make up the whole, add as squares: rms error <= 2^-24 sqrt(L / 3) of the
result's.  L: 3 levels of eight rows, half a step each of the chains of 16 eights and of those chains
(a chain's early sums are small), 5 levels over 32 row lanes; 1.2 for the spread of 2816 elements.
"""

import ctypes
import math

import pytest
import torch

from dwarf_amd import _lib
from dwarf_amd.offsets import OFFSETS_V3

J, D = 44, 64


def _size(lib, a):
    n = ctypes.c_size_t(0)
    _lib.check(lib.dsqg_bwd_workspace_size(ctypes.byref(a), ctypes.byref(n)), "size")
    return n.value


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,rows", [(1, 1, 1, 1), (1, 1, 31 * 64, 31), (3, 11, 64, 33), (1, 3, 64 * 85 + 1, 258),
                                        (2, 8, 2047, 512), (8, 12, 2048, 3072), (5, 16, 64 * 50, 4000),
                                        (4, 16, 16384, 16384)])
def test_rounding_of_deep_sums(gpu_device, B, H, N, rows):
    lib = _lib.load()
    t = torch.zeros(B, H, N, D, device=gpu_device)  # float32: one partial per 64-row tile
    small = torch.zeros(J * max(H, D), device=gpu_device)
    dse = torch.full((J, D), float("nan"), device=gpu_device)
    a = _lib.BwdArgs()
    a.shape = _lib.make_shape(_lib.DSQG_F32, B, H, N, D, OFFSETS_V3)
    st = (ctypes.c_int64 * 4)(*t.stride())
    for name in ("q", "k", "v", "dout", "dq", "dk", "dv"):
        setattr(a, name, t.data_ptr())
        setattr(a, name + "_stride", st)
    a.lse = t.data_ptr()
    a.pos_bias = a.scale_embed = a.dpos_bias = small.data_ptr()
    base = _size(lib, a)
    a.dscale_embed = dse.data_ptr()
    total = _size(lib, a)
    assert total - base == rows * J * D * 4  # the last region of the workspace
    ws = torch.zeros(total, dtype=torch.uint8, device=gpu_device)
    part = ws[base:].view(torch.float32).view(rows, J * D)
    part.normal_(generator=torch.Generator(device=gpu_device).manual_seed(rows))
    a.workspace, a.workspace_bytes = ws.data_ptr(), total
    stream = torch.cuda.current_stream(gpu_device).cuda_stream
    _lib.check(lib.dsqg_bwd_params(ctypes.byref(a), stream), "dsqg_bwd_params")
    ref = part.double().sum(0)
    err = (dse.view(-1).double() - ref).square().mean().sqrt() / ref.square().mean().sqrt()
    eights = math.ceil(rows / 256)
    L = 3 + min(eights, 16) / 2 + eights / 16 / 2 + 5 if rows > 1 else 0
    assert err <= 1.2 * 2.0 ** -24 * math.sqrt(L / 3), f"{rows} partials: {err:.3e}"
