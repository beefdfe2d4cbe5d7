"""Batches per workgroup of the bf16 scale_embed dq: grids whose plan takes one, two or four
batches with a short last group, and the allocation-free entry's compact plan."""

import ctypes

import pytest
import torch

from dwarf_amd import _lib
from dwarf_amd.offsets import OFFSETS_J47, OFFSETS_V3
from tests.test_parity_gpu import _rand_inputs, compare, gpu_run, oracle_chunked


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D,offsets", [
    (3, 2, 200, 64, OFFSETS_V3),      # a handful of tiles: one batch each
    (5, 16, 2048, 64, OFFSETS_V3),    # two batches, the last group of one
    (7, 12, 2048, 64, OFFSETS_V3),    # four, the last group of three
    (3, 8, 2048, 80, OFFSETS_J47),    # two workgroups per CU: two batches, the last group of one
    (5, 8, 1500, 128, OFFSETS_V3),    # two batches, the last group of one, rows of a partial tile
])
def test_batch_plans(gpu_device, B, H, N, D, offsets):
    inp = _rand_inputs(B, H, N, D, offsets, torch.bfloat16, seed=B * N + D, gains=False)
    compare(gpu_run(inp, offsets, gpu_device), oracle_chunked(inp, offsets, torch.float32), "bf16",
            case=f"B{B} H{H} N{N} D{D} J{len(offsets)} batch plan")


def test_noalloc_takes_the_compact_plan():
    """B4 H12 N10240 D64 with dscale_embed: the fastest plan's workspace exceeds the static
    scratch, the four-batch plan's does not, so the call passes the size check."""
    lib = _lib.load()
    a = _lib.BwdArgs()
    B, H, N, D = 4, 12, 10240, 64
    a.shape = _lib.make_shape(_lib.DSQG_BF16, B, H, N, D, OFFSETS_V3)
    st = (_lib._i64x4)(H * N * D, N * D, D, 1)
    for name in ("q", "k", "v", "dout", "dq", "dk", "dv"):
        setattr(a, name, 0x10000)
        setattr(a, name + "_stride", st)
    a.lse = a.alpha_lr = a.pos_bias = a.dpos_bias = a.dscale_embed = 0x10000
    need = ctypes.c_size_t(0)
    assert lib.dsqg_bwd_workspace_size(ctypes.byref(a), ctypes.byref(need)) == _lib.DSQG_OK
    assert need.value > _lib.NOALLOC_SCRATCH_BYTES
    if not torch.cuda.is_available():  # (these pointers must not reach a kernel)
        assert lib.dsqg_bwd_noalloc(ctypes.byref(a), None) == _lib.DSQG_EHIP
