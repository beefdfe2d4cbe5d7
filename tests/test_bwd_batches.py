"""Batches per workgroup of the bf16 scale_embed dq: grids whose plan takes one, two or four
batches with a short last group, and the allocation-free entry's compact plan."""

import ctypes

import pytest
import torch

from dwarf_amd import _lib
from dwarf_amd.offsets import OFFSETS_J47, OFFSETS_V3
from tests.test_parity_gpu import _rand_inputs, compare, gpu_run, oracle_chunked


GENERIC = tuple(range(20)) + (48, 64, 96, 128)  # four long-range taps: the generic-table kernel


def planned_batches(B, H, N, D, offsets, gain):
    """Batches per workgroup of the plan, from the size of dscale_embed's partials ([J x D] floats per
    workgroup: one per batch group, head and 64-row tile)."""
    lib = _lib.load()
    a = _lib.BwdArgs()
    a.shape = _lib.make_shape(_lib.DSQG_BF16, B, H, N, D, offsets)
    for name in ("q", "k", "v", "dout", "dq", "dk", "dv"):
        setattr(a, name, 0x10000)  # (nothing is launched)
        setattr(a, name + "_stride", (_lib._i64x4)(H * N * D, N * D, D, 1))
    a.lse = a.alpha_lr = a.pos_bias = a.dpos_bias = a.scale_embed = 0x10000
    if gain:
        a.score_gain = a.dscore_gain = 0x10000
    sizes = []
    for dse in (None, 0x10000):
        a.dscale_embed = dse
        n = ctypes.c_size_t(0)
        assert lib.dsqg_bwd_workspace_size(ctypes.byref(a), ctypes.byref(n)) == _lib.DSQG_OK
        sizes.append(n.value)
    groups = (sizes[1] - sizes[0]) // (4 * len(offsets) * D) // (H * ((N + 63) // 64))
    return next(b for b in (1, 2, 3, 4) if (B + b - 1) // b == groups)


@pytest.mark.parametrize("B,H,N,D,offsets,plain,gain", [
    # A CU holds four / three workgroups (without / with the score gain's gradient), then three / two,
    # two for a generic table, two / one, two: the same grid fills it to different rounds.
    (16, 8, 2048, 32, OFFSETS_V3, 4, 2), (8, 12, 2048, 64, OFFSETS_V3, 4, 2), (2, 12, 2048, 64, OFFSETS_J47, 1, 2),
    (2, 12, 2048, 64, GENERIC, 2, 2), (4, 8, 2047, 80, OFFSETS_V3, 2, 4), (4, 8, 2048, 128, OFFSETS_V3, 2, 2)])
def test_plan_follows_the_workgroups_a_cu_holds(B, H, N, D, offsets, plain, gain):
    assert planned_batches(B, H, N, D, offsets, False) == plain
    assert planned_batches(B, H, N, D, offsets, True) == gain


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D,offsets,batches", [
    (3, 2, 200, 64, OFFSETS_V3, 1),      # a handful of tiles
    (5, 16, 2048, 64, OFFSETS_V3, 2),    # the last group of one
    (7, 12, 2048, 64, OFFSETS_V3, 4),    # the last group of three
    (3, 8, 2048, 80, OFFSETS_J47, 2),    # two workgroups per CU, the last group of one
    (5, 8, 1500, 128, OFFSETS_V3, 1),    # rows of a partial tile
    (9, 3, 1200, 128, OFFSETS_V3, 2),    # the restaged D = 128 form over a group, the last of one
    (7, 6, 1850, 128, OFFSETS_J47, 4),   # ... the last of three
])
def test_batch_plans(gpu_device, B, H, N, D, offsets, batches):
    assert planned_batches(B, H, N, D, offsets, False) == batches
    inp = _rand_inputs(B, H, N, D, offsets, torch.bfloat16, seed=B * N + D, gains=False)
    compare(gpu_run(inp, offsets, gpu_device), oracle_chunked(inp, offsets, torch.float32), "bf16",
            case=f"B{B} H{H} N{N} D{D} J{len(offsets)} batch plan")


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,D,offsets,batches", [
    (7, 2, 3500, 32, OFFSETS_V3, 2), (7, 6, 2741, 32, OFFSETS_J47, 4), (9, 3, 1200, 64, OFFSETS_J47, 2),
    (7, 6, 1850, 64, OFFSETS_V3, 4), (9, 3, 1200, 64, GENERIC, 2), (5, 2, 1650, 80, OFFSETS_J47, 2),
    (7, 8, 700, 96, OFFSETS_V3, 4), (9, 3, 1200, 128, OFFSETS_V3, 2), (7, 6, 1850, 128, OFFSETS_J47, 4)])
def test_batch_plans_with_the_gain_gradient(gpu_device, B, H, N, D, offsets, batches):
    """The score gain's gradient over a group of batches (its table and sums carried across them), the
    last group short."""
    assert planned_batches(B, H, N, D, offsets, True) == batches and B % batches
    inp = _rand_inputs(B, H, N, D, offsets, torch.bfloat16, seed=B * N + D)
    compare(gpu_run(inp, offsets, gpu_device), oracle_chunked(inp, offsets, torch.float32), "bf16",
            case=f"B{B} H{H} N{N} D{D} J{len(offsets)} batch plan + g, a")


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
