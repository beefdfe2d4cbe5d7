"""float32 MFMA kernels against the oracle at tile edges and tables of every shape, and against
the VALU kernels (the general float32 path) on inputs with infinities and NaN.

The bound against the float64 oracle is the repository's float32 one (tests/tolerance.py:
max|x - ref| <= 1e-5 max|ref|).  The two float32 paths each sum the same products in a different
order; with at most 48 taps of D <= 128 products a sum's rounding is below (48 + 128) 2^-24 of its
terms' magnitude, 1.1e-5, so finite values are compared at 2e-5 of the tensor's scale.
"""

import pytest
import torch

from dwarf_amd import ops
from dwarf_amd.offsets import OFFSETS_J46, OFFSETS_J47, OFFSETS_V3
from tests.test_parity_gpu import _rand_inputs, compare, gpu_run, oracle_chunked

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 80, 96, 128])
@pytest.mark.parametrize("N", [1, 15, 16, 17, 33, 63, 64, 65, 129])
def test_tile_edges(gpu_device, D, N):
    inp = _rand_inputs(2, 3, N, D, OFFSETS_V3, torch.float32, seed=1000 * D + N)
    compare(gpu_run(inp, OFFSETS_V3, gpu_device), oracle_chunked(inp, OFFSETS_V3, torch.float64), "fp32")


@pytest.mark.parametrize("D,se,gains", [(32, True, False), (64, False, True), (80, True, True),
                                        (96, False, False), (128, True, True)])
@pytest.mark.parametrize("offsets", [
    (0,), tuple(range(33)), tuple(range(48)), (0,) + tuple(range(2, 96, 2)), (0, 1, 2, 40, 700),
    OFFSETS_J46, OFFSETS_J47], ids=["one", "window", "15_past", "47_long", "short", "j46", "j47"])
def test_tables(gpu_device, D, se, gains, offsets):
    inp = _rand_inputs(1, 2, 777, D, offsets, torch.float32, seed=D + len(offsets), se=se, gains=gains)
    compare(gpu_run(inp, offsets, gpu_device), oracle_chunked(inp, offsets, torch.float64), "fp32")


def _wide(t, rs):
    """t [1,H,N,D] as a view whose rows are rs floats apart."""
    _, H, N, D = t.shape
    v = torch.empty(N * rs, device=t.device).as_strided(t.shape, (N * rs, D, rs, 1))
    return v.copy_(t)


def _both_paths(inp, offsets, dev):
    d = {k: (None if v is None else v.to(dev)) for k, v in inp.items()}
    N = d["q"].shape[2]
    # Rows so far apart that 32-bit byte offsets do not reach every tap: the VALU kernels' case.
    rs = (-(-(1 << 29) // (N + max(offsets) + 64)) + 3) // 4 * 4
    params = (d["pos_bias"], d["scale_embed"], d["score_gain"], d["if_gain"], list(offsets))
    res = []
    for wide in (False, True):
        q, k, v, dout = (_wide(d[n], rs) if wide else d[n] for n in ("q", "k", "v", "dout"))
        out, lse, alr = ops.dsqg_fwd(q, k, v, *params)
        grads = ops.dsqg_bwd(q, k, v, dout, lse, alr, *params, d["scale_embed"] is not None,
                             d["score_gain"] is not None, d["if_gain"] is not None)
        names = ("dq", "dk", "dv", "dpos_bias", "dscale_embed", "dscore_gain", "dif_gain")
        res.append({"out": out, "lse": lse, **dict(zip(names, grads))})
    torch.cuda.synchronize(dev)
    return res


def _same(a, b, scale_tol=2e-5):
    for key in a:
        x, y = a[key].double().cpu(), b[key].double().cpu()
        assert torch.equal(torch.isnan(x), torch.isnan(y)), f"{key}: NaN in other places"
        assert torch.equal(x.isinf(), y.isinf()) and torch.equal(x[x.isinf()], y[y.isinf()]), key
        fin = torch.isfinite(x)
        if fin.any():
            scale = y[fin].abs().max().item()
            assert (x[fin] - y[fin]).abs().max().item() <= scale_tol * scale, key


@pytest.mark.parametrize("D,se,gains", [(32, True, True), (64, False, False), (80, False, True),
                                        (96, True, True), (128, True, False)])
def test_against_the_general_path(gpu_device, D, se, gains):
    inp = _rand_inputs(1, 2, 130, D, OFFSETS_V3, torch.float32, seed=D, se=se, gains=gains)
    _same(*_both_paths(inp, OFFSETS_V3, gpu_device))


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("tensor", ["q", "k", "v", "dout"])
def test_nonfinite_rows_reach_only_their_taps(gpu_device, tensor, value):
    offsets = (0, 1, 2, 3, 4, 5, 20, 50)
    inp = _rand_inputs(1, 2, 130, 64, offsets, torch.float32, seed=5, gains=False)
    inp[tensor][0, 0, 40, 7] = value
    fast, general = _both_paths(inp, offsets, gpu_device)
    _same(fast, general)
    # Head 1 has none, and no query before row 40 attends it.
    for key in ("out", "dq"):
        assert torch.isfinite(fast[key][0, 1]).all() and torch.isfinite(fast[key][0, 0, :40]).all(), key


def test_nonfinite_parameters(gpu_device):
    # scale_embed infinite at one tap; a bias at the type's lowest value and one at -inf.
    offsets = (0, 1, 2, 3, 4, 5, 20, 50)
    inp = _rand_inputs(1, 2, 130, 64, offsets, torch.float32, seed=6, gains=False)
    inp["scale_embed"][6, 3] = float("inf")
    inp["pos_bias"][3, 0] = torch.finfo(torch.float32).min
    inp["pos_bias"][2, 1] = float("-inf")
    _same(*_both_paths(inp, offsets, gpu_device))
