"""Weight and bias gradients of the linear layers: the kernel against float64 at the edges of its
tiles and row splits, and the layer against nn.Linear through autograd and autocast.

A sum of T products rounded once to the output type is within half an ulp (2^-11 of the value in
float16, 2^-8 in bfloat16, 2^-24 in float32) plus the float32 sum's rounding, below T 2^-24 of its terms' magnitude.
"""

import ctypes

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from dwarf_amd import _lib
from dwarf_amd.modules import FFN, Linear

HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def _close(got, dy, x, name):
    dy, x = dy.double(), x.double()
    ref, mag = (dy.sum(0), dy.abs().sum(0)) if x.numel() == 0 else (dy.t() @ x, dy.abs().t() @ x.abs())
    bound = HALF_ULP[got.dtype] * ref.abs() + len(dy) * 2.0 ** -24 * mag + 2.0 ** -25
    assert ((got.double() - ref).abs() <= bound).all(), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,O,I,pad", [
    (1, 8, 8, 0), (63, 8, 136, 8), (64, 128, 128, 0), (65, 136, 120, 0), (256, 256, 128, 24),
    (257, 128, 264, 0), (1000, 264, 520, 0), (8191, 256, 256, 0), (70001, 8, 8, 0)])
def test_kernel_against_float64(gpu_device, T, O, I, pad, dtype):
    _run_kernel(gpu_device, T, O, I, pad, dtype, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 200, 256, 257])  # one split, straight to the results; two
def test_float32_results_against_float64(gpu_device, T, dtype):
    _run_kernel(gpu_device, T, 136, 264, 8, dtype, torch.float32)


def _run_kernel(gpu_device, T, O, I, pad, dtype, out):
    code = {torch.float16: _lib.DSQG_F16, torch.bfloat16: _lib.DSQG_BF16, torch.float32: _lib.DSQG_F32}
    g = torch.Generator().manual_seed(T + O + I)
    dy = torch.randn(T, O + pad, generator=g).to(gpu_device, dtype)[:, :O]
    x = torch.randn(T, I + pad, generator=g).to(gpu_device, dtype)[:, :I]
    a = _lib.LinearWgradArgs()
    a.T, a.O, a.I = T, O, I
    a.dtype, a.out_dtype = code[dtype], code[out]
    a.dy, a.dy_stride, a.x, a.x_stride = dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0)
    dw = torch.full((O, I), float("nan"), device=gpu_device, dtype=out)
    db = torch.full((O,), float("nan"), device=gpu_device, dtype=out)
    a.dw, a.db = dw.data_ptr(), db.data_ptr()
    n = ctypes.c_size_t(0)
    lib = _lib.load()
    _lib.check(lib.dsqg_linear_wgrad_workspace_size(ctypes.byref(a), ctypes.byref(n)), "size")
    ws = torch.empty(n.value, dtype=torch.uint8, device=gpu_device)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n.value
    stream = torch.cuda.current_stream(gpu_device).cuda_stream
    _lib.check(lib.dsqg_linear_wgrad(ctypes.byref(a), stream), "dsqg_linear_wgrad")
    torch.cuda.synchronize(gpu_device)
    _close(dw, dy, x, "dw")
    _close(db, dy, x[:, :0], "db")


def test_arguments_are_checked_on_the_host():
    lib = _lib.load()
    n = ctypes.c_size_t(0)
    a = _lib.LinearWgradArgs()
    a.T, a.O, a.I, a.dtype, a.out_dtype = 64, 16, 24, _lib.DSQG_BF16, _lib.DSQG_BF16
    assert lib.dsqg_linear_wgrad_workspace_size(ctypes.byref(a), ctypes.byref(n)) == _lib.DSQG_OK
    assert lib.dsqg_linear_wgrad(ctypes.byref(a), None) == _lib.DSQG_EINVAL  # no tensors
    a.dy = a.x = a.dw = a.db = 0x10000
    a.dy_stride, a.x_stride = 16, 24
    assert lib.dsqg_linear_wgrad(ctypes.byref(a), None) == _lib.DSQG_EWORKSPACE
    for field, value in (("O", 12), ("I", 0), ("T", -1), ("dtype", _lib.DSQG_F32), ("out_dtype", _lib.DSQG_F16), ("dy_stride", 8),
                         ("x_stride", 28), ("x", 0x10008)):
        b = _lib.LinearWgradArgs.from_buffer_copy(a)
        setattr(b, field, value)
        assert lib.dsqg_linear_wgrad(ctypes.byref(b), None) == _lib.DSQG_EINVAL, field


def _pair(dev, I, O, bias, dtype):
    torch.manual_seed(1)
    a, b = nn.Linear(I, O, bias=bias), Linear(I, O, bias=bias)
    b.load_state_dict(a.state_dict(), strict=True)
    return a.to(dev, dtype), b.to(dev, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["bf16", "f16", "autocast", "autocast_bf16", "f32"])
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("layout", ["plain", "permuted"])
def test_layer_equals_nn_linear(gpu_device, mode, bias, layout):
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16}.get(mode, torch.float32)
    low = {"autocast": torch.float16, "autocast_bf16": torch.bfloat16}.get(mode, dtype)
    ref, lin = _pair(gpu_device, 48, 72, bias, dtype)
    x = torch.randn(3, 100, 48, device=gpu_device).to(dtype)
    if layout == "permuted":
        x = x.permute(1, 0, 2)
    res = []
    for m in (ref, lin):
        xi = x.detach().requires_grad_(True)
        with torch.amp.autocast("cuda", dtype=low, enabled=mode.startswith("autocast")):
            y = m(xi)
        dy = torch.linspace(-1, 1, y.numel(), device=gpu_device).view(y.shape).to(y.dtype)
        res.append([y.detach(), *torch.autograd.grad(y, [xi, *m.parameters()], dy)])
    for i, (u, v) in enumerate(zip(*res)):
        assert u.dtype == v.dtype and u.shape == v.shape
        if i < 2 or mode == "f32":
            assert torch.equal(u, v)
    if mode != "f32":
        dy2, x2 = dy.reshape(-1, 72), x.to(low).reshape(-1, 48)
        _close(res[1][2], dy2, x2, "weight")  # (float32 under autocast: not rounded to 16 bits)
        if bias:
            _close(res[1][3], dy2, x2[:, :0], "bias")


@pytest.mark.gpu
def test_second_derivatives_under_autocast(gpu_device):
    ref, lin = _pair(gpu_device, 48, 72, True, torch.float32)
    x = torch.randn(64, 48, device=gpu_device)
    res = []
    for m in (ref, lin):
        xi = x.clone().requires_grad_(True)
        with torch.amp.autocast("cuda"):
            y = m(xi)
        (gw,) = torch.autograd.grad(y.float().square().sum(), m.weight, create_graph=True)
        res.append(torch.autograd.grad(gw.float().square().sum(), [xi, m.weight, m.bias]))
    for u, v in zip(*res):  # both round dy and dw to float16 on the way
        assert u.dtype == v.dtype and (u - v).norm() <= 2e-3 * u.norm()


@pytest.mark.gpu
def test_layer_keeps_nn_linears_contract(gpu_device):
    ref, lin = _pair(gpu_device, 48, 72, True, torch.bfloat16)
    x = torch.randn(64, 48, device=gpu_device).bfloat16().requires_grad_(True)
    seen = []
    h = lin.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    # Second derivatives: the gradients are themselves differentiable.
    (gw,) = torch.autograd.grad(lin(x).float().square().sum(), lin.weight, create_graph=True)
    (gx,) = torch.autograd.grad(gw.float().sum(), x)
    w = lin.weight.detach().float()
    xr = x.detach().float().requires_grad_(True)
    wr = w.clone().requires_grad_(True)
    (gwr,) = torch.autograd.grad(F.linear(xr, wr, lin.bias.detach().float()).square().sum(), wr, create_graph=True)
    (gxr,) = torch.autograd.grad(gwr.sum(), xr)
    assert (gx.float() - gxr).norm() <= 2e-2 * gxr.norm()
    h.remove()
    assert seen == [(64, 72)]
    lin.bias.requires_grad_(False)
    (g1,) = torch.autograd.grad(lin(x).float().sum(), lin.weight)
    lin.weight.requires_grad_(False)
    assert torch.autograd.grad(lin(x).float().sum(), x)[0].shape == x.shape and g1.shape == (72, 48)
    with torch.no_grad():
        assert not lin(x).requires_grad
    xb = x.detach().view(4, 16, 48)
    assert torch.equal(torch.vmap(lin)(xb), torch.vmap(ref)(xb))
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x))
        assert torch.autograd.forward_ad.unpack_dual(lin(d)).tangent is not None


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["autocast", "bf16"])
@pytest.mark.parametrize("x_grad", [True, False])
def test_weight_changed_before_the_backward(gpu_device, mode, x_grad):
    """nn.Linear saves what its backward reads: under autocast the cast weight, and no weight where x
    takes no gradient.  A parameter changed in place in between is accepted exactly where it is there."""
    pair = _pair(gpu_device, 48, 72, True, torch.float32 if mode == "autocast" else torch.bfloat16)
    x = torch.randn(64, 48, device=gpu_device).to(torch.float32 if mode == "autocast" else torch.bfloat16)
    res = []
    for m in pair:
        xi = x.clone().requires_grad_(x_grad)
        with torch.amp.autocast("cuda", enabled=mode == "autocast"):
            y = m(xi)
        with torch.no_grad():
            m.weight.add_(1.0)
        leaves = [*([xi] if x_grad else []), m.weight, m.bias]
        try:
            res.append(torch.autograd.grad(y, leaves, torch.linspace(-1, 1, y.numel(), device=gpu_device).view(y.shape).to(y.dtype)))
        except RuntimeError as e:
            res.append("modified by an inplace operation" in str(e))
    if mode == "bf16" and x_grad:
        assert res == [True, True]
        return
    for u, v in zip(*res):  # (dw and db: float32 sums, rounded to 16 bits by nn.Linear)
        assert u.dtype == v.dtype and (u - v).float().norm() <= 4e-3 * u.float().norm()
    if x_grad:
        assert torch.equal(res[0][0], res[1][0])


@pytest.mark.gpu
@pytest.mark.parametrize("leaf", [True, False])
def test_second_derivatives_after_a_weight_change(gpu_device, leaf):
    """Under autocast the graph of the gradients reads the weight as it was at the forward, also where
    it has a history of its own (weight normalisation)."""
    res = []
    for m in _pair(gpu_device, 48, 72, True, torch.float32):
        if not leaf:
            torch.nn.utils.parametrizations.weight_norm(m)
        x = torch.linspace(-1, 1, 64 * 48, device=gpu_device).view(64, 48).requires_grad_(True)
        with torch.amp.autocast("cuda"):
            y = m(x)
        params = list(m.parameters())
        if leaf:
            with torch.no_grad():
                m.weight.mul_(3.0)
        grads = torch.autograd.grad(y.float().square().mean(), [x, *params], create_graph=True)
        res.append(torch.autograd.grad(sum(g.square().sum() for g in grads), [x, *params]))
    for u, v in zip(*res):
        assert u.dtype == v.dtype and (u - v).norm() <= 2e-3 * u.norm()


@pytest.mark.gpu
def test_layer_without_outputs(gpu_device):
    for m in _pair(gpu_device, 48, 0, True, torch.bfloat16):
        x = torch.randn(64, 48, device=gpu_device).bfloat16().requires_grad_(True)
        y = m(x)
        y.sum().backward()
        assert y.shape == (64, 0) and m.weight.grad.shape == (0, 48) and not x.grad.any()


@pytest.mark.gpu
def test_lazily_negated_operands(gpu_device):
    ref, lin = _pair(gpu_device, 48, 72, True, torch.bfloat16)
    x = torch.randn(64, 48, device=gpu_device).bfloat16()
    dy = torch.randn(64, 72, device=gpu_device).bfloat16()
    for xi, g in ((torch._neg_view(x), dy), (x, torch._neg_view(dy))):
        res = [torch.autograd.grad(m(xi), m.weight, g)[0].float() for m in (ref, lin)]
        assert (res[0] - res[1]).norm() <= 4e-3 * res[0].norm()


@pytest.mark.parametrize("trace", [torch.jit.script, torch.fx.symbolic_trace, "export", "compile"],
                         ids=["script", "fx", "export", "compile"])
def test_layers_can_be_traced(trace):
    """What takes a model of nn.Linear layers takes these (here without a GPU)."""
    torch.manual_seed(0)
    ffn = FFN(32, 64).eval()
    x = torch.randn(3, 32)
    if trace == "export":
        run = torch.export.export(ffn, (x,)).module()
    elif trace == "compile":
        run = torch.compile(ffn, backend="eager", fullgraph=True)
    else:
        run = trace(ffn)
    assert torch.equal(run(x), ffn(x))
