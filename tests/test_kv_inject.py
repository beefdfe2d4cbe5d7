"""The K/V injection kernel, through dsqg_attention_qkv, against the casts and adds it replaces
(the custom ops' path): the same bits forward and backward, for every type and layout it takes and
for those left to the casts and adds."""

import ctypes

import pytest
import torch

import dwarf_amd
from dwarf_amd import OFFSETS_V3, _lib, ops

B, H, N = 2, 3, 70


def _deltas(dev, dtype, layout, D):
    if layout == "heads":      # [B,H,N,D] contiguous
        return [torch.randn(B, H, N, D, device=dev).to(dtype) for _ in range(2)]
    if layout == "expanded":   # one delta for all tokens
        return [torch.randn(B, H, 1, D, device=dev).to(dtype).expand(B, H, N, D) for _ in range(2)]
    if layout == "unaligned":
        return [torch.randn(B, H, N, D + 1, device=dev).to(dtype)[..., 1:] for _ in range(2)]
    return [torch.randn(B, N, H, D, device=dev).to(dtype).permute(0, 2, 1, 3) for _ in range(2)]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["tokens", "heads", "expanded", "unaligned"])
@pytest.mark.parametrize("dtype,delta", [(torch.float32,) * 2, (torch.bfloat16,) * 2, (torch.float16,) * 2,
                                         (torch.float16, torch.float32), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("D", [32, 80])
def test_equals_casts_and_adds(gpu_device, D, dtype, delta, layout):
    torch.manual_seed(D)
    qkv = torch.randn(B, N, 3 * H * D, device=gpu_device).to(dtype)
    kd, vd = _deltas(gpu_device, delta, layout, D)
    pb = torch.randn(len(OFFSETS_V3), H, device=gpu_device)
    work = dtype if dtype != torch.float16 else torch.bfloat16
    dout = torch.randn(B, H, N, D, device=gpu_device).to(dtype)
    res = []
    for native in (True, False):
        leaves = [t.detach().requires_grad_(True) for t in (qkv, kd, vd, pb)]
        x, a, b, p = leaves
        out = dwarf_amd.dsqg_attention_qkv(x, H, p, kv_inject=(a, b)) if native else \
            ops.dsqg_fwd_qkv_kv(x.to(work), a, b, H, p, None, None, None, list(OFFSETS_V3))[0].to(dtype)
        res.append([out.detach(), *torch.autograd.grad(out, leaves, dout)])
    for u, v in zip(*res):
        assert u.dtype == v.dtype and u.shape == v.shape and torch.equal(u, v)


@pytest.mark.gpu
def test_lazily_negated_deltas(gpu_device):
    torch.manual_seed(0)
    qkv = torch.randn(B, N, 3 * H * 32, device=gpu_device).bfloat16()
    kd, vd = _deltas(gpu_device, torch.bfloat16, "tokens", 32)
    pb = torch.randn(len(OFFSETS_V3), H, device=gpu_device)
    out = [dwarf_amd.dsqg_attention_qkv(qkv, H, pb, kv_inject=d)
           for d in ((torch._neg_view(kd), torch._neg_view(vd)), (-kd, -vd))]
    assert torch.equal(*out)


def test_arguments_are_checked_on_the_host():
    lib = _lib.load()
    a = _lib.KvInjectArgs()
    a.B, a.H, a.N, a.D = 1, 2, 5, 32
    a.qkv_dtype = a.delta_dtype = a.out_dtype = _lib.DSQG_BF16
    assert lib.dsqg_kv_inject(ctypes.byref(a), None) == _lib.DSQG_EINVAL  # no tensors
    for n in ("qkv", "k_delta", "v_delta", "k_out", "v_out"):
        setattr(a, n, 0x10000)
    a.qkv_stride = (ctypes.c_int64 * 2)(960, 192)
    a.out_stride = (ctypes.c_int64 * 2)(320, 64)
    for field, value in (("D", 12), ("N", -1), ("out_dtype", _lib.DSQG_F16), ("k_out", 0x10008), ("qkv_dtype", 9),
                         ("out_stride", (ctypes.c_int64 * 2)(320, 60)), ("v_delta_stride", (ctypes.c_int64 * 3)(0, 4, 8))):
        b = _lib.KvInjectArgs.from_buffer_copy(a)
        setattr(b, field, value)
        assert lib.dsqg_kv_inject(ctypes.byref(b), None) == _lib.DSQG_EINVAL, field
    a.delta_dtype = _lib.DSQG_F32
    assert lib.dsqg_kv_inject(ctypes.byref(a), None) == _lib.DSQG_EUNSUPPORTED
    a.B = 0
    assert lib.dsqg_kv_inject(ctypes.byref(a), None) == _lib.DSQG_OK
