"""DSQGRingCache.prefill: the ring-load kernel against indexed writes, over prompt lengths around
the ring's, every type and layout it takes in place, and those it leaves to the indexed writes."""

import ctypes

import pytest
import torch

from dwarf_amd import DSQGRingCache, _lib


def _reference(cache, k, v):
    N, S = k.shape[2], cache.S
    idx = torch.arange(max(0, N - S), N, device=k.device)
    kr, vr = cache.k_ring.clone(), cache.v_ring.clone()
    kr[:, :, idx % S] = k[:, :, idx].to(kr.dtype)
    vr[:, :, idx % S] = v[:, :, idx].to(vr.dtype)
    return kr, vr


def _kv(dev, dtype, layout, B, H, N, D):
    if layout == "qkv":        # head views of a projection output
        t = torch.randn(B, N, 3 * H * D, device=dev).to(dtype)
        return [u.view(B, N, H, D).permute(0, 2, 1, 3) for u in t.split(H * D, dim=-1)[1:]]
    if layout == "expanded":   # one sequence for the whole batch
        return [torch.randn(1, H, N, D, device=dev).to(dtype).expand(B, H, N, D) for _ in range(2)]
    if layout == "unaligned":  # rows 2 bytes (4) off: left to the indexed writes
        return [torch.randn(B, H, N, D + 1, device=dev).to(dtype)[..., 1:] for _ in range(2)]
    return [torch.randn(B, H, N, D, device=dev).to(dtype) for _ in range(2)]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["plain", "qkv", "expanded", "unaligned"])
@pytest.mark.parametrize("dtype,ring", [(torch.bfloat16,) * 2, (torch.float32,) * 2, (torch.float16,) * 2,
                                        (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("offsets,N", [((0, 1, 7), n) for n in (1, 7, 8, 9, 29)] + [((0, 1536), 2100)])
def test_prefill_equals_indexed_writes(gpu_device, offsets, N, dtype, ring, layout):
    B, H, D = 2, 3, 32
    cache = DSQGRingCache(B, H, D, offsets, dtype=ring, device=gpu_device)
    cache.k_ring.normal_()
    cache.v_ring.normal_()
    k, v = _kv(gpu_device, dtype, layout, B, H, N, D)
    kr, vr = _reference(cache, k, v)
    version = cache.k_ring._version
    cache.prefill(k, v)
    assert torch.equal(cache.k_ring, kr) and torch.equal(cache.v_ring, vr)
    assert cache.pos.tolist() == [N] * B and cache.k_ring._version > version


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("types", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
def test_rings_of_two_types(gpu_device, types, rows):
    """Each ring takes its rows in its own type: the kernel has one type for all four tensors, so
    this is left to the indexed writes."""
    B, H, D, N = 2, 3, 32, 29
    cache = DSQGRingCache(B, H, D, (0, 1, 7), device=gpu_device)
    cache.k_ring, cache.v_ring = (torch.randn(B, H, cache.S, D, device=gpu_device).to(t) for t in types)
    k, v = _kv(gpu_device, rows, "plain", B, H, N, D)
    kr, vr = _reference(cache, k, v)
    cache.prefill(k, v)
    assert torch.equal(cache.k_ring, kr) and torch.equal(cache.v_ring, vr)
    assert cache.pos.tolist() == [N] * B


@pytest.mark.gpu
def test_left_to_the_indexed_writes(gpu_device):
    """What the indexed writes refuse stays refused, and rows that are more than their stored values
    (lazy negation, tangents, vmap's wrappers) load as there."""
    B, H, D, N = 2, 3, 32, 5
    make = lambda: DSQGRingCache(B, H, D, (0, 1, 7), device=gpu_device)
    k, v = _kv(gpu_device, torch.bfloat16, "plain", B, H, N, D)
    for name in ("k_ring", "v_ring"):
        cache = make()
        getattr(cache, name).requires_grad_(True)
        with pytest.raises(RuntimeError, match="requires grad"):
            cache.prefill(k, v)
        with torch.no_grad():
            cache.prefill(k, v)
        assert torch.equal(cache.v_ring[:, :, :N], v)
    with torch.inference_mode():
        cache = make()
        cache.prefill(k, v)
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        cache.prefill(k, v)
    cache = make()
    cache.prefill(torch._neg_view(k), v)
    assert torch.equal(cache.k_ring[:, :, :N], -k)
    cache = make()
    with torch.autograd.forward_ad.dual_level():
        cache.prefill(torch.autograd.forward_ad.make_dual(k, 2 * k), v)
        tangent = torch.autograd.forward_ad.unpack_dual(cache.k_ring).tangent
        assert torch.equal(tangent[:, :, :N], 2 * k)

    def load(k_ring, v_ring, pos, k, v):
        cache = make()
        cache.k_ring, cache.v_ring, cache.pos = k_ring, v_ring, pos
        cache.prefill(k, v)
        return cache.k_ring, cache.pos

    c = make()
    rings, pos = torch.vmap(load)(*(t.unsqueeze(0).clone() for t in (c.k_ring, c.v_ring, c.pos, k, v)))
    assert torch.equal(rings[0][:, :, :N], k) and pos.tolist() == [[N] * B]


def test_arguments_are_checked_on_the_host():
    lib = _lib.load()
    a = _lib.RingLoadArgs()
    a.dtype, a.B, a.H, a.N, a.S, a.D = _lib.DSQG_BF16, 1, 2, 5, 8, 32
    assert lib.dsqg_ring_load(ctypes.byref(a), None) == _lib.DSQG_EINVAL  # no tensors
    a.k = a.v = a.k_ring = a.v_ring = a.pos = 0x10000
    a.k_stride = a.v_stride = (ctypes.c_int64 * 3)(320, 160, 32)
    for field, value in (("S", 0), ("D", 12), ("dtype", 7), ("N", -1), ("k", 0x10008), ("pos", None),
                         ("v_stride", (ctypes.c_int64 * 3)(320, 160, 36))):
        b = _lib.RingLoadArgs.from_buffer_copy(a)
        setattr(b, field, value)
        assert lib.dsqg_ring_load(ctypes.byref(b), None) == _lib.DSQG_EINVAL, field
    a.H = 70000
    assert lib.dsqg_ring_load(ctypes.byref(a), None) == _lib.DSQG_EUNSUPPORTED
    a.B = 0
    assert lib.dsqg_ring_load(ctypes.byref(a), None) == _lib.DSQG_OK
