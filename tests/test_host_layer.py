"""The native host layer of the eager public functions against the custom ops that traced code
takes: the same results bit for bit over the layouts and types it accepts, and the same refusals."""

import pytest
import torch

import dwarf_amd
from dwarf_amd import OFFSETS_V3, ops

B, H, N, D = 2, 3, 130, 32
gpu = pytest.mark.gpu


@pytest.mark.parametrize("offsets", [[], [1, 2], [0, 2, 2], [0, 5, 3]])
def test_refuses_bad_tables(offsets):
    q = torch.zeros(1, 1, 4, 32)
    with pytest.raises(AssertionError, match="strictly increasing"):
        dwarf_amd.dsqg_attention(q, q, q, torch.zeros(len(offsets), 1), offsets=offsets)


def test_refuses_cpu_tensors_and_bad_shapes():
    q, pb = torch.zeros(1, 2, 4, 32), torch.zeros(44, 2)
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        dwarf_amd.dsqg_attention(q, q, q, pb)
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        dwarf_amd.dsqg_attention_qkv(torch.zeros(1, 4, 192), 2, pb)
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        dwarf_amd.causal_mean_pool_gate(torch.zeros(1, 4, 8), torch.zeros(1, 4, 8))
    for bad in (dict(pos_bias=pb[:, :1]), dict(scale_embed=torch.zeros(44, 16)),
                dict(score_gain=torch.zeros(44, 2)), dict(if_gain=torch.zeros(1))):
        with pytest.raises(AssertionError, match="must be"):
            dwarf_amd.dsqg_attention(q, q, q, bad.pop("pos_bias", pb), offsets=OFFSETS_V3, **bad)
    with pytest.raises(AssertionError, match="same shape"):
        dwarf_amd.dsqg_attention(q, q[:, :1], q, pb)
    with pytest.raises(AssertionError, match="num_heads"):
        dwarf_amd.dsqg_attention_qkv(torch.zeros(1, 4, 190), 2, pb)


BAD_DECODE = [dict(pos_bias=(44, 1)), dict(pos_bias=(43, 2)), dict(scale_embed=(44, 16)), dict(scale_embed=(40, 32)),
              dict(score_gain=(44, 2)), dict(if_gain=(1,))]


@pytest.mark.parametrize("bad", BAD_DECODE, ids=lambda b: "-".join(map(str, *b.items())))
@pytest.mark.parametrize("path", ["eager", "into"])
def test_decode_refuses_short_parameters(bad, path):
    """The kernel indexes the parameters by the ring's head count and dim and the table's length."""
    row, ring = torch.zeros(1, 2, 32), torch.zeros(1, 2, 1537, 32)
    pos = torch.zeros(1, dtype=torch.int64)
    kw = {k: torch.zeros(*s) for k, s in bad.items()}
    pb = kw.pop("pos_bias", torch.zeros(44, 2))
    with pytest.raises(AssertionError, match="must be"):
        if path == "eager":
            dwarf_amd.dsqg_decode_step(row, row, row, ring, ring, pos, pb, offsets=OFFSETS_V3, **kw)
        else:
            ops.decode_step_into(row, row, row, ring, ring, pos, pb, kw.get("scale_embed"), kw.get("score_gain"),
                                 kw.get("if_gain"), list(OFFSETS_V3), torch.empty_like(row))


@gpu
@pytest.mark.parametrize("name,shape", [("scale_embed", (44, 32)), ("score_gain", (2, 44)), ("if_gain", (2,))])
@pytest.mark.parametrize("path", ["eager", "into"])
def test_decode_refuses_cpu_parameters(gpu_device, name, shape, path):
    row, ring = torch.zeros(1, 2, 32, device=gpu_device), torch.zeros(1, 2, 1537, 32, device=gpu_device)
    pos, pb = torch.zeros(1, dtype=torch.int64, device=gpu_device), torch.zeros(44, 2, device=gpu_device)
    kw = {name: torch.zeros(*shape)}
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        if path == "eager":
            dwarf_amd.dsqg_decode_step(row, row, row, ring, ring, pos, pb, offsets=OFFSETS_V3, **kw)
        else:
            ops.decode_step_into(row, row, row, ring, ring, pos, pb, kw.get("scale_embed"), kw.get("score_gain"),
                                 kw.get("if_gain"), list(OFFSETS_V3), torch.empty_like(row))


def _inputs(dev, dtype, form):
    g = torch.Generator().manual_seed(3)
    qkv = torch.randn(B, N, 3 * H * D, generator=g).to(dev, dtype)
    if form == "strided":     # rows of a wider buffer
        qkv = torch.randn(B, N, 3 * H * D + 64, generator=g).to(dev, dtype)[..., :3 * H * D]
    elif form == "inner":     # no unit inner stride: copied
        qkv = torch.randn(B, 3 * H * D, N, generator=g).to(dev, dtype).transpose(1, 2)
    J = len(OFFSETS_V3)
    se = torch.randn(J * D + 1, generator=g).to(dev)[1:].view(J, D)  # 4-byte aligned: copied
    return (qkv, torch.randn(J, H, generator=g).to(dev), se, torch.rand(H, J, generator=g).to(dev) + 0.5,
            torch.rand(H, generator=g).to(dev) + 0.5,
            [torch.randn(B, N, H, D, generator=g).to(dev, torch.float32).permute(0, 2, 1, 3) for _ in range(2)])


def _grads(fn, leaves, dout):
    out = fn(*leaves)
    return [out.detach(), *torch.autograd.grad(out, leaves, dout(out))]


@gpu
@pytest.mark.parametrize("form", ["plain", "strided", "inner"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_equals_the_custom_ops(gpu_device, dtype, form):
    qkv, pb, se, sg, ig, deltas = _inputs(gpu_device, dtype, form)
    work = dtype if dtype != torch.float16 else torch.bfloat16
    douts = (lambda o: torch.ones((), device=o.device, dtype=o.dtype).expand(o.shape),
             lambda o: torch.linspace(-1, 1, o.numel(), device=o.device).to(o.dtype).view(o.shape))
    req = lambda ts: [t.detach().requires_grad_(True) for t in ts]
    for dout in douts:
        for inject in (None, deltas):
            leaves = req([qkv, pb, se, sg, ig, *(inject or ())])
            got = _grads(lambda x, p, s, g, a, *kv: dwarf_amd.dsqg_attention_qkv(
                x, H, p, s, offsets=list(OFFSETS_V3), score_gain=g, if_gain=a, kv_inject=kv or None), leaves, dout)
            fn = ops.dsqg_fwd_qkv_kv if inject else ops.dsqg_fwd_qkv
            ref = _grads(lambda x, p, s, g, a, *kv: fn(
                x.to(work), *kv, H, p, s, g, a, list(OFFSETS_V3))[0].to(x.dtype), req(leaves), dout)
            assert len(got) == len(ref)
            for a, b in zip(got, ref):
                assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
        heads = req(ops.split_qkv(qkv, H))
        leaves = [*heads, *req([pb, se])]
        got = _grads(dwarf_amd.dsqg_attention_v3, leaves, dout)
        ref = _grads(lambda q, k, v, p, s: ops.dsqg_fwd(q.to(work), k.to(work), v.to(work), p, s, None, None,
                                                        list(OFFSETS_V3))[0].to(q.dtype), leaves, dout)
        for a, b in zip(got, ref):
            assert torch.equal(a, b) and a.stride() == b.stride()


@gpu
def test_autograd_contract(gpu_device):
    qkv, pb, se, sg, ig, _ = _inputs(gpu_device, torch.bfloat16, "plain")
    q, k, v = (t.contiguous().requires_grad_(True) for t in ops.split_qkv(qkv, H))
    pb.requires_grad_(True)
    out = dwarf_amd.dsqg_attention(q, k, v, pb)
    ref = torch.autograd.grad(out.float().sum(), (q, pb), retain_graph=True)
    # Saved tensors go through the hooks, and only what is asked for comes back.
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(gpu_device)):
        out2 = dwarf_amd.dsqg_attention(q, k, v, pb)
    for a, b in zip(torch.autograd.grad(out2.float().sum(), (q, pb)), ref):
        assert torch.equal(a, b)
    with torch.no_grad():
        assert not dwarf_amd.dsqg_attention(q, k, v, pb).requires_grad
        k += 1  # a saved input changed in place
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.float().sum().backward()
    with pytest.raises(Exception):
        with torch.autograd.forward_ad.dual_level():
            dwarf_amd.dsqg_attention(torch.autograd.forward_ad.make_dual(q.detach(), q.detach()), k, v, pb)
    with pytest.raises(Exception):
        torch.vmap(lambda t: dwarf_amd.dsqg_attention(t, t, t, pb.detach()))(q.detach().unsqueeze(0))


@gpu
def test_decode_marks_the_rings_changed(gpu_device):
    rows = [torch.randn(B, H, D, device=gpu_device).bfloat16() for _ in range(3)]
    rings = [torch.randn(B, H, 1537, D, device=gpu_device).bfloat16() for _ in range(2)]
    pos = torch.tensor([3, 2000], device=gpu_device)
    pb = torch.randn(44, H, device=gpu_device)
    ref_rings = [r.clone() for r in rings]
    ref = ops.dsqg_decode(*rows, *ref_rings, pos, pb, None, None, None, list(OFFSETS_V3))
    before = [r._version for r in rings]
    out = dwarf_amd.dsqg_decode_step(*rows, *rings, pos, pb)
    assert torch.equal(out, ref) and all(torch.equal(a, b) for a, b in zip(rings, ref_rings))
    assert all(r._version > v for r, v in zip(rings, before))
    # A gradient is still refused, by the op.
    with pytest.raises(RuntimeError):
        dwarf_amd.dsqg_decode_step(rows[0].requires_grad_(True), *rows[1:], *rings, pos, pb).float().sum().backward()


@gpu
def test_decode_of_lazily_negated_operands(gpu_device):
    rows = [torch.randn(B, H, D, device=gpu_device).bfloat16() for _ in range(3)]
    pos, pb = torch.tensor([3, 2000], device=gpu_device), torch.randn(44, H, device=gpu_device)
    rings = torch.randn(2, B, H, 1537, D, device=gpu_device).bfloat16()
    res = []
    for args in ([torch._neg_view(t) for t in (*rows, pb)], [-t for t in (*rows, pb)]):
        kr, vr = rings.clone()
        res.append((dwarf_amd.dsqg_decode_step(*args[:3], kr, vr, pos, args[3]), kr, vr))
    assert all(torch.equal(a, b) for a, b in zip(*res))


class _NoGrad(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@gpu
@pytest.mark.parametrize("call", ["separate", "qkv", "inject"])
def test_absent_output_gradient_is_zero(gpu_device, call):
    """A consumer that returns no gradient: the operands' gradients are zeros, not an error."""
    qkv, pb, se, sg, ig, deltas = _inputs(gpu_device, torch.float32, "plain")
    if call == "separate":
        leaves = [t.contiguous().requires_grad_() for t in qkv.view(B, N, 3, H, D).permute(2, 0, 3, 1, 4)]
        out = dwarf_amd.dsqg_attention(*leaves, pb, se, score_gain=sg, if_gain=ig)
    else:
        leaves = [qkv.requires_grad_(), *(d.requires_grad_() for d in deltas if call == "inject")]
        out = dwarf_amd.dsqg_attention_qkv(qkv, H, pb, se, score_gain=sg, if_gain=ig,
                                           kv_inject=tuple(deltas) if call == "inject" else None)
    for g in torch.autograd.grad(_NoGrad.apply(out).sum(), leaves, allow_unused=True):
        assert g is None or not g.any()
