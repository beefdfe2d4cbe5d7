"""Performance cases of the framework: what its users run, through its public entry points.

Three paths: DSQG attention (forward alone, or forward + backward as a training step runs it),
the ring-buffer decode step, and the interference pool; plus one whole DSQG block.  ``listed()``
are fixed cases, ``draw(rng)`` samples the ranges they stand for:

* attention, bf16 and fp32: B 1..8, H 1..16, N 17..4096 (any N), head dims 32/64/80/96/128, the
  44/46/47-offset tables, scale_embed / score gain / IF gain on or off, separate q, k, v or one
  projection output, with or without the K/V injection;
* prompt prefill: the forward without gradients plus the ring load, prompts of 17..4096 tokens;
* decode: batches of 1..256 sequences;
* pool: bf16 throughout, or the float32 input with a float16 gate that autocast gives.
"""

import math

import torch
import torch.nn.functional as F

import dwarf_amd
from dwarf_amd import DSQGBlock, DSQGRingCache, OFFSETS_J46, OFFSETS_J47, OFFSETS_V3

TABLES = {44: OFFSETS_V3, 46: OFFSETS_J46, 47: OFFSETS_J47}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DEV = "cuda"


def _attn(name, B, H, N, D, J=44, dtype="bf16", call="separate", se=False, gain=False, ifg=False,
          inject=False, grad=True):
    return dict(name=name, kind="attn", B=B, H=H, N=N, D=D, J=J, dtype=dtype, call=call, se=se,
                gain=gain, ifg=ifg, inject=inject, grad=grad)


def listed():
    return [
        # A chat-sized prompt into the 13M model's layer: a forward and the ring load, where
        # launches and host work are everything.
        dict(name="prefill_77", kind="prefill", B=1, H=8, N=77, D=32, J=44, dtype="bf16"),
        # One token of one sequence, the same model: the smallest call there is.
        dict(name="decode_1", kind="decode", B=1, H=8, D=32, J=44, S=1537, dtype="bf16", se=True),
        # Batched serving, the 85M model's layer.
        dict(name="decode_256", kind="decode", B=256, H=12, D=64, J=44, S=1537, dtype="bf16",
             se=False),
        # Training steps of the attention call.  A ragged length and the head dim of the V2
        # kernel's own self-test.
        _attn("train_ragged_d80", 4, 8, 2047, 80),
        # The 13M trainer's layer behind the interference pool: projection output, K/V injection.
        _attn("train_13m_inject", 8, 8, 2048, 32, call="qkv", se=True, ifg=True, inject=True),
        # The 85M-scale call that bench.py quotes.
        _attn("train_85m", 8, 12, 2048, 64),
        # The 85M trainer's module call: head dim 96, scale_embed and IF gain.
        _attn("train_85m_d96", 8, 8, 2048, 96, call="qkv", se=True, ifg=True),
        # Long context with both gains, 46 offsets.
        _attn("train_4096_gains", 4, 8, 4096, 64, J=46, gain=True, ifg=True),
        # Training in float32 (no autocast), a ragged length.
        _attn("train_f32", 2, 8, 2047, 64, dtype="f32", se=True),
        # The interference pool of the 85M model in bf16, forward + backward.
        dict(name="pool_bf16", kind="pool", B=8, N=2048, C=768, x="bf16", g="bf16"),
        # ... and as the 13M trainer's autocast runs it: float32 input, float16 gate.
        dict(name="pool_autocast", kind="pool", B=8, N=2048, C=256, x="f32", g="f16"),
        # One whole interference block of the 13M model under autocast, forward + backward.
        dict(name="block_13m", kind="block", B=8, N=2048, E=256, H=8, F=1024),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "train_f32", "fwd", "prefill", "decode", "pool"])
    dtype = "f32" if kind == "train_f32" else "bf16"
    if kind in ("train", "train_f32", "fwd"):
        J = rng.choice([44, 44, 46, 47])
        call = rng.choice(["separate", "qkv"])
        while True:
            B, H, N, D = rng.randint(1, 8), rng.randint(1, 16), _log_int(rng, 17, 4096), \
                rng.choice([32, 64, 80, 96, 128])
            # No more rows than the largest listed case; float32 costs several times a bf16 row.
            if B * H * N * D <= (8 * 12 * 2048 * 64 if dtype == "bf16" else 2 * 8 * 2047 * 64):
                break
        return dict(kind="attn", B=B, H=H, N=N, D=D, J=J, dtype=dtype, call=call,
                    se=rng.random() < 0.5, gain=rng.random() < 0.25, ifg=rng.random() < 0.5,
                    inject=call == "qkv" and rng.random() < 0.3, grad=kind != "fwd")
    if kind == "prefill":
        return dict(kind="prefill", B=rng.randint(1, 4), H=rng.choice([4, 8, 12]),
                    N=_log_int(rng, 17, 4096), D=rng.choice([32, 64, 96]), J=44, dtype="bf16")
    if kind == "decode":
        return dict(kind="decode", B=_log_int(rng, 1, 256), H=rng.randint(1, 12),
                    D=rng.choice([32, 64]), J=44, S=1537, dtype="bf16", se=rng.random() < 0.5)
    x, g = rng.choice([("bf16", "bf16"), ("f32", "f16")])
    return dict(kind="pool", B=rng.randint(1, 8), N=_log_int(rng, 17, 2048),
                C=8 * rng.randint(8, 96 if x == "bf16" else 32), x=x, g=g)


# ---- Inputs ----------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


def _params(c, g):
    """pos_bias [J,H], scale_embed [J,D], score_gain [H,J], if_gain [H] near what training has:
    the log-linear bias of the modules' initialisation plus noise, small scale_embed, gains
    around one.  Absent ones are None."""
    J, H, D = c["J"], c["H"], c["D"]
    delta = torch.tensor(TABLES[J], dtype=torch.float32, device=DEV)
    pb = -torch.log1p(delta)[:, None] * torch.linspace(0.2, 2.0, H, device=DEV)[None, :]
    pb = pb + _randn(g, J, H, scale=0.1)
    se = _randn(g, J, D, scale=0.05) if c.get("se") else None
    sg = torch.rand((H, J), generator=g, device=DEV) + 0.5 if c.get("gain") else None
    ig = torch.rand((H,), generator=g, device=DEV) * 0.4 + 0.8 if c.get("ifg") else None
    return pb, se, sg, ig


def _block(c):
    torch.manual_seed(11)
    m = DSQGBlock(c["E"], c["H"], c["F"], seq_len=c["N"], dropout=0.0, interference=True)
    return m.to(DEV)


def prepare(case, seed):
    c = case
    g = _gen(seed)
    if c["kind"] == "attn":
        B, H, N, D, dt = c["B"], c["H"], c["N"], c["D"], DTYPES[c["dtype"]]
        st = {"case": c, "offsets": TABLES[c["J"]]}
        if c["call"] == "qkv":
            st["qkv"] = _randn(g, B, N, 3 * H * D, dtype=dt)
        else:
            for k in ("q", "k", "v"):
                st[k] = _randn(g, B, H, N, D, dtype=dt)
        if c["inject"]:  # views of the two projections' outputs, as the block makes them
            for k in ("kd", "vd"):
                st[k] = _randn(g, B, N, H, D, dtype=dt, scale=0.3).permute(0, 2, 1, 3)
        for k, t in zip(("pb", "se", "sg", "ig"), _params(c, g)):
            st[k] = t
        if c["grad"]:
            # The head merge's gradient: token-major, as the modules' backward hands it over.
            st["dout"] = _randn(g, B, N, H, D, dtype=dt).permute(0, 2, 1, 3)
            for k in _leaves(c):
                st[k].requires_grad_(True)
        return st
    if c["kind"] == "prefill":
        pb, se, _, ig = _params(dict(c, se=True, ifg=True), g)
        return {"case": c, "offsets": TABLES[c["J"]], "pb": pb, "se": se, "ig": ig,
                "qkv": _randn(g, c["B"], c["N"], 3 * c["H"] * c["D"], dtype=DTYPES[c["dtype"]]),
                "cache": DSQGRingCache(c["B"], c["H"], c["D"], TABLES[c["J"]],
                                       dtype=DTYPES[c["dtype"]], device=DEV)}
    if c["kind"] == "decode":
        B, H, D, S, dt = c["B"], c["H"], c["D"], c["S"], DTYPES[c["dtype"]]
        pb, se, _, _ = _params(c, g)
        st = {"case": c, "offsets": TABLES[c["J"]], "pb": pb, "se": se}
        for k in ("k_ring", "v_ring"):
            st[k] = torch.randn((B, H, S, D), generator=g, device=DEV, dtype=dt)
        for k in ("q", "k_new", "v_new"):
            st[k] = _randn(g, B, H, D, dtype=dt)
        st["pos"] = torch.randint(S - 1, 8192, (B,), generator=g, device=DEV)
        return st
    if c["kind"] == "pool":
        shape = (c["B"], c["N"], c["C"])
        return {"case": c, "x": _randn(g, *shape, dtype=DTYPES[c["x"]]).requires_grad_(True),
                "gate": _randn(g, *shape, dtype=DTYPES[c["g"]]).requires_grad_(True),
                "dout": _randn(g, *shape, dtype=torch.promote_types(DTYPES[c["x"]], DTYPES[c["g"]]))}
    m = _block(c)
    with torch.no_grad():  # trained-like values where the initialisation is zero or one
        m.attn.scale_embed.copy_(_randn(g, *m.attn.scale_embed.shape, scale=0.05))
        m.attn.if_gain.copy_(torch.rand(c["H"], generator=g, device=DEV) * 0.4 + 0.8)
    return {"case": c, "m": m,
            "x": _randn(g, c["B"], c["N"], c["E"]).requires_grad_(True),
            "dy": _randn(g, c["B"], c["N"], c["E"], scale=1.0)}


def _block_params(m):
    """The block's parameters, less the injected K's bias: it adds the same to all scores of a
    query, so its gradient is zero, and what a run returns for it is rounding alone."""
    return [(n, p) for n, p in m.named_parameters() if n != "inter_k_proj.bias"]


def _leaves(c):
    """Differentiable inputs of an attention case, in the order of the returned gradients."""
    names = ["qkv"] if c["call"] == "qkv" else ["q", "k", "v"]
    names += ["kd", "vd"] if c["inject"] else []
    return names + ["pb"] + [k for k, on in (("se", c["se"]), ("sg", c["gain"]), ("ig", c["ifg"])) if on]


# ---- One pass --------------------------------------------------------------------------------

def _call_attn(st):
    c = st["case"]
    kw = dict(offsets=st["offsets"], score_gain=st["sg"], if_gain=st["ig"])
    if c["call"] == "qkv":
        return dwarf_amd.dsqg_attention_qkv(
            st["qkv"], c["H"], st["pb"], st["se"],
            kv_inject=(st["kd"], st["vd"]) if c["inject"] else None, **kw)
    return dwarf_amd.dsqg_attention(st["q"], st["k"], st["v"], st["pb"], st["se"], **kw)


def run(state):
    st = state
    c = st["case"]
    if c["kind"] == "attn":
        if not c["grad"]:
            with torch.no_grad():
                return {"out": _call_attn(st)}
        out = _call_attn(st)
        names = _leaves(c)
        grads = torch.autograd.grad(out, [st[k] for k in names], st["dout"])
        return {"out": out.detach(), **{"d" + k: t for k, t in zip(names, grads)}}
    if c["kind"] == "prefill":
        with torch.no_grad():
            out = dwarf_amd.dsqg_attention_qkv(st["qkv"], c["H"], st["pb"], st["se"],
                                               offsets=st["offsets"], if_gain=st["ig"])
            B, N, H, D = c["B"], c["N"], c["H"], c["D"]
            k, v = (t.view(B, N, H, D).permute(0, 2, 1, 3)
                    for t in st["qkv"].split(H * D, dim=-1)[1:])
            st["cache"].prefill(k, v)
        return {"out": out, "k_ring": st["cache"].k_ring, "v_ring": st["cache"].v_ring,
                "pos": st["cache"].pos}
    if c["kind"] == "decode":
        out = dwarf_amd.dsqg_decode_step(st["q"], st["k_new"], st["v_new"], st["k_ring"],
                                         st["v_ring"], st["pos"], st["pb"], st["se"],
                                         offsets=st["offsets"])
        return {"out": out, "k_ring": st["k_ring"], "v_ring": st["v_ring"]}
    if c["kind"] == "pool":
        out = dwarf_amd.causal_mean_pool_gate(st["x"], st["gate"])
        dx, dg = torch.autograd.grad(out, (st["x"], st["gate"]), st["dout"])
        return {"out": out.detach(), "dx": dx, "dgate": dg}
    m, x = st["m"], st["x"]
    names, params = zip(*_block_params(m))
    with torch.amp.autocast("cuda"):
        y = m(x)
    grads = torch.autograd.grad(y, (x, *params), st["dy"])
    return {"y": y.detach(), "dx": grads[0], **dict(zip(names, grads[1:]))}


# ---- What a pass cannot do without ------------------------------------------------------------

def _attn_work(c, grad):
    T, D, J, H = c["B"] * c["H"] * c["N"], c["D"], c["J"], c["H"]
    es = 4 if c.get("dtype") == "f32" else 2
    params = 4 * (J * H + (J * D if c.get("se") else 0) + (J * H if c.get("gain") else 0)
                  + (H if c.get("ifg") else 0))
    # q, k, v (and the deltas) in, out out; backward: dout in, the gradients out.
    rows_in, rows_out = 3 + (2 if c.get("inject") else 0), 1
    flops = T * J * 4 * D + (T * J * 2 * D if c.get("se") else 0)
    if grad:
        rows_in, rows_out = rows_in + 1, rows_out + 3 + (2 if c.get("inject") else 0)
        flops += T * J * 8 * D + (T * J * 4 * D if c.get("se") else 0)
    return {"bytes": T * D * es * (rows_in + rows_out) + params * (2 if grad else 1), "flops": flops}


def work(case):
    c = case
    if c["kind"] == "attn":
        return _attn_work(c, c["grad"])
    if c["kind"] == "prefill":
        w = _attn_work(dict(c, se=True, ifg=True), False)
        w["bytes"] += 4 * c["B"] * c["H"] * min(c["N"], max(TABLES[c["J"]]) + 1) * c["D"]  # the rings
        return w
    if c["kind"] == "decode":
        B, H, D, J = c["B"], c["H"], c["D"], c["J"]
        return {"bytes": B * H * D * 2 * (3 + 2 * (J - 1) + 3), "flops": B * H * J * 4 * D}
    if c["kind"] == "pool":
        n = c["B"] * c["N"] * c["C"]
        xs, gs = DTYPES[c["x"]].itemsize, DTYPES[c["g"]].itemsize
        return {"bytes": n * (xs + gs + max(xs, gs) + max(xs, gs) + xs + gs), "flops": 20 * n}
    T, E, Fd = c["B"] * c["N"], c["E"], c["F"]
    per_token = 8 * E * E + 2 * E * Fd  # qkv 3, out, gate, three interference projections; FFN
    attn = _attn_work(dict(B=c["B"], H=c["H"], N=c["N"], D=E // c["H"], J=44, se=True, ifg=True,
                           inject=True), True)
    return {"bytes": 4 * T * E * 4 + 8 * (per_token + 20 * E), "flops": 6 * T * per_token + attn["flops"]}


def tolerance(case):
    c = case
    if c["kind"] == "block":
        return {"rel": 2e-2}
    if c["kind"] == "pool":
        return {"rel": 1e-2 if c["x"] == "bf16" else 1e-3}
    if c.get("dtype") == "f32":
        return {"rel": 1e-5}
    return {"rel": 1e-2}


# ---- 64-bit results ----------------------------------------------------------------------------

def _shift(t, d):
    """Row n of the result is row n - d of t (zero before the start), along dim 2."""
    N = t.shape[2]
    if d >= N:
        return torch.zeros_like(t)
    return F.pad(t[:, :, :N - d], (0, 0, d, 0))


def _unshift(t, d):
    """Row m of the result is row m + d of t (zero past the end), along dim 2."""
    N = t.shape[2]
    if d >= N:
        return torch.zeros_like(t)
    return F.pad(t[:, :, d:], (0, 0, 0, d))


def _attn64(q, k, v, pb, se, sg, ig, offsets, dout=None):
    """Forward (and gradients) of the attention in float64, one tap at a time."""
    B, H, N, D = q.shape
    J, sc = len(offsets), D ** -0.5
    rows = torch.arange(N, device=q.device)
    s = torch.empty((J, B, H, N), dtype=torch.float64, device=q.device)
    qk = torch.empty_like(s)
    for j, d in enumerate(offsets):
        qk[j] = sc * (q * _shift(k, d)).sum(-1)
        x = qk[j] * sg[:, j][None, :, None] if sg is not None else qk[j]
        x = x + pb[j][None, :, None]
        if se is not None:
            x = x + sc * (q @ se[j])
        s[j] = x.masked_fill(rows < d, -math.inf)
    al = torch.softmax(s, dim=0)
    o = torch.zeros_like(q)
    for j, d in enumerate(offsets):
        o += al[j].unsqueeze(-1) * _shift(v, d)
    a = ig[None, :, None] if ig is not None else torch.ones((), dtype=torch.float64, device=q.device)
    out = o * (a.unsqueeze(-1) if ig is not None else 1.0)
    if dout is None:
        return out, None
    Dp = (dout * o).sum(-1)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(q), torch.zeros_like(q)
    dpb = torch.zeros_like(pb)
    dse = torch.zeros_like(se) if se is not None else None
    dsg = torch.zeros_like(sg) if sg is not None else None
    for j, d in enumerate(offsets):
        kj = _shift(k, d)
        dS = a * al[j] * ((dout * _shift(v, d)).sum(-1) - Dp)
        wk = sc * dS * (sg[:, j][None, :, None] if sg is not None else 1.0)
        dq += wk.unsqueeze(-1) * kj
        dk += _unshift(wk.unsqueeze(-1) * q, d)
        dv += _unshift((a * al[j]).unsqueeze(-1) * dout, d)
        dpb[j] = dS.sum((0, 2))
        if se is not None:
            dq += sc * dS.unsqueeze(-1) * se[j]
            dse[j] = sc * (dS.unsqueeze(-1) * q).sum((0, 1, 2))
        if sg is not None:
            dsg[:, j] = (dS * qk[j]).sum((0, 2))
    dig = Dp.sum((0, 2)) if ig is not None else None
    return out, dict(q=dq, k=dk, v=dv, pb=dpb, se=dse, sg=dsg, ig=dig)


def _merge(ts):
    """[B,H,N,D] parts -> the projection layout [B,N,parts*H*D]."""
    B, H, N, D = ts[0].shape
    return torch.cat([t.permute(0, 2, 1, 3).reshape(B, N, H * D) for t in ts], dim=-1)


def _heads64(qkv, H):
    B, N, E3 = qkv.shape
    return [t.reshape(B, N, H, E3 // (3 * H)).permute(0, 2, 1, 3)
            for t in qkv.detach().double().split(E3 // 3, dim=-1)]


def _d(t):
    return None if t is None else t.detach().double()


def exact(case, seed):
    c = case
    st = prepare(c, seed)
    if c["kind"] == "attn":
        q, k, v = _heads64(st["qkv"], c["H"]) if c["call"] == "qkv" \
            else (_d(st["q"]), _d(st["k"]), _d(st["v"]))
        if c["inject"]:
            k, v = k + _d(st["kd"]), v + _d(st["vd"])
        out, gr = _attn64(q, k, v, *(_d(st[n]) for n in ("pb", "se", "sg", "ig")), st["offsets"],
                          _d(st["dout"]) if c["grad"] else None)
        res = {"out": out}
        if c["grad"]:
            gr.update(kd=gr["k"], vd=gr["v"])
            for n in _leaves(c):
                res["d" + n] = _merge([gr["q"], gr["k"], gr["v"]]) if n == "qkv" else gr[n]
        return res
    if c["kind"] == "prefill":
        q, k, v = _heads64(st["qkv"], c["H"])
        out, _ = _attn64(q, k, v, _d(st["pb"]), _d(st["se"]), None, _d(st["ig"]), st["offsets"])
        N, S = c["N"], max(st["offsets"]) + 1
        res = {"out": out}
        idx = torch.arange(max(0, N - S), N, device=DEV)
        for n, t in (("k_ring", k), ("v_ring", v)):
            res[n] = torch.zeros((c["B"], c["H"], S, c["D"]), dtype=torch.float64, device=DEV)
            res[n][:, :, idx % S] = t[:, :, idx]
        res["pos"] = torch.full((c["B"],), N, dtype=torch.int64, device=DEV)
        return res
    if c["kind"] == "decode":
        S, bi = c["S"], torch.arange(c["B"], device=DEV)
        for r, n in (("k_ring", "k_new"), ("v_ring", "v_new")):
            st[r][bi, :, st["pos"] % S] = st[n]
        sc = c["D"] ** -0.5
        offs = torch.tensor(st["offsets"], device=DEV)
        slots = (st["pos"][:, None] - offs) % S                        # [B,J]
        kj = st["k_ring"][bi[:, None], :, slots].double()               # [B,J,H,D]
        vj = st["v_ring"][bi[:, None], :, slots].double()
        q = st["q"].double()[:, None]
        x = sc * (q * kj).sum(-1) + st["pb"].double()
        if st["se"] is not None:
            x = x + sc * (q * st["se"].double()[None, :, None]).sum(-1)
        x = x.masked_fill((st["pos"][:, None] < offs)[:, :, None], -math.inf)
        out = (torch.softmax(x, dim=1).unsqueeze(-1) * vj).sum(1)
        return {"out": out, "k_ring": st["k_ring"], "v_ring": st["v_ring"]}
    if c["kind"] == "pool":
        x, gt, dy = _d(st["x"]), _d(st["gate"]), _d(st["dout"])
        cnt = torch.arange(1, c["N"] + 1, dtype=torch.float64, device=DEV)[None, :, None]
        s, pool = torch.sigmoid(gt), x.cumsum(1) / cnt
        t = dy * s / cnt
        return {"out": s * pool, "dx": t.flip(1).cumsum(1).flip(1), "dgate": dy * pool * s * (1 - s)}
    return _block64(c, st)


def _block64(c, st):
    """The whole block in float64 with torch's autograd around ``_attn64``."""
    P = {n: p.detach().double().requires_grad_(True) for n, p in st["m"].named_parameters()}
    x = _d(st["x"]).requires_grad_(True)
    B, N, E, H = c["B"], c["N"], c["E"], c["H"]

    def lin(t, n):
        return F.linear(t, P[n + ".weight"], P[n + ".bias"])

    def norm(t, n):
        return F.layer_norm(t, (E,), P[n + ".weight"], P[n + ".bias"])

    def heads(t):
        return t.view(B, N, H, E // H).permute(0, 2, 1, 3)

    class Attn(torch.autograd.Function):
        @staticmethod
        def forward(ctx, *a):
            ctx.save_for_backward(*a)
            q, k, v, pb, se, ig = a
            return _attn64(q, k, v, pb, se, None, ig, OFFSETS_V3)[0]

        @staticmethod
        def backward(ctx, dout):
            q, k, v, pb, se, ig = ctx.saved_tensors
            g = _attn64(q, k, v, pb, se, None, ig, OFFSETS_V3, dout)[1]
            return g["q"], g["k"], g["v"], g["pb"], g["se"], g["ig"]

    cnt = torch.arange(1, N + 1, dtype=torch.float64, device=DEV)[None, :, None]
    xi = norm(x, "inter_norm")
    inter = torch.sigmoid(lin(xi, "inter_gate")) * (xi.cumsum(1) / cnt)
    xn = norm(x, "norm1")
    q, k, v = (heads(t) for t in lin(xn, "attn.qkv_proj").split(E, dim=-1))
    o = Attn.apply(q, k + heads(lin(inter, "inter_k_proj")), v + heads(lin(inter, "inter_v_proj")),
                   P["attn.pos_bias"], P["attn.scale_embed"], P["attn.if_gain"])
    o = o.permute(0, 2, 1, 3).reshape(B, N, E) * torch.sigmoid(lin(xn, "attn.gate_proj"))
    y = x + lin(o, "attn.out_proj")
    y = y + lin(F.gelu(lin(norm(y, "norm2"), "ffn.fc1")), "ffn.fc2")
    names = [n for n, _ in _block_params(st["m"])]
    grads = torch.autograd.grad(y, (x, *(P[n] for n in names)), st["dy"].double())
    return {"y": y.detach(), "dx": grads[0], **dict(zip(names, grads[1:]))}
