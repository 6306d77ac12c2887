"""The work whose speed is measured: the calls a serving engine makes on this library, through inferd_amd.ops.

Every case is one operator call (or the producer-consumer pair a route is made of) on weights that were repacked once
at load. The kinds, and what in real use each stands for:

- linear:   one quantized linear of a layer on its T64 copy. One row is the smallest call (a single agent's decode
            step through a square projection); thousands of rows are a prompt's prefill through a wide one. out says
            where the result goes: a new bf16 tensor, added into the residual stream, or fp32.
- mlp:      the dense MLP block (norm, gate and up with SwiGLU, down added into the residual stream) for a batch of
            concurrent agents (up to 128 rows) or a prompt chunk of some hundred rows, ragged as prompts are.
- int8:     a linear on int8 activations, quantizer included: per token (prefill), or per 64-group as decode runs it
            when the weights are flipped.
- linear8:  a linear of an 8-bit layer on its T64x8 copy, for a decode batch.
- moe_step: the mixture-of-experts layer for a decode step of up to 16 tokens.
- moe:      the same layer for larger batches and prompt chunks, the sorted route.

The dense sizes are those of a 5120-wide layer with a 17408-wide MLP, the expert sizes those of a 2048-wide layer with
512 experts of width 512, 10 per token and one shared expert: the sizes of bench.py. Drawn cases take other widths.

Weights are affine 4- or 8-bit groups of 64 whose dequantized values have a variance of 1 / K, as trained layers have
about, so that activations keep their size from layer to layer.
"""
from __future__ import annotations

from types import SimpleNamespace

import torch

from inferd_amd import ops

EPS = 1e-6
DEV = "cuda"


# ---- the cases -----------------------------------------------------------------------------------------------------
def listed():
    return [
        # one agent's decode step through a square projection: launch latency against 15 MB of weights
        dict(name="linear_m1", kind="linear", M=1, N=5120, K=5120, out="new"),
        # the dense MLP of a decode step for a few, some and many concurrent agents
        dict(name="mlp_m8", kind="mlp", M=8, H=5120, I=17408),
        dict(name="mlp_m32", kind="mlp", M=32, H=5120, I=17408),
        dict(name="mlp_m128", kind="mlp", M=128, H=5120, I=17408),
        # a prompt chunk of an ordinary, ragged length
        dict(name="mlp_m777", kind="mlp", M=777, H=5120, I=17408),
        # a long prompt through a wide linear: the largest call
        dict(name="linear_m4096", kind="linear", M=4096, N=17408, K=5120, out="new"),
        # prefill on int8 activations, one scale per token
        dict(name="int8_token_m2048", kind="int8", M=2048, N=5120, K=5120, group=False),
        # a decode batch over flipped weights: int8 activations with a scale per row and 64-group
        dict(name="int8_group_m24", kind="int8", M=24, N=34816, K=5120, group=True),
        # an 8-bit layer in a decode batch
        dict(name="linear8_m8", kind="linear8", M=8, N=34816, K=5120),
        # the expert layer: a decode step of four agents, a batch of a hundred tokens, a long prompt chunk
        dict(name="moe_step_t4", kind="moe_step", T=4, H=2048, I=512, E=512, k=10),
        dict(name="moe_t100", kind="moe", T=100, H=2048, I=512, E=512, k=10),
        dict(name="moe_t2048", kind="moe", T=2048, H=2048, I=512, E=512, k=10),
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "mlp", "mlp", "int8", "int8", "linear8", "moe_step", "moe", "moe"])
    if kind == "linear":
        return dict(kind=kind, M=_log_int(rng, 1, 4096), N=_log_int(rng, 1024, 17408, 16),
                    K=_log_int(rng, 1024, 5120, 256), out=rng.choice(["new", "new", "add", "fp32"]))
    if kind == "mlp":
        return dict(kind=kind, M=_log_int(rng, 1, 1280), H=_log_int(rng, 2048, 5120, 256),
                    I=_log_int(rng, 4096, 17408, 256))
    if kind == "int8":
        group = rng.random() < 0.5
        return dict(kind=kind, M=_log_int(rng, 3, 255) if group else _log_int(rng, 129, 4096),
                    N=_log_int(rng, 2048, 34816 if group else 8192, 64), K=_log_int(rng, 2048, 5120, 256), group=group)
    if kind == "linear8":
        return dict(kind=kind, M=_log_int(rng, 1, 128), N=_log_int(rng, 2048, 34816, 64),
                    K=_log_int(rng, 2048, 5120, 256))
    E = rng.choice([64, 128, 256, 512])
    sizes = dict(H=rng.choice([2048, 2048, 4096]), I=rng.choice([512, 512, 1024]), E=E, k=rng.choice([4, 6, 8, 10]))
    if kind == "moe_step":
        return dict(kind=kind, T=_log_int(rng, 1, 16), **sizes)
    return dict(kind=kind, T=_log_int(rng, 17, 2048), **sizes)


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _affine(g, rows, K, bits):
    """Packed codes, scales and biases of rows of K weights: codes uniform, the zero point near the middle code."""
    words = K * bits // 32
    levels = 1 << bits
    wq = torch.randint(-2 ** 31, 2 ** 31, (rows, words), dtype=torch.int32, device=DEV, generator=g)
    std = levels / 12 ** 0.5  # of the codes
    s = (0.6 + 0.8 * torch.rand((rows, K // 64), device=DEV, generator=g)) / (std * K ** 0.5)
    s = s.to(torch.bfloat16)
    mid = (levels - 1) / 2 * (1 + 0.1 * (torch.rand((rows, K // 64), device=DEV, generator=g) - 0.5))
    return wq, s, (-mid * s.float()).to(torch.bfloat16)


def _layer(g, N, K, bits=4):
    wq, s, b = _affine(g, N, K, bits)
    return SimpleNamespace(wq=wq, s=s, b=b, N=N, K=K, bits=bits)


def _stack(g, E, N, K):
    wq, s, b = _affine(g, E * N, K, 4)
    return SimpleNamespace(wq=wq.view(E, N, -1), s=s.view(E, N, -1), b=b.view(E, N, -1), E=E, N=N, K=K)


def _pack(w):
    """The layer as the loader keeps it: repacked once."""
    if hasattr(w, "E"):
        return ops.pack_t64_stack(ops.MoeW(w.wq, w.s, w.b, w.E, w.N, w.K))
    layer = ops.QLinear(w.wq, w.s, w.b, w.N, w.K, bits=w.bits)
    return ops.pack_t64x8(layer) if w.bits == 8 else ops.pack_t64(layer)


def _rows(g, M, K):
    """Activations: normal values, rows of different size."""
    x = torch.randn((M, K), device=DEV, generator=g) * (0.5 + 1.5 * torch.rand((M, 1), device=DEV, generator=g))
    return x.to(torch.bfloat16)


def _norm_weight(g, H):
    return (0.5 + torch.rand((H,), device=DEV, generator=g)).to(torch.bfloat16)


def _inputs(case, seed):
    """The checkpoint's layers (MLX layout) and the activations, from the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("linear", "int8", "linear8"):
        M, N, K = case["M"], case["N"], case["K"]
        d = dict(w=_layer(g, N, K, 8 if kind == "linear8" else 4), x=_rows(g, M, K))
        if case.get("out") == "add":
            d["c"] = _rows(g, M, N)
        return d
    if kind == "mlp":
        M, H, I = case["M"], case["H"], case["I"]
        return dict(gu=_layer(g, 2 * I, H), dn=_layer(g, H, I), nw=_norm_weight(g, H), x=_rows(g, M, H))
    T, H, I, E = case["T"], case["H"], case["I"], case["E"]
    return dict(gu=_stack(g, E, 2 * I, H), dn=_stack(g, E, H, I), sgu=_layer(g, 2 * I, H), sdn=_layer(g, H, I),
                router=(torch.randn((E + 1, H), device=DEV, generator=g) * H ** -0.5).to(torch.bfloat16),
                x=_rows(g, T, H))


def prepare(case, seed):
    """What the engine holds before the call: activations, and the layers repacked as the loader does."""
    d = _inputs(case, seed)
    kind = case["kind"]
    st = dict(case=case, x=d["x"])
    if kind in ("linear", "int8", "linear8"):
        st["w"] = _pack(d["w"])
        st["c"] = d.get("c")
        if st["c"] is None:
            st["c"] = torch.empty((case["M"], case["N"]), device=DEV,
                                  dtype=torch.float32 if case.get("out") == "fp32" else torch.bfloat16)
    elif kind == "mlp":
        st.update(gu=_pack(d["gu"]), dn=_pack(d["dn"]), nw=d["nw"])
    else:
        st.update(gu=_pack(d["gu"]), dn=_pack(d["dn"]), shared=(_pack(d["sgu"]), _pack(d["sdn"])), router=d["router"],
                  out=torch.zeros_like(d["x"]))
    return st


MODES = {"new": 0, "add": 1, "fp32": 2}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        return ops.gemm_t64(st["x"], st["w"], st["c"], MODES[case["out"]])
    if kind == "linear8":
        return ops.gemm_t64x8(st["x"], st["w"], st["c"])
    if kind == "int8":
        U, XS = ops.a8_quant(st["x"], not case["group"])
        return ops.gemm_t64_w4a8(U, XS, st["w"], st["c"], per_token=not case["group"])
    if kind == "mlp":
        return ops.mlp_decode(st["x"], st["nw"], EPS, st["gu"], st["dn"])
    if kind == "moe_step":
        out, _, _, _, logits = ops.moe_decode_t64(st["x"], st["router"], st["gu"], st["dn"], case["k"],
                                                  shared=st["shared"], out=st["out"])
        return dict(out=out, logits=logits)
    out, idx, wt, sg = ops.moe_ffn_t64(st["x"], st["router"], st["gu"], st["dn"], case["k"], shared=st["shared"],
                                       logits_bf16=case["T"] >= 64, out=st["out"])
    return dict(out=out, wt=wt, sg=sg)


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("linear", "int8", "linear8"):
        M, N, K = case["M"], case["N"], case["K"]
        per = 1.0625 if kind == "linear8" else 0.5625
        out = {"new": 2, "add": 4, "fp32": 4}[case.get("out", "new")]
        return {"bytes": N * K * per + M * K * 2 + M * N * out, "flops": 2.0 * M * N * K}
    if kind == "mlp":
        M, H, I = case["M"], case["H"], case["I"]
        return {"bytes": 3 * H * I * 0.5625 + H * 2 + M * H * 4, "flops": 6.0 * M * H * I}
    T, H, I, E, k = case["T"], case["H"], case["I"], case["E"], case["k"]
    used = E * (1 - (1 - k / E) ** T) + 1  # distinct experts of evenly spread picks, and the shared one
    return {"bytes": used * 3 * H * I * 0.5625 + (E + 1) * H * 2 + 2 * T * H * 2,
            "flops": 6.0 * T * (k + 1) * H * I + 2.0 * T * H * (E + 1)}


def tolerance(case):
    """About four times what a call is off the 64-bit result: the rounding of a bf16 output is 1.7e-3 in the 2-norm, the
    bf16 dequantized weights of larger batches add as much, and the blocks round their intermediate rows too (mlp 2.9e-3,
    the expert layer 5e-3). Int8 activations are the same on every side: their quantizer is exact."""
    kind = case["kind"]
    if kind in ("linear", "linear8", "int8"):
        return {"rel": 8e-3, "max": 4e-2}
    if kind == "mlp":
        return {"rel": 1.1e-2, "max": 6e-2}
    # a token whose last and next expert are a rounding apart may pick the other one
    return {"rel": 1.8e-2, "max": 0.6}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------
def _codes(wq, bits):
    per = 32 // bits
    shift = torch.arange(per, device=wq.device, dtype=torch.int32) * bits
    return ((wq.unsqueeze(-1) >> shift) & ((1 << bits) - 1)).reshape(*wq.shape[:-1], -1)


def _dense(wq, s, b, bits=4):
    """s q + b in 64 bits."""
    q = _codes(wq, bits).double()
    q = q.view(*q.shape[:-1], -1, 64)
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).flatten(-2)


def _product(x, layer, bits=4):
    """x . W^T in 64 bits, a slice of W's rows at a time."""
    step = max(1, (1 << 26) // layer.K)
    return torch.cat([x @ _dense(layer.wq[i:i + step], layer.s[i:i + step], layer.b[i:i + step], bits).T
                      for i in range(0, layer.N, step)], 1)


def _swiglu(gu):
    gate, up = gu.chunk(2, -1)
    return gate * torch.sigmoid(gate) * up


def _quantized(x, group):
    """The int8 activations' values: x / scale rounded to whole numbers, times the scale (one per row or 64-group), with
    the scale and the quotient in fp32 as the format has them."""
    x = x.float()
    v = x.view(x.shape[0], -1, 64) if group else x.unsqueeze(1)
    scale = v.abs().amax(-1, keepdim=True) / 127
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    return (torch.round(v / scale).double() * scale.double()).view(x.shape)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    x = d["x"].double()
    if kind == "linear":
        y = _product(x, d["w"])
        return y + d["c"].double() if case["out"] == "add" else y
    if kind == "linear8":
        return _product(x, d["w"], 8)
    if kind == "int8":
        return _product(_quantized(d["x"], case["group"]), d["w"])
    if kind == "mlp":
        xn = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * d["nw"].double()
        return x + _product(_swiglu(_product(xn, d["gu"])), d["dn"])
    E, k = case["E"], case["k"]
    logits = x @ d["router"].double().T
    if kind == "moe" and case["T"] >= 64:
        seen = logits.to(torch.bfloat16).double()  # the routing reads bf16 logits at these sizes
    else:
        seen = logits
    order = torch.sort(seen[:, :E], dim=-1, descending=True, stable=True).indices[:, :k]
    wt = torch.softmax(seen[:, :E], -1).gather(1, order)
    wt = wt / wt.sum(-1, keepdim=True)
    sg = torch.sigmoid(seen[:, E])
    out = sg[:, None] * _product(_swiglu(_product(x, d["sgu"])), d["sdn"])
    for e in order.unique().tolist():
        t, j = (order == e).nonzero(as_tuple=True)
        h = _swiglu(x[t] @ _dense(d["gu"].wq[e], d["gu"].s[e], d["gu"].b[e]).T)
        out.index_add_(0, t, wt[t, j, None] * (h @ _dense(d["dn"].wq[e], d["dn"].s[e], d["dn"].b[e]).T))
    if kind == "moe_step":
        return dict(out=out, logits=logits)
    return dict(out=out, wt=wt, sg=sg)
