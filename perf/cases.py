"""The work that a program built on this package has it do, as cases that can be timed.

Each listed case stands for one use (its comment says which); ``draw`` gives more cases of the
same ranges.  Four kinds:

* ``core``    -- the fused order-2 op ``flash_poly_attention``, forward and backward;
* ``train``   -- one attention layer (``PolyAttention`` / ``NPolyAttention``), forward and backward
  down to the gradients of its input and of every parameter;
* ``infer``   -- one attention layer without gradients; with ``cache`` it is the prefill of a
  decoding loop and returns the KV cache, with ``graph`` the call is captured once and replayed;
* ``decode``  -- one token through one layer and its ``StaticCache``; with ``graph`` the step is
  captured once and replayed per token, as a decoding loop does.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "poly-attention_amd"))

from poly_attention import NPolyAttention, PolyAttention, StaticCache  # noqa: E402
from poly_attention.flash_poly_attention import flash_poly_attention  # noqa: E402

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _core(b, h, n, d, dtype="bf16", causal=True, softclamp=0.0, pad="none"):
    return {"kind": "core", "b": b, "h": h, "n": n, "d": d, "dtype": dtype, "causal": causal,
            "softclamp": softclamp, "pad": pad}


def _layer(kind, order, b, n, dim, heads, d, kv_heads=0, dtype="bf16", causal=True, rotary="none",
           gated=False, prenorm=False, cache=False, graph=False):
    return {"kind": kind, "order": order, "b": b, "n": n, "dim": dim, "heads": heads,
            "kv_heads": kv_heads or heads, "d": d, "dtype": dtype, "causal": causal,
            "rotary": rotary, "gated": gated, "prenorm": prenorm, "cache": cache, "graph": graph}


def listed():
    cases = {
        # causal language-model training at the headline size (bench.py's config 2)
        "core_train_4k": _core(4, 16, 4096, 64),
        # an encoder over ragged sequences, f16, both directions
        "core_train_encoder": _core(8, 8, 1000, 64, dtype="f16", causal=False),
        # causal training at the larger head dim
        "core_train_d128": _core(2, 16, 2048, 128),
        # causal training with the score soft clamp
        "core_train_softclamp": _core(4, 8, 1000, 64, softclamp=50.0),
        # causal training on a right-padded batch
        "core_train_padded": _core(4, 16, 2048, 64, pad="right"),
        # training in full precision
        "core_train_f32": _core(2, 8, 1024, 64, dtype="f32"),
        # a training step of one order-3 layer with external rotary embeddings
        "layer3_train": _layer("train", 3, 2, 2048, 1024, 16, 64, rotary="external"),
        # a training step of one order-2 layer with its own rotary, root value and gates
        "layer2_train_gated": _layer("train", 2, 4, 1024, 512, 8, 64, rotary="module",
                                     gated=True, prenorm=True),
        # one small full-precision layer call (bench.py's config 1): latency
        "layer2_infer_f32": _layer("infer", 2, 1, 1024, 512, 8, 64, dtype="f32", causal=False),
        # a vision transformer's attention block on 64 patches, captured for serving
        "vit_layer": _layer("infer", 2, 64, 64, 1024, 16, 64, causal=False, prenorm=True,
                            graph=True),
        # a grouped-query layer's token step over a long cache (bench.py's config 5)
        "decode2_gqa": _layer("decode", 2, 32, 8192, 4096, 32, 128, kv_heads=8),
        # an order-3 layer's token step, captured (bench.py's config 4)
        "decode3": _layer("decode", 3, 8, 2049, 1024, 16, 64, rotary="external", graph=True),
    }
    return [dict(c, name=k) for k, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["core", "core", "core", "train", "train", "infer", "infer", "decode",
                       "decode"])
    if kind == "core":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        d = rng.choice([64, 64, 64, 128, 32, 96])
        h = rng.choice([4, 8] if dtype == "f32" else [4, 8, 16])
        n = _log_int(rng, 128, 1024 if dtype == "f32" else 4096)
        tokens = 2048 if dtype == "f32" else 8192
        c = _core(max(1, min(16, rng.randint(tokens // 4, tokens) // n)), h, n, d, dtype=dtype,
                  causal=rng.random() < 0.7, softclamp=rng.choice([0.0, 0.0, 0.0, 30.0]),
                  pad=rng.choice(["none", "none", "right", "left"]))
        # at most about the time of the largest listed case
        most = (4e10 if dtype == "f32" else 9e11) / (6 if c["softclamp"] else 1)
        while work(c)["flops"] > most:
            c["n"] -= c["n"] // 8
        return c
    order = rng.choice([2, 3, 3])
    heads, d = rng.choice([(8, 64), (16, 64), (8, 128)])
    kv_heads = rng.choice([heads, heads, heads // 4])
    dim = heads * d
    rotary = rng.choice(["none", "external", "module"])
    if kind == "decode":
        b = _log_int(rng, 1, 32)
        n = _log_int(rng, 300, 8192)
        return _layer("decode", order, b, n, dim, heads, d, kv_heads=kv_heads,
                      rotary=rng.choice(["none", "external"]), graph=b <= 16)
    dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
    n = _log_int(rng, 64, 512 if dtype == "f32" else 2048)
    tokens = 1024 if dtype == "f32" else 2048 if rotary == "module" else 4096
    b = max(1, min(64, rng.randint(tokens // 4, tokens) // n))
    prefill = kind == "infer" and rng.random() < 0.5
    return _layer(kind, order, b, n, dim, heads, d, kv_heads=kv_heads, dtype=dtype,
                  causal=prefill or rng.random() < 0.7, rotary=rotary,
                  gated=kv_heads == heads and rng.random() < 0.4, prenorm=rng.random() < 0.5,
                  cache=prefill)


# ---------------------------------------------------------------------------------------
# inputs, made from the seed alone


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, shape, dt, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dt)


def _core_inputs(c, seed):
    """q1, q2, q3, v3 as an RMS-normed projection gives them, the upstream gradient, and the
    padding mask (True on kept keys)."""
    g, dt = _gen(seed), _DT[c["dtype"]]
    shape = (c["b"], c["h"], c["n"], c["d"])
    ts = [_randn(g, shape, dt) for _ in range(5)]
    mask = None
    if c["pad"] != "none":
        # the first row of the batch is full, the others keep half to all of their positions
        n = c["n"]
        kept = torch.randint(max(1, n // 2), n + 1, (c["b"],), generator=g, device="cuda")
        kept[0] = n
        pos = torch.arange(n, device="cuda")[None, :]
        mask = pos < kept[:, None] if c["pad"] == "right" else pos >= n - kept[:, None]
    return ts, mask


def _layer_weights(c, seed):
    """Name -> tensor of the layer's parameters, scaled as the default initialisation of a linear
    layer (norm weights around 1)."""
    g, dt = _gen(seed + 7919), _DT[c["dtype"]]
    dim, order = c["dim"], c["order"]
    inner, inner_kv = c["heads"] * c["d"], c["kv_heads"] * c["d"]
    std = (3.0 * dim) ** -0.5

    def linear(out, width):
        return _randn(g, (out, width), dt, std)

    def norm(width):
        return (1.0 + 0.1 * torch.randn(width, generator=g, device="cuda")).to(dt)

    w = {"to_q.weight": linear(inner * (2 if c["gated"] else 1), dim),
         "to_kvs.0.weight": linear(inner_kv * (2 if c["gated"] else 1), dim)}
    for i in range(1, order):
        w["to_kvs.%d.weight" % i] = linear(inner_kv * 2, dim)
    for i in range(order + 1):
        w["q_norms.%d.weight" % i] = norm(c["d"])
    w["to_out.weight"] = linear(dim, inner)
    w["to_out.bias"] = _randn(g, (dim,), dt, std)
    if c["prenorm"]:
        w["norm.weight"] = norm(dim)
    return w


def _make_layer(c, weights):
    opts = dict(dim=c["dim"], heads=c["heads"], kv_heads=c["kv_heads"], dim_head=c["d"],
                causal=c["causal"], use_rotary_embed=c["rotary"] == "module",
                prenorm=c["prenorm"], multiply_root_value=c["gated"], attn_gate=c["gated"])
    with torch.device("cuda"):
        layer = PolyAttention(**opts) if c["order"] == 2 else NPolyAttention(order=c["order"], **opts)
    rotary = layer.rotary_emb  # its frequencies stay in fp32
    layer.rotary_emb = None
    layer = layer.to(_DT[c["dtype"]])
    with torch.no_grad():
        params = dict(layer.named_parameters())
        assert set(params) == set(weights)
        for k, p in params.items():
            p.copy_(weights[k])
    layer.rotary_emb = rotary
    return layer


def _angles(positions, d):
    """[positions, d] rotary angles in fp32: each frequency for a pair of features."""
    freqs = 10000.0 ** -(torch.arange(0, d, 2, device="cuda").float() / d)
    return (positions.float()[:, None] * freqs).repeat_interleave(2, dim=-1)


def _layer_inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    x = _randn(g, (c["b"], c["n"], c["dim"]), dt)
    dy = _randn(g, (c["b"], c["n"], c["dim"]), dt)
    pos = _angles(torch.arange(c["n"], device="cuda"), c["d"]) if c["rotary"] == "external" else None
    return x, dy, pos


def _decode_inputs(c, seed):
    """The new token's hidden state, its rotary angles and a cache of n - 1 positions as a prefill
    leaves it: normed keys, values, each level's outputs (averages of values, so smaller) and
    logsumexps (about log of the number of positions attended)."""
    g, dt = _gen(seed), _DT[c["dtype"]]
    b, n, d, order = c["b"], c["n"] - 1, c["d"], c["order"]
    x = _randn(g, (b, 1, c["dim"]), dt)
    kv, full = (b, c["kv_heads"], n, d), (b, c["heads"], n, d)

    def fill(shape, std=1.0):
        return torch.empty(shape, dtype=dt, device="cuda").normal_(0.0, std, generator=g)

    qs = tuple(fill(kv) for _ in range(order))
    vs = tuple(fill(kv) for _ in range(order - 1))
    rise = torch.log(torch.arange(1, n + 1, device="cuda").float())
    lses, msgs = [], []
    for lvl in range(order - 1):
        lses.append((lvl + 1) * (rise + 0.5) + 0.2 * torch.randn(full[:3], generator=g, device="cuda"))
        msgs.append(fill(full, 0.2))
    pos = _angles(torch.tensor([n], device="cuda"), d)[0] if c["rotary"] == "external" else None
    return x, pos, qs, vs, tuple(lses), tuple(msgs)


class _Replay:
    """A call captured into a HIP graph: replay() leaves the result in the same tensors."""

    def __init__(self, call):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                call()
        torch.cuda.current_stream().wait_stream(side)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.out = call()

    def __call__(self):
        self.graph.replay()
        return self.out


def prepare(case, seed):
    c = case
    if c["kind"] == "core":
        ts, mask = _core_inputs(c, seed)
        return {"case": c, "qs": [t.requires_grad_() for t in ts[:4]], "dout": ts[4], "mask": mask}
    layer = _make_layer(c, _layer_weights(c, seed))
    if c["kind"] == "train":
        x, dy, pos = _layer_inputs(c, seed)
        params = [p for _, p in sorted(layer.named_parameters()) if p.requires_grad]
        return {"case": c, "layer": layer, "x": x.requires_grad_(), "dy": dy, "pos": pos,
                "params": params}
    layer.requires_grad_(False)
    if c["kind"] == "infer":
        x, _, pos = _layer_inputs(c, seed)
        state = {"case": c, "layer": layer, "x": x, "pos": pos}
        if c["graph"]:
            state["replay"] = _Replay(lambda: _infer(layer, x, pos, c))
        return state
    x, pos, qs, vs, lses, msgs = _decode_inputs(c, seed)
    cache = (*qs, *vs, *lses, *msgs) if c["order"] == 2 else (qs, vs, lses, msgs)
    # one layer of a model: the model owns the position count and advances it after its last layer
    static = StaticCache(cache, c["n"] + 64, counter=StaticCache.make_counter(cache))
    state = {"case": c, "layer": layer, "x": x, "pos": pos, "cache": static}
    if c["graph"]:
        state["replay"] = _Replay(lambda: _token(layer, x, pos, static))
    return state


@torch.no_grad()
def _infer(layer, x, pos, c):
    if not c["cache"]:
        return layer(x, rotary_pos_emb=pos)
    return layer(x, rotary_pos_emb=pos, return_cache=True)


@torch.no_grad()
def _token(layer, x, pos, static):
    return layer(x, rotary_pos_emb=pos, cache=static)


def run(state):
    c = state["case"]
    if c["kind"] == "core":
        out = flash_poly_attention(*state["qs"], mask=state["mask"],
                                   softclamp_value=c["softclamp"] or None, is_causal=c["causal"])
        return (out, *torch.autograd.grad(out, state["qs"], state["dout"]))
    if c["kind"] == "train":
        out = state["layer"](state["x"], rotary_pos_emb=state["pos"])
        return (out, *torch.autograd.grad(out, [state["x"], *state["params"]], state["dy"]))
    if "replay" in state:
        out = state["replay"]()
    elif c["kind"] == "infer":
        out = _infer(state["layer"], state["x"], state["pos"], c)
    else:
        out = _token(state["layer"], state["x"], state["pos"], state["cache"])
    if c["kind"] == "decode":
        # the token's entries of the cache are the step's other result
        st, at = state["cache"], c["n"] - 1
        return [out] + [t.select(2, at) for ts in (st.qs, st.vs, st.lses, st.msgs) for t in ts]
    return out


# ---------------------------------------------------------------------------------------
# what a pass cannot do without


def _level_flops(c, heads, n_q, n_k, per_pair):
    share = 0.5 if c.get("causal") and n_q == n_k else 1.0
    return per_pair * share * heads * n_q * n_k * c["d"] * c["b"]


def work(case):
    c = case
    size = 4 if c["dtype"] == "f32" else 2
    if c["kind"] == "core":
        # forward 2 products, backward 5 (S, dP, dQ, dK, dV), at both levels
        rows = c["b"] * c["h"] * c["n"]
        return {"bytes": rows * (10 * c["d"] * size), "flops": 2 * _level_flops(c, c["h"], c["n"], c["n"], 14)}
    order, dim = c["order"], c["dim"]
    inner, inner_kv = c["heads"] * c["d"], c["kv_heads"] * c["d"]
    g = 2 if c["gated"] else 1
    weights = dim * (inner * g + inner_kv * g + inner_kv * 2 * (order - 1) + inner)
    rows = c["b"] * (1 if c["kind"] == "decode" else c["n"])
    flops = 2.0 * rows * weights
    if c["kind"] == "decode":
        pos = c["b"] * c["n"]
        cache = pos * ((2 * order - 1) * inner_kv * size + (order - 1) * (inner * size + 4 * c["heads"]))
        flops += 4.0 * pos * c["d"] * (c["heads"] + (order - 1) * c["kv_heads"])
        return {"bytes": cache + weights * size + 2 * rows * dim * size, "flops": flops}
    levels = c["heads"] + (order - 1) * c["kv_heads"]
    if c["kind"] == "train":
        flops = 3 * flops + _level_flops(c, levels, c["n"], c["n"], 14)
        moved = 4 * rows * dim * size + 2 * weights * size
    else:
        flops += _level_flops(c, levels, c["n"], c["n"], 4)
        moved = 2 * rows * dim * size + weights * size
        if c["cache"]:
            moved += rows * ((2 * order - 1) * inner_kv * size + (order - 1) * (inner * size + 4 * c["heads"]))
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times what the start showed against ``exact``, over all outputs: the f32 ones at most
    1.9e-6 off, the f16 ones 4.5e-4, the bf16 ones of the op 4.4e-3 and of a whole layer, whose
    gradients pass more roundings, up to 1.2e-2 (there no more than is allowed)."""
    if case["dtype"] == "f32":
        return {"rel": 8e-6, "max": 5e-4}
    if case["dtype"] == "f16":
        return {"rel": 2e-3, "max": 0.1}
    if case["kind"] == "core":
        return {"rel": 1.6e-2, "max": 0.6}
    return {"rel": 3e-2, "max": 0.99}


# ---------------------------------------------------------------------------------------
# the same results in 64 bits, in plain torch


def _softclamp64(s, c):
    return c * torch.tanh(s / c) if c else s


def _level64(q, k, v, bias, c, keep, softclamp):
    """One level: (softmax(q k^T + bias) v, logsumexp); keep [b, n] masks keys with the finite fill
    of the type, as causal positions."""
    s = _softclamp64(torch.matmul(q, k.transpose(-1, -2)) * c["d"] ** -0.5, softclamp)
    fill = -torch.finfo(s.dtype).max
    if c["causal"] and s.shape[-2] == s.shape[-1]:
        s = s.masked_fill(torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1), fill)
    if keep is not None:
        s = torch.where(keep[:, None, None, :], s, fill)
    if bias is not None:
        s = s + bias[..., None, :]
    return torch.matmul(s.softmax(-1), v), s.logsumexp(-1)


def _core64(c, seed):
    ts, mask = _core_inputs(c, seed)
    got = [torch.empty(t.shape, dtype=torch.float64, device="cuda") for t in ts]
    for i in range(c["b"]):
        keep = mask[i:i + 1] if mask is not None else None
        for h in range(c["h"]):  # a head at a time: the scores are n x n in 64 bits
            q1, q2, q3, v3, dy = (t[i:i + 1, h:h + 1].detach().double() for t in ts)
            for t in (q1, q2, q3, v3):
                t.requires_grad_()
            msg, lse = _level64(q2, q3, v3, None, c, keep, c["softclamp"])
            out, _ = _level64(q1, q2, msg, lse, c, keep, c["softclamp"])
            grads = torch.autograd.grad(out, (q1, q2, q3, v3), dy)
            for to, t in zip(got, (out.detach(), *grads)):
                to[i, h] = t[0, 0]
    return tuple(got)


def _rms64(x, w):
    return x * (x.square().mean(-1, keepdim=True) + torch.finfo(torch.float32).eps).rsqrt() * w


def _rotate64(t, angles):
    """Interleaved pairs of t [b, h, n, d] turned by angles [n, d] (fp32, as a program has them)."""
    a = angles.double()
    x = t.unflatten(-1, (-1, 2))
    half = torch.stack((-x[..., 1], x[..., 0]), -1).flatten(-2)
    return t * a.cos() + half * a.sin()


def _repeat(t, rep):
    return t.repeat_interleave(rep, dim=1) if rep > 1 else t


def _project64(c, w, x):
    """The raw heads of a layer: queries [q1 .. q_{order+1}], values [v3 ..], root value, gates."""
    d, order = c["d"], c["order"]

    def heads(y, h):
        return y.unflatten(-1, (-1, h, d)).permute(2, 0, 3, 1, 4)  # [parts, b, h, n, d]

    def lin(name):
        return torch.matmul(x, w[name + ".weight"].t())

    q = heads(lin("to_q"), c["heads"])
    first = heads(lin("to_kvs.0"), c["kv_heads"])
    rest = [heads(lin("to_kvs.%d" % i), c["kv_heads"]) for i in range(1, order)]
    qs = [q[0], first[0], *[r[0] for r in rest]]
    return qs, [r[1] for r in rest], first[1] if c["gated"] else None, q[1] if c["gated"] else None


def _finish64(c, w, out, root, gate):
    if root is not None:
        out = _repeat(root, c["heads"] // c["kv_heads"]) * out
    if gate is not None:
        out = out * gate.sigmoid()
    out = out.permute(0, 2, 1, 3).flatten(2)
    return torch.matmul(out, w["to_out.weight"].t()) + w["to_out.bias"]


def _forward64(c, w, x, pos):
    """One layer over a whole sequence: (out, the cache it returns)."""
    h = _rms64(x, w["norm.weight"]) if c["prenorm"] else x
    qs, vs, root, gate = _project64(c, w, h)
    qs = [_rms64(q, w["q_norms.%d.weight" % i]) for i, q in enumerate(qs)]
    if c["rotary"] == "external":
        qs = [_rotate64(q, pos) for q in qs]
    left, right = qs[:-1], qs[1:]
    if c["rotary"] == "module":
        # the layer counts its positions in the type of its queries
        turn = _angles(torch.arange(c["n"], device="cuda", dtype=_DT[c["dtype"]]), c["d"])
        left, right = ([_rotate64(q, turn) for q in side] for side in (left, right))
    rep = c["heads"] // c["kv_heads"]
    out, lse, lses, msgs = None, None, [], []
    for lvl in range(c["order"] - 1, -1, -1):
        if lvl == c["order"] - 1:
            v = vs[-1]
        elif lvl == 0:
            v = out
        else:
            v = vs[lvl - 1] * out
        q, k = left[lvl], right[lvl]
        if lvl == 0:
            k, v, lse = _repeat(k, rep), _repeat(v, rep), _repeat(lse[..., None], rep)[..., 0]
        out, lse = _level64(q, k, v, lse, c, None, 0.0)
        if lvl > 0:
            lses.append(_repeat(lse[..., None], rep)[..., 0])
            msgs.append(_repeat(out, rep))
    out = _finish64(c, w, out, root, gate)
    if c["order"] == 2:
        return out, (*qs[1:], *vs, *lses, *msgs)
    return out, (tuple(qs[1:]), tuple(vs), tuple(lses), tuple(msgs))


def _decode64(c, seed):
    w = {k: t.double() for k, t in _layer_weights(c, seed).items()}
    x, pos, c_qs, c_vs, c_lses, c_msgs = _decode_inputs(c, seed)
    h = _rms64(x.double(), w["norm.weight"]) if c["prenorm"] else x.double()
    qs, vs, root, gate = _project64(c, w, h)
    qs = [_rms64(q, w["q_norms.%d.weight" % i]) for i, q in enumerate(qs)]
    if pos is not None:
        qs = [_rotate64(q, pos[None]) for q in qs]
    order, rep = c["order"], c["heads"] // c["kv_heads"]
    rows = []
    for i in range(c["b"]):  # a batch row at a time: the cache in 64 bits is four times its size
        def at(t):
            return t[i:i + 1].double()

        out = lse = None
        lses, msgs = [], []
        for lvl in range(order - 1, -1, -1):
            k = torch.cat((at(c_qs[lvl]), at(qs[lvl + 1])), 2)
            q = at(qs[lvl])
            val = torch.cat((at(c_vs[lvl - 1]), at(vs[lvl - 1])), 2) if lvl > 0 else None
            if lvl == order - 1:
                v, bias = val, None
            else:
                msg = torch.cat((at(c_msgs[order - 2 - lvl]), out), 2)
                bias = torch.cat((at(c_lses[order - 2 - lvl]), lse), 2)
                v = msg if lvl == 0 else _repeat(val, rep) * msg
                k, q = _repeat(k, rep), _repeat(q, rep) if lvl else q
            out, lse = _level64(q, k, v, bias, c, None, 0.0)
            if lvl > 0:
                out, lse = _repeat(out, c["heads"] // out.shape[1]), _repeat(lse, c["heads"] // lse.shape[1])
                lses.append(lse[:, :, 0])
                msgs.append(out[:, :, 0])
        rows.append((out, *lses, *msgs))
    joined = [torch.cat(ts) for ts in zip(*rows)]
    new = [q[:, :, 0] for q in qs[1:]] + [v[:, :, 0] for v in vs]
    return [_finish64(c, w, joined[0], root, gate), *new, *joined[1:]]


def exact(case, seed):
    c = case
    if c["kind"] == "core":
        return _core64(c, seed)
    if c["kind"] == "decode":
        return _decode64(c, seed)
    w = {k: t.double() for k, t in _layer_weights(c, seed).items()}
    x, dy, pos = _layer_inputs(c, seed)
    x = x.double()
    if c["kind"] == "infer":
        with torch.no_grad():
            parts = [_forward64(c, w, x[i:i + 1], pos) for i in range(c["b"])]

        def join(ts):
            return torch.cat(ts) if isinstance(ts[0], torch.Tensor) else tuple(join(u) for u in zip(*ts))

        return join(parts) if c["cache"] else torch.cat([p[0] for p in parts])
    # a batch row at a time: the parameters' gradients are sums over the rows
    params = [w[k].requires_grad_() for k in sorted(w)]
    outs, dxs, dws = [], [], [torch.zeros_like(p) for p in params]
    for i in range(c["b"]):
        xi = x[i:i + 1].requires_grad_()
        out, _ = _forward64(c, w, xi, pos)
        grads = torch.autograd.grad(out, [xi, *params], dy[i:i + 1].double())
        outs.append(out.detach())
        dxs.append(grads[0])
        for to, gw in zip(dws, grads[1:]):
            to += gw
    return (torch.cat(outs), torch.cat(dxs), *dws)
