"""Performance cases of the GLA framework: the calls a program makes, over the range it makes them.

Three kinds of case, each through the public entry points:

* ``recurrent``: ``fused_recurrent_gla`` forward, from single-token decoding to long sequences;
* ``chunk``    : ``chunk_gla``, forward only (prefill) or forward + backward (training), fixed
                 length or packed sequences, bfloat16 or float32, per-key or per-head gates;
* ``layer``    : ``GatedLinearAttention``, a training step's forward + backward or one decode
                 step with its cache.

A case is a dict of plain values; ``lengths`` (text) gives the packed sequences' lengths.
"""

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "pallas-kernel_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _lengths(total, parts):
    """Text of `parts` shares of `total` tokens (each at least one)."""
    s = sum(parts)
    out = [max(1, int(total * p / s)) for p in parts]
    out[-1] += max(0, total - sum(out))
    return ",".join(str(n) for n in out)


def listed():
    return [
        # one user's next token: 4 wide heads, the smallest call there is
        dict(name="decode_one", kind="recurrent", B=1, T=1, H=4, K=256, V=512, dtype="bf16"),
        # the next token of a serving batch
        dict(name="decode_batch", kind="recurrent", B=64, T=1, H=16, K=128, V=128, dtype="bf16"),
        # short prompts and drafted tokens of a serving batch (the layer's path up to 64 tokens)
        dict(name="short_prompts", kind="recurrent", B=64, T=64, H=16, K=128, V=128,
             dtype="bf16"),
        # a long recurrent pass with final state
        dict(name="recurrent_long", kind="recurrent", B=8, T=2048, H=4, K=256, V=512,
             dtype="bf16"),
        # training on fixed-length sequences, 16 heads of 128 x 128 (the headline workload)
        dict(name="train", kind="chunk", B=4, T=8192, H=16, K=128, V=128, dtype="bf16",
             train=True, gate="key", lengths=""),
        # training on documents of very different lengths packed into one row
        dict(name="train_packed", kind="chunk", B=1, T=16384, H=16, K=128, V=128, dtype="bf16",
             train=True, gate="key",
             lengths="4821,96,1307,33,2650,711,5,1984,402,1023,640,188,2524"),
        # float32 training, the layer's default head sizes (hidden 1024, 4 heads)
        dict(name="train_float32", kind="chunk", B=4, T=2048, H=4, K=128, V=256, dtype="f32",
             train=True, gate="key", lengths=""),
        # training with one constant decay per head
        dict(name="train_head_decay", kind="chunk", B=4, T=8192, H=16, K=128, V=128,
             dtype="bf16", train=True, gate="head", lengths=""),
        # prefill of a batch of prompts, wide heads
        dict(name="prefill", kind="chunk", B=8, T=4096, H=4, K=256, V=512, dtype="bf16",
             train=False, gate="key", lengths=""),
        # prefill of prompts of different lengths packed into one row, wide heads
        dict(name="prefill_packed", kind="chunk", B=1, T=8192, H=4, K=256, V=512, dtype="bf16",
             train=False, gate="key", lengths="1733,290,2049,77,3001,512,530"),
        # a training step's attention layer
        dict(name="layer_train", kind="layer", B=2, T=16384, hidden=2048, H=4, dtype="bf16",
             train=True, conv=False),
        # the attention layer of one decode step of a serving batch
        dict(name="layer_decode", kind="layer", B=32, T=1, hidden=2048, H=4, dtype="bf16",
             train=False, conv=False),
    ]


# (heads, key size, value size) that models come with; 96 is no power of two
HEADS = [(4, 256, 512), (16, 128, 128), (4, 128, 256), (8, 64, 128), (16, 64, 64), (6, 96, 96)]
# the largest listed case (layer_train) bounds the drawn ones: tokens x heads x K x V of the
# attention core, forward and backward counted alike
LARGEST = 2 * 16384 * 4 * 256 * 512


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _documents(rng, total):
    n = _log(rng, 3, 24)
    return _lengths(total, [rng.lognormvariate(0.0, 1.2) for _ in range(n)])


def draw(rng):
    """A case of the listed ones' ranges: decode, recurrent and chunked calls, layers."""
    what = rng.choice(["decode", "decode", "recurrent", "recurrent", "train", "train", "packed",
                       "float32", "head", "prefill", "prefill_packed", "layer", "step"])
    H, K, V = rng.choice(HEADS)
    if what == "decode":
        return dict(kind="recurrent", B=_log(rng, 1, 128), T=rng.choice([1, 1, 1, 2, 4]), H=H, K=K,
                    V=V, dtype=rng.choice(["bf16", "bf16", "f32"]))
    if what == "recurrent":
        T = _log(rng, 5, 2048)
        most = max(1, 8 * 2048 * 4 * 256 * 512 // (T * H * K * V))
        return dict(kind="recurrent", B=_log(rng, 1, min(64, most)), T=T, H=H, K=K, V=V,
                    dtype="bf16")
    if what in ("train", "head", "float32", "prefill"):
        train = what != "prefill"
        if what == "head":   # the reference's simple GLA has heads of 128 x 128
            H, K, V = 16, 128, 128
        T = _log(rng, 200, 2048 if what == "float32" else 16384)
        most = (4 * 2048 * 4 * 128 * 256 if what == "float32" else LARGEST // 2) // (T * H * K * V)
        return dict(kind="chunk", B=_log(rng, 1, min(16, max(1, most))), T=T, H=H, K=K, V=V,
                    dtype="f32" if what == "float32" else "bf16", train=train,
                    gate="head" if what == "head" else "key", lengths="")
    if what in ("packed", "prefill_packed"):
        most = min(16384, LARGEST // 2 // (H * K * V))
        lengths = _documents(rng, _log(rng, 1000, most))
        return dict(kind="chunk", B=1, T=sum(int(n) for n in lengths.split(",")), H=H, K=K, V=V,
                    dtype="bf16", train=what == "packed", gate="key", lengths=lengths)
    hidden = rng.choice([1024, 2048])
    if what == "layer":
        T = _log(rng, 256, 8192)
        return dict(kind="layer", B=_log(rng, 1, max(1, 16384 // T)), T=T, hidden=hidden, H=4,
                    dtype="bf16", train=True, conv=rng.random() < 0.3)
    return dict(kind="layer", B=_log(rng, 1, 128), T=1, hidden=hidden, H=4, dtype="bf16",
                train=False, conv=False)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _cu(case):
    """Offsets of the packed sequences, or None."""
    if not case.get("lengths"):
        return None
    cu = [0]
    for n in case["lengths"].split(","):
        cu.append(cu[-1] + int(n))
    return cu


def _attention_inputs(case, seed):
    """q, k, v ~ N(0, 1), gates logsigmoid(N(0, 1)) / 16, states ~ N(0, 0.1^2)."""
    B, T, H, K, V = (case[n] for n in "BTHKV")
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device=DEV).manual_seed(seed)

    def mk(*shape):
        return torch.randn(*shape, generator=gen, device=DEV)

    cu = _cu(case)
    N = B if cu is None else len(cu) - 1
    x = {"q": mk(B, T, H, K).to(dt), "k": mk(B, T, H, K).to(dt), "v": mk(B, T, H, V).to(dt)}
    if case.get("gate") == "head":   # a decay per head, from fast to slow
        r = torch.rand(H, generator=gen, device=DEV)
        decay = torch.exp2(-3.0 - 5.0 * torch.arange(H, device=DEV) / H - r)
        x["g_gamma"] = -decay.reshape(1, 1, H, 1)
    else:
        x["g"] = (torch.nn.functional.logsigmoid(mk(B, T, H, K)) / 16).to(dt)
    x["h0"] = 0.1 * mk(N, H, K, V)
    if case.get("train"):
        x["do"] = mk(B, T, H, V).to(dt)
        x["dht"] = 0.1 * mk(N, H, K, V)
    return x


def _layer_sizes(case):
    hidden, H = case["hidden"], case["H"]
    return hidden // 2, hidden, hidden // 2 // H, hidden // H   # key dim, value dim, per head


def _layer_inputs(case, seed):
    """Weights ~ N(0, 1 / fan in), hidden states ~ N(0, 1) (after the block's norm)."""
    B, T, hidden, H = case["B"], case["T"], case["hidden"], case["H"]
    kd, vd, K, V = _layer_sizes(case)
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device=DEV).manual_seed(seed)

    def mk(*shape, std=1.0):
        return torch.randn(*shape, generator=gen, device=DEV) * std

    s = hidden ** -0.5
    w = {"q_proj.weight": mk(kd, hidden, std=s).to(dt), "k_proj.weight": mk(kd, hidden, std=s).to(dt),
         "v_proj.weight": mk(vd, hidden, std=s).to(dt), "g_proj.weight": mk(vd, hidden, std=s).to(dt),
         "gk_proj.0.weight": mk(16, hidden, std=s).to(dt),
         "gk_proj.1.weight": mk(kd, 16, std=0.25).to(dt),
         "gk_proj.1.bias": mk(kd, std=0.5).to(dt), "o_proj.weight": mk(hidden, vd, std=s).to(dt),
         "g_norm_swish_gate.weight": 1.0 + mk(V, std=0.1)}
    if case["conv"]:
        for n, d in (("q", kd), ("k", kd), ("v", vd)):
            w[n + "_conv1d.weight"] = mk(d, 1, 4, std=0.5).to(dt)
    x = {"x": mk(B, T, hidden).to(dt)}
    if case["train"]:
        x["do"] = mk(B, T, hidden).to(dt)
    else:
        x["state"] = mk(B, H, K, V)   # the cache after a prompt
    return w, x


def prepare(case, seed):
    if case["kind"] != "layer":
        x = _attention_inputs(case, seed)
        cu = _cu(case)
        st = dict(case=case, x=x, cu=None if cu is None else torch.tensor(cu, dtype=torch.int32))
        if case.get("train"):
            for n in ("q", "k", "v", "g", "h0"):
                if n in x:
                    x[n].requires_grad_(True)
        return st
    from tops.layers import GatedLinearAttention

    w, x = _layer_inputs(case, seed)
    layer = GatedLinearAttention(hidden_size=case["hidden"], num_heads=case["H"], expand_k=0.5,
                                 expand_v=1.0, use_short_conv=case["conv"], layer_idx=0, rngs=0,
                                 dtype=DTYPES[case["dtype"]], device=DEV)
    layer.load_state_dict(w)
    if case["train"]:
        x["x"].requires_grad_(True)
    else:
        layer.requires_grad_(False)
    return dict(case=case, layer=layer, x=x,
                params=[p for _, p in sorted(layer.named_parameters())])


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(state):
    case, x = state["case"], state["x"]
    if case["kind"] == "layer":
        return _run_layer(state)
    import tops.ops.gla as G

    if case["kind"] == "recurrent":
        with torch.no_grad():
            o, ht = G.fused_recurrent_gla(x["q"], x["k"], x["v"], gk=x["g"],
                                          initial_state=x["h0"], output_final_state=True)
        return {"o": o, "ht": ht}
    with torch.set_grad_enabled(case["train"]):
        o, ht = G.chunk_gla(x["q"], x["k"], x["v"], x.get("g"), x.get("g_gamma"),
                            initial_state=x["h0"], output_final_state=True,
                            cu_seqlens=state["cu"], chunk_size=64)
    if not case["train"]:
        return {"o": o, "ht": ht}
    names = [n for n in ("q", "k", "v", "g", "h0") if n in x]
    grads = torch.autograd.grad([o, ht], [x[n] for n in names], [x["do"], x["dht"]])
    return {"o": o.detach(), "ht": ht.detach(), **dict(zip(names, grads))}


def _run_layer(state):
    from tops.layers.gla import LayerCache

    case, x, layer = state["case"], state["x"], state["layer"]
    if case["train"]:
        o, _, _ = layer(x["x"])
        grads = torch.autograd.grad(o, [x["x"], *state["params"]], x["do"])
        return {"o": o.detach(), "grads": list(grads)}
    with torch.no_grad():
        cache = LayerCache()
        cache.update(recurrent_state=x["state"])
        o, _, cache = layer(x["x"], past_key_values=cache, use_cache=True)
        return {"o": o, "state": cache[0]["recurrent_state"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    es = 2 if case["dtype"] == "bf16" else 4
    B, T, H = case["B"], case["T"], case["H"]
    if case["kind"] == "layer":
        kd, vd, K, V = _layer_sizes(case)
        hidden, tok = case["hidden"], B * T
        weights = hidden * (2 * kd + 3 * vd + 16) + 16 * kd + kd + V
        core = tok * H * 4 * K * V
        if case["train"]:   # x, do, o, dx; weights read and their gradients written
            return {"bytes": 4 * tok * hidden * es + 2 * weights * es,
                    "flops": 3 * (2 * tok * weights + core)}
        return {"bytes": 2 * tok * hidden * es + weights * es + 2 * B * H * K * V * 4,
                "flops": 2 * tok * weights + core}
    K, V = case["K"], case["V"]
    tok, cu = B * T * H, _cu(case)
    states = (B if cu is None else len(cu) - 1) * H * K * V * 4
    if case["kind"] == "recurrent":   # o is float32
        return {"bytes": tok * ((3 * K + V) * es + 4 * V) + 2 * states, "flops": tok * 4 * K * V}
    gate = 0 if case["gate"] == "head" else K
    fwd = {"bytes": tok * (2 * K + gate + 2 * V) * es + 2 * states,
           "flops": tok * (4 * K * V + 2 * 64 * (K + V))}
    if not case["train"]:
        return fwd
    # q, k, v, gates and do in; o and the gradients out; h0 and dht in, ht and dh0 out
    return {"bytes": tok * (4 * K + 2 * gate + 4 * V) * es + 4 * states, "flops": 3 * fwd["flops"]}


def tolerance(case):
    """About four times the error measured against ``exact``: 1.8e-7 for the recurrent path's
    float32 sums, 4.5e-7 for the chunked ones, 3.4e-3 in bfloat16, 6.5e-3 through a layer."""
    if case["kind"] == "recurrent":
        return {"rel": 1e-6, "max": 1e-4}
    if case["kind"] == "layer":
        return {"rel": 0.025, "max": 0.5}
    if case["dtype"] == "f32":
        return {"rel": 2e-6, "max": 1e-3}
    return {"rel": 0.014, "max": 0.4}


# ---------------------------------------------------------------------------
# the same values in 64 bits
# ---------------------------------------------------------------------------


def _gla64(q, k, v, g, h0, C=64):
    """Chunked GLA in float64, one batch of sequences of one length: (o, final state)."""
    B, T, H, K = q.shape
    V = v.shape[-1]

    def split(t):   # [B, T, H, D] -> T / C chunks of [B * H, C, D]
        D = t.shape[-1]
        t = torch.nn.functional.pad(t, (0, 0, 0, 0, 0, -T % C))
        return t.permute(1, 0, 2, 3).reshape(-1, C, B * H, D).transpose(1, 2).unbind(0)

    mask = torch.ones(C, C, dtype=torch.float64, device=q.device).tril()
    S = h0.reshape(B * H, K, V)
    out = []
    for qc, kc, vc, gc in zip(split(q * K ** -0.5), split(k), split(v), split(g)):
        G = gc.cumsum(1)
        ref = G[:, -1:] / 2   # the factors stay within e^{|chunk's decay| / 2}
        qg, kg = qc * (G - ref).exp(), kc * (ref - G).exp()
        A = (qg @ kg.transpose(1, 2)) * mask
        out.append(A @ vc + (qc * G.exp()) @ S)
        S = G[:, -1].exp()[..., None] * S + (kc * (G[:, -1:] - G).exp()).transpose(1, 2) @ vc
    o = torch.stack(out).transpose(1, 2).reshape(-1, B, H, V)[:T].permute(1, 0, 2, 3)
    return o, S.reshape(B, H, K, V)


def _gla64_any(q, k, v, g, h0, cu):
    if cu is None:
        return _gla64(q, k, v, g, h0)
    parts = [_gla64(*(t[:, a:b] for t in (q, k, v, g)), h0[i:i + 1])
             for i, (a, b) in enumerate(zip(cu, cu[1:]))]
    return torch.cat([p[0] for p in parts], 1), torch.cat([p[1] for p in parts], 0)


def exact(case, seed):
    if case["kind"] == "layer":
        return _exact_layer(case, seed)
    x = {n: t.double() for n, t in _attention_inputs(case, seed).items()}
    train = bool(case.get("train"))
    names = [n for n in ("q", "k", "v", "g", "h0") if n in x]
    for n in names:
        x[n].requires_grad_(train)
    with torch.set_grad_enabled(train):
        g = x["g"] if "g" in x else x["g_gamma"].expand(x["q"].shape)
        o, ht = _gla64_any(x["q"], x["k"], x["v"], g, x["h0"], _cu(case))
    if not train:
        return {"o": o, "ht": ht}
    grads = torch.autograd.grad([o, ht], [x[n] for n in names], [x["do"], x["dht"]])
    return {"o": o.detach(), "ht": ht.detach(), **dict(zip(names, grads))}


def _conv64(x, w):
    """Causal depthwise convolution over time and SiLU."""
    W = w.shape[-1]
    p = torch.nn.functional.pad(x, (0, 0, W - 1, 0))
    y = sum(p[:, i:i + x.shape[1]] * w[:, 0, i] for i in range(W))
    return torch.nn.functional.silu(y)


def _exact_layer(case, seed):
    w, x = _layer_inputs(case, seed)
    train, H = case["train"], case["H"]
    w = {n: t.double().requires_grad_(train) for n, t in w.items()}
    h = x["x"].double().requires_grad_(train)
    B, T, _ = h.shape
    _, _, K, V = _layer_sizes(case)
    with torch.set_grad_enabled(train):
        q, k, v, gate = (h @ w[n + "_proj.weight"].t() for n in "qkvg")
        gk = (h @ w["gk_proj.0.weight"].t()) @ w["gk_proj.1.weight"].t() + w["gk_proj.1.bias"]
        if case["conv"]:
            q, k, v = (_conv64(t, w[n + "_conv1d.weight"]) for t, n in ((q, "q"), (k, "k"), (v, "v")))
        g = torch.nn.functional.logsigmoid(gk) / 16
        s0 = x["state"].double() if "state" in x else h.new_zeros(B, H, K, V)
        q, k, g, v = (t.reshape(B, T, H, -1) for t in (q, k, g, v))
        o, s = _gla64(q, k, v, g, s0)
        o = o * (o.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * w["g_norm_swish_gate.weight"]
        o = (o * torch.nn.functional.silu(gate.reshape(B, T, H, V))).reshape(B, T, H * V)
        o = o @ w["o_proj.weight"].t()
    if not train:
        return {"o": o, "state": s}
    grads = torch.autograd.grad(o, [h] + [w[n] for n in sorted(w)], x["do"].double())
    return {"o": o.detach(), "grads": list(grads)}
