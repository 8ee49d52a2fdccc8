"""GPU parity of fused_recurrent_gla's bf16 forward on the matrix cores (16 tokens at a time;
sequences of 24 tokens and more, packed ones of 24 on average) against the oracle, at the float32
bar (max-abs error <= 1e-4) and at the sizes where its tiles end: tokens around multiples of 16,
key sizes around 64 / 128 / 256 and odd ones (element loads), column counts around the 16-column
tiles and the 64- and 128-column blocks, packed sequences of one token, reversed order; gates
beyond the factoring's range and non-finite inputs, which it takes as the recurrence is written."""

import numpy as np
import pytest
import torch

import oracle as orc
from gla_cases import check, logsigmoid, round_bf16, to_dev, to_np

pytestmark = pytest.mark.gpu

CASES = [
    dict(B=1, T=24, H=1, K=16, V=1),
    dict(B=2, T=31, H=3, K=63, V=17),
    dict(B=1, T=32, H=2, K=64, V=64, reverse=True),
    dict(B=1, T=33, H=2, K=65, V=65),
    dict(B=3, T=49, H=1, K=128, V=128),
    dict(B=1, T=47, H=2, K=130, V=40, reverse=True),
    dict(B=1, T=100, H=1, K=256, V=130),
    dict(B=40, T=31, H=8, K=72, V=136),                    # 32 columns a wave, partial tiles
    dict(B=64, T=40, H=5, K=40, V=128, gate="none"),
    dict(B=64, T=41, H=5, K=40, V=128, gate="none"),
    dict(B=33, T=50, H=8, K=64, V=64),                     # more blocks than CUs: the VALU scan
    dict(B=32, T=50, H=8, K=64, V=64),                     # as many
    dict(B=1, T=170, H=2, K=96, V=96, cu=[0, 1, 2, 18, 35, 36, 170]),
    dict(B=1, T=90, H=2, K=33, V=20, cu=[0, 16, 69, 70], reverse=True),   # tokens past the last
    dict(B=1, T=90, H=2, K=128, V=70, gate_mul=12.0),      # every chunk beyond the range
    dict(B=1, T=150, H=2, K=256, V=64, strong=(37, 60)),   # some chunks
    dict(B=2, T=80, H=1, K=64, V=32, strong=(20, 21), reverse=True),
    dict(B=1, T=23, H=2, K=64, V=64),                      # below: the VALU scan
]


def _inputs(c, seed=11):
    r = np.random.default_rng(seed)
    B, T, H, K, V = (c[n] for n in "BTHKV")
    q, k, v = (round_bf16(r.standard_normal((B, T, H, D))) for D in (K, K, V))
    g = logsigmoid(r.standard_normal((B, T, H, K))) * c.get("gate_mul", 1.0) / (
        1.0 if "gate_mul" in c else 4.0)
    if "strong" in c:
        g[:, slice(*c["strong"])] -= 30.0
    g = None if c.get("gate") == "none" else round_bf16(g)
    N = len(c["cu"]) - 1 if "cu" in c else B
    return q, k, v, g, r.standard_normal((N, H, K, V))


def _call(q, k, v, g, s0, c):
    import tops.ops.gla as G

    d = lambda x: None if x is None else to_dev(x, "bf16")  # noqa: E731
    cu = c.get("cu")
    o, ht = G.fused_recurrent_gla(d(q), d(k), d(v), gk=d(g), initial_state=to_dev(s0, "state"),
                                  output_final_state=True, reverse=c.get("reverse", False),
                                  cu_seqlens=None if cu is None else torch.tensor(cu))
    torch.cuda.synchronize()
    return to_np(o), to_np(ht)


def _oracle(q, k, v, g, s0, c):
    return orc.fused_recurrent_gla(q, k, v, gk=g, initial_state=s0, output_final_state=True,
                                   reverse=c.get("reverse", False), cu_seqlens=c.get("cu"))


@pytest.mark.parametrize("c", CASES, ids=lambda c: "-".join(f"{a}{b}" for a, b in c.items()))
def test_recurrent_chunk(c):
    print(f"recurrent chunk {c}", flush=True)
    x = _inputs(c)
    for name, got, ref in zip(("o", "ht"), _call(*x, c), _oracle(*x, c)):
        check(name, got, ref, "f32")


@pytest.mark.parametrize("where", ["q", "k", "v", "g", "s0"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_recurrent_chunk_non_finite(where, value):
    """A non-finite input reaches the outputs that the recurrence carries it to, and no other
    (a gate of -inf clears its row of the state)."""
    c = dict(B=1, T=50, H=2, K=64, V=40)
    x = dict(zip(("q", "k", "v", "g", "s0"), _inputs(c)))
    x[where][(0, 1, 21, 3) if where == "s0" else (0, 21, 1, 3)] = value
    print(f"recurrent chunk, {value} in {where}", flush=True)
    args = (x["q"], x["k"], x["v"], x["g"], x["s0"])
    with np.errstate(all="ignore"):
        refs = _oracle(*args, c)
    for name, got, ref in zip(("o", "ht"), _call(*args, c), refs):
        assert np.array_equal(np.isfinite(got), np.isfinite(ref)), name
        m = np.isfinite(ref)
        check(name, got[m], ref[m], "f32")


def _same_non_finite(name, got, ref):
    """The same infinities and NaN in the same places, the rest at the float32 bar."""
    assert np.array_equal(np.isnan(got), np.isnan(ref)), name
    assert np.array_equal(got == np.inf, ref == np.inf), name
    assert np.array_equal(got == -np.inf, ref == -np.inf), name
    m = np.isfinite(ref)
    check(name, got[m], ref[m], "f32")


# steps in the order of the scan: the first and last row of a 16-token chunk's halves, of the first
# chunk (which has no decay before it) and of a later one
@pytest.mark.parametrize("step", [0, 7, 8, 15, 16, 23, 24, 31])
@pytest.mark.parametrize("value", [-np.inf, -3e38, np.nan])
@pytest.mark.parametrize("c", [dict(B=1, T=50, H=2, K=64, V=40),
                               dict(B=1, T=50, H=2, K=130, V=40, reverse=True),
                               dict(B=1, T=70, H=2, K=64, V=40, cu=[0, 19, 70])],
                         ids=["forward", "reverse", "packed"])
def test_recurrent_chunk_clearing_gate(c, value, step):
    """A gate whose e^g is 0 clears its row of the state at any row of a chunk; one that is NaN
    reaches its row of the state and the outputs from there on. The row that is a chunk's first
    has its gate in the chunk's decays alone, not in its operands."""
    x = dict(zip(("q", "k", "v", "g", "s0"), _inputs(c)))
    t = c["T"] - 1 - step if c.get("reverse") else c["cu"][1] + step if "cu" in c else step
    x["g"][0, t, 1, 3] = value
    print(f"recurrent chunk {c}, gate {value} at step {step}", flush=True)
    args = (x["q"], x["k"], x["v"], x["g"], x["s0"])
    with np.errstate(all="ignore"):
        refs = _oracle(*args, c)
    for name, got, ref in zip(("o", "ht"), _call(*args, c), refs):
        _same_non_finite(name, got, ref)


@pytest.mark.parametrize("c", [dict(B=1, T=50, H=2, K=64, V=40),
                               dict(B=1, T=50, H=2, K=130, V=40, reverse=True),
                               dict(B=1, T=70, H=1, K=256, V=70, cu=[0, 30, 70]),
                               dict(B=40, T=31, H=8, K=72, V=136),
                               dict(B=1, T=900, H=2, K=96, V=40, grow=0.125, start=1.0)],
                         ids=["K64", "K130-reverse", "K256-packed", "wide-tiles", "slowly"])
def test_recurrent_chunk_state_overflows(c):
    """A state that grows out of the float range during the scan (gates of +2 on one key column of
    a state near 1e29, or of +0.125 on one near 1) gives the infinities of the recurrence in
    float32, in its value column alone: columns that stay in range, and the tokens before, keep
    their values."""
    x = dict(zip(("q", "k", "v", "g", "s0"), _inputs(c)))
    V = c["V"]
    # without keys the row only grows: no term cancels another
    x["g"][..., 3], x["q"][..., 3], x["k"][..., 3] = c.get("grow", 2.0), 1.0, 0.0
    x["s0"][..., 3, : V // 2] *= c.get("start", 1e29)
    x["s0"][..., 3, V // 2:] *= c.get("start", 1.0) * 1e-30 if "start" in c else 1.0
    x["s0"] = x["s0"].astype(np.float32).astype(np.float64)
    print(f"recurrent chunk {c}, a state that overflows", flush=True)
    args = (x["q"], x["k"], x["v"], x["g"], x["s0"])
    with np.errstate(all="ignore"):
        refs = orc.fused_recurrent_gla(*args[:3], gk=args[3], initial_state=args[4],
                                       output_final_state=True, reverse=c.get("reverse", False),
                                       cu_seqlens=c.get("cu"), dtype=np.float32)
    for name, got, ref in zip(("o", "ht"), _call(*args, c), refs):
        assert np.isinf(ref).any() and np.isfinite(ref).any()
        assert np.array_equal(np.isnan(got), np.isnan(ref)), name
        assert np.array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(ref), ref, 0)), name
        m = np.isfinite(ref)
        # T roundings of a state, and of e^g T times, 2^-23 each at most; other rows add order one
        err = np.abs(got[m] - ref[m]) / np.maximum(np.abs(ref[m]), 1.0)
        assert err.max() <= max(2e-5, c["T"] * 2 ** -22), (name, err.max())


# the chunk at which the scan leaves the matrix cores (a strong gate, or a value of v that is not
# finite or large, there): the first, another, the last, one of a packed sequence's; sizes around
# the 64-column blocks and odd ones, 32 columns a wave
@pytest.mark.parametrize("c", [dict(B=1, T=41, H=2, K=33, V=20),
                               dict(B=2, T=40, H=1, K=64, V=130, reverse=True),
                               dict(B=1, T=64, H=2, K=100, V=65),
                               dict(B=1, T=57, H=1, K=256, V=72, reverse=True),
                               dict(B=1, T=57, H=1, K=200, V=33),
                               dict(B=1, T=150, H=2, K=128, V=40, cu=[0, 37, 90, 150]),
                               dict(B=40, T=35, H=8, K=72, V=136),
                               dict(B=40, T=35, H=8, K=64, V=128, gate="none")],
                         ids=lambda c: "-".join(f"{a}{b}" for a, b in c.items()))
@pytest.mark.parametrize("at", ["first", "second", "last"])
@pytest.mark.parametrize("what", ["gate", "nan v", "large v"])
def test_recurrent_chunk_leaves_the_matrix_cores(c, at, what):
    x = dict(zip(("q", "k", "v", "g", "s0"), _inputs(c)))
    if what == "gate" and x["g"] is None:
        pytest.skip("no gates")
    t0, t1 = (c["cu"][1], c["cu"][2]) if "cu" in c else (0, c["T"])
    step = {"first": 5, "second": 16, "last": t1 - t0 - 1}[at]
    t = t1 - 1 - step if c.get("reverse") else t0 + step
    if what == "gate":
        x["g"][0, t, 0, 1::2] = -50.0
    else:
        x["v"][0, t, 0, 3] = np.nan if what == "nan v" else 2.0 ** 21
    print(f"recurrent chunk {c}, {what} in the {at} chunk", flush=True)
    args = (x["q"], x["k"], x["v"], x["g"], x["s0"])
    refs = _oracle(*args, c)
    for name, got, ref in zip(("o", "ht"), _call(*args, c), refs):
        assert np.array_equal(np.isfinite(got), np.isfinite(ref)), name
        m = np.isfinite(ref)
        # column 3 may hold the large value in sums (float32: some ulps of the largest term)
        col = np.broadcast_to(np.arange(ref.shape[-1]) == 3, ref.shape)
        check(name, got[m & ~col], ref[m & ~col], "f32")
        scale = 2.0 ** 21 if what == "large v" else 1.0
        if (m & col).any():
            check(name, got[m & col], ref[m & col], "f32", atol=max(1e-4, scale * 2 ** -18))


# strong gates at these steps of the scan: it leaves the matrix cores there and returns after 8
# chunks of 16 tokens, then after 32: once and back, twice and back, to the end in either phase
@pytest.mark.parametrize("c,steps", [
    (dict(B=1, T=300, H=2, K=64, V=40), [5]),
    (dict(B=2, T=1000, H=1, K=96, V=70), [40, 260]),
    (dict(B=1, T=999, H=1, K=256, V=64, reverse=True), [40, 260]),
    (dict(B=1, T=400, H=2, K=130, V=20), [20, 200]),
    (dict(B=40, T=330, H=8, K=72, V=136), [5, 200]),
    (dict(B=40, T=300, H=8, K=48, V=128), [130]),
    (dict(B=1, T=700, H=2, K=128, V=33, cu=[0, 290, 305, 700]), [20, 60]),
], ids=lambda x: "-".join(f"{a}{b}" for a, b in x.items()) if isinstance(x, dict) else str(x))
def test_recurrent_chunk_returns_to_the_matrix_cores(c, steps):
    x = dict(zip(("q", "k", "v", "g", "s0"), _inputs(c)))
    cu = c.get("cu", [0, c["T"]])
    for i in steps:
        for a, b in zip(cu, cu[1:]):
            if i < b - a:
                x["g"][:, b - 1 - i if c.get("reverse") else a + i, :, 2::3] = -45.0
    print(f"recurrent chunk {c}, strong gates at {steps}", flush=True)
    args = (x["q"], x["k"], x["v"], x["g"], x["s0"])
    for name, got, ref in zip(("o", "ht"), _call(*args, c), _oracle(*args, c)):
        check(name, got, ref, "f32")


@pytest.mark.parametrize("where", ["v", "s0"])
@pytest.mark.parametrize("c", [
    dict(B=1, T=300, H=2, K=64, V=40), dict(B=1, T=300, H=2, K=130, V=70, reverse=True),
    dict(B=40, T=190, H=8, K=72, V=136), dict(B=1, T=420, H=1, K=256, V=33, cu=[0, 400, 420])],
    ids=lambda c: "-".join(f"{a}{b}" for a, b in c.items()))
def test_recurrent_chunk_carries_nan(c, where):
    """A NaN in the state stays in its column, with infinities beside it, over strong gates and the
    sequence's end."""
    x = dict(zip(("q", "k", "v", "g", "s0"), _inputs(c)))
    if where == "v":
        x["v"][0, 21, 0, 3] = np.nan
    else:
        x["s0"][0, 0, 1, 3] = np.nan
        x["s0"][0, 0, 2, 4] = np.inf
    x["g"][0, 170, 0, 5] = -45.0
    x["g"][0, 185, 0, 6] = -np.inf
    print(f"recurrent chunk {c}, NaN in {where}", flush=True)
    args = (x["q"], x["k"], x["v"], x["g"], x["s0"])
    with np.errstate(all="ignore"):
        refs = _oracle(*args, c)
    for name, got, ref in zip(("o", "ht"), _call(*args, c), refs):
        _same_non_finite(name, got, ref)
