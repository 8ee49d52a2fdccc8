"""GPU parity of packed (varlen) sequences cut into segments: lengths around the segment and
chunk boundaries, against the oracle at the bf16 bar (max-abs error / max |ref| <= 2e-2).

The full-head kernels cut a packed sequence of more chunks than the plan's segment (at least
5 chunks of 64) into pieces that run in parallel, each folding its entry state from the
pieces before it; wide heads also stream the per-chunk gating workspace."""

import pytest
import torch

import oracle as orc
from gla_cases import check, make_inputs, round_bf16, to_dev, to_np

pytestmark = pytest.mark.gpu

# one piece / exactly one full piece / one row over / several pieces, one-row pieces at the end;
# sequences of one token between long ones; a single long sequence
LENS = {
    "edges": [320, 321, 1, 640, 641, 64, 65, 63],
    "long_between": [1, 1500, 1, 1, 970, 2],
    "one": [2049],
}
SHAPES = [(2, 128, 128), (1, 64, 40), (3, 72, 128), (2, 128, 256), (1, 256, 192), (1, 256, 72)]


def _cu(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


def _run(H, K, V, lens, seed, strong=None):
    import tops.ops.gla as G

    cu = _cu(lens)
    T, N = cu[-1], len(lens)
    q, k, v, g, s0, do, dht = make_inputs(1, T, H, K, V, seed, gate_div=16.0, h0=True, dht=True,
                                          N=N, dtype="bf16")
    if strong is not None:   # per-token decays near 4 in these tokens: beyond the factoring
        g[:, strong[0]:strong[1]] = round_bf16(g[:, strong[0]:strong[1]] * 80.0)
    tq, tk, tv, tg = (to_dev(x, "bf16").requires_grad_() for x in (q, k, v, g))
    th0 = to_dev(s0, "state").requires_grad_()
    o, ht = G.chunk_gla(tq, tk, tv, tg, initial_state=th0, output_final_state=True,
                        cu_seqlens=torch.tensor(cu), chunk_size=64)
    grads = torch.autograd.grad([o, ht], [tq, tk, tv, tg, th0],
                                [to_dev(do, "bf16"), to_dev(dht, "state")])
    with torch.no_grad():   # no gradients wanted: the forward that keeps no states
        o2, ht2 = G.chunk_gla(tq, tk, tv, tg, initial_state=th0, output_final_state=True,
                              cu_seqlens=torch.tensor(cu), chunk_size=64)
    torch.cuda.synchronize()
    on, hn = orc.naive_recurrent_gla(q, k, v, g, initial_state=s0, output_final_state=True,
                                     cu_seqlens=cu)
    ref = orc.chunk_gla_bwd(q, k, v, g, None, None, K ** -0.5, s0, None, None, do, dht,
                            cu_seqlens=cu, chunk_size=16)
    names = ["o", "ht", "o (no grad)", "ht (no grad)", "dq", "dk", "dv", "dg", "dh0"]
    for name, x, r in zip(names, [o, ht, o2, ht2, *grads], [on, hn, on, hn, *ref]):
        check(name, to_np(x), r, "bf16")


@pytest.mark.parametrize("lens", list(LENS), ids=list(LENS))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "H%dK%dV%d" % s)
def test_packed_segments(shape, lens):
    print(f"packed {shape} {LENS[lens]}", flush=True)
    _run(*shape, LENS[lens], seed=71)


@pytest.mark.parametrize("shape", [(2, 128, 128), (1, 256, 192)], ids=lambda s: "H%dK%dV%d" % s)
def test_packed_segments_strong_gates(shape):
    """The gate-range flags of one sequence's middle piece reach the recurrent fallback."""
    lens = [330, 70, 1400, 5, 400]
    print(f"packed, strong gates {shape} {lens}", flush=True)
    _run(*shape, lens, seed=72, strong=(1000, 1100))


def test_packed_segments_head_decay():
    import tops.ops.gla as G

    H, K, V = 2, 128, 128
    lens = LENS["long_between"]
    cu = _cu(lens)
    print(f"packed, per-head decay {lens}", flush=True)
    q, k, v, _, s0, do, dht = make_inputs(1, cu[-1], H, K, V, 73, h0=True, dht=True,
                                          N=len(lens), dtype="bf16")
    gg = torch.tensor([-0.03, -0.5]).reshape(1, 1, H, 1)
    xs = [to_dev(x, "bf16").requires_grad_() for x in (q, k, v)]
    th0 = to_dev(s0, "state").requires_grad_()
    o, ht = G.chunk_gla(*xs, g_gamma=gg.cuda(), initial_state=th0, output_final_state=True,
                        cu_seqlens=torch.tensor(cu), chunk_size=64)
    grads = torch.autograd.grad([o, ht], [*xs, th0],
                                [to_dev(do, "bf16"), to_dev(dht, "state")])
    torch.cuda.synchronize()
    g = gg.expand(1, cu[-1], H, K).double().numpy()
    on, hn = orc.naive_recurrent_gla(q, k, v, g, initial_state=s0, output_final_state=True,
                                     cu_seqlens=cu)
    ref = orc.chunk_gla_bwd(q, k, v, g, None, None, K ** -0.5, s0, None, None, do, dht,
                            cu_seqlens=cu, chunk_size=16)
    refs = [on, hn, ref[0], ref[1], ref[2], ref[4]]
    for name, x, r in zip(["o", "ht", "dq", "dk", "dv", "dh0"], [o, ht, *grads], refs):
        check(name, to_np(x), r, "bf16")
