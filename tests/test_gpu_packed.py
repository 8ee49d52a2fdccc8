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


def _ref64(q, k, v, g, h0, cu):
    """Every sequence alone, in float64 on the GPU (weak gates)."""
    from torch_ref import chunk_gla_torch

    parts = [chunk_gla_torch(*(t[:, a:b] for t in (q, k, v, g)), h0=h0[i:i + 1])
             for i, (a, b) in enumerate(zip(cu, cu[1:]))]
    return torch.cat([p[0] for p in parts], 1), torch.cat([p[1] for p in parts], 0)


# 132 chunks: pieces of up to 13 where heads x V tiles are 32 (63 chunks in 5 pieces, 40 in 4, 24
# in 2; short sequences between them), of up to 7 where they are 16
LONG = [4000, 64, 1, 2500, 1500, 130]


@pytest.mark.parametrize("shape", [(32, 64, 64), (16, 128, 128), (32, 72, 128), (8, 128, 256),
                                   (4, 256, 512)], ids=lambda s: "H%dK%dV%d" % s)
def test_packed_long_pieces(shape):
    import tops.ops.gla as G
    from tops import _lib

    H, K, V = shape
    cu, N = _cu(LONG), len(LONG)
    T = cu[-1]
    print(f"packed, long pieces {shape}", flush=True)
    # the plan cuts: the workspace holds segment states
    q1 = _lib.load().tops_gla_chunk_ws_bytes
    assert q1(1, T, H, K, V, 64, N, 2, 1, 2) > q1(1, T, H, K, V, 64, N, 1, 1, 2)
    gen = torch.Generator(device="cuda").manual_seed(H + K + V)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    xs = [mk(1, T, H, K).bfloat16(), mk(1, T, H, K).bfloat16(), mk(1, T, H, V).bfloat16(),
          (torch.nn.functional.logsigmoid(mk(1, T, H, K)) / 16).bfloat16(), mk(N, H, K, V)]
    do, dht = mk(1, T, H, V).bfloat16(), mk(N, H, K, V)
    ys = [x.double().requires_grad_() for x in xs]
    ref = _ref64(*ys, cu)
    ref = [*ref, *torch.autograd.grad(list(ref), ys, [do.double(), dht.double()])]
    xs = [x.requires_grad_() for x in xs]
    o, ht = G.chunk_gla(*xs[:4], initial_state=xs[4], output_final_state=True,
                        cu_seqlens=torch.tensor(cu), chunk_size=64)
    got = [o, ht, *torch.autograd.grad([o, ht], xs, [do, dht])]
    for name, x, r in zip(("o", "ht", "dq", "dk", "dv", "dg", "dh0"), got, ref):
        err = (x.detach().double() - r).abs().max().item() / r.abs().max().item()
        assert err <= 2e-2, (name, err)


@pytest.mark.parametrize("shape", [(32, 64, 64), (8, 256, 256), (8, 256, 200)],
                         ids=lambda s: "H%dK%dV%d" % s)
def test_packed_long_pieces_head_decay(shape):
    """Scalar gates; heads wider than 128 forward only (their backward takes another path)."""
    import tops.ops.gla as G

    H, K, V = shape
    cu, N = _cu(LONG), len(LONG)
    T = cu[-1]
    print(f"packed, long pieces, per-head decay {shape}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(H + K + V)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    xs = [mk(1, T, H, K).bfloat16(), mk(1, T, H, K).bfloat16(), mk(1, T, H, V).bfloat16(),
          mk(N, H, K, V)]
    do, dht = mk(1, T, H, V).bfloat16(), mk(N, H, K, V)
    gg = -torch.rand(1, 1, H, 1, generator=gen, device="cuda") / 8 - 1e-3
    train = K <= 128
    ys = [x.double().requires_grad_(train) for x in xs]
    ref = list(_ref64(*ys[:3], gg.double().expand(1, T, H, K), ys[3], cu))
    xs = [x.requires_grad_(train) for x in xs]
    with torch.set_grad_enabled(train):
        got = list(G.chunk_gla(*xs[:3], g_gamma=gg, initial_state=xs[3], output_final_state=True,
                               cu_seqlens=torch.tensor(cu), chunk_size=64))
    if train:
        ref += torch.autograd.grad(ref, ys, [do.double(), dht.double()])
        got += torch.autograd.grad(got, xs, [do, dht])
    for name, x, r in zip(("o", "ht", "dq", "dk", "dv", "dh0"), got, ref):
        err = (x.detach().double() - r).abs().max().item() / r.abs().max().item()
        assert err <= 2e-2, (name, err)
