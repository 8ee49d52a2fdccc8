"""float32 chunk-64 output and dv kernels (chunk_f32.hip) against float64 over their tile edges."""

import pytest
import torch


def _ref(q, k, v, g, h0, do, dht, cu):
    """float64 recurrence, token by token; gradients by autograd."""
    xs = [t.detach().double().requires_grad_(True) for t in (q, k, v, g, h0)]
    q, k, v, g, h0 = xs
    outs, hts = [], []
    scale = q.shape[-1] ** -0.5
    for i, (a, b) in enumerate(zip(cu, cu[1:])):
        S = h0[i]
        for t in range(a, b):
            S = S * g[0, t].exp()[..., None] + k[0, t][..., None] * v[0, t][:, None, :]
            outs.append((q[0, t][..., None] * S).sum(1) * scale)
        hts.append(S)
    o, ht = torch.stack(outs)[None], torch.stack(hts)
    grads = torch.autograd.grad([o, ht], xs, [do.double(), dht.double()])
    return [o, ht, *grads]


# K around 64-column tiles and 16-row contraction steps, V around 64, 128 and 256 columns,
# sequence lengths around 16-row tiles and chunks of 64
@pytest.mark.gpu
@pytest.mark.parametrize("K,V", [(4, 4), (64, 64), (60, 68), (96, 96), (128, 132), (132, 256),
                                 (100, 260), (256, 512)])
@pytest.mark.parametrize("lengths", [(1,), (64,), (17, 130, 63), (65, 48)])
def test_chunk_f32(K, V, lengths):
    import tops.ops.gla as G

    H = 2
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    T, N = cu[-1], len(lengths)
    gen = torch.Generator(device="cuda").manual_seed(K * 1000 + V + T)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    print(f"chunk f32 K {K} V {V} lengths {lengths}", flush=True)
    q, k, v, h0 = mk(1, T, H, K), mk(1, T, H, K), mk(1, T, H, V), mk(N, H, K, V)
    g = torch.nn.functional.logsigmoid(mk(1, T, H, K)) / 4
    do, dht = mk(1, T, H, V), mk(N, H, K, V)
    ref = _ref(*(t.cpu() for t in (q, k, v, g, h0, do, dht)), cu)
    xs = [t.requires_grad_(True) for t in (q, k, v, g, h0)]
    o, ht = G.chunk_gla(*xs[:4], initial_state=h0, output_final_state=True, chunk_size=64,
                        cu_seqlens=torch.tensor(cu) if N > 1 else None)
    got = [o, ht, *torch.autograd.grad([o, ht], xs, [do, dht])]
    # float32 sums of at most K + 64 products: 2-norm error about 1e-6
    for name, a, b in zip(("o", "ht", "dq", "dk", "dv", "dg", "dh0"), got, ref):
        err = (a.detach().cpu().double() - b).norm() / b.norm().clamp_min(1e-30)
        assert err < 4e-6, (name, float(err))


# chunks around the state pass's batches of 8, one and two sequences, and the rows' value columns
@pytest.mark.gpu
@pytest.mark.parametrize("V", [60, 128, 320])
@pytest.mark.parametrize("chunks", [7, 8, 9, 16, 17, 25])
def test_two_pass_states_match_the_scan(chunks, V, monkeypatch):
    """Without the workspace's last part the one-pass scan runs: the same float32 values but for
    the order of the sums and one rounding of a decay."""
    import tops.ops.gla as G
    from tops import _lib

    T, N, H, K = 64 * chunks - 5, 2, 2, 68
    gen = torch.Generator(device="cuda").manual_seed(chunks * V)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    xs = [mk(N, T, H, K), mk(N, T, H, K), mk(N, T, H, V),
          torch.nn.functional.logsigmoid(mk(N, T, H, K)) / 16, mk(N, H, K, V)]
    xs = [x.requires_grad_(True) for x in xs]
    do, dht = mk(N, T, H, V), mk(N, H, K, V)

    def run():
        o, ht = G.chunk_gla(*xs[:4], initial_state=xs[4], output_final_state=True, chunk_size=64)
        return [o, ht, *torch.autograd.grad([o, ht], xs, [do, dht])]

    two = run()
    real = _lib.seg_workspace
    part = (N * chunks * H * K * 4 + 255) // 256 * 256
    monkeypatch.setattr(_lib, "seg_workspace",
                        lambda *a, **kw: (lambda ws, n: (ws, n - part))(*real(*a, **kw)))
    for name, a, b in zip(("o", "ht", "dq", "dk", "dv", "dg", "dh0"), two, run()):
        assert (a - b).norm() < 2e-6 * b.norm(), name


# packed sequences of more chunks than the state pass's two batches of 8, short ones between them
@pytest.mark.gpu
@pytest.mark.parametrize("H,K,V", [(2, 68, 128), (1, 256, 320)])
def test_packed_sequences_longer_than_the_batches(H, K, V):
    import tops.ops.gla as G
    from torch_ref import chunk_gla_torch

    lengths = (64 * 17 + 1, 30, 64 * 9 - 5, 1, 64 * 25)
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    T, N = cu[-1], len(lengths)
    gen = torch.Generator(device="cuda").manual_seed(K + V)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    print(f"chunk f32 packed K {K} V {V} lengths {lengths}", flush=True)
    xs = [mk(1, T, H, K), mk(1, T, H, K), mk(1, T, H, V),
          torch.nn.functional.logsigmoid(mk(1, T, H, K)) / 16, mk(N, H, K, V)]
    do, dht = mk(1, T, H, V), mk(N, H, K, V)
    ys = [x.double().requires_grad_() for x in xs]
    parts = [chunk_gla_torch(*(t[:, a:b] for t in ys[:4]), h0=ys[4][i:i + 1])
             for i, (a, b) in enumerate(zip(cu, cu[1:]))]
    ref = [torch.cat([p[0] for p in parts], 1), torch.cat([p[1] for p in parts], 0)]
    ref += torch.autograd.grad(ref, ys, [do.double(), dht.double()])
    xs = [x.requires_grad_() for x in xs]
    o, ht = G.chunk_gla(*xs[:4], initial_state=xs[4], output_final_state=True,
                        cu_seqlens=torch.tensor(cu), chunk_size=64)
    got = [o, ht, *torch.autograd.grad([o, ht], xs, [do, dht])]
    # float32 sums of at most K + 64 products: 2-norm error about 1e-6
    for name, a, b in zip(("o", "ht", "dq", "dk", "dv", "dg", "dh0"), got, ref):
        err = (a.detach().double() - b).norm() / b.norm()
        assert err < 4e-6, (name, float(err))


def test_two_pass_workspace_part():
    """The decays are counted with bit 1 of `backward` alone, where the two-pass scan can run."""
    from tops import _lib

    q = _lib.load().tops_gla_chunk_ws_bytes
    part = 4 * 32 * 4 * 128 * 4
    assert q(4, 2048, 4, 128, 256, 64, 4, 0, 0, 3) == q(4, 2048, 4, 128, 256, 64, 4, 0, 0, 1) + part
    assert q(4, 2048, 4, 128, 256, 64, 4, 0, 0, 2) == q(4, 2048, 4, 128, 256, 64, 4, 0, 0, 0) + part
    for K, V, C, dt in ((388, 256, 64, 0), (128, 255, 64, 0), (128, 256, 32, 0), (128, 256, 64, 1)):
        assert q(4, 2048, 4, K, V, C, 4, 0, dt, 2) == q(4, 2048, 4, K, V, C, 4, 0, dt, 0)


@pytest.mark.gpu
def test_rows_past_a_sequence_stay_out():
    """Non-finite values in the next sequence's rows do not reach a partial chunk."""
    import tops.ops.gla as G

    T, H, K, V = 70, 1, 64, 128
    gen = torch.Generator(device="cuda").manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    q, k, v, g = mk(1, T, H, K), mk(1, T, H, K), mk(1, T, H, V), -mk(1, T, H, K).abs() / 8
    v[:, 35:] = float("inf")
    cu = torch.tensor([0, 35, T])
    o, _ = G.chunk_gla(q, k, v, g, chunk_size=64, cu_seqlens=cu)
    alone, _ = G.chunk_gla(q[:, :35], k[:, :35], v[:, :35], g[:, :35], chunk_size=64)
    assert torch.equal(o[:, :35], alone)


@pytest.mark.gpu
def test_unaligned_rows_take_the_other_kernel():
    """V of no multiple of four: the same values as the first columns of a wider call."""
    import tops.ops.gla as G

    gen = torch.Generator(device="cuda").manual_seed(6)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    q, k, v, g = mk(1, 80, 2, 64), mk(1, 80, 2, 64), mk(1, 80, 2, 68), -mk(1, 80, 2, 64).abs() / 8
    o, _ = G.chunk_gla(q, k, v, g, chunk_size=64)
    o2, _ = G.chunk_gla(q, k, v[..., :67].contiguous(), g, chunk_size=64)
    assert (o[..., :67] - o2).norm() / o2.norm() < 2e-6   # another order of float32 sums


# the steep column in the first and last 64 key columns, in whole and partial chunks: the output
# and dv kernels flag the chunk, and the recurrent kernels take the sequence and head
@pytest.mark.gpu
@pytest.mark.parametrize("V", [64, 260])
@pytest.mark.parametrize("row,col", [(0, 0), (40, 99), (129, 70)])
def test_gates_beyond_the_factors_range(row, col, V):
    import tops.ops.gla as G

    T, H, K = 130, 2, 100
    gen = torch.Generator(device="cuda").manual_seed(row + col)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    q, k, v, h0 = mk(1, T, H, K), mk(1, T, H, K), mk(1, T, H, V), mk(1, H, K, V)
    g = torch.nn.functional.logsigmoid(mk(1, T, H, K)) / 4
    g[0, row, 1, col] = -300.0
    do, dht = mk(1, T, H, V), mk(1, H, K, V)
    ref = _ref(*(t.cpu() for t in (q, k, v, g, h0, do, dht)), [0, T])
    xs = [t.requires_grad_(True) for t in (q, k, v, g, h0)]
    o, ht = G.chunk_gla(*xs[:4], initial_state=h0, output_final_state=True, chunk_size=64)
    got = [o, ht, *torch.autograd.grad([o, ht], xs, [do, dht])]
    for name, a, b in zip(("o", "ht", "dq", "dk", "dv", "dg", "dh0"), got, ref):
        assert torch.isfinite(a).all(), name
        err = (a.detach().cpu().double() - b).norm() / b.norm()
        assert err < 4e-6, (name, float(err))
