"""The layer's few-row kernels: projections and low-rank gate against float64, and the decode
step through them against the same layer taking one library call per projection."""

import pytest
import torch


def _close(got, ref, tol):
    err = (got.double() - ref).abs().max().item() / ref.abs().max().item()
    assert err <= tol, err


# rows around the 16-row tiles; weight rows below, at and above a 16-row tile
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 64, 65, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_small_linear(rows, dtype):
    from tops.layers.gla import _small_linear

    gen = torch.Generator(device="cuda").manual_seed(rows)
    for K in (256, 1280):
        print(f"small linear rows {rows} K {K} {dtype}", flush=True)
        x = torch.randn(rows, K, generator=gen, device="cuda").to(dtype)
        ws = [torch.randn(n, K, generator=gen, device="cuda").bfloat16() for n in (4, 16, 100)]
        ys = _small_linear(x, ws, (1,) if dtype == torch.bfloat16 else ())
        for i, (y, w) in enumerate(zip(ys, ws)):
            ref = x.double() @ w.double().t()
            if dtype == torch.float32:   # float32 sums of K products
                assert y.dtype == torch.float32
                _close(y, ref, 1e-6)
            else:   # one rounding to bf16
                assert y.dtype == (torch.float32 if i == 1 else torch.bfloat16)
                assert torch.equal(y.bfloat16().to(y.dtype), y)
                _close(y, ref, 2 ** -8)


@pytest.mark.gpu
def test_small_linear_scratch_values():
    """float32 rows with infinities, NaN and values above the largest bfloat16 (3.3895e38): as
    F.linear in float32 gives them (weights of +-1 and powers of two: exact products)."""
    import torch.nn.functional as F

    from tops.layers.gla import _small_linear

    x = torch.zeros(6, 256, device="cuda")
    x[0, 3], x[1, 3], x[2, 3] = float("inf"), float("-inf"), float("nan")
    x[3, 3], x[4, 3], x[5, 200] = 3.4e38, -3.4028234663852886e38, 1e-30
    w = torch.full((16, 256), 0.5, device="cuda").bfloat16()
    w[1] = -1.0
    y = _small_linear(x, [w])[0]
    assert torch.equal(torch.nan_to_num(y, 7.0), torch.nan_to_num(F.linear(x, w.float()), 7.0))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 20])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_small_linear_non_finite_weights(rows, value):
    """A weight that is not finite meets x as in F.linear, also where x is a bfloat16 value (one
    that needs no second and third part), 0 or infinite; other outputs keep their values."""
    import torch.nn.functional as F

    from tops.layers.gla import _small_linear

    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, 512, generator=gen, device="cuda")
    x[:, 3] = torch.tensor([1.5, 0.1, -2.0, 0.0, -0.3], device="cuda").repeat(4)[:rows]
    x[-1, 300] = float("inf")
    w = torch.randn(16, 512, generator=gen, device="cuda").bfloat16()
    w[2, 3] = w[5, 300] = value
    print(f"small linear, {value} in the weights, {rows} rows", flush=True)
    y, ref = _small_linear(x, [w])[0], F.linear(x, w.float())
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(y), inf) and torch.equal(y[inf], ref[inf])
    m = torch.isfinite(ref)
    # float32 sums of 512 products, largest sums about 100
    assert (y[m] - ref[m]).abs().max().item() <= 1e-4 if m.any() else True


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,clamp,bias", [(1, 256, None, True), (5, 300, -0.03, True),
                                               (128, 1024, None, False)])
def test_low_rank_gate(rows, n, clamp, bias):
    from tops.layers.gla import Linear, _low_rank_gate
    from tops.modules._norm import GateLogSigmoidFn

    gen = torch.Generator(device="cuda").manual_seed(n)
    up = Linear(16, n, bias, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        for p in up.parameters():
            p.copy_(torch.randn(p.shape, generator=gen, device="cuda"))
        x = torch.randn(1, rows, 16, generator=gen, device="cuda").bfloat16()
        y = _low_rank_gate(x, up, 16.0, clamp)
        # the product may round to the next bf16: then so may the gate
        ref = GateLogSigmoidFn.apply(up(x), 16.0, clamp)
        assert y.shape == ref.shape and y.dtype == ref.dtype
        _close(y, ref.double(), 2 ** -7)


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", [
    dict(hidden_size=1024, num_heads=4),
    dict(hidden_size=512, num_heads=4, num_kv_heads=2, use_output_gate=False),
    dict(hidden_size=512, num_heads=2, use_short_conv=True, fuse_norm=False, clamp_min=-0.1),
], ids=["default", "gqa-nogate", "conv-unfused"])
@pytest.mark.parametrize("batch,tokens", [(1, 1), (33, 1), (2, 40), (1, 100)])
def test_decode_step_matches_library_path(cfg, batch, tokens):
    from tops.layers import GatedLinearAttention
    from tops.layers.gla import LayerCache

    m = GatedLinearAttention(rngs=3, dtype=torch.bfloat16, device="cuda", layer_idx=0, **cfg)
    gen = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.randn(batch, tokens, cfg["hidden_size"], generator=gen, device="cuda").bfloat16()
    outs = []
    with torch.no_grad():
        for hooked in (False, True):
            if hooked:   # a hook on a projection keeps every call on the library path
                for lin in (m.q_proj, m.gk_proj[1], m.o_proj):
                    lin.register_forward_hook(lambda *a: None)
            cache = LayerCache()
            o, _, cache = m(x, past_key_values=cache, use_cache=True)
            o2, _, cache = m(x, past_key_values=cache, use_cache=True)
            outs.append([o, o2, cache[0]["recurrent_state"]])
    for a, b in zip(*outs):
        assert a.shape == b.shape and a.dtype == b.dtype
        _close(a, b.double(), 2e-2)


def _layer(hidden=256):
    from tops.layers import GatedLinearAttention

    return GatedLinearAttention(rngs=3, dtype=torch.bfloat16, layer_idx=0, hidden_size=hidden,
                                num_heads=2)


def test_few_row_route_takes_plain_projections_only():
    """What the few-row kernels would not see keeps the library path: a weight of another width
    (F.linear's error), another forward, hooks."""
    from tops.layers.gla import _plain_gate, _plain_linear

    m, x = _layer(), torch.zeros(1, 1, 256, dtype=torch.bfloat16)
    low = torch.zeros(1, 1, 16, dtype=torch.bfloat16)
    assert _plain_linear(m.q_proj, x) and _plain_gate(m.gk_proj[1], low)
    assert not _plain_linear(m.q_proj, torch.zeros(1, 1, 512, dtype=torch.bfloat16))
    assert not _plain_gate(m.gk_proj[1], x)
    assert not _plain_linear(m.gk_proj[1], low)   # has a bias
    m.q_proj.forward = lambda t: t
    m.k_proj.register_forward_hook(lambda *a: None)
    m.gk_proj[1].bias = torch.nn.Parameter(m.gk_proj[1].bias.detach()[:8])
    assert not _plain_linear(m.q_proj, x) and not _plain_linear(m.k_proj, x)
    assert not _plain_gate(m.gk_proj[1], low)


def test_few_row_route_leaves_wide_ranks_and_empty_weights():
    """Sizes that the entry points refuse keep the library path: a gate rank above 4096, a weight
    without rows."""
    from tops.layers.gla import Linear, _plain_gate, _plain_linear

    low = torch.zeros(1, 1, 4104, dtype=torch.bfloat16)
    assert _plain_gate(Linear(4096, 8, True, dtype=torch.bfloat16), low[..., :4096])
    assert not _plain_gate(Linear(4104, 8, True, dtype=torch.bfloat16), low)
    x = torch.zeros(1, 1, 256, dtype=torch.bfloat16)
    lin = Linear(256, 4, dtype=torch.bfloat16)
    assert _plain_linear(lin, x)
    lin.weight = torch.nn.Parameter(lin.weight.detach()[:0])
    assert not _plain_linear(lin, x)


@pytest.mark.gpu
def test_norm_gate_hooks_see_the_gate_in_its_own_dtype():
    """A hooked or replaced gated norm gets the output gate as g_proj gives it, and the layer's
    result with a hook that only looks is the one without."""
    m = _layer().cuda()
    x = torch.randn(2, 1, 256, generator=torch.Generator("cuda").manual_seed(1),
                    device="cuda").bfloat16()
    with torch.no_grad():
        plain = m(x)[0]
        seen = []
        h = m.g_norm_swish_gate.register_forward_pre_hook(
            lambda mod, a: seen.append([t.dtype for t in a]))
        hooked = m(x)[0]
        h.remove()
        inner = m.g_norm_swish_gate

        class Norm(torch.nn.Module):
            def forward(self, o, g):
                seen.append([o.dtype, g.dtype])
                return inner(o, g)

        m.g_norm_swish_gate = Norm()
        replaced = m(x)[0]
    assert seen == [[torch.float32, torch.bfloat16]] * 2
    assert torch.equal(plain, hooked) and torch.equal(plain, replaced)


@pytest.mark.gpu
def test_few_row_route_leaves_tangents_and_global_hooks():
    import torch.autograd.forward_ad as fwd
    from torch.nn.modules.module import register_module_forward_hook

    m = _layer().cuda()
    x = torch.ones(1, 1, 256, device="cuda").bfloat16()
    from tops.layers.gla import _small_rows

    with torch.no_grad():
        assert _small_rows(x)
        with fwd.dual_level():
            assert not _small_rows(x)
        seen = []
        h = register_module_forward_hook(lambda mod, a, o: seen.append(mod))
        try:
            m(x)
        finally:
            h.remove()
        assert any(s is m.q_proj for s in seen) and any(s is m.o_proj for s in seen)


def test_entry_points_refuse_bad_arguments():
    """Host checks (no GPU call is made)."""
    import ctypes

    from tops import _lib

    lib = _lib.load()
    arr = lambda t, *v: (t * len(v))(*v)  # noqa: E731
    P, I64 = ctypes.c_void_p, ctypes.c_int64

    def rc(dt=1, n=64, nw=1, M=4, K=256, x=4096, w=4096):
        return lib.tops_gla_small_linear(x, dt, arr(P, w), arr(I64, n), nw, M, K, arr(P, 4096),
                                         0, None)

    assert rc(dt=7) == 1 and rc(nw=9) == 1 and rc(x=None) == 1 and rc(w=8) == 1
    assert rc(M=129) == 2 and rc(K=128) == 2 and rc(n=6) == 2
    gate = lib.tops_gla_low_rank_gate
    assert gate(4096, 4096, None, 4096, 1, 8, 12, 16.0, 0, 0.0, None) == 2
    assert gate(4096, 4096, None, 4096, 1, 8, 16, 0.0, 0, 0.0, None) == 1
    assert gate(None, 4096, None, 4096, 1, 8, 16, 16.0, 0, 0.0, None) == 1
