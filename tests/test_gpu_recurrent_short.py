"""The short scan of a few tokens over up to 256 state rows, against float64."""

import pytest
import torch


# rows around 128 and 256, partial row groups and column tiles; one block a CU and more
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 2, 4])
@pytest.mark.parametrize("B,K,V", [(128, 128, 64), (128, 129, 60), (64, 160, 65), (64, 256, 130),
                                   (40, 255, 512)])
def test_short_scan(B, K, V, T, dtype):
    import tops.ops.gla as G

    H = 2
    gen = torch.Generator(device="cuda").manual_seed(K + V + T)
    mk = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    print(f"short scan B {B} K {K} V {V} T {T} {dtype}", flush=True)
    q, k, v = (mk(B, T, H, d).to(dtype) for d in (K, K, V))
    g = torch.nn.functional.logsigmoid(mk(B, T, H, K)).to(dtype)
    h0 = mk(B, H, K, V)
    o, ht = G.fused_recurrent_gla(q, k, v, gk=g, initial_state=h0, output_final_state=True)
    S, ref = h0.double(), []
    for t in range(T):
        S = S * g[:, t].double().exp()[..., None] \
            + k[:, t].double()[..., None] * v[:, t].double()[:, :, None]
        ref.append((q[:, t].double()[..., None] * S).sum(2) * K ** -0.5)
    ref = torch.stack(ref, 1)
    # float32 sums of K products: 2-norm error about 1e-7
    assert (o.double() - ref).norm() < 1e-6 * ref.norm()
    assert (ht.double() - S).norm() < 1e-6 * S.norm()
