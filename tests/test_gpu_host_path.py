"""The calls' host path: the stream a kernel goes to, inputs converted on the way, and the
gradient-free forward of the gated norm against the differentiable one."""

import pytest
import torch

from tops import _lib
from tops.modules._norm import RMSNormGatedFn, rms_norm_gated
from tops.ops.gla import fused_recurrent_gla


def test_shape_errors_name_the_argument():
    q = torch.zeros(1, 2, 1, 8)
    with pytest.raises(_lib.ArgumentError, match="Expected k shape"):
        fused_recurrent_gla(q, q[:, :1], q)
    with pytest.raises(_lib.ArgumentError, match="Expected gv shape"):
        fused_recurrent_gla(q, q, q, gv=q[..., :4])
    with pytest.raises(_lib.ArgumentError, match="Expected initial_state shape"):
        fused_recurrent_gla(q, q, q, initial_state=torch.zeros(1, 1, 8, 4))


@pytest.mark.gpu
def test_current_stream():
    dev = torch.device("cuda", torch.cuda.current_device())
    assert _lib.stream_of(dev).value == (torch.cuda.current_stream(dev).cuda_stream or None)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert _lib.stream_of(dev).value == s.cuda_stream
    assert _lib.stream_of(torch.device("cuda")).value == _lib.stream_of(dev).value


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 3, 40])
def test_converted_inputs(T):
    """Strided and half-precision inputs give the bits of their float32 copies."""
    torch.manual_seed(T)
    q, k, v, g = (torch.randn(2, 4, T, 64, device="cuda").half().transpose(1, 2)
                  for _ in range(4))
    g = -g.abs() / 16
    h0 = torch.randn(2, 4, 64, 64, device="cuda").transpose(2, 3)
    a = fused_recurrent_gla(q, k, v, gk=g, initial_state=h0, output_final_state=True)
    f = [x.float().contiguous() for x in (q, k, v, g)]
    b = fused_recurrent_gla(f[0], f[1], f[2], gk=f[3], initial_state=h0.contiguous(),
                            output_final_state=True)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gated", [False, True])
def test_norm_without_gradients(dtype, gated):
    torch.manual_seed(0)
    x = torch.randn(5, 3, 96, device="cuda").to(dtype)
    g = torch.randn(5, 3, 96, device="cuda").to(dtype) if gated else None
    w = torch.randn(96, device="cuda")
    want = RMSNormGatedFn.apply(x, g, w, 1e-5)
    with torch.no_grad():
        got = rms_norm_gated(x, g, w, 1e-5)
    assert got.dtype == dtype and torch.equal(got, want)


def test_full_head_query_of_each_direction():
    """Wide heads: full-head forward (no per-chunk states without gradients), per-chunk backward."""
    from tops import _lib

    assert _lib.full_head(256, 512, 64, torch.bfloat16, False)
    assert not _lib.full_head(256, 512, 64, torch.bfloat16, True)
    assert _lib.full_head(128, 128, 64, torch.bfloat16, True)
    assert not _lib.full_head(128, 128, 64, torch.float32, False)
