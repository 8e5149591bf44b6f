"""What the training gradient's bf16 roundings rest on: the order of the sums in
front of them and the library's erff and expf.

A last-place difference in front of a rounding to bf16 is another value for every
layer behind it, so these are compared bit for bit: the data gradient with the
forward convolution's sums (one order for both), gelu' with torch's float32 erf
and exp in the same expression, the head with its channels added one after
another.  Against 64 bits, gelu' is within one bf16 rounding (2^-8 relative) and
4 FP32 roundings of its largest term (2^-22, |v phi(v)| <= 0.25, Phi <= 1).
"""
import math

import pytest
import torch

from tests.test_gpu_unet import _call, bf, unbf

pytestmark = pytest.mark.gpu


def gelu_grad_f32(z):
    """The derivative op by op in float32 with torch's erf and exp."""
    return 0.5 * (1.0 + torch.erf(z * (0.5 ** 0.5))) \
        + z * (2.0 * math.pi) ** -0.5 * torch.exp((-0.5 * z) * z)


# a 32-channel gradient (blocks of 16 and of 4 rows), and wider ones on each tile
@pytest.mark.parametrize("N,H,W,c,cin", [
    (1, 1, 1, 32, 32), (1, 17, 33, 32, 96), (2, 145, 161, 32, 32), (1, 9, 31, 64, 32),
    (1, 5, 19, 64, 192), (2, 4, 33, 128, 64), (1, 3, 17, 128, 384), (1, 5, 18, 160, 64),
    (1, 6, 15, 256, 512), (1, 3, 20, 384, 128), (1, 4, 17, 40, 24), (1, 2, 18, 544, 32)])
def test_data_gradient_order(N, H, W, c, cin):
    from seistorch_amd import _lib
    g = torch.Generator().manual_seed(c * 5 + cin + H)
    dz = bf(torch.randn((N, H, W, c), generator=g)).cuda()
    w = bf(torch.randn((cin, 9 * c), generator=g) * (9 * c) ** -0.5).cuda()
    z = bf(torch.randn((N, H, W, cin), generator=g) * 2).cuda()
    y = torch.empty((N, H, W, cin), dtype=torch.int16, device="cuda")
    fused = torch.empty_like(y)
    dx = torch.empty((N, H, W, cin), device="cuda")
    s, P = _lib.stream_of(dx), _lib.ptr
    _call("seis_unet_conv3x3", P(dz), N, H, W, c, P(w), None, cin, 0, None, P(y), None, s)
    _call("seis_unet_conv3x3", P(dz), N, H, W, c, P(w), None, cin, 0, None, None, P(dx), s)
    _call("seis_unet_conv3x3_gelu_grad", P(dz), N, H, W, c, P(w), cin, P(z), P(fused), s)
    assert torch.equal(bf(dx), y)
    assert torch.equal(fused, bf(dx * gelu_grad_f32(unbf(z))))


@pytest.mark.parametrize("dy", [1.0, -0.37, 1.1e-4])
def test_gelu_derivative(dy):
    from seistorch_amd import _lib
    z = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16)
    z = z[unbf(z).isfinite()].cuda()
    d = torch.full(z.shape, dy, device="cuda")
    out = torch.empty_like(z)
    _call("seis_unet_gelu_bwd", _lib.ptr(d), _lib.ptr(z), z.numel(), _lib.ptr(out),
          _lib.stream_of(d))
    v = unbf(z)
    assert torch.equal(out, bf(d * gelu_grad_f32(v)))
    v = v.double()
    ref = dy * (0.5 * torch.erfc(-v * 0.5 ** 0.5)
                + v * (2.0 * math.pi) ** -0.5 * torch.exp(-0.5 * v * v))
    err = (unbf(out).double() - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -8 + abs(dy) * 2.0 ** -22).all()


@pytest.mark.parametrize("P", [1, 255, 4099])
def test_head_order(P):
    from seistorch_amd import _lib
    g = torch.Generator().manual_seed(P)
    x = bf(torch.randn((P, 32), generator=g)).cuda()
    w, b = torch.randn(32, generator=g).cuda(), torch.randn(1, generator=g).cuda()
    out = torch.empty(P, device="cuda")
    _call("seis_unet_head", _lib.ptr(x), P, 32, _lib.ptr(w), _lib.ptr(b), _lib.ptr(out),
          _lib.stream_of(out))
    v, s = unbf(x), torch.zeros(P, device="cuda")
    for c in range(32):
        s = s + v[:, c] * w[c]
    assert torch.equal(out, s + b)
