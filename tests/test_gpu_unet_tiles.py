"""The U-Net kernels' tiles and fused forms at their edges.

Tolerances: a result stored in bf16 is within one rounding (2^-8 relative) of
the exact one plus the FP32 accumulation, bounded by 2^-24 * sqrt(K) times the
sum of the products' magnitudes (taken as 1e-5 of the largest result); fused
forms round at the same places as the separate kernels, so they differ by at
most one bf16 rounding where an FP32 sum's order differs, and not at all where it
does not; FP32 weight gradients agree to rel-L2 1e-5.
"""
import pytest
import torch

from tests.test_gpu_unet import _call, bf, unbf

pytestmark = pytest.mark.gpu


def conv64(x, w, b, cout, cin):
    return torch.nn.functional.conv2d(
        x.double().permute(0, 3, 1, 2), w.double().reshape(cout, 3, 3, cin).permute(0, 3, 1, 2),
        b.double(), padding=1).permute(0, 2, 3, 1)


# every tile of the forward convolution, its edges in both axes, one pixel
@pytest.mark.parametrize("N,H,W,cin,cout", [
    (1, 1, 1, 8, 32), (2, 9, 33, 8, 32), (1, 17, 31, 32, 32), (2, 8, 32, 96, 32),
    (1, 5, 17, 32, 64), (1, 3, 47, 64, 64), (2, 4, 16, 64, 128), (1, 5, 19, 128, 128),
    (1, 7, 33, 160, 64), (1, 4, 32, 192, 64), (1, 5, 18, 128, 256), (2, 3, 17, 256, 256),
    (1, 5, 65, 384, 128), (1, 6, 15, 512, 256), (1, 3, 20, 544, 64)])
def test_forward_tiles(N, H, W, cin, cout):
    from seistorch_amd import _lib
    g = torch.Generator().manual_seed(cin * 7 + cout + H)
    x = bf(torch.randn((N, H, W, cin), generator=g))
    w = bf(torch.randn((cout, 9 * cin), generator=g) * (9 * cin) ** -0.5)
    b = torch.randn(cout, generator=g)
    ref = conv64(unbf(x), unbf(w), b, cout, cin)
    d = [t.cuda() for t in (x, w, b)]
    z = torch.empty((N, H, W, cout), dtype=torch.int16, device="cuda")
    y = torch.empty_like(z)
    s = _lib.stream_of(d[2])
    _call("seis_unet_conv3x3", _lib.ptr(d[0]), N, H, W, cin, _lib.ptr(d[1]), _lib.ptr(d[2]), cout,
          1, _lib.ptr(z), _lib.ptr(y), None, s)
    tol = ref.abs() * 2.0 ** -8 + 1e-5 * ref.abs().max()
    assert ((unbf(z.cpu()).double() - ref).abs() <= tol).all()
    act = torch.nn.functional.gelu(unbf(z.cpu()).double())
    # y is the activation of the unrounded sum: gelu's slope is at most 1.13
    tol = act.abs() * 2.0 ** -8 + 1.13 * tol
    assert ((unbf(y.cpu()).double() - act).abs() <= tol).all()
    if cin % 64 == 32 and cin > 64 or cin in (192, 384, 512):
        # the concatenation read in place: the same sums in the same order
        c1 = (cin // 96) * 64 if cin < 512 else 256
        H2, W2 = H + H % 2, W + W % 2
        low = bf(torch.randn((N, H2 // 2, W2 // 2, c1), generator=g)).cuda()
        skip = bf(torch.randn((N, H2, W2, cin - c1), generator=g)).cuda()
        u = torch.empty((N, H2, W2, cin), dtype=torch.int16, device="cuda")
        _call("seis_unet_up_concat", _lib.ptr(low), _lib.ptr(skip), N, H2, W2, c1, cin - c1,
              _lib.ptr(u), s)
        o = [torch.empty((N, H2, W2, cout), dtype=torch.int16, device="cuda") for _ in range(4)]
        _call("seis_unet_conv3x3", _lib.ptr(u), N, H2, W2, cin, _lib.ptr(d[1]), _lib.ptr(d[2]),
              cout, 1, _lib.ptr(o[0]), _lib.ptr(o[1]), None, s)
        _call("seis_unet_conv3x3_cat", _lib.ptr(low), c1, _lib.ptr(skip), cin - c1, N, H2, W2,
              _lib.ptr(d[1]), _lib.ptr(d[2]), cout, 1, _lib.ptr(o[2]), _lib.ptr(o[3]), s)
        assert torch.equal(o[0], o[2]) and torch.equal(o[1], o[3])


@pytest.mark.parametrize("N,H,W,c1,c2,cout", [
    (1, 2, 2, 0, 8, 32), (2, 9, 33, 0, 8, 32), (1, 17, 31, 0, 32, 64), (1, 8, 34, 64, 32, 32),
    (2, 10, 18, 128, 64, 64), (1, 16, 64, 0, 256, 256), (1, 40, 66, 0, 64, 64)])
def test_weight_gradient_workspace(N, H, W, c1, c2, cout):
    from seistorch_amd import _lib
    g = torch.Generator().manual_seed(c1 + c2 + cout + W)
    cin = c1 + c2
    skip = bf(torch.randn((N, H, W, c2), generator=g))
    low = bf(torch.randn((N, H // 2, W // 2, c1), generator=g)) if c1 else None
    dz = bf(torch.randn((N, H, W, cout), generator=g))
    x = unbf(skip)
    if c1:
        up = unbf(low).repeat_interleave(2, 1).repeat_interleave(2, 2)
        x = torch.cat([up, x], -1)
    xp = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    d64 = unbf(dz).double()
    ref = torch.stack([torch.einsum("nhwo,nhwi->oi", d64, xp[:, t // 3:t // 3 + H,
                                                            t % 3:t % 3 + W]) for t in range(9)], 1)
    start = torch.randn((cout, 9 * cin), generator=g)
    dw, db = start.clone().cuda(), torch.zeros(cout, device="cuda")
    n = int(_lib.load().seis_unet_wgrad_workspace(N, H, W, cin, cout))
    work = torch.full((n,), float("nan"), device="cuda")
    dev = [None if t is None else t.cuda() for t in (low, skip, dz)]
    _call("seis_unet_conv3x3_wgrad_ws", _lib.ptr(dev[0]), c1, _lib.ptr(dev[1]), c2,
          _lib.ptr(dev[2]), N, H, W, cout, _lib.ptr(dw), _lib.ptr(db), _lib.ptr(work),
          _lib.stream_of(dw))
    got = dw.cpu().double() - start.double()
    ref = ref.reshape(cout, 9 * cin)
    assert (got - ref).norm() <= 1e-5 * (ref.norm() + start.double().norm())
    rb = d64.sum((0, 1, 2))
    assert (db.cpu().double() - rb).norm() <= 1e-5 * d64.abs().sum((0, 1, 2)).norm()


@pytest.mark.parametrize("N,H,W,c1,c2", [(1, 2, 2, 64, 32), (2, 6, 34, 128, 64), (1, 10, 18, 256, 128)])
def test_fused_backward(N, H, W, c1, c2):
    """Data gradient through an activation, the two parts of a concatenation, the
    head and the flipped weights against the separate kernels."""
    from seistorch_amd import _lib
    g = torch.Generator().manual_seed(c1 + W)
    C = c1 + c2

    def rnd(*s):
        return torch.randn(s, generator=g).cuda()

    def out(*s, dt=torch.int16):
        return torch.empty(s, dtype=dt, device="cuda")

    def close(a, b):
        a, b = unbf(a.cpu()).double(), unbf(b.cpu()).double()
        assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6 * b.abs().max()).all()

    P = _lib.ptr
    w = bf(rnd(2 * c2 * 9 * c2 + c1 * 9 * c2))
    s = _lib.stream_of(w)
    layers = torch.tensor([[0, c2, c2], [c2 * 9 * c2, c1, c2], [c2 * 9 * (c1 + c2), c2, c2]],
                          dtype=torch.int64)
    both, one = out(w.numel()), out(w.numel())
    _call("seis_unet_flip_layers", P(w), 3, P(layers), P(both), s)
    for o, co, ci in layers.tolist():
        _call("seis_unet_flip_weights", P(w[o:]), co, ci, P(one[o:]), s)
    assert torch.equal(both, one)

    dz, z = bf(rnd(N, H, W, c2)), bf(rnd(N, H, W, c2) * 3)
    dx, sep, fus = out(N, H, W, c2, dt=torch.float32), out(N, H, W, c2), out(N, H, W, c2)
    _call("seis_unet_conv3x3", P(dz), N, H, W, c2, P(both), None, c2, 0, None, None, P(dx), s)
    _call("seis_unet_gelu_bwd", P(dx), P(z), dx.numel(), P(sep), s)
    _call("seis_unet_conv3x3_gelu_grad", P(dz), N, H, W, c2, P(both), c2, P(z), P(fus), s)
    assert torch.equal(sep, fus)

    dout, dpool = rnd(N, H, W, C), rnd(N, H // 2, W // 2, c2)
    zl = bf(rnd(N, H // 2, W // 2, c1) * 3)
    dlow, dskip = rnd(N, H // 2, W // 2, c1), out(N, H, W, c2, dt=torch.float32)
    _call("seis_unet_up_concat_bwd", P(dout), N, H, W, c1, c2, P(dlow), P(dskip), 0, s)
    sep, fus = out(*zl.shape), out(*zl.shape)
    _call("seis_unet_gelu_bwd", P(dlow), P(zl), dlow.numel(), P(sep), s)
    _call("seis_unet_up_gelu_bwd", P(dout), N, H, W, c1, c2, P(zl), P(fus), s)
    close(fus, sep)
    _call("seis_unet_avgpool2_bwd", P(dpool), N, H, W, c2, P(dskip), 1, s)
    sep, fus = out(*z.shape), out(*z.shape)
    _call("seis_unet_gelu_bwd", P(dskip), P(z), dskip.numel(), P(sep), s)
    _call("seis_unet_skip_gelu_bwd", P(dout), P(dpool), N, H, W, c1, c2, P(z), P(fus), s)
    close(fus, sep)

    n = N * H * W
    x, zh, do, hw = bf(rnd(n, 32)), bf(rnd(n, 32) * 3), rnd(n), rnd(32)
    a = [torch.zeros(32, device="cuda"), torch.zeros(1, device="cuda")]
    b = [torch.zeros(32, device="cuda"), torch.zeros(1, device="cuda")]
    dh, sep, fus = out(n, 32, dt=torch.float32), out(n, 32), out(n, 32)
    _call("seis_unet_head_bwd", P(x), P(do), n, 32, P(hw), P(dh), P(a[0]), P(a[1]), s)
    _call("seis_unet_gelu_bwd", P(dh), P(zh), dh.numel(), P(sep), s)
    _call("seis_unet_head_gelu_bwd", P(x), P(do), n, P(hw), P(zh), P(fus), P(b[0]), P(b[1]), s)
    assert torch.equal(sep, fus)
    scale = (do.abs()[:, None] * unbf(x).abs()).sum(0)
    assert ((a[0] - b[0]).abs() <= 1e-5 * scale + 1e-6).all()
    assert (a[1] - b[1]).abs() <= 1e-5 * do.abs().sum() + 1e-6
