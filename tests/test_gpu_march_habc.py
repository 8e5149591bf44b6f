"""The HABC loops with up to four steps per launch away from the edges against one
step per launch: the smallest grids they take, widths that divide by 1, 2 and 4,
time axes and snapshot intervals that leave every remainder, receivers and sources
in the frame, at the edge of the marched part and inside it, both boundaries.

Records are the same bit for bit.  The adjoint field is rounded in another order
away from the edges: per step and operation 2^-24, which over the steps of these
problems stays below a relative L2 of 2e-5 of the gradient."""
import pytest
import torch

from seistorch_amd.equations2d import acoustic_habc as ah
from seistorch_amd.habc import generate_habc_coefficients_2d
from tests.test_gpu_march import DEV

pytestmark = pytest.mark.gpu
CORE = 57  # first row of the marched part


def _problem(nz, nx, B, nt, deep, multiple=False):
    g = torch.Generator().manual_seed(nz + nx)
    vp = (2000 + 1500 * torch.rand(nz, nx, generator=g)).to(DEV)
    b = generate_habc_coefficients_2d((nz, nx), 50, multiple=multiple).to(DEV)
    w = torch.randn(nt, generator=g).to(DEV)
    sz = torch.tensor([51, CORE - 1, CORE, CORE + 3, nz // 2])[torch.arange(B) % 5]
    src = torch.stack([sz, torch.randint(51, nx - 51, (B,), generator=g)], 1).int().to(DEV)
    rows = (0, 20, 51, 54) + ((CORE - 1, CORE, CORE + 1, CORE + 4, nz // 2) if deep else ())
    rec = torch.cat([s * nz * nx + z * nx + torch.randint(0, nx, (31,), generator=g)
                     for s in range(B) for z in rows])
    rec = torch.cat([rec, rec[-5:]]).to(DEV)
    return vp, b, w, src, rec, B, 1e-3, 10.0


def _run(P, multiple, K, shape=None, monkeypatch=None):
    used, kw = [], dict(shots_per_group=1)
    if shape is not None:
        kw, f, bw = {}, ah._march_forward, ah._march_backward
        monkeypatch.setattr(ah, "_march_fits", lambda *a: True)
        monkeypatch.setattr(ah, "_march_forward",
                            lambda *a: (used.append(1), f(*a, shape=shape))[1])
        monkeypatch.setattr(ah, "_march_backward",
                            lambda *a: (used.append(1), bw(*a, shape=shape))[1])
    vp = P[0].clone().requires_grad_(True)
    r = ah.propagate(vp, *P[1:], multiple=multiple, snapshot_every=K, **kw)
    g = torch.Generator().manual_seed(1)
    r.backward(torch.randn(r.shape, generator=g).to(DEV))
    if shape is not None:
        assert len(used) == 2
        monkeypatch.undo()
    return r.detach(), vp.grad


@pytest.mark.parametrize("nz,nx,B,nt,multiple,deep", [
    (130, 136, 1, 1, False, True), (131, 133, 2, 2, False, True), (141, 259, 3, 39, False, False),
    (153, 302, 9, 61, True, True), (202, 400, 5, 75, False, True)])
@pytest.mark.parametrize("K", [0, 1, 7, 50])
def test_marching_loops_equal_one_step_loops(nz, nx, B, nt, multiple, deep, K, monkeypatch):
    P = _problem(nz, nx, B, nt, deep, multiple)
    r0, g0 = _run(P, multiple, K)
    for shape in [(0, 0), (1, 5), (2, 1000), (4, 33)]:
        if shape[0] and nx % shape[0]:
            continue
        r, g = _run(P, multiple, K, shape, monkeypatch)
        assert torch.equal(r, r0), shape
        assert float((g - g0).double().norm()) <= 2e-5 * float(g0.double().norm()), shape
