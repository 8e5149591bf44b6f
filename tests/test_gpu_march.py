"""The marching acoustic loops (up to four time steps per launch) against the
one-step-per-launch loops, at the edges of their tiles and schedules: widths
that divide by 1, 2 and 4, segments shorter and longer than the grid, time
axes and snapshot intervals that leave every remainder, receivers on
neighbouring rows, twice in one cell and on the grid's edge, both boundaries."""
import math

import pytest
import torch

from seistorch_amd.equations2d import acoustic as ac
from seistorch_amd.pml import generate_pml_coefficients_2d

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _problem(nz, nx, B, nt, free, seed=3):
    g = torch.Generator().manual_seed(seed)
    top = 0 if free else 50
    vp = (2000 + 1500 * torch.rand(nz, nx, generator=g)).to(DEV)
    d = generate_pml_coefficients_2d((nz, nx), 50, multiple=free).to(DEV)
    w = torch.randn(nt, generator=g).to(DEV)
    src = torch.stack([torch.randint(top, nz - 51, (B,), generator=g),
                       torch.randint(51, nx - 51, (B,), generator=g)], 1).int().to(DEV)
    rows = (0, top + 1, top + 2, nz // 2, nz - 1)
    rec = torch.cat([b * nz * nx + z * nx + torch.randint(0, nx, (23,), generator=g)
                     for b in range(B) for z in rows])
    rec = torch.cat([rec, rec[:5]]).to(DEV)
    return vp, d, w, src, rec, B, 1e-3, 10.0


def _run(P, free, K, shape=None, monkeypatch=None):
    """Records and gradient; shape (steps, cells per lane, rows) of the marching
    loops, or None: one step per launch."""
    if shape is not None:
        f, b = ac._march_forward, ac._march_backward
        used = []
        monkeypatch.setattr(ac, "_march_forward",
                            lambda *a: (used.append(1), f(*a, shape=shape))[1])
        monkeypatch.setattr(ac, "_march_backward",
                            lambda *a: (used.append(1), b(*a, shape=shape))[1])
    vp = P[0].clone().requires_grad_(True)
    kw = {} if shape is not None else dict(shots_per_group=1, two_step=False)
    r = ac.propagate(vp, *P[1:], multiple=free, snapshot_every=K, **kw)
    g = torch.Generator().manual_seed(1)
    r.backward(torch.randn(r.shape, generator=g).to(DEV))
    if shape is not None:
        assert len(used) == 2  # both directions took the marching loops
        monkeypatch.undo()
    return r.detach(), vp.grad


@pytest.mark.parametrize("nz,nx,B,nt,free", [
    (109, 103, 1, 2, False), (107, 105, 2, 3, False), (141, 259, 3, 38, False),
    (153, 302, 9, 61, True), (202, 500, 2, 75, False)])
@pytest.mark.parametrize("K", [0, 1, 7, 50])
def test_marching_loops_equal_one_step_loops(nz, nx, B, nt, free, K, monkeypatch):
    P = _problem(nz, nx, B, nt, free)
    r0, g0 = _run(P, free, K)
    # the gradient's terms are added in another order: a sum of n = nt * B
    # roundings of 2^-24 each, taken as a random walk with a factor of 4
    tol = 4 * math.sqrt(nt * B) * 2.0 ** -24
    for shape in [(0, 0, 0), (1, 1, 16), (2, 2, 7), (4, 1, 5), (4, 2, 1000), (4, 4, 33)]:
        if shape[1] and nx % shape[1]:
            continue
        r, g = _run(P, free, K, shape, monkeypatch)
        assert torch.equal(r, r0), shape
        e = float((g - g0).double().norm() / g0.double().norm().clamp_min(1e-300))
        assert e <= tol, (shape, e, tol)


def test_receivers_on_many_rows_and_none():
    """A well's receivers keep the one-step loops; no receivers at all work."""
    vp, d, w, src, _, B, dt, h = _problem(180, 204, 2, 20, False)
    nz, nx = vp.shape
    well = (torch.arange(B)[:, None] * nz * nx + torch.arange(50, 130)[None, :] * nx + 100)
    well = well.reshape(-1).to(DEV)
    assert ac._march_rows(well, nz, nx) is None
    a = ac.propagate(vp, d, w, src, well, B, dt, h)
    b = ac.propagate(vp, d, w, src, well, B, dt, h, two_step=False)
    assert torch.equal(a, b)
    none = torch.zeros(0, dtype=torch.int64, device=DEV)
    assert ac.propagate(vp, d, w, src, none, B, dt, h).shape == (20, 0)
