"""The fused elastic adjoint's work between two reverse steps in one launch: its
gradients against the stage-by-stage adjoint, which takes a launch for each part,
with sources inside, on a row and a column of the ring, at its corner, next to it
and in the frame, in stresses and velocities, and no receivers.  Both round the same
operations in the same order; only atomic additions of receivers that share a cell
and the sums over shots may differ: relative L2 1e-6."""
import pytest
import torch

from seistorch_amd.equations2d import elastic as el
from tests.test_gpu_march import DEV, _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,free,receivers", [
    (("txx", "tzz"), False, True), (("vx", "txz"), False, True), (("vz", "txx"), True, True),
    (("vx", "vz", "txx", "tzz", "txz"), False, True), (("txx",), False, False)])
@pytest.mark.parametrize("nt,K", [(1, 0), (2, 0), (3, 1), (24, 7), (24, 0)])
def test_fused_adjoint_with_sources_on_the_ring(src, free, receivers, nt, K):
    vp, d, w, _, rec, _, dt, h = _problem(131, 152, 7, nt, free)
    nz, nx = vp.shape
    m = el.NPML
    cells = [(60, 70), (m, 80), (70, m), (nz - 1 - m, 90), (m, m), (m + 1, m + 1), (30, 20)]
    zx = torch.tensor(cells, dtype=torch.int32, device=DEV)
    rec = rec.unique() if receivers else rec[:0]
    g = torch.Generator().manual_seed(2)
    out = []
    weight = torch.randn((nt, rec.numel(), 2), generator=g).to(DEV)
    start = None
    for fused in (True, False):
        models = [t.clone().requires_grad_(True) for t in (vp, vp / 1.8, 1500 + 0.2 * vp)]
        r = el.propagate(*models, d, 1e-6 * w, zx, rec, 7, dt, h, src_type=src, multiple=free,
                         snapshot_every=K, fused=fused, shots_per_group=2)
        r.backward(weight)
        out.append([t.grad for t in models])
        assert start is None or torch.equal(start, r.detach())
        start = r.detach()
    for a, b in zip(*out):
        assert (a - b).norm() <= 1e-6 * b.norm()
