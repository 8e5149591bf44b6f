"""The batched marching loops (up to four steps of every instance per launch)
against the batched one-step loops: uneven grids, shots and time axes (one and
two steps among them), every remainder of the launches, snapshot intervals and
lane widths, an instance without receivers, and the forward alone.

Records are the same bit for bit.  Gradients differ by the order of FP32
additions over steps and shots and by the separate rounding of 2c: relative L2
1e-5 at most."""
import types

import pytest
import torch

from seistorch_amd.equations2d import acoustic_batch as ab
from tests.test_gpu_march import DEV, _problem

pytestmark = pytest.mark.gpu

SIZES = [(141, 256, 3, 61), (109, 104, 1, 1), (164, 180, 9, 38), (107, 108, 2, 2),
         (130, 300, 2, 75), (120, 132, 4, 64)]


def _instances(odd):
    out = []
    for q, (nz, nx, B, nt) in enumerate(SIZES):
        vp, d, w, src, rec, B, dt, h = _problem(nz, nx + odd, B, nt, False, seed=q)
        if q == 4:
            rec = rec[:0]
        out.append(ab.BatchInstance(vp, d, w, src, rec, B, dt * (1 - 0.05 * q), h + q))
    return out


def _run(insts, grad, monkeypatch, march=None, **kw):
    real, used = ab._BatchLoop, []
    if march is not None:
        def apply(*a):
            assert a[-1] == (0, 0)  # the default call takes the marching loops
            return real.apply(*a[:-1], march)
        monkeypatch.setattr(ab, "_BatchLoop", types.SimpleNamespace(apply=apply))
        call = ab._lib.call
        monkeypatch.setattr(ab._lib, "call", lambda n, *a: (used.append(n), call(n, *a))[1])
    for it in insts:
        it.vp = it.vp.detach().clone().requires_grad_(grad)
    recs = ab.propagate_batch(insts, **kw)
    if grad:
        g = torch.Generator().manual_seed(1)
        sum((r * torch.randn(r.shape, generator=g).to(DEV)).sum() for r in recs).backward()
    if march is not None:
        monkeypatch.undo()
        assert "seis_acoustic_march_batch_forward" in used
        assert ("seis_acoustic_march_batch_backward" in used) == grad
    return [r.detach() for r in recs], [it.vp.grad for it in insts]


@pytest.mark.parametrize("K", [0, 1, 7, 50])
@pytest.mark.parametrize("march,odd", [((0, 0), 0), ((4, 13), 0), ((2, 5), 2), ((1, 40), 1)])
def test_batched_marching_equals_one_step(K, march, odd, monkeypatch):
    insts = _instances(odd)
    r0, g0 = _run(insts, True, monkeypatch, shots_per_group=1, rows_per_thread=1, vec_x=1,
                  two_step=False, use_graph=False, snapshot_every=K)
    r1, g1 = _run(insts, True, monkeypatch, march=march, snapshot_every=K)
    for q, (a, b, x, y) in enumerate(zip(r0, r1, g0, g1)):
        assert torch.equal(a, b), f"instance {q}: records differ"
        assert (x - y).norm() <= 1e-5 * x.norm(), q
        assert float(x.abs().max()) > 0 or SIZES[q][3] <= 2 or q == 4


def test_forward_alone(monkeypatch):
    insts = _instances(0)
    r0, _ = _run(insts, False, monkeypatch, shots_per_group=1, two_step=False, use_graph=False)
    r1, _ = _run(insts, False, monkeypatch, march=(0, 0))
    assert all(torch.equal(a, b) for a, b in zip(r0, r1))
