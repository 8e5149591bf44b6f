"""The marching loops where their larger sets of buffers do not fit: each direction
falls back by itself to the loops that need fewer, from buffers that are asked for last.

Records are the same bit for bit.  Gradients are sums of one rounding of 2^-24 per
step and shot in another order (HABC: another order per operation as well), below a
relative L2 of 2e-5 for these problems."""
import pytest
import torch

from seistorch_amd.equations2d import acoustic as ac
from seistorch_amd.equations2d import acoustic_batch as ab
from seistorch_amd.equations2d import acoustic_habc as ah
from seistorch_amd.habc import generate_habc_coefficients_2d
from tests.test_gpu_march import DEV, _problem

pytestmark = pytest.mark.gpu


def _run(kind, P, K):
    vp, rest = P[0].clone().requires_grad_(True), P[1:]
    if kind == "batch":
        one = ab.BatchInstance(vp, *rest)
        two = ab.BatchInstance(vp[:, :-4].contiguous(), rest[0][:, :-4].contiguous(), rest[1][:-3],
                               rest[2], rest[3][:0], *rest[4:])
        r = ab.propagate_batch([one, two], snapshot_every=K)[0]
    elif kind == "habc":
        r = ah.propagate(vp, *rest, snapshot_every=K)
    else:
        r = ac.propagate(vp, *rest, snapshot_every=K)
    g = torch.Generator().manual_seed(1)
    r.backward(torch.randn(r.shape, generator=g).to(DEV))
    return r.detach(), vp.grad


def _make(kind, nz, nx, B, nt):
    P = list(_problem(nz, nx, B, nt, False))
    if kind == "habc":
        P[1] = generate_habc_coefficients_2d((nz, nx), 50).to(DEV)
    return P


MOD = {"acoustic": ac, "batch": ab, "habc": ah}


def _same(got, want):
    assert torch.equal(got[0], want[0])
    assert float((got[1] - want[1]).double().norm()) <= 2e-5 * float(want[1].double().norm())


@pytest.mark.parametrize("kind", ["acoustic", "batch", "habc"])
@pytest.mark.parametrize("short", ["forward", "backward", "both"])
@pytest.mark.parametrize("nt,K", [(38, 0), (61, 7)])
def test_each_direction_falls_back(kind, short, nt, K, monkeypatch):
    P, mod = _make(kind, 153, 204, 5, nt), MOD[kind]
    if kind == "habc":
        monkeypatch.setattr(mod, "_march_fits", lambda *a: False)
    else:
        monkeypatch.setattr(mod, "_march_rows", lambda *a: None)
    want = _run(kind, P, K)
    monkeypatch.undo()
    if kind == "habc":
        monkeypatch.setattr(mod, "_march_fits", lambda *a: True)
    real, calls = mod._march_buffers, []

    def buffers(*a):
        calls.append("forward" if not calls else "backward")
        return None if short in (calls[-1], "both") else real(*a)
    monkeypatch.setattr(mod, "_march_buffers", buffers)
    _same(_run(kind, P, K), want)
    assert calls == ["forward", "backward"]


@pytest.mark.parametrize("kind", ["acoustic", "batch", "habc"])
@pytest.mark.parametrize("grad", [True, False])
def test_the_larger_set_comes_after_what_every_loop_needs(kind, grad, monkeypatch):
    """So that a survey whose records, rings and snapshots fit beside the smaller set
    falls back instead of running out of memory."""
    nz, nx, B, nt, K = 153, 204, 5, 61, 7
    P, mod = _make(kind, nz, nx, B, nt), MOD[kind]
    if kind == "habc":
        monkeypatch.setattr(mod, "_march_fits", lambda *a: True)
    need = 4 * nt * P[4].shape[0]
    if grad:
        need += 4 * (nt - 1) * B * ac.ring_len(nz, nx) + 4 * ((nt - 2) // K) * 2 * B * nz * nx
    real, calls = mod._march_buffers, []

    def buffers(*a):
        calls.append(torch.cuda.memory_allocated() - before)
        return real(*a)
    monkeypatch.setattr(mod, "_march_buffers", buffers)
    before = torch.cuda.memory_allocated()
    if grad:
        _run(kind, P, K)
    elif kind == "batch":
        with torch.no_grad():
            ab.propagate_batch([ab.BatchInstance(*P)])
    else:
        with torch.no_grad():
            mod.propagate(*P)
    assert len(calls) == 1 + grad and calls[0] >= need
