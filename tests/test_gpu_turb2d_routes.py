"""The two routes of a turb_2d ensemble's step (GPU): both halves of the
nonlinear term in each pass, for batches that leave the chip room, and the two
halves one after the other, for batches that fill it.

Each against the FP64 oracle at the bars of the scheme's other tests (nonlinear
term 1e-12 / 2e-5, five steps 1e-11 / 1e-4; FP64 / FP32), graph replay equal to
eager steps to the bit.  A batch that fills the chip keeps the memory of the
second route: seven fields."""
import numpy as np
import pytest

import speccodelib_amd as scl
from oracle import turb2d as t2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def par(n):
    return dict(nu=0.5, eta=5.0, kf=4.0, sigma=1.0 / (0.4 * n))


def field(n, seed):
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((n, n // 2)) + 1j * rng.standard_normal((n, n // 2))
    w = w * np.exp(-t2.kgrid(n)[2] / (2 * (n / 8) ** 2))
    for iy in range(1, n // 2):  # Hermitian kx = 0 column
        w[n - iy, 0] = np.conj(w[iy, 0])
    return t2.symmetrize(w)


def relerr(a, b):
    return np.abs(np.asarray(a, np.complex128) - b).max() / np.abs(b).max()


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("prec,tol,step_tol", [(scl.DP, 1e-12, 1e-11), (scl.SP, 2e-5, 1e-4)])
@pytest.mark.parametrize("n", [32, 64, 128, 256, 512, 1024])
def test_routes_match_the_oracle(monkeypatch, split, prec, tol, step_tol, n):
    monkeypatch.setenv("SCL_TURB2D_SPLIT", split)
    ct = np.complex128 if prec == scl.DP else np.complex64
    w = [field(n, n + j) for j in range(2)]
    got = []
    for graph in (True, False):
        e = scl.Ensemble2D([(n, 2)], prec=prec, dt=1e-3, scheme=1, use_graph=graph, **par(n))
        assert relerr(e.rhs(0, 1, w[1].astype(ct)), t2.nonlinear(w[1])) < tol
        for j in range(2):
            e.set_member(0, j, w[j].astype(ct))
        e.step(1)
        e.step(4)
        got.append([e.get_member(0, j).copy() for j in range(2)])
        e.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
    for j in range(2):
        o = t2.Turb2D(t2.Turb2DParams(n=n, dt=1e-3, **par(n)), w[j])
        for _ in range(5):
            o.step()
        assert relerr(got[0][j], o.w) < step_tol


@pytest.mark.parametrize("n,members,prec", [(1024, 16, scl.SP), (512, 64, scl.SP), (256, 64, scl.DP), (128, 512, scl.DP)])
def test_memory_of_a_batch_that_fills_the_chip(n, members, prec):
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible to torch")
    scl.Ensemble2D([(n, 1)], prec=prec, dt=1e-3, scheme=1, **par(n)).close()  # what a first use allocates
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    e = scl.Ensemble2D([(n, members)], prec=prec, dt=1e-3, scheme=1, **par(n))
    used = before - torch.cuda.mem_get_info()[0]
    e.close()
    f = members * n * (n // 2 + 1) * (8 if prec == scl.SP else 16)
    print(f"{used / f:.2f} fields of {f >> 20} MB", flush=True)
    assert used < 8 * f


@pytest.mark.parametrize("n,members,per_member", [(256, 4096, False), (1024, 256, True)])
def test_batches_that_only_fit_in_seven_fields(n, members, per_member):
    """Sizes that take nine fields where there is room (forced off: the members
    that are not set stay zero)."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible to torch")
    w = field(n, 3).astype(np.complex64)
    got = []
    for fill in (False, True):
        hold = None
        m = members if fill else 2
        if fill:
            f = members * n * (n // 2 + 1) * 8
            torch.cuda.empty_cache()
            free = torch.cuda.mem_get_info()[0]
            if free < 16 * f:
                pytest.skip("not enough free memory on this device")
            hold = torch.empty(free - 8 * f, dtype=torch.uint8, device="cuda")
        try:
            e = scl.Ensemble2D([(n, m)], prec=scl.SP, dt=1e-3, scheme=1, per_member=per_member, use_graph=False,
                               forced=False, **par(n))
            e.set_member(0, m - 1, w)
            e.step(4)
            got.append(e.get_member(0, m - 1).copy())
            e.close()
        finally:
            del hold
            torch.cuda.empty_cache()
    assert np.abs(got[0] - got[1]).max() < 1e-5 * np.abs(got[0]).max()
