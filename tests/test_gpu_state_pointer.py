"""A state changed through the pointer of scl_dns_state (GPU).

The change is scl_ifrk4_integrate in place (its right-hand side is not
truncated, so it leaves modes beyond the radius).  By the solver's own callback,
which tells the solver, the pointer can be an old one; by another solver's, the
pointer is asked for again.  The next step has to take the state as it is: a
fresh solver set from it gives the same bits, and so does asking again."""
import numpy as np
import pytest

import speccodelib_amd as scl

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# fields of 2 MB and more: steps leave out what lies beyond the radius
GRIDS = [((64, 64, 64), scl.DP), ((128, 64, 64), scl.SP), ((256, 64, 64), scl.SP)]
KINDS = [dict(sgs=1, cs2=0.03), dict(scalar=True, grad=1.0, schmidt=0.7),
         dict(sgs=1, cs2=0.03, scalar=True, grad=1.0, schmidt=0.7), dict(sgs=2, cs2=0.03, iupdate=2)]


def state_of(d):
    return [*d.get_velocity()] + ([d.get_scalar()] if d.params.scalar else [])


def solver(p, v, **kw):
    d = scl.DNS(p, nu=0.02, dt=1e-3, forced=1, fkmax=2.5, eps=0.1, **kw)
    d.set_velocity(*v[:3])
    if d.params.scalar:
        d.set_scalar(v[3])
    return d


@pytest.mark.parametrize("i", range(len(GRIDS)))
@pytest.mark.parametrize("kind", range(len(KINDS)))
@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("stepper", [0, 2])
def test_change_through_a_kept_pointer(i, kind, graph, own, stepper):
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible to torch")
    dims, prec = GRIDS[i]
    kw = dict(KINDS[kind], stepper=stepper, use_graph=graph)
    p = scl.Plan3D(*dims, prec)
    v = [*scl.initialize(*dims, 1, 4.0, 1.0, prec)]
    v.append(v[1])
    got = []
    for ask in (not own, True):
        d = solver(p, v, **kw)
        d.step(3)  # with a captured step, where graphs are used
        ptr, n = d.state()
        d.step(3)
        cb = d if own else solver(p, v, **kw)
        rate = torch.empty(n, dtype=torch.float32 if prec == scl.SP else torch.float64, device="cuda")
        d.rates(rate.data_ptr())
        d.sync()
        scl.ifrk4_integrate(prec, n, ptr, rate.data_ptr(), 0.0, 1e-3, 1, scl.dns_derivs_cb_ptr(), cb.h.value)
        changed = state_of(d)
        if ask:
            d.state()
        d.step(1)
        one = state_of(d)
        d.step(2)
        got.append((changed, one, state_of(d)))
        if cb is not d:
            cb.close()
        d.close()
    kx, ky, kz = (np.arange(dims[0] // 2 + 1), *(np.fft.fftfreq(n, 1.0 / n) for n in dims[1:]))
    k2 = kx[None, None, :] ** 2 + ky[None, :, None] ** 2 + kz[:, None, None] ** 2
    out = k2 >= (2.0 * (dims[0] // 2) / 3.0) ** 2 * (1 + 1e-6)
    assert any(x[out].any() for x in got[0][0])
    for a, b in zip(*got):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)
    assert not any(x[out].any() for x in got[0][1])
    if not stepper and kw.get("sgs") != 2:
        d = solver(p, got[0][0], **kw)
        d.step(1)
        for x, y in zip(got[0][1], state_of(d)):
            np.testing.assert_array_equal(x, y)
        d.close()
    p.close()
