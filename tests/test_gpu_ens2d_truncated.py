"""Scheme 0 steps that leave out what lies beyond the 2/3 cut: a state set with
modes out there (its first step takes them as they are), runs grouped into
calls in every way, and a state set again in the middle of a run.

FP64 against the oracle at the bar of the other 2D steps (1e-10 of the largest
entry); groupings of the same steps to the bit."""
import numpy as np
import pytest

import speccodelib_amd as scl
from oracle import vort2d as v2

pytestmark = pytest.mark.gpu

KW = dict(dt=2e-3, c_hyper=1e-5, n_hyper=4, damp=0.1, fkmin=4.0, fkmax=5.0, eps=0.01)


def full_state(n, seed):
    """A state with entries on both sides of the cut, symmetric as a step leaves it."""
    w = v2.initialize2d(n, -seed, 8.0, 0.5)
    rng = np.random.default_rng(seed)
    w = w + 1e-3 * (rng.standard_normal(w.shape) + 1j * rng.standard_normal(w.shape))
    w[n // 2, :] = 0
    w[:, n // 2] = 0
    w[0, 0] = 0
    w[n // 2 + 1:, 0] = np.conj(w[1: n // 2, 0][::-1])
    return w


def oracle_steps(n, w, steps):
    o = v2.Vort2D(v2.Vort2DParams(n=n, **KW))
    for _ in range(steps):
        w = o.rk4_step(w)
    return w


@pytest.mark.parametrize("n,members", [(32, 1), (32, 5), (64, 3), (128, 2), (256, 1)])
@pytest.mark.parametrize("graph", [0, 1])
def test_steps_of_untruncated_states(n, members, graph):
    e = scl.Ensemble2D([(n, members)], prec=scl.DP, use_graph=graph, **KW)
    w = [full_state(n, 3 + j) for j in range(members)]
    for j in range(members):
        e.set_member(0, j, w[j])
    e.step(1)
    e.step(3)
    for j in range(members):
        want = oracle_steps(n, w[j], 4)
        assert np.abs(e.get_member(0, j) - want).max() < 1e-10 * np.abs(want).max()
    # the last member set again: the others go on, none loses what is beyond the cut
    other = full_state(n, 40)
    w = [e.get_member(0, j) for j in range(members)]
    w[-1] = other
    e.set_member(0, members - 1, other)
    e.step(12)
    for j in range(members):
        want = oracle_steps(n, w[j], 12)
        assert np.abs(e.get_member(0, j) - want).max() < 1e-10 * np.abs(want).max()


@pytest.mark.parametrize("n,e_pts,cw", [(64, 8, 8), (64, 16, 8), (128, 8, 16), (256, 8, 4), (1024, 8, 8)])
def test_groupings_of_steps_are_the_same(n, e_pts, cw):
    w = full_state(n, 9).astype(np.complex64)
    out = []
    for runs in ([13], [1, 12], [5, 5, 3], [1] * 13):
        e = scl.Ensemble2D([(n, 2)], prec=scl.SP, **KW)
        e.set_schedule(0, e_pts, cw, 0)
        for j in range(2):
            e.set_member(0, j, w)
        for k in runs:
            e.step(k)
        out.append(e.get_member(0, 1))
    for o in out[1:]:
        assert np.array_equal(o, out[0])
