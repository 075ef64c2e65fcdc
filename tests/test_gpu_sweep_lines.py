"""FP64 sweeps on lines at the edges of the line engine's split (against the oracle).

Along x a wavefront exchanges its lines in quads of threads, eight points a
thread: lines of an odd number of eights and of a number that is no multiple
of four leave part of a wavefront idle, short lines put several into one, and
a line longer than 512 points spans wavefronts.  Tolerances are the parity
tests' (1e-12 for right-hand sides and steps; 1e-13 for a filter, times the
condition (1 + 2 a) / (1 - 2 a) of its implicit matrix over the one at 0.35).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def _state(shape, seed):
    rng = np.random.default_rng(seed)
    q = np.zeros(shape + (5,), order="F")
    q[..., 0] = 1 + 0.05 * rng.random(shape)
    q[..., 1:4] = 0.3 * rng.standard_normal(shape + (3,))
    q[..., 4] = 5 + 0.1 * rng.random(shape)
    return q


SHAPES = [(16, 16, 16), (24, 40, 16), (72, 16, 24), (104, 24, 16), (520, 16, 16), (16, 520, 16), (16, 16, 520),
          (1032, 16, 16)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("scheme", [O.PERIODIC, O.OPEN])
def test_sweeps_match_oracle(shape, scheme):
    from public_amd import Cruna
    dx = (0.13, 0.2, 0.26)
    q, qs = _state(shape, 3), np.asfortranarray(np.random.default_rng(4).standard_normal(shape + (5,)))
    kw = dict(mu0=0.01, T0=5.0, dt=1e-4, scheme=(scheme,) * 3)
    cfg = O.Cfg(shape, dx, **kw)
    with Cruna(shape, dx, **kw) as g:
        assert rel(g.right_hand_side_direct_3d(q), O.rhs_direct(cfg, q)) < 1e-12
        assert rel(g.right_hand_side_adjoint_3d(qs, q), O.rhs_adjoint(cfg, qs, q)) < 1e-12
        g.set_state(q)
        g.run_direct(2)
        assert rel(g.get_state(), O.run_direct(cfg, q, 2)) < 1e-12


@pytest.mark.parametrize("shape", SHAPES[:5])
@pytest.mark.parametrize("alpha", [0.0, 0.45, 0.497, 0.498, 0.4995])
def test_filters_up_to_the_slowest(shape, alpha):
    """Beyond alpha = 0.4972 the recursion's factor exceeds 0.9 and cyclic reduction takes over."""
    from public_amd import Cruna
    q = np.asfortranarray(np.random.default_rng(2).standard_normal(shape + (5,)))
    tol = 1e-13 * max(1.0, (1 + 2 * alpha) / (1 - 2 * alpha) * 0.3 / 1.7)
    for scheme in (O.PERIODIC, O.OPEN):
        kw = dict(scheme=(scheme,) * 3, filter_alpha=alpha)
        cfg = O.Cfg(shape, (1, 1, 1), **kw)
        with Cruna(shape, (1, 1, 1), **kw) as g:
            for d in range(3):
                err = rel(g.filter(d, q), O.filter4d(cfg, d, q))
                assert err < tol, (scheme, d, err)
