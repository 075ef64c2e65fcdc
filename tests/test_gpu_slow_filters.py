"""Step loops with filters that decay slowly, against the oracle.

From alpha 0.376 on the FP64 recursions sum more terms than they keep addresses
for, also in the x filter that the last stage applies; beyond 0.4972 the filters
run on cyclic reduction as passes of their own.  Tolerances: the parity tests'
1e-12 for the steps, and per step and direction a filter's 1e-13 times the
condition (1 + 2 a) / (1 - 2 a) of its implicit matrix over the one at 0.35.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

STEPS = 3


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def _state(shape, seed):
    rng = np.random.default_rng(seed)
    q = np.zeros(shape + (5,), order="F")
    q[..., 0] = 1 + 0.05 * rng.random(shape)
    q[..., 1:4] = 0.3 * rng.standard_normal(shape + (3,))
    q[..., 4] = 5 + 0.1 * rng.random(shape)
    return q


@pytest.mark.parametrize("alpha", [0.37, 0.38, 0.45, 0.497, 0.498])
@pytest.mark.parametrize("shape, scheme", [((64, 48, 72), O.PERIODIC), ((64, 48, 72), O.OPEN), ((41, 60, 65), O.OPEN),
                                           ((16, 24, 136), O.PERIODIC), ((136, 16, 17), O.OPEN)])
def test_filtered_steps_match_oracle(shape, scheme, alpha):
    from public_amd import Cruna
    scheme = tuple(O.OPEN if scheme == O.OPEN else O.PERIODIC for _ in range(3))
    kw = dict(mu0=0.01, T0=5.0, dt=1e-4, scheme=scheme, filter_alpha=alpha, filter_freq=(1, 1, 1))
    q, dx = _state(shape, 7), (0.13, 0.2, 0.26)
    tol = 1e-12 + STEPS * 3 * 1e-13 * max(1.0, (1 + 2 * alpha) / (1 - 2 * alpha) * 0.3 / 1.7)
    with Cruna(shape, dx, **kw) as g:
        g.set_state(q)
        g.run_direct(STEPS)
        err = rel(g.get_state(), O.run_direct(O.Cfg(shape, dx, **kw), q, STEPS))
        assert err < tol, err


@pytest.mark.parametrize("alpha, freq, batched", [(0.45, 1, True), (0.498, 1, False), (0.498, 0, True)])
def test_ensembles_of_slow_filters_match_their_members(alpha, freq, batched):
    """Filters on cyclic reduction run member by member; without filters alpha does not matter."""
    from public_amd import FORWARD, Cruna, Ensemble
    steps, members, states = 4, [], []
    for k, n in enumerate((32, 48)):
        members.append(dict(n=(n,) * 3, dx=(0.2,) * 3, mu0=0.01, T0=5.0, dt=1e-4, filter_alpha=alpha,
                            filter_freq=(freq,) * 3))
        states.append(_state((n,) * 3, k))
    with Ensemble(members) as ens:
        for i, q in enumerate(states):
            ens[i].set_state(q)
            ens.set_role(i, FORWARD, 0)
        ens.run(steps)
        assert (ens.batched_steps() > 0) == batched
        for i, q in enumerate(states):
            kw = dict(members[i])
            with Cruna(kw.pop("n"), kw.pop("dx"), **kw) as g:
                g.set_state(q)
                g.run_direct(steps)
                assert np.array_equal(ens[i].get_state(), g.get_state())
