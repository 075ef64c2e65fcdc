"""Characteristic rows on q launched together (GPU against the oracle).

Consecutive rows of the types 201, 202 and 203 share a launch of up to 12 rows
in which a point is updated by one thread, row after row: boxes that overlap in
edges, corners and whole, more rows than fit into a launch, and rows of
other types between them (200, 401), which end one.  The tolerance is the parity
tests' 1e-12 for runs of a few steps.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPE = (33, 20, 17)
N1, N2, N3 = SHAPE
FACES = [(201, 1, 1, 1, N2, 1, N3, -1, 0, 0), (201, N1, N1, 1, N2, 1, N3, 1, 0, 0),
         (201, 1, N1, 1, 1, 1, N3, 0, -1, 0), (201, 1, N1, N2, N2, 1, N3, 0, 1, 0),
         (201, 1, N1, 1, N2, 1, 1, 0, 0, -1), (201, 1, N1, 1, N2, N3, N3, 0, 0, 1)]
BLOCKS = [(201, 3 + m, 9 + m, 2, 8, 1 + m, 6 + m, 0.6, 0.0, 0.8) for m in range(8)]
ROWS = {
    "one": FACES[:1],
    "faces": FACES,
    "fourteen": FACES + BLOCKS,
    "mixed": FACES[:2] + [(203, 0, 0, 0, 0, 0, 0, 0), (202, 1, N1, 1, 1, 1, N3)] + FACES[2:4]
    + [(200, 1, N1, 1, N2, N3, N3, 0, 0, 1)] + FACES[4:5] + [(401, 1, N1, 1, N2, 1, N3)] + BLOCKS[:2],
}


@pytest.mark.parametrize("rows", sorted(ROWS))
def test_rows_match_oracle(rows):
    from public_amd import Cruna
    rng = np.random.default_rng(5)
    q = np.zeros(SHAPE + (5,), order="F")
    q[..., 0] = 1 + 0.05 * rng.random(SHAPE)
    q[..., 1:4] = 0.1 * rng.standard_normal(SHAPE + (3,))
    q[..., 4] = 1 / 1.4 + 0.02 * rng.random(SHAPE)
    qref = q.copy(order="F")
    qref[..., 0] *= 1.02
    qref[..., 1] += 0.05
    kv = np.asfortranarray(rng.standard_normal(SHAPE + (3,)))
    kv /= np.linalg.norm(kv, axis=-1, keepdims=True)
    shp = np.asfortranarray(0.1 * rng.random(SHAPE))
    kw = dict(scheme=(O.OPEN,) * 3, mu0=0.01, T0=1 / 1.4, dt=1e-3, bc=ROWS[rows])
    dx = tuple(1.0 / (n - 1) for n in SHAPE)
    cfg = O.Cfg(SHAPE, dx, kvector=kv, **kw)
    ref = O.run_direct(cfg, q, 2, qref=qref, shape=shp)
    with Cruna(SHAPE, dx, **kw) as g:
        g.set_qref(qref)
        g.set_kvector(kv)
        g.set_sponge_shape(shp)
        g.set_state(q)
        g.run_direct(2)
        got = g.get_state()
    for v in range(5):
        err = np.linalg.norm(got[..., v] - ref[..., v]) / np.linalg.norm(ref[..., v])
        assert err < 1e-12, (v, err)
