"""Weight gradients of batches and windows, whatever their tiles.

One training sample, so every batch has the whole field's gradient: as one box
or several (one to several tiles per work-group), periodic, or as a window of
the sample's size with its halo of zeros outside (24 points: partial tiles in
x).  One Adam step moves every parameter by lr g / (|g| + eps), nearly lr sign g,
so two gradients that agree to FP32 summation error (1e-6 of the terms' sum) give
equal steps except for the few entries that are themselves that small: at
most one in 200 with a step that differs by more than 1 %.
"""
import numpy as np
import pytest

from test_gpu_closure import IN_STD, OUT_STD, P_REF, S, _state

pytestmark = pytest.mark.gpu


def _step(batch, crop, seed):
    from public_amd import Closure
    net = Closure(S, seed=6)
    net.set_norm(IN_STD, OUT_STD, P_REF)
    q = _state(4)
    target = np.asfortranarray(np.random.default_rng(1).standard_normal(q.shape) * OUT_STD)
    net.add_sample(q, target)
    p0 = net.get_params()
    net.train(1, lr=1e-3, batch=batch, crop=crop, seed=seed)
    d = net.get_params() - p0
    net.close()
    return d


@pytest.mark.parametrize("batch,crop", [(2, 0), (31, 0), (40, 0), (1, S), (9, S)])
def test_batches_and_windows_have_the_whole_fields_gradient(batch, crop):
    ref = _step(1, 0, 0)
    got = _step(batch, crop, 3)
    used = ref != 0.0
    assert used.mean() > 0.5
    assert np.array_equal(got != 0.0, used)
    assert (np.abs(got - ref)[used] > 1e-5).mean() < 5e-3
