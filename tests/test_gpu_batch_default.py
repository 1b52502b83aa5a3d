"""Uneven batches by the size rule against the same batch with the depth and
tile set by hand, value for value, on both sides of each of its lines."""
import numpy as np
import pytest

import taufactor_amd as tau
from taufactor_amd import autotune

pytestmark = pytest.mark.gpu


def _batch(shapes):
    rng = np.random.default_rng(len(shapes))
    return [(rng.random(s) < 0.6).astype(np.uint8) for s in shapes]


@pytest.mark.parametrize("shapes,config", [
    ([(5, 6, 7), (33, 17, 40), (18, 70, 66)], (5, (8, 2, 16))),
    ([(128, 127, 129), (17, 3, 2)], (5, (8, 2, 16))),
    ([(128, 127, 129), (17, 3, 5)], (5, (16, 2, 16))),
    ([(289, 300, 290), (40, 9, 11)], (5, (16, 2, 16))),
    ([(290, 300, 290), (40, 9, 11)], (5, (16, 2, 32)))])
def test_size_rule(shapes, config):
    imgs = _batch(shapes)
    a, b = tau.BatchSolver(imgs), tau.BatchSolver(imgs)
    assert a._launch_config() == config
    b.half_sweeps_per_pass, b.tile = 4, (8, 2, 64)
    a.solve(iter_limit=200)
    b.solve(iter_limit=200)
    assert np.array_equal(a.iters, b.iters) and np.array_equal(a.tau, b.tau)
    for v in range(len(shapes)):
        assert np.array_equal(np.asarray(a.field(v).cpu()), np.asarray(b.field(v).cpu()))


def test_large_batches_are_tuned():
    assert autotune.batch_default(2 ** 26 - 1) == (5, (16, 2, 32))
    assert autotune.batch_default(2 ** 26) == (None, None)
