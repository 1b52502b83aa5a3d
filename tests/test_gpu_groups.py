"""Solver codes in groups of four rows: the layout, and the streaming sweep
that reads them against the CPU oracle, at the edges of groups and tiles."""
import numpy as np
import pytest

import taufactor_amd as tau
from oracle.restate import OracleSolver
from taufactor_amd import _lib, autotune

pytestmark = pytest.mark.gpu


def _binary(shape, seed):
    return (np.random.default_rng(seed).random(shape) < 0.6).astype(np.uint8)


def _grouped(img, H, tile, monkeypatch):
    """A solver that streams with the given depth and tile, as the tuner's choice."""
    monkeypatch.setattr(autotune, "MIN_VOXELS", 0)
    s = tau.Solver(img)
    s._resident, s._auto_cfg = False, (H, tile)
    return s


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 2, 4), (2, 3, 5), (4, 5, 6), (2, 37, 64)])
def test_layout(shape, monkeypatch):
    img = np.stack([_binary(shape, 0), _binary(shape, 1)])
    img[:, :, 0, 0] = 1
    s = _grouped(img, 6, (16, 2, 0), monkeypatch)
    X, Y, Z = shape
    Q, P = (Y + 2) // 4 + 1, (Z + 1) // 2
    got = s._sweep_groups().cpu().numpy().reshape(2, X + 2, Q, P, 4, 2)
    codes = np.zeros((2, X + 2, 4 * Q, 2 * P), np.uint8)
    codes[:, :, 1:Y + 3] = s._codes.cpu().numpy()[:, :, :, 1:2 * P + 1] * 8
    assert np.array_equal(got, codes.reshape(2, X + 2, Q, 4, P, 2).transpose(0, 1, 2, 4, 3, 5))


@pytest.mark.parametrize("H,tile", [(6, (16, 2, 0)), (4, (16, 2, 0)), (6, (12, 4, 0)), (4, (12, 4, 0)),
                                    (6, (16, 2, 4)), (6, (12, 4, 4))])
@pytest.mark.parametrize("shape", [(2, 3, 4), (7, 36, 53), (9, 37, 116), (13, 75, 129), (6, 41, 185), (5, 110, 300)])
def test_matches_oracle(H, tile, shape, monkeypatch):
    """From both colours: five half-sweeps first (an ungrouped launch where H
    is 4 or 6), then blocks of H and a remainder."""
    img = _binary(shape, 3)
    img[:, 0, 0] = 1
    s, o = _grouped(img, H, tile, monkeypatch), OracleSolver(img)
    done = 0
    for n in (5, 2 * H, 2 * H + 3):
        done += n
        s.solve(iter_limit=done, verbose=False, conv_crit=0.0)
        assert np.array_equal(s.field.cpu().numpy(), o.run(n).field.numpy())
    assert s._groups is not None
