"""CPU: the x tile of uneven batches whose largest volumes fill the device."""
import numpy as np
import pytest
import torch

from taufactor_amd import _lib
from taufactor_amd.batch import BatchSolver


@pytest.mark.parametrize("edges,tx", [([64, 130], 16), ([190], 16), ([205], 24), ([205, 100, 60], 24), ([240], 32),
                                      ([280], 48), ([190] * 3, 48), ([160] * 4, 32), ([120] * 8, 24),
                                      (list(range(32, 113, 3)), 16), ([289], 16)])
def test_one_round_of_the_largest(edges, tx, monkeypatch):
    b = object.__new__(BatchSolver)
    b.shapes = [(e, e, e) for e in edges]
    b._lib, b.device = _lib.load(), torch.device("cpu")
    b.half_sweeps_per_pass, b.tile, b.autotune = None, None, True
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: type("P", (), {"multi_processor_count": 256}))
    if edges == [289]:
        b.shapes = [(289, 300, 290)]
    assert b._launch_config() == (5, (16, 2, tx))
    largest = [s for s in b.shapes if np.prod(s) >= 0.9 * max(np.prod(s) for s in b.shapes)]
    tiles = sum(b._tile_count(s, 5, _lib.Tile(16, 2, tx)) for s in largest)
    assert tiles <= 256 or edges == [289]
