"""GPU: solvers that change between resident and streaming launches, or stop
between checks, against the oracle's field."""
import numpy as np
import pytest

import taufactor_amd as tau
from oracle.restate import (OracleAnisotropicSolver, OracleElectrodeSolver, OracleFieldSolver, OracleMultiPhaseSolver,
                            OraclePeriodicElectrodeSolver, OraclePeriodicSolver, OracleSolver)
from taufactor_amd import solver

pytestmark = pytest.mark.gpu


def _labels(shape, n, seed):
    return np.random.default_rng(seed).integers(0, n, size=shape).astype(np.uint8)


D3 = {0: 0.0, 1: 1.0, 2: 0.1}


@pytest.mark.parametrize("cls,ocls,n,extra", [(tau.Solver, OracleSolver, 2, ()),
                                              (tau.MultiPhaseSolver, OracleMultiPhaseSolver, 3, (D3,))])
def test_back_from_a_hand_set_depth(cls, ocls, n, extra):
    """Streaming up to a check, then the default: the converged field is that
    of the last check."""
    img = _labels((22, 20, 21), n, 3)
    img[:, 4:9, 5:12] = 1
    s = cls(img, *(dict(e) for e in extra))
    s.half_sweeps_per_pass = 4
    s.solve(iter_limit=200, verbose=False, conv_crit=0.0)
    s.half_sweeps_per_pass = None
    s.solve(verbose=False)
    assert s.converged and s.iter > 200 and s._resident
    assert np.array_equal(s.field.cpu().numpy(), ocls(img, *(dict(e) for e in extra)).run(s.iter).field.numpy())


def test_periodic_with_other_electrode_values():
    """The x ghosts of a field that is set before the first solve hold in
    every buffer of a resident periodic solve."""
    img = (np.random.default_rng(6).random((18, 20, 22)) < 0.7).astype(np.uint8)
    s, o = tau.PeriodicSolver(img), OraclePeriodicSolver(img)
    f = o.field.clone()
    f[:, 0], f[:, -1] = f[:, 0] * 0.5, f[:, -1] * 2
    o.field = f.clone()
    s.field = f.to(s.device)
    for n in (230, 170):
        o.run(n)
        s.solve(iter_limit=s.iter + n, verbose=False, conv_crit=0.0)
        assert s._resident and np.array_equal(s.field.cpu().numpy(), o.field.numpy())


@pytest.mark.parametrize("cls,ocls", [(tau.Solver, OracleSolver), (tau.PeriodicSolver, OraclePeriodicSolver)])
@pytest.mark.parametrize("by_hand", [False, True])
def test_lost_waits_of_solves_that_end_between_checks(cls, ocls, by_hand):
    """With a single poll per wait the first launch is lost; what it read is
    not written again before the loss is known."""
    img = (np.random.default_rng(6).random((40, 44, 46)) < 0.65).astype(np.uint8)
    s, o = cls(img), ocls(img)
    assert s._resident_sweep()
    s._resident.spin = 1
    for n in (50, 10, 70):
        o.run(n)
        s.solve(iter_limit=s.iter + n, verbose=False, conv_crit=0.0)
        assert s._resident is False, "no wait ran out"
        if by_hand:
            s.half_sweeps_per_pass = 4
    assert np.array_equal(s.field.cpu().numpy(), o.field.numpy())


@pytest.mark.parametrize("cls,ocls,shape", [(tau.Solver, OracleSolver, (5, 9, 600)), (tau.Solver, OracleSolver, (14, 1030)),
                                            (tau.PeriodicSolver, OraclePeriodicSolver, (6, 8, 1024)),
                                            (tau.MultiPhaseSolver, OracleMultiPhaseSolver, (3, 7, 300))])
def test_measured_against_the_streaming_sweep(cls, ocls, shape):
    """Layouts of which it is not known which sweep is the faster change from
    one to the other inside a solve; the next solver takes the faster one."""
    extra = (dict(D3),) if cls is tau.MultiPhaseSolver else ()
    img = _labels(shape, 3 if extra else 2, 9) if extra else (np.random.default_rng(9).random(shape) < 0.8).astype(np.uint8)
    field = ocls(img, *extra).run(630).field.numpy()
    for _ in range(2):
        s = cls(img, *extra)
        s.solve(iter_limit=630, verbose=False, conv_crit=0.0)
        assert s._resident.measured and s._resident.key in solver._resident_faster
        assert np.array_equal(s.field.cpu().numpy(), field)


@pytest.mark.parametrize("kind", ["field", "multiphase", "anisotropic", "electrode", "periodic electrode"])
def test_lost_waits_of_every_kind(kind):
    """With a single poll per wait a launch is lost, the solver knows, and its
    field is the repeated one."""
    shape = (40, 44, 46)
    if kind == "field":
        k = np.random.default_rng(4).uniform(0.05, 2.0, size=(2, *shape)).astype(np.float32)
        s, o = tau.FieldSolver(k), OracleFieldSolver(k)
    elif kind == "multiphase":
        img = _labels(shape, 3, 5)
        s, o = tau.MultiPhaseSolver(img, dict(D3)), OracleMultiPhaseSolver(img, dict(D3))
    elif kind == "anisotropic":
        img = _labels(shape, 2, 5)
        s, o = (c(img, (1.0, 1.3, 2.0)) for c in (tau.AnisotropicSolver, OracleAnisotropicSolver))
    else:
        img = _labels(shape, 3, 5)
        cls, ocls = ((tau.ElectrodeSolver, OracleElectrodeSolver) if kind == "electrode" else
                     (tau.PeriodicElectrodeSolver, OraclePeriodicElectrodeSolver))
        s, o = cls(img), ocls(img)
    assert s._resident_sweep()
    s._resident.spin = 1
    s.solve(iter_limit=130, verbose=False, conv_crit=0.0)
    assert s._resident is False, "no wait ran out"
    assert np.array_equal(s.field.cpu().numpy(), o.run(130).field.numpy())
