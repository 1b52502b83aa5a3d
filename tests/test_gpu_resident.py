"""GPU: the resident sweep (a volume kept in registers, faces exchanged
through a mailbox) against the oracle, value for value, at the edges of its
layout: rows shorter and longer than a wave's lanes, odd sizes, partly filled
patches and tiles, 2-D images, batches, every kind that has it, and a launch
whose waits run out."""
import numpy as np
import pytest
import torch

import taufactor_amd as tau
from oracle.restate import (OracleAnisotropicSolver, OracleElectrodeSolver, OracleFieldSolver, OracleMultiPhaseSolver,
                            OraclePeriodicElectrodeSolver, OraclePeriodicSolver, OracleSolver)

pytestmark = pytest.mark.gpu


def _binary(shape, seed, p=0.65):
    return (np.random.default_rng(seed).random(shape) < p).astype(np.uint8)


def _same(s, o, n):
    """s after n iterations (resident, two blocks) holds o's field."""
    s.solve(iter_limit=n, verbose=False, conv_crit=0.0)
    assert s._resident, "the resident sweep did not run"
    assert np.array_equal(s.field.cpu().numpy(), o.run(n).field.numpy())


# one voxel; rows of 1, 2, 63..65 pairs; rows of 4, 8, 16 and 32 voxels per
# lane; last patch and last tile partly filled in x and y
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 2), (5, 7, 9), (9, 6, 127), (4, 5, 128), (6, 9, 129),
                                   (7, 10, 255), (3, 4, 257), (17, 33, 30), (66, 5, 3), (5, 9, 600), (2, 3, 1100)])
def test_solver_shapes(shape):
    img = _binary(shape, sum(shape))
    # (a check of a single layer has no fluxes to compare)
    _same(tau.Solver(img), OracleSolver(img), 109 if shape[0] > 1 else 57)


# one volume per compiled shape that the small ones above do not take: (voxels
# per lane and row, patch, waves) of the plan
@pytest.mark.parametrize("shape,plan", [
    ((100, 60, 9), (2, 1, 2, 16)), ((120, 72, 9), (2, 2, 2, 16)), ((130, 130, 9), (2, 2, 4, 16)),
    ((230, 138, 9), (2, 4, 4, 16)), ((330, 198, 9), (2, 6, 8, 8)), ((100, 60, 140), (4, 1, 2, 16)),
    ((120, 72, 140), (4, 2, 2, 16)), ((130, 130, 140), (4, 2, 3, 16)), ((215, 129, 140), (4, 2, 4, 16)),
    ((230, 138, 140), (4, 4, 6, 8)), ((290, 174, 140), (4, 4, 8, 8)), ((420, 252, 5), (2, 8, 8, 8)),
    ((100, 60, 260), (8, 1, 2, 16)), ((150, 90, 260), (8, 2, 2, 16)), ((120, 72, 260), (8, 2, 3, 8)), ((130, 130, 260), (8, 3, 4, 8)),
    ((100, 60, 520), (16, 2, 2, 8))])
def test_every_patch(shape, plan):
    img = _binary(shape, 5)
    s = tau.Solver(img)
    assert s._resident_sweep()
    p = s._resident.plan
    assert (p.elems, p.px, p.py, p.waves) == plan
    _same(s, OracleSolver(img), 7)


@pytest.mark.parametrize("shape", [(1, 2), (33, 40), (16, 129), (40, 300), (9, 515), (35, 1030)])
def test_images(shape):
    img = _binary(shape, shape[0], p=0.8)
    s = tau.Solver(img)
    assert s._resident_sweep() and s._resident.plan.lane_y
    _same(s, OracleSolver(img), 109 if shape[0] > 1 else 57)


@pytest.mark.parametrize("shape", [(20, 21, 22), (120, 72, 9), (130, 130, 9)])
def test_resumed_on_the_other_colour(shape):
    """A launch that starts on an odd iteration (patches with even sides have
    a kernel per first colour)."""
    img = _binary(shape, 8)
    s, o = tau.Solver(img), OracleSolver(img)
    _same(s, o, 5)
    s.solve(iter_limit=9, verbose=False, conv_crit=0.0)
    assert s._resident and np.array_equal(s.field.cpu().numpy(), o.run(4).field.numpy())


def test_batch():
    img = np.stack([_binary((18, 21, 23), i) for i in range(3)])
    _same(tau.Solver(img), OracleSolver(img), 109)


@pytest.mark.parametrize("shape", [(12, 2, 2), (9, 10, 12), (8, 34, 128), (20, 18, 132)])
def test_periodic(shape):
    """Rows and lanes wrap round, inside a workgroup and across; the ghosts
    end as the reference's."""
    img = _binary(shape, 3)
    _same(tau.PeriodicSolver(img), OraclePeriodicSolver(img), 109)


@pytest.mark.parametrize("shape", [(9, 11, 13), (14, 40), (6, 9, 131)])
def test_anisotropic(shape):
    img = _binary(shape, 4)
    _same(tau.AnisotropicSolver(img, (1.0, 1.3, 2.0)), OracleAnisotropicSolver(img, (1.0, 1.3, 2.0)), 109)


@pytest.mark.parametrize("periodic", [False, True])
def test_electrode(periodic):
    img = np.random.default_rng(8).choice([0, 1, 5], size=(2, 15, 12, 18), p=[0.3, 0.6, 0.1])
    cls, ocls = ((tau.PeriodicElectrodeSolver, OraclePeriodicElectrodeSolver) if periodic else
                 (tau.ElectrodeSolver, OracleElectrodeSolver))
    _same(cls(img, spacing=0.5), ocls(img, spacing=0.5), 109)


@pytest.mark.parametrize("cls,ocls", [(tau.Solver, OracleSolver), (tau.PeriodicSolver, OraclePeriodicSolver)])
def test_a_wait_that_runs_out(cls, ocls):
    """With a single poll per wait the exchange is lost; the iterations are
    repeated by the streaming sweep and end on the same field."""
    img = _binary((40, 44, 46), 6)
    s = cls(img)
    assert s._resident_sweep()
    s._resident.spin = 1
    s.solve(iter_limit=330, verbose=False, conv_crit=0.0)
    assert np.array_equal(s.field.cpu().numpy(), ocls(img).run(330).field.numpy())
    s.reset()
    s.solve(iter_limit=230, verbose=False, conv_crit=0.0)
    assert np.array_equal(s.field.cpu().numpy(), ocls(img).run(230).field.numpy())


def test_tiny_values_take_the_division():
    """Subnormal and tiny fields: the quotients the reciprocal does not give."""
    img = _binary((12, 10, 70), 9, p=0.8)
    for cls, ocls, extra in ((tau.Solver, OracleSolver, ()), (tau.AnisotropicSolver, OracleAnisotropicSolver,
                                                             ((1.0, 1.2, 0.7),)),
                             (tau.ElectrodeSolver, OracleElectrodeSolver, ())):
        s, o = cls(img, *extra), ocls(img, *extra)
        rng = np.random.default_rng(2)
        f = o.field.numpy().copy()
        tiny = np.ldexp(rng.standard_normal(f.shape), rng.integers(-149, -95, f.shape)).astype(np.float32)
        f[:, 1:-1, 1:-1, 1:-1] = tiny[:, 1:-1, 1:-1, 1:-1] * (f[:, 1:-1, 1:-1, 1:-1] != 0)
        f[:, [0, -1]] = 0.0  # nothing large flows in
        o.field = torch.from_numpy(f.copy())
        s.field = torch.from_numpy(f)
        _same(s, o, 11)


def test_streams_take_turns():
    """Solvers on streams of their own, in threads: their resident launches
    wait for each other's end on the device, none runs out of its waits."""
    import threading

    imgs = [_binary((120, 110, 100), i) for i in range(3)]
    solvers = [None] * len(imgs)

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            s = solvers[i] = tau.Solver(imgs[i])
            s.solve(iter_limit=310, verbose=False, conv_crit=0.0)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(imgs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for s, img in zip(solvers, imgs):
        assert s._resident
        assert np.array_equal(s.field.cpu().numpy(), OracleSolver(img).run(310).field.numpy())


def _map(shape, seed):
    """Voxel diffusivities, a fifth of them 0."""
    rng = np.random.default_rng(seed)
    k = rng.uniform(0.05, 2.0, size=shape).astype(np.float32)
    k[rng.random(shape) < 0.2] = 0.0
    return k


@pytest.mark.parametrize("shape,plan", [
    ((3, 4, 5), (2, 1, 1, 16)), ((9, 8, 127), (2, 1, 1, 16)), ((100, 60, 5), (2, 1, 2, 16)),
    ((120, 72, 5), (2, 2, 2, 16)), ((130, 130, 5), (2, 2, 3, 16)), ((215, 129, 5), (2, 4, 4, 8)),
    ((7, 5, 140), (4, 1, 1, 16)), ((100, 60, 140), (4, 1, 2, 16)), ((120, 72, 140), (4, 1, 3, 16)),
    ((150, 90, 140), (4, 2, 4, 8)), ((130, 130, 140), (4, 3, 3, 8)), ((6, 3, 260), (8, 1, 1, 16)),
    ((100, 60, 260), (8, 1, 3, 8)), ((80, 80, 260), (8, 2, 2, 8)), ((6, 3, 520), (16, 1, 1, 8))])
def test_field_every_patch(shape, plan):
    k = _map(shape, 2)
    s = tau.FieldSolver(k)
    assert s._resident_sweep()
    p = s._resident.plan
    assert (p.elems, p.px, p.py, p.waves) == plan
    _same(s, OracleFieldSolver(k), 7)


def test_field_batch_in_groups():
    """Five volumes of which two fit at once, checks and a resumed solve."""
    k = _map((5, 112, 100, 90), 3)
    s = tau.FieldSolver(k)
    assert s._resident_sweep() and 1 < s._resident.per < 5
    _same(s, OracleFieldSolver(k), 103)


def _labels(shape, n, seed):
    return np.random.default_rng(seed).integers(0, n, size=shape).astype(np.uint8)


D3 = {0: 0.0, 1: 1.0, 2: 0.1}
D7 = {0: 0.0, 1: 1.0, 2: 0.5, 3: 0.25, 4: 0.12, 5: 2.0, 6: 1 / 3}


@pytest.mark.parametrize("shape,plan", [
    ((3, 4, 5), (2, 1, 1, 16)), ((9, 8, 127), (2, 1, 1, 16)), ((100, 60, 5), (2, 1, 2, 16)),
    ((120, 72, 5), (2, 2, 2, 16)), ((130, 130, 5), (2, 2, 4, 16)), ((230, 138, 5), (2, 4, 6, 8)),
    ((7, 5, 140), (4, 1, 1, 16)), ((100, 60, 140), (4, 1, 2, 16)), ((120, 72, 140), (4, 2, 2, 16)),
    ((130, 130, 140), (4, 3, 3, 8)), ((185, 111, 140), (4, 2, 6, 8)), ((215, 129, 140), (4, 4, 4, 8)),
    ((290, 174, 5), (2, 4, 8, 8)), ((6, 3, 260), (8, 1, 1, 16)), ((100, 60, 260), (8, 1, 2, 16)),
    ((120, 72, 260), (8, 2, 3, 8)), ((150, 90, 260), (8, 2, 4, 8)), ((6, 3, 520), (16, 1, 1, 8)),
    ((60, 36, 520), (16, 1, 2, 8))])
def test_multiphase_every_patch(shape, plan):
    img = _labels(shape, 3, 7)
    s = tau.MultiPhaseSolver(img, dict(D3))
    assert s._resident_sweep()
    p = s._resident.plan
    assert (p.elems, p.px, p.py, p.waves) == plan
    _same(s, OracleMultiPhaseSolver(img, dict(D3)), 7)


@pytest.mark.parametrize("Ds,n", [(D3, 3), (D7, 7)])
@pytest.mark.parametrize("shape", [(14, 13, 12), (8, 9, 131), (33, 150), (2, 9, 8, 70)])
def test_multiphase_blocks(Ds, n, shape):
    """Face codes and (seven values) class codes over two blocks, first and
    last layers, images and batches."""
    img = _labels(shape, n, 11)
    _same(tau.MultiPhaseSolver(img, dict(Ds)), OracleMultiPhaseSolver(img, dict(Ds)), 109)


def test_field_and_multiphase_lost_waits():
    k, img = _map((3, 60, 61, 62), 4), _labels((50, 51, 52), 3, 5)
    for s, o in ((tau.FieldSolver(k), OracleFieldSolver(k)),
                 (tau.MultiPhaseSolver(img, dict(D3)), OracleMultiPhaseSolver(img, dict(D3)))):
        assert s._resident_sweep()
        s._resident.spin = 1
        s.solve(iter_limit=130, verbose=False, conv_crit=0.0)
        assert np.array_equal(s.field.cpu().numpy(), o.run(130).field.numpy())
