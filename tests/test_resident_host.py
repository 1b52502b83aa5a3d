"""CPU: the host logic of the resident and streaming launches (which buffer a
launch reads and writes, launches ahead of a check that are dropped, launches
whose waits ran out) on a stand-in for the device.

The stand-in's field holds, in every interior voxel, the number of iterations
behind it, and in its x ghosts the boundary value it was given; a launch
requires its source to hold an iteration of its colour.  As on the device, a
lost resident launch stores its number in the status and leaves dst void, and
later resident launches write nothing until the status is cleared."""
import contextlib
import ctypes
import random
import threading

import numpy as np
import pytest
import torch

import taufactor_amd as tau
from taufactor_amd import _lib, solver as solver_module

VOID = -1e6  # what a lost launch leaves
X = Y = Z = 4


class Device:
    """The library entry points that a solve calls, on host memory."""

    def __init__(self):
        self.lost = set()  # resident launches (counted from 1) whose waits run out
        self.launches = 0
        self.boundary = 0.5
        self.clock, self.cost = 0.0, {"resident": 1.0, "streaming": 2.0}  # time of a half-sweep
        self.ran = []  # (path, half-sweeps) of each launch
        self.status = None  # of the solver made last
        self.solver = None

    def _view(self, p, dtype, n):
        return np.ctypeslib.as_array((dtype * n).from_address(p))

    def _field(self, p):
        return self._view(p, ctypes.c_float, (X + 2) * (Y + 2) * (Z + 2)).reshape(X + 2, Y + 2, Z + 2)

    def _run(self, src, dst, n, colour):
        s, d = self._field(src), self._field(dst)
        it = s[1, 1, 1]
        assert np.all(s[1:-1, 1:-1, 1:-1] == it) and it >= 0, "a void field was read"
        assert np.all(s[[0, -1], 1:-1, 1:-1] == self.boundary), "a field with other boundary values was read"
        assert int(it) & 1 == colour, f"iteration {it} read for a launch of colour {colour}"
        d[1:-1, 1:-1, 1:-1] = it + n

    def took(self, path, n):
        self.clock += self.cost[path] * n
        self.ran.append((path, n))

    def tf_sweep(self, src, dst, codes, hm, n_table, kind, B, nx, ny, nz, w, colour, h, tile, stream):
        self.took("streaming", h)
        r = self.solver._resident
        if r and self.status is not None and self.status[0] and any(e[0] >= self.status[0] for e in r.log):
            # the host does not know of the loss yet: whatever was read
            self._field(dst)[1:-1, 1:-1, 1:-1] = VOID
        else:
            self._run(src, dst, h, colour)
        return 0

    def tf_resident_plan(self, kind, B, nx, ny, nz, cus, plan):
        p = plan._obj
        p.elems, p.px, p.py, p.waves, p.wy, p.tiles, p.mail_bytes = 2, 1, 1, 16, 4, 1, 64
        return 1

    def tf_sweep_resident(self, src, dst, codes, table, n_table, kind, B, nx, ny, nz, w, colour, n, plan, section,
                          mail, mail_bytes, tag, status, launch_id, spin, stream):
        st = self.status = self._view(status, ctypes.c_int32, 1)
        self.launches += 1
        self.took("resident", n)
        if st[0]:
            return 0
        if self.launches in self.lost:
            st[0] = launch_id
            self._field(dst)[1:-1, 1:-1, 1:-1] = VOID
        else:
            self._run(src, dst, n, colour)
        return 0

    def tf_wrap_ghosts_from(self, src, dst, *args):
        a, b = (self._field(p)[1, 1, 1] for p in (src, dst))
        assert a == b - 1 or b == VOID, "ghosts of another field than the one before"
        return 0

    def tf_hbm_copy(self, src, dst, n, stream):
        ctypes.memmove(dst, src, n)
        return 0

    def tf_layer_sums_ws(self, field, codes, hm, n_classes, kind, B, nx, ny, nz, flux, conc, ws, n_ws, stream):
        # the value of the field that is checked
        self._view(flux, ctypes.c_double, 1)[0] = self._field(field)[1, 1, 1]
        return 0


class _Event:
    device = None

    def __init__(self, *a, **k):
        pass

    def record(self, *a):
        self.at = self.device.clock

    def synchronize(self):
        pass

    def query(self):
        return True

    def elapsed_time(self, end):
        return end.at - self.at


class _Stream:
    cuda_stream = 7

    def wait_event(self, e):
        pass

    def record_event(self, e=None):
        return e or _Event()

    def __eq__(self, other):
        return self.cuda_stream == other.cuda_stream

    __hash__ = None


@pytest.fixture
def device(monkeypatch):
    for name, f in {"device": lambda d: contextlib.nullcontext(), "synchronize": lambda d=None: None,
                    "Event": _Event, "current_stream": lambda d=None: _Stream(),
                    "get_device_properties": lambda d: type("P", (), {"multi_processor_count": 256})}.items():
        monkeypatch.setattr(torch.cuda, name, f)
    monkeypatch.setattr(solver_module, "_resident_turn", {})
    monkeypatch.setattr(_lib, "stream_handle", lambda d: _Stream.cuda_stream)
    monkeypatch.setattr(solver_module, "_resident_faster", {})
    _Event.device = Device()
    return _Event.device


def make(cls, device, spare=True):
    """A solver of the class on the stand-in, its fields at iteration 0."""

    class Stub(cls):
        stop = None  # iteration at which the check finds convergence
        broken = None  # iteration from which a check is interrupted

        def _launch_operands(self, H, tile):
            return self.kind | self._sweep_flags, 0, None, 0, tile

        def compute_metrics(self):
            if self.broken is not None and self.iter >= self.broken:
                raise KeyboardInterrupt
            flux, _ = self._layer_sums()
            assert self._sums_host[0] == self.iter, "another field was checked"
            done = self.stop is not None and self.iter >= self.stop
            return np.ones(1), np.full(1, 0.0 if done else 1.0)

        def _end_simulation(self, iterations, verbose):
            pass

    s = object.__new__(Stub)
    s.batch_size, s.Nx, s.Ny, s.Nz = 1, X, Y, Z
    s.device = torch.device("cpu")
    s._lib, device.solver = device, s
    s._w32, s.omega = 1.5, 1.5
    s.half_sweeps_per_pass = s.tile = s._auto_cfg = None
    s.autotune = True
    shape = (1, X + 2, Y + 2, Z + 2)
    s._fields = [_lib.slack_buffer(shape, torch.float32, s.device) for _ in range(2)]
    for f in s._fields:
        f[:, [0, -1], 1:-1, 1:-1] = device.boundary
    s._field_init = _lib.slack_buffer(shape, torch.float32, s.device)
    s._copy_field(s._fields[0], s._field_init)
    s._spare = None
    if spare and s._zero_yz_ghosts:
        s._spare = _lib.slack_buffer(shape, torch.float32, s.device)
        s._copy_field(s._field_init, s._spare)
    s._codes = s._sweep_codes = torch.zeros(4096, dtype=torch.uint8)
    s._groups = s._hm_lut = s._launch_events = s._checked = None
    s._n_classes = 0
    s._sums = torch.zeros(2 * X + 1, dtype=torch.float64)
    s._sums_host = torch.zeros(2 * X + 1, dtype=torch.float64)
    s._sums_ws = torch.zeros(1, dtype=torch.float64)
    s._resident = s._sums_ready = None
    s._cur = s._ahead = s.iter = s.old_tau = 0
    s.converged = False
    s.tau = s.tau_x = s.D_eff = None
    return s


def holds(s, device):
    """The solver's field is that of its iteration, with its boundary."""
    f = s.field[0].numpy()
    assert np.all(f[1:-1, 1:-1, 1:-1] == s.iter), (f[1, 1, 1], s.iter)
    assert np.all(f[[0, -1], 1:-1, 1:-1] == device.boundary)


def run(s, limit, stop=None):
    s.stop, s.converged = stop, False
    s.solve(iter_limit=limit, verbose=False)


def test_back_from_a_hand_set_depth(device):
    """A solve that streams (depth set by hand) and ends on a check, then the
    default again: a resident solve that converges ends on its own field, not
    on one that the streaming solve's last decision kept."""
    s = make(tau.Solver, device)
    s.half_sweeps_per_pass = 4
    run(s, 200)
    s.half_sweeps_per_pass = None
    run(s, 10000, stop=400)
    assert s.converged and s.iter == 400
    holds(s, device)


def test_boundary_set_before_the_third_buffer(device):
    """A field with other x ghosts, set before a periodic solver's first
    launch, holds in the third buffer too."""
    s = make(tau.PeriodicSolver, device)
    f = s.field.clone()
    f[:, [0, -1], 1:-1, 1:-1] = device.boundary = 0.25
    s.field = f
    run(s, 330)
    assert s._resident.third is not None
    holds(s, device)


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
@pytest.mark.parametrize("lost", [1, 2, 3])
def test_lost_launch_of_solves_that_end_between_checks(cls, lost, device):
    """A solve that ends between checks returns a field that is known: a lost
    launch is repeated before the buffer that it read is written again."""
    s = make(cls, device)
    device.lost = {lost}
    for limit in (50, 60, 130, 250):
        run(s, limit)
        assert s.iter == limit and not (s._resident and s._resident.log)
        holds(s, device)
    assert s._resident is False


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
def test_lost_launch_then_a_hand_set_depth(cls, device):
    s = make(cls, device)
    device.lost = {1}
    run(s, 50)
    s.half_sweeps_per_pass = 4
    run(s, 130)
    holds(s, device)


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
@pytest.mark.parametrize("spare", [False, True])
@pytest.mark.parametrize("measured", [None, "resident", "streaming"])
@pytest.mark.parametrize("seed", range(25))
def test_any_sequence(cls, spare, measured, seed, device, monkeypatch):
    """Solves to any iteration, converged or not, with the depth set by hand
    or not, interrupted in a check, resets, new fields, lost launches, the two
    sweeps measured against each other: the field is always that of the
    solver's iteration."""
    rng = random.Random(seed)
    if measured:
        monkeypatch.setattr(solver_module, "_resident_unsure", lambda *a: True)
        device.cost[measured] = 0.5
    s = make(cls, device, spare)
    device.lost = set(rng.sample(range(1, 40), rng.randint(0, 2)))
    for _ in range(12):
        act = rng.random()
        if act < 0.1:
            s.reset()
            device.boundary = 0.5
        elif act < 0.2:
            f = s.field.clone()
            f[:, [0, -1], 1:-1, 1:-1] = device.boundary = rng.choice([0.25, 0.5, 1.0])
            s.field = f
        elif act < 0.35:
            s.half_sweeps_per_pass = rng.choice([None, None, 3, 4])
        elif act < 0.45:
            s.broken = s.iter + rng.randint(0, 200)
            with contextlib.suppress(KeyboardInterrupt):
                run(s, s.iter + 300)
            s.broken = None
        else:
            run(s, s.iter + rng.choice([1, 7, 40, 100, 100 - s.iter % 100, 230]),
                rng.choice([None, s.iter + 100, s.iter + 200]))
        if rng.random() < 0.7:
            holds(s, device)
    holds(s, device)


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
def test_field_read_in_a_check_after_a_lost_launch_ahead(cls, device):
    """The launch ahead of the check at 100 is lost and a check that looks at
    the field finds out: there is nothing to repeat."""
    s = make(cls, device)
    device.lost = {2}
    metrics = s.compute_metrics

    def look():
        out = metrics()
        if s.iter == 100:  # (later checks have streaming launches ahead)
            holds(s, device)
        return out

    s.compute_metrics = look
    run(s, 230)
    assert s._resident is False
    holds(s, device)


def test_repeated_on_the_solvers_device(device, monkeypatch):
    """A field read outside of solve() that finds a lost launch repeats it on
    the solver's device, whichever is current."""
    current = []

    @contextlib.contextmanager
    def on(d):
        current.append(d)
        try:
            yield
        finally:
            current.pop()

    monkeypatch.setattr(torch.cuda, "device", on)
    s = make(tau.Solver, device)
    device.lost = {1}
    s.broken = 100
    with contextlib.suppress(KeyboardInterrupt):
        run(s, 200)
    sweep = device.tf_sweep

    def checked(*args):
        assert current and current[-1] == s.device
        return sweep(*args)

    device.tf_sweep = checked
    holds(s, device)
    assert s._resident is False and s.iter == 100


def test_walltime_includes_a_repetition(device, monkeypatch):
    """solve() waits for the device after its last launch, that of a
    repetition too."""
    s = make(tau.Solver, device)
    device.lost = {1}
    calls = []
    sweep = device.tf_sweep
    device.tf_sweep = lambda *a: calls.append("sweep") or sweep(*a)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda d=None: calls.append("wait"))
    run(s, 50)
    assert "sweep" in calls and calls[-1] == "wait"


class _Turn:
    """Streams and events that note what was asked of them."""

    def __init__(self, monkeypatch, device):
        self.log = []
        self.stream_of = {}  # of each thread
        turn = self

        class Event(_Event):
            def record(self, stream=None):
                self.at = device.launches

        class Stream:
            def __init__(self, handle):
                self.cuda_stream, self.gone = handle, False

            def __eq__(self, other):
                return self.cuda_stream == other.cuda_stream

            def wait_event(self, e):
                turn.log.append((self.cuda_stream, e.at))

            def record_event(self, e=None):
                assert not self.gone, "a stream that is gone was used"
                e = e or Event()
                e.record(self)
                return e

        self.stream = Stream
        monkeypatch.setattr(torch.cuda, "Event", Event)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: self.stream_of[threading.get_ident()])

    def run(self, stream, s, limit):
        self.stream_of[threading.get_ident()] = stream
        run(s, limit)


@pytest.mark.parametrize("interrupted", [False, True])
def test_a_stream_that_is_gone(interrupted, device, monkeypatch):
    """A solve on a stream that is destroyed after it, then one on another
    stream: the first stream is not used again, and launches that an
    interrupted solve left on it are waited for."""
    turn = _Turn(monkeypatch, device)
    first, second = make(tau.Solver, device), make(tau.Solver, device)
    a, b = turn.stream(1), turn.stream(2)
    first.broken = 100 if interrupted else None
    with contextlib.suppress(KeyboardInterrupt):
        turn.run(a, first, 150)
    launches = device.launches
    a.gone = True
    turn.run(b, second, 50)
    assert turn.log == ([(2, launches)] if interrupted else [])


def test_turns_of_threads(device, monkeypatch):
    """A solve on a stream of its own in another thread, while the first one
    stands in a check: each waits for the other's launches."""
    turn = _Turn(monkeypatch, device)
    first, second = make(tau.Solver, device), make(tau.Solver, device)
    a, b = turn.stream(1), turn.stream(2)
    metrics = first.compute_metrics

    def meanwhile():
        if first.iter == 100:
            t = threading.Thread(target=turn.run, args=(b, second, 50))
            t.start()
            t.join()
        return metrics()

    first.compute_metrics = meanwhile
    turn.run(a, first, 150)
    # launches 1, 2 (ahead) and 4 of the first solve, 3 of the second, which
    # had ended before 4
    assert turn.log == [(2, 2)]
    assert first.iter == 150 and second.iter == 50
    assert solver_module._resident_turn == {}


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
def test_no_wait_for_the_status_inside_a_solve(cls, device):
    """The status comes with the sums of a check; only a solve's end asks."""
    s = make(cls, device)
    asked = []
    settle = s._settle
    s._settle = lambda: asked.append(s.iter) or settle()
    run(s, 1000, stop=500)
    assert asked == [500]


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
@pytest.mark.parametrize("what", ["zeros", "slack_buffer"])
def test_no_memory_for_the_resident_sweep(cls, what, device, monkeypatch):
    """A solver whose mailbox or third buffer does not fit streams."""
    s = make(cls, device)

    def full(*args, **kwargs):
        raise torch.cuda.OutOfMemoryError("full")

    monkeypatch.setattr(torch if what == "zeros" else _lib, what, full)
    run(s, 230)
    assert bool(s._resident) == (what == "slack_buffer" and cls is tau.Solver)
    holds(s, device)


def test_no_memory_for_code_groups(device, monkeypatch):
    """A volume whose codes in groups do not fit sweeps without them."""
    s = make(tau.Solver, device)
    device.tf_sweep_groups_bytes = lambda *a: 64

    def full(*args, **kwargs):
        raise torch.cuda.OutOfMemoryError("full")

    monkeypatch.setattr(solver_module.autotune, "MIN_VOXELS", 0)
    monkeypatch.setattr(torch, "empty", full)
    assert s._sweep_groups() is None
    assert s._sweep_groups() is None and not device.launches


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
def test_tuned_after_a_lost_launch(cls, device, monkeypatch):
    """A large volume that leaves the resident sweep is tuned as one that
    streams from the start, and not before."""
    tuned = []
    monkeypatch.setattr(solver_module.autotune, "MIN_VOXELS", 1)
    monkeypatch.setattr(solver_module.autotune, "tune_solver", lambda s, H, tile: tuned.append(s.iter) or (3, (8, 2, 0)))
    s = make(cls, device)
    device.lost = {4}
    run(s, 150)
    assert not tuned and s._resident
    run(s, 400)
    assert len(tuned) == 1 and s._resident is False and s._launch_config() == (3, (8, 2, 0))
    holds(s, device)


@pytest.mark.parametrize("cls", [tau.Solver, tau.PeriodicSolver])
@pytest.mark.parametrize("faster", ["resident", "streaming"])
def test_unsure_layouts_are_measured(cls, faster, device, monkeypatch):
    """Two periods resident, two streaming, then the faster of them; the next
    solver of the shape starts with that one, one of another shape does not."""
    monkeypatch.setattr(solver_module, "_resident_unsure", lambda *a: True)
    device.cost[faster] = 0.5

    def main(s, n):
        """The path of each period's launches (a periodic one ends on a
        streaming half-sweep), without those ahead of a check."""
        out = []
        for _ in range(n):
            del device.ran[:]
            run(s, s.iter + 100)
            out.append(max(device.ran, key=lambda r: r[1])[0])
        holds(s, device)
        return out

    assert main(make(cls, device), 7) == ["resident"] * 2 + ["streaming"] * 2 + [faster] * 3
    assert main(make(cls, device), 2) == [faster] * 2
    s = make(cls, device)
    s.solve(iter_limit=1000, verbose=False)
    holds(s, device)
    monkeypatch.setattr(solver_module, "_resident_faster", {})
    s = make(cls, device)
    s.solve(iter_limit=1000, verbose=False)
    holds(s, device)
    assert list(solver_module._resident_faster.values()) == [faster == "resident"]


def test_which_layouts_are_unsure():
    """On both sides of each line: ordinary volumes and images are not."""
    def unsure(kind, shape, per=None):
        B, X, Y, Z = shape
        p = _lib.Resident()
        assert _lib.load().tf_resident_plan(kind, per or B, X, Y, Z, 256, ctypes.byref(p)) == 1
        return solver_module._resident_unsure(kind, p, per or B, B, X, Y, Z, 256)

    S, F, M = _lib.KIND_SOLVER, _lib.KIND_FIELD, _lib.KIND_MULTIPHASE_FACES
    for kind, shape in [(S, (1, 32, 32, 32)), (S, (1, 203, 157, 181)), (S, (1, 256, 256, 256)), (S, (4, 96, 96, 96)),
                        (S, (1, 611, 803, 1)), (S, (1, 16, 1030, 1)), (S, (1, 4, 300, 300)), (S, (1, 2, 300, 256)),
                        (S, (1, 40, 40, 512)), (S, (1, 350, 350, 60)), (F, (1, 128, 128, 128)), (M, (1, 160, 160, 160))]:
        assert not unsure(kind, shape)
    assert not unsure(F, (4, 128, 128, 128), 2) and unsure(F, (4, 100, 100, 100), 2)
    assert unsure(M, (4, 128, 128, 128), 2)
    for shape in [(1, 15, 1030, 1), (1, 3, 300, 300), (1, 40, 40, 513), (1, 8, 8, 2000), (1, 350, 350, 56)]:
        assert unsure(S, shape)
