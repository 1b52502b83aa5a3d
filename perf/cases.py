"""Timed cases of the framework: the solves its users run, from the smallest to the largest.

A case is a dict of plain values.  ``prepare(case, seed)`` makes the inputs
(images or diffusivity maps from the seed) and, for the cases that keep one,
the solver object; ``run(state)`` is one pass through the public entry points;
``exact(case, seed)`` gives the same outputs in 64 bits from plain torch and
numpy.

Case fields:
  path      which entry point (see listed())
  batch     volumes per call (of one shape; for "uneven" the count of volumes)
  x, y, z   voxels per volume; z = 0: a 2-D image of x by y pixels (for
            "uneven": x, y = the smallest and largest cube edge)
  porosity  conductive fraction
  sigma     Gaussian smoothing of the noise in voxels, 0: independent voxels
  whole     True: a pass builds the solver from the host image and solves, as
            a script that meets each image once does; False: the solver is
            kept and a pass is reset() and solve(), as in a program that
            solves a resident volume again
"""
from __future__ import annotations

import math

import numpy as np
import torch

import taufactor_amd as tau

SPACING = (1.0, 1.0, 2.0)  # slices twice as far apart as pixels
THREE_PHASE = {0: 0.0, 1: 1.0, 2: 0.1}
SEVEN_PHASE = {0: 0.0, 1: 1.0, 2: 0.5, 3: 0.25, 4: 0.12, 5: 2.0, 6: 0.05}


def listed():
    def c(name, path, x, y, z, porosity=0.5, sigma=3.0, batch=1, whole=False):
        return dict(name=name, path=path, batch=batch, x=x, y=y, z=z, porosity=porosity, sigma=sigma, whole=whole)

    return [
        # a small subvolume, image to tau: what a scan over many representative
        # volumes or a first try calls; all latency
        c("whole_32", "solver", 32, 32, 32, 0.5, 2.0, whole=True),
        # the 100^3 volume of independent voxels of the benchmark, solver kept
        c("plain_100", "solver", 100, 100, 100, 0.5, 0.0),
        # one 2-D micrograph
        c("image_2d", "solver", 611, 803, 0, 0.7, 4.0),
        # an ordinary tomogram crop of ragged size, image to tau
        c("whole_ragged", "solver", 203, 157, 181, 0.4, 3.0, whole=True),
        # the headline volume of the benchmark: 512^3 at porosity 0.35
        c("solver_512", "solver", 512, 512, 512, 0.35, 4.0),
        # a periodic structure of the size of the documentation's volumes
        c("periodic_256", "periodic", 256, 256, 256, 0.45, 4.0),
        # a stack of slices with another spacing along z
        c("anisotropic", "anisotropic", 160, 241, 97, 0.5, 3.0),
        # transport with reaction in a three-phase electrode
        c("electrode", "electrode", 128, 128, 128, 0.45, 3.0),
        # three labels, two of them conducting, and the per-phase gradient
        c("multiphase_320", "three_phase", 320, 320, 320, 0.6, 3.0),
        # seven labels with seven diffusivities
        c("multiphase_7", "seven_phase", 121, 130, 143, 0.8, 3.0),
        # many volumes of different sizes in one call
        c("uneven_48", "uneven", 32, 112, 0, 0.5, 3.0, batch=48),
        # one step of an optimisation of a diffusivity map: forward and backward
        c("field_step", "field", 128, 128, 128, 1.0, 3.0, batch=4, whole=True),
    ]


# smallest and largest edge a path is drawn with
RANGES = {"solver": (24, 400), "image": (96, 1600), "periodic": (32, 256), "anisotropic": (32, 224),
          "electrode": (32, 160), "three_phase": (32, 320), "seven_phase": (32, 160), "uneven": (16, 128),
          "field": (24, 128)}


def draw(rng):
    kind = rng.choice(sorted(RANGES))
    lo, hi = RANGES[kind]

    def edge():
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    n = edge()
    x, y, z = (min(hi, max(lo, int(round(n * rng.uniform(0.7, 1.4))))) for _ in range(3))
    batch, path, whole = 1, kind, False
    porosity = round(rng.uniform(0.4, 0.6), 3)
    sigma = round(rng.uniform(1.0, 4.0), 2)
    if kind == "solver":
        whole = rng.random() < 0.5
        if rng.random() < 0.25:
            sigma = 0.0
        if n <= 96:
            batch = rng.choice([1, 1, 2, 4])  # equal volumes in one call
    elif kind == "image":
        path, z, porosity = "solver", 0, round(rng.uniform(0.65, 0.8), 3)
    elif kind == "periodic":
        y, z = y // 2 * 2, z // 2 * 2
    elif kind == "three_phase":
        porosity = round(rng.uniform(0.5, 0.7), 3)
    elif kind == "seven_phase":
        porosity = round(rng.uniform(0.6, 0.9), 3)
    elif kind == "uneven":
        x, y, z = max(lo, n // 3), max(n, lo + 8), 0
        batch = rng.randint(6, 48)
    elif kind == "field":
        batch, porosity, whole = rng.randint(1, 4), 1.0, True
    return dict(path=path, batch=batch, x=x, y=y, z=z, porosity=porosity, sigma=sigma, whole=whole)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _noise(shape, sigma, gen):
    """Standardised Gaussian-smoothed noise (periodic), float32 on the GPU."""
    t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    if sigma > 0:
        r = int(math.ceil(3 * sigma))
        for dim in range(len(shape)):
            if shape[dim] == 1:
                continue
            acc = torch.zeros_like(t)
            for k in range(-r, r + 1):
                acc += math.exp(-0.5 * (k / sigma) ** 2) * torch.roll(t, k, dim)
            t = acc
    return (t - t.mean()) / t.std()


def _cut(p):
    """The value a standard normal variable stays below with probability p."""
    return math.sqrt(2) * torch.erfinv(torch.tensor(2 * p - 1, dtype=torch.float64)).item()


def _shape(case):
    return (case["x"], case["y"], case["z"]) if case["z"] else (case["x"], case["y"])


def _uneven_shapes(case):
    """The edges of the batch: fixed by the case, the voxels by the seed."""
    rng = np.random.default_rng([case["batch"], case["x"], case["y"]])
    return [int(e) for e in rng.integers(case["x"], case["y"] + 1, size=case["batch"])]


def _images(case, seed):
    """The host image (or list of images, or the device map) of a case."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    path, p, sigma = case["path"], case["porosity"], case["sigma"]

    def labels(shape):
        z = _noise(shape, sigma, gen)
        if path in ("solver", "periodic", "anisotropic", "uneven"):
            return (z < _cut(p)).to(torch.uint8)
        if path == "electrode":
            # 1 pores, 0 reacting solid, 2 an inert tenth
            img = (z < _cut(p)).to(torch.uint8)
            img[z > _cut(0.9)] = 2
            return img
        # multiphase: label 0 isolating above the cut, the rest split evenly
        # by a second field
        n = len(THREE_PHASE if path == "three_phase" else SEVEN_PHASE) - 1
        split = _noise(shape, sigma, gen)
        img = torch.ones(shape, dtype=torch.uint8, device="cuda")
        for k in range(1, n):
            img += (split > _cut(k / n)).to(torch.uint8)
        img[z >= _cut(p)] = 0
        return img

    if path == "field":
        z = torch.stack([_noise(_shape(case), sigma, gen) for _ in range(case["batch"])])
        return torch.sigmoid(4.0 * z)
    if path == "uneven":
        return [labels((e, e, e)).cpu().numpy() for e in _uneven_shapes(case)]
    vols = [labels(_shape(case)) for _ in range(case["batch"])]
    return (torch.stack(vols) if case["batch"] > 1 else vols[0]).cpu().numpy()


def _solver(case, img):
    path = case["path"]
    if path == "solver":
        return tau.Solver(img)
    if path == "periodic":
        return tau.PeriodicSolver(img)
    if path == "anisotropic":
        return tau.AnisotropicSolver(img, SPACING)
    if path == "electrode":
        return tau.ElectrodeSolver(img)
    return tau.MultiPhaseSolver(img, dict(THREE_PHASE if path == "three_phase" else SEVEN_PHASE))


def prepare(case, seed):
    img = _images(case, seed)
    state = {"case": case}
    if case["path"] == "field":
        state["k"] = img.requires_grad_(True)
    elif case["path"] == "uneven":
        state["solver"] = tau.BatchSolver(img)
    elif case["whole"]:
        state["img"] = img
    else:
        state["solver"] = _solver(case, img)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    path = case["path"]
    if path == "field":
        k = state["k"]
        k.grad = None
        d = tau.effective_diffusivity(k)
        d.sum().backward()
        return {"D_eff": d.detach(), "grad": k.grad}
    s = _solver(case, state["img"]) if case["whole"] else state["solver"]
    if path == "uneven":
        s.solve()
        return {"tau": s.tau, "D_eff": s.D_eff, "iter": s.iters, "field": [s.field(v) for v in range(s.n_volumes)]}
    if not case["whole"]:
        s.reset()
    s.solve(verbose=False)
    out = {"tau": s.tau, "iter": s.iter, "field": s.field}
    if path == "electrode":
        out["c_x"] = s.c_x
    else:
        out["D_eff"] = s.D_eff
    if path in ("three_phase", "seven_phase"):
        out["grad"] = s.grad_D_eff()
    return out


def _iterations(case):
    """Iterations of a typical solve at these sizes (they grow with the edge
    along the flux)."""
    n = case["y"] if case["path"] == "uneven" else case["x"]
    return max(300, 3.5 * n)


def work(case):
    """Image in (1 byte a voxel; 4 for a diffusivity map), field out (4 bytes
    a voxel) and the arithmetic of the iteration: a voxel is updated every
    second iteration, with 5 additions, a division and 3 more operations (10
    products and 10 sums where the faces have conductances)."""
    if case["path"] == "uneven":
        lo, hi = case["x"], case["y"]
        vox = case["batch"] * sum(e ** 3 for e in range(lo, hi + 1)) / (hi - lo + 1)
    else:
        vox = case["batch"] * case["x"] * case["y"] * max(case["z"], 1)
    ops = 20 if case["path"] in ("field", "three_phase", "seven_phase") else 9
    return {"bytes": vox * (8 if case["path"] == "field" else 5), "flops": vox * _iterations(case) / 2 * ops}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
EXACT_MOST = 60_000_000  # voxels: more would take too long in plain torch
_IN = (slice(None), slice(1, -1), slice(1, -1), slice(1, -1))


def _pad64(t, first=0.0, last=0.0):
    p = torch.nn.functional.pad(t, (1, 1, 1, 1, 1, 1))
    p[:, 0, 1:-1, 1:-1], p[:, -1, 1:-1, 1:-1] = first, last
    return p


def _wrap(p):
    p[:, :, 0, :] = p[:, :, -2, :]
    p[:, :, -1, :] = p[:, :, 1, :]
    p[:, :, :, 0] = p[:, :, :, -2]
    p[:, :, :, -1] = p[:, :, :, 1]


def _neighbours(p):
    return (p[:, 2:, 1:-1, 1:-1], p[:, :-2, 1:-1, 1:-1], p[:, 1:-1, 2:, 1:-1], p[:, 1:-1, :-2, 1:-1],
            p[:, 1:-1, 1:-1, 2:], p[:, 1:-1, 1:-1, :-2])


def _hm(a, b):
    return torch.where(a + b > 0, 2 * a * b / (a + b).clamp_min(1e-300), torch.zeros_like(a))


def _impedance(R, C, w):
    z = np.full_like(w, 1e50, dtype=complex)
    for i in range(R.shape[1] - 1, -1, -1):
        z = R[:, i:i + 1] + 1 / (1j * w * C[:, i:i + 1] + 1 / z)
    return z[:, 0].real


class _Exact:
    """The red-black iteration of one [B, X, Y, Z] volume in float64 torch."""

    def __init__(self, path, img):
        self.path = path
        img = img if img.dim() == 4 else img.view((1,) + tuple(img.shape) + (1,) * (3 - img.dim()))
        self.B, X, self.Y, self.Z = img.shape
        self.X = X
        if path == "field":
            d = img.double()
        elif path in ("three_phase", "seven_phase"):
            table = THREE_PHASE if path == "three_phase" else SEVEN_PHASE
            d = torch.tensor([table[i] for i in range(len(table))], dtype=torch.float32).double().cuda()[img.long()]
        else:
            d = (img == 1).double()
        self.d, mask = d, (d > 0).double()
        x = torch.arange(X, device="cuda", dtype=torch.float64).view(1, X, 1, 1)
        if path == "electrode":
            self.c = _pad64(mask * torch.cosh(1 - (x + 0.5) / X) / math.cosh(1), 2.0, 0.0)
            near = sum(_neighbours(_pad64(mask, 2.0, 0.0)))
            reac = sum(_neighbours(_pad64((img == 0).double()))) * mask
            self.a_x = reac.mean((2, 3))
            self.k_0 = mask.mean((1, 2, 3)) / self.a_x.mean(1) / X ** 2
            f = (near + self.k_0.view(-1, 1, 1, 1) * reac) * mask
        else:
            self.c = _pad64(mask * ((x + 0.5) / X - 0.5), -1.0, 1.0)
            if path in ("field", "three_phase", "seven_phase"):
                p = _pad64(d)
                p[:, 0], p[:, -1] = p[:, 1], p[:, -2]
                self.g = [_hm(d, n) for n in _neighbours(p)]
                f = sum(self.g)
                f[:, 0] += self.g[1][:, 0]
                f[:, -1] += self.g[0][:, -1]
            else:
                p = _pad64(mask, 2.0, 2.0)
                if path == "periodic":
                    _wrap(p)
                xq, xm, yq, ym, zq, zm = _neighbours(p)
                ky = (SPACING[0] / SPACING[1]) ** 2 if path == "anisotropic" else 1.0
                kz = (SPACING[0] / SPACING[2]) ** 2 if path == "anisotropic" else 1.0
                self.k = (ky, kz)
                f = (xq + xm + ky * (yq + ym) + kz * (zq + zm)) * mask
        self.f = torch.where(f == 0, torch.full_like(f, math.inf), f)
        par = (torch.arange(X, device="cuda").view(-1, 1, 1) + torch.arange(self.Y, device="cuda").view(1, -1, 1)
               + torch.arange(self.Z, device="cuda").view(1, 1, -1)) % 2
        w = 2 - math.pi / (1.5 * X)
        self.w = [w * (par == 0).double(), w * (par == 1).double()]
        self.vol_x = mask.mean((2, 3))
        self.D_mean = d.mean((1, 2, 3))

    def step(self, it):
        c = self.c
        if self.path == "periodic":
            _wrap(c)
        n = _neighbours(c)
        if self.path in ("field", "three_phase", "seven_phase"):
            s = n[0] * self.g[0]
            for a, b in zip(n[1:], self.g[1:]):
                s.addcmul_(a, b)
        elif self.path == "anisotropic":
            s = n[0] + n[1] + self.k[0] * (n[2] + n[3]) + self.k[1] * (n[4] + n[5])
        else:
            s = n[0] + n[1]
            for a in n[2:]:
                s += a
        s /= self.f
        s -= c[_IN]
        c[_IN].addcmul_(s, self.w[it & 1])

    def metrics(self, last):
        """(tau, relative error) per volume; last: c_x of the check before."""
        c = self.c[_IN]
        vol = self.vol_x
        c_x = torch.where(vol > 0, c.mean((2, 3)) / vol.clamp_min(1e-300), torch.zeros_like(vol))
        self.c_x = c_x
        if self.path == "electrode":
            prev = self.c[:, :-2, 1:-1, 1:-1]
            fl = prev - c
            fl[:, 0] = 2 * (1 - c[:, 0])
            fl = torch.where((c == 0) | (prev == 0), torch.zeros_like(fl), fl).mean((2, 3))
            one = torch.cat([2 * (1 - c_x[:, :1]), c_x[:, :-1] - c_x[:, 1:]], 1)
            eps = torch.cat([vol[:, :1], (vol[:, :-1] + vol[:, 1:]) / 2], 1)
            fl, one, eps, a = (t.cpu().numpy() for t in (fl, one, eps, self.a_x))
            w = eps.mean(1, keepdims=True) / a.mean(1, keepdims=True) / self.X ** 2 / 8
            mean_a = np.repeat(a.mean(1, keepdims=True), self.X, 1)
            mean_r = np.repeat(1 / eps.mean(1, keepdims=True), self.X, 1)
            t = _impedance(one / fl, a, w) / _impedance(mean_r, mean_a, w)
            return t, (c_x - last).abs().amax(1).cpu().numpy()
        d = self.c[:, 2:-1, 1:-1, 1:-1] - self.c[:, 1:-2, 1:-1, 1:-1]
        if self.path in ("field", "three_phase", "seven_phase"):
            d = d * self.g[0][:, :-1]
        else:
            d = torch.where((self.f[:, :-1] > 8) | (self.f[:, 1:] > 8), torch.zeros_like(d), d)
        fl = d.mean((2, 3))
        D = fl.mean(1) * self.X
        self.D = D.cpu().numpy()
        hi, lo = fl.amax(1), fl.amin(1)
        return (self.D_mean / D).cpu().numpy(), ((hi - lo) / hi).cpu().numpy()

    def solve(self, crit=1e-2):
        old, last, it = 0.0, torch.zeros((), device="cuda", dtype=torch.float64), 0
        while it < 10000:
            self.step(it)
            it += 1
            if it % 100 == 0:
                t, err = self.metrics(last)
                last, before, old = self.c_x, old, t
                if np.all(err < crit) and np.max(np.abs(t - before)) < 2e-3:
                    break
        self.tau = t
        return self

    def dissipation_gradient(self):
        """dD/dk of every voxel: the change of the dissipation at the fixed
        point; where k is 0, the one-sided change, with the voxel at the mean
        of its conducting neighbours and electrodes."""
        p, dp = self.c.clone(), _pad64(self.d)
        n, dn = _neighbours(p), _neighbours(dp)
        c, d = p[_IN], self.d
        g, count, total, square = (torch.zeros_like(c) for _ in range(4))
        for a, b in zip(n, dn):
            on = (b > 0).double()
            g += torch.where(d > 0, on * (a - c) ** 2 * 2 * b ** 2 / (d + b).clamp_min(1e-300) ** 2, torch.zeros_like(c))
            count += on
            total += on * a
            square += on * a ** 2
        for at, bc in ((0, -0.5), (-1, 0.5)):
            g[:, at] += 2 * (c[:, at] - bc) ** 2
            count[:, at] += 1
            total[:, at] += bc
            square[:, at] += bc ** 2
        mean = total / count.clamp_min(1)
        g = torch.where(d > 0, g, 2 * (square - count * mean ** 2))
        return g * (self.X / (self.Y * self.Z))


def exact(case, seed):
    path = case["path"]
    if path == "uneven":
        got = [_Exact("solver", torch.from_numpy(i).cuda()).solve() for i in _images(case, seed)]
        return {"tau": np.concatenate([e.tau for e in got]), "D_eff": np.concatenate([e.D for e in got]),
                "iter": None, "field": [e.c[0] for e in got]}
    if case["batch"] * case["x"] * case["y"] * max(case["z"], 1) > EXACT_MOST:
        return None
    img = _images(case, seed)
    e = _Exact(path, img if path == "field" else torch.from_numpy(img).cuda())
    e.solve(1e-3 if path == "field" else 1e-2)
    if path == "field":
        return {"D_eff": e.D, "grad": e.dissipation_gradient()}
    out = {"tau": e.tau, "iter": None, "field": e.c}
    if path == "electrode":
        out["c_x"] = e.c_x.cpu().numpy()
    else:
        out["D_eff"] = e.D
    if path in ("three_phase", "seven_phase"):
        g = e.dissipation_gradient()
        lab = torch.from_numpy(img).cuda()[None]
        out["grad"] = {k: np.array([(g * (lab == k)).sum().item()])
                       for k in range(len(THREE_PHASE if path == "three_phase" else SEVEN_PHASE))}
    return out
