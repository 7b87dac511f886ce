"""Performance cases: the calls a lattice simulation makes on its way from
initial conditions to output, through the public Python interface.

A case names what it runs (`kind`), the lattice, and the options a run sets in
its configuration.  Kinds:

  evolve     Yoshida / leapfrog steps of the resident state (every run's inner
             loop), the state left on the device
  output     one output interval: Yoshida steps, energies and the output
             spectra of every field
  gw         steps with the six metric perturbations, then the GW spectrum
  ensemble   realisations of uneven lattice sizes advanced together
  laplacian  the host-array Laplacian of the Fortran drop-in (laplacian_3d)
  corrector  corrected coarse steps of the learned corrector (its forward pass)
  gradients  loss and weight gradients of the corrector (its training pass)

Fields are a homogeneous part plus white-noise fluctuations; the physics
constants are those of the repository's benchmark.  Box sides are scaled with
the lattice (dx of a 256^3 lattice with L = 10), so the time step dx / 40
resolves the chi mass at every size.  Outputs that are FP64 numbers computed
from FP32 transforms are returned in FP32, the precision that they carry.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "lattice-dev_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import lattice_amd as la  # noqa: E402

PHI0, DPHI0 = 1.0093430384226378929425913902459, -0.7137133070120812430962278466136
G2 = 2.5e5
G2_COARSE = 2e4  # a coupling whose coarse leapfrog step (8 dt) is stable: the corrector's range
DX = 10.0 / 256
AMP = 1e-4  # fluctuation amplitude of fields and momenta
U_MPL = 1.0  # reduced Planck mass of the tensor source


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest production lattice: lambda phi^4, conformal time, one
        # field; launches and latency decide
        dict(name="phi4_64_f64", kind="output", nx=64, ny=64, nz=64, prec="f64", lap="spectral", model="phi4",
             order=4, steps=5),
        # the 256^3 drop-in configuration, two fields, spectral, both forms
        dict(name="spectral_256_f64", kind="evolve", nx=256, ny=256, nz=256, prec="f64", lap="spectral",
             model="twofield", order=4, steps=2),
        dict(name="spectral_256_mixed", kind="evolve", nx=256, ny=256, nz=256, prec="mixed", lap="spectral",
             model="twofield", order=4, steps=2),
        # the same lattice with the 7-point finite-difference Laplacian
        dict(name="fd7_256_mixed", kind="evolve", nx=256, ny=256, nz=256, prec="mixed", lap="fd7",
             model="twofield", order=4, steps=4),
        # the isotropic 27-point stencil on an uneven box
        dict(name="fd27_box_f64", kind="evolve", nx=192, ny=96, nz=128, prec="f64", lap="fd27",
             model="twofield", order=2, steps=6),
        # the headline lattice, mixed form
        dict(name="spectral_1024_mixed", kind="evolve", nx=1024, ny=1024, nz=1024, prec="mixed", lap="spectral",
             model="twofield", order=4, steps=1),
        # an output interval on an uneven box: energies and all spectra
        dict(name="output_box_f64", kind="output", nx=256, ny=192, nz=128, prec="f64", lap="spectral",
             model="twofield", order=4, steps=2),
        # gravitational waves: six tensor components beside the fields
        dict(name="gw_256_mixed", kind="gw", nx=256, ny=256, nz=256, prec="mixed", lap="spectral",
             model="twofield", order=4, steps=1),
        # a coupling scan over uneven lattice sizes
        dict(name="ensemble_mixed", kind="ensemble", prec="mixed", n64=16, n96=4, n128=8, order=4, steps=3),
        # the Fortran drop-in's operator on host arrays
        dict(name="laplacian_host_128", kind="laplacian", nx=128, ny=128, nz=128),
        # the learned corrector at its training size: forward pass in a
        # corrected coarse step, and the training pass
        dict(name="corrector_step_128", kind="corrector", n=128, cf=8, steps=1),
        dict(name="corrector_grad_128", kind="gradients", n=128),
    ]


_SIZES = (8, 16, 32, 48, 64, 96, 128, 192, 256, 512)


def _box(rng, lo, hi, cubic):
    """Lattice sides between lo and hi; their product log-uniform-ish."""
    ok = [s for s in _SIZES if lo <= s <= hi]
    a = rng.choice(ok)
    if cubic:
        return a, a, a
    near = [s for s in ok if a / 2 <= s <= 2 * a]
    return a, rng.choice(near), rng.choice(near)


def draw(rng):
    kind = rng.choice(["evolve", "evolve", "evolve", "evolve", "output", "output", "gw", "ensemble", "laplacian",
                       "corrector", "gradients"])
    if kind == "evolve":
        lap = rng.choice(["spectral", "spectral", "fd7", "fd27"])
        nx, ny, nz = _box(rng, 16, 512, rng.random() < 0.5)
        case = dict(kind=kind, nx=nx, ny=ny, nz=nz, prec=rng.choice(["f64", "mixed"]), lap=lap,
                    model=rng.choice(["phi4", "twofield", "twofield"]), order=rng.choice([2, 4, 4, 6]),
                    steps=rng.randint(1, 4))
        if nx * ny * nz > 2 ** 25:  # no longer than a step of the headline lattice
            case["steps"] = 1
        return case
    if kind == "output":
        lap = rng.choice(["spectral", "spectral", "fd7"])
        nx, ny, nz = _box(rng, 16, 256, rng.random() < 0.5)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, prec=rng.choice(["f64", "mixed"]), lap=lap,
                    model=rng.choice(["phi4", "twofield"]), order=4, steps=rng.randint(1, 5))
    if kind == "gw":
        nx, ny, nz = _box(rng, 32, 256, rng.random() < 0.7)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, prec=rng.choice(["f64", "mixed"]),
                    lap=rng.choice(["spectral", "spectral", "fd7"]), model=rng.choice(["phi4", "twofield"]), order=4,
                    steps=rng.randint(1, 2))
    if kind == "ensemble":
        return dict(kind=kind, prec=rng.choice(["f64", "mixed"]), n64=rng.randint(1, 16), n96=rng.randint(0, 6),
                    n128=rng.randint(0, 8), order=rng.choice([2, 4]), steps=rng.randint(1, 4))
    if kind == "laplacian":
        nx, ny, nz = _box(rng, 16, 256, rng.random() < 0.5)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz)
    n = rng.choice([16, 32, 48, 64, 96, 128, 192])
    if kind == "corrector":
        return dict(kind=kind, n=n, cf=rng.choice([4, 8]), steps=rng.randint(1, 3))
    return dict(kind=kind, n=n)


# ---------------------------------------------------------------- inputs
def _length(case):
    return DX * case["nx"]


def _dt(case):
    # config 0 steps with dx / 20, the two-field runs with dx / 40
    return DX / 20 if case.get("model") == "phi4" else DX / 40


def _nfld(case):
    return 1 if case.get("model") == "phi4" else 2


def _background(case):
    """Homogeneous fields and momenta."""
    if case.get("model") == "phi4":
        return [1.0], [-1.0 / (3.0 * math.sqrt(1.0 / 12.0))]
    return [PHI0, 0.0], [DPHI0, 0.0]


def _noise(shape, seed):
    """White-noise fluctuations with zero mean per field, FP64, on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(AMP).to(torch.float64)
    return x - x.mean(dim=(-3, -2, -1), keepdim=True)


def _fluctuations(case, seed, member=0):
    """(fields, momenta) as (nfld, nz, ny, nx) FP64 fluctuations, rounded to
    FP32 in the mixed form."""
    shape = (_nfld(case), case["nz"], case["ny"], case["nx"])
    f, p = (_noise(shape, 4 * (1000 * int(seed) + member) + q) for q in range(2))
    if case.get("prec") == "mixed":
        f, p = f.float(), p.float()
    return f, p


class _DeviceArray:
    """A state array of a lattice as torch sees it; keeps the lattice alive."""

    def __init__(self, lat, ptr, shape, dtype):
        self.lat = lat
        self.__cuda_array_interface__ = {"shape": shape, "typestr": dtype, "data": (ptr, False), "version": 2}


def _device_state(lat, case):
    shape = (_nfld(case), case["nz"], case["ny"], case["nx"])
    dtype = "<f4" if case.get("prec") == "mixed" else "<f8"
    return [torch.as_tensor(_DeviceArray(lat, p, shape, dtype), device="cuda") for p in lat.device_state()]


def _fill(lat, case, seed, member=0):
    """Initial state of a lattice: the homogeneous part, the fluctuations
    written in place, the metric from the Friedmann constraint.  Returns the
    state arrays as tensors."""
    phi, pi = _background(case)
    mixed = case.get("prec") == "mixed"
    if mixed:  # the sampler sets the homogeneous part that the FP32 arrays are fluctuations about
        for l in range(_nfld(case)):
            lat.sample_field(l, 0, phi[l], -0.25, 1.0, 2e5, 1, 0)
            lat.sample_field(l, 1, pi[l], 0.25, 1.0, 2e5, 1, 1)
    lat.synchronize()
    state = _device_state(lat, case)
    for dst, src, mean in zip(state, _fluctuations(case, seed, member), (phi, pi)):
        for l in range(_nfld(case)):
            dst[l].copy_(src[l] if mixed else src[l] + mean[l])
    torch.cuda.synchronize()
    lat.set_scalars(1.0, 0.0)
    lat.calc_metric()
    return state


def _lattice(case):
    phi4 = case.get("model") == "phi4"
    return la.Lattice((case["nx"], case["ny"], case["nz"]), nfld=_nfld(case), length=_length(case),
                      precision=la.MIXED if case.get("prec") == "mixed" else la.F64,
                      laplacian=la.LAP_SPECTRAL if case.get("lap", "spectral") == "spectral" else la.LAP_STENCIL,
                      stencil=la.STENCIL_27PT if case.get("lap") == "fd27" else la.STENCIL_7PT,
                      time_var=la.CONFORMAL if phi4 else la.COSMIC,
                      model=la.MODEL_PHI4 if phi4 else la.MODEL_TWOFIELD,
                      model_params=(1.0,) if phi4 else (1.0, case.get("g2", G2)), gw=case["kind"] == "gw", gw_mpl=U_MPL)


def _classes(case):
    return [(n, case["n%d" % n], DX * n) for n in (64, 96, 128) if case["n%d" % n] > 0]


def _members(case):
    """(size, coupling) of every member, class-major."""
    out = []
    for n, count, _ in _classes(case):
        out += [(n, 1e4 * 10.0 ** (1.4 * m / max(1, count - 1))) for m in range(count)]
    return out


def _member_case(case, n):
    return dict(kind="evolve", nx=n, ny=n, nz=n, prec=case["prec"], lap="spectral", model="twofield",
                order=case["order"], steps=case["steps"])


def _cube(case):
    return dict(case, nx=case["n"], ny=case["n"], nz=case["n"], model="twofield", g2=G2_COARSE)


def _layers(seed):
    """Weights of a small trained-like network: (w, b) per layer."""
    rng = np.random.default_rng(seed)
    out = []
    for li, (cin, cout) in enumerate(la.Corrector.SHAPES):
        sd = math.sqrt(2.0 / (27 * cin)) * (0.1 if li == 3 else 1.0)
        out.append(((rng.standard_normal((cout, 27, cin)) * sd).astype(np.float32),
                    (rng.standard_normal(cout) * 0.05).astype(np.float32)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "laplacian":
        s["lat"] = la.Lattice((case["nx"], case["ny"], case["nz"]), nfld=1, length=_length(case),
                              model=la.MODEL_PHI4, model_params=(1.0,))
        s["f"] = _noise((case["nz"], case["ny"], case["nx"]), seed).cpu().numpy()
        return s
    if kind == "ensemble":
        members = _members(case)
        ens = la.Ensemble(_classes(case), nfld=2, precision=la.MIXED if case["prec"] == "mixed" else la.F64,
                          members=[(1.0, g2) for _, g2 in members])
        s["ens"] = ens
        s["dt"] = np.full(len(_classes(case)), DX / 40)
        s["out"] = []
        for m, (n, _) in enumerate(members):
            view = ens.member(m)
            s["out"] += _fill(view, _member_case(case, n), seed, m)
        return s
    if kind in ("corrector", "gradients"):
        case = _cube(case)
        s["lat"] = _lattice(case)
        state = _fill(s["lat"], case, seed)
        if kind == "corrector":
            s["out"] = state
        s["corr"] = la.Corrector(seed=1)
        for li, (w, b) in enumerate(_layers(5)):
            s["corr"].set_layer(li, w, b)
        s["corr"].set_norm(np.full(4, 1e-3))
        if kind == "gradients":
            rng = np.random.default_rng(seed)
            n = case["n"]
            s["target"] = rng.standard_normal((n, n, n, 4), dtype=np.float32)
        return s
    s["lat"] = _lattice(case)
    s["out"] = _fill(s["lat"], case, seed)
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "laplacian":
        return s["lat"].laplacian_3d(s["f"])
    if kind == "ensemble":
        s["ens"].symp(case["order"], s["dt"], case["steps"])
        return s["out"]
    if kind == "corrector":
        st = s["corr"].step(s["lat"], DX / 40, case["cf"], nsteps=case["steps"], threshold=1e-2)
        return s["out"] + [st["fallbacks"]]
    if kind == "gradients":
        loss, grads = s["corr"].gradients(s["lat"], s["target"])
        return [np.float32(loss)] + [x for layer in grads for x in layer]
    lat = s["lat"]
    lat.symp(case["order"], _dt(case), case["steps"])
    if kind == "evolve":
        return s["out"]
    if kind == "gw":
        spectrum = lat.gw_spectrum()
        return s["out"] + [spectrum.astype(np.float32) if case["prec"] == "mixed" else spectrum]
    e = lat.energies()
    spectra = [lat.output_spectra(l) for l in range(_nfld(case))]
    if case["prec"] == "mixed":
        spectra = [x.astype(np.float32) for x in spectra]
    # the Friedmann residual is a difference of nearly equal numbers: its
    # terms are returned instead
    return s["out"] + [np.array([e[k] for k in ("a", "hubble", "rho", "ke", "pe", "ge", "grav", "mean1")])] + spectra


# ---------------------------------------------------------------- the least work
_STAGES = {2: 1, 4: 3, 6: 7, 8: 15}


def _fft_flops(sites):
    return 2.5 * sites * math.log2(sites)


def work(case):
    """Bytes that a pass cannot do without (the state read and written once
    per call; a force evaluation that does not fit the caches needs one read
    and one write of the state more) and its floating-point operations."""
    kind = case["kind"]
    if kind == "laplacian":
        nv = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": 16.0 * nv, "flops": 2 * _fft_flops(nv) + 6 * nv}
    if kind == "ensemble":
        w = [work(_member_case(case, n)) for n, _ in _members(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if kind in ("corrector", "gradients"):
        nv = float(case["n"]) ** 3
        macs = nv * 27 * (8 * 32 + 2 * 32 * 32 + 32 * 4)
        if kind == "corrector":
            step = work(dict(_cube(case), kind="evolve", prec="f64", lap="spectral", order=2, steps=1))
            return {"bytes": case["steps"] * step["bytes"], "flops": case["steps"] * (step["flops"] + 2 * macs)}
        # forward, weight gradients and the data gradients of layers 2-4; the
        # state and target in
        return {"bytes": nv * (32 + 16),
                "flops": 2 * (2 * macs + nv * 27 * (2 * 32 * 32 + 32 * 4))}
    nv = float(case["nx"]) * case["ny"] * case["nz"]
    nf = _nfld(case)
    w = 4.0 if case["prec"] == "mixed" else 8.0
    kicks = _STAGES[case["order"]] * case["steps"]
    arrays = nf + (6 if kind == "gw" else 0)
    # per kick: fields and momenta read and written once
    nbytes = kicks * arrays * 4 * w * nv
    spectral = case.get("lap", "spectral") == "spectral"
    per = 2 * _fft_flops(nv) if spectral else (14.0 if case["lap"] == "fd7" else 54.0) * nv
    flops = kicks * (arrays * (per + 10 * nv) + 20 * nv)
    if kind == "output":
        nbytes += 2 * nf * w * nv
        flops += 2 * nf * (_fft_flops(nv) + 10 * nv)
    if kind == "gw":
        nbytes += 12 * w * nv
        flops += 12 * (_fft_flops(nv) + 50 * nv)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------- the same in 64 bits
def _wave(n):
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    return torch.where(k <= n // 2, k, n - k)


def _k2(case):
    dk = 2.0 * math.pi / _length(case)
    kx = torch.arange(case["nx"] // 2 + 1, device="cuda", dtype=torch.float64)
    ky, kz = _wave(case["ny"]), _wave(case["nz"])
    return (kx * kx)[None, None, :], (ky * ky)[None, :, None], (kz * kz)[:, None, None], dk * dk


def _laplacian(case, f):
    lap = case.get("lap", "spectral")
    if lap == "spectral":
        F = torch.fft.rfftn(f)
        kx, ky, kz, dk2 = _k2(case)
        for k in range(case["nz"]):  # plane by plane: no k^2 array of the lattice's size
            F[k] *= -dk2 * (kx[0] + ky[0] + kz[k])
        return torch.fft.irfftn(F, s=f.shape)
    c0, c1, c2, c3, cc = (-128.0, 14.0, 3.0, 1.0, 30.0) if lap == "fd27" else (-6.0, 1.0, 0.0, 0.0, 1.0)
    out = c0 * f
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                rank = abs(dx) + abs(dy) + abs(dz)
                c = (0.0, c1, c2, c3)[rank]
                if c:
                    out = out + c * torch.roll(f, (dz, dy, dx), (0, 1, 2))
    return out / (cc * DX * DX)


class _Exact:
    """H = H_fields + H_gravity by symplectic splitting, FP64: phi' = pi / y^2
    and so on; y = a (conformal) or a^(3/2) (cosmic)."""

    def __init__(self, case, seed, g2=G2, member=0):
        self.case, self.g2 = case, g2
        self.phi4 = case.get("model") == "phi4"
        f, p = _fluctuations(case, seed, member)
        phi, pi = _background(case)
        self.f = [f[l].double() + phi[l] for l in range(len(phi))]
        self.p = [p[l].double() + pi[l] for l in range(len(pi))]
        self.u = self.pu = None
        if case["kind"] == "gw":
            self.u = [torch.zeros_like(self.f[0]) for _ in range(6)]
            self.pu = [torch.zeros_like(self.f[0]) for _ in range(6)]
        self.y = 1.0
        e = self.energies()
        self.q = -math.sqrt(12.0 * e["rho"]) if self.phi4 else -math.sqrt(16.0 / 3.0 * e["rho"])

    def v(self):
        if self.phi4:
            return float((0.25 * self.f[0] ** 4).mean())
        return float((0.5 * self.f[0] ** 2).mean() + (0.5 * self.g2 * (self.f[0] * self.f[1]) ** 2).mean())

    def energies(self):
        y = self.y
        a = y if self.phi4 else y ** (2.0 / 3.0)
        ke = 0.5 * sum(float((p * p).mean()) for p in self.p) / (y ** 6 if self.phi4 else y ** 4)
        ge = 0.5 * sum(-float((f * _laplacian(self.case, f)).mean()) for f in self.f) / (a * a)
        pe = self.v()
        e = dict(a=a, ke=ke, pe=pe, ge=ge, rho=ke + pe + ge, mean1=float(self.f[0].mean()))
        if hasattr(self, "q"):
            e["hubble"] = -self.q / 6.0 / y ** 2 if self.phi4 else -self.q / y / 4.0
            e["grav"] = -3.0 * e["hubble"] ** 2
        return e

    def drift(self, h):
        c = h / self.y ** 2
        self.q += h * sum(float((p * p).mean()) for p in self.p) / self.y ** 3
        for f, p in zip(self.f, self.p):
            f.add_(p, alpha=c)
        for u, p in zip(self.u or [], self.pu or []):
            u.add_(p, alpha=c)

    def grav(self, h):
        self.y -= h * self.q / 6.0 if self.phi4 else h * self.q * 3.0 / 8.0

    def kick(self, h):
        y = self.y
        a2 = y * y if self.phi4 else y ** (4.0 / 3.0)
        hA = h * y * y if self.phi4 else h * y * y / a2
        hB = h * y ** 4 if self.phi4 else h * y * y
        if self.phi4:
            dv = [self.f[0] ** 3]
        else:
            f0, f1 = self.f
            dv = [f0 + self.g2 * f0 * f1 * f1, self.g2 * f0 * f0 * f1]
        ge = 0.0
        for l, f in enumerate(self.f):
            lap = _laplacian(self.case, f)
            ge -= float((f * lap).mean())
            self.p[l] += hA * lap - hB * dv[l]
            del lap
        if self.u:
            g = [[(torch.roll(f, -1, ax) - torch.roll(f, 1, ax)) / (2 * DX) for ax in (2, 1, 0)] for f in self.f]
            pairs = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
            for c, (i, j) in enumerate(pairs):
                src = sum(d[i] * d[j] for d in g)
                self.pu[c] += hA * (_laplacian(self.case, self.u[c]) + 2.0 / U_MPL ** 2 * src)
        if self.phi4:
            self.q -= y ** 3 * (ge / a2 + 4.0 * self.v()) * h
        else:
            self.q -= y * (ge / a2 / 3.0 + 2.0 * self.v()) * h

    def part(self, h, index):
        if index == 3:
            self.kick(h)
        elif (index == 1) == self.phi4:
            self.drift(h)
        else:
            self.grav(h)

    def symp(self, order, dt, steps):
        if order == 2:
            w = [1.0]
        elif order == 4:
            w1 = 1.0 / (2.0 - 2.0 ** (1.0 / 3.0))
            w = [w1, 1.0 - 2.0 * w1, w1]
        else:
            w1, w2, w3 = -1.17767998417887, 0.235573213359357, 0.784513610477560
            w = [w3, w2, w1, 1.0 - 2.0 * (w1 + w2 + w3), w1, w2, w3]
        w = w * steps
        self.part(w[0] * dt / 2, 1)
        for a, b in zip(w, w[1:] + [0.0]):
            self.part(a * dt / 2, 2)
            self.part(a * dt, 3)
            self.part(a * dt / 2, 2)
            self.part((a + b) * dt / 2, 1)

    def state(self):
        f, p = torch.stack(self.f), torch.stack(self.p)
        if self.case.get("prec") == "mixed":  # the FP32 arrays are fluctuations
            f -= f.mean(dim=(1, 2, 3), keepdim=True)
            p -= p.mean(dim=(1, 2, 3), keepdim=True)
        return [f, p]

    def _bins(self, value):
        """Shell averages of a function of the plane index over a half-complex
        array, with the two-bin weights (1 - d^2)^2."""
        c = self.case
        ns = _num_bins(c)
        kx, ky, kz, _ = _k2(c)
        mult = torch.full((c["nx"] // 2 + 1,), 2.0, device="cuda", dtype=torch.float64)
        mult[0] = mult[-1] = 1.0
        S, W = None, torch.zeros(ns + 2, device="cuda", dtype=torch.float64)
        for k in range(c["nz"]):
            r = torch.sqrt(kx[0] + ky[0] + kz[k])
            b = torch.floor(r)
            vals = value(k)
            if S is None:
                S = torch.zeros(len(vals), ns + 2, device="cuda", dtype=torch.float64)
            for add in (0, 1):
                w = (1.0 - (b + add - r) ** 2) ** 2 * mult[None, :]
                idx = (b.long() + add).clamp_(max=ns + 1).reshape(-1)
                W.index_add_(0, idx, w.reshape(-1))
                for ch, x in enumerate(vals):
                    S[ch].index_add_(0, idx, (w * x).reshape(-1))
        return torch.where(W[None, :ns] != 0, S[:, :ns] / W[None, :ns], S[:, :ns])

    def spectra(self, l):
        A, B = torch.fft.rfftn(self.f[l]), torch.fft.rfftn(self.p[l])

        def value(k):
            a, b = A[k], B[k]
            x = b * a.conj()
            return [a.real ** 2 + a.imag ** 2, b.real ** 2 + b.imag ** 2, x.real, x.imag]

        return self._bins(value)

    def gw_spectrum(self):
        c = self.case
        out = []
        for arr in (self.pu, self.u):
            F = [torch.fft.rfftn(x) for x in arr]

            def value(k):
                kx = torch.arange(c["nx"] // 2 + 1, device="cuda", dtype=torch.float64)[None, :]
                signed = lambda n: torch.where(torch.arange(n, device="cuda") <= n // 2,  # noqa: E731
                                               torch.arange(n, device="cuda"), torch.arange(n, device="cuda") - n)
                ky = signed(c["ny"]).double()[:, None]
                kz = float(k if k <= c["nz"] // 2 else k - c["nz"])
                shape = (c["ny"], c["nx"] // 2 + 1)
                kv = torch.stack([kx.expand(shape), ky.expand(shape), torch.full(shape, kz, device="cuda", dtype=torch.float64)], -1)
                k2 = (kv * kv).sum(-1)
                eye = torch.eye(3, device="cuda", dtype=torch.float64)
                P = (eye - kv[..., :, None] * kv[..., None, :] / torch.where(k2 > 0, k2, 1.0)[..., None, None])
                U = torch.stack([F[q][k] for q in (0, 1, 2, 1, 3, 4, 2, 4, 5)], -1).reshape(shape + (3, 3))

                def mul(x, y):  # 3 x 3 products, entry by entry
                    return (x[..., :, :, None] * y[..., None, :, :]).sum(-2)

                M = mul(P.to(U.dtype), U)
                T = mul(M, P.to(U.dtype)) - 0.5 * P * M.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
                n2 = (T.real ** 2 + T.imag ** 2).sum((-2, -1))
                return [torch.where(k2 > 0, n2, 0.0)]

            out.append(self._bins(value)[0])
        return torch.stack(out)


def _num_bins(c):
    """Number of shells: floor(sqrt(1 + sum of the squared half sides))."""
    return int(math.floor(math.sqrt(1.0 + sum((c[k] // 2 + 1) ** 2 for k in ("nx", "ny", "nz")))))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("corrector", "gradients"):
        return None  # a BF16 network: its 64-bit value says nothing about the kernels
    if kind == "laplacian":
        f = _noise((case["nz"], case["ny"], case["nx"]), seed)
        return _laplacian(dict(case, lap="spectral"), f)
    if kind == "ensemble":
        out = []
        for m, (n, g2) in enumerate(_members(case)):
            x = _Exact(_member_case(case, n), seed, g2, m)
            x.symp(case["order"], DX / 40, case["steps"])
            out += x.state()
        return out
    x = _Exact(case, seed)
    x.symp(case["order"], _dt(case), case["steps"])
    out = x.state()
    if kind == "evolve":
        return out
    if kind == "gw":
        return out + [x.gw_spectrum()]
    e = x.energies()
    return (out + [np.array([e[k] for k in ("a", "hubble", "rho", "ke", "pe", "ge", "grav", "mean1")])]
            + [x.spectra(l) for l in range(_nfld(case))])
