"""GPU parity of the evolution path (splits, Yoshida compositions, calc_metric,
energies) against the CPU oracle on identical seeded initial conditions."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

PHI0_C, DPHI0_C = 1.0093430384226378929425913902459, -0.7137133070120812430962278466136


def two_field_ic(n, L, seed, mpl=2e5):
    """Seeded vacuum-like fluctuations (oracle sampler, Philox streams) on top of
    the homogeneous two-field background of hamiltonian_cosmic.f90:18-22."""
    m2eff = 1.0
    fld = np.empty((2, n, n, n))
    fldp = np.empty_like(fld)
    fld[0] = PHI0_C + O.sample(n, L, -0.25, m2eff, mpl, seed, 0)
    fldp[0] = DPHI0_C + O.sample(n, L, 0.25, m2eff, mpl, seed, 1)
    fld[1] = O.sample(n, L, -0.25, m2eff, mpl, seed, 2)
    fldp[1] = O.sample(n, L, 0.25, m2eff, mpl, seed, 3)
    return fld, fldp


def one_field_ic(n, L, seed, phi0=1.0, mpl=1e7 / 3.0):
    m2eff = 3.0 * phi0**2
    dphi0 = -phi0**3 / (3.0 * np.sqrt(phi0**4 / 12.0))
    fld = (phi0 + O.sample(n, L, -0.25, m2eff, mpl, seed, 0))[None]
    fldp = (dphi0 + O.sample(n, L, 0.25, m2eff, mpl, seed, 1))[None]
    return fld, fldp


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def run_pair(gpu, n, L, nfld, time_var, model, mp, lap, stencil, fld, fldp, plan):
    with gpu.Lattice(n, nfld=nfld, length=L, time_var=time_var, model=model, model_params=mp,
                     laplacian=lap, stencil=stencil) as lat:
        sim = O.Simulation(n, nfld, L, time_var, lap_kind=lap, stencil=stencil, model=model, mp=mp)
        lat.set_state(fld, fldp, 1.0, 0.0)
        sim.set_state(fld, fldp, 1.0, 0.0)
        lat.calc_metric()
        sim.calc_metric()
        y0, p0 = lat.scalars
        assert abs(p0 - sim.ysclp) <= 1e-13 * abs(sim.ysclp)
        for kind, args in plan:
            getattr(lat, kind)(*args)
            if kind == "symp":
                sim.symp(*args)
            elif kind == "Hamiltonian_Split":
                sim.split(*args)
            elif kind == "symp_o2step":
                sim.symp_o2step(*args)
        gf, gp, gy, gpy = lat.get_state()
        ge = lat.energies()
        oe = sim.energies()
        return (gf, gp, gy, gpy, ge), (sim.fld.copy(), sim.fldp.copy(), sim.yscl, sim.ysclp, oe)


CASES = {
    "conformal_phi4_spectral": dict(nfld=1, time_var=O.CONFORMAL, model=O.MODEL_PHI4, mp=(1.0,),
                                    lap=O.LAP_SPECTRAL, stencil=(-6, 1, 0, 0, 1)),
    "cosmic_twofield_spectral": dict(nfld=2, time_var=O.COSMIC, model=O.MODEL_TWOFIELD, mp=(1.0, 2.5e5),
                                     lap=O.LAP_SPECTRAL, stencil=(-6, 1, 0, 0, 1)),
    "cosmic_twofield_fd7": dict(nfld=2, time_var=O.COSMIC, model=O.MODEL_TWOFIELD, mp=(1.0, 2.5e5),
                                lap=O.LAP_STENCIL, stencil=(-6.0, 1.0, 0.0, 0.0, 1.0)),
    "conformal_phi4_fd27": dict(nfld=1, time_var=O.CONFORMAL, model=O.MODEL_PHI4, mp=(1.0,),
                                lap=O.LAP_STENCIL, stencil=(-128.0, 14.0, 3.0, 1.0, 30.0)),
    # the chi mass of the Discrete model (model.f90:35-55), m2psi = 3e3
    "cosmic_twofield_mchi_fd7": dict(nfld=2, time_var=O.COSMIC, model=O.MODEL_TWOFIELD, mp=(1.0, 2.5e5, 3.0e3),
                                     lap=O.LAP_STENCIL, stencil=(-6.0, 1.0, 0.0, 0.0, 1.0)),
}


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("order", [2, 4, 6, 8])
def test_symp_matches_oracle(gpu, case, order):
    print("case", case, order, flush=True)
    c = CASES[case]
    n, L = 16, 10.0 if c["nfld"] == 2 else 20.0
    # two-field: m_chi,eff = g phi ~ 500 needs omega*dt well inside the symp stability region
    dt = 1e-3 if c["nfld"] == 2 else (L / n) / 40.0
    fld, fldp = (two_field_ic(n, L, 101) if c["nfld"] == 2 else one_field_ic(n, L, 37))
    g, o = run_pair(gpu, n, L, c["nfld"], c["time_var"], c["model"], c["mp"], c["lap"], c["stencil"],
                    fld, fldp, [("symp", (order, dt, 5)), ("symp", (order, dt, 3))])
    assert rel(g[0], o[0]) < 1e-12
    assert rel(g[1], o[1]) < 1e-12
    assert abs(g[2] - o[2]) < 1e-13 * abs(o[2])
    assert abs(g[3] - o[3]) < 1e-11 * abs(o[3])
    for k in ("rho", "ke", "pe", "ge", "resid", "a", "hubble"):
        assert abs(g[4][k] - o[4][k]) <= 1e-11 * abs(o[4][k]) + 1e-15, k


@pytest.mark.parametrize("case", list(CASES))
def test_single_splits_match_oracle(gpu, case):
    c = CASES[case]
    n, L = 16, 10.0
    fld, fldp = (two_field_ic(n, L, 5) if c["nfld"] == 2 else one_field_ic(n, L, 6))
    plan = [("Hamiltonian_Split", (0.01, 1)), ("Hamiltonian_Split", (0.02, 3)), ("Hamiltonian_Split", (0.01, 2)),
            ("symp_o2step", (0.01, 0.7, 0.3)), ("Hamiltonian_Split", (0.005, 3))]
    g, o = run_pair(gpu, n, L, c["nfld"], c["time_var"], c["model"], c["mp"], c["lap"], c["stencil"],
                    fld, fldp, plan)
    assert rel(g[0], o[0]) < 1e-13
    assert rel(g[1], o[1]) < 1e-13
    assert abs(g[2] - o[2]) < 1e-14 * abs(o[2])
    assert abs(g[3] - o[3]) < 1e-12 * abs(o[3])


@pytest.mark.parametrize("shape", [(16, 16, 8), (32, 32, 64), (48, 48, 16), (64, 64, 32), (96, 96, 8), (128, 128, 16)])
@pytest.mark.parametrize("nfld", [1, 2])
def test_plane_sweeps_match_oracle(gpu, shape, nfld):
    """Spectral steps of lattices with nx = ny (the plane sweeps; at 128 per
    side FP64 takes the inverse one with one field only) and nz of its own."""
    print("case planes", shape, nfld, flush=True)
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + nz)
    fld = 1e-3 * rng.standard_normal((nfld, nz, ny, nx))
    fldp = 1e-3 * rng.standard_normal((nfld, nz, ny, nx))
    fld[0] += 1.0
    fldp[0] -= 0.6
    phi4 = nfld == 1
    g, o = run_pair(gpu, shape, 0.05 * nx, nfld, O.CONFORMAL if phi4 else O.COSMIC,
                    O.MODEL_PHI4 if phi4 else O.MODEL_TWOFIELD, (1.0,) if phi4 else (1.0, 2.5e5), O.LAP_SPECTRAL,
                    (-6, 1, 0, 0, 1), fld, fldp, [("symp", (4, 1e-3, 2)), ("Hamiltonian_Split", (1e-3, 3))])
    assert rel(g[0], o[0]) < 1e-12 and rel(g[1], o[1]) < 1e-12
    assert abs(g[2] - o[2]) < 1e-13 * abs(o[2]) and abs(g[3] - o[3]) < 1e-11 * abs(o[3])
    for k in ("rho", "ke", "pe", "ge"):
        assert abs(g[4][k] - o[4][k]) <= 1e-11 * abs(o[4][k]), k


FD_SHAPES = [(8, 8, 64), (16, 48, 8), (96, 32, 8), (192, 8, 16), (64, 192, 8), (128, 16, 96)]


@pytest.mark.parametrize("shape", FD_SHAPES)
@pytest.mark.parametrize("stencil", [(-6.0, 1.0, 0.0, 0.0, 1.0), (-128.0, 14.0, 3.0, 1.0, 30.0)])
def test_fd_tiles_match_oracle(gpu, shape, stencil):
    """Finite-difference kicks on boxes whose rows, planes and chunks leave
    partial tiles (nx, ny, nz from 8 to 192), an even and an odd number of kicks
    per call (the odd one runs its first kick unfused)."""
    print("case fd tiles", shape, stencil, flush=True)
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + ny + nz)
    fld = 1e-3 * rng.standard_normal((2, nz, ny, nx))
    fldp = 1e-3 * rng.standard_normal((2, nz, ny, nx))
    fld[0] += PHI0_C
    fldp[0] += DPHI0_C
    g, o = run_pair(gpu, shape, 0.05 * nx, 2, O.COSMIC, O.MODEL_TWOFIELD, (1.0, 2.5e5), O.LAP_STENCIL, stencil,
                    fld, fldp, [("symp", (2, 1e-3, 2)), ("symp", (2, 1e-3, 3)), ("symp", (4, 1e-3, 1))])
    assert rel(g[0], o[0]) < 1e-12 and rel(g[1], o[1]) < 1e-12
    assert abs(g[2] - o[2]) < 1e-13 * abs(o[2]) and abs(g[3] - o[3]) < 1e-11 * abs(o[3])
    for k in ("rho", "ke", "pe", "ge"):
        assert abs(g[4][k] - o[4][k]) <= 1e-11 * abs(o[4][k]), k


@pytest.mark.parametrize("shape", [(512, 256, 48), (512, 512, 16)])
@pytest.mark.parametrize("stencil", [(-6.0, 1.0, 0.0, 0.0, 1.0), (-128.0, 14.0, 3.0, 1.0, 30.0)])
@pytest.mark.parametrize("nfld", [1, 2])
def test_fd_partial_chunks_match_oracle(gpu, shape, stencil, nfld):
    """Finite-difference kicks in chunks of 32 planes (boxes with enough tiles for
    them) whose last chunk is shorter: 16 of 48 planes, and the only one 16 of
    16.  A drift sweep with a kick in place, and fused sweeps."""
    print("case fd partial chunks", shape, stencil, nfld, flush=True)
    nx, ny, nz = shape
    rng = np.random.default_rng(nfld + nz)
    fld = 1e-3 * rng.standard_normal((nfld, nz, ny, nx))
    fldp = 1e-3 * rng.standard_normal((nfld, nz, ny, nx))
    fld[0] += PHI0_C
    fldp[0] += DPHI0_C
    tv, model, par = (O.COSMIC, O.MODEL_TWOFIELD, (1.0, 2.5e5)) if nfld == 2 else (O.CONFORMAL, O.MODEL_PHI4, (1.0,))
    plan = [("symp", (2, 1e-3, 2)), ("symp", (2, 1e-3, 1))]
    g, o = run_pair(gpu, shape, 0.05 * nx, nfld, tv, model, par, O.LAP_STENCIL, stencil, fld, fldp, plan)
    assert rel(g[0], o[0]) < 1e-12 and rel(g[1], o[1]) < 1e-12
    for k in ("rho", "ke", "pe", "ge"):
        assert abs(g[4][k] - o[4][k]) <= 1e-11 * abs(o[4][k]), k


class _Device:
    """n reals at a device address, for torch.as_tensor."""

    def __init__(self, ptr, shape, dtype):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr=np.dtype(dtype).str, version=3)


@pytest.mark.parametrize("precision,shape,n", [("f64", (1024, 1024, 192), 64), ("mixed", (1024, 512, 1024), 64),
                                               ("f64", (512, 512, 48), 16), ("mixed", (512, 512, 48), 16)])
@pytest.mark.parametrize("stencil", [(-6.0, 1.0, 0.0, 0.0, 1.0), (-128.0, 14.0, 3.0, 1.0, 30.0)])
def test_fd_large_lattices_match_their_period(gpu, precision, shape, n, stencil):
    """A state with the period of an n^3 lattice against that lattice, three
    leapfrog steps (an unfused and two fused kicks): lattices with more tiles and
    chunks than the 8192 blocks of a kick, so that blocks take a second item,
    and chunks of 32 planes of which the last is half full.  Sites see the same
    operations with background coefficients from sums in another order: a few
    roundings of the largest value."""
    import torch

    print("case fd period", precision, shape, n, stencil, flush=True)
    tile = {"f64": 64 * 8 * 32, "mixed": 64 * 16 * 32}[precision]  # sites of an item
    assert n == 16 or shape[0] * shape[1] * shape[2] // tile > 8192
    dtype = np.float64 if precision == "f64" else np.float32
    kw = dict(nfld=1, precision=gpu.F64 if precision == "f64" else gpu.MIXED, model=gpu.MODEL_PHI4,
              model_params=(0.7,), laplacian=gpu.LAP_STENCIL, stencil=stencil)
    rng = np.random.default_rng(8)
    init = [torch.from_numpy(rng.standard_normal((n, n, n)).astype(dtype)).cuda() for _ in range(2)]
    reps = tuple(shape[2 - d] // n for d in range(3))

    def view(lat):
        return [torch.as_tensor(_Device(ptr, (lat.nz, lat.ny, lat.nx), dtype), device="cuda")
                for ptr in lat.device_state()]

    with gpu.Lattice(n, length=0.125 * n, **kw) as small, gpu.Lattice(shape, length=0.125 * shape[0], **kw) as big:
        for lat in (small, big):
            lat.set_scalars(1.0, 0.0)
            for v, x in zip(view(lat), init):
                v.copy_(x if lat is small else x.repeat(reps))
            torch.cuda.synchronize()
            lat.calc_metric()
            lat.symp2(2e-3, 3)
            lat.synchronize()
        eps = float(np.finfo(dtype).eps)
        y = [lat.scalars for lat in (small, big)]
        assert abs(y[0][0] - y[1][0]) <= 1e-13 * abs(y[0][0]) and abs(y[0][1] - y[1][1]) <= 1e-12 * abs(y[0][1])
        for a, b in zip(view(small), view(big)):
            top, worst = float(a.abs().max()), 0.0
            for k in range(0, shape[2], n):
                worst = max(worst, float((b[k:k + n] - a.repeat(1, reps[1], reps[2])).abs().max()))
            print("largest difference", worst, "of", top, flush=True)
            assert worst <= 16 * eps * top


@pytest.mark.parametrize("shape", [(8, 16, 32), (16, 8, 48), (48, 32, 8), (64, 16, 96), (32, 192, 16), (192, 48, 8),
                                   (16, 256, 8), (256, 8, 16), (8, 8, 512), (16, 512, 8)])
@pytest.mark.parametrize("nfld", [1, 2])
def test_column_tiles_match_oracle(gpu, shape, nfld):
    """y and z sweeps whose tiles of columns run over the ends of rows (pitches
    8 to 136, tiles of 4 to 64 columns): FP64 against the oracle; the mixed form
    against FP64, 34 roundings of FP32 (2 per radix-2 level of 2^17 sites)."""
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + 3 * ny + 5 * nz)
    fld = 1e-3 * rng.standard_normal((nfld, nz, ny, nx))
    fldp = 1e-3 * rng.standard_normal((nfld, nz, ny, nx))
    fld[0] += PHI0_C
    fldp[0] += DPHI0_C
    tv, model, par = (O.COSMIC, O.MODEL_TWOFIELD, (1.0, 2.5e5)) if nfld == 2 else (O.CONFORMAL, O.MODEL_PHI4, (1.0,))
    print("case column tiles", shape, nfld, flush=True)
    g, o = run_pair(gpu, shape, 0.05 * nx, nfld, tv, model, par, O.LAP_SPECTRAL, (-6, 1, 0, 0, 1), fld, fldp,
                    [("symp", (2, 1e-3, 1))])
    assert rel(g[0], o[0]) < 1e-12 and rel(g[1], o[1]) < 1e-12
    for k in ("rho", "ke", "pe", "ge"):
        assert abs(g[4][k] - o[4][k]) <= 1e-11 * abs(o[4][k]), k
    with gpu.Lattice(shape, nfld=nfld, length=0.05 * nx, precision=gpu.MIXED, time_var=tv, model=model,
                     model_params=par) as lat:
        lat.set_state(fld, fldp, 1.0, 0.0)
        lat.calc_metric()
        lat.symp(2, 1e-3, 1)
        m = lat.get_state()
    for a, b in zip(m[:2], g[:2]):
        for l in range(nfld):
            d = a[l] - b[l]
            assert np.linalg.norm(d - d.mean()) < 34 * 2.0**-24 * np.linalg.norm(b[l] - b[l].mean())


@pytest.mark.parametrize("members", [None, 3])
@pytest.mark.parametrize("precision,tol", [("f64", 1e-13), ("mixed", 2e-6)])
def test_fd_fused_kicks_match_single_steps(gpu, precision, tol, members):
    """One call of four leapfrog steps (fused drift + kick sweeps) against four
    calls of one step (a drift sweep and a kick each), single and batched: the
    same fluctuations to a few roundings per step."""
    print("case fd fused", precision, members, flush=True)
    n, L, dt = (48, 32, 16), 2.4, 1e-3
    rng = np.random.default_rng(3)
    fld = 1e-3 * rng.standard_normal((2, 16, 32, 48))
    fldp = 1e-3 * rng.standard_normal((2, 16, 32, 48))
    fld[0] += PHI0_C
    fldp[0] += DPHI0_C
    kw = dict(nfld=2, length=L, laplacian=gpu.LAP_STENCIL, precision=gpu.F64 if precision == "f64" else gpu.MIXED)
    got = []
    for calls in ((4,), (1, 1, 1, 1)):
        with gpu.Lattice(n, members=None if members is None else [(1.0, 2.5e5)] * members, **kw) as lat:
            views = [lat] if members is None else [lat.member(m) for m in range(members)]
            for v in views:
                v.set_state(fld, fldp, 1.0, 0.0)
                v.calc_metric()
            for k in calls:
                lat.symp2(dt, k)
            got.append(views[-1].get_state())
            if members is not None:
                for v in views:
                    v.close()
    for a, b in zip(got[0][:2], got[1][:2]):
        for l in range(2):
            assert np.linalg.norm(a[l] - b[l]) < tol * np.linalg.norm(b[l] - b[l].mean())
    assert abs(got[0][2] - got[1][2]) < 1e-13 * abs(got[1][2])


def test_state_roundtrip_ghost_layout(gpu):
    """AoS ghosted fld(nfld,0:nx+1,...) in, periodic ghosts out (wrap_fields)."""
    n = 8
    rng = np.random.default_rng(0)
    fld = rng.standard_normal((2, n, n, n))
    fldp = rng.standard_normal((2, n, n, n))
    g = np.zeros((n + 2, n + 2, n + 2, 2))
    g[1:-1, 1:-1, 1:-1, :] = np.moveaxis(fld, 0, -1)
    O.wrap_fields(g)
    with gpu.Lattice(n, nfld=2, length=10.0) as lat:
        lat.set_state_aos(g, np.ascontiguousarray(np.moveaxis(fldp, 0, -1)), 1, 1.25, -0.5)
        aos, aosp, y, p = lat.get_state_aos(1)
    assert np.array_equal(aos, g)
    assert np.array_equal(aosp, np.moveaxis(fldp, 0, -1))
    assert (y, p) == (1.25, -0.5)
