"""The work whose speed is followed, case by case, through the library's public entry points.

A `step` case is one analysis step of one run through the C ABI of include/spo_hip.h, the calls that a driver makes
between two records: spo_hip_propagate_analysis_step, spo_hip_analyse, the specular wave for the analysis surface,
and what it writes out (the whole wave for a restart file, or the densities and the analysis plane of a big grid). A
`batch` case is the same for several runs stepped together. The tables are those of include/spo_hip.h with the
structure and the magnitudes of a real run (unit-modulus kinetic and rotational phases, absorbers close to 1, a Gauss-
Legendre rule, a potential of -5 to 10 eV times the time step) and the wave fills the grid, as it does late in a run.
A `train` / `predict` case is the potential surrogate, a `crp` / `scm` case the CRP surface on given geometries.

The ranges that draw() covers: (Z, r) grids of 32 x 12 to 176 x 64 points, 4 x 4 to 16 x 16 (x, y) points, molecules
with two equal atoms up to JMax 28 and with unequal ones up to JMax 15, both precisions, with and without a symmetry-
reduced potential; batches of 16 to 16384 rows; 1 to 2^20 geometries.
"""

import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cpp-spo-dvr_amd"))

import spodvr_amd  # noqa: E402

GOLDEN = os.path.join(ROOT, "tests", "golden")


def step(name, **k):
    return {"name": name, "kind": "step", "homonuclear": True, "sym": False, "needs_shift": False, **k}


def listed():
    return [
        # The smallest grid with all six degrees of freedom: a first look at a surface, a convergence series.
        step("smoke_fp64", nz=64, nr=16, nxy=4, nzsp=128, nzpot=50, jmax=4, precision="fp64", steps=5, read="wave"),
        # The HardWallPES workload: 128 x 32 x 8 x 8, JMax 10 (6 theta x 22 phi), analysis on 200 energies.
        step("hardwall_fp64", nz=128, nr=32, nxy=8, nzsp=192, nzpot=43, jmax=10, precision="fp64", steps=5,
             read="densities"),
        # One surface of a series of distorted slabs (CRP + SCM): 110 x 48 x 6 x 6, 20 time steps per analysis step,
        # oblique incidence (the momentum shift is not the identity).
        step("distorted_slab_fp64", nz=110, nr=48, nxy=6, nzsp=198, nzpot=100, jmax=4, precision="fp64", steps=20,
             needs_shift=True, read="densities"),
        # HD: every J, twice the theta points, no symmetry; a ragged 90 x 40 x 10 x 10 grid in complex64.
        step("hd_mixed", nz=90, nr=40, nxy=10, nzsp=180, nzpot=63, jmax=9, precision="mixed", steps=5,
             homonuclear=False, read="densities"),
        # The reference's published run: 160 x 40 x 12 x 12, JMax 28 (15 theta x 60 phi).
        step("thesis_fp64", nz=160, nr=40, nxy=12, nzsp=320, nzpot=110, jmax=28, precision="fp64", steps=5, sym=True,
             read="densities"),
        # The Dai-Light H2/Cu(111) workload of bench.py: 96 x 48 x 16 x 16, JMax 24, MJMax 23 (13 theta x 48 phi),
        # in both precisions.
        step("dz_fp64", nz=96, nr=48, nxy=16, nzsp=512, nzpot=66, jmax=24, mjmax=23, precision="fp64", steps=5,
             sym=True, read="densities"),
        step("dz_mixed", nz=96, nr=48, nxy=16, nzsp=512, nzpot=66, jmax=24, mjmax=23, precision="mixed", steps=5,
             sym=True, read="densities"),
        # Four runs of uneven size stepped together (spo_hip_propagate_batch): the reduced members of the batched workload
        # (JMax 12 and 18, NR 32) on an 8 x 8 (x, y) grid.
        {"name": "batch_mixed", "kind": "batch", "nz": 96, "nr": 32, "nxy": 8, "nzsp": 256, "nzpot": 66,
         "precision": "mixed", "jmaxs": "12,18,12,18", "steps": 5, "sym": True},
        # The surrogate's training: Adam steps of 4096 rows over a data set resident on the host.
        {"name": "train_4096", "kind": "train", "batch": 4096, "rows": 65536, "steps": 32},
        # The surrogate on a slab of grid points, a count that fills no tile.
        {"name": "predict_500k", "kind": "predict", "batch": 4096, "rows": 500003},
        # Single geometries of the CRP surface, as a trajectory or a cut through the potential asks for them.
        {"name": "crp_1000", "kind": "crp", "n": 1000},
        # A chunk of the potential grid of a distorted slab (CRP + SCM, the 73-atom example slab).
        {"name": "scm_300k", "kind": "scm", "n": 300007},
    ]


# ---- drawn cases ------------------------------------------------------------------------------------------------

def smooth(n):
    for p in (2, 3, 5, 7, 11):
        while n % p == 0:
            n //= p
    return n == 1


def sizes(lo, hi):
    """The even FFT lengths of a grid axis."""
    return [n for n in range(lo, hi + 1) if n % 2 == 0 and smooth(n)]


def log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["batch", "train", "predict", "crp", "scm"])
    if kind == "train":
        return {"kind": "train", "batch": 16 * log_uniform(rng, 1, 1024), "rows": 65536, "steps": rng.randint(1, 32)}
    if kind == "predict":
        return {"kind": "predict", "batch": 4096, "rows": log_uniform(rng, 1, 1 << 19)}
    if kind in ("crp", "scm"):
        return {"kind": kind, "n": log_uniform(rng, 1, 1 << 18)}
    precision = rng.choice(["fp64", "mixed"])
    if kind == "batch":
        jmaxs = ",".join(str(rng.choice([4, 6, 8, 10, 12, 18])) for _ in range(rng.randint(2, 4)))
        nz = rng.choice(sizes(32, 96))
        return {"kind": "batch", "nz": nz, "nr": rng.choice(sizes(12, 32)), "nxy": rng.choice([4, 6, 8]),
                "nzsp": rng.choice(sizes(2 * nz, 3 * nz)), "nzpot": int(nz * rng.uniform(0.3, 0.9)),
                "precision": precision, "jmaxs": jmaxs, "steps": 5, "sym": rng.random() < 0.5}
    while True:
        homonuclear = rng.random() < 0.7
        c = {"kind": "step", "nz": rng.choice(sizes(32, 176)), "nr": rng.choice(sizes(12, 64)),
             "nxy": rng.choice(sizes(4, 16)), "jmax": 2 * rng.randint(1, 14) if homonuclear else rng.randint(3, 15),
             "homonuclear": homonuclear, "sym": rng.random() < 0.5, "needs_shift": rng.random() < 0.3,
             "precision": precision, "steps": rng.choice([1, 5, 5, 20]), "read": "wave"}
        c["nzsp"] = rng.choice(sizes(c["nz"], 3 * c["nz"]))
        c["nzpot"] = int(c["nz"] * rng.uniform(0.3, 0.95))
        values = c["nz"] * c["nr"] * c["nxy"] ** 2 * len(basis(c)[1])
        if 2e5 < values * c["steps"] / 5 and values < 1.5e7 and values * c["steps"] < 1.2e8:
            c["read"] = "wave" if values < 2e6 else "densities"
            return c


# ---- the tables of a run ----------------------------------------------------------------------------------------

def basis(c):
    """theta points, [(J, m)] in mJ blocks and phi points of a case."""
    jmax, step_j = c["jmax"], 2 if c["homonuclear"] else 1
    mmax = c.get("mjmax", jmax)
    j0 = jmax % 2 if c["homonuclear"] else 0
    states = [(j, m) for m in range(-mmax, mmax + 1) for j in range(j0, jmax + 1, step_j) if j >= abs(m)]
    n_theta = (jmax - j0) // step_j + 1
    n_phi = 2 * mmax + 2
    while not smooth(n_phi):
        n_phi += 2
    return n_theta, states, n_phi


def legendre(c):
    """sqrt(w / n_phi) P_J^m(theta), one (n_theta, n_J) matrix per mJ block; normalised so that n_phi L^T L = 1."""
    n_theta, states, n_phi = basis(c)
    jmax = c["jmax"]
    x, w = np.polynomial.legendre.leggauss(jmax + 1)
    x, w = x[::-1][:n_theta], w[::-1][:n_theta].copy()
    if c["homonuclear"]:
        w *= 2.0
        if jmax % 2 == 0:
            w[-1] *= 0.5  # theta = pi / 2 counted once
    out = {}
    for m in sorted({m for _, m in states}):
        a = abs(m)
        p = {a: np.sqrt(np.prod([(2 * k + 1) / (2 * k) for k in range(1, a + 1)]) / 2) * (1 - x * x) ** (a / 2)}
        if m > 0 and a % 2:
            p[a] = -p[a]
        prev = np.zeros_like(x)
        for j in range(a + 1, jmax + 1):
            f = math.sqrt((4 * j * j - 1) / (j * j - a * a))
            g = math.sqrt(((j - 1) ** 2 - a * a) / (4 * (j - 1) ** 2 - 1)) if j > a + 1 else 0.0
            p[j] = f * (x * p[j - 1] - g * prev)
            prev = p[j - 1]
        js = [j for j, mm in states if mm == m]
        out[m] = np.stack([p[j] * np.sqrt(w / n_phi) for j in js], axis=1)
    return out


def phase(a):
    return np.exp(-1j * a)


def tables(c, seed):
    """Every array of spo_hip_tables and spo_hip_analysis as numpy arrays and torch tensors, from the seed alone."""
    rng = np.random.default_rng(seed)
    n_theta, states, n_phi = basis(c)
    n_rot, nz, nr, nx, nzsp = len(states), c["nz"], c["nr"], c["nxy"], c["nzsp"]
    n_xy, n_tp = nx * nx, n_theta * n_phi
    dt, mass, mu = 2.0, 3674.0, 918.6
    t = {"n_theta": n_theta, "n_phi": n_phi, "n_rot": n_rot, "n_xy": n_xy, "states": states}

    def kinetic(n, d, m):
        k = 2 * np.pi * np.fft.fftfreq(n, d)
        return k * k / (2 * m)

    dz, dr = 0.135 * rng.uniform(0.95, 1.05), 0.11 * rng.uniform(0.95, 1.05)
    er = kinetic(nr, dr, mu)
    exy = (kinetic(nx, 4.82 / nx, mass)[:, None] + kinetic(nx, 4.82 / nx, mass)[None, :]).reshape(-1)
    for tag, f in (("full", 1.0), ("half", 0.5)):
        t["zr_" + tag] = phase(f * dt * (kinetic(nz, dz, mass)[:, None] + er[None, :])).reshape(-1)
        t["specular_" + tag] = phase(f * dt * (kinetic(nzsp, dz, mass)[:, None] + er[None, :])).reshape(-1)
        t["xy_" + tag] = phase(f * dt * exy)
    t["scales"] = (dz / math.sqrt(2 * math.pi), dr / math.sqrt(2 * math.pi), math.sqrt(4.82 / nx) / math.sqrt(nx),
                   math.sqrt(4.82 / nx) / math.sqrt(nx))
    r = 0.8 + dr * np.arange(nr)
    j = np.array([s[0] for s in states])
    rot = phase(dt / 2 * (j * (j + 1))[None, :] / (2 * mu * r[:, None] ** 2))  # [ir][irot]
    vasy = rng.uniform(-0.17, 0.1, nr)

    def absorber(n):
        x = np.clip((np.arange(n) - 0.8 * n) / (0.2 * n), 0, None)
        return np.exp(-0.02 * x * x)

    t["z_optical"], t["z_specular_optical"] = absorber(nz), absorber(nzsp)
    t["r_absorber_first"] = int(0.8 * nr)
    t["r_optical"] = absorber(nr)
    t["rotation_half"] = rot.reshape(-1)
    t["before_interaction"] = (t["r_optical"][:, None] * rot).reshape(-1)
    t["gas_phase_step"] = (t["r_optical"][:, None] * rot * phase(vasy * dt)[:, None] * rot).reshape(-1)
    t["ichn"] = states.index((j.min(), 0))
    t["specular_gas_phase"] = rot[:, t["ichn"]] ** 2 * phase(vasy * dt)
    k0 = rng.uniform(0.5, 3.0, 2) if c["needs_shift"] else np.zeros(2)
    a = (k0[0] * np.arange(nx)[:, None] / nx + k0[1] * np.arange(nx)[None, :] / nx).reshape(-1)
    cell = 4.82 ** 2 * math.sin(math.pi / 3)
    t["shift_forward"], t["shift_backward"] = phase(a), phase(-a)
    t["specular_to_scattering"] = phase(-a) / math.sqrt(cell)
    t["scattering_to_specular"] = phase(a) / math.sqrt(cell) * (cell / n_xy)
    t["legendre"] = legendre(c)
    blocks = sorted(t["legendre"])
    t["block_size"] = np.array([t["legendre"][m].shape[1] for m in blocks], dtype=np.int32)
    t["block_first"] = (np.cumsum(t["block_size"]) - t["block_size"]).astype(np.int32)
    # Symmetry: under C6v about an eighth of the sites hold a potential, the others map to one of them with the
    # azimuth turned and mirrored.
    if c["sym"]:
        n_rep, n_op = max(1, n_xy // 8), 12
        t["representative_of"] = rng.permutation(n_xy).astype(np.int32) % n_rep
        t["operation_of"] = rng.integers(0, n_op, n_xy).astype(np.int32)
        ip = np.arange(n_phi)
        t["phi_index"] = np.stack([((ip if o < 6 else -ip) + (o % 6) * n_phi // 6) % n_phi for o in range(n_op)])
    else:
        n_rep, n_op = n_xy, 1
        t["representative_of"], t["operation_of"] = np.arange(n_xy, dtype=np.int32), np.zeros(n_xy, dtype=np.int32)
        t["phi_index"] = np.arange(n_phi)[None, :]
    t["phi_index"] = np.ascontiguousarray(t["phi_index"], dtype=np.int32)
    t["n_rep"], t["n_op"] = n_rep, n_op
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    angle = torch.rand((c["nzpot"] * nr, n_rep, n_tp), generator=gen, device="cuda", dtype=torch.float64) * 1.1 - 0.75
    t["exp_potential"] = torch.polar(torch.ones((), device="cuda", dtype=torch.float64), angle)
    # The wave, (irot, ixy, izr) with irot fastest as the host holds it, and the specular wave.
    psi = torch.randn((nz * nr, n_xy, n_rot, 2), generator=gen, device="cuda", dtype=torch.float64)
    t["wave"] = torch.view_as_complex(psi.mul_(1e-3))
    spec = torch.randn((nzsp, nr, 2), generator=gen, device="cuda", dtype=torch.float64)
    t["spec"] = torch.view_as_complex(spec.mul_(1e-2))
    # Analysis: the states up to about half the basis, all diffraction channels of the grid, three vibrations.
    t["rotation_index"] = np.flatnonzero(j <= max(j.min(), 0.6 * c["jmax"])).astype(np.int32)
    t["diffraction_slot"] = rng.permutation(n_xy).astype(np.int32)[:max(1, int(0.8 * n_xy))]
    n_v, q = 3, (r - 1.5) / 0.3
    radial = np.stack([np.exp(-q * q / 2), q * np.exp(-q * q / 2), (2 * q * q - 1) * np.exp(-q * q / 2)])
    t["initial_radial"] = radial
    stretch = rng.uniform(0.9, 1.1, len(t["rotation_index"]))
    t["radial_weight"] = radial[:, None, :] * stretch[None, :, None] * dr  # [v][irotana][ir]
    t["n_v"], t["dr"], t["xy_scale"] = n_v, dr, 4.82 ** 2 / n_xy
    t["iz_analysis"], t["iz_specular"] = int(0.78 * nz), int(0.7 * nzsp)
    t["energies"] = np.linspace(0.2, 1.0, 100) / 27.2114
    return t


# ---- the C ABI --------------------------------------------------------------------------------------------------

_D, _I, _V = ctypes.c_double, ctypes.c_int, ctypes.c_void_p


def _struct(name, fields):
    return type(name, (ctypes.Structure,), {"_fields_": fields})


Shape = _struct("Shape", [(n, _I) for n in (
    "n_rot nx ny nr nz nz_specular nz_potential n_theta n_phi n_representatives n_operations initial_channel mj_max "
    "steps_per_analysis r_absorber_first r_absorber_last needs_shift precision").split()])
Tables = _struct("Tables", [(n, _V) for n in "zr_full zr_half xy_full xy_half specular_full specular_half".split()]
                 + [("fft_scale_" + n, _D) for n in "zrxy"]
                 + [(n, _V) for n in (
                     "rotation_half before_interaction gas_phase_step specular_gas_phase z_optical r_optical "
                     "z_specular_optical shift_forward shift_backward specular_to_scattering scattering_to_specular "
                     "legendre block_first block_size exp_potential representative_of operation_of "
                     "phi_index").split()])
Analysis = _struct("Analysis", [(n, _I) for n in (
    "n_states n_v n_rotation n_diffraction n_energies iz_analysis initial_state").split()]
    + [(n, _V) for n in "rotation_index diffraction_slot radial_weight initial_radial".split()]
    + [(n, _D) for n in "dr xy_scale analysis_time_step".split()] + [("total_energy_hartree", _V)])

_lib = None


def library():
    global _lib
    if _lib is None:
        spodvr_amd.host_library()
        _lib = ctypes.CDLL(spodvr_amd.library_path("libspo_hip.so"))
        _lib.spo_hip_last_error.restype = ctypes.c_char_p
        _lib.spo_hip_create.argtypes = [_V] * 5
        _lib.spo_hip_analyse.argtypes = [_V, _I, _I, _D, _V]
        _lib.spo_hip_get_z_plane.argtypes = [_V, _I, _V]
        _lib.spo_hip_upload_wave.argtypes = _lib.spo_hip_download_wave.argtypes = [_V, _V, _V]
        _lib.spo_hip_get_specular.argtypes = _lib.spo_hip_block_densities.argtypes = [_V, _V]
        _lib.spo_hip_propagate_batch.argtypes = [_V, _I]
        _lib.spo_hip_destroy.argtypes = _lib.spo_hip_propagate_analysis_step.argtypes = [_V]
    return _lib


def call(status):
    if status:
        raise RuntimeError(library().spo_hip_last_error().decode())


def _ptr(a):
    return a.ctypes.data


class Backend:
    """One run of the C ABI: its handle and the host arrays that its results go to."""

    def __init__(self, c, seed):
        self.handle, lib, t = None, library(), tables(c, seed)
        n_states = len(t["rotation_index"]) * len(t["diffraction_slot"])
        initial = int(np.flatnonzero(t["rotation_index"] == t["ichn"])[0]) * len(t["diffraction_slot"])
        shape = Shape(t["n_rot"], c["nxy"], c["nxy"], c["nr"], c["nz"], c["nzsp"], c["nzpot"], t["n_theta"], t["n_phi"],
                      t["n_rep"], t["n_op"], t["ichn"], max(m for _, m in t["states"]), c["steps"],
                      t["r_absorber_first"], c["nr"] - 1, int(c["needs_shift"]), int(c["precision"] == "mixed"))
        t["legendre"] = np.concatenate([t["legendre"][m].reshape(-1) for m in sorted(t["legendre"])])
        t["exp_potential"] = t["exp_potential"].cpu().numpy()
        spec = t["spec"].cpu().numpy()
        keep, tab = [], Tables()
        for name, kind in Tables._fields_:
            if kind is _V:
                keep.append(np.ascontiguousarray(t[name]))
                setattr(tab, name, _ptr(keep[-1]))
        tab.fft_scale_z, tab.fft_scale_r, tab.fft_scale_x, tab.fft_scale_y = t["scales"]
        weights = np.ascontiguousarray(t["radial_weight"])
        radial, energies = np.ascontiguousarray(t["initial_radial"]), np.ascontiguousarray(t["energies"])
        ana = Analysis(n_states, t["n_v"], len(t["rotation_index"]), len(t["diffraction_slot"]), len(energies),
                       t["iz_analysis"], initial, _ptr(t["rotation_index"]), _ptr(t["diffraction_slot"]), _ptr(weights),
                       _ptr(radial), t["dr"], t["xy_scale"], 2.0 * c["steps"], _ptr(energies))
        handle = _V()
        call(lib.spo_hip_create(ctypes.byref(shape), ctypes.byref(tab), ctypes.byref(ana), _ptr(spec),
                                ctypes.byref(handle)))
        self.handle = handle
        wave = t.pop("wave").cpu().numpy()
        call(lib.spo_hip_upload_wave(handle, _ptr(wave), _ptr(spec)))
        self.iz, self.iz_specular, self.time, self.dt = t["iz_analysis"], t["iz_specular"], 0.0, 2.0 * c["steps"]
        n_izr = c["nz"] * c["nr"]
        self.bk = np.empty((t["n_v"], n_states), dtype=np.complex128)
        self.specular = np.empty((c["nzsp"], c["nr"]), dtype=np.complex128)
        if c.get("read") == "wave":
            self.wave = np.empty((n_izr, t["n_xy"], t["n_rot"]), dtype=np.complex128)
        else:
            self.densities = np.empty(n_izr)
            self.plane = np.empty((c["nr"], t["n_xy"], t["n_rot"]), dtype=np.complex128)
        self.read = c.get("read")

    def results(self):
        """The analysis at the new time, and what is written out."""
        lib = library()
        self.time += self.dt
        call(lib.spo_hip_analyse(self.handle, 1, self.iz_specular, self.time, _ptr(self.bk)))
        if self.read == "wave":
            call(lib.spo_hip_download_wave(self.handle, _ptr(self.wave), _ptr(self.specular)))
            return {"bk": self.bk, "specular": self.specular, "wave": self.wave}
        call(lib.spo_hip_get_specular(self.handle, _ptr(self.specular)))
        call(lib.spo_hip_block_densities(self.handle, _ptr(self.densities)))
        call(lib.spo_hip_get_z_plane(self.handle, self.iz, _ptr(self.plane)))
        return {"bk": self.bk, "specular": self.specular, "densities": self.densities, "plane": self.plane}

    def __del__(self):
        if self.handle:
            library().spo_hip_destroy(self.handle)


def members(c):
    return [{**c, "kind": "step", "jmax": int(j), "homonuclear": True, "needs_shift": False, "read": "densities"}
            for j in c["jmaxs"].split(",")]


# ---- surrogate and CRP ------------------------------------------------------------------------------------------

def network(rng):
    w = [rng.normal(0, 1 / math.sqrt(a), (a, b)) for a, b in ((6, 128), (128, 128), (128, 128), (128, 1))]
    b = [rng.normal(0, 0.05, n) for n in (128, 128, 128, 1)]
    return np.concatenate([x.reshape(-1) for pair in zip(w, b) for x in pair]).astype(np.float32)


def samples(rng, n):
    x = rng.uniform(-1, 1, (n, 6)).astype(np.float32)
    t = (np.sin(2 * x[:, 0]) * x[:, 3] + x[:, 1] ** 2 - 0.5 * x[:, 2] * x[:, 5]).astype(np.float32)
    return x, t


def geometries(rng, n):
    """u v Z r theta phi over a cell of the SRP48 data set's Cu(111) surface, the range of a potential grid."""
    lo, hi = np.array([0.0, 0.0, 1.0, 0.9, 0.0, 0.0]), np.array([4.8, 4.8, 8.0, 4.0, math.pi, 2 * math.pi])
    return lo + (hi - lo) * rng.random((n, 6))


CRP_DATA = os.path.join(GOLDEN, "crp", "cu111_srp48", "dataset")


# ---- the interface ----------------------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return {"kind": kind, "run": Backend(case, seed)}
    if kind == "batch":
        runs = [Backend(m, seed + 7919 * k) for k, m in enumerate(members(case))]
        return {"kind": kind, "runs": runs, "handles": (_V * len(runs))(*[r.handle for r in runs])}
    rng = np.random.default_rng(seed)
    if kind in ("train", "predict"):
        net = spodvr_amd.Mlp(case["batch"])
        net.params = network(rng)
        n = case["rows"] // case["batch"] * case["batch"] if kind == "train" else case["rows"]
        x, t = samples(rng, n)
        return {"kind": kind, "net": net, "x": x, "t": t, "steps": case.get("steps")}
    if kind == "crp":
        return {"kind": kind, "surface": spodvr_amd.CrpSurface(CRP_DATA), "points": geometries(rng, case["n"])}
    example = os.path.join(GOLDEN, "scm", "example")
    surface = spodvr_amd.ScmSurface(CRP_DATA, os.path.join(example, "params.dat"),
                                    os.path.join(example, "examplePosfile.dat"))
    return {"kind": kind, "surface": surface, "points": geometries(rng, case["n"])}


def run(state):
    kind = state["kind"]
    if kind == "step":
        call(library().spo_hip_propagate_analysis_step(state["run"].handle))
        return state["run"].results()
    if kind == "batch":
        call(library().spo_hip_propagate_batch(state["handles"], len(state["runs"])))
        return [r.results() for r in state["runs"]]
    if kind == "train":
        losses = state["net"].train(state["x"], state["t"], state["steps"], 1e-3)
        return {"losses": losses, "params": state["net"].params}
    if kind == "predict":
        return state["net"].predict(state["x"])
    if kind == "crp":
        return state["surface"].device_qd(state["points"])
    return state["surface"].device_values(state["points"])


def work(case):
    kind = case["kind"]
    if kind == "batch":
        each = [work(m) for m in members(case)]
        return {k: sum(w[k] for w in each) for k in each[0]}
    if kind in ("train", "predict"):
        macs = 6 * 128 + 2 * 128 * 128 + 128
        if kind == "predict":
            return {"bytes": case["rows"] * 28.0, "flops": 2.0 * macs * case["rows"]}
        rows = case["batch"] * case["steps"]
        return {"bytes": rows * 28.0 + case["steps"] * 7 * 4 * 34049.0, "flops": 6.0 * macs * rows}
    if kind in ("crp", "scm"):
        return {"bytes": 56.0 * case["n"], "flops": (10e3 if kind == "crp" else 25e3) * case["n"]}
    n_theta, states, n_phi = basis(case)
    n_xy, n_zr, n_pot, n_rot = case["nxy"] ** 2, case["nz"] * case["nr"], case["nzpot"] * case["nr"], len(states)
    b = 16.0 if case["precision"] == "fp64" else 8.0
    psi, steps = float(n_xy) * n_zr * n_rot, case["steps"]
    n_rep = max(1, n_xy // 8) if case["sym"] else n_xy
    table = float(n_theta) * n_phi * n_rep * n_pot
    # each T_Zr and each T_xy reads and writes the wave once, each V its share of it and the potential's phases
    step_bytes = (steps + 1) * 4 * psi * b + steps * (2 * psi * n_pot / n_zr + table) * b
    out = (psi if case.get("read") == "wave" else n_xy * n_rot * case["nr"] + n_zr / 2) * 16.0 + psi * b
    fft = 10 * psi * (math.log2(n_zr) + math.log2(n_xy))
    per_m = sum(sum(1 for j, mm in states if mm == m) for m in {m for _, m in states})
    dvr = float(n_xy) * n_pot * (8 * n_theta * per_m + 10 * n_theta * n_phi * math.log2(n_phi))
    return {"bytes": step_bytes + out, "flops": (steps + 1) * fft + steps * dvr}


# ---- 64-bit values, in plain torch ------------------------------------------------------------------------------

def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def exact_step(c, seed):
    t = tables(c, seed)
    nz, nr, nx, n_xy, n_rot, nzpot = c["nz"], c["nr"], c["nxy"], t["n_xy"], t["n_rot"], c["nzpot"]
    n_pot, n_phi, n_theta, ichn = nzpot * nr, t["n_phi"], t["n_theta"], t["ichn"]
    psi = t.pop("wave").permute(1, 2, 0).contiguous()  # [ixy][irot][izr]
    spec = t["spec"]
    table = t.pop("exp_potential")  # [izr][rep][itp]
    g = {k: _cuda(v) for k, v in t.items() if isinstance(v, np.ndarray)}
    rot = g["rotation_half"].reshape(nr, n_rot)
    before, gas = g["before_interaction"].reshape(nr, n_rot), g["gas_phase_step"].reshape(nr, n_rot)
    inside = torch.arange(nz, device="cuda") < nzpot
    diagonal = torch.where(inside[:, None, None], before[None], gas[None]) * g["z_optical"][:, None, None]
    diagonal = diagonal.reshape(nz * nr, n_rot).t().contiguous()
    rot_pot = rot.repeat(nzpot, 1).t().contiguous()
    mats = [(m, int(f), _cuda(t["legendre"][m])) for m, f in zip(sorted(t["legendre"]), t["block_first"])]

    def angular(ixy):
        x = psi[ixy, :, :n_pot]
        grid = torch.zeros((n_theta, n_phi, n_pot), device="cuda", dtype=torch.complex128)
        xr = torch.view_as_real(x).reshape(n_rot, 2 * n_pot)
        for m, f, L in mats:
            grid[:, m % n_phi] = torch.view_as_complex((L @ xr[f:f + L.shape[1]]).reshape(n_theta, n_pot, 2))
        grid = torch.fft.ifft(grid, dim=1, norm="forward")
        maps = g["phi_index"][int(t["operation_of"][ixy])].long()
        u = table[:, int(t["representative_of"][ixy])].reshape(n_pot, n_theta, n_phi)[:, :, maps]
        grid = torch.fft.fft(grid * u.permute(1, 2, 0), dim=1)
        for m, f, L in mats:
            d = torch.view_as_real(grid[:, m % n_phi].contiguous()).reshape(n_theta, 2 * n_pot)
            y = torch.view_as_complex((L.t().contiguous() @ d).reshape(L.shape[1], n_pot, 2))
            psi[ixy, f:f + L.shape[1], :n_pot] = y * rot_pot[f:f + L.shape[1]]

    def block(half, kinetic_only):
        nonlocal psi, spec
        tag = "half" if half else "full"
        spec = torch.fft.ifft2(torch.fft.fft2(spec) * g["specular_" + tag].reshape(-1, nr))
        if not kinetic_only:
            spec[nzpot:] *= g["specular_gas_phase"]
            spec = spec * g["z_specular_optical"][:, None]
            spec[:, t["r_absorber_first"]:] *= g["r_optical"][t["r_absorber_first"]:]
        zr, xy = g["zr_" + tag].reshape(nz, nr), g["xy_" + tag].reshape(nx, nx)[:, :, None]
        for ixy in range(n_xy):
            p = psi[ixy].reshape(n_rot, nz, nr)
            psi[ixy] = torch.fft.ifft2(torch.fft.fft2(p) * zr).reshape(n_rot, -1)
        for irot in range(n_rot):
            p = (psi[:, irot] * g["shift_forward"][:, None]).reshape(nx, nx, -1)
            p = torch.fft.ifft2(torch.fft.fft2(p, dim=(0, 1)) * xy, dim=(0, 1)).reshape(n_xy, -1)
            p = p * g["shift_backward"][:, None]
            psi[:, irot] = p if kinetic_only else p * diagonal[irot]
        if kinetic_only or n_pot == 0:
            return
        chi = spec[:nzpot].reshape(-1)
        psi[:, ichn, :n_pot] += g["specular_to_scattering"][:, None] * (rot_pot[ichn] * chi)[None, :]
        for ixy in range(n_xy):
            angular(ixy)
        chi = (psi[:, ichn, :n_pot] * g["scattering_to_specular"][:, None]).sum(0)
        spec[:nzpot] = chi.reshape(nzpot, nr)
        psi[:, ichn, :n_pot] -= g["specular_to_scattering"][:, None] * chi

    block(True, False)
    for _ in range(c["steps"] - 1):
        block(False, False)
    block(True, True)
    plane = psi[:, :, t["iz_analysis"] * nr:(t["iz_analysis"] + 1) * nr]
    n_ana, n_dif, n_v = len(t["rotation_index"]), len(t["diffraction_slot"]), t["n_v"]
    shifted = plane[:, g["rotation_index"].long()] * g["shift_forward"][:, None, None]
    bk = torch.empty((n_v, n_ana, n_dif), device="cuda", dtype=torch.complex128)
    for v in range(n_v):
        overlap = (shifted * g["radial_weight"][v][None]).sum(2)
        channels = torch.fft.fft2(overlap.reshape(nx, nx, n_ana), dim=(0, 1)).reshape(n_xy, n_ana)
        bk[v] = channels[g["diffraction_slot"].long()].t() * t["xy_scale"]
    initial = int(np.flatnonzero(t["rotation_index"] == ichn)[0])
    bk[:, initial, 0] = (g["initial_radial"] * spec[t["iz_specular"]]).sum(1) * t["dr"]
    out = {"bk": bk.reshape(n_v, -1).cpu().numpy(), "specular": spec.cpu().numpy()}
    if c.get("read") == "wave":
        out["wave"] = psi.permute(2, 0, 1).contiguous().cpu().numpy()
    else:
        out["densities"] = sum(p.abs().square().sum(0) for p in psi).cpu().numpy()
        out["plane"] = plane.permute(2, 0, 1).contiguous().cpu().numpy()
    return out


def unpack(p):
    cut = np.cumsum([6 * 128, 128, 128 * 128, 128, 128 * 128, 128, 128])
    shapes = ((6, 128), (128,), (128, 128), (128,), (128, 128), (128,), (128, 1), (1,))
    return [a.reshape(s) for a, s in zip(torch.tensor_split(p, [int(k) for k in cut]), shapes)]


def forward(p, x):
    w1, b1, w2, b2, w3, b3, w4, b4 = unpack(p)
    h = torch.nn.functional.silu(x @ w1 + b1)
    h = torch.nn.functional.silu(h @ w2 + b2)
    h = torch.nn.functional.silu(h @ w3 + b3)
    return (h @ w4 + b4)[:, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return exact_step(case, seed)
    if kind == "batch":
        return [exact_step(m, seed + 7919 * k) for k, m in enumerate(members(case))]
    if kind in ("crp", "scm"):
        return None  # a spline library of its own
    rng = np.random.default_rng(seed)
    p = _cuda(network(rng).astype(np.float64))
    if kind == "predict":
        x, _ = samples(rng, case["rows"])
        return forward(p, _cuda(x.astype(np.float64))).cpu().numpy()
    b = case["batch"]
    n = case["rows"] // b * b
    x, t = (_cuda(a.astype(np.float64)) for a in samples(rng, n))
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    for k in range(case["steps"]):
        at = k * b % n
        q = p.clone().requires_grad_(True)
        loss = (forward(q, x[at:at + b]) - t[at:at + b]).square().mean()
        grad, = torch.autograd.grad(loss, q)
        losses.append(float(loss.detach()))
        m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad * grad
        p = p - 1e-3 * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return {"losses": np.array(losses), "params": p.cpu().numpy()}
