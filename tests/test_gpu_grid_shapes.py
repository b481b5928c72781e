"""Grids of every kind of shape against the CPU oracle on one full T block: the radices of the T_Zr passes, the (x, y)
line lengths and the angular bases for which the kernels choose between their paths. FP64 to the parity bar of
test_gpu_parity.py (max |a - b| / max |a| < 1e-12), complex64 to single-precision rounding (< 1e-5)."""

import os

import numpy as np
import pytest

from tests import cases
from tests.util import pseudo_random, relative_difference

pytestmark = pytest.mark.gpu


def _grid(nz, nr, nxy, jmax, **more):
    """SMOKE_DAILIGHT on another grid of the same extent, its absorbers ending at the last grid points."""
    dz, dr = 10.08 / (nz - 1), 4.5 / (nr - 1)
    nzsp = 2 * nz
    return dict(cases.SMOKE_DAILIGHT, Title=f"{nz} x {nr} x {nxy} x {nxy}, JMax {jmax}", nZ=nz, dZ=dz,
                nR=nr, dR=dr, nX=nxy, nY=nxy, JMax=jmax, MJMax=more.pop("mjmax", jmax), nZSpecular=nzsp, ZOptEnd=-1.0 + dz * (nz - 1),
                ROptEnd=0.8 + dr * (nr - 1), ZSpOptEnd=-1.0 + dz * (nzsp - 1), **more)


def _check(name, params, seed, precisions=("fp64", "mixed"), blocks=((False, False),)):
    import spodvr_amd
    from oracle import oracle
    path = cases.write_case(name, params)
    cpu = oracle.run(path)
    scattering, specular = pseudo_random(cpu.scattering_size, seed), pseudo_random(cpu.specular_size, seed + 1)
    for half, kinetic_only in blocks:
        cpu.set_wave(scattering, specular)
        cpu.kinetic_and_potential(half, kinetic_only)
        want = cpu.get_wave()
        for precision in precisions:
            print(f"{name} seed {seed} {precision} half {half} kinetic_only {kinetic_only}", flush=True)
            os.environ["SPO_HIP_POTENTIAL"] = "host"
            try:
                gpu = spodvr_amd.Run(path, {"Precision": precision}, device="hip")
            finally:
                os.environ.pop("SPO_HIP_POTENTIAL", None)
            gpu.set_wave(scattering, specular)
            gpu.kinetic_and_potential(half, kinetic_only)
            got = gpu.get_wave()
            gpu.close()
            ds, dp = (relative_difference(a, b) for a, b in zip(want, got))
            print(f"  scattering {ds:.3e} specular {dp:.3e}", flush=True)
            assert np.isfinite(got[0].view(float)).all()
            assert ds < (1e-12 if precision == "fp64" else 1e-5) and dp < (1e-12 if precision == "fp64" else 1e-5)
    cpu.close()


# (NZ, NR): a prime radix alone (22 = 2 x 11), every radix up to 16 in each pass, axes of one radix and of two equal
# ones, a length that is no product of two radices (the run-time engine), and a plane that fills a CU's LDS in FP64.
@pytest.mark.parametrize("nz,nr", [(66, 12), (110, 14), (126, 22), (80, 30), (144, 18), (210, 20), (128, 56),
                                   (112, 36), (160, 40), (192, 16), (264, 12), (132, 64)])
def test_zr_plane_shapes(nz, nr):
    _check(f"zr_{nz}_{nr}", _grid(nz, nr, 4, 2), 100 + nz + nr, blocks=((False, False), (True, True)))


# Planes beyond the in-place kernel in FP64: 160 x 64 fits a CU's LDS only without the padding of its rows (the run-time
# engine on the plane), 176 x 64 does not fit at all (line transforms). In complex64 both are in place.
@pytest.mark.parametrize("nz,nr", [(160, 64), (176, 64)])
def test_zr_planes_beyond_the_in_place_kernel(nz, nr):
    _check(f"zr_{nz}_{nr}", _grid(nz, nr, 4, 2), 100 + nz + nr, blocks=((False, False), (True, True)))


# Specular grids (NZSpecular, NR) on both sides of each choice: in one launch, with small radices and with 18, 20 and 22
# along Z, before the scattering wave's step (up to 5120 points) and beside it; no product of two radices (420), and
# more points than a CU's LDS holds (360 x 36), which take the line transforms.
@pytest.mark.parametrize("nzsp,nr", [(30, 10), (198, 12), (360, 12), (396, 12), (440, 12), (308, 24), (420, 12), (360, 36)])
def test_specular_grids(nzsp, nr):
    p = _grid(22, nr, 4, 2)
    p.update(Title=f"specular {nzsp} x {nr}", nZSpecular=nzsp, ZSpOptEnd=-1.0 + p["dZ"] * (nzsp - 1))
    _check(f"sp_{nzsp}_{nr}", p, 400 + nzsp + nr, blocks=((False, False), (True, True)))


# Every (x, y) line length of the register kernel, with izr counts that leave a partial tile, and one beyond it.
@pytest.mark.parametrize("nxy", [2, 6, 10, 12, 14, 18])
@pytest.mark.parametrize("nz,nr", [(22, 10), (28, 12)])
def test_xy_line_lengths(nxy, nz, nr):
    _check(f"xy_{nxy}_{nz}_{nr}", _grid(nz, nr, nxy, 2), 200 + nxy + nz, blocks=((False, False), (True, True)))


# Angular bases for every phi length with a kernel of its own (JMax, MJMax, two equal atoms), the longest block that it
# takes (16 J), one J more (another kernel), and truncated mJ.
@pytest.mark.parametrize("jmax,mjmax,homonuclear", [
    (0, 0, True), (1, 1, False), (2, 2, True), (3, 3, False), (4, 4, True), (5, 5, False), (6, 6, True), (7, 7, False),
    (8, 8, True), (9, 9, False), (10, 10, True), (11, 11, False), (12, 12, True), (14, 14, True), (15, 15, False),
    (16, 16, True), (16, 16, False), (18, 18, True), (20, 20, True), (22, 20, True), (22, 22, True), (24, 23, True),
    (24, 24, True), (28, 28, True), (30, 30, True), (12, 3, False), (24, 2, True)])
@pytest.mark.parametrize("sym", [False, True])
def test_angular_bases(jmax, mjmax, homonuclear, sym):
    _check(f"ang_{jmax}_{mjmax}_{homonuclear}_{sym}",
           _grid(22, 10, 4, jmax, mjmax=mjmax, HomoNuc=homonuclear, UseSymmetry=sym), 300 + 2 * jmax + mjmax)
