"""Every launch variant that SPO_HIP_TUNE can pick, in every list that SPO_HIP_INTERACTION leaves, on one full T block
against the CPU oracle: FP64 to the parity bar of test_gpu_parity.py (max |a - b| / max |a| < 1e-12), complex64 to
single-precision rounding (< 1e-5). The lists are walked to their ends, whatever their lengths."""

import os
import re

import numpy as np
import pytest

from tests import cases
from tests.test_gpu_grid_shapes import _grid
from tests.util import pseudo_random, relative_difference

pytestmark = pytest.mark.gpu


def _run(path, precision, tune, interaction=None):
    import spodvr_amd
    env = {"SPO_HIP_TUNE": tune, "SPO_HIP_INTERACTION": interaction, "SPO_HIP_POTENTIAL": "host"}
    saved = {k: os.environ.pop(k, None) for k in env}
    os.environ.update({k: v for k, v in env.items() if v is not None})
    try:
        return spodvr_amd.Run(path, {"Precision": precision}, device="hip")
    finally:
        for k, v in saved.items():
            os.environ.pop(k, None)
            if v is not None:
                os.environ[k] = v


def _length(path, precision, family, interaction=None):
    """The length of a family's list, from the message that refuses a place past its end (a list of one variant, or
    none, is not tuned)."""
    import spodvr_amd
    try:
        _run(path, precision, f"{family}=#100", interaction).close()
    except spodvr_amd.SpoError as e:
        return int(re.search(rf"{family} has (\d+) variants", str(e)).group(1))
    return 0


def _check(name, params, seed, family, precisions=("fp64", "mixed"), interactions=(None,), least=2):
    from oracle import oracle
    path = cases.write_case(name, params)
    cpu = oracle.run(path)
    wave = pseudo_random(cpu.scattering_size, seed), pseudo_random(cpu.specular_size, seed + 1)
    cpu.set_wave(*wave)
    cpu.kinetic_and_potential(False, False)
    want = cpu.get_wave()
    cpu.close()
    for precision in precisions:
        for interaction in interactions:
            n = _length(path, precision, family, interaction)
            print(f"{name} seed {seed} {precision} SPO_HIP_INTERACTION={interaction}: {n} {family} variants", flush=True)
            assert interaction is not None or n >= least
            for k in range(n):
                run = _run(path, precision, f"{family}=#{k}", interaction)
                run.set_wave(*wave)
                run.kinetic_and_potential(False, False)
                got = run.get_wave()
                run.close()
                ds, dp = (relative_difference(a, b) for a, b in zip(want, got))
                print(f"  #{k}: scattering {ds:.3e} specular {dp:.3e}", flush=True)
                assert np.isfinite(got[0].view(float)).all()
                tol = 1e-12 if precision == "fp64" else 1e-5
                assert ds < tol and dp < tol, (interaction, k)


# Angular bases of every phi length that these grids take up to MJMax 31 (2, 4, ... 24, 28, 30, 32, 36, 40, 42, 44, 48,
# 56, 60 and 64 points; 56 in FP64 has MFMA kernels alone), an (izr) count that fills no tile, with the MFMA and buffer
# kernels' own lists where they have one.
@pytest.mark.parametrize("jmax,mjmax,homonuclear", [
    (0, 0, True), (1, 1, False), (2, 2, True), (3, 3, False), (4, 4, True), (5, 5, False), (6, 6, True), (7, 7, False),
    (8, 8, True), (9, 9, False), (10, 10, True), (11, 11, False), (12, 12, True), (14, 14, True), (15, 15, False),
    (16, 16, True), (18, 18, True), (20, 20, True), (22, 21, True), (24, 23, True), (24, 24, True), (28, 28, True),
    (30, 30, True)])
def test_every_interaction_variant(jmax, mjmax, homonuclear):
    _check(f"var_{jmax}_{mjmax}", _grid(22, 10, 4, jmax, mjmax=mjmax, HomoNuc=homonuclear), 500 + 2 * jmax + mjmax,
           "interaction", interactions=(None, "buf", "mfma"))


# A shape of the compile-time T_Zr list and two without one (a plane that fills a CU's LDS in FP64, a small one).
@pytest.mark.parametrize("nz,nr", [(96, 32), (160, 40), (42, 18)])
def test_every_zr_variant(nz, nr):
    _check(f"varzr_{nz}_{nr}", _grid(nz, nr, 4, 2), 600 + nz + nr, "zr")


@pytest.mark.parametrize("nxy", [4, 8, 10, 12, 14, 16])
def test_every_xy_variant(nxy):
    _check(f"varxy_{nxy}", _grid(22, 10, nxy, 2), 700 + nxy, "xy")
