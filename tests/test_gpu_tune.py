"""SPO_HIP_TUNE=auto: a run whose launch variants were timed at its set-up starts from the same waves as any other and
gives its results to rounding. Every test prints its case before touching the GPU."""

import os

import numpy as np
import pytest

from tests import cases
from tests.util import relative_difference

pytestmark = pytest.mark.gpu

# dz_angular: the in-place interaction kernels, then the MFMA (FP64) or buffer ones (complex64), in the list.
CASES = {
    "dz_angular": lambda: cases.write_case("dz_angular", cases.DZ_ANGULAR),
    "smoke": lambda: cases.write_case("smoke_dailight", cases.SMOKE_DAILIGHT),
}


def _run(case, precision, tune=None, **overrides):
    import spodvr_amd
    print(f"case {case} {precision} SPO_HIP_TUNE={tune} {overrides}", flush=True)
    env = {"SPO_HIP_TUNE": tune, "SPO_HIP_TUNE_LOG": "1"}
    saved = {k: os.environ.pop(k, None) for k in env}
    os.environ.update({k: v for k, v in env.items() if v is not None})
    try:
        return spodvr_amd.Run(CASES[case](), dict(overrides, Precision=precision), device="hip")
    finally:
        for k, v in saved.items():
            os.environ.pop(k, None)
            if v is not None:
                os.environ[k] = v


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_tuned_run_starts_from_an_empty_scattering_wave(case, precision):
    """The specular wave as in an untuned run, bit for bit, and no scattering wave; three analysis steps then give the
    untuned run's BK records to the variants' rounding (FP64 1e-12, complex64 1e-5 of the largest)."""
    plain = _run(case, precision)
    try:
        scattering, specular = plain.get_wave()
        assert not scattering.any() and specular.any()
        plain.steps(3)
        want = plain.bk_records()
        assert plain.get_wave()[0].any()
    finally:
        plain.close()
    for again in range(2):  # the second finds its variants timed
        tuned = _run(case, precision, "auto")
        try:
            scattering, tuned_specular = tuned.get_wave()
            assert not scattering.any(), again
            assert np.array_equal(tuned_specular, specular)
            tuned.steps(3)
            assert relative_difference(want, tuned.bk_records()) < (1e-12 if precision == "fp64" else 1e-5)
        finally:
            tuned.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_variants_are_timed_for_each_shape_and_list(precision, capfd):
    """A choice is reused by a run of the same shape with the same variants to choose from, and by no other: not where
    the interaction region is shorter, nor where SPO_HIP_INTERACTION leaves some kernels out of the list."""
    def timed(**overrides):
        capfd.readouterr()
        run = _run("dz_angular", precision, "auto", **overrides)
        try:
            assert np.isfinite(run.bk_records()).all()
            run.propagate()
            assert np.isfinite(run.get_wave()[0]).all()
        finally:
            run.close()
        return sorted(line.split()[2].split(":")[0] for line in capfd.readouterr().err.splitlines()
                      if line.startswith("spo_hip tune"))

    # regions of their own, which no other test of this process has timed
    first = {"ZmaxSwitch": 7.3}
    assert "interaction" in timed(**first)
    assert timed(**first) == []
    assert "interaction" in timed(ZmaxSwitch=6.3)
    os.environ["SPO_HIP_INTERACTION"] = "mfma"
    try:
        assert timed(**first) == ["interaction"]
        assert timed(**first) == []
    finally:
        os.environ.pop("SPO_HIP_INTERACTION", None)
    assert timed(**first) == []
