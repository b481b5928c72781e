"""The CRP kernels at the sizes where they change: a lane, a workgroup's 64 points and one more, the last count that
takes a workgroup a CU and the first beyond it (64 x 256 points), and a corrugation function short enough for LDS or
longer. Against the host restatement, to the bar of test_gpu_crp.py (the same statements; the device's sin / cos and the
sums in runs leave a few ulp of the terms)."""

import os
import shutil

import numpy as np
import pytest

from tests.test_gpu_crp import CRP_DIR, FLOOR_EV, SCM_DIR, SCM_RUNS, TOL, _note, _points, _relative

pytestmark = pytest.mark.gpu


def _check(directory, counts, seed):
    import spodvr_amd
    s = spodvr_amd.CrpSurface(directory)
    try:
        pts = _points(s, max(counts), seed)
        host = s.qd(pts)
        for n in counts:
            _note("values of", n, "points, seed", seed)
            assert _relative(s.device_qd(pts[:n]), host[:n], FLOOR_EV) <= TOL
    finally:
        s.close()


@pytest.mark.parametrize("case", ["cu111_srp48", "c6v_pairwise", "c4v_pairwise"])
def test_point_counts(case):
    _check(os.path.join(CRP_DIR, case, "dataset"), [1, 63, 64, 65, 1000, 16384, 16385], 21)


@pytest.mark.parametrize("case", ["cu111_srp48", "c4v_pairwise"])
@pytest.mark.parametrize("knots", [128, 129, 178, 179, 400])
def test_corrugation_knots(case, knots, tmp_path):
    """The data set's corrugation function resampled to `knots` points, ends and slopes kept."""
    where = tmp_path / "dataset"
    shutil.copytree(os.path.join(CRP_DIR, case, "dataset"), where)
    table = where / "Atom" / "intrep.dat"
    lines = [line for line in table.read_text().splitlines() if line.strip()]
    count = 2  # after the slopes at both ends
    n = int(lines[count].split()[0])
    x, f = np.array([[float(v) for v in line.split()[:2]] for line in lines[count + 1:count + 1 + n]]).T
    fine = np.linspace(x[0], x[-1], knots)
    table.write_text("\n".join(lines[:count] + [str(knots)] + [f"{a:.16e} {b:.16e}" for a, b in
                                                                zip(fine, np.interp(fine, x, f))]) + "\n")
    _check(str(where), [500, 17000], 22)


@pytest.mark.parametrize("case", ["cu111_srp48", "c4v_pairwise"])
def test_a_value_does_not_depend_on_the_points_beside_it(case):
    """A geometry's value bit for bit the same alone, among few points and among many (the kernel's two workgroup
    sizes)."""
    import spodvr_amd
    s = spodvr_amd.CrpSurface(os.path.join(CRP_DIR, case, "dataset"))
    try:
        pts = _points(s, 20000, 23)
        _note("values of 20000 points and of runs of them", case)
        many = s.device_qd(pts)
        for n in (1, 65, 1000):
            assert np.array_equal(s.device_qd(pts[:n]), many[:n]), n
    finally:
        s.close()


@pytest.mark.parametrize("run", ["example/rescaling_on", "synthetic/v3_slab3_rescaling_on"])
def test_a_slab_value_does_not_depend_on_the_points_beside_it(run):
    import spodvr_amd
    f = np.load(os.path.join(SCM_DIR, run + ".npz"))
    par, slab = SCM_RUNS[run]
    s = spodvr_amd.ScmSurface(os.path.join(CRP_DIR, "cu111_srp48", "dataset"), os.path.join(SCM_DIR, par),
                              os.path.join(SCM_DIR, slab), int(f["slab_number"]), float(f["cutoff"]),
                              bool(f["rescaling"]))
    try:
        _note("SCM values of 20000 points and of runs of them", run)
        pts = np.resize(f["points"], (20000, 6))
        many = s.device_values(pts)
        for n in (1, 65, 1000):
            assert np.array_equal(s.device_values(pts[:n]), many[:n]), n
    finally:
        s.close()


def test_threads_with_tables_of_other_lengths():
    """Two threads, each with its own surface (corrugation functions of 46 and 5 knots, both in LDS), give bit for bit
    what each gives alone."""
    import threading
    import spodvr_amd
    surfaces = [spodvr_amd.CrpSurface(os.path.join(CRP_DIR, case, "dataset"))
                for case in ("cu111_srp48", "c3v_impulse_15")]
    try:
        points = [_points(s, 1000, 24) for s in surfaces]
        _note("values of two surfaces, one after the other, then from two threads")
        alone = [s.device_qd(p) for s, p in zip(surfaces, points)]
        assert not np.array_equal(*alone)
        same = [[], []]

        def work(k):
            for _ in range(50):
                same[k].append(np.array_equal(surfaces[k].device_qd(points[k]), alone[k]))

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert same == [[True] * 50] * 2
    finally:
        for s in surfaces:
            s.close()
