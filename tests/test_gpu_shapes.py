"""The kernels of passes over many rows (cell walks, one lane per row) against the row kernels
(a workgroup per row), at the sizes where their tiles, windows and queues can go wrong: grids of
2-4 cells a side (no relative coordinates), cells of more than 64 rows, candidate counts that are
no multiple of a tile, radii far below the cell side, partly active rows, strong shocks (every
rung of the Riemann ladder).

Both shapes add each row's terms in ascending partner order, so every field agrees bit for bit,
in both arithmetic forms; the row kernels are held to the oracle in test_gpu_parity.py and
test_gpu_riemann.py.
"""
import numpy as np
import pytest

from gizmo_amd import ics
from gizmo_amd.batch import Batch
from gizmo_amd.hydro import GZ_FP32_MIXED, GZ_FP64, Hydro

pytestmark = pytest.mark.gpu

FIELDS = ("h", "numngb", "rho", "press", "nvt", "nvt_fw", "cn", "fce", "drkern", "divvel", "grad_rho", "grad_p", "grad_v",
          "accel", "dtu", "maxsig", "wakeup")

BOXES = {
    "two_cells": lambda: ics.lattice_box(8, 21, kernel=3, des_num_ngb=32.0, mach_sigma=0.3),
    "four_cells": lambda: ics.lattice_box(13, 22, kernel=6, des_num_ngb=64.0, mach_sigma=1.0),
    "eight_cells": lambda: ics.lattice_box(21, 23, kernel=6, des_num_ngb=64.0, mach_sigma=2.0),
    "odd": lambda: ics.lattice_box(27, 24, kernel=3, des_num_ngb=32.0, mach_sigma=0.2),
    # one grid sized by the largest radius: dense cells of hundreds of rows with radii of a
    # fraction of the cell
    "clustered": lambda: ics.lognormal_box(6000, 25, ng=16),
    "blast": lambda: ics.sedov_box(18, 26, kernel=6, des_num_ngb=64.0),
}


def run(ic, few_rows, precision, active, fd, wide=False):
    g = Hydro(dict(ic["params"]), len(ic["mass"]), precision)
    if wide:
        g.set_option("wide_search", 1)
    g.set_option("few_rows", few_rows)
    if fd:
        g.set_option("fd_correction", 1)
    g.load({k: ic[k] for k in ("pos", "vel", "mass", "u", "h")})
    g.hydro_pass()
    if active < 1.0:
        rng = np.random.Generator(np.random.Philox(7))
        g.set_active(rng.random(len(ic["mass"])) < active)
        g.hydro_pass()
    out = g.store(FIELDS)
    g.close()
    return out


@pytest.mark.parametrize("precision", [GZ_FP64, GZ_FP32_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name,active,fd", [("two_cells", 1.0, False), ("four_cells", 0.3, False), ("eight_cells", 1.0, True),
                                            ("eight_cells", 0.05, False), ("odd", 1.0, False), ("clustered", 1.0, False),
                                            ("clustered", 0.4, False), ("blast", 1.0, False)])
def test_many_rows_equal_row_kernels(name, active, fd, precision):
    ic = BOXES[name]()
    print(f"shapes: {name} n={len(ic['mass'])} active={active} fd={fd} precision={precision}", flush=True)
    a = run(ic, 0, precision, active, fd)
    b = run(ic, 10 ** 9, precision, active, fd)
    for k in FIELDS:
        same = a[k].view(np.int64 if a[k].dtype == np.float64 else a[k].dtype) == b[k].view(np.int64 if b[k].dtype == np.float64 else b[k].dtype)
        assert np.isfinite(a[k]).all() and same.all(), (k, int((~same).sum()), same.size)


@pytest.mark.parametrize("precision", [GZ_FP64, GZ_FP32_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name,active", [("two_cells", 1.0), ("four_cells", 0.3), ("eight_cells", 1.0), ("clustered", 1.0), ("clustered", 0.4),
                                         ("blast", 1.0)])
def test_groups_of_many_levels_equal_row_kernels(name, active, precision):
    """The symmetric list of the search over many levels, by groups of rows and row by row: coarse
    levels (2 and 4 cells a side, where differences wrap), long walks, particles of coarser levels."""
    ic = BOXES[name]()
    print(f"levels: {name} n={len(ic['mass'])} active={active} precision={precision}", flush=True)
    a = run(ic, 0, precision, active, False, wide=True)
    b = run(ic, 10 ** 9, precision, active, False, wide=True)
    for k in FIELDS:
        same = a[k].view(np.int64 if a[k].dtype == np.float64 else a[k].dtype) == b[k].view(np.int64 if b[k].dtype == np.float64 else b[k].dtype)
        assert np.isfinite(a[k]).all() and same.all(), (k, int((~same).sum()), same.size)


INTEG = dict(courant_fac=0.2, err_tol_int_accuracy=0.02, max_size_timestep=0.01, min_size_timestep=0.0, time_begin=0.0, time_max=1.0,
             min_egy_spec=0.0)


@pytest.mark.parametrize("precision", [GZ_FP64, GZ_FP32_MIXED], ids=["fp64", "mixed"])
def test_batch_rounds_by_row_equal_cell_walks(precision):
    """A batch whose rows need different numbers of density rounds: the later rounds' few rows by row
    (one wavefront, four wavefronts each) against the pass that takes every round by row."""
    rng = np.random.Generator(np.random.Philox(11))
    boxes = [ics.lattice_box(s, 30 + s, kernel=6, des_num_ngb=64.0, mach_sigma=0.5) for s in (12, 17)]
    for ic in boxes:
        far = rng.random(len(ic["h"])) < 0.3  # radii that the rounds have to bring back
        ic["h"] = np.where(far, ic["h"] * rng.uniform(0.7, 1.3, len(ic["h"])), ic["h"])
    out = {}
    for few_rows in (10 ** 9, 0, 1500):
        b = Batch(dict(boxes[0]["params"]), sum(len(ic["mass"]) for ic in boxes), 2, precision)
        b.set_option("few_rows", few_rows)
        ids = [b.add({k: ic[k] for k in ("pos", "vel", "mass", "u", "h")}, ic["params"], INTEG) for ic in boxes]
        print(f"batch rounds: few_rows={few_rows} precision={precision}", flush=True)
        b.begin()
        for _ in range(3):
            b.step()
        out[few_rows] = [b.store(i, ("h", "rho", "numngb", "accel", "dtu")) for i in ids]
        b.close()
    for few_rows in (0, 1500):
        for x, y in zip(out[few_rows], out[10 ** 9]):
            for k in x:
                assert np.isfinite(x[k]).all() and np.array_equal(x[k], y[k]), (few_rows, k)
