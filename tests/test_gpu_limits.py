"""Paths of the kernels that ordinary inputs seldom or never take: long walks with skipped runs,
scratch that the device refuses, the finest grids, values at the limits of the FP32 form, faces
that just reach vacuum.  Each is compared with the general path bit for bit, or with the oracle.
"""
import numpy as np
import pytest

from gizmo_amd.hydro import GZ_FP32_MIXED, GZ_FP64, Hydro

pytestmark = pytest.mark.gpu

BOTH = pytest.mark.parametrize("precision", [GZ_FP64, GZ_FP32_MIXED], ids=["fp64", "mixed"])
DENSITY_OUT = ("h", "numngb", "rho", "press", "nvt", "nvt_fw", "cn", "fce", "drkern", "divvel")


def params(**kw):
    p = dict(box=1.0, kernel=6, gamma=5.0 / 3.0, des_num_ngb=64.0, max_num_ngb_dev=0.1, min_kernel_radius=0.0,
             max_kernel_radius=0.25, time=0.0, time_begin=0.0)
    p.update(kw)
    return p


def same_bits(a, b, rows=slice(None)):
    for k in a:
        x, y = a[k][rows], b[k][rows]
        assert np.isfinite(x).all() and np.array_equal(x.view(np.uint8), y.view(np.uint8)), (k, int((x != y).sum()), x.size)


@BOTH
def test_long_walk_with_skipped_runs(precision):
    """A long walk's runs of 256 candidates that lie within reach and out of it in turn, with fewer
    partners between two of them than a round of sums takes: no barrier but that of the ranks then
    separates the walked runs of a row's four wavefronts.  Against one wavefront per row.

    8^3 cubes of side 1/16, each of 256 particles in its middle: consecutive in Morton order, so a run
    is a cube.  The rows sit in the middle of cubes, with a radius that reaches part of the next
    cube along an axis (and along two) and nothing of the one after that."""
    rng = np.random.Generator(np.random.Philox(41))
    side, first, cubes, per = 1.0 / 16, 4, 8, 256
    ijk = np.stack(np.meshgrid(*[np.arange(first, first + cubes)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = np.repeat((ijk + 0.5) * side, per, axis=0) + rng.uniform(-0.4, 0.4, (len(ijk) * per, 3)) * side
    rows = np.flatnonzero(((ijk >= first + 2) & (ijk < first + 6)).all(1)) * per
    pos[rows] = (ijk[rows // per] + 0.5) * side
    n = len(pos)
    active = np.zeros(n, dtype=np.uint8)
    active[rows] = 1
    out = {}
    for few_rows in (0, 10 ** 9):
        g = Hydro(params(), n, precision)
        g.set_option("wide_search", 1)
        g.set_option("few_rows", few_rows)
        g.load(dict(pos=pos, vel=np.sin(37.0 * pos), mass=np.full(n, 1.0 / n), u=np.ones(n), h=np.full(n, 0.07)))
        g.set_active(active)
        print(f"skipped runs: n={n} rows={len(rows)} few_rows={few_rows} precision={precision}", flush=True)
        g.density()
        out[few_rows] = g.store(DENSITY_OUT)
        g.close()
    same_bits(out[0], out[10 ** 9], rows)


@BOTH
def test_grid_of_512_cells_a_side(precision):
    """Many rows on the second finest grid (radii below box / 512; 134 million cells, whose stencils
    take as many threads as a launch cannot hold), against the row kernels, which find their cells
    themselves."""
    rng = np.random.Generator(np.random.Philox(42))
    side = 14
    pos = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3) * 7e-4
    pos = 0.5 + pos + rng.uniform(-1e-4, 1e-4, pos.shape)
    n = len(pos)
    out = {}
    for few_rows in (0, 10 ** 9):
        print(f"512 cells a side: n={n} few_rows={few_rows} precision={precision}", flush=True)
        g = Hydro(params(), n, precision)
        g.set_option("few_rows", few_rows)
        g.load(dict(pos=pos, vel=np.sin(900.0 * pos), mass=np.full(n, 1.0 / n), u=np.ones(n), h=np.full(n, 0.0015)))
        g.density()
        out[few_rows] = g.store(DENSITY_OUT)
        g.close()
    same_bits(out[0], out[10 ** 9])
