"""Paths of the kernels that ordinary inputs seldom or never take: long walks with skipped runs,
scratch that the device refuses, the finest grids, values at the limits of the FP32 form, faces
that just reach vacuum.  Each is compared with the general path bit for bit, or with the oracle.
"""
import numpy as np
import pytest

from gizmo_amd import ics
from gizmo_amd.batch import Batch
from gizmo_amd.hydro import GZ_FP32_MIXED, GZ_FP64, GizmoHipError, Hydro

pytestmark = pytest.mark.gpu

BOTH = pytest.mark.parametrize("precision", [GZ_FP64, GZ_FP32_MIXED], ids=["fp64", "mixed"])
DENSITY_OUT = ("h", "numngb", "rho", "press", "nvt", "nvt_fw", "cn", "fce", "drkern", "divvel")


def params(**kw):
    p = dict(box=1.0, kernel=6, gamma=5.0 / 3.0, des_num_ngb=64.0, max_num_ngb_dev=0.1, min_kernel_radius=0.0,
             max_kernel_radius=0.25, time=0.0, time_begin=0.0)
    p.update(kw)
    return p


INTEG = dict(courant_fac=0.2, err_tol_int_accuracy=0.02, max_size_timestep=0.01, min_size_timestep=0.0, time_begin=0.0, time_max=1.0,
             min_egy_spec=0.0)
FORCE_OUT = ("accel", "dtu", "maxsig", "wakeup")


def streams(side, mach, seed):
    """Gas streams that collide at x = 1/2 and part at x = 0: many faces past the Riemann ladder's
    common case."""
    ic = ics.lattice_box(side, seed, kernel=6, des_num_ngb=64.0, mach_sigma=0.3)
    cs = np.sqrt(ic["params"]["gamma"])
    ic["vel"][:, 0] += np.where(ic["pos"][:, 0] < 0.5, mach, -mach) * cs
    return ic


def loaded(ic, precision, capacity=None, **options):
    g = Hydro(dict(ic["params"]), capacity or len(ic["mass"]), precision)
    for k, v in options.items():
        g.set_option(k, v)
    g.load({k: ic[k] for k in ("pos", "vel", "mass", "u", "h")})
    return g


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


@BOTH
@pytest.mark.parametrize("room,spare", [(1e18, 1), (0, 1), (0, 8), (100000, 1), (2e6, 1)])
def test_force_pass_with_less_room(room, spare, precision):
    """The force pass over many rows without its scratch (the device refuses 10^18 bytes; none allowed)
    or with less of it: the density sums' room and short segments.  Against whole segments, twice
    (the refusal must not reach a later launch check), and against the row kernels."""
    ic = streams(15, 5.0, 43)
    n = len(ic["mass"])
    out = {}
    for name, options in (("whole", dict(few_rows=0)), ("less", dict(few_rows=0, force_room=room)), ("rows", dict(few_rows=10 ** 9))):
        print(f"force room: {name} room={room} spare={spare} n={n} precision={precision}", flush=True)
        g = loaded(ic, precision, spare * n, **options)
        g.hydro_pass()
        g.hydro_pass()
        assert name == "rows" or g.stat("force_rare_rows") > 0
        out[name] = g.store(FORCE_OUT)
        g.close()
    same_bits(out["less"], out["whole"])
    same_bits(out["rows"], out["whole"])


def test_force_pass_without_any_room_is_refused():
    """So few particles that even the density sums hold less than an entry for each workgroup."""
    rng = np.random.Generator(np.random.Philox(44))
    n = 100
    ic = dict(pos=rng.random((n, 3)), vel=rng.normal(size=(n, 3)), mass=np.full(n, 1.0 / n), u=np.ones(n), h=np.full(n, 0.2))
    f = dict(ic, rho=np.ones(n), press=np.full(n, 2.0 / 3.0), numngb=np.full(n, 4.0), drkern=np.ones(n), divvel=np.zeros(n), cn=np.ones(n),
             fce=np.zeros(n), nvt=np.tile([100.0, 100.0, 100.0, 0.0, 0.0, 0.0], (n, 1)), grad_rho=np.zeros((n, 3)), grad_p=np.zeros((n, 3)),
             grad_v=np.zeros((n, 9)))
    for room in (0, -1):
        print(f"no room: n={n} force_room={room}", flush=True)
        g = Hydro(params(), n, GZ_FP64)
        g.set_option("few_rows", 0)
        g.set_option("force_room", room)
        g.load(f)
        if room == 0:
            with pytest.raises(GizmoHipError, match="no room"):
                g.hydro_force()
        else:
            g.hydro_force()
            assert np.isfinite(g.store(["accel"])["accel"]).all()
        g.close()


@BOTH
def test_batch_with_less_room(precision):
    boxes = [streams(s, 3.0, 45 + s) for s in (11, 14)]
    out = {}
    for room in (-1, 1e18, 0):
        b = Batch(dict(boxes[0]["params"]), sum(len(ic["mass"]) for ic in boxes), 2, precision)
        b.set_option("few_rows", 0)
        b.set_option("force_room", room)
        ids = [b.add({k: ic[k] for k in ("pos", "vel", "mass", "u", "h")}, ic["params"], INTEG) for ic in boxes]
        print(f"batch room: {room} precision={precision}", flush=True)
        b.begin()
        for _ in range(2):
            b.step()
        out[room] = [b.store(i, ("h", "rho", "accel", "dtu")) for i in ids]
        b.close()
    for room in (1e18, 0):
        for x, y in zip(out[room], out[-1]):
            same_bits(x, y)


@BOTH
def test_batch_later_rounds_walk_and_by_row(precision):
    """A batch whose second density round keeps so many rows that its groups are walked again, and whose
    later rounds then take the rest by row, against the pass that takes every round by row."""
    rng = np.random.Generator(np.random.Philox(47))
    boxes = [ics.lattice_box(s, 50 + s, kernel=6, des_num_ngb=64.0, mach_sigma=0.5) for s in (31, 47)]
    for ic in boxes:  # nearly every radius needs a second round, some need more
        ic["h"] = ic["h"] * rng.uniform(0.85, 1.15, len(ic["h"]))
    out = {}
    for few_rows in (0, 10 ** 9):
        b = Batch(dict(boxes[0]["params"]), sum(len(ic["mass"]) for ic in boxes), 2, precision)
        b.set_option("few_rows", few_rows)
        ids = [b.add({k: ic[k] for k in ("pos", "vel", "mass", "u", "h")}, ic["params"], INTEG) for ic in boxes]
        print(f"batch later rounds: few_rows={few_rows} precision={precision}", flush=True)
        b.begin()
        b.step()
        out[few_rows] = [b.store(i, ("h", "rho", "numngb", "accel", "dtu")) for i in ids]
        print(f"rounds: {b.stat('density_iterations'):.0f}", flush=True)
        b.close()
    for x, y in zip(out[0], out[10 ** 9]):
        same_bits(x, y)


@BOTH
def test_rarefactions_that_just_reach_vacuum(oracle_lib, precision):
    """Two streams that part at exactly the speed at which their rarefactions reach vacuum: the exact
    solver's first pressure is 0, where a rarefaction's slope is infinite and the pressure stays 0
    (gamma = 3, with which every quantity of the state is exact in both forms)."""
    c = np.zeros((2, 24))
    c[:, 0:2] = c[:, 5:7] = [1.0, 3.0]
    c[:, 2], c[:, 7] = [-3.0, -2.5], [3.0, 3.5]  # sound speed 3 on both sides
    c[:, 10] = 1.0
    c[:, 14:16], c[:, 16:18] = 3.0, 1.0
    c[:, 18], c[:, 21] = c[:, 7], c[:, 2]
    for mode in (4, 1, 0) if precision == GZ_FP64 else (4,):
        print(f"vacuum edge: mode={mode} precision={precision}", flush=True)
        g = Hydro(params(gamma=3.0), 16, precision)
        dev, rung = g.riemann_probe(mode, c)
        g.close()
        ora, want = oracle_lib.riemann_probe(mode, 3.0, c)
        assert np.array_equal(dev, ora) and np.array_equal(rung, want), (mode, dev, ora)
        if mode == 4:
            assert (ora[:, 0] == 0).all() and np.array_equal(ora[:, 1], [0.0, 0.5])


@BOTH
@pytest.mark.parametrize("side", [11, 21], ids=["four_cells", "eight_cells"])
@pytest.mark.parametrize("scale", [1.0, 1e-46], ids=["unit", "below_fp32"])
def test_retired_and_light_particles_in_the_cell_walk(side, scale, precision):
    """Partners are the particles of positive mass: retired ones (mass 0, or below) are none, and ones
    whose mass rounds to 0 in the FP32 form count as neighbours all the same.  The cell walk against
    the row kernels."""
    ic = ics.lattice_box(side, 48, kernel=6, des_num_ngb=64.0, mach_sigma=0.3)
    rng = np.random.Generator(np.random.Philox(49))
    n = len(ic["mass"])
    ic["mass"] = np.where(rng.random(n) < 0.1, rng.choice([0.0, -1.0, -1e-300], n), ic["mass"] * scale)
    out = {}
    for few_rows in (0, 10 ** 9):
        print(f"light particles: n={n} scale={scale} few_rows={few_rows} precision={precision}", flush=True)
        g = loaded(ic, precision, few_rows=few_rows)
        g.density()
        out[few_rows] = g.store(DENSITY_OUT)
        g.close()
    assert abs(np.median(out[0]["numngb"][ic["mass"] > 0]) ** 3 - 64.0) < 1.0  # (kept as the cube root of the number)
    same_bits(out[0], out[10 ** 9])


@pytest.mark.parametrize("ncoarse", [700, 767, 768, 769, 1500])
def test_groups_with_many_coarse_partners(oracle_lib, ncoarse):
    """The symmetric list of a tight clump inside the radii of ncoarse particles of three coarser
    levels: collected and merged up to 768 of them, inserted into the finished rows one by one
    beyond.  Groups of rows against one wavefront per row, and the sets against the oracle's."""
    rng = np.random.Generator(np.random.Philox(50))
    clump = 0.4 + rng.uniform(-0.004, 0.004, (150, 3))
    away = rng.normal(size=(ncoarse, 3))
    away *= (rng.uniform(0.03, 0.11, ncoarse) / np.linalg.norm(away, axis=1))[:, None]
    pos = np.concatenate((clump, 0.4 + away))
    h = np.concatenate((np.full(150, 0.003), rng.choice([0.125, 0.2, 0.24], ncoarse)))
    n = len(pos)
    lists = {}
    for few_rows in (0, 10 ** 9):
        print(f"coarse partners: n={n} few_rows={few_rows}", flush=True)
        g = loaded(dict(params=params(), pos=pos, vel=np.zeros((n, 3)), mass=np.ones(n), u=np.ones(n), h=h), GZ_FP64, wide_search=1,
                   few_rows=few_rows)
        lists[few_rows] = g.neighbors(1)
        g.close()
    for a, b in zip(lists[0], lists[10 ** 9]):
        assert np.array_equal(a, b)
    off, nbr = lists[0]
    assert (np.diff(off)[:150] >= ncoarse).all()
    ref_off, ref = oracle_lib.neighbors(params(), pos, h, 1)
    assert np.array_equal(off, ref_off)
    for i in range(n):
        assert np.array_equal(np.sort(nbr[off[i]:off[i + 1]]), ref[off[i]:off[i + 1]]), i


def patchy(side, seed, share):
    """Quiet gas with a slab of violent motion, `share` of the box: the rows with a face past the Riemann
    ladder's common case."""
    ic = ics.lattice_box(side, seed, kernel=6, des_num_ngb=64.0, mach_sigma=0.003)
    rng = np.random.Generator(np.random.Philox(seed))
    ic["vel"][ic["pos"][:, 0] < share] += rng.normal(size=(int((ic["pos"][:, 0] < share).sum()), 3)) * 0.8
    return ic


@pytest.mark.parametrize("share,active", [(0.0, 1.0), (0.1, 1.0), (0.1, 0.95)])
def test_quiet_gas_by_lanes(share, active):
    """The FP32 form's pass over many rows of quiet gas: from the second pass on one lane per row takes the
    rows of the common case and leaves the others to the general kernel, which takes all of them
    with the option force_split at 0.  Wake-up flags, too, where some neighbours are inactive."""
    ic = patchy(59, 51, share)
    n = len(ic["mass"])
    rows = np.random.Generator(np.random.Philox(52)).random(n) < active
    out, rare = {}, {}
    for split in (0, -1, 1):
        print(f"quiet gas: n={n} share={share} active={active} force_split={split}", flush=True)
        g = loaded(ic, GZ_FP32_MIXED, force_split=split)
        for _ in range(2):
            g.hydro_pass()
        if active < 1.0:
            g.set_active(rows)
        g.timing_reset()
        g.hydro_pass()
        rare[split] = g.stat("force_rare_rows") / rows.sum()
        out[split] = g.store(FORCE_OUT)
        g.close()
    print(f"rows past the common case: {rare[-1]:.3f}", flush=True)
    # (a row has such a face only with a moving particle within reach: in the slab, or a radius from it)
    assert rare[0] == 0 and rare[-1] == rare[1] <= 0.25 and share <= rare[1] <= (share + 2 * ic["h"].max() if share else 0)
    same_bits(out[-1], out[0])
    same_bits(out[1], out[0])


def test_quiet_gas_by_lanes_in_a_batch():
    boxes = [patchy(s, 53 + s, x) for s, x in ((48, 0.0), (50, 0.1))]
    out = {}
    for few_rows in (8192, 10 ** 9):
        b = Batch(dict(boxes[0]["params"]), sum(len(ic["mass"]) for ic in boxes), 2, GZ_FP32_MIXED)
        b.set_option("few_rows", few_rows)
        ids = [b.add({k: ic[k] for k in ("pos", "vel", "mass", "u", "h")}, ic["params"], INTEG) for ic in boxes]
        print(f"quiet batch: few_rows={few_rows}", flush=True)
        b.begin()
        for _ in range(3):
            b.step()
        out[few_rows] = [b.store(i, ("h", "rho", "accel", "dtu", "vel")) for i in ids]
        b.close()
    for x, y in zip(out[8192], out[10 ** 9]):
        same_bits(x, y)


@pytest.mark.parametrize("box", [1.0, 1e-21, 3e-22, 3e24])
def test_wide_search_in_other_units(box):
    """Long walks of the search over many levels in a box of any size (FP64): the squares of distances
    lie far below and above what FP32 holds.  Against one grid, bit for bit."""
    ic = ics.lognormal_box(20000, 57, ng=32)
    s = box
    ic["params"] = dict(ic["params"], box=s, max_kernel_radius=0.25 * s)
    out = {}
    for wide in (0, 1):
        print(f"wide units: box={box} wide={wide}", flush=True)
        g = Hydro(ic["params"], len(ic["mass"]), GZ_FP64)
        g.set_option("wide_search", wide)
        g.load(dict(pos=ic["pos"] * s, vel=ic["vel"], mass=ic["mass"], u=ic["u"], h=ic["h"] * s))
        g.density()
        out[wide] = (g.store(DENSITY_OUT), g.neighbors(1))
        g.close()
    same_bits(out[1][0], out[0][0])
    for a, b in zip(out[1][1], out[0][1]):
        assert np.array_equal(a, b)
