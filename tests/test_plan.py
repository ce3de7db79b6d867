"""The launch arithmetic (gizmo_amd/csrc/gz_plan.h), compiled with g++ and asked on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "plan_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "gizmo_amd", "csrc"),
                    os.path.join(ROOT, "tests", "plan_check.cpp"), "-o", str(exe)], check=True)

    def run(questions):
        r = subprocess.run([str(exe)], input="\n".join(" ".join(str(x) for x in q) for q in questions), capture_output=True,
                           text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        return [[float(x) for x in line.split()] for line in r.stdout.splitlines()]
    return run


def test_stencil_launch_fits_at_every_level(ask):
    """Fewer than 2^32 threads along x, which is the most that a launch takes, and a thread group per
    cell while that fits."""
    for level, (blocks,) in enumerate(ask([("stencil", 8 ** level) for level in range(11)])):
        assert 1 <= blocks and blocks * 256 < 2 ** 32
        if level <= 8:
            assert blocks == max(1, 8 ** level * 32 // 256)


@pytest.mark.parametrize("form,width", [("force32", 4), ("force64", 8)])
def test_force_plan_of_any_room(ask, form, width):
    """The stored fluxes' launch keeps within its room, takes whole eights of workgroups, and says
    segment 0 (with which the kernel would not end: the callers refuse it) exactly where the room
    does not hold an entry of 64 rows x 4 values for each of eight workgroups."""
    entry = 64 * 4 * width
    rooms = [0, 1, entry, 8 * entry - 1, 8 * entry, 8 * entry + 1, 63 * entry, 64 * entry, 100 * entry, 512 * 8 * entry - 1,
             512 * 8 * entry, 512 * 96 * entry, 2 ** 63]
    for nrows in (1, 64, 65, 121, 8193, 32768, 10 ** 9):
        whole = min(-(-nrows // 64), 512)
        for room, (blocks, segment, size) in zip(rooms, ask([(form, nrows, room) for room in rooms])):
            assert size <= room and size == blocks * segment * entry
            assert blocks % 8 == 0 and 8 <= blocks <= -(-whole // 8) * 8 and segment <= 96
            assert (segment == 0) == (room < 8 * entry), (nrows, room)


def test_few_groups_share_their_rows_out(ask):
    """Groups that leave the chip's places for wavefronts idle are taken by several workgroups each, as
    many as fit and at most eight; groups that fill them by one."""
    for ngroups, (parts,) in zip((0, 1, 511, 512, 1500, 4095, 4096, 10 ** 7), ask([("parts", g) for g in (0, 1, 511, 512, 1500, 4095, 4096, 10 ** 7)])):
        assert 1 <= parts <= 8 and (parts == 1 or parts * ngroups <= 4096)
        assert parts == 8 or (parts + 1) * ngroups > 4096


# Later density rounds of batches as measured on the MI355X (FP32 form, then FP64, then mixtures of
# boxes): the boxes (count x particles / cells), the groups, the rows still iterating, microseconds of
# the walk and by row
ROUNDS = [
    ("24x8000/64", 1142, 34573, 150, 116),
    ("24x8000/64", 1336, 90389, 217, 260),
    ("3x10648/512 21x10648/64", 1669, 33965, 411, 126),
    ("7x10648/512 17x10648/64", 4016, 120472, 493, 387),
    ("5x13824/512 15x13824/64", 1650, 15555, 459, 81),
    ("12x13824/512 8x13824/64", 6656, 171327, 743, 530),
    ("12x21952/512", 4863, 34589, 184, 85),
    ("12x21952/512", 6144, 164142, 225, 330),
    ("10x32768/512", 3629, 74692, 167, 168),
    ("10x32768/512", 3595, 135111, 202, 295),
    ("8x46656/512", 2436, 46512, 280, 136),
    ("8x46656/512", 3629, 183604, 326, 465),
    ("6x59319/512", 1841, 22617, 173, 76),
    ("6x59319/512", 3072, 192438, 298, 537),
    ("2x91125/4096 4x91125/512", 6309, 72441, 761, 268),
    ("3x91125/512 3x91125/4096", 13354, 249613, 1390, 798),
    ("6x140608/4096", 20006, 105506, 591, 226),
    ("5x140608/4096 1x140608/512", 20992, 475775, 1927, 1782),
    ("8x262144/4096", 24950, 404623, 822, 942),
    ("8x262144/4096", 16490, 539596, 755, 1267),
    ("4x512000/4096", 10022, 89923, 787, 315),
    ("4x512000/4096", 16384, 1014366, 1386, 2936),
    ("4x1000000/32768", 111269, 556076, 3153, 1248),
    ("3x1000000/32768 1x1000000/4096", 102400, 2037913, 9305, 8544),
    ("2x2097152/32768", 35048, 496640, 1134, 1200),
    ("2x2097152/32768", 65536, 1685263, 2202, 4093),
    ("5x13824/512 15x13824/64", 1650, 15554, 446, 107),
    ("12x13824/512 8x13824/64", 6656, 171327, 776, 757),
    ("8x46656/512", 2436, 46507, 322, 191),
    ("8x46656/512", 3629, 183606, 412, 684),
    ("8x262144/4096", 24950, 404623, 1097, 1380),
    ("8x262144/4096", 16490, 539582, 989, 1784),
    ("4x1000000/32768", 111269, 556046, 4336, 1875),
    ("3x1000000/32768 1x1000000/4096", 102400, 2037926, 12072, 12461),
    ("1x32768/512 1x42875/512 1x54872/512 2x636056/4096 1x300763/4096", 9752, 666810, 1466, 2202),
    ("1x32768/512 1x42875/512 1x54872/512 2x636056/4096 1x300763/4096", 7973, 230986, 641, 523),
    ("1x456533/4096 1x804357/4096 1x1157625/32768 1x493039/4096", 45056, 1892330, 4857, 7279),
    ("1x456533/4096 1x804357/32768 1x1157625/4096 1x493039/4096", 13106, 81387, 1007, 389),
    ("1x166375/4096 1x205379/4096 1x262144/4096 1x148877/4096 1x636056/4096 1x681472/4096", 24576, 1320940, 4695, 5818),
    ("1x166375/4096 1x205379/4096 1x262144/4096 1x148877/4096 1x636056/4096 1x681472/4096", 18956, 129162, 800, 630),
]


def test_later_density_rounds_take_no_slower_way(ask):
    """The way that the rule takes costs at most a tenth more than the walk of any measured round, and
    all of them together at most a twentieth more than the faster ways."""
    questions = []
    for boxes, groups, remaining, _, _ in ROUNDS:
        kinds = [k.replace("/", "x").split("x") for k in boxes.split()]
        questions.append(["by_row", groups, remaining, len(kinds)] + [x for k in kinds for x in k])
    taken = [row if by_row else walk for (_, _, _, walk, row), (by_row, _) in zip(ROUNDS, ask(questions))]
    for r, t in zip(ROUNDS, taken):
        assert t <= 1.1 * r[3], r
    assert sum(taken) <= 1.05 * sum(min(r[3:]) for r in ROUNDS)


def test_particles_per_cell_of_the_fullest_eighth(ask):
    """Weighted by cells: one small box of full cells among large ones does not set it, half of the
    boxes do; no boxes and boxes of one cell are answered too."""
    got = [a[1] for a in ask([("by_row", 1, 1, 2, 1, 1728, 8, 1, 16384, 512), ("by_row", 1, 1, 2, 2, 1000000, 32768, 2, 1000000, 4096),
                              ("by_row", 1, 1, 1, 3, 50, 1), ("by_row", 1, 1, 0), ("by_row", 1, 1, 1, 1, 0, 1)])]
    want = [(8 * 216 + 57 * 32) / 65, (8192 * 1e6 / 4096 + 1024 * 1e6 / 32768) / 9216, 50, 0, 0]
    assert got == pytest.approx(want, rel=1e-12)


# The FP32 form's force pass as measured on the MI355X: rows, the share of them with a face past the
# Riemann ladder's common case, the evenness of the lists, microseconds of the general kernel alone
# and behind one lane per row
PASSES = [(140608, 0, 0.92, 403, 362), (140608, 0.0004, 0.92, 413, 463), (140608, 0.2374, 0.92, 509, 607), (262144, 0, 0.92, 598, 473),
          (262144, 0, 0.92, 687, 456), (262144, 0.0187, 0.92, 805, 564), (262144, 0.2377, 0.92, 880, 715), (262144, 0.7338, 0.92, 933, 1177),
          (512000, 0, 0.92, 1387, 920), (512000, 0.0983, 0.92, 1719, 1142), (1030301, 0.2388, 0.92, 3541, 2689),
          (1030301, 0.7333, 0.92, 3732, 4408), (2097152, 0, 0.93, 4744, 3319), (2097152, 0, 0.92, 5542, 3407), (2097152, 0.0006, 0.92, 5591, 3522),
          (2097152, 0.1631, 0.92, 6972, 4656), (2097152, 0.7333, 0.92, 7491, 8775), (512000, 0, 0.7926, 1427, 943), (512000, 0, 0.709, 1196, 1369),
          (250000, 0, 0.6675, 657, 864), (250000, 0, 0.5226, 1079, 2107), (600000, 0.1109, 0.5482, 2489, 3684), (572550, 0, 0.9535, 1450, 1241),
          (1000000, 0.0042, 0.5256, 3087, 4021), (4194304, 0.2007, 0.5391, 14793, 15294), (4194304, 0, 0.5391, 11527, 11343),
          (515150, 0, 0.9237, 1505, 1195), (257575, 0, 0.9236, 784, 784), (257575, 0.1622, 0.9236, 985, 1007)]


def test_quiet_force_passes_go_by_lanes(ask):
    """At most a tenth and 50 us more than the faster way of every measured pass."""
    for (rows, share, even, general, lanes), (by_lanes,) in zip(PASSES, ask([("lanes", *p[:3]) for p in PASSES])):
        assert (lanes if by_lanes else general) <= 1.1 * min(general, lanes) + 50, (rows, share, even)
