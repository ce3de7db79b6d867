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
