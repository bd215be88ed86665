"""What the solving C entries do when memory runs out or a cooperative launch is
refused, and what they do again on a repeated call.  A compiled caller
(batch_entry.cpp) links the library's objects with a stand-in for the GPU
runtime; it makes a context by hand and runs no kernel.
"""
import os
import subprocess
from collections import namedtuple

import pytest

from pigfem_assignment_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
ENV = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1")
Call = namedtuple("Call", "status coop plain host_bytes threads_per_row")


@pytest.fixture(scope="module")
def entry(tmp_path_factory):
    objs = [os.path.join(build.OBJ, os.path.basename(s) + ".o") for s in build.HOST_SRC + build.HIP_SRC]
    assert all(os.path.exists(o) for o in objs), "the library is not built; run `python -m pigfem_assignment_amd.build`"
    out = str(tmp_path_factory.mktemp("entry") / "batch_entry")
    obj = out + ".o"
    subprocess.run([build.HIPCC, "-O1", "-std=c++17", "--offload-arch=" + build.ARCH, "--offload-host-only", "-x", "hip", "-c",
                    os.path.join(HERE, "batch_entry.cpp"), "-o", obj], check=True)
    subprocess.run([build.HIPCC, "--offload-arch=" + build.ARCH, "-o", out, obj] + objs + ["-lgomp"], check=True)
    return out


def run(exe, *args):
    r = subprocess.run([exe] + [str(a) for a in args], env=ENV, capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0, "ended with %d" % r.returncode
    return [Call(*map(int, line.split())) for line in r.stdout.splitlines()]


def test_no_device(entry):
    (c,) = run(entry, "batch", 4, 1, 1, "device")
    assert c.status == -4


# 100 kB: a thread's table of the system's columns (640 kB), in the parallel
# region; 1 MB: the steps of all shares (2.6 MB), behind it.  The launches
# need host blocks of that size too.
@pytest.mark.parametrize("limit", [100000, 1000000])
def test_host_memory_of_a_batch_fails(entry, limit):
    (c,) = run(entry, "batch", 400, 1, 1, "host", limit)
    assert c.status == -4 and c.coop == 0


def test_host_memory_of_the_layout_alone_fails(entry):
    """The tables of a layout for 40 x 40 rows take more than 20 kB, the launches'
    vectors 13 kB."""
    (c,) = run(entry, "batch", 40, 1, 1, "host", 20000)
    assert c.status == 0 and c.coop == 0 and c.plain > 0 and c.threads_per_row > 0


# the layout's tables, positions, slots and columns, and the solve's vectors
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
def test_batch_short_of_device_memory_takes_the_launches(entry, k):
    (c,) = run(entry, "batch", 40, 1, 1, "short", k)
    assert c.status == 0 and c.coop == 0 and c.plain > 0 and c.threads_per_row > 0


@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_solve_short_of_device_memory_takes_the_launches(entry, k):
    for c in run(entry, "single", 40, 1, 2, "short", k):
        assert c.status == 0 and c.coop == 0 and c.plain > 0


def test_refused_launches(entry):
    for c in run(entry, "batch", 40, 2, 2, "refused"):
        assert c.status == 0 and c.coop == 1 and c.plain > 0 and c.threads_per_row > 0
    for c in run(entry, "single", 40, 1, 2, "refused"):
        assert c.status == 0 and c.coop == 1 and c.plain > 0


def test_a_system_that_fits_no_team_is_planned_once(entry):
    """640,000 rows on 256 blocks are 2,500 a block, with about 1,600 columns of
    other blocks: 2,500 + 4,100 values for each of four right-hand sides, more
    than the 158 KiB of LDS.  The second call allocates what the launches need
    and copies of the ranges, no layout."""
    first, again = run(entry, "batch", 800, 4, 2, "none")
    assert first.coop == again.coop == 0 and first.threads_per_row > 0
    launches = 3 * 4 * 8 * 640000  # host copies of the right-hand sides and the solution; the tiles: 1 MB
    assert first.host_bytes > launches + 20000000 and again.host_bytes < launches + 5000000
