"""pgf_batch_pcg returns a status when memory runs out, no exception leaves the
C entry, and systems that fit no team are not laid out again on every call.  A compiled caller (batch_entry.cpp) makes a context by hand and no
GPU is visible to it, so every device allocation fails."""
import os
import subprocess

import pytest

from pigfem_assignment_amd import build, _lib as L

HERE = os.path.dirname(os.path.abspath(__file__))
ENV = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1")


@pytest.fixture(scope="module")
def entry(tmp_path_factory):
    objs = [os.path.join(build.OBJ, os.path.basename(s) + ".o") for s in build.HOST_SRC + build.HIP_SRC]
    assert all(os.path.exists(o) for o in objs), "the library is not built; run `python -m pigfem_assignment_amd.build`"
    out = str(tmp_path_factory.mktemp("entry") / "batch_entry")
    obj = out + ".o"
    subprocess.run([build.HIPCC, "-O1", "-std=c++17", "--offload-arch=" + build.ARCH, "--offload-host-only", "-x", "hip", "-c",
                    os.path.join(HERE, "batch_entry.cpp"), "-o", obj], check=True, capture_output=True)
    subprocess.run([build.HIPCC, "--offload-arch=" + build.ARCH, "-o", out, obj] + objs + ["-lgomp"], check=True,
                   capture_output=True)
    return out


def run(exe, *args):
    r = subprocess.run([exe] + [str(a) for a in args], env=ENV, capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0, "ended with %d" % r.returncode
    return r.stdout


def test_device_memory_of_a_solve_fails(entry):
    out = run(entry, "workspace")
    assert out.startswith("status -4, ") and len(out.split(": ")[1]) > 4


# 100 kB: a thread's table of the system's columns (640 kB), in the parallel
# region; 1 MB: the steps of all shares (2.6 MB), behind it
@pytest.mark.parametrize("limit", [100000, 1000000])
def test_host_memory_of_the_layout_fails(entry, limit):
    assert run(entry, "plan", limit).startswith("status -4, ")


def test_a_system_that_fits_no_team_is_planned_once(entry):
    """640,000 rows on 256 blocks are 2,500 a block, with about 1,600 columns of
    other blocks: 2,500 + 4,100 values for each of four right-hand sides, more
    than the 158 KiB of LDS.  The second call allocates copies of the ranges and
    error texts, no layout."""
    first, again = [int(line.split()[2]) for line in run(entry, "unfit").splitlines()]
    assert first > 100000 and again < 10000
