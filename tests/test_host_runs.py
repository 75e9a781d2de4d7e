"""Host code of the library on a HIP runtime without a device
(tests/hip_host.cpp): what it launches, and what it leaves behind when an
allocation fails.  Every run is a process of its own, in which that runtime
is loaded before the library."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
host = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
host.host_launch_name.restype = ctypes.c_char_p
host.host_launch_ptr.restype = ctypes.c_void_p
host.host_mallocs.restype = host.host_live.restype = host.host_launches.restype = ctypes.c_long
host.host_pointer_queries.restype = ctypes.c_long
host.host_busy.argtypes = [ctypes.c_long]
host.host_fail_malloc.argtypes = [ctypes.c_long]
host.host_launch_name.argtypes = [ctypes.c_long]
host.host_launch_ptr.argtypes = [ctypes.c_long, ctypes.c_int]
sys.path.insert(0, sys.argv[2])
import numpy as np
from camille_amd import *

def launches():
    return [host.host_launch_name(k).decode() for k in range(host.host_launches())]

def tables():  # the operand table and tile list of every batch launch
    return [(host.host_launch_ptr(k, 0), host.host_launch_ptr(k, 1)) for k, n in enumerate(launches()) if "k_batch_" in n]

def block(ni, nj):
    x, y = np.meshgrid(0.5 * np.arange(ni), 0.5 * np.arange(nj))
    mean = np.zeros((5, nj, ni))
    mean[4] = 1 / 1.4
    return dict(x=x, y=y, mean=mean)
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip_host") / "libhip_host.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_host.cpp"), "-o", so], check=True)

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), so, os.path.dirname(HERE)],
                           capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-2000:]
        return p.stdout
    return run


BATCH = """
def batch():
    b = Batch([dict(block(70, 40), mode="FIX_DT", value=0.01) for _ in range(2)], precision=FP32)
    for k in range(2):
        b.set_solution(np.zeros((5, 40, 70)), k)
    host.host_forget()
    return b

def solved(b, fail=0):
    host.host_fail_malloc(fail)
    try:
        b.solve(3)
        return True
    except LeeError:
        return False
    finally:
        host.host_fail_malloc(0)

b = batch()
host.host_fail_malloc(0)
b.solve(3)
total = host.host_mallocs()
assert total > 10 and any("k_batch_pair" in n for n in launches())
b.close()
"""


def test_batch_after_a_failed_allocation(runtime):
    """Whichever allocation of a batch's first solve fails, the solve says so
    and the next one runs on whole tables."""
    runtime(BATCH + """
for k in range(1, total + 1):
    b = batch()
    assert not solved(b, fail=k), k
    host.host_forget()
    assert solved(b), k
    assert launches() and all(p and q for p, q in tables()), k
    b.close()
""")


def test_batch_whose_tuner_failed(runtime):
    """A tuner that stops at a failed allocation leaves neither events nor the
    tables it times on: a pinned shape then runs on the state.  Stage 1 reads
    Y2 and Y0; on the scratch tables it would read Y2 twice (the pointers
    after the six integers of StageArgs)."""
    runtime(BATCH + """
clean = host.host_live()
for k in range(1, total + 1):
    b = batch()
    assert not solved(b, fail=k), k
    b.set_tile_shape(1, 4)
    host.host_forget()
    assert solved(b), k
    mid = [p for (p, _), n in zip(tables(), launches()) if "k_batch_stageIfLb0ELi1ELi1E" in n]
    assert mid and len(tables()) == len(launches()), k
    yin, yn = (ctypes.c_void_p * 2).from_address(mid[0] + 24)
    assert yin != yn, k
    b.close()
    assert host.host_live() == clean, (k, host.host_live())
""")


def test_batch_after_a_failed_schedule(runtime):
    """A schedule that could not grow is not taken for the shorter one before."""
    runtime(BATCH + """
b = batch()
assert solved(b)
host.host_fail_malloc(1)
try:
    b.solve(50)
    assert False
except LeeError:
    pass
host.host_fail_malloc(0)
b.solve(2)
b.solve(60)
b.close()
""")


def test_boundary_faces_read_within_their_reach(tmp_path):
    """What a face's conditions read lies in bc_reach, by which faces and
    early receivers share the boundary launch."""
    exe, root = str(tmp_path / "bc_reads"), os.path.dirname(HERE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-fpermissive", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(root, "include"), "-I" + os.path.join(root, "camille_amd", "csrc"),
                    os.path.join(HERE, "bc_reads.cpp"), "-o", exe], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout


OVERSET = """
sys.path.insert(0, sys.argv[2] + "/tests")
from boundary_tables import DIMS, WALL, tables

def phase(*kinds, **kw):
    blocks = [block(*d) for d in DIMS]
    s = Solver(blocks, overset=tables(*kinds, **kw), mode="FIX_DT", value=0.01, boundaries=[WALL])
    host.host_forget()
    s.update_boundary([np.zeros((5,) + b["x"].shape) for b in blocks])
    s.close()
    names = [n for n in launches() if "k_b" in n or "k_ov" in n]
    assert names and any("k_boundary" in n for n in names) != any("k_ov_scatter" in n for n in names), names
    return any("k_boundary" in n for n in names)
"""


def test_boundary_phase_is_one_launch_where_its_tail_is_short(runtime):
    """One launch for few held receivers and few that read what faces write;
    with more, one workgroup would work through them, pass by pass (41 times
    the time of the separate launches for 16000 receivers along a wall)."""
    runtime(OVERSET + """
assert phase(0, 0, 1) and phase(2, 0, 5000) and phase(150, 12, 3000) and phase(384 - 25, 25, 10)
assert phase(20, 10, 200, 30, 8)
assert not phase(385, 0, 10) and not phase(3000, 0, 0)
assert not phase(0, 26, 1000) and not phase(0, 4000, 0)
assert not phase(2, 2, 100, twice=True) and not phase(20, 10, 200, 30, 8, twice=True)
""")


def test_result_pages_are_mapped_while_there_is_work_only(runtime):
    """A fetch with nothing to wait for goes straight to the copy; beside work
    in flight the result's pages are written as they are."""
    runtime("""
y = np.random.default_rng(0).standard_normal((5, 40, 70))
y[3] = 0
for prec in (FP64, FP32):
    s = Solver([block(70, 40)], precision=prec, mode="FIX_DT", value=0.01)
    s.set_solution(y)
    before = host.host_pointer_queries()
    out = s.solution()
    assert host.host_pointer_queries() == before
    host.host_busy(2)  # ends while the pages are mapped
    out = s.solution()
    assert host.host_pointer_queries() == before + 1
    if prec == FP64:
        assert np.array_equal(out, y)
    s.solve(1)  # the stream's "not ready" is no failure of what follows
    s.close()
""")
