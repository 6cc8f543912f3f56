"""Device memory the library asks for, and what it does when there is none: librtx.so on
a HIP runtime that allocates host memory within a limit and runs no kernels
(host/fake_hip.cpp), each case in a process of its own."""
import os
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

HOST = os.path.join(ROOT, "tests", "host")
MIB = 1 << 20


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("host") / "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w",
                    os.path.join(HOST, "fake_hip.cpp"), "-o", lib], check=True)
    return lib


SETUP = """
import ctypes, sys
fake = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
for f in ("fake_live", "fake_largest", "fake_peak"):
    getattr(fake, f).restype = ctypes.c_size_t
fake.fake_limit.argtypes = [ctypes.c_size_t]
sys.path.insert(0, {package!r})
import numpy as np
import rtx
MIB = 1 << 20
ctx = rtx.Context(0)
"""


def _run(lib, body):
    code = SETUP.format(lib=lib, package=os.path.join(ROOT, "treelet-prefetching-for-rt_amd")) + textwrap.dedent(body)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


def test_prediction_after_a_failed_allocation(fake_hip):
    """Memory for one of prediction's two buffers only: the call fails and keeps neither, and
    the next one, with memory, has both."""
    _run(fake_hip, """
        net = ctx.mlp(100, 200)
        samples = net.upload(np.zeros(50, rtx.MLP_SAMPLE_DTYPE))
        net.predict(samples, n=50)
        both = fake.fake_largest()
        net2 = ctx.mlp(100, 200)
        before = fake.fake_live()
        fake.fake_reset()
        fake.fake_limit(before + both + MIB)  # the outputs and the first buffer
        try:
            net2.predict(samples, n=50)
            sys.exit("no error")
        except rtx.RtxError as e:
            assert e.status == 12, e.status
        assert fake.fake_launches() == 0
        kept = fake.fake_live() - before
        assert kept < MIB, kept
        fake.fake_limit(2**63)
        net2.predict(samples, n=50)
        assert fake.fake_live() - before > 16 * MIB
    """)


TRACE = """
scene = rtx.workload_scene(rtx.workload_desc(rtx.WORKLOAD_SPHERE_AND_QUAD, slices=16, stacks=8, width=8, height=8, seed=1))
ctx.set_scene(scene.arena, scene.tlas_offset)
owner = np.zeros(len(scene.arena) // 64, np.uint32)
tlas = np.array([scene.tlas_offset], np.uint64)
ctx.set_treelets(8192, tlas, np.array([0, 1], np.uint64), tlas, owner)
dummy = rtx.DeviceBuffer(ctx, 64)  # (no kernel runs: rays and hits are never read)
def trace(n, mode, **kw):
    fake.fake_reset()
    before = fake.fake_live()
    status = ctx.trace_device(dummy, n, dummy, mode=mode, **kw)
    return status, (fake.fake_peak() - before) / MIB
"""


@pytest.mark.parametrize("mode", [0, 1])
def test_eight_lanes_per_ray_take_no_spill_area(fake_hip, mode):
    """The eight-lanes kernel keeps its stacks in LDS: a call of any size that asks for it
    allocates nothing for them."""
    _run(fake_hip, TRACE + f"""
status, mib = trace(50_000_000, {mode}, lanes_per_ray=8)
assert status == 0 and mib < 1, (status, mib)
status, mib = trace(1000, {mode})
assert status == 0 and mib < 1, (status, mib)
""")


def test_a_spill_area_of_the_size_asked_for_is_enough(fake_hip):
    """A launch that fills the GPU asks for more than its own spill area, so that one with
    other options finds room; where that cannot be had, its own is enough."""
    _run(fake_hip, TRACE + """
fake.fake_limit(fake.fake_live() + 300 * MIB)
status, mib = trace(2_000_000, 0)
assert status == 0 and 0 < mib <= 300, (status, mib)
status, mib = trace(2_000_000, 0)
assert status == 0 and mib == 0, (status, mib)
status, _ = trace(2_000_000, 1)  # 512 MiB of its own
assert status == 7, status
fake.fake_limit(2**63)
status, mib = trace(2_000_000, 1)
assert status == 0 and mib > 500, (status, mib)
""")
