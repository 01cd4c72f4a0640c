"""The host side on a machine without a GPU, on tests/host_runtime.c: a kernel launch that the runtime refuses
is an error of the call that made it, not a result (the entry points whose kernels write the caller's
data); the slots of the field readback; how many batches of iterations go out; the mesh reader's threads."""
import os
import subprocess
import sys

import pytest

from srx_amd import inputs

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes as C, sys
import numpy as np
rt = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
import srx_amd
L = srx_amd.lib()
E_HIP = 2003
def each_launch_refused(call):
    rt.host_fail_launch(-1)
    assert call() == 0
    n, held = rt.host_launches(), rt.host_device_blocks()
    assert n > 0
    for k in range(n):
        rt.host_fail_launch(k)
        assert call() == E_HIP, k
        assert rt.host_device_blocks() == held, k
    rt.host_fail_launch(-1)
    assert call() == 0
"""
FFT = """
n, nc = (12, 10, 8), 3
x = np.zeros(nc * 12 * 10 * 8)
X = np.zeros(nc * 12 * 10 * 5 * 2)
for prec in (srx_amd.PREC_FP64, srx_amd.PREC_MIXED):
    each_launch_refused(lambda: L.srx_fft_forward(srx_amd._dptr(x), nc, *n, prec, srx_amd._dptr(X)))
    each_launch_refused(lambda: L.srx_fft_inverse(srx_amd._dptr(X), nc, *n, prec, 1.0, srx_amd._dptr(x)))
    L.srx_fft_forward_noalloc.argtypes = L.srx_fft_forward.argtypes
    each_launch_refused(lambda: L.srx_fft_forward_noalloc(srx_amd._dptr(x), nc, *n, prec, srx_amd._dptr(X)))
"""
FIELD = """
s = srx_amd.Solver(sys.argv[2])
for name, (fid, nc) in srx_amd.FIELDS.items():
    if name in ("grain", "rho_g1", "rho_g2"):   # kept on the host; GND option only
        continue
    out = np.empty(s.nxyz * nc)
    each_launch_refused(lambda: L.srx_get_field(s.h, fid, srx_amd._dptr(out), out.size))
"""
SLOTS = """
s = srx_amd.Solver(sys.argv[2])
for name in ("sig", "rho_s", "rho_tot"):
    fid, nc = srx_amd.FIELDS[name]
    out = np.empty(s.nxyz * nc)
    rt.host_watch_pointer(3)   # where k_gather writes
    assert L.srx_get_field(s.h, fid, srx_amd._dptr(out), out.size) == 0
    assert rt.host_pointer_offsets() % 512 == 0, (name, rt.host_pointer_offsets())
"""
PINNED = """
s = srx_amd.Solver(sys.argv[2])
before = rt.host_pinned_bytes()
for name in ("sig", "rho_s", "rho_tot"):   # the first read, and larger and smaller fields after it
    s.field(name)
most = s.nxyz * 12 * 8
threads = s.nxyz * 9 * 8 >= 8 << 20   # fields that helper threads copy
assert rt.host_pinned_bytes() - before <= (most + 4096 if most <= 2 << 20 else max(most // 4, threads * (8 << 20)) + 4 * 4096)
"""
AHEAD = """
s = srx_amd.Solver(sys.argv[2], reserved=[0, 1])   # launch by launch
def launches(iters):
    rt.host_stop_after(iters)
    rt.host_fail_launch(-1)
    assert s.step()["iters"] == iters
    return rt.host_launches()
first, again = launches(8), launches(8)    # one batch, with nothing known of the iteration count
per_batch = launches(16) - again           # two batches
for few in (3, 8, 20):
    launches(900)
    assert launches(few) <= again + (few // 8 + 8) * per_batch, few
"""
MESH = """
want = np.array([int(line.split()[6]) for line in open(sys.argv[3])], float)
for threads in (0, 1, 2, 3, 16):
    s = srx_amd.Solver(sys.argv[2], nthreads=threads)
    np.testing.assert_array_equal(s.field("grain"), want)
    s.close()
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("rt") / "host_runtime.so")
    obj = lib + ".o"
    subprocess.check_call(["gcc", "-c", "-fPIC", "-O1", "-o", obj, os.path.join(HERE, "host_runtime.c")])
    subprocess.check_call(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-o", lib, os.path.join(HERE, "host_control.cpp"), obj])
    return lib


def run(body, *args):
    p = subprocess.run([sys.executable, "-c", PRELUDE + body, *args], cwd=os.path.dirname(HERE), capture_output=True,
                       text=True, timeout=110)
    assert p.returncode == 0, p.stderr[-2000:]


def test_transforms_report_a_refused_launch(runtime):
    run(FFT, runtime)


@pytest.mark.parametrize("n", [(6, 5, 4), (48, 40, 60)])   # one chunk; several, some of them in flight
def test_field_reads_report_a_refused_launch(runtime, tmp_path, n):
    run(FIELD, runtime, inputs.make_case(str(tmp_path), n=n, grains=3, seed=1, nsteps=1, timestep=0.1))


@pytest.mark.parametrize("n", [(75, 75, 75), (81, 81, 81), (120, 81, 75)])
def test_field_chunks_start_aligned(runtime, tmp_path, n):
    """The gather kernel stores 8-byte values in runs of 512 B: every chunk's slot starts at a multiple of
    that from the first, also where the slots' size follows from the number of voxels."""
    run(SLOTS, runtime, inputs.make_case(str(tmp_path), n=n, grains=3, seed=1, nsteps=1, timestep=0.1))


@pytest.mark.parametrize("n", [(4, 4, 4), (27, 27, 27), (32, 32, 32), (48, 48, 48), (75, 60, 45)])
def test_first_field_read_pins_a_quarter_of_a_field(runtime, tmp_path, n):
    """Pinned memory is paid for by a context's first read (its pages are mapped on first touch): no more of it
    than a quarter of the largest field, or one such field where that is small, or four slots of 2 MiB
    where helper threads share the page faults."""
    run(PINNED, runtime, inputs.make_case(str(tmp_path), n=n, grains=3, seed=1, nsteps=1, timestep=0.1))


def test_a_quick_increment_after_a_long_one(runtime, tmp_path):
    """Batches of 8 iterations go out ahead by the last increment's count: an increment that needs fewer
    stops the host within eight batches of its own last one."""
    run(AHEAD, runtime, inputs.make_case(str(tmp_path), n=(6, 5, 4), grains=3, seed=1, nsteps=20, timestep=0.1))


@pytest.mark.parametrize("n", [(5, 4, 3), (16, 16, 16), (16, 16, 32), (27, 15, 18), (27, 27, 30)])
def test_mesh_is_read_whole_by_any_number_of_threads(runtime, tmp_path, n):
    """Threads take ranges of 4096 voxels in turn: fewer than one range, whole ranges, remainders, more
    threads than ranges."""
    deck = inputs.make_case(str(tmp_path), n=n, grains=40, seed=6, nsteps=1, timestep=0.1)
    run(MESH, runtime, deck, str(tmp_path / "mesh.txt"))
