"""What calls of the library ask of the HIP runtime, on the CPU: the host code
built without device code against a stand-in (tests/host/mock_calls.cc) that
records launches."""
import ctypes as C
import os
import shutil
import subprocess
import threading
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
SOURCES = [ROOT / "kernels_amd/csrc" / f for f in ("prk_api.hip", "batch.hip", "autotune.hip", "transpose.hip")]
SOURCES.append(ROOT / "tests/host/mock_calls.cc")

pytestmark = pytest.mark.skipif(not (os.path.exists(HIPCC) and SOURCES[-1].exists()), reason="needs hipcc")


class Solve(C.Structure):
    _fields_ = [(f, C.c_int) for f in ("pattern", "radius", "dtype", "n", "iterations", "init")] + [
        ("seed", C.c_uint64)]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("calls")

    def compile_one(src):
        obj = tmp / (src.name + ".o")
        subprocess.run([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-fPIC", f"-I{ROOT / 'include'}",
                        f"-I{ROOT / 'kernels_amd/csrc'}", "-x", "hip", "-c", str(src), "-o", str(obj)],
                       check=True, capture_output=True, text=True)
        return str(obj)

    objs = [compile_one(s) for s in SOURCES]
    # the device code that the host code would register does not exist here
    names = subprocess.run(["nm", "-u", *objs], check=True, capture_output=True, text=True).stdout.split()
    defs = [f"-Wl,--defsym={s}=0" for s in sorted(set(names)) if s.startswith("__hip_fatbin")]
    so = tmp / "libcalls.so"
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", str(so), *objs, *defs, "-lpthread"], check=True, capture_output=True,
                   text=True)
    L = C.CDLL(str(so))
    L.prk_last_error.restype = C.c_char_p
    L.mock_reset()
    return L


def check(L, rc):
    assert rc == 0, L.prk_last_error()


def kernels(L):
    v = (C.c_uint * 3)()
    out = []
    for i in range(L.mock_kernels()):
        L.mock_kernel(i, v)
        out.append(tuple(v))
    return out


def sweeps(L):
    """(sweeps, any, rows, workgroups per CU, reach, in, in_next) of each launch."""
    v = (C.c_longlong * 7)()
    out = []
    for i in range(L.mock_sweeps()):
        L.mock_sweep(i, v)
        out.append(tuple(v))
    return out


def test_batch_output_runs_on_the_batch_s_device(lib):
    # the thread that fetches a grid has another device current than the one
    # the batch was made on: the rows are packed where they lie, and the
    # thread's device is as it was
    L, n = lib, 100
    batch = C.c_void_p()
    L.hipSetDevice(1)
    try:
        check(L, L.prk_batch_create(C.byref(Solve(0, 1, 1, n, 2, 1, 5)), 1, 0, 0, C.byref(batch)))
    finally:
        L.hipSetDevice(0)
    before = L.mock_bytes_on(0)
    seen = []

    def fetch():
        host = np.zeros((n, n), np.float32)
        L.mock_reset()
        rc = L.prk_batch_output(batch, 0, 0, host.ctypes.data_as(C.c_void_p), C.c_size_t(host.nbytes))
        dev = C.c_int(-1)
        L.hipGetDevice(C.byref(dev))
        seen.extend([rc, dev.value, [k[2] for k in kernels(L)]])

    t = threading.Thread(target=fetch)
    t.start()
    t.join()
    assert seen == [0, 0, [1]] and L.mock_bytes_on(0) == before
    L.prk_batch_destroy(batch)


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_sweep_reads_stay_inside_the_grid(lib, dtype):
    # rows off 16-byte boundaries are read in vectors that may run past their
    # row; a row before the last must not read past the last one's elements
    L, es = lib, (8, 4, 2)[dtype]
    for n in range(3, 20):
        for pitch in range(n, n + 9):
            for offset in (0, 4, 8):
                p = [C.c_void_p((k << 20) + offset) for k in (1, 2, 3)]
                L.mock_reset()
                check(L, L.prk_sweep(0, 1, dtype, n, C.c_longlong(pitch), *p, None))
                (s,) = sweeps(L)
                assert s[4] <= ((n - 1) * pitch + n) * es, (n, pitch, offset)


@pytest.mark.parametrize("dtype,n", [(0, 92680), (0, 92681), (0, 92682), (0, 130001), (1, 131071), (1, 131072),
                                     (2, 185363), (2, 185364), (2, 300000)])
def test_add_of_very_large_grids_is_launched(lib, dtype, n):
    # a launch holds fewer than 2^32 threads: larger dense grids go row by row
    lib.mock_reset()
    check(lib, lib.prk_add_ex(dtype, n, C.c_longlong(n), C.c_void_p(1 << 20), None))
    assert len(kernels(lib)) == 1


@pytest.mark.parametrize("n,least", [(1000, 128), (2000, 256), (3001, 256)])
def test_tiles_of_a_small_slab_fill_the_chip(lib, n, least):
    # the height goes by the slab's own rows: an eighth of a grid's rows in
    # tiles chosen for the whole grid left most of the 256 CUs idle
    L, rows = lib, n // 8
    p = [C.c_void_p(k << 30) for k in (1, 2, 3)]
    L.mock_reset()
    pitch = C.c_longlong((n + 15) // 16 * 16)
    check(L, L.prk_sweep_slab(0, 2, 0, n, 3 * rows, rows, pitch, *p, None))
    (s,) = sweeps(L)
    groups = ((n + 127) // 128 + 3) // 4
    assert groups * -(-(rows + 4) // s[2]) >= least


class Tuning(C.Structure):
    _fields_ = [(f, C.c_int) for f in ("variant", "rows_per_wave", "wgs_per_cu", "order")] + [("gbs", C.c_double)]


@pytest.mark.parametrize("pattern,radius,dtype,n,rows,wgs", [
    (1, 8, 0, 3600, 24, 2), (1, 8, 0, 5400, 24, 2),      # 32 rows: 282 -> 300 us, 542 -> 573
    (0, 4, 0, 18000, 16, 2), (0, 5, 0, 11000, 24, 2), (0, 6, 0, 14000, 24, 2),
    (0, 8, 0, 2800, 24, 2), (0, 4, 1, 4200, 16, 2), (0, 8, 1, 15000, 24, 2),
    (1, 2, 2, 15000, 12, 4), (1, 2, 2, 18000, 12, 3),
    (1, 5, 1, 4800, 32, 4), (1, 5, 0, 16384, 32, 4)])
def test_default_tilings(lib, pattern, radius, dtype, n, rows, wgs):
    # sizes at which the rules of small, middle and large grids meet
    t = Tuning()
    check(lib, lib.prk_tuning_get(pattern, radius, dtype, n, C.byref(t)))
    assert (t.rows_per_wave, t.wgs_per_cu) == (rows, wgs)


@pytest.mark.parametrize("n", [1, 2, 63, 129, 513, 46340])
def test_default_height_is_inside_the_grid(lib, n):
    t = Tuning()
    for pattern in (0, 1):
        for radius in range(1, 9):
            for dtype in (0, 1, 2):
                check(lib, lib.prk_tuning_get(pattern, radius, dtype, n, C.byref(t)))
                assert 1 <= t.rows_per_wave <= n


def test_batch_heights_of_passes_are_not_tuned(lib):
    # a stencil that runs in passes ignores the table of heights: nothing is
    # timed for it, and what the table holds leaves the schedule as it is
    L, keys, rows = lib, C.c_int(), C.c_int()
    solves = (Solve * 6)(*[Solve(0, 2, 1, 300 + k, 9, 1, k) for k in range(3)],
                         *[Solve(1, 6, 1, 300 + k, 9, 1, k) for k in range(3)])

    def plan():
        batch, info = C.c_void_p(), (C.c_longlong(), C.c_longlong(), C.c_int())
        check(L, L.prk_batch_create(solves, 6, 0, 0, C.byref(batch)))
        check(L, L.prk_batch_info(batch, *[C.byref(v) for v in info]))
        L.prk_batch_destroy(batch)
        return [v.value for v in info]

    try:
        before = plan()
        L.mock_reset()
        check(L, L.prk_batch_autotune(solves, 3, 2, 1, C.byref(keys)))
        assert keys.value == 1 and L.mock_kernels() == 0
        check(L, L.prk_batch_tuning_set(0, 2, 1, 300, 128))
        assert plan()[1:] == before[1:]
        check(L, L.prk_batch_autotune(solves, 6, 2, 1, C.byref(keys)))
        assert keys.value == 2 and L.mock_kernels() > 0
    finally:
        L.prk_batch_tuning_clear()


@pytest.mark.parametrize("iterations", [1, 2, 3, 4, 10, 11, 255, 256, 257, 511, 512, 600])
def test_run_of_passes_ends_in_its_buffer(lib, iterations):
    # launches hand the in buffers over in turn, add up to iterations + 1
    # sweeps, and end in the buffer that one sweep per launch would end in; a
    # last sweep alone leaves the in before the last in the other buffer, after
    # a pass that buffer is refreshed
    L, n, final = lib, 512, C.c_int(-1)
    p = [C.c_void_p(k << 30) for k in (1, 2, 3)]
    L.mock_reset()
    check(L, L.prk_run(0, 2, 0, n, C.c_longlong(n), iterations, *p, None, C.byref(final), None))
    calls = sweeps(L)
    assert sum(s[0] for s in calls) == iterations + 1 and final.value == (iterations + 1) % 2
    src = 1 << 30
    for s in calls:
        assert s[5] == src and s[6] == (3 << 30) - src
        src = s[6]
    assert src == p[final.value].value
    assert L.mock_kernels() == (0 if calls[-1][0] == 1 else 1)
    assert all(s[1] == (s is calls[0]) for s in calls if s[0] > 1)  # the caller's values: the first pass alone


@pytest.mark.parametrize("order,tiles", [
    (1024, 32 * 16), (1408, 22 * 11), (1409, 23 * 23), (1495, 24 * 24), (1600, 25 * 25), (1601, 26 * 13),
    (2496, 39 * 20), (2497, 40 * 40), (2560, 40 * 40), (2561, 41 * 21)])
def test_transpose_tiles_where_turns_of_the_chip_end(lib, order, tiles):
    # 64 x 128 tiles that come to little more than whole turns of the CUs left
    # most of them idle (odd order 1495: 14.8 -> 16.5 us)
    lib.mock_reset()
    check(lib, lib.prk_transpose_ex(order, C.c_void_p(1 << 30), C.c_void_p(2 << 30), None))
    (k,) = kernels(lib)
    assert k[0] == tiles
