"""The depth order's kernels (3dgs-project_amd/csrc/gs_sample_sort.h), compiled for the CPU and run
under the two extreme schedules of a workgroup's wavefronts (emulation/sample_sort.cpp): between two
barriers the first wavefront runs ahead of all others, or the last one does. A word of LDS that one
wavefront stores while another has still to read it, with no barrier between, gives another result
under one of them; on a GPU such an overlap is rare and timing alone decides it."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "3dgs-project_amd" / "csrc"


@pytest.fixture(scope="module")
def emulation(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    so = tmp_path_factory.mktemp("emulation") / "sample_sort.so"
    subprocess.run([cxx, "-std=c++17", "-O2", "-fPIC", "-shared", "-fno-strict-aliasing", "-w", f"-I{CSRC}",
                    str(HERE / "emulation" / "sample_sort.cpp"), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.emulate_sample_sort.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_int,
                                        ctypes.c_void_p, ctypes.c_void_p]
    lib.sample_positions.argtypes = [ctypes.c_int64, ctypes.c_void_p]
    lib.sample_positions.restype = ctypes.c_int64
    return lib


def keys_of(kind, n, rng, lib):
    if kind == "descending":  # the first wavefront holds the largest keys
        return np.arange(n, 0, -1).astype(np.uint32) * np.uint32(1000)
    if kind == "ascending":  # ... and the last one
        return np.arange(1, n + 1).astype(np.uint32) * np.uint32(1000)
    if kind == "culled_mix":  # a third equal to the largest
        k = rng.integers(1 << 20, 1 << 29, n).astype(np.uint32)
        k[rng.random(n) < 0.33] = np.uint32(1 << 30)
        return k
    if kind == "few_distinct":  # the digit passes in LDS
        return rng.integers(0, 5, n).astype(np.uint32) * np.uint32(70_001)
    if kind == "equal":
        return np.full(n, 77, np.uint32)
    assert kind == "beyond_lds"  # every sampled key below all others: one bucket of nearly all keys
    k = rng.integers(1 << 16, 1 << 18, n).astype(np.uint32)
    pos = np.zeros(lib.sample_positions(n, None), np.uint32)
    lib.sample_positions(n, pos.ctypes.data)
    k[pos] = np.arange(len(pos))
    return k


@pytest.mark.parametrize("last_first", [0, 1])
@pytest.mark.parametrize("kind,n", [
    *((k, n) for k in ("descending", "ascending", "culled_mix", "few_distinct", "equal") for n in (65, 2048, 4096, 9000)),
    ("descending", 1), ("culled_mix", 2049), ("beyond_lds", 9000),
])
def test_order_does_not_depend_on_the_schedule(emulation, kind, n, last_first):
    rng = np.random.default_rng(n)
    keys = keys_of(kind, n, rng, emulation)
    counts = rng.integers(0, 9, n).astype(np.uint32)
    order, offsets = np.full(n, -1, np.int32), np.full(n + 1, -1, np.int32)
    assert emulation.emulate_sample_sort(keys.ctypes.data, counts.ctypes.data, n, last_first, order.ctypes.data,
                                         offsets.ctypes.data), "a thread waits for ever"
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(order, want)
    assert np.array_equal(offsets, np.concatenate([[0], np.cumsum(counts[want])]))
