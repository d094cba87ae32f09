"""Host side of the transfers (csrc/hip/rhllc_records): no GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "radrhd_solver_amd", "csrc", "hip")

FILL_ONCE = r"""
#include "rhllc_records.h"
#include <cassert>
#include <cstdio>
int main() {
  static int array[4];
  int *slot = nullptr, allocs = 0, fills = 0, releases = 0, alloc_error = 0, fill_error = 0;
  auto use = [&] {
    return rhllc_records::fill_once(
        slot, [&](int **p) { ++allocs; *p = alloc_error ? nullptr : array; return alloc_error; },
        [&](int *p) { ++fills; assert(p == array); return fill_error; }, [&](int *p) { ++releases; assert(p == array); });
  };
  alloc_error = 2;
  assert(use() == 2 && !slot && allocs == 1 && fills == 0 && releases == 0);
  alloc_error = 0, fill_error = 1;
  assert(use() == 1 && !slot && allocs == 2 && fills == 1 && releases == 1);  // not seen as filled by the next use
  fill_error = 0;
  assert(use() == 0 && slot == array && allocs == 3 && fills == 2 && releases == 1);
  assert(use() == 0 && slot == array && allocs == 3 && fills == 2 && releases == 1);
  std::puts("ok");
}
"""


def test_an_array_is_in_use_only_once_it_is_filled(tmp_path):
    """The face map of rhllc_download_face_flux is uploaded on first use; a failed copy must not leave
    a map of unset indices for the next call."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(FILL_ONCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-UNDEBUG", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=60).stdout == "ok\n"


THREADS = r"""
import ctypes, os, sys
import numpy as np
lib = ctypes.CDLL(sys.argv[1])
copy = lib["_ZN13rhllc_records4copyEPvPKvm"]
tasks = lambda: len(os.listdir("/proc/self/task"))
src = np.random.default_rng(1).integers(0, 255, (8 << 20) + 13, dtype=np.uint8)
dst = np.zeros_like(src)
before = tasks()
copy(ctypes.c_void_p(dst.ctypes.data), ctypes.c_void_p(src.ctypes.data), ctypes.c_size_t(1000))
small = tasks()
copy(ctypes.c_void_p(dst.ctypes.data), ctypes.c_void_p(src.ctypes.data), ctypes.c_size_t(src.nbytes))
assert np.array_equal(src, dst)
print(small - before, tasks() - before)
"""


def test_copies_take_a_bounded_number_of_threads():
    """Several ranks of a node share its cores: a copy starts 15 threads beside the caller's at most,
    however many OpenMP would use, fewer where OpenMP is told so, and none for a small one."""
    lib = os.path.join(ROOT, "radrhd_solver_amd", "librhllc_hip.so")
    for limit, most in ((64, 15), (3, 2)):
        env = dict(os.environ, OMP_NUM_THREADS=str(limit), OMP_DYNAMIC="false", OPENBLAS_NUM_THREADS="1")
        r = subprocess.run([sys.executable, "-c", THREADS, lib], env=env, capture_output=True, text=True, timeout=60,
                           check=True)
        assert r.stdout.split() == ["0", str(most)]
