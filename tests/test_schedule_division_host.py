"""The schedule's division (schedule.h, sched_div_by), compiled for the host: the arithmetic that the device runs, a float reciprocal and
two corrections, must give the quotient exactly for the reciprocals one unit in the last place around 1 / b.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cmath>
#include <initializer_list>
#include "schedule.h"
// wrong quotients among `count` pairs, over the three reciprocals
extern "C" int wrong(const int* a, const int* b, int count, int* first) {
  int bad = 0;
  for (int i = 0; i < count; i++) {
    const float exact = (float)(1.0 / (double)(float)b[i]);
    for (const float inverse : {exact, std::nextafter(exact, 0.f), std::nextafter(exact, 2.f)})
      if (esmoe::sched_div_by(a[i], b[i], inverse) != a[i] / b[i] && bad++ == 0) *first = i;
  }
  return bad;
}
"""
TOP = 3 * 2**29   # of the dividend


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("division")
    (folder / "host.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(folder / "host.cpp"),
                    "-o", str(folder / "host.so")], check=True)
    return ctypes.CDLL(str(folder / "host.so"))


def _check(host, a, b):
    a, b = (np.ascontiguousarray(v, dtype=np.int32) for v in (a, b))
    ptr, first = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), ctypes.c_int(-1)
    bad = host.wrong(ptr(a), ptr(b), len(a), ctypes.byref(first))
    assert bad == 0, (bad, int(a[first.value]), int(b[first.value]))


def test_small_numbers_all(host):
    b = np.arange(1, 513)
    for lo in range(0, 8192, 1024):
        a = np.arange(lo, lo + 1024)
        _check(host, np.repeat(a, len(b)), np.tile(b, len(a)))


def test_around_multiples_and_the_ends_of_the_range(host):
    rng = np.random.default_rng(0)
    edges = [1, 2, 3, 5, 7, 16, 127, 128, 192, 255, 256, 257, 65535, 65537, 2**23 - 1, 2**24 + 1, 2**30 - 1, 2**30 + 1, 2**31 - 2, 2**31 - 1]
    b = np.concatenate([np.array(edges * 200, dtype=np.int64), np.exp2(rng.uniform(0, 31, 400_000)).astype(np.int64).clip(1, 2**31 - 1)])
    for most in (16, 4096, 2**20, TOP):
        q = np.minimum((rng.random(len(b)) * (np.minimum(TOP // b, most) + 1)).astype(np.int64), TOP // b)
        for a in (q * b, q * b - 1, q * b + b - 1, q * b + rng.integers(0, b), TOP // b * b, TOP // b * b - 1, np.full(len(b), TOP)):
            _check(host, a.clip(0, TOP), b)
