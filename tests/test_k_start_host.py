"""First K block of an expert's K order (schedule.h, sched_k_start), compiled for the host: spread over all places by scales as
quantisers write them, block 0 for equal scales, the same for scales that differ by a common power of two."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from tests import helpers as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "schedule.h"
using namespace esmoe;
extern "C" {
int k_start(const unsigned* s) { return sched_k_start(s[0], s[1], s[2], s[3]); }
int spread(int k) { return sched_spread_k(k); }
int word(int e, int start) { return rec_expert_word(e, start); }
int expert(int w) { return rec_expert(w); }
int first_kb(int w) { return rec_first_kb(w); }
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("kstart")
    (folder / "host.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(folder / "host.cpp"), "-o", str(folder / "host.so")], check=True)
    return ctypes.CDLL(str(folder / "host.so"))


def _start(host, words):
    w = np.ascontiguousarray(words, dtype=np.uint32)
    assert w.size == 4
    return host.k_start(w.ctypes.data_as(ctypes.c_void_p))


def test_starts_are_spread_and_go_by_scale_differences(host):
    rng = np.random.default_rng(0)
    weights = np.abs(rng.standard_normal((4000, 4, 1024)).astype(np.float32)).max(axis=2)
    fp32 = (weights * np.float32(0.02 / 448)).astype(np.float32)
    pow2 = np.exp2(rng.integers(-12, -8, size=(4000, 4))).astype(np.float32)      # scales rounded to powers of two
    e8m0 = rng.integers(115, 119, size=(4000, 16)).astype(np.uint8)
    for words, shifted in ((fp32.view(np.uint32), (fp32 * np.float32(8)).view(np.uint32)), (pow2.view(np.uint32), (pow2 * np.float32(0.25)).view(np.uint32)),
                           (e8m0.view(np.uint32), (e8m0 + np.uint8(5)).view(np.uint32))):
        got = np.array([_start(host, w) for w in words])
        count = np.bincount(got, minlength=8)
        assert len(count) == 8 and count.min() > 4000 // 8 // 2 and count.max() < 4000 // 8 * 2, count
        assert [_start(host, w) for w in shifted[:200]] == got[:200].tolist()
        assert [H.k_start_blocks(np.ascontiguousarray(w).tobytes()) for w in words[:500]] == (4 * got[:500]).tolist()
    for value in (0, 0x3f800000, 0x7f7f7f7f, 0xffffffff):
        assert _start(host, [value] * 4) == 0


def test_record_word_and_condition(host):
    for e in (0, 1, 511, 1023):
        for start in range(8):
            w = host.word(e, start)
            assert w >= 0 and host.expert(w) == e and host.first_kb(w) == 4 * start and host.first_kb(w) + 4 <= 32
    assert [k for k in range(128, 12289, 128) if host.spread(k)] == [4096, 8192, 12288]
