"""The rule of permute_rule.h, compiled for the host: which rows are stored plainly, and which pairs are looked at."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SAMPLES = 128

SOURCE = r"""
#include "permute_rule.h"
extern "C" {
int plain_from(long tokens, int topk, long row_bytes) { return esmoe::permute_plain_from(tokens, topk, row_bytes); }
long sample_step(long pairs) { return esmoe::permute_sample_step(pairs); }
int samples() { return esmoe::kPermuteSamples; }
int run() { return esmoe::kPermuteRun; }
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    (d / "host.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(d / "host.cpp"), "-o", str(d / "host.so")], check=True)
    lib = ctypes.CDLL(str(d / "host.so"))
    lib.plain_from.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_long]
    lib.sample_step.argtypes, lib.sample_step.restype = [ctypes.c_long], ctypes.c_long
    assert lib.samples() == SAMPLES and SAMPLES % lib.run() == 0
    return lib


# (tokens, top-k, bytes of a row, share of local pairs) -> plain stores are the faster ones (both measured on MI355X)
@pytest.mark.parametrize("tokens,topk,row_bytes,share,plain", [
    (1024, 4, 8192, 1, False), (700, 4, 14336, 1, False), (1500, 4, 8192, 1, False), (1003, 8, 14336, 1, True), (4096, 2, 8192, 1, True),
    (2048, 8, 8192, 1 / 8, False), (4096, 8, 4096, 1 / 8, False), (4096, 8, 4096, 1 / 4, False), (1024, 8, 14336, 1 / 4, False),
    (8192, 8, 14336, 1 / 64, False), (8192, 8, 14336, 1 / 8, True), (16384, 8, 8192, 1 / 16, True), (4096, 8, 14336, 1 / 8, True),
])
def test_rows_are_stored_plainly_by_what_is_written(host, tokens, topk, row_bytes, share, plain):
    need = host.plain_from(tokens, topk, row_bytes)
    assert 1 <= need <= SAMPLES + 1
    assert (SAMPLES * share >= need) == plain


def test_small_calls_are_never_looked_at(host):
    for tokens, topk, row_bytes in ((1, 2, 16), (64, 8, 14336), (512, 8, 8192), (15, 8, 1 << 20), (1, 64, 1 << 40)):
        assert host.plain_from(tokens, topk, row_bytes) == SAMPLES + 1


@pytest.mark.parametrize("pairs", [128, 129, 143, 144, 1000, 65536, (1 << 31) - 1])
def test_samples_are_pairs_of_the_call(host, pairs):
    step, runs = host.sample_step(pairs), SAMPLES // host.run()
    assert step >= host.run()                                   # no pair is looked at twice
    assert (runs - 1) * step + host.run() <= pairs
