"""Index functions of schedule.h that the short tiles use, compiled for the host.

The output of a short tile leaves through a buffer descriptor with 32-bit offsets: every element of the tile's rows must be
stored where 64-bit arithmetic puts it, and everything else (rows past the expert's last, the absent half of a last column
tile of 128 columns) must be dropped.
"""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "schedule.h"
using namespace esmoe;
extern "C" {
int by_buffer(int n) { return strip_by_buffer(n); }
unsigned buffer_bytes(int rows, int n, int active) { return strip_buffer_bytes(rows, n, active != 0); }
int draw(int total, int seen, int workgroups, int kblocks, int strips) { return sched_light_draw(total, seen, workgroups, kblocks, strips != 0); }
unsigned buffer_offset(int row, int n, int col) { return strip_buffer_offset(row, n, col); }
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    (d / "host.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(d / "host.cpp"), "-o", str(d / "host.so")], check=True)
    lib = ctypes.CDLL(str(d / "host.so"))
    lib.buffer_bytes.restype = lib.buffer_offset.restype = ctypes.c_uint
    return lib


# 8388736: the first width with a last tile of 128 columns whose 64 rows end past 2^30 bytes
@pytest.mark.parametrize("n", [128, 384, 7168, 8388608, 8388736, (1 << 24) - 128, 1 << 24])
def test_stores_through_a_buffer_reach_their_element_or_are_dropped(host, n):
    assert host.by_buffer(n)
    row_tile = 16
    for rows in (1, 15, 16, 17, 33, 63, 64):
        for n0 in {0, (n - 1) // 256 * 256}:                  # the first and the last column tile
            for nw in range(0, 256, 32):                      # a wavefront's first column
                active = n0 + nw < n
                size = host.buffer_bytes(rows, n, active)
                for row in range(0, 64, row_tile):            # (a lane's row r, a tile's row mt * 16)
                    for r in (0, 1, 15):
                        for col in (0, 12, 28):               # four columns of a lane, 8 bytes
                            off = (host.buffer_offset(r, n, n0 + nw) + host.buffer_offset(row, n, col)) % (1 << 32)
                            exact = ((row + r) * n + n0 + nw + col) * 2
                            written = off + 8 <= size
                            assert written == (active and row + r < rows), (rows, n0, nw, row, r, col)
                            assert off == exact and (written or off >= size)


@pytest.mark.parametrize("n", [(1 << 24) + 128, 1 << 25, (1 << 31) - 128])
def test_wider_outputs_do_not_use_a_buffer(host, n):
    assert not host.by_buffer(n)


@pytest.mark.parametrize("kblocks", [1, 2, 3, 4, 5, 8, 11, 12, 16, 17, 31, 32, 33, 56, 256])
@pytest.mark.parametrize("workgroups", [1, 8, 255, 256, 304])
def test_a_draw_is_at_most_a_strip(host, kblocks, workgroups):
    for total in (1, 2, 15, 16, 255, 257, 1000, 7168, 1 << 20):
        for seen in sorted({0, 1, total // 3, total // 2, total - 1}):
            draw = host.draw(total, seen, workgroups, kblocks, 1)
            assert draw >= 1 and (draw == 1 or draw * kblocks <= 32)
            # no more than half a workgroup's share of what was left, but in a launch that has two such draws for everyone
            # tickets of up to 16 K blocks
            assert draw <= max(1, (total - seen) // (2 * workgroups), min(16 // kblocks, total // (2 * workgroups)))
            assert host.draw(total, seen, workgroups, kblocks, 0) == 1   # kernels without strips


def test_draws_at_benchmark_sizes(host):
    """256 workgroups; 256 experts x 7168 columns at K = 256, 70 x 8192 at K = 512, 32 x 7168 at K = 2048."""
    assert [host.draw(256 * 28, seen, 256, 2, 1) for seen in (0, 4000, 7000)] == [14, 8, 8]
    assert host.draw(70 * 32, 0, 256, 4, 1) == 4
    assert host.draw(32 * 28, 0, 256, 16, 1) == 1
