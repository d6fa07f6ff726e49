"""Index functions of schedule.h that the short tiles and their strips use, compiled for the host.

The output of a short tile leaves through a buffer descriptor with 32-bit offsets: every element of the tile's rows must be
stored where 64-bit arithmetic puts it, and everything else (rows past the expert's last, the absent half of a last column
tile of 128 columns) must be dropped.  A draw of light tickets is at most a strip long, and however the workgroups' draws
fall, the strips and single tiles cut from them cover every column of every expert once.
"""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "schedule.h"
using namespace esmoe;
extern "C" {
int by_buffer(int n) { return strip_by_buffer(n); }
unsigned buffer_bytes(int rows, int n, int active) { return strip_buffer_bytes(rows, n, active != 0); }
int draw(int total, int seen, int workgroups, int kblocks, int strips) { return sched_light_draw(total, seen, workgroups, kblocks, strips != 0); }
int strip_tiles(int v, int end, int split, int local, int n, int half) { return sched_strip_tiles(v, end, split, local, n, half); }
int item_of_ticket(int ticket, int split, int* half) { return sched_light_item_of_ticket(ticket, split, half); }
unsigned buffer_offset(int row, int n, int col) { return strip_buffer_offset(row, n, col); }
}
"""


def schedule_functions(folder):
    (folder / "host.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(folder / "host.cpp"), "-o", str(folder / "host.so")], check=True)
    lib = ctypes.CDLL(str(folder / "host.so"))
    lib.buffer_bytes.restype = lib.buffer_offset.restype = ctypes.c_uint
    return lib


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    return schedule_functions(tmp_path_factory.mktemp("host"))


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


def light_tickets(native, rows, n, kind=0):
    """(light tickets of a launch, the first that is a half item, records [experts + 1, 4]) from the host mirror."""
    e = len(rows)
    ps = np.array([[m, n, 512] for m in rows], dtype=np.int32)
    ws = np.zeros(native.lib.esmoe_gemm_workspace_bytes(e) // 4, dtype=np.int32)
    rc = native.lib.esmoe_host_schedule(ps.ctypes.data_as(ctypes.c_void_p), e, n, 0, kind, ws.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0, native.last_error()
    first = 64 + 32 * 8
    return int(ws[1]), int(ws[4]), ws[first:first + 4 * (e + 1)].reshape(e + 1, 4)


@pytest.mark.parametrize("n,k,experts", [(128, 128, 9), (256, 128, 300), (384, 128, 900), (640, 256, 256), (3200, 128, 200), (4224, 128, 512),
                                         (7168, 256, 256), (7168, 2048, 32), (2176, 384, 160), (16384, 128, 130)])
@pytest.mark.parametrize("workgroups", [3, 256])
def test_strips_cover_every_column_once(host, n, k, experts, workgroups):
    """The hand-out loop's light side with the workgroups' draws in random order."""
    from expert_specialization_moe_amd import _native

    rng = random.Random(n + k + experts)
    rows = [rng.choice((0, 1, 16, 33, 64, 300)) for _ in range(experts)]
    total, split, rec = light_tickets(_native, rows, n)
    firsts = rec[:, 1]
    cover = np.zeros((experts, n // 128), dtype=np.int32)
    half = ctypes.c_int()
    counter, active, longest, crossing = 0, [[0, w] for w in range(workgroups)], 1, 0
    while active:
        i = rng.randrange(len(active))
        draw = host.draw(total, active[i][0], workgroups, k // 128, 1)
        v, counter = counter, counter + draw
        if v >= total:
            active.pop(i)
            continue
        active[i][0] = v
        end, experts_of_draw = min(v + draw, total), set()
        while v < end:
            idx = host.item_of_ticket(v, split, ctypes.byref(half))
            pos = int(np.searchsorted(firsts[:experts], idx, side="right")) - 1
            e, local, m = int(rec[pos, 2]), idx - int(firsts[pos]), int(rec[pos, 3])
            assert 0 < m <= 64 and 0 <= local < (n + 255) // 256
            experts_of_draw.add(e)
            h = half.value
            tiles = host.strip_tiles(v, end, split, local, n, h)
            if tiles > 1 or (h >= 0 and tiles):
                assert (local + tiles) * 256 <= n and (tiles == 1 or tiles * k <= 32 * 128)
            if h < 0:
                cols, used, first, width = max(tiles, 1), max(tiles, 1), local * 2, 2 * max(tiles, 1)
            elif tiles:
                cols, used, first, width = tiles, 2 * tiles, local * 2, 2 * tiles
            else:
                cols, used, first, width = 1, 1, local * 2 + h, 1
            cover[e, first:min(first + width, n // 128)] += 1
            longest = max(longest, cols)
            v += used
        assert v == end
        crossing += len(experts_of_draw) > 1
    for e, m in enumerate(rows):
        assert (cover[e] == (1 if 0 < m <= 64 else 0)).all(), e
    if workgroups == 3 and k < 2048 and n >= 512:
        assert longest > 1 and (crossing > 0 or n * k >= 4096 * 1024)


def test_tiles_of_very_wide_outputs_are_no_strips(host):
    n = (1 << 24) + 256
    assert host.strip_tiles(0, 8, 100, 0, n, -1) == 1 and host.strip_tiles(100, 108, 100, 0, n, 0) == 1
    assert host.strip_tiles(0, 8, 100, 0, 1 << 24, -1) == 8
