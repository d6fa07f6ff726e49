"""First tickets (schedule.h, sched_first_tickets), compiled for the host.

A workgroup's first ticket goes by its index and the counters hand out what lies behind: together they give every light ticket
and every ticket of every XCD's queue that may be a tile once, whatever the kinds, the share, the tiles of a block and the number
of workgroups, and a queue is named undrawn exactly where nothing lies behind.
"""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "schedule.h"
using namespace esmoe;
extern "C" {
int queue_tickets(int xcd, int hblocks) { return sched_queue_tickets(xcd, hblocks); }
int first(int wgs, int hblocks, int block_tiles, int ltotal, int share, int draw, int wg, int* light, int* heavy_base, int* light_base, int* undrawn) {
  const SchedFirst f = sched_first_tickets(wgs, hblocks, sched_log2_ceil(block_tiles), ltotal, share, draw);
  *light = sched_first_is_light(wg, f);
  *heavy_base = f.heavy_base;
  *light_base = f.light_base;
  *undrawn = sched_undrawn_queues(hblocks, ltotal, f);
  return sched_first_ticket(wg, f);
}
int seen(int wgs, int hblocks, int block_tiles, int ltotal, int share, int draw, int wg) {
  return sched_first_seen(wg, sched_first_tickets(wgs, hblocks, sched_log2_ceil(block_tiles), ltotal, share, draw));
}
int home_queue(int wg) { return sched_home_queue(wg); }
int drawn_queue(int wg, int step) { return sched_drawn_queue(wg, step); }
int next_block(int ticket, int heavy_base) { return sched_next_block(ticket, heavy_base); }
int light_draw(int total, int seen, int workgroups, int kblocks) { return sched_light_draw(total, seen, workgroups, kblocks, true); }
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("first")
    (folder / "host.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(folder / "host.cpp"), "-o", str(folder / "host.so")], check=True)
    return ctypes.CDLL(str(folder / "host.so"))


@pytest.mark.parametrize("workgroups", [1, 7, 8, 9, 255, 256, 304])
def test_first_and_drawn_tickets_cover_every_ticket_once(host, workgroups):
    rng = random.Random(workgroups)
    out = [ctypes.c_int() for _ in range(4)]
    refs = [ctypes.byref(o) for o in out]
    cases = [(0, 0), (0, 1), (1, 0), (0, workgroups), (0, workgroups + 1), (8, 0), (9, 0), (16, 0), (17, 0), (7, 5), (8, 400), (40, 2000)]
    cases += [(rng.randrange(80), rng.randrange(1500)) for _ in range(40)]
    for hblocks, ltotal in cases:
        share, draw = rng.randrange(33) if hblocks and ltotal else 0, rng.choice((1, 1, 2, 5, 14, 32))
        tiles = rng.choice((1, 2, 3, 5, 8, 9, 16, 17, 24, 32))   # of a block: its first tickets, the others are no tiles
        queues = [host.queue_tickets(x, hblocks) for x in range(8)]
        assert sum(queues) == 32 * hblocks
        light, heavy = [0] * ltotal, [[0] * q for q in queues]
        for wg in range(workgroups):
            t = host.first(workgroups, hblocks, tiles, ltotal, share, draw, wg, *refs)
            assert t >= 0
            if out[0].value:
                for v in range(t, min(t + draw, ltotal)):
                    light[v] += 1
            elif t < queues[wg % 8]:
                heavy[wg % 8][t] += 1
        heavy_base, light_base, undrawn = (o.value for o in out[1:])
        for v in range(light_base, ltotal):
            light[v] += 1
        for q in heavy:
            for v in range(heavy_base, len(q)):
                q[v] += 1
        assert all(c == 1 for c in light), (hblocks, ltotal, share, draw)
        assert all(c == 1 or (c == 0 and t % 32 >= tiles) for q in heavy for t, c in enumerate(q)), (hblocks, tiles, ltotal, share)
        want = (256 if light_base >= ltotal else 0) | sum(1 << x for x in range(8) if heavy_base >= queues[x])
        assert undrawn == want


def test_a_heavy_first_ticket_says_nothing_about_the_light_queue(host):
    """A workgroup that starts on a heavy ticket has seen no light one, whatever the ticket's number (also where it gets none: of a
    queue's 24 workgroups the last eight, behind one block of 16 tiles), and its first light draw is that of a workgroup that has seen nothing;
    one that starts on light tickets has seen its own."""
    out = [ctypes.c_int() for _ in range(4)]
    refs = [ctypes.byref(o) for o in out]
    for hblocks, tiles, ltotal, share, draw in ((90, 16, 4000, 8, 4), (16, 32, 4000, 8, 4), (300, 4, 2000, 20, 1), (1, 1, 500, 16, 2)):
        none = 0
        for wg in range(256):
            ticket = host.first(256, hblocks, tiles, ltotal, share, draw, wg, *refs)
            seen = host.seen(256, hblocks, tiles, ltotal, share, draw, wg)
            none += ticket > 1 << 30
            assert seen == (ticket if out[0].value else 0), (wg, ticket, seen)
            if not out[0].value:
                assert host.light_draw(ltotal, seen, 256, 1) == min(max(ltotal >> 9, 1), 32)
        assert none == (64 if tiles == 16 else 0)


def test_a_raised_counter_is_drawn_from_next(host):
    """The counter of a heavy queue is raised past a block's empty tickets by an atomic that only the workgroup's next draw waits for.  So
    that draw must be from the same queue, also behind a first ticket, and a queue that is never drawn from must never be raised."""
    for wg in range(256):
        assert host.drawn_queue(wg, 0) == host.home_queue(wg)
        assert sorted(host.drawn_queue(wg, step) for step in range(8)) == list(range(8))
    out = [ctypes.c_int() for _ in range(4)]
    refs = [ctypes.byref(o) for o in out]
    rng = random.Random(3)
    raised = 0
    for workgroups in (1, 8, 100, 256, 304, 512):
        for hblocks in [1, 2, 7, 8, 9, 16, 17, 64, 65] + [rng.randrange(1, 200) for _ in range(20)]:
            ltotal = rng.choice((0, 1, 300))
            share, tiles = rng.randrange(33) if ltotal else 0, rng.choice((1, 2, 3, 5, 8, 9, 16, 17, 24, 31))
            for wg in range(workgroups):
                t = host.first(workgroups, hblocks, tiles, ltotal, share, 1, wg, *refs)
                light, heavy_base, _, undrawn = (o.value for o in out)
                queue = host.home_queue(wg)
                if light or t >= host.queue_tickets(queue, hblocks):
                    continue
                raise_to = host.next_block(t, heavy_base)
                assert raise_to + heavy_base == (t // 32 + 1) * 32
                raised += raise_to > 0
                assert raise_to <= 0 or not undrawn >> queue & 1, (workgroups, hblocks, tiles, ltotal, share, wg)
    assert raised
