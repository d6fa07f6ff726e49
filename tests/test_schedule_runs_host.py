"""The schedule of launches whose queues hold runs (K > 512), through its host mirror, and the statements of the 96- and 160-row tiles.
No GPU."""
import ctypes
import os
import random
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "expert_specialization_moe_amd", "csrc")


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _schedule(lib, rows, n, kind, k=640):
    ps = np.array([[m, n, k] for m in rows], dtype=np.int32)
    ws = np.zeros(lib.esmoe_gemm_workspace_bytes(len(rows)) // 4, dtype=np.int32)
    assert lib.esmoe_host_schedule(_ptr(ps), len(rows), n, 0, kind, _ptr(ws)) == 0
    return ps, ws


@pytest.mark.parametrize("seed", range(8))
def test_every_ticket_is_a_tile_and_every_output_element_is_covered_once(esmoe, seed):
    """Numbers of heavy tiles around 256 and 512, where the length of a run changes; experts of more than eight row tiles, whose columns
    are cut; every height of a last row tile."""
    from expert_specialization_moe_amd import _native

    lib, rng = _native.lib, random.Random(seed)
    for rows, n in (([65, 96, 97, 128, 129, 160, 161, 192, 193, 208, 209, 224, 256, 257, 288, 289, 352, 384, 0, 64, 1, 1700], 768),
                    ([70] * (252 + seed) + [200, 256], 256), ([70] * (508 + seed) + [200, 256], 256), ([70] * (254 + seed), 256), ([70] * (510 + seed), 256), ([2000] * (3 + seed), 1280), ([5] * 9, 384),
                    ([rng.choice((0, rng.randrange(65), rng.randrange(65, 4000))) for _ in range(rng.randrange(1, 60))], 128 * rng.randrange(1, 30))):
        k = (640, 640, 2048, 3072, 2176, 3200, 3968, 4096)[seed]
        ps, ws = _schedule(lib, rows, n, seed % 4, k)
        tiles, out = int(ws[64 + 32 * 8 + 4 * len(rows)]), np.zeros(5, dtype=np.int32)
        cover = [np.zeros((m, n // 128), dtype=np.int32) for m in rows]
        queues = []
        for xcd in range(8):
            ticket = 0
            while True:
                rc = lib.esmoe_host_decode_heavy(_ptr(ps), _ptr(ws), len(rows), n, 0, seed % 4, xcd, ticket, _ptr(out))
                if rc == 2:
                    break
                e, bm, bn, m0, n0 = (int(v) for v in out)
                last = rows[e] - m0
                assert rc == 0 and rows[e] > 64 and bn == 256 and m0 % 64 == 0
                # (from 193 rows to 224 or 256: two tall tiles, the first of 128 rows; odd seeds are MXFP8)
                most = (64 if tiles <= 512 else 0) if k >= 4096 else 0 if tiles > 256 else 64 if k > 3072 and seed % 2 else 32 if k > 2048 or seed % 2 else 0
                two = 192 < rows[e] <= 192 + most
                want = 128 if two and m0 == 0 else 192 if last > 160 else -(-last // 32) * 32 if last > 64 else 16 if last <= 16 else 32 if last <= 32 else 64
                assert bm == want, (rows[e], m0, bm)
                cover[e][m0:m0 + bm, n0 // 128:(n0 + bn) // 128] += 1
                ticket += 1
            queues.append(ticket)
        assert sum(queues) == tiles == sum(-(-m // 192) * -(-n // 256) for m in rows if m > 64)
        assert max(queues) - min(queues) <= (32 if tiles > 512 else 15)   # of up to two runs the last one is at most so much shorter
        for e, m in enumerate(rows):
            assert (cover[e] == (1 if m > 64 else 0)).all(), (e, m)


def test_a_launch_of_one_round_starts_on_all_its_heavy_tiles(esmoe):
    """Word 3: workgroups of every 32 that start on the light items."""
    from expert_specialization_moe_amd import _native

    rows = [70] * 33 + [60] * 73      # 99 heavy tiles, 219 light items at n = 768
    _, ws = _schedule(_native.lib, rows, 768, 0)
    assert (32 - int(ws[3])) * 8 >= 99


def test_statements_of_three_and_five_row_tiles_follow_the_ring():
    """The checks that test_pp_bookkeeping.py and test_pp_lds_waits.py make of the other two, on these; the header is the generator's."""
    from tests import test_pp_bookkeeping as B
    from tests import test_pp_lds_waits as L

    gen = B._gen()
    for mtw in (3, 5):
        for mx in (False, True):
            for kb_count in (1, 2, 3, 4, 7, 57):
                B.test_statement_advances_its_operands_as_the_ring_prescribes(mx, mtw, kb_count)
        for fuse in (False, True):
            p, q = gen.Plan(mtw, fuse), gen.MxPlan(mtw, fuse)
            for name, lines in ((f"fp8 {mtw} {fuse}", gen.memory_phase(p) + gen.matrix_phase(p)), (f"mx {mtw} {fuse}", gen.mx_memory_phase(q) + gen.mx_matrix_phase(q))):
                L.test_barrier_waits_for_weight_slot_reads_and_mfmas_for_their_operands(name, lines)
                L.test_reads_left_out_at_the_first_barrier_are_the_groups_own(name, lines)
                last_roll = max(i for i, l in enumerate(lines) if l.startswith("ds_read_b128") and ("%[al]" in l or "%[ah]" in l))
                assert next(i for i, l in enumerate(lines) if l.startswith("v_add_u32 %[al]")) > last_roll
    out = subprocess.run([sys.executable, os.path.join(CSRC, "gen_pp_phase.py"), "odd"], capture_output=True, text=True, check=True).stdout
    assert out == open(os.path.join(CSRC, "pp_phase_odd.h")).read(), "pp_phase_odd.h is stale: python gen_pp_phase.py odd > pp_phase_odd.h"
