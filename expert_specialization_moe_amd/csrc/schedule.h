// Tile schedule of the persistent grouped GEMM: how one expert's M x N output is
// cut into workgroup tiles and how a linear work-item index maps back to a tile.
//
// This takes the place of the reference's three M-bucket problem lists
// (expert_specialization/csrc/cuda/es_fp8_blockwise_functor.cuh:121-256): instead
// of routing whole experts to one of three differently tiled kernels, every
// expert is cut into full "big" row tiles plus one remainder tile whose height is
// the smallest menu entry that covers the leftover rows (sched_cover_mt,
// sched_last_mt), and all tiles of all experts feed one persistent kernel.
//
// The same functions compile for the device (hipcc) and for the host (plain C++),
// so the index math is unit-tested on the CPU.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define ESMOE_HD __host__ __device__ __forceinline__
#else
#define ESMOE_HD inline
#endif

namespace esmoe {

// Row-tile heights are MT * 16 rows with MT in {1, 2, 4, 8, 12} (sched_valid_mt), with runs also 6 and 10; a workgroup tile
// is (MT * 16) rows by 256 columns.
struct SchedPolicy {
  int force_mt;   // 0 = choose per expert; else every tile uses this MT
  int big_mt;     // MT of the full tiles of a many-row expert (8 or 12)
  int order;      // 0: heavy experts by rows ascending, light ones descending (sched_order_key); 1: expert index order;
                  // 2: most rows first for both kinds
  int light_share;  // workgroups (of every 32) that start on the light items; -1 = from the cost estimate
  int narrow_tail;  // the last so many light items are handed out as two 128-column halves each (0: none)
  int narrow_fit;   // 1, 2: only where halves fill idle workgroups (sched_halves_fit; 1: of a launch of one round)
  int runs;         // 1: the queues hold runs of tiles instead of blocks, and last row tiles come in steps of 32 rows (sched_use_runs)
};

struct TileCoord {
  int mt;  // tile height / 16
  int nt;  // tile width / 64
  int m0;  // first row inside the expert
  int n0;  // first column
};

// a / b for 0 <= a <= 3 * 2^29 (more rows than the card has memory for), b > 0.  On the device an integer division by a
// variable is a chain of some forty instructions, and the schedule of an expert with more than 64 rows takes three of them in
// front of the first tile, every heavy ticket six.  The float quotient is off by less than 2^9, that of what it leaves by less
// than one, and the last remainder says which way.  `inverse`: 1 / b, up to one unit in the last place off either way.
ESMOE_HD int sched_div_by(int a, int b, float inverse) {
  const int q = (int)((float)a * inverse), left = (int)((uint32_t)a - (uint32_t)q * (uint32_t)b);
  const int more = (int)((float)left * inverse), r = left - more * b;
  return q + more + (r >= b ? 1 : 0) - (r < 0 ? 1 : 0);
}
ESMOE_HD int sched_div(int a, int b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return sched_div_by(a, b, __builtin_amdgcn_rcpf((float)b));
#else
  return a / b;
#endif
}

// The tile heights that can be forced (the kernels also have 6 and 10: sched_last_mt).
ESMOE_HD bool sched_valid_mt(int mt) { return mt == 1 || mt == 2 || mt == 4 || mt == 8 || mt == 12; }

// Smallest tile height of the menu {1, 2, 4, 8, 12} (x16 rows) that covers `rows`, at most max_mt.
ESMOE_HD int sched_cover_mt(int rows, int max_mt) {
  const int need = (rows + 15) / 16;
  int mt = 1;
  if (need > 1) mt = 2;
  if (need > 2) mt = 4;
  if (need > 4) mt = 8;
  if (need > 8) mt = 12;
  return mt < max_mt ? mt : max_mt;
}

// Height / 16 of the last row tile of a heavy expert, `rows` (1 .. 192) rows of it, where the queues hold runs: tall tiles in steps of 32
// rows.  What lies past the expert's rows is copied, read from LDS and multiplied like the rest: 8192 rows, 32 experts, 4096 x 7168
// (MXFP8) had 11 % of such rows with 128 and 192 alone and has 6 %, 297.6 -> 292.6 us, of 6579 rows (FP8) 266.6 -> 262.7.  Up to 64 rows a
// short tile costs less than a tall one (K = 1536: 64 rows 15.3 us, 96 or 128 rows 17 us).
ESMOE_HD int sched_last_mt(int rows) { return rows > 64 ? (rows + 31) >> 5 << 1 : sched_cover_mt(rows, 4); }

// Every compiled shape is 256 columns wide (NT = 4 units of 64).
ESMOE_HD int sched_nt_for(int, const SchedPolicy&) { return 4; }

ESMOE_HD int sched_ntiles(int n, int nt) { return (n + nt * 64 - 1) / (nt * 64); }

// ---- XCD-aware hand-out ------------------------------------------------------------------
// The 256 CUs sit in 8 XCDs with one L2 each, and workgroup i of a launch runs on XCD i % 8.  Tiles
// of one expert that share token rows or weight rows should therefore run at the same time on the
// same XCD: every expert with more than 64 rows ("heavy") has its tile grid cut into blocks of
// up to 32 tiles (one per CU of an XCD, at most kBlkM tiles high), block b of the launch belongs to XCD b % 8, and the
// workgroups of an XCD draw tickets from that XCD's counter: ticket t is tile t % 32 of the XCD's
// (t / 32)-th block.  A dense 6144 x 4096 x 7168 problem fetches 302 MB into L2 this way against
// 557 MB with tiles handed out in plain order.  Tickets that fall outside the grid (edge blocks) are
// skipped.  An XCD that runs out of blocks helps the others.  Experts with at most 64 rows ("light")
// have one short tile per 256 columns that streams its weights once; nothing is shared, and they come
// from one launch-wide counter.  Heavy tiles are bound by the LDS feed of the matrix cores and light
// items by HBM, so the two kinds run side by side: a share of the workgroups (sized by the cost
// estimates below) starts on the light items while the rest start on the heavy tickets, and each
// side moves on to the other kind when its own runs out.
constexpr int kBlkM = 8;
constexpr int kBlkLog = 5, kBlkTiles = 1 << kBlkLog;
constexpr int kXcds = 8;

ESMOE_HD bool sched_is_heavy(int m, const SchedPolicy& p) { return p.force_mt ? m > 0 : m > 64; }

// Sort key of the hand-out order (smallest first, ties by expert index).  The heavy experts and the light ones are
// handed out from separate queues, so only the order inside each kind matters.  Light items: most rows first, the
// longest items first.  Heavy experts: fewest rows first (order 0): the launch then ends on the tiles of the experts with
// the most rows, many of which share an operand panel behind an L2, where an expert of few rows streams its own weights.  Measured
// against most rows first (order 2): where the queues hold runs, 36 drawn launches of more than a round of heavy tiles -2.8 % (-13 to
// +0.2), 153 of experts of about the same size -0.4 % (-9 to +13); as blocks, where an expert of one block also ended on a single
// queue, C4 -2.5 %, C3 at 2048 tokens -1.8 %, C1 and C3 at 8192 tokens -0.3 to -0.8 %.
ESMOE_HD int sched_order_key(int m, const SchedPolicy& p) {
  if (p.order == 2 || !sched_is_heavy(m, p)) return (1 << 30) - m;
  return m;
}

// Row tiles of an expert: full big tiles plus one remainder tile.
ESMOE_HD int sched_mtiles(int m, const SchedPolicy& p) {
  const int rows = (p.force_mt ? p.force_mt : p.big_mt) * 16;
  return sched_div(m + rows - 1, rows);
}

// ---- Runs --------------------------------------------------------------------------------
// From K = 640 on the queues hold runs instead of blocks: all heavy tiles of the launch stand in one line, expert after expert, each
// down its columns (of at most eight tiles), and queue x has the x-th, (x + 8)-th, ... run of 32 of them.  Every ticket is a tile: blocks
// leave holes where they have fewer than 32 tiles, and a hole costs a draw and a look-up, 2 to 3 us.  32 tiles that stand together
// are 4 columns of eight tiles to 32 of one, so what an XCD works on at a time are a few weight panels and the token rows of mostly one
// expert, however many of its workgroups are on heavy tiles; a block of 6 x 4 tiles leaves eight of them to the next one, of other rows.
// (Nothing holds a column's tiles together: a run ends inside one where 32 is no multiple of its height, 191 of 286 times with 131072
// rows, 128 experts, 3072 x 4096, and the column's panel then goes through two L2s, 0.2 GB in all.)  Fetched into L2
// (MB): 131072 rows, 128 experts, 3072 x 4096 5400 -> 3870, 6579 rows, 32 experts, 4096 x 7168 1470 -> 1250, 4012 rows (MXFP8) 1255 -> 1100.  us:
// 1646 -> 1596, 257.4 -> 251.3, 204.0 -> 197.2; 44 experts, 11384 rows, 768 x 640 (MXFP8) 29.0 -> 16.4, 10 experts, 974 rows, 4096 x 1024
// 26.2 -> 16.7; 110 drawn shapes of K = 640 to 7168 1.11 times as fast.  Row by row instead of down the columns: -2 % on the large
// launches; one run of an eighth of the launch per queue: +0.4 % on these, -0.6 % on the drawn ones.
// Slower than blocks are launches of one to four rounds of heavy experts of about the same size, two row tiles each: tall and short tiles
// alternate in a column, and where a few tiles are left for another round half of them are tall ones, while a block, laid row by row,
// ends on the short row.  us, blocks / runs: 12 experts x 367 rows, 2816 x 3712 (MXFP8) 62.9 / 72.8, 24 x 194 rows, 2304 x 768 (MXFP8,
// fused) 28.8 / 33.1, 22 x 256 rows, 3072 x 7040 199 / 204; but 28 x 232 rows, 2304 x 768 35.3 / 27.7, 100 x 201 rows, 512 x 1152 36.5 /
// 32.6.  420 drawn launches of that kind 1.02 times as fast as with blocks (0.86 to 1.27), one in five more than 2 % slower.  Tried on
// these: row by row -0.3 %, runs of equal length +0.2 %, most rows first -0.4 %, all last row tiles behind the others -6 % (a column's
// panel is then read twice).
// Up to K = 512 the queues hold blocks.  That line is not one of speed: the host mirrors and their tests hold such schedules.  53 drawn
// launches of K = 128 to 512 with heavy experts are 1.10 times as fast with runs (0.92 to 1.86): those of few tiles gain most (11 experts,
// 2234 rows, 2688 x 256 MXFP8 19.9 / 10.7 us), FP8 ones of many rounds lose (62552 rows, 175 experts, 4480 x 512 327 / 353).
ESMOE_HD bool sched_use_runs(int k) { return k > 512; }
// Tiles of a run: 32, one per CU of an XCD.  In launches of at most 512 an eighth or a sixteenth of them, so that the queues hold one or
// two runs each and about as many tiles.
ESMOE_HD int sched_run_tiles(int tiles) {
  constexpr int kAll = kXcds * kBlkTiles;
  return tiles > 2 * kAll ? kBlkTiles : tiles > kAll ? (tiles + 2 * kXcds - 1) / (2 * kXcds) : (tiles + kXcds - 1) / kXcds;
}

// Block shape for an expert with mtl x ntl tiles: at most kBlkM tiles high and kBlkTiles tiles in all, with
// the rows and the columns of the grid split evenly over the blocks (21 x 16 tiles -> blocks of 7 x 4;
// 6 x 16 -> 6 x 4; 1 x 16 -> 1 x 16).  Near-square blocks (in bytes) fetch the least per tile.
// rb = ceil(mtl / 8) rows of blocks are bm = ceil(mtl / rb) <= 8 tiles high, and since mtl > 8 (rb - 1) >= bm (rb - 1) it takes all
// rb of them; the same for the columns.
struct SchedBlocks {
  int bm, rb;      // tiles of a block's column, rows of blocks
  int width, cb;   // most tiles of a block's row, columns of blocks (a block's row: sched_block_cols)
};
ESMOE_HD SchedBlocks sched_block_shape(int mtl, int ntl) {
  static_assert(kBlkM == 8 && kBlkTiles == 32, "the table of widths");
  SchedBlocks b;
  b.rb = (mtl + kBlkM - 1) / kBlkM;
  b.bm = sched_div(mtl + b.rb - 1, b.rb);
  b.width = (int)(0x04040506080a1020ull >> ((b.bm - 1) * 8)) & 0xff;   // kBlkTiles / bm for bm = 1 .. 8
  b.cb = sched_div(ntl + b.width - 1, b.width);
  return b;
}
ESMOE_HD int sched_block_cols(const SchedBlocks& b, int ntl) { return sched_div(ntl + b.cb - 1, b.cb); }

ESMOE_HD int sched_heavy_blocks(int m, int n, const SchedPolicy& p) {
  if (!sched_is_heavy(m, p)) return 0;
  const SchedBlocks b = sched_block_shape(sched_mtiles(m, p), sched_ntiles(n, 4));
  return b.rb * b.cb;
}

// No block of a heavy expert has more tiles.  (Exact with one column of blocks; with several a block has at least half as many.)
ESMOE_HD int sched_block_tiles(int m, int n, const SchedPolicy& p) {
  const int ntl = sched_ntiles(n, 4);
  const SchedBlocks b = sched_block_shape(sched_mtiles(m, p), ntl);
  return b.bm * (ntl < b.width ? ntl : b.width);
}

ESMOE_HD int sched_light_items(int m, int n, const SchedPolicy& p) {
  return (m > 0 && !sched_is_heavy(m, p)) ? sched_ntiles(n, 4) : 0;
}

// Tile `idx` (0..31) of block `lb` of a heavy expert; false if it falls outside the expert's grid (`past`: and so do the block's
// tickets behind it).
ESMOE_HD bool sched_decode_heavy(int lb, int idx, int m, int n, const SchedPolicy& p, TileCoord* t, bool* past) {
  const int mtl = sched_mtiles(m, p), ntl = sched_ntiles(n, 4);
  const SchedBlocks b = sched_block_shape(mtl, ntl);
  const int bm = b.bm, bn = sched_block_cols(b, ntl);
  const int rb = sched_div(lb, b.cb), rows = mtl - rb * bm < bm ? mtl - rb * bm : bm;   // (the last row of blocks may be lower)
  *past = idx >= rows * bn;
  if (*past) return false;
  const int r = sched_div(idx, bn);
  const int mi = rb * bm + r, ni = (lb - rb * b.cb) * bn + idx - r * bn;
  if (ni >= ntl) return false;
  const int big = p.force_mt ? p.force_mt : p.big_mt;
  const int m0 = mi * big * 16;
  t->mt = p.force_mt ? p.force_mt : m - m0 >= big * 16 ? big : sched_cover_mt(m - m0, big);
  t->nt = 4;
  t->m0 = m0;
  t->n0 = ni * 256;
  return true;
}

constexpr int kRunRows = 192;   // row tiles of a launch whose queues hold runs
ESMOE_HD int sched_run_mtiles(int m) { return (m + kRunRows - 1) / kRunRows; }
ESMOE_HD int sched_heavy_tiles(int m, int n) { return sched_run_mtiles(m) * sched_ntiles(n, 4); }
// Most rows behind a first full tile that make two tall tiles of the expert's rows, of 128 and of 96 or 128, where 192 rows would leave a
// short one to the rest.  For launches of up to 256 heavy tiles, all of one round: it lasts as long as its longest tile, and a short tile
// beside a tall one, on the same panel, lasts longer than a tall one; for up to 512 from K = 4096 on (84 FP8 launches of 216 to 256 rows an
// expert, 512 to 2560 columns, K = 4096 to 7168 1.08 times as fast, 0.975 to 1.22: 3 % slower 24 experts x 248 rows, 2560 x 5120, 1 to 1.5 %
// 40 x 240 to 256 rows, 1024 x 7168).  `tiles`: of the launch.
// us, 192 + rest against two tall tiles, 2048 columns.  14 experts x 208 rows MXFP8: K = 7168 66.1 / 43.8, K = 3200 35.5 / 26.3, K = 1024
// 18.0 / 15.1; FP8: K = 7168 67.1 / 54.2, K = 3200 32.4 / 28.2, K = 2176 23.1 / 22.4, K = 2048 21.7 / 21.7.  14 x 256 rows MXFP8: K = 3200
// 33.8 / 27.3, K = 1024 14.8 / 15.2; FP8: K = 4096 36.6 / 35.5, K = 3968 35.6 / 35.8.  Two rounds, 32 experts: x 208 rows MXFP8 K = 7168
// 154.9 / 134.9, K = 4096 90.3 / 79.2, K = 3200 64.1 / 65.1, K = 2048 45.3 / 49.0; FP8 K = 4096 94.3 / 86.0; x 256 rows MXFP8 K = 4096
// 89.8 / 86.2, K = 3200 60.4 / 69.6, FP8 K = 4096 92.9 / 91.8.  Past two rounds what counts is the sum of the work: 100 experts x 256
// rows, 1024 x 4096 fused 165.5 / 179.3, 131072 rows, 128 experts, 3072 x 4096 1600 / 1610 (with experts of any size).
ESMOE_HD int sched_pair_rows(int tiles, int k, bool mx) {
  constexpr int kRound = kXcds * kBlkTiles;
  if (k >= 4096) return tiles <= 2 * kRound ? 64 : 0;
  return tiles > kRound ? 0 : mx && k > 3072 ? 64 : mx || k > 2048 ? 32 : 0;
}
// First row of an expert's last row tile.
ESMOE_HD int sched_run_last_row(int m, int mtl, int pair_rows) {
  return mtl == 2 && m - kRunRows <= pair_rows ? kRunRows - 64 : (mtl - 1) * kRunRows;
}
ESMOE_HD float sched_run_cost(int m, int n) {
  const int tiles = sched_run_mtiles(m), above = (tiles - 1) * kRunRows;
  return (float)(above + sched_last_mt(m - above) * 16 + 16 * tiles) * (float)sched_ntiles(n, 4);
}
// Tile `local` of an expert of m rows.
ESMOE_HD TileCoord sched_decode_run(int local, int m, int n, int pair_rows) {
  const int mtl = sched_run_mtiles(m), ntl = sched_ntiles(n, 4);
  int rows = mtl, left = local, first = 0;   // of the row of blocks: tiles of a column, the tile's place, its first row tile
  if (mtl > kBlkM) {
    const int rbs = (mtl + kBlkM - 1) / kBlkM, bm = sched_div(mtl + rbs - 1, rbs), rb = sched_div(local, bm * ntl);
    first = rb * bm;
    left -= first * ntl;
    rows = mtl - first < bm ? mtl - first : bm;
  }
  const int ni = sched_div(left, rows), mi = first + left - ni * rows;
  TileCoord t;
  const int last = sched_run_last_row(m, mtl, pair_rows);
  t.m0 = mi < mtl - 1 ? mi * kRunRows : last;
  t.mt = mi < mtl - 2 ? kRunRows / 16 : mi < mtl - 1 ? (last - t.m0) >> 4 : sched_last_mt(m - last);
  t.nt = 4;
  t.n0 = ni * 256;
  return t;
}

// Light items are handed out whole (256 columns) except the last `narrow_tail` of the launch, which go out as two
// 128-column halves each: a launch ends on light items (they are the last of the light-first workgroups' queue, and
// what the others turn to when the heavy tickets are gone), fewer of them are left than there are workgroups, and an
// item holds a CU for as long as a tall tile, so halves spread the end of the launch over twice the CUs.
// Where a draw takes several tickets (sched_light_draw, K of up to 1024 in launches of many items) most halves of the tail
// come out of one draw together and run as the whole tile again (sched_strip_tiles); only what a draw begins or ends with
// stays a half.
// Tickets [0, split) are the whole items 0 .. split-1, tickets split + 2j and split + 2j + 1 the halves of item split + j.
//
// A fused launch's halves (MXFP8) are not much shorter than its whole items: both read all token rows, quantise and write.  They pay
// only where they fill workgroups that would have nothing to do (`fit`, SchedPolicy::narrow_fit).  us, whole / halves:
//   in a launch of one round of workgroups without heavy tiles where all halves are one round too: 52 items, K = 1536 14.5 / 11.1; 112,
//     K = 1920 17.6 / 14.0; 100, K = 512 8.3 / 7.8; K = 128 5.8 / 5.9, not taken.  But 133 items, K = 1280 14.5 / 20.4, 189, K = 2944 29.5 /
//     35.0; and beside heavy tiles, which last longer than any item, 18 + 126, K = 1280 22.1 / 25.7;
//   in a longer one, from K = 1024 on, where up to half a round is left for the end: 264 items, K = 6784 108.0 / 90.7, 48 heavy tiles and
//     222 items, K = 6016 96.4 / 86.2.  But 60 + 370 (174 left), K = 5632 106.8 / 112.8, 429 items (173), K = 4096 75.7 / 81.3; K = 768, 1290
//     items 65.3 / 67.4;
//   where a whole round of tall tiles runs before the items, whatever is left: 400 + 272, K = 7168 213.0 / 206.5, 1044 + 1152, K = 4096
//     376.3 / 372.2.
// 284 drawn fused launches of K = 128 to 7168 1.11 times as fast as with whole items (0.99 to 1.60); halves in every one 1.07 (0.68 to 1.60).
ESMOE_HD bool sched_halves_fit(int items, int heavy, int fit) {   // `heavy`: heavy tiles
  constexpr int kRound = kXcds * kBlkTiles;
  if (items + heavy <= kRound) return heavy == 0 && 2 * items <= kRound;
  const int last = (items + heavy) % kRound;
  return fit > 1 && (heavy >= kRound || (last > 0 && 2 * last <= kRound));
}
ESMOE_HD int sched_light_split(int items, int heavy, int fit, const SchedPolicy& p) {
  const int narrow = fit && !sched_halves_fit(items, heavy, fit) ? 0 : p.narrow_tail < items ? p.narrow_tail : items;
  return items - (narrow > 0 ? narrow : 0);
}
ESMOE_HD int sched_light_item_of_ticket(int ticket, int split, int* half) {
  if (ticket < split) {
    *half = -1;
    return ticket;
  }
  *half = (ticket - split) & 1;
  return split + ((ticket - split) >> 1);
}

// Light tickets that a workgroup takes with one draw, when the last light ticket it saw was `seen` (0 at first): half its
// share of what was left then, within bounds that go by the item's length in K blocks.  Neighbouring tickets of one expert run
// as one strip (grouped_gemm.hip, gemm_tile), so the upper bound is also a strip's: 32 K blocks, 1 MB of weights.  Longer
// strips put the workgroups' streams further apart in memory and run slower: 64 experts x 8 rows, upper bound 16 / 32 / 64 /
// 256 blocks: K = 256 209 / 206 / 219 / 220 us, K = 1024 187 / 181 / 189 / 189 us (single tickets: 282 and 190 us).  The lower
// bound is 16 K blocks, for launches that give every workgroup two such draws: below it the draw and the first stages'
// trip from memory, about 5 us, outweigh the even end of the launch.  The whole share instead of half: up to 15 % slower.
// `strips`: false in the kernels with a fused epilogue, which walk every tile by itself: several tickets at once only make the
// end of their launch uneven (SwiGLU + 1x128 quantisation, 64 experts x 48 rows, 7168 x 512: 73 us with single tickets, 82
// with up to eight).
// All quotients are by the next power of two: a division is a chain of some forty instructions, and this stands in front of
// a workgroup's first tile.
constexpr int kStripBlocks = 32;
ESMOE_HD int sched_log2_ceil(int v) { return v > 1 ? 32 - __builtin_clz((unsigned)v - 1) : 0; }
ESMOE_HD int sched_light_draw(int total, int seen, int workgroups, int kblocks, bool strips) {
  if (!strips) return 1;
  const int lk = sched_log2_ceil(kblocks), lw = sched_log2_ceil(workgroups) + 1;
  const int most = kStripBlocks >> lk;
  int least = (kStripBlocks / 2) >> lk;
  if (least > total >> lw) least = total >> lw;
  int draw = (total - seen) >> lw;
  if (draw < least) draw = least;
  if (draw > most) draw = most;
  return draw > 1 ? draw : 1;
}

// Short 256-column tiles (and strips of them) store their output through a buffer descriptor of the tile's rows: 32-bit byte
// offsets from row m0, and whatever lies at or past the descriptor's size is dropped.  So the size has to be exact, every
// offset of a row past the last must stay past it, and a wavefront whose columns do not exist (the absent half of a last
// tile of 128 columns, which would land in the next row) gets a descriptor of size 0.  64 rows fit 32 bits up to
// n = 2^25; wider outputs, beyond 2^24, take 64-bit addresses and one tile at a time.
constexpr int kMaxStripN = 1 << 24;
ESMOE_HD bool strip_by_buffer(int n) { return n <= kMaxStripN; }
ESMOE_HD uint32_t strip_buffer_bytes(int rows, int n, bool wave_active) { return wave_active ? (uint32_t)rows * (uint32_t)n * 2 : 0; }
ESMOE_HD uint32_t strip_buffer_offset(int row, int n, int col) { return ((uint32_t)row * (uint32_t)n + (uint32_t)col) * 2; }

// Whole column tiles that run as one strip from light ticket `v` on (half `half` of column tile `local` of its expert): the
// tickets in hand, up to `end`, that are whole items of the expert, or both halves of such.  0: the ticket is a half by itself;
// a 128-column last tile is never part of a strip.
ESMOE_HD int sched_strip_tiles(int v, int end, int split, int local, int n, int half) {
  int tiles = half < 0 ? (end < split ? end : split) - v : half == 0 ? (end - v) >> 1 : 0;
  if (tiles > (n >> 8) - local) tiles = (n >> 8) - local;
  if (tiles > 1 && !strip_by_buffer(n)) tiles = 1;
  return tiles > 0 ? tiles : 0;
}

// Item `item` of a light expert; half = -1: the whole 256-column item, 0 / 1: its first / second 128 columns.
ESMOE_HD TileCoord sched_decode_light(int item, int m, const SchedPolicy& p, int half = -1) {
  TileCoord t;
  t.mt = sched_cover_mt(m, p.big_mt);
  t.nt = half < 0 ? 4 : 2;
  t.m0 = 0;
  t.n0 = item * 256 + (half > 0 ? 128 : 0);
  return t;
}

// Cost estimates in units of one tile row streamed through a CU: a heavy tile costs its padded rows; a light
// item is bound by streaming its 256 weight rows (and its few token rows) from HBM at one CU's rate, which
// takes as long as about 75 rows of a heavy tile.
ESMOE_HD float sched_heavy_cost(int m, int n, const SchedPolicy& p) {
  if (!sched_is_heavy(m, p)) return 0;
  const int big = (p.force_mt ? p.force_mt : p.big_mt) * 16, tiles = sched_mtiles(m, p), above = (tiles - 1) * big;
  const int rows = above + (p.force_mt ? big : sched_cover_mt(m - above, p.big_mt) * 16);
  return (float)(rows + 16 * tiles) * (float)sched_ntiles(n, 4);
}
ESMOE_HD float sched_light_cost(int m, int n, const SchedPolicy& p) {
  return (float)sched_light_items(m, n, p) * (float)(75 + m / 3);
}
// `run_tiles`: heavy tiles where the queues hold runs.  Up to 256 of them are all first tickets, and of a launch of about two rounds half: a
// tall tile drawn when the other workgroups end theirs is the longest end a launch can have, and where nothing is drawn from the
// heavy queues no workgroup has to look at all of them when the light items are used up.  106 experts, 6462 rows, 768 x 7168 (99 heavy
// tiles) 148.4 -> 121.9 us, 64 experts, 4131 rows, 1536 x 1024 (132) 38.8 -> 29.6, 66 experts, 13232 rows, 1536 x 1536 (384) 71.9 -> 62.0, 32
// experts, 256 rows, 7168 x 2048 (28) 77.2 -> 74.3.
// Workgroups of every 32 that start on the light items.  (Floats: it is an estimate, and a 64-bit division and sum of both costs
// stood 0.8 us in front of the first tile.)
ESMOE_HD int sched_light_share(float heavy_cost, float light_cost, int run_tiles, const SchedPolicy& p) {
  if (p.light_share >= 0) return p.light_share > 32 ? 32 : p.light_share;
  if (heavy_cost <= 0 || light_cost <= 0) return 0;
  if (run_tiles > 0) {
    const int tiles = (run_tiles + kXcds - 1) / kXcds;
    if (tiles <= kBlkTiles) return kBlkTiles - tiles;
    const float rounds = (float)run_tiles * (heavy_cost + light_cost) / (heavy_cost * (kXcds * kBlkTiles));
    if (rounds < 2.75f && tiles <= 2 * kBlkTiles) return kBlkTiles - (tiles + 1) / 2;
  }
  return (int)(32 * light_cost / (heavy_cost + light_cost) + 0.5f);
}

// Heavy ticket `ticket` of XCD `xcd` -> launch-wide block index (the caller compares it with the block total).
ESMOE_HD int sched_ticket_block(int xcd, int ticket) { return (ticket / kBlkTiles) * kXcds + xcd; }

// Tickets of XCD `xcd`'s queue when the launch has `hblocks` heavy blocks: queue x holds the blocks x, x + 8, ..., 32 tickets each.
ESMOE_HD int sched_queue_tickets(int xcd, int hblocks) { return xcd < hblocks ? (hblocks - xcd + kXcds - 1) / kXcds * kBlkTiles : 0; }

// Where the queues hold runs, queue x holds the runs x, x + 8, ... and every ticket is a tile: ticket -> tile of the launch, tickets of
// a queue.  (Runs of less than 32 tiles: a queue has no more than two.)
ESMOE_HD int sched_run_tile(int xcd, int ticket, int run) {
  const int q = run == kBlkTiles ? ticket / kBlkTiles : ticket >= run ? 1 : 0;
  return (q * kXcds + xcd) * run + ticket - q * run;
}
ESMOE_HD int sched_run_tickets(int xcd, int tiles, int run) {
  const int round = kXcds * run, full = run == kBlkTiles ? tiles / (kXcds * kBlkTiles) : tiles >= round ? 1 : 0;   // rounds of all queues
  const int left = tiles - full * round - xcd * run;
  return full * run + (left < 0 ? 0 : left < run ? left : run);
}

// Queue that a workgroup draws heavy tickets from when it has found `step` queues empty: first the one its first ticket is of, the
// queue of its XCD (the hardware deals the workgroups of a launch out in turn, workgroup i to XCD i % 8), then the others in turn.
// That the first draw is from the queue of the first ticket is more than locality: see sched_next_block.
ESMOE_HD int sched_home_queue(int workgroup) { return workgroup % kXcds; }
ESMOE_HD int sched_drawn_queue(int workgroup, int step) { return (sched_home_queue(workgroup) + step) % kXcds; }

// What a queue's counter has to be at least when the tickets behind `ticket` in its block are no tiles (0 or less: nothing to do, the
// rest of the block is not drawn from the counter).  Raising the counter is an atomic maximum that nobody waits for.  It must
// have happened before the workgroup counts itself out, since the last one out zeroes the counters; it has, because the workgroup
// goes on with a draw from the same queue, an add to the same address by the same thread, and waits for that.
ESMOE_HD int sched_next_block(int ticket, int heavy_base) { return (ticket / kBlkTiles + 1) * kBlkTiles - heavy_base; }

// First tickets: a workgroup's first ticket goes by its index, and the counters hand out what lies behind these.  Atomic adds to
// one address are served one every 12 ns, so 256 workgroups that all begin with a draw wait 3 us for the last of them, and as
// long again to count themselves out; a launch whose tickets are all first ones needs neither.
// `heavy_ranks`: the workgroups 8 r + x with r below it start on queue x, the others on the light tickets, `light_draw` neighbouring
// ones each.  Where no block of the launch has more than 16 tiles (`block_log`: sched_log2_ceil of the most), a queue's first workgroups
// take the tiles of its first `blocks` blocks, a power of two of tickets of each, and nobody draws the rest of those blocks' tickets,
// which are no tiles; otherwise they take the tickets of its first block.  When the later blocks had to be drawn a queue's 32
// workgroups stood in line for them, and many found no tile: 14 experts, 1717 rows, 2944 x 1536 27.3 -> 23.6 us, 10 experts,
// 1602 rows, 768 x 3072 44.7 -> 40.1, 18 experts, 9341 rows, 768 x 4864 49.7 -> 46.9; launches of larger blocks pay some 0.1 us
// for the look.
struct SchedFirst {
  int heavy_ranks;
  int blocks, share_log;   // a first workgroup r of a queue: ticket r % 2^share_log of block r >> share_log, if below `blocks`
  int heavy_base;          // first ticket of a queue that is drawn from its counter
  int light_draw;
  int light_base;          // first light ticket that is
};
ESMOE_HD SchedFirst sched_first_tickets(int workgroups, int hblocks, int block_log, int ltotal, int light_share, int light_draw) {
  SchedFirst f;
  const int per_xcd = workgroups / kXcds;
  if (hblocks == 0) f.heavy_ranks = 0;
  else if (ltotal == 0) f.heavy_ranks = per_xcd;   // (the workgroups past a multiple of eight begin with a draw)
  else f.heavy_ranks = ((kBlkTiles - light_share) * per_xcd + kBlkTiles - 1) / kBlkTiles;
  f.share_log = block_log;
  f.blocks = f.heavy_ranks >> f.share_log;
  f.heavy_base = f.blocks * kBlkTiles;
  if (block_log >= kBlkLog || f.blocks == 0) {
    f.share_log = 31;   // one block, as many tickets of it as there are workgroups
    f.blocks = 1;
    f.heavy_base = f.heavy_ranks;
  }
  f.light_draw = light_draw;
  const int light_first = workgroups - f.heavy_ranks * kXcds;
  f.light_base = light_first > 0 ? light_first * light_draw : 0;
  return f;
}
ESMOE_HD bool sched_first_is_light(int workgroup, const SchedFirst& f) { return workgroup >= f.heavy_ranks * kXcds; }
// First ticket of `workgroup`, of the light ones or of queue workgroup % 8; may lie past the last ticket there is.
ESMOE_HD int sched_first_ticket(int workgroup, const SchedFirst& f) {
  if (sched_first_is_light(workgroup, f)) return (workgroup - f.heavy_ranks * kXcds) * f.light_draw;
  const int r = workgroup / kXcds, block = r >> f.share_log;
  return block < f.blocks ? block * kBlkTiles + (r - (block << f.share_log)) : 0x7fffffff - kBlkTiles;
}
// Last light ticket that `workgroup` knows of before its first draw (`seen` of sched_light_draw): its own first one if that is a
// light one; a heavy ticket says nothing about the light queue.
ESMOE_HD int sched_first_seen(int workgroup, const SchedFirst& f) { return sched_first_is_light(workgroup, f) ? sched_first_ticket(workgroup, f) : 0; }
// Queues that hold nothing but first tickets: bits 0-7 the XCDs' queues, bit 8 the light tickets (all nine: no counter is used).
constexpr int kAllQueues = (1 << (kXcds + 1)) - 1;
ESMOE_HD int sched_undrawn_queues(int hblocks, int ltotal, const SchedFirst& f) {
  // a queue of b blocks has 32 b tickets: the queues with no more than `rounds` blocks, and they come last
  const int rounds = f.heavy_base / kBlkTiles, more = hblocks - rounds * kXcds;   // blocks past that many rounds of all queues
  const int drawn = more <= 0 ? 0 : more < kXcds ? more : kXcds;
  return (f.light_base >= ltotal ? 1 << kXcds : 0) | (((1 << kXcds) - 1) & ~((1 << drawn) - 1));
}

// First K block of an expert's K order.  With K a multiple of 4096 all rows of a weight panel share address bits 7-11: a K block of a
// tile goes through one L2 channel of sixteen, and tiles that all begin with block 0 stay in step and queue for one channel
// after the other (128 experts x 8 rows: 768 x 4096 88.3 us in step, 68.6 apart; 4096 x 4096 337 and 325; the projection of a 64-token
// expert MLP with hidden size 4096 19 us less).  So every expert begins at a place of its own, a multiple of four K blocks in the first
// 32, and wraps; large launches, bound by the matrix cores, take as long either way.  The place goes by the expert's weight scales,
// so that its bytes depend on its rows and weights alone, not on where or among which others it is listed: a hash of the differences
// between its first scales (four fp32 block scales, or sixteen E8M0 bytes as four words), which a common power of two in all
// scales does not change.  Equal scales: block 0.  One place for all columns, since a tile of 256 has one K loop: a call on a part of
// the expert's weight rows takes the same order only if it begins with the same row.
ESMOE_HD bool sched_spread_k(int k) { return (k & 4095) == 0; }
constexpr int kStartUnit = 4;
ESMOE_HD int sched_k_start(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t s3) {   // in units of kStartUnit K blocks
  uint32_t h = (s1 - s0) * 0x9e3779b1u;
  h = ((h << 13 | h >> 19) ^ (s2 - s0)) * 0x85ebca6bu;
  h = ((h << 13 | h >> 19) ^ (s3 - s0)) * 0xc2b2ae35u;
  h = (h ^ h >> 16) * 0x7feb352du;
  return (int)(h >> 29);
}

// Workspace layout (int32 words).
constexpr int kWsLightCounter = 32;  // next light ticket to hand out (every counter has a 128-byte line of its own)
constexpr int kWsLightTotal = 1;     // number of light tickets: whole items, then two per item of the narrow tail
constexpr int kWsHeavyBlocks = 2;    // number of heavy blocks (runs: of 32 tiles)
constexpr int kWsLightShare = 3;     // workgroups of every 32 that start on the light items
constexpr int kWsLightSplit = 4;     // first light ticket that is a half item (sched_light_split)
constexpr int kWsBlockLog = 5;       // sched_log2_ceil of the most tiles of a heavy block (sched_block_tiles)
constexpr int kWsRun = 6;            // tiles of a run (sched_run_tiles), 0: the queues hold blocks
constexpr int kWsExitCounter = 16;   // workgroups of the launch that have left the hand-out loop: the last one zeroes every counter
constexpr int kWsXcdCounter = 64;    // next heavy ticket of XCD x at word kWsXcdCounter + 32 * x (ws_xcd_counter)
constexpr int kWsHeader = 64 + 32 * kXcds;   // then one record of kRecWords per schedule position, E + 1 of them
// Record of schedule position p: first heavy block (runs: first heavy tile), first light item, expert index, rows (clamped at 0).
// Record E closes the prefix sums: {heavy blocks (tiles), light items, -1, 0}.
constexpr int kRecWords = 4;
constexpr int kRecBlock = 0, kRecItem = 1, kRecExpert = 2, kRecRows = 3;
// The expert's word also holds where its K order starts (sched_k_start).
ESMOE_HD int rec_expert_word(int expert, int k_start) { return expert | k_start << 16; }
ESMOE_HD int rec_expert(int word) { return word & 0xffff; }
ESMOE_HD int rec_first_kb(int word) { return (word >> 16) * kStartUnit; }
ESMOE_HD int ws_xcd_counter(int xcd) { return kWsXcdCounter + 32 * xcd; }
ESMOE_HD int ws_rec(int pos) { return kWsHeader + pos * kRecWords; }
ESMOE_HD int ws_words(int num_experts) { return kWsHeader + (num_experts + 1) * kRecWords; }

// One launch per call: when the counters of a workspace are known to be zero (a workspace the library owns: it is
// zeroed when it is allocated, and the last workgroup to leave a launch zeroes the counters again), the GEMM kernel
// needs no schedule kernel in front of it: every workgroup ranks the experts, builds the records itself and writes them (the same
// values from every workgroup) for its own scalar loads.  Up to 64 experts its first wavefront does so alone, a lane for an expert,
// while the others wait (wave_schedule), past that all of its 512 threads (self_schedule), so no more experts than that.
constexpr int kWaveScheduleMaxExperts = 64;
constexpr int kSelfScheduleMaxExperts = 512;

}  // namespace esmoe
