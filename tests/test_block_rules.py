"""Which transposed views are moved in skewed blocks and in strips of blocks, and which streamed chunks
run in line: the rules of csrc/axr_internal.h, compiled on their own."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include "axr_internal.h"
using namespace axr;
int main() {
  unsigned e, square, tensor_lines, payload_lines;
  unsigned long long a, b, payload;
  while (std::scanf("%u %llu %llu %u %llu %u %u", &e, &a, &b, &square, &payload, &tensor_lines, &payload_lines) == 7) {
    const BlockRule r = block_rule(e, a, b, square, payload, tensor_lines, payload_lines);
    std::printf("%d%d%d\n", r.strips, r.skew_pack, r.skew_unpack);
  }
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rule")
    src, exe = str(folder / "rule.cpp"), str(folder / "rule")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src, "-o", exe], check=True, timeout=120)

    def ask(cases):
        """[(element bytes, A, B, MiB, tensor rows on lines, payload rows on lines)] -> [(strips, pack, unpack)]"""
        edge = {1: 128, 2: 64, 4: 32, 8: 32, 16: 16}
        lines = "".join(f"{e} {a} {b} {int(a >= edge[e] and b >= edge[e])} {int(mib * (1 << 20))} {t} {p}\n"
                        for e, a, b, mib, t, p in cases)
        out = subprocess.run([exe], input=lines, capture_output=True, text=True, check=True, timeout=60).stdout.split()
        assert len(out) == len(cases)
        return [tuple(c == "1" for c in o) for o in out]
    return ask


def test_small_bundles_and_whole_lines_stay_plain(rule):
    cases = [(e, 2001, 2003, mib, t, p) for e in (1, 2, 4, 8, 16)
             for mib, t, p in ((8, 0, 0), (26, 0, 0), (28 - 2 * (e == 8), 1, 0), (200, 1, 1))]
    assert set(rule(cases)) == {(False, False, False)}


def test_short_rows_are_not_skewed(rule):
    """Rows of little more than a block, where staging the neighbour's elements costs up to 40 %."""
    for mib in (33, 70, 190):
        cases = [(e, 300001, b, mib, 0, 0) for e, short in ((2, (65, 101, 211, 511)), (4, (33, 41, 101, 211, 1023)),
                                                             (8, (33, 41, 101, 127))) for b in short]
        cases += [(e, n, n, mib, 0, 0) for e, n in ((2, 422), (4, 298), (4, 705), (8, 119))]     # batches of small matrices
        assert set(rule(cases)) == {(False, False, False)}


def test_large_matrices_are_skewed_on_the_side_that_straddles_lines(rule):
    for e in (2, 4, 8):
        for mib in (29 - 2 * (e == 8), 34, 134):
            both, tensor_odd, payload_odd = rule([(e, 2001, 2003, mib, 0, 0), (e, 2048, 2003, mib, 0, 1),
                                                  (e, 2001, 2048, mib, 1, 0)])
            assert both[1:] == (True, True) and tensor_odd[1:] == (False, True) and payload_odd[1:] == (True, False)
            assert both[0] == tensor_odd[0] == (mib > 96) and payload_odd[0]
    assert {r[1:] for r in rule([(e, 2001, 2003, 134, 0, 0) for e in (1, 16)])} == {(False, False)}


def test_strips_where_b_is_long_or_the_cache_is_left(rule):
    """Long B: strips from 28 MiB on (8-byte elements 26), very long ones from 24; else 16-byte elements, and flat ones at no
    size."""
    assert all(r[0] for r in rule([(e, 211, 4001, mib, 0, 0) for e in (2, 4, 8, 16) for mib in (29, 70, 190)]))
    assert all(r[0] for r in rule([(e, 211, 6007, mib, 0, 0) for e in (2, 4, 8, 16) for mib in (25, 70, 190)]))
    assert not any(r[0] for r in rule([(e, 211, b, mib, 0, 0) for e in (2, 4, 8, 16) for b, mib in ((4001, 26), (6007, 24))]))
    # a short A beyond 192 MiB: only with a very long B
    assert [r for e in (2, 4, 8) for r in rule([(e, 72, 4001, 193, 0, 0)])] == [(False, False, False)] * 3
    assert all(r[0] for r in rule([(e, a, b, mib, 0, 0) for e in (2, 4, 8) for a, b, mib in ((72, 6007, 230), (72, 4001, 192), (150, 4001, 230))]))
    assert not any(r[0] for r in rule([(16, 1459, 1461, 70, 0, 0), (16, 30001, 801, 190, 0, 0), (16, 1456, 1461, 190, 0, 1),
                                       (1, 211, 90001, 190, 0, 0)]))
    assert rule([(16, 1459, 1461, 190, 0, 0)])[0][0]
    # one dimension shorter than a square block
    assert [r[0] for r in rule([(e, 12, 90001, 70, 0, 0) for e in (1, 2, 4, 8, 16)])] == [False] * 4 + [True]


def test_plane_blocks_do_not_overlap(tmp_path):
    """Every element of a plane belongs to one block, but for the last block's end, which may reach
    less than a vector beyond the extent (and is moved back by that much)."""
    source = r"""
#include "axr_internal.h"
using namespace axr;
constexpr bool covered(uint32_t e, uint32_t planes) {
  for (uint64_t extent = kVecBytes / e; extent < 6000; ++extent) {
    const uint64_t edge = plane_edge(e, planes, extent), blocks = (extent + edge - 1) / edge;
    if (edge % (kVecBytes / e) != 0 || edge * e > plane_rounds(e, planes) * kRowBytes) return false;
    if (blocks == 1 && edge - extent >= kVecBytes / e) return false;
  }
  return true;
}
static_assert(covered(1, 2) && covered(1, 3) && covered(1, 4), "bytes");
static_assert(covered(2, 2) && covered(2, 3) && covered(2, 4), "2-byte elements");
static_assert(covered(4, 2) && covered(4, 3) && covered(4, 4), "4-byte elements");
static_assert(in_planes(1, 16) && !in_planes(1, 15) && in_planes(4, 201) && !in_planes(4, 200) && !in_planes(8, 4096), "range");
"""
    src = str(tmp_path / "planes.cpp")
    with open(src, "w") as f:
        f.write(source)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-fconstexpr-ops-limit=100000000", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src], check=True, timeout=120)


def test_short_blocks_of_planes(tmp_path):
    """In blocks of one round on the side that was measured to be faster: (element bytes, planes, elements of a plane, MB, alone)."""
    short = [(1, 3, 50176, 37, 1), (1, 3, 7501, 24, 1), (1, 4, 30011, 40, 1), (1, 4, 3072, 256, 1), (1, 3, 50176, 300, 1), (2, 3, 7501, 180, 1),
             (2, 3, 3563, 24, 1), (1, 3, 50176, 9, 0), (1, 4, 7501, 10, 0), (2, 3, 32400, 4, 0), (2, 3, 7501, 36, 0), (2, 3, 7501, 130, 0),
             (2, 3, 50176, 3500, 0)]
    two = [(1, 3, 7501, 180, 1), (1, 4, 7501, 300, 1), (1, 4, 50000, 64, 1), (1, 2, 42000, 25, 1), (2, 4, 16256, 17, 1), (2, 2, 40000, 10, 1),
           (4, 3, 50176, 38, 1), (1, 3, 50176, 38, 0), (1, 3, 38190, 15, 0), (1, 4, 50176, 40, 0), (2, 3, 32400, 19, 0), (2, 3, 32400, 28, 0), (2, 2, 3000, 2, 0),
           (2, 3, 3000, 300, 1), (2, 3, 809, 298, 1), (2, 3, 3000, 36, 0),
           (2, 3, 50177, 3500, 0), (2, 3, 5000, 3500, 0), (2, 3, 20001, 2300, 0), (2, 3, 20001, 6000, 0)]
    checks = "".join(f"static_assert({no}plane_short_blocks({e}, {c}, {n}, {mb}000000ull, {alone}), \"{e} {c} {n} {mb} {alone}\");\n"
                     for cases, no in ((short, ""), (two, "!")) for e, c, n, mb, alone in cases)
    src = str(tmp_path / "short.cpp")
    with open(src, "w") as f:
        f.write('#include "axr_internal.h"\nusing namespace axr;\n' + checks)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src], check=True, timeout=120)


def test_chunks_in_line(tmp_path):
    """On the side that was measured to be faster, for sizes where the two differ by more than 4 %."""
    turn = [(2, 2, 136), (2, 2, 148), (3, 3, 94), (3, 3, 105), (4, 4, 68), (4, 4, 84), (4, 2, 136), (6, 3, 84), (2, 2, 269),
            (2, 2, 537), (3, 3, 336), (8, 8, 16)]
    line = [(2, 2, 164), (2, 2, 175), (2, 2, 268), (3, 3, 116), (4, 4, 105), (6, 6, 105), (4, 2, 148), (6, 3, 110), (2, 1, 16),
            (8, 1, 600), (1, 1, 16)]
    checks = "".join(f"static_assert({no}chunks_in_line({mb}000000ull, {lanes}, {streams}, 256ull << 20), \"{lanes} {streams} {mb}\");\n"
                     for cases, no in ((turn, "!"), (line, "")) for lanes, streams, mb in cases)
    src = str(tmp_path / "line.cpp")
    with open(src, "w") as f:
        f.write('#include "axr_internal.h"\nusing namespace axr;\n' + checks)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src], check=True, timeout=120)


def test_row_slots(tmp_path):
    """Rows of every length from every start: the slots of its 64-byte units cover a row, a tile holds two rows
    at least and no more than its lanes and its LDS, and the payload pieces of a tile fit theirs."""
    source = r"""
#include "axr_internal.h"
using namespace axr;
constexpr bool fits(uint64_t run, uint32_t start, bool mixed) {
  const uint32_t slots = row_slots(run, start), lanes = row_slots_per_lane(slots, mixed) * kWaveLanes, rows = lanes / slots;
  if (slots % 4 != 0 || slots * kVecBytes < start + run || rows < 2 || rows * slots > lanes) return false;
  if ((kUnitBytes - 1 + rows * run + kVecBytes - 1) / kVecBytes > lanes + kWaveLanes) return false;
  return kUnitBytes - 1 + rows * run <= rows_lds_bytes(static_cast<uint32_t>(rows), run) && rows_lds_bytes(rows, run) <= 16384;
}
constexpr bool all(uint32_t start, bool mixed) {
  for (uint64_t run = kVecBytes; run <= kMaxRowBytes; ++run)
    if (!fits(run, start, mixed)) return false;
  return true;
}
constexpr bool every_start(bool mixed) {
  for (uint32_t start = 0; start < kUnitBytes; ++start)
    if (!all(start, mixed)) return false;
  return true;
}
static_assert(every_start(false) && every_start(true), "rows");
"""
    src = str(tmp_path / "rows.cpp")
    with open(src, "w") as f:
        f.write(source)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-fconstexpr-ops-limit=200000000", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src], check=True, timeout=120)


def test_row_rule(tmp_path):
    """The slots a row gets cover it, a tile holds two rows at least and no more than its lanes and its LDS, and the
    payload pieces of a tile fit theirs, for every length, every start, both sides and payloads of every class."""
    source = r"""
#include "axr_internal.h"
using namespace axr;
constexpr bool fits(uint64_t run, uint64_t pitch, uint32_t start, bool receiver, uint64_t payload, bool streams) {
  const RowRule r = row_rule(run, pitch, start, receiver, payload, streams);
  const uint32_t lanes = r.per_lane * kWaveLanes, rows = lanes / r.slots;
  if (r.per_lane < 2 || r.per_lane > kMaxRowSlots || r.slots < 2 || r.slots * kVecBytes < run || rows < 2) return false;
  if ((kUnitBytes - 1 + rows * run + kVecBytes - 1) / kVecBytes > lanes + kWaveLanes) return false;
  return kUnitBytes - 1 + rows * run <= rows_lds_bytes(rows, run) && rows_lds_bytes(rows, run) <= 16384;
}
constexpr bool all() {
  for (uint64_t run = kVecBytes; run <= kMaxRowBytes; ++run)
    for (uint64_t pitch : {run, run + 1, run + 64, uint64_t(0), uint64_t(1) << 40})
      for (uint32_t start : {0u, 1u, 16u, 48u, 63u})
        for (uint64_t payload : {uint64_t(1), kRowUnitsPayload, kRowCachedPayload, kRowFilledPayload, uint64_t(1) << 38})
          for (int receiver = 0; receiver < 2; ++receiver)
            if (!fits(run, pitch, start, receiver != 0, payload, false) || !fits(run, pitch, start, receiver != 0, payload, true)) return false;
  return true;
}
static_assert(all(), "rows");
constexpr bool is(RowRule r, uint32_t slots, uint32_t per_lane) { return r.slots == slots && r.per_lane == per_lane; }
constexpr uint64_t M = 1 << 20;
// rows of one to two units: slots for a start on a unit whatever the start is
static_assert(is(row_rule(72, 73, 63, false, 32 * M, false), 8, 4) && is(row_rule(72, 73, 63, false, 200 * M, false), 8, 2));
static_assert(is(row_rule(100, 101, 63, true, 100 * M, false), 8, 2) && is(row_rule(100, 128, 0, false, 100 * M, false), 8, 2));
static_assert(is(row_rule(64, 65, 63, true, 32 * M, false), 4, 2) && is(row_rule(130, 131, 63, false, 32 * M, false), 12, 3));
// longer ones: slots for the worst start on the side that is written and where the payload streams
static_assert(is(row_rule(200, 201, 63, false, 100 * M, false), 16, 2) && is(row_rule(200, 201, 63, true, 100 * M, false), 20, 2));
static_assert(is(row_rule(200, 201, 63, true, 12 * M, false), 16, 2) && is(row_rule(200, 201, 63, false, 300 * M, true), 20, 2));
static_assert(is(row_rule(256, 292, 60, false, 32 * M, false), 20, 2) && is(row_rule(128, 129, 63, false, 32 * M, false), 8, 2));
// where they cost no row of a tile
static_assert(is(row_rule(666, 667, 63, false, 32 * M, false), 48, 3) && is(row_rule(600, 601, 63, false, 32 * M, false), 40, 2));
// very short rows next to each other
static_assert(is(row_rule(16, 24, 56, false, 8 * M, false), 2, 2) && is(row_rule(36, 37, 63, true, 200 * M, false), 3, 3));
static_assert(is(row_rule(32, 64, 0, false, 12 * M, false), 2, 2) && is(row_rule(32, 64, 0, false, 100 * M, false), 4, 2) &&
              is(row_rule(32, 128, 0, false, 12 * M, false), 4, 2));
"""
    src = str(tmp_path / "rule.cpp")
    with open(src, "w") as f:
        f.write(source)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-fconstexpr-ops-limit=400000000", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src], check=True, timeout=240)


def test_rows_that_share_a_launch(tmp_path):
    """Many tiles of short rows share a launch with each other and not with bundles of other kinds; few do."""
    source = r"""
#include "axr_internal.h"
using namespace axr;
static_assert(rows_share_launch(uint64_t(1) << 40, false) && rows_share_launch(0, true));
static_assert(rows_share_launch(2048, true) && !rows_share_launch(2049, true));
"""
    src = str(tmp_path / "share.cpp")
    with open(src, "w") as f:
        f.write(source)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "execution-ucx_amd", "csrc"), src], check=True, timeout=120)
