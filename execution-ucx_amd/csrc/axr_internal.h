// Internal declarations shared by the planner (host only), the runtime shim
// and the HIP kernels.  Nothing here is part of the C ABI.
#ifndef AXR_INTERNAL_H_
#define AXR_INTERNAL_H_

#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <new>
#include <string>
#include <vector>

#include "axon_rocm.h"

namespace axr {

// ---------------------------------------------------------------- device tables
//
// One pack or unpack is ONE kernel launch that walks a segment table resident
// in HBM.  A segment is one tensor (or one slice of a tensor with many strided
// outer dimensions); it is cut into tiles of at most kTileBytes that never
// cross a contiguous run, and tiles are numbered consecutively over the whole
// bundle.  Each wavefront owns a contiguous range of tile ids.

constexpr uint32_t kWaveLanes = 64;
constexpr uint32_t kVecBytes = 16;                           // one dwordx4 per lane
constexpr uint32_t kRowBytes = kWaveLanes * kVecBytes;       // 1 KiB per wave-wide access
constexpr uint32_t kMaxTileRows = 16;
constexpr uint32_t kMaxThreadsPerWorkgroup = 1024;
constexpr uint32_t kMaxElementThreads = 256;   // kernels that decode elements or transpose: more registers
constexpr uint32_t kXcds = 8;   // accelerator dies; workgroup i is dispatched to die i % 8
constexpr uint32_t kMaxOuterDims = 6;

constexpr uint32_t kSegPadMask = 0xfffu;         // meta bits 0..11: zero bytes after segment
constexpr uint32_t kSegDimsShift = 12;           // meta bits 12..31: 1 + dims index
constexpr uint32_t kSegFillOnly = 0xfffffu;      // dims field value: segment only writes zeros
constexpr uint32_t kSegGroup = 0xffffeu;         // dims field value: one tile that holds several short tensors
constexpr uint32_t kMaxAlign = 4096;
constexpr uint32_t kDirectSegShift = 0xffu;      // seg_shift value: every segment is exactly one tile
constexpr uint32_t kOneSegShift = 0xfdu;         // seg_shift value: one segment, a view moved otherwise than in runs
constexpr uint32_t kGroupBlocksShift = 0xfeu;    // seg_shift value: every tile is a group block at a fixed stride
// run_bytes of a contiguous (not strided) segment carries, in its top byte, the number
// of leading bytes (< 128) that tile 0 moves in addition to its own range: with them
// peeled off, every tile of the segment starts on a 128-byte line of the written side.
constexpr uint32_t kSegHeadShift = 56;
constexpr uint64_t kSegRunMask = (1ull << kSegHeadShift) - 1;
constexpr uint32_t kLineBytes = 128;

struct Seg {              // 32 bytes
  uint64_t ptr;           // tensor-side address of the first element
  uint64_t off;           // payload offset of the segment's first byte
  uint64_t run_bytes;     // bytes per contiguous run (whole segment when not strided)
  uint32_t tile_begin;    // id of the segment's first tile
  uint32_t meta;          // pad | (dims index + 1) << 12
};
static_assert(sizeof(Seg) == 32, "Seg layout");

// A group tile: several whole short contiguous tensors that follow each other in the bundle
// are moved by ONE wavefront.  Every group has a block of kGroupBlockBytes in the table block
// (behind the tile-block index): a GroupHead, then up to kGroupMaxMembers Member records.  The
// group's Seg carries, in `ptr`, the byte offset of that block from the start of the segment
// table.  A bundle that consists of group tiles only needs neither its Seg records nor the
// index on the device: tile t's block lies at t * kGroupBlockBytes (seg_shift ==
// kGroupBlocksShift; the kernel's `dims` argument then points at the blocks), which takes
// one dependent memory access out of every wavefront's path.
// A member of n bytes followed by `pad` zero bytes occupies max(1, ceil(n / 16)) data slots,
// then ceil(pad / 16) zero slots when pad >= 16; a slot is one 16-byte access of one lane, the
// last data (zero) slot covering the member's (gap's) final 16 bytes.  Members shorter than 16
// bytes and gaps shorter than 16 bytes move in pieces of 8, 4, 2 and 1 bytes in the lane of
// the member's last data slot.
constexpr uint32_t kGroupMaxMembers = 16;
constexpr uint32_t kGroupMaxSlots = 128;         // two 16-byte accesses per lane
constexpr uint32_t kGroupMaxMemberBytes = 1023;
struct Member {           // 16 bytes
  uint64_t ptr;           // tensor-side address
  uint32_t off_pad;       // bits 0-19: payload offset from the group's first byte; bits 20-31: pad
  uint16_t nbytes;        // 1 .. kGroupMaxMemberBytes
  uint16_t begin;         // first slot of the member
};
static_assert(sizeof(Member) == 16, "Member layout");
struct GroupHead {        // 32 bytes
  uint64_t starts[2];     // bit j of starts[r]: lane slot 64 r + j is the first slot of a member, so
                          // that a slot finds its member by counting bits instead of searching
  uint64_t off;           // payload offset of the group's first member
  uint32_t members;
  uint32_t slots;
};
static_assert(sizeof(GroupHead) == 32, "GroupHead layout");
// A group as the host stages it for the device to write its block: its members' records lie side
// by side in an array of their own.
struct GroupStage {       // 16 bytes
  uint64_t off;           // GroupHead.off
  uint32_t first;         // index of the first member's record
  uint16_t members, slots;
};
static_assert(sizeof(GroupStage) == 16, "GroupStage layout");
constexpr uint32_t kGroupBlockBytes = sizeof(GroupHead) + kGroupMaxMembers * sizeof(Member);   // 288
constexpr uint32_t kMemberOffBits = 20;
constexpr uint32_t group_data_slots(uint32_t nbytes) { return nbytes >= kVecBytes ? (nbytes + kVecBytes - 1) / kVecBytes : 1u; }
constexpr uint32_t group_pad_slots(uint32_t pad) { return pad >= kVecBytes ? (pad + kVecBytes - 1) / kVecBytes : 0u; }

constexpr uint32_t kModeRunTiles = 0;   // every tile is a piece of one contiguous run
constexpr uint32_t kModeElements = 1;   // tile covers packed bytes; lanes decode granules
// kModeRows and above: the tile goes through LDS
constexpr uint32_t kModeRows = 2;       // tile covers whole runs, cut on each side's own 64-byte boundaries
// kModeTranspose and above: the tile is a block transposed through LDS
constexpr uint32_t kModeTranspose = 3;  // plain blocks in plain rows
constexpr uint32_t kModeWalked = 4;     // skewed blocks, or blocks in strips (see block_rule)
constexpr uint32_t kModePlanes = 5;     // few planes against the same elements interleaved
// Kernels are built for the segments a bundle has: runs and groups of short tensors only, views of one
// mode above kModeRunTiles only (the kind is that mode), or anything.
constexpr uint32_t kKindRuns = 0, kKindAny = 6;

// Transposed blocks are T x T elements; a block row is 128 bytes (eight 16-byte
// vectors) for elements up to 4 bytes and 256 bytes for wider ones, so that a
// block is 4 to 16 KiB.  In LDS every row carries one dword of padding.
constexpr uint32_t transpose_edge(uint32_t element_bytes) {
  return (element_bytes <= 4 ? 128u : 256u) / element_bytes;   // 128, 64, 32, 32, 16
}
constexpr uint32_t transpose_lds_pitch(uint32_t element_bytes) {
  return transpose_edge(element_bytes) * element_bytes + 4u;
}
// Skewed blocks (2- to 8-byte elements; written rows that do not start on 64-byte boundaries) stage
// up to 64 / E - 1 more rows than a block has, rounded up to what one wave-wide access covers.
constexpr uint32_t kSkewBytes = 64;
constexpr uint32_t transpose_skew_rows(uint32_t element_bytes) {
  const uint32_t per_access = kWaveLanes / (transpose_edge(element_bytes) * element_bytes / kVecBytes);
  return (transpose_edge(element_bytes) + kSkewBytes / element_bytes - 1 + per_access - 1) / per_access * per_access;
}
// The four wavefronts of a workgroup in the kernel of walked blocks alone take kSkewGroup skewed blocks that follow
// each other along the written rows, and stage their rows together: the rows of the next block are staged once for
// four blocks.  The rows, rounded up to what a round of the four covers.
constexpr uint32_t kSkewGroup = 4;
constexpr uint32_t transpose_group_rows(uint32_t element_bytes) {
  const uint32_t round = kSkewGroup * (kWaveLanes / (transpose_edge(element_bytes) * element_bytes / kVecBytes));
  return (kSkewGroup * transpose_edge(element_bytes) + kSkewBytes / element_bytes - 1 + round - 1) / round * round;
}
constexpr uint32_t kBlockStrip = 8;
constexpr uint32_t kSkewPack = 16, kSkewUnpack = 32;   // Dims.nt_allowed bits 4, 5: blocks of that direction are skewed
// How the blocks of a transposition are cut and walked when rows straddle lines: plain or skewed
// blocks; in plain rows (along B, the dimension that is contiguous in the tensor, then along A, the one
// that is contiguous in the payload) or in strips of kBlockStrip blocks along A.  Microseconds are pack +
// unpack in turn, each pass on another of several copies, 1.2 GB in all.
//  - Bundles up to 28 MiB (8-byte elements 26), most of what the eight L2s hold, stay plain, partly written
//    lines are completed there (7379 x 989 2-byte elements, twice, 29.2 MB, 26.3 plain / 28.4 skewed; 29.7 MB
//    30.9 / 29.1, 34 MB of odd rows 41.9 / 40.0; 8-byte elements 26.4 MB 23.5 / 24.1, 28.3 MB 30.2 / 25.8; 400
//    shapes: means 1.01 of plain at 26 MB, 0.94 at 28, 0.91 from 30 MB on).
//  - Skewed blocks stage up to 1.5 times the elements they write, and twice as many where a row holds
//    little more than a block: both extents have to reach skew_min_row (70 MB in rows of 101 2-byte
//    elements 68 plain / 95 skewed, 100 matrices of 428 x 428 4-byte elements 62 / 68; one odd matrix of
//    70 MB 82 / 67, 4- and 8-byte elements 72 / 62 and 70 / 59).
//  - Strips bring blocks that share payload lines, neighbours along A, close to each other where B is long
//    (70 MB of 211 x n 4-byte elements 82 in plain rows / 64, 16-byte ones 77 / 68; very long ones from
//    24 MiB on: 72 x 16001 2-byte elements, 25.3 MB, 33.5 / 29.6, but 72 x 2003, 26.0 MB, 26.0 / 30.4, and
//    30.9 MB 36.6 / 34.9; beyond 192 MiB not where A is short and B not very long: 72 x 2003 2- and 4-byte
//    elements are 9 % behind plain rows at 240 MB, level and 8 % ahead at 130 MB) and where only the
//    payload's rows straddle lines (34 MB of 8-byte elements 34.0 / 32.8).
//    Elsewhere plain rows are ahead as long as the last-level cache holds most of a pass (45 MB, payload
//    rows on lines and odd tensor rows, 39.1 / 40.8; 16-byte elements 3 to 10 % up to 70 MB); beyond that
//    strips are (one odd matrix of 190 MB 198 / 188, 16-byte elements 188 / 171), save for 16-byte matrices
//    that are flat (1.02) or have their payload rows on lines (1.03).  128 x 128 blocks of bytes gain
//    nowhere, blocks shorter than a square one only with 16-byte elements (18 x n, 70 MB 82 / 66).
constexpr uint64_t kLongMinPayload = 24u << 20, kStripMinPayload = 96u << 20, kThinMaxPayload = 192u << 20;
constexpr uint64_t kLongRow = 6000, kThinRows = 128;
constexpr uint64_t skew_min_payload(uint32_t element_bytes) { return (element_bytes == 8 ? 26u : 28u) << 20; }
constexpr uint32_t skew_min_row(uint32_t element_bytes) {
  return element_bytes == 4 ? 1024u : element_bytes == 8 ? 128u : 512u;
}
struct BlockRule {
  bool strips = false, skew_pack = false, skew_unpack = false;
};
// `square`: blocks of transpose_edge x transpose_edge, otherwise one dimension is shorter than that.
constexpr BlockRule block_rule(uint32_t element_bytes, uint64_t ext_a, uint64_t ext_b, bool square, uint64_t payload_bytes,
                               bool tensor_lines, bool payload_lines) {
  BlockRule rule;
  if (tensor_lines && payload_lines) return rule;
  const uint64_t row = skew_min_row(element_bytes);
  const bool large = ext_a >= row && ext_b >= row && payload_bytes > skew_min_payload(element_bytes);
  const bool thin = ext_a < kThinRows && ext_b < kLongRow && payload_bytes > kThinMaxPayload;
  const bool long_b = element_bytes > 1 && ext_b >= row && ext_b / 4 >= ext_a && !thin &&
                      payload_bytes > (ext_b >= kLongRow ? kLongMinPayload : skew_min_payload(element_bytes));
  const bool beyond_cache = payload_bytes > kStripMinPayload;
  if (element_bytes == 16) {
    rule.strips = long_b || (square && large && beyond_cache && !payload_lines && ext_b >= ext_a / 2);
  } else if (square && element_bytes > 1 && (large || long_b)) {
    rule.strips = long_b || beyond_cache || tensor_lines;
    rule.skew_pack = !payload_lines && ext_a >= row;
    rule.skew_unpack = !tensor_lines;
  }
  return rule;
}
// Streamed chunks that the receiver borrows: in turn on their lanes' streams, or in line on one stream
// and slot.  Where the payloads of all streams fit the last-level cache, the overlap of two launches'
// ramps and tails is worth more than a slot that stays there, and where one alone does not, nothing stays
// either way.  In between the slots evict each other, but not before they exceed the cache by more than
// a launch that is just ending has left behind, and sooner where more lanes than streams take turns.
// Twelve chunks through kept plans, from the first submission to the end of the wait, in turn / in line in us
// (rows of 4 KiB; rows of 1 KiB and 64 KiB agree within 5 MB):
//   2 lanes, 2 streams: 136 MB 1005 / 1102, 153 MB 1187 / 1212, 158 MB 1263 / 1248, 175 MB 1509 / 1358
//   3, 3:               94 MB 722 / 825, 105 MB 853 / 899, 110 MB 931 / 928, 116 MB 1023 / 971
//   4, 4:               84 MB 729 / 760, 94 MB 810 / 829, 100 MB 886 / 867;  6, 6: 84 MB 744 / 764, 94 MB 855 / 837
//   4, 2:               136 MB 1048 / 1103, 142 MB 1106 / 1145, 148 MB 1259 / 1187;  6, 3: 94 MB 803 / 833, 105 MB 940 / 903
// 8 x 268 MB on two streams 1645 / 1340 (a plain copy of the bytes: 1282), 8 x 336 MB 1690 / 1719, 8 x 537 MB
// 2684 / 2695.
constexpr bool chunks_in_line(uint64_t nbytes, size_t lanes, size_t streams, uint64_t cache) {
  if (streams <= 1) return true;
  const uint64_t spare = lanes > streams ? cache / 24 : cache / 12;
  return nbytes <= cache && nbytes > cache / streams + spare && nbytes > cache / 20 * 7;
}
// When one of the two block dimensions is shorter than a square block's edge the
// block becomes a rectangle of about this many bytes, its long edge capped.
constexpr uint32_t kRectBlockBytes = 8192;
constexpr uint32_t kRectMaxEdge = 1024;
constexpr uint32_t kMinBlockBytes = 1024;   // smaller blocks than this are left to element mode
// Two to four planes of 1- to 4-byte elements against the same elements interleaved: a lane moves
// 16 bytes of every plane, a wavefront up to plane_rounds times that per lane.  Bytes and 2-byte
// elements take two rounds; 4-byte elements as many as the 8 KiB rectangle of the other blocks with
// a short dimension has (1024, 680 and 512 elements of each of 2, 3 and 4 planes).
constexpr uint32_t plane_rounds(uint32_t element_bytes, uint32_t planes) {
  return element_bytes < 4 || planes == 4 ? 2u : planes == 3 ? 3u : 4u;
}
// The elements of every plane that lie in one round.
constexpr uint32_t plane_round_elements(uint32_t element_bytes) { return kWaveLanes * kVecBytes / element_bytes; }
// Planes whose blocks have a routine of one round as well, for blocks that hold no more.
constexpr bool plane_single_round(uint32_t element_bytes, uint32_t planes) {
  return element_bytes < 4 && (planes == 3 || (planes == 4 && element_bytes == 1));
}
// Whether planes are moved in blocks of one round: a wavefront has less to do and needs less LDS, more of them run at once and the
// last of them end closer together, but there are twice as many, and twice as many ends of blocks that share a line (pack +
// unpack, blocks of two rounds / of one, unless said otherwise as a share of the time with two).
//  - Three planes of bytes alone, up to kShortBlocksMaxPayload: 256 images of 224 x 224 28.8 / 27.4 us, 3 MB 0.92 to 0.98,
//    24 MB 0.92 to 1.02, 40 MB 0.96 to 1.04, four planes 0.88 to 0.97, 0.92 to 1.05, 0.96 to 1.03.  Beyond that planes of whole
//    rounds only (300 MB of 50,176 x 3 204.6 / 199.4): 180 MB of 7501 x 3 151.1 / 157.9, 300 MB of 7501 x 4 222.9 / 252.9.
//  - Three planes of 2-byte elements alone likewise (24 MB of 3563 26.0 / 24.9), and beyond that those of kShortBlocksLongPlane
//    elements and more (180 MB of 7501 159.0 / 135.3, of 50,176 124.8 / 122.8, but 300 MB of 3000 227.0 / 234.2, of 809 packed and
//    unpacked in one launch 201.6 / 243.5).
//  - Next to other tensors, in the kernel for any mode, which holds 5 wavefronts on a SIMD whatever their LDS, where (nearly)
//    all of them run at once: with 1 MiB of compact tensor 1 MB 0.84 to 0.97, 3 MB 0.85 to 0.96, 10 MB 0.89 to 1.03,
//    16 MB of three planes 0.92 to 1.11, 256 images of 224 x 224 x 3 bytes 31.2 / 33.5.  Such long planes of 2-byte elements beyond
//    kShortBlocksMinMixed again: 36 MB 0.89 to 0.97, 64 MB 0.90 to 0.99, 130 MB 0.92 to 0.98 (28 MB of 32,400 x 3 25.0 / 26.4).
//  - Beyond kShortBlocksMaxLong, where the default tile ends and with it the kernel of planes alone, long planes of whole rounds
//    only (3.5 GB of 50,176 2300 / 2273, of 50,177 2650 / 2873, of 5000 2730 / 2895, 2.3 GB of 20,001 1720 / 1820, 6 GB 4570 /
//    4920; slower for one length in eight, whose blocks of two rounds leave the short last ones to the same die, up to
//    3 GB: 2.3 GB of 7501 1890 / 1820).
//  - Not where a round gives a wavefront 2 KiB (two planes: 300 of 210 x 200 bytes 18.8 / 19.5), nor for four planes of 2-byte
//    elements (128 of 128 x 127 14.3 / 15.0, 150 of 200 x 200 33.1 / 33.6).  4-byte elements keep the 8 KiB of the other
//    blocks with a short dimension (in one round 64 of 224 x 224 x 3 took 27.1 us instead of 31.1).
constexpr uint64_t kShortBlocksMaxPayload = 48u << 20, kShortBlocksMixedRounds = 4096, kShortBlocksMinMixed = 28u << 20, kShortBlocksMaxLong = 2ull << 30;
constexpr uint64_t kShortBlocksLongPlane = 4096;
constexpr bool plane_short_blocks(uint32_t element_bytes, uint32_t planes, uint64_t extent, uint64_t payload_bytes, bool alone) {
  if (!plane_single_round(element_bytes, planes)) return false;
  const bool whole = extent % plane_round_elements(element_bytes) == 0;
  const bool long_planes = element_bytes == 2 && extent >= kShortBlocksLongPlane && (whole || payload_bytes <= kShortBlocksMaxLong);
  if (!alone) return payload_bytes <= kShortBlocksMixedRounds * planes * kRowBytes || (long_planes && payload_bytes > kShortBlocksMinMixed);
  return long_planes || payload_bytes <= kShortBlocksMaxPayload || whole;
}
constexpr uint32_t kMaxPlanes = 4;
// Dims.lanes_per_run of such a segment: which side holds the planes, and above that the routine that moves its blocks.
constexpr uint32_t kPlanesInPayload = 1, kPlanesInTensor = 2, kPlaneRoutineShift = 2;
constexpr uint32_t plane_routine(uint32_t element_bytes, uint32_t planes, bool one_round) {
  const uint32_t all = (element_bytes >> 1) * 3 + planes - 2;   // 0 to 8
  return one_round ? 9 + (element_bytes == 2 ? 2 : planes - 3) : all;
}
static_assert(plane_routine(1, 2, false) == 0 && plane_routine(4, 4, false) == 8 && plane_routine(1, 3, true) == 9 &&
                  plane_routine(2, 3, true) == 11, "one after the other");
// LDS of a wavefront, one vector of padding behind every eight.
constexpr uint32_t planes_lds_bytes(uint32_t element_bytes, uint32_t planes, bool single) {
  return (single ? 1u : plane_rounds(element_bytes, planes)) * kWaveLanes * planes * kVecBytes / 8 * 9;
}
// Whether planes of `extent` elements are moved like this.  Whole vectors of 4-byte elements that one
// access per lane holds are not: rectangles take no second round for them (38 MB in three planes of 200
// elements 44 us for pack + unpack, 50 in rounds).
constexpr bool in_planes(uint32_t element_bytes, uint64_t extent) {
  return element_bytes <= 4 && extent * element_bytes >= kVecBytes &&
         !(element_bytes == 4 && extent <= kWaveLanes * kVecBytes / 4 && extent % 4 == 0);
}
// Elements of every plane that a block takes of `extent` of them: whole vectors, as many as fit; the
// block behind the last whole one takes what is left.
constexpr uint32_t plane_edge(uint32_t element_bytes, uint32_t planes, uint64_t extent) {
  const uint32_t vec = kVecBytes / element_bytes, square = kRectBlockBytes / 4 / planes;
  const uint32_t block = element_bytes < 4 ? plane_rounds(element_bytes, planes) * plane_round_elements(element_bytes)
                                           : (square < kRectMaxEdge ? square : kRectMaxEdge) / vec * vec;
  return extent < block ? static_cast<uint32_t>((extent + vec - 1) / vec * vec) : block;
}
constexpr uint32_t kMaxBatchDims = 4;
constexpr uint32_t kMinElementTileBytes = 8192;   // element-mode work unit (measured: 8 KiB beats 2, 4 and 16)
// kModeRows: the 16-byte slots a row needs, in whole 64-byte units, when its first byte lies up to
// `start` bytes behind one; the slots a lane moves; LDS for the rows of a tile.
constexpr uint32_t kUnitBytes = 64;
constexpr uint32_t kMaxRowSlots = 4;
constexpr uint64_t kMaxRowBytes = kMaxRowSlots * kRowBytes / 2 - kUnitBytes;   // two rows to a tile at least
constexpr uint32_t row_slots(uint64_t run_bytes, uint32_t start) {
  return static_cast<uint32_t>((start + run_bytes + kUnitBytes - 1) / kUnitBytes * (kUnitBytes / kVecBytes));
}
// Two, or three where that leaves a tenth less of a wavefront's slots without a row; four only for rows of
// which three would hold one.  (Three pieces: 36 bytes at 37, 32 MiB, two 22.8, three 19.8 us for two packs.)
// `mixed`: next to tensors that are moved otherwise.  The kernel for those holds fewer wavefronts, and larger
// tiles make up for it (2^18 rows of 128 bytes at 131, pack + unpack, next to 1 MiB of compact tensor 35.3 us with two
// slots per lane, 32.8 with three, 32.5 with four; next to a transposed matrix 47.1 / 39.7 / 36.9).
constexpr uint32_t row_slots_per_lane(uint32_t slots, bool mixed) {
  const uint32_t two = 2 * kWaveLanes / slots, three = 3 * kWaveLanes / slots;   // rows to a tile
  return mixed || three < 2 ? kMaxRowSlots : slots == 3 || 20 * three > 33 * two ? 3u : 2u;
}
// The slots of rows that lie `pitch` bytes apart and start up to `start` bytes behind a unit.
// Slots for the worst start cut every row on its units, but a row of one to two units then takes three of them,
// and what the lanes without a piece cost is more than the requests that are saved.  So they are taken where
// they cost no row of a tile, and for two to seven units where the bundle has left the caches: by receivers,
// which write the rows, from 24 MiB on, by senders of whole units, three or more, as well (such rows have no slot
// to spare for another start: 256 at 292, 32 MiB, pack + unpack in turn 28.4 -> 26.7 us, two packs in a launch
// 22.6 -> 23.9), by the others where the payload streams.  Slots for the worst start against slots for a start on a
// unit, time of pack / unpack alone: 72 bytes at 73, 32 MiB 20.0 / 19.6 us against 13.1 / 15.0; 200 at 201, 12 MiB
// 1.16 / 1.15 times, 100 MiB 1.18 / 0.83, 200 MiB 1.25 / 0.73; 130 at 131, 200 MiB 1.37 / 0.72; 500 at 501, 100 MiB
// 1.30 / 1.08; 144 at 168, 400 MiB 1.01 / 0.99 and 0.78 in one launch.
// Rows of up to 48 bytes whose neighbour lies in the same unit, or in the next one of a bundle that the caches
// hold, take as many slots as they have pieces (16 bytes at 24 0.6 times the time of whole units for pack and
// 0.7 for unpack up to 100 MiB; 32 at 128 1.03 times).
// Where a quarter of the slots of a row or more stay empty, more slots per lane make up for it: three, and for
// rows of 65 to 80 bytes, five pieces of eight, four as long as the caches help (130 at 131, 200 MiB, pack alone: two
// slots 1.43 times the time of three; 72 at 73, 32 MiB, two packs in a launch: two 26.5 us, three 21.8, four 20.1; 72 at
// 128, 300 MiB 8 % slower with four than with two).
constexpr uint64_t kRowUnitsPayload = 24ull << 20, kRowCachedPayload = 64ull << 20, kRowFilledPayload = 128ull << 20;
struct RowRule {
  uint32_t slots, per_lane;
};
constexpr RowRule row_rule(uint64_t run_bytes, uint64_t pitch, uint32_t start, bool receiver, uint64_t payload_bytes, bool streams) {
  const uint32_t pieces = static_cast<uint32_t>((run_bytes + kVecBytes - 1) / kVecBytes);
  if (pieces <= 3 && pitch < (payload_bytes < kRowCachedPayload ? 2 : 1) * kUnitBytes) {
    const uint32_t slots = pieces < 2 ? 2u : pieces;
    return {slots, row_slots_per_lane(slots, false)};
  }
  const uint32_t whole = row_slots(run_bytes, 0), worst = row_slots(run_bytes, start);
  if (run_bytes >= 2 * kUnitBytes && run_bytes < 7 * kUnitBytes &&
      (streams || (payload_bytes >= kRowUnitsPayload && (receiver || (run_bytes > 2 * kUnitBytes && run_bytes % kUnitBytes == 0)))))
    return {worst, 2u};
  uint32_t per_lane = row_slots_per_lane(whole, false);
  if (whole >= 8 && pieces * 4 <= whole * 3)
    per_lane = pieces != 5 ? 3u : payload_bytes < kRowFilledPayload ? kMaxRowSlots : 2u;
  const uint32_t lanes = per_lane * kWaveLanes;
  return {lanes / worst == lanes / whole ? worst : whole, per_lane};
}
// Whether bundles may share a launch that hold so many tiles of rows alone, and other kinds or not.  In the kernel for any mode the tiles of rows alone lose more
// than a launch costs once there are a few thousand of them (rows of 300 bytes at 512 and 1 MiB of compact tensor, joined /
// launched in turn: 640 tiles 5.2 / 6.9 us, 1280 7.5 / 7.7, 2560 11.7 / 10.9, 10240 34.5 / 28.6).
constexpr uint32_t kRowTilesJoined = 2048;
constexpr bool rows_share_launch(uint64_t row_tiles, bool others) { return !others || row_tiles <= kRowTilesJoined; }
constexpr uint32_t rows_lds_bytes(uint32_t rows, uint64_t run_bytes) {
  return static_cast<uint32_t>(rows * run_bytes) + kUnitBytes;
}

struct Dims {             // 176 bytes, one per strided segment
  uint32_t mode;
  uint32_t ndim;          // outer (non-run) dimensions after collapsing, <= kMaxOuterDims;
                          // transposed: batch dimensions (<= kMaxBatchDims)
  uint32_t tiles_per_run; // kModeRunTiles; kModeRows: runs per tile; kModeWalked: blocks per strip
                          // (kBlockStrip, or 1, or kSkewGroup in plain rows whose pack is skewed)
  uint32_t granule;       // kModeElements: bytes moved per lane access (1,2,4,8,16);
                          // kModeRunTiles: 1 + log2(tiles_per_run) when a power of two;
                          // transposed: element size
  uint64_t nbytes;        // bytes of the whole segment
  uint32_t shape[kMaxOuterDims];
  int64_t stride[kMaxOuterDims];   // bytes, outermost first, right-aligned
  // transposed: A is the innermost packed dimension (strided in the tensor), B the
  // dimension that is contiguous in the tensor; the rest are batch dimensions.
  uint64_t pstride[kMaxBatchDims]; // packed byte strides of the batch dims (aligned with shape[2..5])
  int64_t stride_a;                // tensor byte stride of A
  uint64_t pstride_b;              // packed byte stride of B
  uint32_t ext_a, ext_b;
  uint32_t tiles_a, tiles_b;       // kModeWalked alone: along a dimension in which blocks are skewed rounded up to
                                   // kSkewGroup, and the segment's tiles likewise; those past the extents are empty
  uint32_t edge_a, edge_b;         // block extent along A and B (elements)
  uint32_t lanes_per_run;          // kModeRows: the lane slots a run occupies (pstride[0] holds the
                                   // number of runs, edge_a the slots per lane);
                                   // kModePlanes: which side holds the planes (kPlanesInPayload,
                                   // kPlanesInTensor), and plane_routine << kPlaneRoutineShift
  uint32_t nt_allowed;             // kModeElements, transposed: sides that may keep the launch's
                                   // non-temporal hint when packing (bit 0 tensor, bit 1 payload) and when
                                   // unpacking (bits 2, 3).  Transposed block rows that straddle 128-byte
                                   // lines share them with the neighbouring blocks and are written through
                                   // the cache; rows shorter than a line are read and written through it.
                                   // Bits 4, 5: kSkewPack, kSkewUnpack
};
static_assert(sizeof(Dims) == 176, "Dims layout");

// Workgroup indices a die takes in a row: a power of two, or one run per die (`whole`).
constexpr uint32_t kRemapShiftBit = 27, kRemapRunMask = (1u << kRemapShiftBit) - 1u;
constexpr uint32_t remap_code(uint32_t run, bool whole) {
  return run | (whole ? 31u : static_cast<uint32_t>(__builtin_ctz(run))) << kRemapShiftBit;
}

struct KernelArgs {
  const Seg* segs;            // nseg + 1 entries, last is a sentinel with tile_begin == ntiles
  const Dims* dims;
  const uint32_t* wave_seg;   // segment holding tile (k << seg_shift), for every k
  uint8_t* payload;
  uint32_t nseg;
  uint32_t ntiles;
  uint32_t tiles_per_wave;
  uint32_t xcd_remap;         // 0, or remap_code of the workgroup indices a die takes in a row
  uint32_t seg_shift;         // log2 of the tile-block size of wave_seg
  int64_t tensor_delta = 0;   // added to every tensor-side address of the tables
};

// One launch serving several bundles: job k owns the workgroups [wg_begin[k], wg_begin[k+1]).
constexpr uint32_t kMaxJobs = 16;   // 1 KiB of kernel arguments
struct JobDesc {              // 64 bytes
  uint64_t segs, dims, wave_seg, payload;   // device addresses
  int64_t tensor_delta;
  uint32_t ntiles, tiles_per_wave, seg_shift, wg_begin;
  uint32_t unpack;            // 0: tensors -> payload, 1: payload -> tensors
  uint32_t reserved;
};
static_assert(sizeof(JobDesc) == 64, "JobDesc layout");
constexpr uint32_t kNoJobBegin = 0x7fffffffu;        // beyond every workgroup index of a launch
constexpr uint32_t kJobTableKernargOffset = 64;      // the table follows 14 scalar arguments, 16-byte aligned
struct alignas(16) JobTable {
  uint32_t count, lds_per_wave, nt_bits;
  uint32_t interleaved;       // 1: two jobs of equal grids, job = workgroup & 1, local workgroup = workgroup >> 1
  // first workgroup of every job once more, side by side (kNoJobBegin past the last job): the kernel
  // gets the first eleven as scalar arguments as well and reads the rest here, instead of walking
  // the descriptors with a dependent load per step
  uint32_t begins[kMaxJobs];
  JobDesc job[kMaxJobs];
};

// Tables of a small bundle handed to the kernel by value.  bytes[0..16) is a head
// (a mark the kernel checks, then padding), the Seg array follows at kInlineTablesHead,
// Dims and the tile-block index at the offsets the launch passes.
constexpr uint32_t kInlineTableBytes = 3584;
constexpr uint32_t kInlineTablesHead = 16;
constexpr uint64_t kInlineTablesMark = 0x31454c4254525841ull;   // "AXRTBLE1"
struct alignas(16) InlineTables {
  uint8_t bytes[kInlineTableBytes];
};

struct LaunchConfig {
  uint32_t workgroups = 0;
  uint32_t tiles_per_wave = 0;
  uint32_t tile_rows = 2;
  uint32_t threads = 128;   // per workgroup, a multiple of 64
  uint32_t seg_shift = 0;   // wave_seg has one entry per 2^seg_shift tiles
  uint32_t nontemporal = 3;   // bit 0: tensor-side accesses, bit 1: payload-side accesses
  bool elements = false;   // some segment's mode is above kModeRunTiles
  uint32_t kind = kKindAny;   // the mode of every segment where all have the same and one kernel is built for it
  uint32_t lds_per_wave = 0;   // bytes of LDS each wavefront needs (kModeRows and above)
  uint32_t lds_walked = 0;     // and in the kernel of walked blocks alone
  uint32_t cached_tail = 0;    // MiB at the end of a streaming payload that a pack leaves in the cache (runs in
                           // 1 KiB tiles only; see finish_geometry)
  uint32_t xcd_remap = 0;  // 0, or remap_code of the workgroup indices each die takes in a row (the grid is a
                           // multiple of 8 such runs)
};

// ---------------------------------------------------------------- tunables

// Read by planning threads while axr_tune_set may write: every knob is an atomic.
struct Tunables {
  // Tile = tile_rows KiB moved by one wavefront.  0 picks the smallest of
  // 2, 4, 8, 16 that keeps the bundle within max_tiles tiles (and one tile per
  // run for bundles of short strided runs): small tiles and a grid of one tile
  // per wave measured fastest on MI355X (the hardware dispatcher balances the
  // load); larger tiles only bound the grid for multi-GiB bundles.
  std::atomic<int64_t> tile_rows{0};
  std::atomic<int64_t> max_tiles{1 << 20};
  std::atomic<int64_t> max_waves{1 << 20};    // beyond this many tiles a wave takes several
  std::atomic<int64_t> threads{0};            // workgroup size; 0 = 256 below 65,536 tiles (fewer dispatches
                                  // for short kernels), 128 above (finer balance at the tail)
  // Non-temporal hint: bit 0 tensor-side accesses, bit 1 payload-side accesses;
  // -1 = automatic: tensors always stream (read or written once), the payload
  // streams only when it is larger than payload_cache_bytes.  A smaller payload
  // is written with ordinary stores so that it is still in the 256 MB
  // last-level cache when the consumer (unpack, or the transport's copy) reads it.
  std::atomic<int64_t> nontemporal{-1};
  std::atomic<int64_t> payload_cache_bytes{256ll << 20};
  // Strided runs shorter than this are not moved as run tiles when they are 16 bytes or
  // longer, anything else up to a fifth of it (measured crossovers).
  std::atomic<int64_t> gather_run_bytes{1280};
  std::atomic<int64_t> xcd_remap{-1};         // contiguous wave ranges per die: 1 always, 0 never, -1 when
                                  // transposed blocks that share lines with their neighbours dominate
                                  // (larger bundles then in squares of blocks, see finish_geometry)
  std::atomic<int64_t> transpose{1};          // move transposed views as square blocks through LDS
  std::atomic<int64_t> ragged_runs{1};        // short runs of 16+ bytes move in whole rows (kModeRows) instead
                                  // of in granules of a power of two that divides them
  // Contiguous segments longer than a tile start their tiles on a multiple of this many
  // bytes of the written side (0: tiles start at the segment's first byte).  Measured on the
  // 4096-tensor bundle: 16 lifts the tight layout by 2 % (every 16-byte store aligned) and
  // costs the 256-byte aligned layout nothing; 64 and 128 are no better for either.
  std::atomic<int64_t> head_align{16};
  // The loopback transport moves a device payload to device memory of the same GPU with the
  // library's copy kernel (1) or with hipMemcpyAsync (0).
  std::atomic<int64_t> loopback_copy_kernel{1};
  // Bundles of at least this many tensors, all of them contiguous device tensors, get their
  // tables in one pass over the tensors into pinned memory plus a kernel that brings them to
  // the device and writes the tile-block index (0: the general host path always).  Fresh bundles of 256 B
  // to 64 KiB, pack + unpack, host tables read in place / device tables: 300 tensors 53.4 / 54.8 us, 340 55.6 / 56.2, 380
  // 58.3 / 58.1, 420 61.1 / 59.7; of 600 to 4000 bytes 320 50.7 / 55.3, 480 61.6 / 63.4, 600 68.7 / 69.0; of 64 KiB 320
  // 53.2 / 56.1, 440 61.8 / 63.3.
  std::atomic<int64_t> device_tables{384};
  // axr_stream_synchronize may first poll, for up to this many microseconds, a word of pinned
  // memory that a one-wave kernel enqueued behind the stream's work writes, before it falls
  // back to the runtime's wait (0, the default: the runtime's wait only).  See the header.
  std::atomic<int64_t> spin_wait_us{0};
  std::atomic<int64_t> host_threads{4};       // threads (the caller included) for host-side staging copies
  // Contiguous device tensors of at most this many bytes that follow each other in a bundle
  // share wavefronts (group tiles, up to 64 tensors or 2 KiB of lane slots each); 0: every
  // tensor gets its own wavefronts.
  std::atomic<int64_t> group_bytes{512};
  std::atomic<int64_t> group_slots{kGroupMaxSlots};   // lane slots per group tile: 64 or 128
  // The two jobs of an axr_submit launch whose grids are equal and whose payloads are larger than
  // payload_cache_bytes take the workgroups in turn (even / odd) instead of one range each (1, the
  // default; 0: never; 2: also smaller payloads that were asked to stream).  With a pack and an
  // unpack in one launch the memory then sees reads and writes of both throughout: the 405 MB
  // layer bundle 6.50 -> 6.65 TB/s.  Smaller payloads are better off with the pack's range first,
  // cached (48 MB mixed bundle: 6.18 against 6.11 TB/s) or streaming (5.78 against 5.51).
  std::atomic<int64_t> submit_interleave{1};
  // Failure injection for tests of the streamed transfer's error handling: N > 0 makes the
  // N-th chunk submitted from now on fail after its send has been queued, as if the message
  // that arrived did not match the receiver's plan (and counts down to 0 = off).
  std::atomic<int64_t> transfer_fail_after_send{0};
  std::atomic<int64_t> inline_tables{16384};  // bundles of up to this many tiles whose tables fit the kernel
                                  // arguments are launched without a table upload (larger ones
                                  // outside of captures, see large_inline), and read theirs in pinned
                                  // memory (see first_launch_reads_host_block); 0: never
};
Tunables& tunables();

// ---------------------------------------------------------------- errors

int fail(int status, const std::string& message);   // records thread-local message
int check_hip(int hip_error, const char* what);     // 0 or AXR_ERR_HIP
// Host-side copies of the staging paths (pageable memory <-> pinned blocks).  One core
// moves about 25 GB/s, less than the PCIe link; jobs of 2 MiB and more in total are cut
// into byte-balanced shares for up to `host_threads` short-lived threads.
struct HostCopyJob {
  void* dst;
  const void* src;
  size_t bytes;
};
void host_copy(const HostCopyJob* jobs, size_t count);
// A staging block moved unit by unit from the front, by the caller and up to `helpers` short-lived threads in turn.
struct HostUnits {
  size_t span = 0, unit = 1, helpers = 0;   // the block's bytes [0, span), in units of `unit`
  // Whether unit `u` may be moved; waits for it.  False (an error, known to the caller's thread) ends the thread's share.
  virtual bool ready(size_t u, bool caller) = 0;
  virtual void copy(size_t lo, size_t hi) = 0;   // moves bytes [lo, hi); from any of the threads
  virtual int done(size_t u) = 0;                // units 0 .. u have been moved; in order, on the caller's thread
  virtual void stop() {}                         // the caller gives up: no ready() may wait any longer
  virtual ~HostUnits() = default;
};
// Units of a block that the device fills from the front, raising a flag behind every `piece` bytes.  A flag is looked at
// `looks` times in a row; then the caller's thread waits for the device and the others look again now and then.
struct FlaggedUnits : HostUnits {
  const uint32_t* flags = nullptr;
  size_t piece = 1;
  uint32_t looks = 0;
  int status = AXR_OK;           // what ended the caller's share
  virtual int arrive() = 0;      // returns once every flag has been raised (or with an error); on the caller's thread
  bool ready(size_t u, bool caller) override;
  void stop() override { stopped_.store(true, std::memory_order_relaxed); }

 private:
  std::atomic<bool> stopped_{false};
};
int host_copy_units(HostUnits& units);   // what done() returned, or AXR_OK
// The least that goes to the payload at once of a staging block of `span` bytes, `sent` of which have gone (the rules of
// staging blocks are in axr_plan.cpp).  Rounded up: four such pieces hold the block, whatever its length.
constexpr size_t kStageUnit = 64u << 10, kStageSend = 256u << 10;
constexpr size_t stage_piece(size_t span, size_t sent) {
  const size_t part = ((sent ? 5 * span : span) + 15) / 16;
  return part > kStageSend ? part : kStageSend;
}

// True for a handle that axr_stream_destroy has destroyed (and no later
// axr_stream_create has returned again).
bool stream_retired(void* stream);
// Launch marks order what the library enqueues, process-wide.  A launch takes a mark after
// it has been enqueued; a wait reads the current mark before it starts, and once it has seen
// the stream drain, every launch on that stream with a mark up to that value is known to be
// finished, so that a plan released next need not wait for the stream again.
uint64_t stream_mark_launch();
uint64_t stream_launch_mark();
void stream_note_drained(void* stream, uint64_t mark);
bool stream_drained(void* stream, uint64_t mark);
void stream_forget(void* stream);   // the stream is being destroyed
// A kernel that writes device-visible HOST memory has been enqueued on `stream`: the next
// axr_stream_synchronize of that stream must be the runtime's wait (which makes such writes
// visible to the CPU), not the polled one.  take: true once per note, then forgotten.
void stream_note_host_writes(void* stream);
bool stream_take_host_writes(void* stream);
int fail_nothrow(int status, const char* message) noexcept;

// Every extern "C" entry point runs its body through this: no C++ exception
// (std::bad_alloc from a container, in practice) crosses the C boundary.
template <typename Body>
int guarded(Body&& body) noexcept {
  try {
    return body();
  } catch (const std::bad_alloc&) {
    return fail_nothrow(AXR_ERR_NOMEM, "out of host memory");
  } catch (...) {
    return fail_nothrow(AXR_ERR_INVALID, "unexpected C++ exception");
  }
}

// ---------------------------------------------------------------- kernels (axr_kernels.hip)

int launch_bundle_kernel(bool pack, const KernelArgs& args, const LaunchConfig& cfg,
                         void* stream);
// Same launch with the tables inside the kernel arguments (two geometries only: 2 KiB tiles, tensor side
// streaming, payload side cacheable; runs in tiles of 1 KiB, both sides streaming; no die remapping).
int launch_bundle_kernel_inline(bool pack, const KernelArgs& args, const LaunchConfig& cfg,
                                const InlineTables& tables, uint32_t dims_at, uint32_t wave_at,
                                void* stream);
// One launch for up to kMaxJobs bundles that share `cfg` (tile size, workgroup size, cache
// hints; cfg.workgroups is the whole grid, cfg.lds_per_wave the largest need of any job).
int launch_bundle_jobs(const JobTable& jobs, const LaunchConfig& cfg, void* stream);
int launch_fill(void* dst, int value, size_t bytes, void* stream);
// Enqueues a one-wave kernel that stores `value` into *flag (pinned host memory).
int launch_notify(uint32_t* flag, uint32_t value, void* stream);
// staged: n + 1 segment records in device-accessible memory (pinned host memory will do);
// segs and wave_seg are device memory.  Copies the records and writes the tile-block index.
int launch_expand_tables(const Seg* staged, uint32_t n, Seg* segs, uint32_t* wave_seg, uint32_t seg_shift,
                         void* stream);
// members and groups are pinned host memory, blocks device memory: writes the blocks of `n` groups.
int launch_expand_groups(const Member* members, const GroupStage* groups, uint32_t n, void* blocks, void* stream);
// tables[0, bytes) = staged[0, bytes), rounded up to 16 bytes: a table block's pinned half into its
// device half.
int launch_upload_tables(const void* staged, void* tables, size_t bytes, void* stream);
// dst[0, bytes) = src[0, bytes), no alignment needed; dst in memory of the current device, src there or in pinned host memory.
int launch_stream_copy(void* dst, const void* src, size_t bytes, bool nontemporal, void* stream);
// dst[0, bytes) = src[0, bytes) from device memory to pinned host memory; flags[i] (pinned, cleared by the
// caller) becomes 1 once bytes [i, i + 1) * kStagePieceBytes are there.
constexpr uint32_t kStagePieceBytes = 16384, kStageGroups = 16;
int launch_stage_out(void* dst, const void* src, size_t bytes, uint32_t* flags, void* stream);
// Device address, on the current device, of the kStaticTableBytes bytes that hold the
// tables of axr_pack_noalloc (a __device__ array of the code object: never allocated,
// shared by every call on that device).
constexpr size_t kStaticTableBytes = 1u << 20;
int static_table_area(void** ptr);

// ---------------------------------------------------------------- runtime (axr_runtime.cpp)

int device_compute_units(int* cus);
// Cached pinned-host + device block pair used for plan tables.
struct TableBlock {
  void* host = nullptr;
  void* device = nullptr;
  size_t bytes = 0;
  int device_id = -1;
};
int table_block_acquire(size_t bytes, TableBlock* block);
void table_block_release(TableBlock* block);
// Events without timing for the current device, recycled: creating one costs more than a
// microsecond, and every fresh plan that uploads tables needs one.  An event goes back
// only once it has fired (or was never recorded).
// They release to the system.  A kernel behind one that does not (hipEventDisableSystemFence) starts 1.6 us sooner
// (140 views that all differ, fresh, pack + unpack, 56.1 -> 54.5 us), but nothing then promises that what is in
// front of it is visible; with hipEventReleaseToDevice, which would be enough, it does not start sooner (56.3).
int event_acquire(void** event, int* device);
void event_release(void* event, int device);

}  // namespace axr

#endif  // AXR_INTERNAL_H_
