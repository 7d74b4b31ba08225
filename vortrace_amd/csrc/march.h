// The march: rays advanced from cell to cell through neighbour lists, instead
// of by the split-point recursion's nearest-neighbour queries.
//
// Along a ray x(s), the squared distance to generator g less |x(s)|^2 is a
// line in s, so the cells a ray crosses are the lower envelope of lines.  The
// march builds that envelope cell by cell: the exit of cell c is the smallest
// s at which another generator is as near as c, found among the generators
// nearest to c (neighbors.h).  The reference's recursion (src/ray.cpp:187-430)
// inserts cells at split points of pairs and closes a boundary once one of the
// pair is nearest there; where no generator comes within the reference's
// tolerance of a tie, it inserts exactly the envelope's cells and its
// boundaries are the split points of adjacent cells.  So after the march
//  * every boundary is verified: no third generator within the tolerance
//    (plus rounding) of the two that meet there;
//  * the recursion is replayed on the known envelope: the split point of every
//    pair it visits must fall inside a cell, clear of that cell's boundaries
//    by more than the tolerance.
// A ray that fails any check -- ties, grazing bisectors, tiny chords, image
// choices that depend on the interval -- is left to the ray engine (engine.h),
// which repeats the reference's steps one by one.  A ray that passes has the
// engine's segments, bit for bit: each boundary is computed by the
// reference's own expression from the same two generators.
#pragma once
#include "boxes.h"
#include "record.h"
#include "sinks.h"

namespace vt {

// Per-cell neighbour lists (neighbors.h).
constexpr int kNbMax = 64;       // entries per list
constexpr int kNbSlotBits = 27;  // an entry is slot | image << 27
constexpr uint32_t kNbSlotMask = (1u << kNbSlotBits) - 1u;
constexpr uint32_t kNbCentre = 13u;  // image code of no shift: (ix+1)*9 + (iy+1)*3 + (iz+1)
constexpr size_t kNbMaxPoints = (size_t)1 << kNbSlotBits;

struct NbLists {
  const uint32_t *nb;  // [n][kNbMax], nearest first, kNone past the end
  const float *r2;     // [n] every generator closer than this is in the list
  const BNode *boxes;  // per inner node (boxes.h)
};

// The rays of one batch: slot j is ray order[base + j], or the 8x8-tile ray of
// fetch slot base + j.
struct MarchRays {
  const double *start, *end;
  int64_t base, n;  // the batch's slots are [base, base + n)
  const uint32_t *order;
  uint32_t tile_row, tile_n;
};

// Work buffers of a march, one row per batch slot.
struct MarchBufs {
  // [slot][cap], entry k: position where cell k is entered, cell | image, zone
  // half-width.
  uint4 *seq;
  // Per slot: the entry to march from (kNone: not at all), then the number
  // of cells (0: left to the engine).
  uint32_t *c0;
  // kMarchCounters words: slots taken of each part of the queue, and the starts
  // left to k_locate_far.
  uint32_t *ctr;
  int cap;
};

constexpr int kMarchCounters = kParts + 1;

struct MarchCall {
  DevCloud C;
  Scratch S;      // for the start cells' searches
  NbLists N;
  MarchRays R;
  MarchBufs B;
  uint32_t *fall;  // rays left to the engine
  ErrRec *err;
  Stats *stats;
  int cus;
  int pool;  // intervals a wave holds for its lanes to share
  hipStream_t st;
};

// Builds the neighbour lists of a cloud (gen: slot order).
void march_build_lists(const DevCloud &C, uint32_t *nb, float *r2, hipStream_t st);
// Builds the boxes of its `nodes` inner nodes; `work` holds 2 * nodes + n words.
void march_build_boxes(const DevCloud &C, uint32_t nodes, BNode *boxes, uint32_t *work,
                       hipStream_t st);
// Start cells and envelopes of a batch's rays.
void march_batch(const MarchCall &m, bool periodic);
// Checks the batch's envelopes and hands their segments to `io`'s sinks.
template <class IO>
void march_finish(const MarchCall &m, bool periodic, const IO &io);
// The most workgroups k_locate_far runs, as many as its stacks in LDS let the chip
// hold (its scratch is sized by it).
int march_locate_grid(int cus);

// Records a ray's segments in one run of the pool (RecordIO for the march).
template <class InnerIO>
struct MarchRecordIO {
  InnerIO inner;
  RecPool pool;
};

}  // namespace vt
