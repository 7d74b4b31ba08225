// Segment lists and segment records: the forward side of the adjoint.
#pragma once
#include "device_common.h"

namespace vt {

// Segments of a ray at its offset: slot of the cell and ds.
struct SegSink {
  uint32_t *slot;
  double *ds;
  uint64_t cap;
  uint64_t n;
  __device__ void init() { n = 0; }
  __device__ __forceinline__ void seg(uint32_t cell, double a, double b) {
    if (n < cap) {
      gst(slot + n, cell);
      gst(ds + n, b - a);
    }
    ++n;
  }
};

struct SegIO {
  using Sink = SegSink;
  const int64_t *offsets;
  uint32_t *slot;
  double *ds;
  __device__ void begin(int64_t ray, Sink &sk) const {
    const int64_t off = gld(offsets + ray);
    sk.slot = slot + off;
    sk.ds = ds + off;
    sk.cap = (uint64_t)(gld(offsets + ray + 1) - off);
    sk.init();
  }
  __device__ int end(int64_t, Sink &sk) const {
    return sk.n == sk.cap ? kErrNone : kErrFillOverflow;
  }
};

// One segment recorded by a forward pass: the cell's slot, the ray, its
// position k along the ray, and ds.  ray == kNone marks a record of a
// lane's last chunk that the lane did not fill.
struct alignas(16) SegRec {
  uint32_t slot, ray, k, pad;
  double ds, pad2;
};
static_assert(sizeof(SegRec) == 32, "segment record must be 32 bytes");

// Pool the records go to: lanes take chunks of kRecChunk records from `head`
// and fill them in order; `overflow` is set when the pool runs out.  A lane
// marks the records of its last chunk that it did not fill (ray = kNone)
// after its last ray, so every record below the final head is either written
// or marked and the pool needs no clearing beforehand.
struct RecPool {
  SegRec *rec;
  unsigned long long cap;
  unsigned long long *head;
  int *overflow;
};
constexpr int kRecChunk = 32;

// A projection IO that also records every segment.  The sink's chunk state
// survives from ray to ray (begin() leaves it alone).  A ray left to the
// K_EXPAND launch records a prefix of its segments twice, with the same
// values: the backward pass writes both to the same place.
template <class InnerIO>
struct RecordIO {
  // The inner sink with recording added; its segment count `n` is the
  // place of the next segment along the ray.
  struct Sink : InnerIO::Sink {
    using Base = typename InnerIO::Sink;
    RecPool pool;  // set once per lane before the first ray (setup), the same in every lane
    uint32_t ray;
    // Next record of this lane's current chunk; a multiple of kRecChunk
    // means the chunk is used up (chunks start at multiples of kRecChunk).
    unsigned long long next = 0;
    __device__ __forceinline__ void seg(uint32_t cell, double a, double b) {
      const uint32_t k = (uint32_t)this->n;  // the segment's place along the ray
      Base::seg(cell, a, b);
      if ((next & (unsigned long long)(kRecChunk - 1)) == 0ull)
        next = atomicAdd(pool.head, (unsigned long long)kRecChunk);
      if (next < pool.cap) {
        SegRec *r = pool.rec + next;
        // Records are read only by a later kernel.  Measured at 2M clustered
        // cells, 512^2: HBM reads of the recording forward 13.7 -> 8.0 GB.
        gst_nt(reinterpret_cast<uint4 *>(r), make_uint4(cell, ray, k, 0u));
        gst_nt(&r->ds, b - a);
      } else {
        atomicOr(pool.overflow, 1);
      }
      ++next;
    }
  };
  InnerIO inner;
  RecPool pool;
  __device__ void setup(Sink &sk) const { sk.pool = pool; }
  // After the lane's last ray: the rest of its current chunk is unwritten.
  __device__ void finish(Sink &sk) const {
    unsigned long long j = sk.next;
    while ((j & (unsigned long long)(kRecChunk - 1)) != 0ull && j < pool.cap) {
      gst(&pool.rec[j].ray, kNone);
      ++j;
    }
  }
  __device__ void begin(int64_t ray, Sink &sk) const {
    inner.begin(ray, static_cast<typename Sink::Base &>(sk));
    sk.ray = (uint32_t)ray;
  }
  __device__ int end(int64_t ray, Sink &sk) const {
    return inner.end(ray, static_cast<typename Sink::Base &>(sk));
  }
};

}  // namespace vt
