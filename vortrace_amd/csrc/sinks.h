// Reduction sinks and per-ray I/O of the ray kernels: what a walk or a march
// does with a ray's segments, in order (src/reduction.cpp:8-83), and where a
// ray's results go.
#pragma once
#include "device_common.h"

#pragma clang fp contract(off)

namespace vt {

// ---------------------------------------------------------------- sinks ----

template <int NF>
struct SumSink {  // reduce_sum, src/reduction.cpp:8-21
  const double *fields;
  double acc[NF];
  uint64_t n;
  __device__ void init() {
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = 0.0;
    n = 0;
  }
  __device__ __forceinline__ void seg(uint32_t cell, double a, double b) {
    const double ds = b - a;
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = acc[f] + ds * gld(fields + (size_t)cell * NF + f);
    ++n;
  }
  __device__ void store(double *out) const {
#pragma unroll
    for (int f = 0; f < NF; ++f) gst(out + f, acc[f]);
  }
};

struct SumSinkDyn {  // reduce_sum for any number of fields, accumulated in place
  const double *fields;
  int nf;
  double *out;
  uint64_t n;
  __device__ void init() {
    for (int f = 0; f < nf; ++f) gst(out + f, 0.0);
    n = 0;
  }
  __device__ void seg(uint32_t cell, double a, double b) {
    const double ds = b - a;
    for (int f = 0; f < nf; ++f)
      gst(out + f, gld(out + f) + ds * gld(fields + (size_t)cell * nf + f));
    ++n;
  }
  __device__ void store(double *) const {}
};

template <bool kMax>
struct ExtSink {  // reduce_max / reduce_min, src/reduction.cpp:23-53
  const double *fields;
  int nf;
  double *out;
  uint64_t n;
  __device__ void init() {
    for (int f = 0; f < nf; ++f) gst(out + f, kMax ? -(double)INFINITY : (double)INFINITY);
    n = 0;
  }
  __device__ void seg(uint32_t cell, double, double) {
    for (int f = 0; f < nf; ++f) {
      const double v = gld(fields + (size_t)cell * nf + f);
      const double cur = gld(out + f);
      if (kMax ? (v > cur) : (v < cur)) gst(out + f, v);
    }
    ++n;
  }
  __device__ void store(double *) const {}
};

struct VolSink {  // reduce_volume_render, src/reduction.cpp:55-83
  const double *fields;
  double T, c[3];
  uint64_t n;
  __device__ void init() {
    T = 1.0;
    c[0] = c[1] = c[2] = 0.0;
    n = 0;
  }
  __device__ __forceinline__ void seg(uint32_t cell, double a, double b) {
    const double2 *fv = reinterpret_cast<const double2 *>(fields + (size_t)cell * 4);
    const double2 rg = gld(fv), ba = gld(fv + 1);
    const double col[3] = {rg.x, rg.y, ba.x};
    const double alpha = ba.y;
    const double ds = b - a;
    const double opacity = 1.0 - exp(-alpha * ds);
#pragma unroll
    for (int k = 0; k < 3; ++k) c[k] += T * col[k] * opacity;
    T *= (1.0 - opacity);
    ++n;
  }
  __device__ void store(double *out) const {
    gst(out, c[0]);
    gst(out + 1, c[1]);
    gst(out + 2, c[2]);
  }
};

struct CountSink {
  uint64_t n;
  __device__ void init() { n = 0; }
  __device__ __forceinline__ void seg(uint32_t, double, double) { ++n; }
  __device__ void store(double *) const {}
};

template <class Inner>
struct FillSink {  // segments at the ray's offset, plus the reduced values
  Inner in;
  const uint32_t *slot_id;
  int64_t *ids;
  double *se, *sx;
  uint64_t cap;  // room the count pass reserved for this ray
  uint64_t n;
  __device__ void init() {
    in.init();
    n = 0;
  }
  __device__ __forceinline__ void seg(uint32_t cell, double a, double b) {
    if (n < cap) {
      gst(ids + n, (int64_t)gld(slot_id + cell));
      gst(se + n, a);
      gst(sx + n, b);
    }
    ++n;
    in.seg(cell, a, b);
  }
  __device__ void store(double *out) const { in.store(out); }
};

// ------------------------------------------------------------ ray I/O ----
// Per-ray sink set-up and output for run_engine (engine.h).

// Every projection IO also writes the ray's segment count when `counts` is
// given (the forward pass of a differentiable projection keeps them for the
// adjoint).
__device__ __forceinline__ void put_count(int64_t *counts, int64_t ray, uint64_t n) {
  if (counts) gst(counts + ray, (int64_t)n);
}

template <int NF>
struct SumIO {
  using Sink = SumSink<NF>;
  const double *fields;
  double *out;
  int nout;
  int64_t *counts;
  __device__ void begin(int64_t, Sink &sk) const {
    sk.fields = fields;
    sk.init();
  }
  __device__ int end(int64_t ray, Sink &sk) const {
    sk.store(out + ray * nout);
    put_count(counts, ray, sk.n);
    return kErrNone;
  }
};

struct SumDynIO {
  using Sink = SumSinkDyn;
  const double *fields;
  int nf;
  double *out;
  int nout;
  int64_t *counts;
  __device__ void begin(int64_t ray, Sink &sk) const {
    sk.fields = fields;
    sk.nf = nf;
    sk.out = out + ray * nout;
    sk.init();
  }
  __device__ int end(int64_t ray, Sink &sk) const {
    put_count(counts, ray, sk.n);
    return kErrNone;
  }
};

template <bool kMax>
struct ExtIO {
  using Sink = ExtSink<kMax>;
  const double *fields;
  int nf;
  double *out;
  int nout;
  int64_t *counts;
  __device__ void begin(int64_t ray, Sink &sk) const {
    sk.fields = fields;
    sk.nf = nf;
    sk.out = out + ray * nout;
    sk.init();
  }
  __device__ int end(int64_t ray, Sink &sk) const {
    put_count(counts, ray, sk.n);
    return kErrNone;
  }
};

struct VolIO {
  using Sink = VolSink;
  const double *fields;
  double *out;
  int nout;
  int64_t *counts;
  __device__ void begin(int64_t, Sink &sk) const {
    sk.fields = fields;
    sk.init();
  }
  __device__ int end(int64_t ray, Sink &sk) const {
    sk.store(out + ray * nout);
    put_count(counts, ray, sk.n);
    return kErrNone;
  }
};

struct CountIO {
  using Sink = CountSink;
  int64_t *counts;
  __device__ void begin(int64_t, Sink &sk) const { sk.init(); }
  __device__ int end(int64_t ray, Sink &sk) const {
    gst(counts + ray, (int64_t)sk.n);
    return kErrNone;
  }
};

// Segments at the ray's offset (from the count pass) plus the reduced values.
template <class InnerIO>
struct FillIO {
  using Sink = FillSink<typename InnerIO::Sink>;
  InnerIO inner;
  const int64_t *offsets;
  const uint32_t *slot_id;
  int64_t *ids;
  double *se, *sx;
  __device__ void begin(int64_t ray, Sink &sk) const {
    const int64_t off = gld(offsets + ray);
    sk.slot_id = slot_id;
    sk.ids = ids + off;
    sk.se = se + off;
    sk.sx = sx + off;
    sk.cap = (uint64_t)(gld(offsets + ray + 1) - off);
    inner.begin(ray, sk.in);
    sk.n = 0;
  }
  __device__ int end(int64_t ray, Sink &sk) const {
    inner.end(ray, sk.in);
    return sk.n == sk.cap ? kErrNone : kErrFillOverflow;
  }
};

}  // namespace vt
