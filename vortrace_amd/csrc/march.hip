// The march's kernels: start cells, envelopes, and the replay of the
// recursion that hands the segments on (march.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "boxes.h"
#include "engine.h"
#include "march.h"
#include "neighbors.h"

#pragma clang fp contract(off)

namespace vt {

namespace {

// What a third generator must stay clear of in r^2: the reference's tolerance
// plus the rounding of squared distances between points of this size (the
// expressions here and the reference's differ by some tens of roundings of
// numbers up to scale^2).
__device__ __forceinline__ double clearance(const DevCloud &C, const RayGeom &r, double &scale) {
  double m = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    m = fmax(m, fmax(fabs(r.a[d]), fabs(r.a[d] + r.len * r.d[d])));
    m = fmax(m, fmax(fabs(C.rb_lo[d]), fabs(C.rb_hi[d])) + C.box[d]);
  }
  scale = m;
  return 1.05 * kTol + 1e-14 * m * m;
}

__device__ __forceinline__ int64_t march_ray(const MarchRays &R, int64_t j) {
  const int64_t k = R.base + j;
  if (R.order) return (int64_t)gld(R.order + k);
  return R.tile_row ? (int64_t)tile_ray((uint32_t)k, R.tile_row, R.tile_n) : k;
}

// 1 / b to about 1e-14.
__device__ __forceinline__ double fast_rcp(double b) {
  const double r = __builtin_amdgcn_rcp(b);
  return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}

// Image shift of `code` along axis d.
__device__ __forceinline__ int image_axis(uint32_t code, int d) {
  const uint32_t hi = (code * 57u) >> 9, q = (code * 43u) >> 7;  // code / 9, code / 3
  return d == 0 ? (int)hi - 1 : (d == 1 ? (int)(q - 3u * hi) - 1 : (int)(code - 3u * q) - 1);
}

__device__ __forceinline__ uint32_t image_code(int x, int y, int z) {
  return (uint32_t)((x + 1) * 9 + (y + 1) * 3 + (z + 1));
}

// Blocks are dealt to the XCDs in turn; give each XCD a contiguous share.
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t nb) {
  const int64_t share = (nb + kParts - 1) / kParts;
  return (b % kParts) * share + b / kParts;
}

// A value from another lane of a group of 4 or 16: lanes 1 or 2 apart, or
// mirrored within 8 or 16 (after the steps before, each of those lanes holds
// its own quad's or half's result).
template <int STEP>
__device__ __forceinline__ uint32_t group_swap(uint32_t v) {
  constexpr int ctrl = STEP == 0 ? 0xB1 : (STEP == 1 ? 0x4E : (STEP == 2 ? 0x141 : 0x140));
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true);
}
// The value of a group's first lane.
template <int G>
__device__ __forceinline__ uint32_t group_first(uint32_t v) {
  static_assert(G == 4 || G == 8 || G == 16, "groups are quads, half rows or rows");
  const int i = (int)v;
  if constexpr (G == 4) return (uint32_t)__builtin_amdgcn_update_dpp(i, i, 0x00, 0xF, 0xF, true);
  // Lane 0 of every row of 16, and for the second half of a row its lane 8.
  const int row = __builtin_amdgcn_update_dpp(i, i, 0x150, 0xF, G == 8 ? 0x3 : 0xF, false);
  if constexpr (G == 16) return (uint32_t)row;
  return (uint32_t)__builtin_amdgcn_update_dpp(row, i, 0x158, 0xF, 0xC, false);
}

// The nearest generator so far.
struct Near {
  double d2 = INFINITY;
  uint32_t name = kNone;
  __device__ __forceinline__ void offer(double d, uint32_t id) {
    name = d < d2 ? +id : +name;
    d2 = fmin(d, d2);
  }
  template <int STEP>
  __device__ __forceinline__ void swap_in() {
    const uint64_t b = (uint64_t)__double_as_longlong(d2);
    const uint32_t lo = group_swap<STEP>((uint32_t)b), hi = group_swap<STEP>((uint32_t)(b >> 32));
    const uint32_t id = group_swap<STEP>(name);
    offer(__longlong_as_double((long long)(((uint64_t)hi << 32) | lo)), id);
  }
  // The nearest of a group's lanes; equals: any of them, alike in every lane.
  template <int G>
  __device__ __forceinline__ void reduce() {
    swap_in<0>();
    swap_in<1>();
    if constexpr (G > 8) {
      swap_in<2>();
      swap_in<3>();
    }
    name = __shfl(name, (threadIdx.x & 63) & ~(G - 1));
  }
};

__device__ __forceinline__ void load_gen(const DevCloud &C, uint32_t slot, double (&g)[3]) {
  const double2 xy = gld(reinterpret_cast<const double2 *>(C.gen + slot));
  g[0] = xy.x;
  g[1] = xy.y;
  g[2] = gld(&C.gen[slot].z);
}

// Every ray's start cell as entry 0 of its column, and 0 as the entry to march
// from -- or kNone when the march cannot vouch for the start.  Also empties the
// batch's queues.
//
// G lanes per ray: the tree is descended once, to the start's leaf; from the
// nearest generator there the lists lead to the nearest of all (any nearer one
// is within twice its distance, and a list that reaches that far has it).  Starts
// whose lists do not reach that far are left to k_locate_far, in `rest`.  Bound
// by the chain of reads, some ten of the descent and two per cell: with a search
// of the tree per lane 256 rays took 212 us (its images and backtracking, lanes
// apart) and 262,144 rays 720 us; now 11 us, and 118 + 234 us.
template <bool PER, int G>
__global__ __launch_bounds__(kBlock) void k_locate(DevCloud C, NbLists N, MarchRays R, MarchBufs B,
                                                   uint32_t *rest) {
  constexpr int kChunk = 4 * G;
  const int tid = threadIdx.x;
  const int gtid = blockIdx.x * kBlock + tid;
  const int gl = tid & (G - 1), lead = (tid & 63) & ~(G - 1);
  if (gtid < kParts) gst(B.ctr + gtid, 0u);
  for (int64_t j = gtid / G; j < R.n; j += (int64_t)gridDim.x * (kBlock / G)) {
    const int64_t ray = march_ray(R, j);
    RayGeom r;
    make_ray(R.start + 3 * ray, R.end + 3 * ray, r);
    double scale;
    const double delta = clearance(C, r, scale);
    const bool sane = r.len > 1e-6 && r.len < 1e30 && scale < 1e15;
    uint32_t c = kNone, code = kNbCentre;
    bool sure = false;
    if (sane) {
      // The leaf of the start, folded into the box.
      double q[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        q[d] = r.a[d];
        if constexpr (PER) {
          const double off = q[d] - 0.5 * (C.rb_lo[d] + C.rb_hi[d]);
          if (off > 0.5 * C.box[d]) q[d] -= C.box[d];
          if (off < -0.5 * C.box[d]) q[d] += C.box[d];
        }
      }
      uint32_t cur = C.rroot;
      while (!(cur & kRefLeaf)) {
        const DRecV rec = load_rec(C.recs, cur);
        double cut;
        cur = choose(rec.x, sel3(q[0], q[1], q[2], rec.x.dim), cut) ? rec.x.c1 : rec.x.c2;
        if (!(cur & kRefLeaf)) {
          const DNodeV nd = rec_child(rec, cur & 1u);
          cur = choose(nd, sel3(q[0], q[1], q[2], nd.dim), cut) ? nd.c1 : nd.c2;
        }
      }
      const uint32_t s0 = cur & kSlotMask, end = (uint32_t)gld(&C.gen[s0].end);
      Near near;
      for (uint32_t t = s0 + gl; t < end; t += G) {
        double g[3], d2 = 0.0;
        load_gen(C, t, g);
#pragma unroll
        for (int d = 0; d < 3; ++d) d2 = __builtin_fma(g[d] - q[d], g[d] - q[d], d2);
        near.offer(d2, t);
      }
      near.template reduce<G>();
      c = near.name;
      double gb[3], w[3];
      load_gen(C, c, gb);
      if constexpr (PER) {
        // The image nearest to the start.
        int im[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double e = r.a[d] - gb[d];
          im[d] = e > 0.5 * C.box[d] ? 1 : (e < -0.5 * C.box[d] ? -1 : 0);
        }
        code = image_code(im[0], im[1], im[2]);
      }
      bool go = true;
      for (int move = 0; go && move < 64; ++move) {
        double v2 = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          w[d] = r.a[d] - gb[d];
          if (PER && code != kNbCentre) w[d] -= image_axis(code, d) * C.box[d];
          v2 = __builtin_fma(w[d], w[d], v2);
        }
        const double complete = gld(N.r2 + c);
        near = Near();
        go = false;
        for (int pos = 0; pos < kNbMax / kChunk; ++pos) {
          const uint4 ids =
              gld(reinterpret_cast<const uint4 *>(N.nb + (size_t)c * kNbMax + pos * kChunk) + gl);
          const uint32_t id[4] = {ids.x, ids.y, ids.z, ids.w};
          double g[4][3];
#pragma unroll
          for (int i = 0; i < 4; ++i) load_gen(C, id[i] == kNone ? c : id[i] & kNbSlotMask, g[i]);
          double last = 0.0;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t rel = id[i] >> kNbSlotBits;
            bool named = true;
            double dd = 0.0, d2 = 0.0;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
              double e = g[i][d] - gb[d];
              if (PER && id[i] != kNone) {
                if (rel != kNbCentre) e += image_axis(rel, d) * C.box[d];
                named &= abs(image_axis(rel, d) + image_axis(code, d)) <= 1;
              }
              dd = __builtin_fma(e, e, dd);
              d2 = __builtin_fma(e - w[d], e - w[d], d2);
            }
            if (id[i] != kNone) near.offer(d2, named ? id[i] : kNone);
            last = id[i] == kNone ? (double)INFINITY : dd;
          }
          near.template reduce<G>();
          last = __shfl(last, lead + G - 1);
          if (near.d2 < v2) {
            go = near.name != kNone;  // (an image the march cannot name: searched for)
            break;
          }
          const bool ended = last == (double)INFINITY || pos + 1 == kNbMax / kChunk;
          const double lim = ended ? complete : last * 0.999998;
          const double gap = lim - delta;
          if (gap > 0.0 && gap * gap > 4.000008 * lim * v2) {
            sure = true;
            break;
          }
          if (ended) break;
        }
        if (go) {
          c = near.name & kNbSlotMask;
          if constexpr (PER) code += (near.name >> kNbSlotBits) - kNbCentre;
          load_gen(C, c, gb);
        }
        if (sure && !(near.d2 - v2 > delta)) c = kNone;  // a tie: the engine's
      }
    }
    if (gl == 0) {
      if (sane && !sure) {
        gst(rest + atomicAdd(B.ctr + kParts, 1u), (uint32_t)j);
      } else {
        if (c != kNone)
          gst(B.seq + (size_t)j * B.cap, make_uint4(0u, 0u, c | (code << kNbSlotBits), 0u));
        gst(B.c0 + j, c != kNone ? 0u : kNone);
      }
    }
  }
}

// The starts k_locate left: a search of the tree each.
template <bool PER>
__global__ __launch_bounds__(kBlock) void k_locate_far(DevCloud C, Scratch S, MarchRays R,
                                                       MarchBufs B, const uint32_t *rest) {
  const int tid = threadIdx.x;
  const int gtid = blockIdx.x * kBlock + tid;
  const LaneInfo li{tid, gtid, gtid >> 6, (int)(tid & 63)};
  KStack st = make_stack(S, li);
  const uint32_t n = gld(B.ctr + kParts);
  // Spread over the waves, as a wave's searches take different ways (262,144
  // rays through clumps: 234 us, with full waves 700 us).
  const uint32_t waves = gridDim.x * (kBlock / 64);
  for (uint32_t i = (tid & 63) * waves + (gtid >> 6); i < n; i += 64 * waves) {
    const uint32_t j = gld(rest + i);
    const int64_t ray = march_ray(R, j);
    RayGeom r;
    make_ray(R.start + 3 * ray, R.end + 3 * ray, r);
    double scale;
    const double delta = clearance(C, r, scale);
    uint32_t id[2];
    double d[2];
    query_reg<2, PER>(C, r.a[0], r.a[1], r.a[2], id, d, st);
    const bool ok = id[0] != kNone && d[1] - d[0] > delta && !st.overflow;
    if (ok) {
      uint32_t code = kNbCentre;
      if constexpr (PER) {
        // The generator's image nearest to the start.
        double g[3];
        load_gen(C, id[0], g);
        int im[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double e = r.a[k] - g[k];
          im[k] = e > 0.5 * C.box[k] ? 1 : (e < -0.5 * C.box[k] ? -1 : 0);
        }
        code = image_code(im[0], im[1], im[2]);
      }
      gst(B.seq + (size_t)j * B.cap, make_uint4(0u, 0u, id[0] | (code << kNbSlotBits), 0u));
    }
    gst(B.c0 + j, ok ? 0u : kNone);
  }
}

// The three nearest candidates' places (where they come within the clearance;
// floats, good to kKeyTol), and the names of the nearer two.  Floats order all
// but a millionth of the exits; the rest, and every exit taken, are computed
// again in FP64.  Keeping the places and their g'.d in FP64 through the
// selects and the lanes' exchange took a third of the scan's instructions.
//
// A key (key_of) is off by the rounding of its numerator and of g'.d to float
// (2^-24 of themselves each), the reciprocal's last place (2^-23) and the
// product's rounding (2^-24; halving is exact): 5 2^-24 = 3.0e-7 of itself.  Two
// keys compared may be 6.0e-7 of the larger apart from their FP64 values'
// order, and kKeyTol leaves two fifths of itself above that.  A key that
// underflows lies within any zone of the entry, where no exit is accepted.
constexpr double kKeyTol = 1e-6;
struct Best {
  float t1, t2, t3;
  uint32_t n1, n2;
  __device__ __forceinline__ void clear() {
    t1 = INFINITY;
    n1 = kNone;
    clear_rest();
  }
  // All but the nearest.
  __device__ __forceinline__ void clear_rest() {
    t2 = t3 = INFINITY;
    n2 = kNone;
  }
  __device__ __forceinline__ void offer(float t, uint32_t id) {
    const bool l1 = t < t1, l2 = t < t2;
    const uint32_t second = l2 ? +id : +n2;
    n2 = l1 ? +n1 : +second;
    n1 = l1 ? +id : +n1;
    t3 = __builtin_amdgcn_fmed3f(t, t2, t3);
    t2 = __builtin_amdgcn_fmed3f(t, t1, t2);
    t1 = fminf(t, t1);
  }
  // The candidates of both, which have none in common.
  __device__ __forceinline__ void merge(const Best &other) {
    // By value: a choice between members becomes a choice between addresses,
    // which keeps both records in scratch memory.
    const Best o = other;
    const uint32_t a1 = n1, b1 = n2, a2n = o.n1, b2n = o.n2;
    const bool l1 = o.t1 < t1;
    const bool l2 = l1 ? o.t2 < t1 : o.t1 < t2;
    const uint32_t keep = l1 ? +a1 : +b1, take = l1 ? +b2n : +a2n;
    const uint32_t s1 = l2 ? +take : +keep;
    const float a3 = fminf(fminf(t3, o.t3), fminf(fmaxf(t1, o.t2), fmaxf(t2, o.t1)));
    const float a2 = fminf(fmaxf(t1, o.t1), fminf(t2, o.t2));
    n1 = l1 ? +a2n : +a1;
    n2 = s1;
    t1 = fminf(t1, o.t1);
    t2 = a2;
    t3 = a3;
  }
  template <int STEP>
  __device__ __forceinline__ void swap_in() {
    Best o;
    o.t1 = __uint_as_float(group_swap<STEP>(__float_as_uint(t1)));
    o.t2 = __uint_as_float(group_swap<STEP>(__float_as_uint(t2)));
    o.t3 = __uint_as_float(group_swap<STEP>(__float_as_uint(t3)));
    o.n1 = group_swap<STEP>(n1);
    o.n2 = group_swap<STEP>(n2);
    merge(o);
  }
  // The candidates of a group's lanes, alike in every lane: of equal keys, each
  // lane of a pair keeps its own in front, so the names are the first lane's.
  template <int G>
  __device__ __forceinline__ void reduce() {
    swap_in<0>();
    swap_in<1>();
    if constexpr (G > 4) swap_in<2>();
    if constexpr (G > 8) swap_in<3>();
    n1 = group_first<G>(n1);
    n2 = group_first<G>(n2);
  }
};

enum : int { kMpScan = 0, kMpBall = 1, kMpDone = 2 };

// One ray's march.  Distances along the ray are relative to the entry of the
// current cell c: with w = x(entry) - c, d the direction and g' = g - c, the
// generator g becomes as near as c at tau = (|g'|^2 - 2 g'.w) / (2 g'.d), and
// its squared distance less c's is 2 g'.d (tau_g - tau) there.  Candidates are
// compared by where they come within the clearance, tau' (delta earlier in
// r^2), so that the exit is verified when the next one's tau' lies beyond it.
// What a ray's march needs at crossings only (its group's, in LDS: these
// registers held a third wave per SIMD off).
struct Held {
  double a[3], len;  // the ray
  double s;          // entry of the cell
  double zone;       // half-width of a boundary's zone, but for the clearance
  double x[3];       // centre of a search's ball
  double reach;      // and how far ahead it looks while there is no exit
  uint32_t j;        // slot
  int k;             // entries so far
  float tent;        // zone half-width at the entry
};

// The images of a box: their shifts, and for each the relative images (codes
// as bits) whose sum with it is an image.
struct Images {
  double shift[27][3];
  uint32_t sums[27];
};

template <bool PER>
struct Marcher {
  Held *h;
  const Images *im;
  double dir[3];
  double delta;
  uint32_t c;      // current cell
  uint32_t ic;     // and its image's code
  double gb[3];    // its generator, in the primary box
  double w[3];
  double tend;     // distance left on the ray
  Best b;
  int pos;

  __device__ __forceinline__ void enter(uint32_t cell, const double (&g)[3],
                                        const double (&p)[3], double at) {
    c = cell;
    h->s = at;
    tend = h->len - at;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      gb[d] = g[d];
      w[d] = (h->a[d] + at * dir[d]) - p[d];
    }
    b.clear();
    pos = 0;
  }
  // A generator's image, as the reference shifts it.
  __device__ __forceinline__ void image(const double (&g)[3], uint32_t code, double (&p)[3]) const {
#pragma unroll
    for (int d = 0; d < 3; ++d) p[d] = g[d];
    if (PER && code != kNbCentre) {
#pragma unroll
      for (int d = 0; d < 3; ++d) p[d] = g[d] + im->shift[code][d];
    }
  }
  // From c to a generator, base coordinates g, named by slot | relative image.
  __device__ __forceinline__ void apart(const double (&g)[3], uint32_t name, double (&e)[3]) const {
#pragma unroll
    for (int d = 0; d < 3; ++d) e[d] = g[d] - gb[d];
    if (PER && (name >> kNbSlotBits) != kNbCentre) {
#pragma unroll
      for (int d = 0; d < 3; ++d) e[d] += im->shift[name >> kNbSlotBits][d];
    }
  }
  __device__ __forceinline__ void dots(const double (&e)[3], double &dd, double &dw,
                                       double &dh) const {
    dd = __builtin_fma(e[2], e[2], __builtin_fma(e[1], e[1], e[0] * e[0]));
    dw = __builtin_fma(e[2], w[2], __builtin_fma(e[1], w[1], e[0] * w[0]));
    dh = __builtin_fma(e[2], dir[2], __builtin_fma(e[1], dir[1], e[0] * dir[0]));
  }
  // tau' of a generator at e from c as a key, infinite when it recedes.
  __device__ __forceinline__ float key_of(const double (&e)[3], float &dd2) const {
    double dd, dw, dh;
    dots(e, dd, dw, dh);
    dd2 = (float)dd;
    const float a = (float)(__builtin_fma(-2.0, dw, dd) - delta);
    const float t = a * 0.5f * __builtin_amdgcn_rcpf((float)dh);
    return dh > 1e-18 ? t : INFINITY;
  }
  // Its exit, and how far before it it comes within the clearance.
  __device__ __forceinline__ double exit_of(const double (&e)[3], double &dh, double &slack) const {
    double dd, dw;
    dots(e, dd, dw, dh);
    const double ih = 0.5 * fast_rcp(dh);
    slack = delta * ih;
    return __builtin_fma(-2.0, dw, dd) * ih;
  }
  __device__ __forceinline__ void load(const DevCloud &C, uint32_t name, double (&g)[3]) const {
    const uint32_t n = name & kNbSlotMask;
    const double2 xy = gld(reinterpret_cast<const double2 *>(C.gen + n));
    g[0] = xy.x;
    g[1] = xy.y;
    g[2] = gld(&C.gen[n].z);
  }
  // Squared distance from c of the point `tau` after the entry.
  __device__ __forceinline__ double r2_at(double tau) const {
    double s2 = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double v = __builtin_fma(tau, dir[d], w[d]);
      s2 = __builtin_fma(v, v, s2);
    }
    return s2;
  }
  // Whether nothing at least sqrt(lim) from c can be within the clearance of
  // the exit: |x - g| >= |g - c| - |x - c|, so when D^2 - delta > 2 D |x - c|.
  __device__ __forceinline__ bool clear_of(double lim, double v2) const {
    const double q = lim - delta;
    return q > 0.0 && q * q > 4.000008 * lim * v2;
  }
};

// References of nodes still to be searched for an exit, per group, in LDS (a
// step pushes up to two per lane).
constexpr int ball_stack(int G) { return G == 4 ? 112 : (G == 8 ? 192 : 384); }

// At most the squared distance from q to a box; q is the nearest float of a
// point, which lies within `eps` of it along every axis.
__device__ __forceinline__ float box_below2(const float (&lo)[3], const float (&hi)[3],
                                            const float (&q)[3], float eps) {
  float s = 0.0f;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float t = fmaxf(fmaxf(lo[d] - q[d], q[d] - hi[d]) - eps, 0.0f);
    s = __builtin_fmaf(t, t, s);
  }
  return s * 0.999999f;
}

// G lanes march one ray: each takes a share of every list chunk, and they hold
// the ray's state alike.  4 lanes where rays are plentiful, 8 or 16 where they
// are not (see march_batch_p).
//
// A cell whose list does not reach far enough for its exit has the tree
// searched: boxes that touch the ball around the exit are opened, G at a time;
// every generator found inside moves the exit closer and shrinks the ball (the
// part of a ball ahead of the entry contains the later, smaller ones).  A
// wave's rays wait until some need a search (or none can go on), so that the
// searches' steps run for several rays at once.
//
// Groups take rays from a queue of the batch's slots, one part per XCD.
//
// 2M clustered cells, 512^2 rays (126 crossings each): 7.1 ms, of which the 1.1 %
// of crossings that search take a quarter; 1M such cells, 1024^2 rays: 2 x 10.1
// ms.  Counters of the former: VALU issues in 58 % of the SIMDs' cycles (71 wave
// instructions a crossing, 35 lanes active, 29 % of them FP64), the address units
// are busy in 56 %, 68 % of the reads hit L1, and the 2.5 waves a SIMD holds wait
// for half of their time: the chain list -> generators -> exit -> next list.  With
// FP64 keys, the image shifts computed at each use and all of the ray in
// registers it was 8.0 and 2 x 11.5 ms; the keys in scratch memory (see merge)
// cost 1.2 ms, two waves per SIMD 1.4 ms, and four, which spill here, nothing
// less.  A ray's own lane descending the tree alone took 65 ms (chains of up to
// 300 dependent reads in clumps).
template <bool PER, int G, int kShare>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(G == 4 ? 3 : 4))) void k_march(
    DevCloud C, NbLists N, MarchRays R, MarchBufs B, double far, Stats *stats, int batch) {
  constexpr int kChunk = G * kShare;  // list entries a group takes at once
  static_assert(kShare % 4 == 0 && kNbMax % kChunk == 0, "lists are read in whole chunks");
  constexpr int kRays = 64 / G;
  // Generators of a leaf whose loads are in flight together.
  constexpr int kSearchChunk = G == 4 ? 5 : 3;
  constexpr int kBallStack = ball_stack(G);
  __shared__ uint32_t stack_all[kRays * kBallStack];
  __shared__ Held held[kRays];
  __shared__ Images im;
  const int lane = threadIdx.x;
  const int gl = lane & (G - 1), lead = lane & ~(G - 1);
  uint32_t *stk = stack_all + (lane / G) * kBallStack;
  const uint32_t below = (1u << gl) - 1u;
  constexpr uint64_t leads = G == 4   ? 0x1111111111111111ull
                             : G == 8 ? 0x0101010101010101ull
                                      : 0x0001000100010001ull;
  auto slice = [&](uint64_t m) { return (uint32_t)(m >> lead) & ((1u << G) - 1u); };
  if constexpr (PER) {
    if (lane < 27) {
      uint32_t sums = 0u;
      for (uint32_t rel = 0; rel < 27u; ++rel) {
        bool is = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) is &= abs(image_axis(lane, d) + image_axis(rel, d)) <= 1;
        sums |= (is ? 1u : 0u) << rel;
      }
      im.sums[lane] = sums;
#pragma unroll
      for (int d = 0; d < 3; ++d) im.shift[lane][d] = image_axis(lane, d) * C.box[d];
    }
    __syncthreads();
  }
  Marcher<PER> M;
  M.h = held + lane / G;  // (every lane of a group writes it, alike)
  M.im = &im;
  int ph = kMpDone;
  uint32_t nball = 0;
  uint32_t id[kShare];   // this lane's share of the next chunk
  uint32_t list = 0;     // the cell whose list is read: c, or its exit's other cell
  float complete = 0.0f;  // c's list holds everything closer than this (squared)
  float lim = 0.0f;       // everything closer than this has been seen (infinite: searched)
  auto read_ids = [&](int pos) {
    const uint4 *p =
        reinterpret_cast<const uint4 *>(N.nb + (size_t)list * kNbMax + kChunk * pos + kShare * gl);
#pragma unroll
    for (int i = 0; i < kShare; i += 4) {
      const uint4 q = gld(p + i / 4);
      id[i] = q.x;
      id[i + 1] = q.y;
      id[i + 2] = q.z;
      id[i + 3] = q.w;
    }
  };
  // The queue's parts, this block's own first.
  const uint32_t psize = (uint32_t)((R.n + kParts - 1) / kParts);
  int part = (int)(blockIdx.x & (kParts - 1));
  int tries = 0;
  bool more = true;  // the queue may hold rays (uniform in the wave)
  for (;;) {
    // Free groups take the next rays.
    while (more) {
      const uint64_t idle = __ballot(ph == kMpDone) & leads;
      if (!idle) break;
      const int need = __popcll(idle);
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(B.ctr + part, (uint32_t)need);
      base = __shfl(base, 0);
      const uint32_t lo = part * psize, hi = min(lo + psize, (uint32_t)R.n);
      const uint32_t at = lo + base + __popcll(idle & ((1ull << lead) - 1ull));
      if (ph == kMpDone && at < hi) {
        if (gld(B.c0 + at) == kNone) {
          if (gl == 0) gst(B.c0 + at, 0u);
        } else {
          const int64_t ray = march_ray(R, at);
          RayGeom r;
          make_ray(R.start + 3 * ray, R.end + 3 * ray, r);
          double scale;
          M.delta = clearance(C, r, scale);
          M.h->zone = 1e-13 * scale;
          M.h->j = at;
          M.h->k = 0;
          M.h->tent = 0.0f;
          M.h->len = r.len;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            M.h->a[d] = r.a[d];
            M.dir[d] = r.d[d];
          }
          const uint4 e = gld(B.seq + (size_t)at * B.cap);
          list = e.z & kNbSlotMask;
          M.ic = e.z >> kNbSlotBits;
          read_ids(0);
          complete = gld(N.r2 + list);
          double g[3], p[3];
          M.load(C, list, g);
          M.image(g, M.ic, p);
          M.enter(list, g, p, 0.0);
          // (A start too far from its cell's generator: see `far` below.)
          if (M.r2_at(0.0) < far * far) {
            ph = kMpScan;
          } else if (gl == 0) {
            gst(B.c0 + at, 0u);
          }
        }
      }
      if (lo + base + need >= hi) {
        // This part is used up.
        part = (part + 1) & (kParts - 1);
        more = ++tries < kParts;
      }
    }
    const uint64_t scan = __ballot(ph == kMpScan), wait = __ballot(ph == kMpBall);
    if (!(scan | wait)) break;
    bool settle = false;  // the exit is certain: cross (or end)
    const bool search = __popcll(wait) >= batch * G || !scan;
    if (ph == kMpScan && !search) {
      // This lane's share of one chunk of the list; its names were read when
      // the chunk before it was done.
      double2 gxy[kShare];
      double gz[kShare];
#pragma unroll
      for (int i = 0; i < kShare; ++i) {
        const uint32_t sl = id[i] == kNone ? M.c : (id[i] & kNbSlotMask);
        gxy[i] = gld(reinterpret_cast<const double2 *>(C.gen + sl));
        gz[i] = gld(&C.gen[sl].z);
      }
      const uint32_t sums = PER ? im.sums[M.ic] : 0u;
      float last = 0.0f;
      Best b;
      b.clear();
#pragma unroll
      for (int i = 0; i < kShare; ++i) {
        const double g[3] = {gxy[i].x, gxy[i].y, gz[i]};
        bool valid = id[i] != kNone;
        double e[3];
        const uint32_t name = valid ? id[i] : (kNbCentre << kNbSlotBits);
        M.apart(g, name, e);
        if constexpr (PER) valid &= (sums >> (name >> kNbSlotBits)) & 1u;
        float dd;
        const float t = M.key_of(e, dd);
        b.offer(valid ? t : INFINITY, id[i]);
        last = id[i] == kNone ? INFINITY : dd;
      }
      b.template reduce<G>();
      M.b.merge(b);
      if constexpr (G > 1) last = __shfl(last, lead + G - 1);  // the chunk's farthest
      ++M.pos;
      const bool ended = last == INFINITY || M.pos == kNbMax / kChunk;
      // Generators not seen yet are at least this far from c; those of the
      // other cell's list were all seen.  The exit's key will do here, with
      // some room: the exit taken is held against `lim` again.
      if (list == M.c) lim = ended ? complete : last * 0.999998f;
      const double near = M.r2_at(fmin((double)M.b.t1, M.tend)) * 1.00002;
      if (list == M.c ? M.clear_of((double)lim, near)
                      : ended && (M.b.n1 & kNbSlotMask) == list) {
        settle = true;
      } else if (!ended) {
        read_ids(M.pos);
      } else {
        ph = kMpBall;
        M.h->reach = 2.0 * sqrt((double)complete);
        M.b.clear_rest();  // the searches meet them again
        // The ball around the exit also passes through the exit's other cell:
        // its list may reach far enough.
        if (list == M.c && (M.b.n1 >> kNbSlotBits) == kNbCentre && (double)M.b.t1 < M.tend) {
          const uint32_t n = M.b.n1 & kNbSlotMask;
          const float other = gld(N.r2 + n);
          if (n != M.c && M.clear_of((double)other, near)) {
            lim = other;
            list = n;
            M.pos = 0;
            read_ids(0);
            ph = kMpScan;
          }
        }
      }
    }
    // The waiting rays' searches, until all of them have ended.  Their state is
    // alike in a group's lanes.
    double br2 = 0.0;
    uint32_t images = 0;
    int code = 0, first = 0, steps = 0;
    int sp = -1;  // not begun
    while (search && __ballot(ph == kMpBall && !settle)) {
      const bool on = ph == kMpBall && !settle;
      auto centre = [&]() {
        // The ball around the exit known so far, no farther than `reach` while
        // there is none.
        double te = M.h->reach;
        if (M.b.n1 != kNone) {
          double g[3], e[3], h, slack;
          M.load(C, M.b.n1, g);
          M.apart(g, M.b.n1, e);
          te = M.exit_of(e, h, slack);
        }
        te = fmin(te, M.tend);
        br2 = M.r2_at(te) + M.delta;
        double p[3];
        M.image(M.gb, M.ic, p);
#pragma unroll
        for (int d = 0; d < 3; ++d) M.h->x[d] = p[d] + __builtin_fma(te, M.dir[d], M.w[d]);
      };
      if (on && sp < 0) {
        if (gl == 0) ++nball;
        centre();
        sp = 0;
        images = 1u << kNbCentre;
        first = (int)kNbCentre;
        if constexpr (PER) {
          // Images whose generators can be within the ball, the nearest first.
          uint32_t ms[3];
          const double r = sqrt(br2);
          first = 0;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            ms[d] = 0u;
            double nearest = DBL_MAX;
            int at = 1;
#pragma unroll
            for (int k = -1; k <= 1; ++k) {
              const double q = M.h->x[d] - k * C.box[d];
              const double o = fmax(fmax(C.rb_lo[d] - q, q - C.rb_hi[d]), 0.0);
              if (o <= r) ms[d] |= 1u << (k + 1);
              if (o < nearest) {
                nearest = o;
                at = k + 1;
              }
            }
            first = 3 * first + at;
          }
          images = 0u;
#pragma unroll
          for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b)
              if (((ms[0] >> a) & (ms[1] >> b) & 1u) != 0u) images |= ms[2] << (a * 9 + b * 3);
        }
      }
      if (on && sp == 0 && images) {
        // The next image: its root.
        code = first;
        if (!((images >> code) & 1u)) code = __ffs(images) - 1;
        images &= ~(1u << code);
        if (gl == 0) stk[0] = C.root;
        sp = 1;
      }
      __builtin_amdgcn_wave_barrier();
      __threadfence_block();
      // The centre in the image's frame, and what its floats may be off.
      double q1[3];
      float qf[3], eps = 0.0f;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        q1[d] = PER ? M.h->x[d] - im.shift[code][d] : M.h->x[d];
        qf[d] = (float)q1[d];
        eps = fmaxf(eps, fabsf(qf[d]) * 1.2e-7f);
      }
      const float bf = (float)br2 * 1.000001f;
      const int take = on ? min(sp, G) : 0;
      uint32_t ref = 0u;
      const bool have = gl < take;
      if (have) ref = stk[sp - take + gl];
      sp -= take;
      const bool leaf = have && (ref & kRefLeaf);
      const bool inner = have && !(ref & kRefLeaf);
      uint32_t kn = 0u, kf = 0u;
      bool pn = false, pf = false;
      if (inner) {
        const uint4 *p = reinterpret_cast<const uint4 *>(N.boxes + ref);
        const uint4 v0 = gld(p), v1 = gld(p + 1), v2 = gld(p + 2), v3 = gld(p + 3);
        const float lo1[3] = {__uint_as_float(v0.x), __uint_as_float(v0.y), __uint_as_float(v0.z)};
        const float hi1[3] = {__uint_as_float(v0.w), __uint_as_float(v1.x), __uint_as_float(v1.y)};
        const float lo2[3] = {__uint_as_float(v1.z), __uint_as_float(v1.w), __uint_as_float(v2.x)};
        const float hi2[3] = {__uint_as_float(v2.y), __uint_as_float(v2.z), __uint_as_float(v2.w)};
        const float d1 = box_below2(lo1, hi1, qf, eps), d2 = box_below2(lo2, hi2, qf, eps);
        const bool first1 = d1 <= d2;
        kn = first1 ? v3.x : v3.y;
        kf = first1 ? v3.y : v3.x;
        pn = fminf(d1, d2) < bf;
        pf = fmaxf(d1, d2) < bf;
      }
      // Far children below near ones: the near ones are taken next.
      const uint32_t mf = slice(__ballot(pf)), mn = slice(__ballot(pn));
      const int nf = __popc(mf), nn = __popc(mn);
      bool fail = on && (sp + nf + nn > kBallStack || ++steps > 8192);
      if (!fail) {
        if (pf) stk[sp + __popc(mf & below)] = kf;
        if (pn) stk[sp + nf + __popc(mn & below)] = kn;
        sp += nf + nn;
      }
      bool found = false;
      Best b;
      b.clear();
      if (leaf) {
        const uint32_t s0 = ref & kSlotMask;
        const uint32_t end = (uint32_t)gld(&C.gen[s0].end);
        // The current candidate under its absolute name.
        uint32_t nslot = kNone;
        int ncode = (int)kNbCentre;
        if (M.b.n1 != kNone) {
          nslot = M.b.n1 & kNbSlotMask;
          if constexpr (PER) {
            // Codes of base 3 add up, one centre too many.
            ncode = (int)(M.ic + (M.b.n1 >> kNbSlotBits)) - (int)kNbCentre;
          }
        }
        const int ccode = PER ? (int)M.ic : (int)kNbCentre;
        // Half a leaf at a time, its loads in flight together (past the
        // leaf's end they stay within the padding records).
#pragma unroll
        for (int h0 = 0; h0 < kLeafMaxSize; h0 += kSearchChunk) {
          if (h0 && s0 + h0 >= end) break;
          double2 xy[kSearchChunk];
          double z[kSearchChunk];
#pragma unroll
          for (int i = 0; i < kSearchChunk; ++i) {
            xy[i] = gld(reinterpret_cast<const double2 *>(C.gen + s0 + h0 + i));
            z[i] = gld(&C.gen[s0 + h0 + i].z);
          }
          uint32_t in = 0u;
#pragma unroll
          for (int i = 0; i < kSearchChunk; ++i) {
            const uint32_t t = s0 + (uint32_t)(h0 + i);
            const double e0 = q1[0] - xy[i].x, e1 = q1[1] - xy[i].y, e2 = q1[2] - z[i];
            const double d2 = __builtin_fma(e2, e2, __builtin_fma(e1, e1, e0 * e0));
            if (t < end && d2 < br2 && !(t == M.c && code == ccode) &&
                !(t == nslot && code == ncode))
              in |= 1u << i;
          }
          while (in) {
            const uint32_t t = s0 + (uint32_t)(h0 + __ffs(in) - 1);
            in &= in - 1u;
            uint32_t rel = kNbCentre;
            bool named = true;
            if constexpr (PER) {
              rel = (uint32_t)code - M.ic + kNbCentre;
#pragma unroll
              for (int d = 0; d < 3; ++d)
                named &= abs(image_axis((uint32_t)code, d) - image_axis(M.ic, d)) <= 1;
            }
            double g[3], e[3];
            M.load(C, t, g);
            if (named) M.apart(g, t | (rel << kNbSlotBits), e);
            float dd;
            // A generator that recedes, or two images away, is no exit the
            // march can name: leave the ray to the engine.
            const float tv = named ? M.key_of(e, dd) : INFINITY;
            if (tv == INFINITY)
              fail = true;
            else
              b.offer(tv, t | (rel << kNbSlotBits));
            found = true;
          }
        }
      }
      if (slice(__ballot(fail))) {
        if (gl == 0) gst(B.c0 + M.h->j, 0u);
        ph = kMpDone;
      } else if (slice(__ballot(found))) {
        b.template reduce<G>();
        M.b.merge(b);
        centre();
      }
      if (ph == kMpBall && sp == 0 && !images) {
        if (M.b.n1 == kNone && M.h->reach < M.tend) {
          M.h->reach *= 4.0;
          sp = -1;
        } else {
          settle = true;
          lim = INFINITY;
        }
      }
    }
    if (settle) {
      int cells = 0;  // 0: left to the engine
      bool done = true;
      // `far` (periodic boxes): each boundary's generators must be the images
      // nearest to every point of the two cells' chords, so cells and their
      // distances stay a fifth of the box.
      uint32_t name = M.b.n1;
      bool ends = !((double)M.b.t1 <= M.tend * (1.0 + kKeyTol));
      if (!ends) {
        list = name & kNbSlotMask;
        read_ids(0);
        complete = gld(N.r2 + list);
        double g[3], e[3], h, slack;
        M.load(C, name, g);
        M.apart(g, name, e);
        double exit = M.exit_of(e, h, slack);
        bool ok = exit < M.tend;
        if (fmin(exit, M.tend) >= (double)M.b.t2 * (1.0 - kKeyTol)) {
          // The keys cannot tell which of two is first.
          double g2[3], e2[3], h2, slack2;
          M.load(C, M.b.n2, g2);
          M.apart(g2, M.b.n2, e2);
          const double exit2 = M.exit_of(e2, h2, slack2);
          if (exit2 < exit - slack) {
            name = M.b.n2;
            list = name & kNbSlotMask;
            read_ids(0);
            complete = gld(N.r2 + list);
            exit = exit2;
            h = h2;
            slack = slack2;
#pragma unroll
            for (int d = 0; d < 3; ++d) g[d] = g2[d];
            ok = exit < M.tend;
          } else {
            ok = ok && exit < exit2 - slack2;
          }
          ok &= exit < (double)M.b.t3 * (1.0 - kKeyTol);
        } else {
          ends = exit - slack > M.tend;
        }
        const uint32_t n = list, rc = name >> kNbSlotBits;
        const double v2 = M.r2_at(exit);
        // Codes of base 3 add up, one centre too many.
        const uint32_t in = PER ? M.ic + rc - kNbCentre : kNbCentre;
        double p1[3], p2[3];
        M.image(M.gb, M.ic, p1);
        M.image(g, in, p2);
        RayGeom r;
        r.len = M.h->len;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          r.a[d] = M.h->a[d];
          r.d[d] = M.dir[d];
        }
        const double sv = split_analytic(r, p1, p2);
        const double zone = slack * 1.000001 + M.h->zone;
        const float tent = M.h->tent;
        const int k = M.h->k + 1;
        const double chord = sv - M.h->s;
        ok &= h > 1e-10 && fabs(chord - exit) <= zone &&
              chord > (double)tent + zone && chord < far && v2 < far * far && n != M.c &&
              k < B.cap && (lim == INFINITY || M.clear_of((double)lim, v2));
        if (ok) {
          // The next float up keeps the stored half-width at least the zone.
          const float out = __uint_as_float(__float_as_uint((float)zone) + 1u);
          M.h->k = k;
          M.h->tent = out;
          M.ic = in;
          const uint64_t sb = (uint64_t)__double_as_longlong(sv);
          if (gl == 0)
            gst(B.seq + (size_t)M.h->j * B.cap + k,
                make_uint4((uint32_t)sb, (uint32_t)(sb >> 32), n | (in << kNbSlotBits),
                           __float_as_uint(out)));
          M.enter(n, g, p2, sv);
          ph = kMpScan;
          done = false;
        }
      }
      if (ends) {
        // The ray ends in this cell, clear of its entry and of every exit.
        const double v2 = M.r2_at(M.tend);
        if (M.tend > (double)M.h->tent && M.tend < far && v2 < far * far &&
            (lim == INFINITY || M.clear_of((double)lim, v2)))
          cells = M.h->k + 1;
      }
      if (done) {
        if (gl == 0) gst(B.c0 + M.h->j, (uint32_t)cells);
        ph = kMpDone;
      }
    }
  }
  for (int o = 32; o; o >>= 1) nball += __shfl_xor(nball, o);
  if (lane == 0 && nball) atomicAdd(&stats->queries, (unsigned long long)nball);
}

// Rays per wave of the replay, and cells whose entries it holds in LDS (at least
// the longest ray's).
constexpr int kReplayRays = 4;
constexpr int kReplayCells = 576;

// The replay of the recursion (see march.h) over the lanes of a wave.  An item
// is an interval (i, j), j >= i + 2, of a ray's cells that the recursion visits
// as a pair; its split point inserts a cell k between them and leaves (i, k)
// and (k, j).  Intervals do not depend on one another, so any lane takes any
// interval of the wave's rays.  A ray's entries are one contiguous run, copied
// to LDS first: the search for the split point's cell is a chain of reads, and
// with the entries in device memory it took 2.7 of the 11.7 ms of a call (2M
// clustered cells, 512^2 rays).  Four rays keep a wave's lanes busy (a ray has
// one interval per cell) in 15 KB, so that ten waves share a CU.
template <bool PER>
__global__ __launch_bounds__(64) void k_replay(DevCloud C, MarchRays R, MarchBufs B, int room,
                                               int pool, uint32_t *fall, Stats *stats) {
  extern __shared__ uint4 dyn[];  // room entries, then where the recursion inserts them
  uint4 *ent = dyn;
  double *ins = reinterpret_cast<double *>(dyn + room);
  uint64_t *item = reinterpret_cast<uint64_t *>(ins + (PER ? room : 0));  // the pool
  __shared__ double geo[7][kReplayRays];
  __shared__ int cells[kReplayRays], start[kReplayRays];
  __shared__ uint32_t bad[kReplayRays];
  const int lane = threadIdx.x;
  if (blockIdx.x == 0 && lane == 0) gst(B.ctr + kParts, 0u);  // for the next batch's starts
  const int64_t j0 = xcd_block(blockIdx.x, gridDim.x) * kReplayRays;
  const int64_t j = j0 + lane;
  const bool mine = lane < kReplayRays && j < R.n;
  int K = 0;
  int64_t ray = 0;
  RayGeom r;
  if (mine) {
    ray = march_ray(R, j);
    K = (int)gld(B.c0 + j);
    make_ray(R.start + 3 * ray, R.end + 3 * ray, r);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      geo[d][lane] = r.a[d];
      geo[3 + d][lane] = r.d[d];
    }
    geo[6][lane] = r.len;
  }
  if (lane < kReplayRays) {
    cells[lane] = K;
    bad[lane] = mine && K == 0 ? 1u : 0u;
  }
  __syncthreads();
  auto at = [](const uint4 &e) {
    return __longlong_as_double((long long)(((uint64_t)e.y << 32) | e.x));
  };
  // The cell k of [lo, hi] that s falls in, clear of both its boundaries, of a
  // ray of n cells from entry `e0`; -1: none.
  auto locate = [&](int e0, int n, double len, double s, int lo, int hi) {
    if (s < at(ent[e0 + lo])) return -1;
    while (hi > lo) {
      const int mid = (lo + hi + 1) >> 1;
      if (at(ent[e0 + mid]) <= s)
        lo = mid;
      else
        hi = mid - 1;
    }
    const uint4 ek = ent[e0 + lo];
    double next = len, zn = 0.0;
    if (lo + 1 < n) {
      const uint4 en = ent[e0 + lo + 1];
      next = at(en);
      zn = (double)__uint_as_float(en.w);
    }
    const double zk = lo > 0 ? (double)__uint_as_float(ek.w) : -1.0;
    return (s - at(ek) > zk && next - s > zn) ? lo : -1;
  };
  auto pack = [](int owner, int depth, int i, int k) {
    return (uint64_t)owner | ((uint64_t)depth << 8) | ((uint64_t)i << 16) | ((uint64_t)k << 32);
  };
  uint32_t given = 0, back = 0;
  for (int r0 = 0; r0 < kReplayRays;) {
    // As many rays as fit, one at least (a ray has at most `room` cells).
    int r1 = r0, held = 0;
    while (r1 < kReplayRays && (r1 == r0 || held + cells[r1] <= room)) held += cells[r1++];
    __syncthreads();
    if (lane == 0) {
      int at0 = 0;
      for (int q = r0; q < r1; ++q) {
        start[q] = at0;
        at0 += cells[q];
      }
    }
    __syncthreads();
    for (int q = r0; q < r1; ++q)
      for (int k = lane; k < cells[q]; k += 64)
        ent[start[q] + k] = gld(B.seq + (size_t)(j0 + q) * B.cap + k);
    __syncthreads();
    // The rays' first intervals, by their own lanes.
    uint64_t first[2] = {0, 0};
    int nfirst = 0;
    if (lane >= r0 && lane < r1 && K > 0) {
      const int e0 = start[lane];
      const uint32_t a = ent[e0].z & kNbSlotMask, b = ent[e0 + K - 1].z & kNbSlotMask;
      bool fail = false;
      if constexpr (PER) {
        ins[e0] = 0.0;
        ins[e0 + K - 1] = r.len;
        if (a == b) {
          // Same cell at both ends: dyadic probes for another one
          // (src/ray.cpp:220-246).
          fail = true;
          bool go = K > 1;
          for (int lv = 1; go && lv <= 10; ++lv)
            for (int i = 1; go && i < (1 << lv); i += 2) {
              const double mid = r.len * i / (1 << lv);
              const int k = locate(e0, K, r.len, mid, 0, K - 1);
              if (k < 0) {
                go = false;
              } else if ((ent[e0 + k].z & kNbSlotMask) != a) {
                go = false;
                fail = false;
                ins[e0 + k] = mid;
                if (k >= 2) first[nfirst++] = pack(lane, 1, 0, k);
                if (K - 1 - k >= 2) first[nfirst++] = pack(lane, 0, k, K - 1);
              }
            }
        } else if (K >= 3) {
          first[nfirst++] = pack(lane, 0, 0, K - 1);
        }
      } else {
        fail = a == b && K > 1;
        if (!fail && K >= 3) first[nfirst++] = pack(lane, 0, 0, K - 1);
      }
      if (fail) bad[lane] = 1u;
    }
    int count = 0;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const bool put = nfirst > q;
      const uint64_t m = __ballot(put);
      const int p = count + __popcll(m & ((1ull << lane) - 1ull));
      if (put) {
        if (p < pool) {
          item[p] = first[q];
        } else {
          bad[lane] = 1u;
          ++back;
        }
      }
      count = min(pool, count + (int)__popcll(m));
    }
    __syncthreads();
    while (count > 0) {
      const int take = count < 64 ? count : 64;
      count -= take;
      uint64_t it = 0;
      const bool work = lane < take;
      if (work) it = item[count + lane];
      __syncthreads();
      uint64_t child[2] = {0, 0};
      bool put[2] = {false, false};
      int owner = 0;
      if (work) {
        owner = (int)(it & 255u);
        const int depth = (int)((it >> 8) & 255u);
        const int i = (int)((it >> 16) & 0xFFFFu), jj = (int)((it >> 32) & 0xFFFFu);
        if (owner != lane) ++given;
        if (!bad[owner]) {
          const int e0 = start[owner], n = cells[owner];
          RayGeom g;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            g.a[d] = geo[d][owner];
            g.d[d] = geo[3 + d][owner];
          }
          g.len = geo[6][owner];
          const uint32_t ci = ent[e0 + i].z & kNbSlotMask, cj = ent[e0 + jj].z & kNbSlotMask;
          bool ok = ci != cj && depth < 120;
          double s = 0.0, p1[3], p2[3];
          double sc = 0.0, sn = g.len;
          if constexpr (PER) {
            sc = ins[e0 + i];
            sn = ins[e0 + jj];
          }
          const bool analytic = split_point<PER>(C, g, ci, cj, sc, sn, s, p1, p2);
          int k = -1;
          if (ok && analytic) {
            if constexpr (PER) {
              const double l2 = sc + 1e-15, h2 = sn - 1e-15;
              s = (s < l2) ? l2 : ((h2 < s) ? h2 : s);
            }
            k = locate(e0, n, g.len, s, i, jj);
          } else if (PER && ok) {
            // The reference's bisection between the two cells.
            double lo = sc, hi = sn;
            for (int q = 0; q < 64; ++q) {
              const double mid = 0.5 * (lo + hi);
              const int km = locate(e0, n, g.len, mid, i, jj);
              if (km < 0) break;
              const uint32_t cm = ent[e0 + km].z & kNbSlotMask;
              if (cm != ci && cm != cj) {
                const double l2 = sc + 1e-15, h2 = sn - 1e-15;
                s = (mid < l2) ? l2 : ((h2 < mid) ? h2 : mid);
                k = s == mid ? km : -1;
                break;
              }
              if (cm == ci)
                lo = mid;
              else
                hi = mid;
              if (hi - lo < 1e-11) break;
            }
          }
          if (k <= i || k >= jj) {
            ok = false;
          } else {
            const uint32_t ck = ent[e0 + k].z & kNbSlotMask;
            ok = ok && ck != ci && ck != cj;
          }
          if (!ok) {
            bad[owner] = 1u;
          } else {
            if constexpr (PER) ins[e0 + k] = s;
            put[0] = jj - k >= 2;
            child[0] = pack(owner, depth, k, jj);
            put[1] = k - i >= 2;
            child[1] = pack(owner, depth + 1, i, k);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint64_t m = __ballot(put[q]);
        const int p = count + __popcll(m & ((1ull << lane) - 1ull));
        if (put[q]) {
          if (p < pool) {
            item[p] = child[q];
          } else {
            bad[owner] = 1u;  // no room: the engine walks the ray
            ++back;
          }
        }
        count = min(pool, count + (int)__popcll(m));
      }
      __syncthreads();
    }
    r0 = r1;
  }
  if (mine && bad[lane]) {
    if (K) gst(B.c0 + j, 0u);
    const unsigned long long q = atomicAdd(&stats->fallback, 1ull);
    gst(fall + q, (uint32_t)ray);
  }
  for (int o = 32; o; o >>= 1) {
    given += __shfl_xor(given, o);
    back += __shfl_xor(back, o);
  }
  if (lane == 0) {
    if (given) atomicAdd(&stats->intervals, (unsigned long long)given);
    if (back) atomicAdd(&stats->intervals_back, (unsigned long long)back);
  }
}

// The IO that takes a lane's segments, and the record pool when there is one.
template <class IO>
struct Emit {
  using Inner = IO;
  static constexpr bool kRecord = false;
  static __device__ __forceinline__ const IO &inner(const IO &io) { return io; }
};
template <class I>
struct Emit<MarchRecordIO<I>> {
  using Inner = I;
  static constexpr bool kRecord = true;
  static __device__ __forceinline__ const I &inner(const MarchRecordIO<I> &io) { return io.inner; }
};

// Hands the segments of the batch's rays to the sinks, one ray per lane; with
// records, the wave then writes them ray by ray, its lanes along the ray, so
// that a ray's records are one run of whole lines (a lane writing its own ray's
// took 2.4 ms more at 2M cells, 512^2 rays).
template <class IO>
__global__ __launch_bounds__(64) void k_emit(MarchRays R, MarchBufs B, IO io, ErrRec *err,
                                             Stats *stats) {
  const int lane = threadIdx.x;
  const int64_t j0 = xcd_block(blockIdx.x, gridDim.x) * 64;
  const int64_t j = j0 + lane;
  const bool mine = j < R.n;
  const int K = mine ? (int)gld(B.c0 + j) : 0;
  const uint4 *ent = B.seq + (size_t)(mine ? j : 0) * B.cap;
  auto at = [](const uint4 &e) {
    return __longlong_as_double((long long)(((uint64_t)e.y << 32) | e.x));
  };
  int64_t ray = 0;
  double len = 0.0;
  if (K > 0) {
    ray = march_ray(R, j);
    RayGeom r;
    make_ray(R.start + 3 * ray, R.end + 3 * ray, r);
    len = r.len;
    const auto &in = Emit<IO>::inner(io);
    typename Emit<IO>::Inner::Sink sk;
    in.begin(ray, sk);
    // Four segments at a time, their reads in flight together.
    uint4 e = gld(ent);
    int k = 0;
    for (; k + 4 < K; k += 4) {
      uint4 n[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) n[i] = gld(ent + k + 1 + i);
      sk.seg(e.z & kNbSlotMask, at(e), at(n[0]));
#pragma unroll
      for (int i = 0; i < 3; ++i) sk.seg(n[i].z & kNbSlotMask, at(n[i]), at(n[i + 1]));
      e = n[3];
    }
    for (; k < K; ++k) {
      uint4 n = e;
      double b = len;
      if (k + 1 < K) {
        n = gld(ent + k + 1);
        b = at(n);
      }
      sk.seg(e.z & kNbSlotMask, at(e), b);
      e = n;
    }
    const int rc = in.end(ray, sk);
    if (rc) report_error(err, rc, ray, 0.0, 0.0, 0.0, 0u, 0u);
  }
  int inc = K;
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o);
    if (lane >= o) inc += v;
  }
  const int total = __shfl(inc, 63);
  if (lane == 0 && total) atomicAdd(&stats->segments, (unsigned long long)total);
  if constexpr (Emit<IO>::kRecord) {
    // One run of whole chunks; the rest of the last one is marked unwritten.
    const int whole = (total + kRecChunk - 1) / kRecChunk * kRecChunk;
    unsigned long long base = 0;
    if (lane == 0 && whole) base = atomicAdd(io.pool.head, (unsigned long long)whole);
    base = __shfl(base, 0);
    if (base + (unsigned long long)whole > io.pool.cap) {
      if (lane == 0) atomicOr(io.pool.overflow, 1);
      return;
    }
    if (lane < whole - total) gst(&io.pool.rec[base + total + lane].ray, kNone);
    for (int q = 0; q < 64; ++q) {
      const int n = __shfl(K, q), off = __shfl(inc, q) - n;
      const uint32_t id = (uint32_t)__shfl((int)ray, q);
      const double end = __shfl(len, q);
      const uint4 *src = B.seq + (size_t)(j0 + q) * B.cap;
      for (int k = lane; k < n; k += 64) {
        const uint4 e = gld(src + k);
        const double b = k + 1 < n ? at(gld(src + k + 1)) : end;
        SegRec *o = io.pool.rec + base + off + k;
        // Both halves whole, through the cache, which joins them: 1.51 ms for
        // 52M segments of 8M cells, against 2.22 with the padding left out and
        // streaming stores.
        const uint64_t ds = (uint64_t)__double_as_longlong(b - at(e));
        gst(reinterpret_cast<uint4 *>(o), make_uint4(e.z & kNbSlotMask, id, (uint32_t)k, 0u));
        gst(reinterpret_cast<uint4 *>(o) + 1,
            make_uint4((uint32_t)ds, (uint32_t)(ds >> 32), 0u, 0u));
      }
    }
  }
}

}  // namespace

void march_build_lists(const DevCloud &C, uint32_t *nb, float *r2, hipStream_t st) {
  const unsigned grid = (C.n + kNbWindow - 1) / kNbWindow;
  if (C.periodic)
    k_neighbors<true><<<grid, 64, 0, st>>>(C, nb, r2);
  else
    k_neighbors<false><<<grid, 64, 0, st>>>(C, nb, r2);
}

void march_build_boxes(const DevCloud &C, uint32_t nodes, BNode *boxes, uint32_t *work,
                       hipStream_t st) {
  if (!nodes) return;
  uint32_t *parent = work, *arrived = work + nodes, *leaf_parent = work + 2 * (size_t)nodes;
  k_box_parents<<<(nodes + 255) / 256, 256, 0, st>>>(C.nodes, nodes, C.root, boxes, parent,
                                                     leaf_parent, arrived);
  k_box_climb<<<(C.n + 255) / 256, 256, 0, st>>>(C.gen, C.n, boxes, parent, leaf_parent, arrived);
}

int march_locate_grid(int cus) { return 2 * cus; }

template <bool PER>
static void march_batch_p(const MarchCall &m) {
  // (The batch's own part of the list of rays left to the engine, empty yet.)
  uint32_t *rest = m.fall + m.R.base;
  auto locate = [&](auto kernel, int lanes) {
    const int64_t blocks = (m.R.n * lanes + kBlock - 1) / kBlock;
    kernel<<<(int)std::min<int64_t>(32ll * m.cus, blocks), kBlock, 0, m.st>>>(m.C, m.N, m.R, m.B,
                                                                             rest);
  };
  if (m.R.n >= 64ll * m.cus)
    locate(k_locate<PER, 4>, 4);
  else
    locate(k_locate<PER, 16>, 16);
  const int64_t far_blocks = (m.R.n + 1) / 2;
  k_locate_far<PER><<<(int)std::min<int64_t>(march_locate_grid(m.cus), far_blocks), kBlock, 0,
                      m.st>>>(m.C, m.S, m.R, m.B, rest);
  // As many waves as the chip holds at once, or as the rays need.
  double far = DBL_MAX;
  if (PER) far = 0.2 * std::min(m.C.box[0], std::min(m.C.box[1], m.C.box[2]));
  auto go = [&](auto kernel, int rays, int batch) {
    const unsigned waves =
        (unsigned)std::min<int64_t>(16ll * m.cus, (m.R.n + rays - 1) / rays);
    kernel<<<waves, 64, 0, m.st>>>(m.C, m.N, m.R, m.B, far, m.stats, batch);
  };
  // Rays per wave.  The fewer rays there are, the more lanes are worth a ray:
  // its crossings are a chain, and the last rays' chains end the launch.
  // Measured with 4, 8 and 16 lanes (ms): 512^2 rays through clustered periodic
  // cells 7.1, 8.4, 10.5; 384^2 4.8, 4.2, 5.6; 256^2 4.9, 3.9, 4.1; 16^2 .17,
  // .17, .10; without images, where searches are cheaper, 300 x 257 rays 2.8,
  // 3.2, 3.9; 128^2 .61, .52, .65.  Chunks of 32 or 64 entries save rounds (16
  // entries: 384^2 4.6, 300 x 257 3.0, 128^2 .57), but with images and 4 lanes
  // they cost registers (512^2 7.8).
  const int64_t many = (PER ? 768ll : 256ll) * m.cus;
  if (m.R.n >= many)
    go(k_march<PER, 4, PER ? 4 : 8>, 16, 4);  // (searches for 3, 6 or 8 waiting rays: no better)
  else if (m.R.n >= 64ll * m.cus)
    go(k_march<PER, 8, 4>, 8, 2);
  else
    go(k_march<PER, 16, 4>, 4, 1);
}

void march_batch(const MarchCall &m, bool periodic) {
  if (periodic)
    march_batch_p<true>(m);
  else
    march_batch_p<false>(m);
}

template <class IO>
void march_finish(const MarchCall &m, bool periodic, const IO &io) {
  auto waves = [&](int64_t rays) {
    return (unsigned)(((m.R.n + rays - 1) / rays + kParts - 1) / kParts * kParts);
  };
  const int room = std::max(kReplayCells, m.B.cap);
  // Intervals a wave holds: breadth grows by a wave's worth per level below the
  // 64th interval, so rays of up to 640 cells need 256 (an overflow leaves the
  // ray to the engine).  512 for all took a wave per CU: 2M cells, 512^2 rays
  // .96 ms against .88, 4M cells 3.07 against 2.78.
  const int pool = std::min(m.pool, m.B.cap <= 640 ? 256 : 512);
  const size_t lds = (size_t)room * (sizeof(uint4) + (periodic ? sizeof(double) : 0)) +
                     (size_t)pool * sizeof(uint64_t);
  if (periodic)
    k_replay<true><<<waves(kReplayRays), 64, lds, m.st>>>(m.C, m.R, m.B, room, pool, m.fall,
                                                          m.stats);
  else
    k_replay<false><<<waves(kReplayRays), 64, lds, m.st>>>(m.C, m.R, m.B, room, pool, m.fall,
                                                           m.stats);
  k_emit<IO><<<waves(64), 64, 0, m.st>>>(m.R, m.B, io, m.err, m.stats);
}

#define VT_FINISH(...) template void march_finish<__VA_ARGS__>(const MarchCall &, bool, const __VA_ARGS__ &);
VT_FINISH(SumIO<1>)
VT_FINISH(SumIO<2>)
VT_FINISH(SumIO<3>)
VT_FINISH(SumIO<4>)
VT_FINISH(SumDynIO)
VT_FINISH(ExtIO<true>)
VT_FINISH(ExtIO<false>)
VT_FINISH(VolIO)
VT_FINISH(CountIO)
VT_FINISH(SegIO)
VT_FINISH(FillIO<SumDynIO>)
VT_FINISH(FillIO<ExtIO<true>>)
VT_FINISH(FillIO<ExtIO<false>>)
VT_FINISH(FillIO<VolIO>)
VT_FINISH(MarchRecordIO<SumIO<1>>)
VT_FINISH(MarchRecordIO<SumDynIO>)
VT_FINISH(MarchRecordIO<VolIO>)
#undef VT_FINISH

}  // namespace vt
