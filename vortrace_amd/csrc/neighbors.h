// Neighbour lists: for every generator the kNbMax generators nearest to it
// (images included in periodic boxes), nearest first, and the radius within
// which the list is complete.
//
// One wave per kNbWindow consecutive slots builds the lists of the leaves that
// start there, leaf by leaf: a radius is estimated from the generators around
// the leaf in slot order, every generator within that radius of the leaf's box
// is collected from the kd-tree (64 nodes tested at a time), and each
// generator of the leaf ranks the collected ones by distance.  A leaf's
// generators share one traversal and one set of candidates.  Bound by VALU
// issue, the ranking a third of it: 2M clustered points 12.1 ms, 8M 29.0 (13.9
// and 39.7 with ties ranked in the same pass).  64 entries: at 48, 2 % of the
// crossings of a clustered mesh have more generators in reach than the list
// holds, at 64 1.2 %, at 96 0.9 %.
#pragma once
#include "knn.h"
#include "march.h"

namespace vt {

constexpr int kNbWindow = 16;
constexpr int kNbCand = 1024;   // candidates collected per leaf
constexpr int kNbStack = 512;   // pending nodes of the traversal
constexpr int kNbLeaves = 512;  // leaves found by it
constexpr int kNbSort = 128;    // candidates ranked per generator

struct NbShared {
  uint32_t stack[kNbStack];
  uint32_t leaves[kNbLeaves];
  uint32_t cand[kNbCand];
  alignas(16) float key[kNbSort];
  uint32_t ent[kNbSort];
};

__device__ __forceinline__ int lane_prefix(uint64_t m, int lane) {
  return __popcll(m & ((1ull << lane) - 1ull));
}
__device__ __forceinline__ double wave_min(double v) {
  for (int o = 32; o; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
  for (int o = 32; o; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// Squared distance from generator coordinates to a box.
__device__ __forceinline__ double box_d2(const double (&g)[3], const double (&lo)[3],
                                         const double (&hi)[3]) {
  double s = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double t = fmax(fmax(lo[d] - g[d], g[d] - hi[d]), 0.0);
    s += t * t;
  }
  return s;
}

// Appends the generators within sqrt(r2) of the box (lo, hi), as seen through
// image `code` (box already shifted into that image's frame), to sh.cand.
// Returns false when a buffer is full.
__device__ inline bool nb_collect(const DevCloud &C, NbShared &sh, int lane,
                                  const double (&lo)[3], const double (&hi)[3], double r,
                                  double r2, uint32_t code, int &nc) {
  if (lane == 0) {
    if (C.root & kRefLeaf)
      sh.leaves[0] = C.root;
    else
      sh.stack[0] = C.root;
  }
  int ns = (C.root & kRefLeaf) ? 0 : 1, nl = (C.root & kRefLeaf) ? 1 : 0;
  __syncthreads();
  while (ns > 0) {
    const int take = ns < 64 ? ns : 64;
    ns -= take;
    uint32_t c[2] = {kNone, kNone};
    if (lane < take) {
      const DNodeV nd = load_node(C.nodes, sh.stack[ns + lane]);
      const double ql = sel3(lo[0], lo[1], lo[2], nd.dim) - r;
      const double qh = sel3(hi[0], hi[1], hi[2], nd.dim) + r;
      if (ql <= nd.lo) c[0] = nd.c1;
      if (qh >= nd.hi) c[1] = nd.c2;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const bool leaf = c[b] != kNone && (c[b] & kRefLeaf);
      const bool inner = c[b] != kNone && !(c[b] & kRefLeaf);
      const uint64_t ml = __ballot(leaf), mi = __ballot(inner);
      if (nl + __popcll(ml) > kNbLeaves || ns + __popcll(mi) > kNbStack) return false;
      if (leaf) sh.leaves[nl + lane_prefix(ml, lane)] = c[b];
      if (inner) sh.stack[ns + lane_prefix(mi, lane)] = c[b];
      nl += __popcll(ml);
      ns += __popcll(mi);
    }
    __syncthreads();
  }
  for (int l0 = 0; l0 < nl; l0 += 64) {
    const bool have = l0 + lane < nl;
    uint32_t s0 = 0, cnt = 0;
    if (have) {
      s0 = sh.leaves[l0 + lane] & kSlotMask;
      cnt = (uint32_t)gld(&C.gen[s0].end) - s0;
    }
    for (uint32_t t = 0; t < (uint32_t)kLeafMaxSize; ++t) {
      if (!__ballot(t < cnt)) break;
      bool in = false;
      if (t < cnt) {
        const Gen *p = C.gen + s0 + t;
        const double2 xy = gld(reinterpret_cast<const double2 *>(p));
        const double g[3] = {xy.x, xy.y, gld(&p->z)};
        in = box_d2(g, lo, hi) <= r2;
      }
      const uint64_t m = __ballot(in);
      if (nc + __popcll(m) > kNbCand) return false;
      if (in) sh.cand[nc + lane_prefix(m, lane)] = (s0 + t) | (code << kNbSlotBits);
      nc += __popcll(m);
    }
  }
  __syncthreads();
  return true;
}

template <bool PER>
__global__ __launch_bounds__(64) void k_neighbors(DevCloud C, uint32_t *nb, float *nr2) {
  __shared__ NbShared sh;
  const int lane = threadIdx.x;
  const uint32_t w0 = blockIdx.x * kNbWindow;
  const uint32_t w1 = min(w0 + (uint32_t)kNbWindow, C.n);
  uint32_t s0 = w0;
  // The first leaf that starts in the window.
  if (s0 < w1) {
    const uint32_t st = (uint32_t)gld(&C.gen[s0].start);
    if (st != s0) s0 = (uint32_t)gld(&C.gen[s0].end);
  }
  double rmax = DBL_MAX;
  if constexpr (PER) rmax = 0.499 * fmin(C.box[0], fmin(C.box[1], C.box[2]));
  while (s0 < w1) {
    const uint32_t s1 = (uint32_t)gld(&C.gen[s0].end);
    const int m = (int)(s1 - s0);
    // The leaf's box.
    double lo[3], hi[3];
    {
      const uint32_t s = s0 + (uint32_t)(lane < m ? lane : 0);
      const double2 xy = gld(reinterpret_cast<const double2 *>(C.gen + s));
      const double g[3] = {xy.x, xy.y, gld(&C.gen[s].z)};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        lo[d] = wave_min(g[d]);
        hi[d] = wave_max(g[d]);
      }
    }
    // A radius that holds about kNbMax generators: the distance from the
    // leaf's centre of the 56th nearest of the 256 generators around it in
    // slot order.
    double r2;
    {
      const uint32_t span = min(256u, C.n);
      uint32_t a = s0 + (uint32_t)(m / 2);
      a = a > span / 2 ? a - span / 2 : 0u;
      if (a + span > C.n) a = C.n - span;
      float d2[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t k = (uint32_t)(lane + 64 * i);
        const uint32_t s = a + (k < span ? k : 0u);
        const double2 xy = gld(reinterpret_cast<const double2 *>(C.gen + s));
        const double e0 = xy.x - 0.5 * (lo[0] + hi[0]), e1 = xy.y - 0.5 * (lo[1] + hi[1]),
                     e2 = gld(&C.gen[s].z) - 0.5 * (lo[2] + hi[2]);
        d2[i] = k < span ? (float)(e0 * e0 + e1 * e1 + e2 * e2) : INFINITY;
      }
      const int want = min(56, (int)span);
      uint32_t t = 0;  // the largest float (by bits) with fewer than `want` at or below it
      for (int b = 30; b >= 12; --b) {
        const uint32_t u = t | (1u << b);
        if (u > 0x7F7FFFFFu) continue;
        const float f = __uint_as_float(u);
        int cnt = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) cnt += __popcll(__ballot(d2[i] <= f));
        if (cnt < want) t = u;
      }
      r2 = (double)__uint_as_float(t + (1u << 12));
      if (!(r2 < 1e36)) r2 = 0.0;  // squares near the end of float: no list
    }
    if constexpr (PER) r2 = fmin(r2, rmax * rmax);
    // Collect every generator within the radius of the leaf's box.  Where that
    // finds too many (a dense clump beside a sparse leaf), each generator of
    // the leaf collects around itself, within a radius reduced until they fit.
    int nc = 0;
    auto collect = [&](const double (&blo)[3], const double (&bhi)[3], double rr) {
      const double r = sqrt(rr) * (1.0 + 1e-12);
      nc = 0;
      bool ok = true;
      if constexpr (PER) {
        for (int code = 0; ok && code < 27; ++code) {
          const int ish[3] = {code / 9 - 1, (code / 3) % 3 - 1, code % 3 - 1};
          double l2[3], h2[3];
          bool hit = true;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            l2[d] = blo[d] - ish[d] * C.box[d];
            h2[d] = bhi[d] - ish[d] * C.box[d];
            hit &= l2[d] - r <= C.rb_hi[d] && h2[d] + r >= C.rb_lo[d];
          }
          if (hit) ok = nb_collect(C, sh, lane, l2, h2, r, rr, (uint32_t)code, nc);
        }
      } else {
        ok = nb_collect(C, sh, lane, blo, bhi, r, rr, kNbCentre, nc);
      }
      __syncthreads();
      return ok;
    };
    const bool together = collect(lo, hi, r2);
    const double r2leaf = r2;
    for (int p = 0; p < m; ++p) {
      const uint32_t self = s0 + (uint32_t)p;
      const double2 cxy = gld(reinterpret_cast<const double2 *>(C.gen + self));
      const double cz = gld(&C.gen[self].z);
      if (!together) {
        const double own[3] = {cxy.x, cxy.y, cz};
        r2 = r2leaf;
        for (int tries = 0; !collect(own, own, r2); ++tries) {
          r2 *= 0.6;
          if (tries == 64) {
            r2 = -1.0;
            nc = 0;
            break;
          }
        }
      }
      const int nch = (nc + 63) / 64;
      float d2[kNbCand / 64];
      const float lim = (float)r2 * 0.999998f;
#pragma unroll
      for (int i = 0; i < kNbCand / 64; ++i) {
        d2[i] = INFINITY;
        if (i < nch) {
          const int k = lane + 64 * i;
          if (k < nc) {
            const uint32_t e = sh.cand[k];
            const uint32_t s = e & kNbSlotMask;
            const double2 xy = gld(reinterpret_cast<const double2 *>(C.gen + s));
            double e0 = xy.x - cxy.x, e1 = xy.y - cxy.y, e2 = gld(&C.gen[s].z) - cz;
            const uint32_t code = e >> kNbSlotBits;
            if (PER && code != kNbCentre) {
              e0 += ((int)(code / 9) - 1) * C.box[0];
              e1 += ((int)(code / 3) % 3 - 1) * C.box[1];
              e2 += ((int)(code % 3) - 1) * C.box[2];
            }
            const float f = (float)(e0 * e0 + e1 * e1 + e2 * e2);
            if (e != (self | (kNbCentre << kNbSlotBits)) && f <= lim) d2[i] = f;
          }
        }
      }
      auto count = [&](float t) {
        int c = 0;
#pragma unroll
        for (int i = 0; i < kNbCand / 64; ++i)
          if (i < nch) c += __popcll(__ballot(d2[i] <= t));
        return c;
      };
      // The largest radius with at most kNbSort candidates (at least kNbMax
      // when the ties allow it).
      float t = lim;
      int cnt = count(t);
      if (cnt > kNbSort) {
        uint32_t a = 0u, b = __float_as_uint(t);  // count(a) <= kNbSort < count(b)
        int ca = count(0.0f);
        if (ca > kNbSort) {
          a = 0u;
          b = 0u;
          ca = 0;
        }
        while (b > a + 1u) {
          const uint32_t mid = a + (b - a) / 2u;
          const int c = count(__uint_as_float(mid));
          if (c <= kNbSort) {
            a = mid;
            ca = c;
            if (c >= kNbMax) break;
          } else {
            b = mid;
          }
        }
        t = b == 0u ? -1.0f : __uint_as_float(a);
        cnt = ca;
      }
      int n = 0;
#pragma unroll
      for (int i = 0; i < kNbCand / 64; ++i) {
        if (i < nch) {
          const bool in = d2[i] <= t;
          const uint64_t mk = __ballot(in);
          if (in) {
            const int q = n + lane_prefix(mk, lane);
            sh.key[q] = d2[i];
            sh.ent[q] = sh.cand[lane + 64 * i];
          }
          n += __popcll(mk);
        }
      }
      if (lane < 4 && n + lane < kNbSort) sh.key[n + lane] = INFINITY;
      __syncthreads();
      // Rank by (distance, place); each lane places up to two candidates.  The
      // places are only looked at when two distances are equal (the ranks then
      // do not add up to 0 + 1 + ... + n - 1).
      float k0 = lane < n ? sh.key[lane] : INFINITY;
      float k1 = lane + 64 < n ? sh.key[lane + 64] : INFINITY;
      int r0 = 0, r1 = 0;
      for (int j = 0; j < n; j += 4) {
        const float4 k = *reinterpret_cast<const float4 *>(sh.key + j);
        r0 += (k.x < k0) + (k.y < k0) + (k.z < k0) + (k.w < k0);
        r1 += (k.x < k1) + (k.y < k1) + (k.z < k1) + (k.w < k1);
      }
      int sum = (lane < n ? r0 : 0) + (lane + 64 < n ? r1 : 0);
      for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o);
      if (sum != n * (n - 1) / 2) {
        for (int j = 0; j < n; ++j) {
          const float kj = sh.key[j];
          r0 += (kj == k0 && j < lane) ? 1 : 0;
          r1 += (kj == k1 && j < lane + 64) ? 1 : 0;
        }
      }
      uint32_t *out = nb + (size_t)self * kNbMax;
      if (lane < n && r0 < kNbMax) gst(out + r0, sh.ent[lane]);
      if (lane + 64 < n && r1 < kNbMax) gst(out + r1, sh.ent[lane + 64]);
      if (lane >= n && lane < kNbMax) gst(out + lane, kNone);
      // Complete below: the radius searched, or the last entry's distance.
      const uint64_t l0 = __ballot(lane < n && r0 == kNbMax - 1);
      const uint64_t l1 = __ballot(lane + 64 < n && r1 == kNbMax - 1);
      float comp = t < lim ? t : lim;
      if (l0) comp = __shfl(k0, __ffsll((unsigned long long)l0) - 1);
      if (l1) comp = __shfl(k1, __ffsll((unsigned long long)l1) - 1);
      if (lane == 0) gst(nr2 + self, fmaxf(comp * 0.999998f, 0.0f));
      __syncthreads();
    }
    s0 = s1;
  }
}

}  // namespace vt
