// The kd-tree's boxes: for every inner node the tight boxes of its two
// children, in floats rounded outward, so that a search around a point that
// moves (the exit of a march) tests a subtree from one 64-byte record and
// keeps nothing but references on its stack.  Built on the device, from the
// leaves up: the second child to arrive carries the union to the parent.
#pragma once
#include "device_common.h"

namespace vt {

struct alignas(64) BNode {
  float lo1[3], hi1[3];  // child1
  float lo2[3], hi2[3];  // child2
  uint32_t c1, c2;       // references as in DNode, dimension bits removed
  uint32_t pad[2];
};
static_assert(sizeof(BNode) == 64, "box node must be 64 bytes");

// A float at or below / at or above v.
__device__ __forceinline__ float float_below(double v) {
  float f = (float)v;
  if ((double)f > v) f = __uint_as_float(f > 0.0f ? __float_as_uint(f) - 1u
                                                  : (f < 0.0f ? __float_as_uint(f) + 1u
                                                              : 0x80000001u));
  return f;
}
__device__ __forceinline__ float float_above(double v) { return -float_below(-v); }

// Children references, and who a node's or leaf's parent is: 2 * node + which
// (leaves by their first slot).
static __global__ void k_box_parents(const DNode *nodes, uint32_t n, uint32_t root, BNode *bn,
                              uint32_t *parent, uint32_t *leaf_parent, uint32_t *arrived) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DNodeV nd = load_node(nodes, i);
  bn[i].c1 = nd.c1;
  bn[i].c2 = nd.c2;
  arrived[i] = 0u;
  if (i == root) parent[i] = kNone;
  const uint32_t c[2] = {nd.c1, nd.c2};
#pragma unroll
  for (uint32_t b = 0; b < 2; ++b) {
    if (c[b] & kRefLeaf)
      leaf_parent[c[b] & kSlotMask] = 2 * i + b;
    else
      parent[c[b]] = 2 * i + b;
  }
}

static __global__ void k_box_climb(const Gen *gen, uint32_t n, BNode *bn, const uint32_t *parent,
                            const uint32_t *leaf_parent, uint32_t *arrived) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || gld(&gen[s].start) != s) return;
  const uint32_t end = gld(&gen[s].end);
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint32_t t = s; t < end; ++t) {
    const double g[3] = {gld(&gen[t].x), gld(&gen[t].y), gld(&gen[t].z)};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = fminf(lo[d], float_below(g[d]));
      hi[d] = fmaxf(hi[d], float_above(g[d]));
    }
  }
  uint32_t p = gld(leaf_parent + s);
  for (;;) {
    BNode *b = bn + (p >> 1);
    float *mine = (p & 1u) ? b->lo2 : b->lo1;  // lo then hi, six floats
    float *other = (p & 1u) ? b->lo1 : b->lo2;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      __hip_atomic_store(mine + d, lo[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(mine + 3 + d, hi[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // The sibling's box is visible to the second arrival.
    if (__hip_atomic_fetch_add(arrived + (p >> 1), 1u, __ATOMIC_ACQ_REL,
                               __HIP_MEMORY_SCOPE_AGENT) == 0u)
      return;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = fminf(lo[d], __hip_atomic_load(other + d, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT));
      hi[d] = fmaxf(hi[d], __hip_atomic_load(other + 3 + d, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT));
    }
    p = gld(parent + (p >> 1));
    if (p == kNone) return;
  }
}

}  // namespace vt
