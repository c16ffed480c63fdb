// uniform_load.h -- wave-uniform reads through the scalar cache.
//
// A 16-byte-per-lane vector load holds the address unit for 16 or more cycles
// whatever the lanes; an address that is the same in every lane is read once
// per wave through the scalar cache instead.  Only for memory that no kernel
// running at the same time writes.
#pragma once
#include "common.h"
#include "cubql_amd/traversal.hip.h"

namespace cubql {

typedef float vec4f __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) vec4f *uniform_vec4;

__device__ __forceinline__ uniform_vec4 uniform_ptr(const void *p) { return (uniform_vec4)(uintptr_t)p; }

// The child pair at nodes[i0], i0 the same in every lane.
__device__ __forceinline__ void load_pair_uniform(const cubql_node3f *nodes, uint32_t i0, cubql_dev::QNode &n0,
                                                  cubql_dev::QNode &n1) {
  const uniform_vec4 p = uniform_ptr(nodes + i0);
  const vec4f a = p[0], b = p[1], c = p[2], d = p[3];
  n0.a = make_float4(a.x, a.y, a.z, a.w);
  n0.b = make_float4(b.x, b.y, b.z, b.w);
  n1.a = make_float4(c.x, c.y, c.z, c.w);
  n1.b = make_float4(d.x, d.y, d.z, d.w);
}

}  // namespace cubql
