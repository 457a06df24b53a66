// (tile, stage) units of a product dealt over one workgroup per CU: who owns what, and the exchange of
// partial sums between the workgroups of a tile (gemm_i4.hip, gemm_i4_exact.hip).
#pragma once

#include "krm_internal.h"

namespace krm {
namespace {

// One span of units dealt over all workgroups, in contiguous ranges that differ by one unit, or (tile_groups
// > 0) the units of each tile dealt so over workgroups of its own.
struct UnitDeal {
  uint32_t stages_per_tile;
  uint32_t tile_groups;
  uint32_t units_lo, extra;  // workgroup i of a span owns units_lo + (i < extra) units
  float* partials;           // [2 * workgroups] slots of 128 x 256 floats
  uint32_t* tickets;         // one counter per tile, kTicketStride words apart, zero at rest
};
// (a division by what only the launch knows is twenty instructions: none where there is one span)
__device__ inline uint32_t deal_begin(const UnitDeal& d, uint32_t v) {
  const uint32_t tile = d.tile_groups ? v / d.tile_groups : 0u, i = v - tile * d.tile_groups;
  return tile * d.stages_per_tile + i * d.units_lo + (i < d.extra ? i : d.extra);
}
__device__ inline uint32_t deal_units(const UnitDeal& d, uint32_t v) {
  const uint32_t i = d.tile_groups ? v % d.tile_groups : v;
  return d.units_lo + (i < d.extra ? 1u : 0u);
}
__device__ inline uint32_t deal_owner(const UnitDeal& d, uint32_t unit) {
  const uint32_t tile = d.tile_groups ? unit / d.stages_per_tile : 0u, at = unit - tile * d.stages_per_tile;
  const uint32_t big = d.extra * (d.units_lo + 1u);
  return tile * d.tile_groups + (at < big ? at / (d.units_lo + 1u) : d.extra + (at - big) / d.units_lo);
}
constexpr uint32_t kPartialFloats = 128u * 256u;

typedef float float4_t __attribute__((ext_vector_type(4)));
// 16 bytes written through to / read from memory that every XCD sees (device scope).
__device__ inline void publish4(float4_t* p, float4_t v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
__device__ inline float4_t observe4(const float4_t* p) {
  float4_t v;
  asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=v"(v) : "v"(p) : "memory");
  return v;
}

// The eight requests above have landed; the values pass through so that no use moves ahead.
__device__ inline void landed(float4_t (&p)[8]) {
  asm volatile("s_waitcnt vmcnt(0)"
               : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]), "+v"(p[4]), "+v"(p[5]), "+v"(p[6]),
                 "+v"(p[7])::"memory");
}

}  // namespace
}  // namespace krm
