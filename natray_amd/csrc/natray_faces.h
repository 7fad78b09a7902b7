// Which tagged halo words a lane of the solve's quads reads, waits for and publishes: the rules
// alone, on plain values, so that a host program can check what the kernels run by (a solve
// whose waves disagree on them loses words or waits for ever).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace natray {

// A lane of a set of four consecutive blocks: lane 16 q + 4 x + y holds the column of cells
// (x, y, 0..3) of the set's block q.
struct QuadLane {
  uint32_t ln, q, col;      // lane, block of the set, column 4 x + y
  bool x0, x3, y0, y3, odd; // odd: the column's red cells are z = 1 and 3
};
__host__ __device__ __forceinline__ QuadLane quad_lane(uint32_t ln) {
  const uint32_t col = ln & 15u, x = col >> 2, y = col & 3u;
  return {ln, ln >> 4, col, x == 0u, x == 3u, y == 0u, y == 3u, ((x + y) & 1u) != 0u};
}

// No block. (A macro elsewhere: the same value.)
constexpr uint32_t QUAD_NONE = 0xffffffffu;
// A lane's four halo links: across its x and y faces (lanes at 3 the neighbour below, at 0 the
// one above: the columns a rotation of the row by one brings to the lanes that need them), below
// and above. Each is one of the block's face neighbours, -x, +x, -y, +y, -z, +z: its place in this
// workgroup, or QUAD_FAR | a block of another workgroup, or QUAD_NONE.
constexpr uint32_t QUAD_FAR = 0x80000000u;
struct QuadLinks {
  uint32_t x, y, m, p;
};
__host__ __device__ __forceinline__ bool quad_far(uint32_t k) { return k != QUAD_NONE && (k & QUAD_FAR); }
// A set's face flags, per lane: bits 0..3 and 4..7 the water cells (z order) of the x and y halo
// columns, 8 and 9 the cells below and above; 10..13 whether x, y, below and above lie in another
// workgroup; 14..17 whether this lane's own faces (its x face, y face, bottom, top) do, and
// 18..21 whether they face a block at all. nbm: Dev::nbm; b0: the workgroup's first block.
__host__ __device__ __forceinline__ uint32_t quad_flags(const uint32_t* nbm, const uint32_t* nb, const QuadLinks& k,
                                                        const QuadLane& l, uint32_t b0) {
  uint32_t w = 0;
  auto cells = [](uint4 v) -> uint32_t { return (v.x >> 6 & 1u) | (v.y >> 5 & 2u) | (v.z >> 4 & 4u) | (v.w >> 3 & 8u); };
  auto id = [&](uint32_t link) -> uint32_t { return (link & QUAD_FAR) ? link & ~QUAD_FAR : b0 + link; };
  if (k.x != QUAD_NONE) w |= cells(*reinterpret_cast<const uint4*>(nbm + (size_t)id(k.x) * 64u + l.col * 4u));
  if (k.y != QUAD_NONE) w |= cells(*reinterpret_cast<const uint4*>(nbm + (size_t)id(k.y) * 64u + l.col * 4u)) << 4;
  if (k.m != QUAD_NONE) w |= (nbm[(size_t)id(k.m) * 64u + l.col * 4u + 3u] >> 6 & 1u) << 8;
  if (k.p != QUAD_NONE) w |= (nbm[(size_t)id(k.p) * 64u + l.col * 4u] >> 6 & 1u) << 9;
  w |= (quad_far(k.x) ? 1u << 10 : 0u) | (quad_far(k.y) ? 1u << 11 : 0u) | (quad_far(k.m) ? 1u << 12 : 0u) |
       (quad_far(k.p) ? 1u << 13 : 0u);
  const uint32_t own[4] = {l.x0 ? nb[0] : (l.x3 ? nb[1] : QUAD_NONE), l.y0 ? nb[2] : (l.y3 ? nb[3] : QUAD_NONE), nb[4], nb[5]};
#pragma unroll
  for (uint32_t f = 0; f < 4u; ++f) {
    if (own[f] != QUAD_NONE) w |= 1u << (18u + f);
    if (quad_far(own[f])) w |= 1u << (14u + f);
  }
  return w;
}
// The faces (x, y, bottom, top) a lane publishes: all that face a block, or (far) those that face
// another workgroup's.
__host__ __device__ __forceinline__ uint32_t quad_faces(uint32_t w, bool far) { return w >> (far ? 14 : 18) & 15u; }
// The halo words whose values a lane uses, the water cells': all, or (far) those of other
// workgroups. (Bits 0..3 and 4..7 the x and y halo columns, 8 and 9 the cells below and above.)
__host__ __device__ __forceinline__ uint32_t quad_want(uint32_t w, bool far) {
  if (!far) return w & 0x3ffu;
  return w & (((w >> 10 & 1u) ? 15u : 0u) | ((w >> 11 & 1u) ? 240u : 0u) | ((w >> 12 & 3u) << 8));
}
// The halo words to wait for in exchanges that follow each other in the same buffers with no
// reduction between: every word across a face, water or not. A wave may write the next words
// over a face's last ones only once the block across has read them, and it knows that from having
// that block's own words of the exchange after. So the waits have to be mutual. The water cells'
// words alone are not: a dry block beside a wet one waited for words the wet one, which wanted none
// of its, had already written over; the wait then never ended but by its limit.
__host__ __device__ __forceinline__ uint32_t quad_exchange(const QuadLinks& k) {
  return (k.x != QUAD_NONE ? 15u : 0u) | (k.y != QUAD_NONE ? 240u : 0u) | (k.m != QUAD_NONE ? 256u : 0u) |
         (k.p != QUAD_NONE ? 512u : 0u);
}

}  // namespace natray
