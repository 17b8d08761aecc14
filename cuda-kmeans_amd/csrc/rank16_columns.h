/*
 * Which points the wavefronts of rank16_impl.h read of SoA points, 64 of a column per request. Plain code without a HIP header: the tests
 * look at every read of a launch against the points there are.
 */
#ifndef KMX_RANK16_COLUMNS_H
#define KMX_RANK16_COLUMNS_H

#include <cstdint>

namespace kmx {

/* A wavefront's points begin at `first`, which in the last unit of a work-group may lie behind all n of them: a request then begins at the last point. */
constexpr uint32_t rank16_column_base(uint32_t first, uint32_t n) { return first < n ? first : n - 1; }
/* the point of a lane, counted from the base: lanes behind the last point have that one again */
constexpr uint32_t rank16_column_inside(uint32_t base, uint32_t lane, uint32_t n) { return lane < n - base ? lane : n - 1 - base; }

} // namespace kmx

#endif
