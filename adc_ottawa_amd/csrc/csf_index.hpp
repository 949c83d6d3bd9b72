// Index rules of the CSF kernels that a host program can check too.
#pragma once

namespace adc2g {

// The up kernel takes x1 in tiles of CSF_UP_ROWS rows c, lane group g (0..3) the
// rows tile + g and tile + 4 + g, and masks those past the last virtual.  From
// five virtuals on a tile's end is within 2 v rows, that is within the t1
// entries behind x1; with fewer (one tile) the group keeps to rows that exist:
// eight rows of o = v = 2 are 16 entries, the whole vector has 14.
constexpr int CSF_UP_ROWS = 8;
constexpr int csf_up_first(int g, int v) { return g < v ? g : v - 1; }  // row of group g in the first tile
constexpr int csf_up_half(int v) { return v > 4 ? 4 : 0; }              // from it to the group's second row

}  // namespace adc2g
