// How attention tiles are dealt to several work-groups: what host and kernels agree on.  Plain C++ (constexpr functions run on
// either side), so that a test can compile it by itself.
#pragma once

namespace fgrpo {

constexpr int kAttnMaxParts = 8;      // parts of a tile at most

// The merge launches read from a table how many parts a tile has and which work-group took the first; the others' lie `stride`
// behind one another, and what is read starts `skip` behind (the heads of a query tile that further work-groups take).  An entry
// is written by the work-group of the tile's first part: of a tile that an order list of the caller's leaves out it is whatever
// the workspace held.  Only an entry whose work-groups all are in the launch is followed; the sums of any other would be read
// from outside the workspace.
constexpr bool attn_parts_inside(int np, int first, int skip, int stride, int grid) {
  return np > 1 && np <= kAttnMaxParts && first >= 0 && first <= grid - 1 - skip - (np - 1) * stride;
}

}  // namespace fgrpo
