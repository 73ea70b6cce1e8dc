// Which sorted position a lane slot of a row reads.  In a header of its own so that the bounds are checked on the host.
#pragma once

namespace tgt {

// Position of edge `slot` of a row with n edges from position `start` on; a slot past the end repeats the row's last edge.  A row
// without edges reads position 0: its own start may be one past the last edge of the graph (isolated rows at the end), and its
// lanes load although nothing of theirs is used.  The graph has at least one edge.
__host__ __device__ __forceinline__ int edge_of_slot(const int start, const int n, const int slot) {
    return n > 0 ? start + (slot < n ? slot : n - 1) : 0;
}

}  // namespace tgt
