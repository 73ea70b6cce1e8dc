// Linears of any width (linear_tiles.hip) for linear.hip.
#pragma once
#include "common.h"

namespace tgt {

struct LinArgs {
    const void* A[3];      // forward: A[0] = x [N, K]; input gradient: A[j] = dy_j [N, M]
    const void* W[3];      // [M, K] row-major (nn.Linear.weight)
    const void* bias[3];   // forward only; entries may be null
    void* out[3];          // forward: y_j [N, M]; input gradient: out[0] = dx [N, K]
    int nw;
    int64_t N;
    int K, M;
};

// y_j = x W_j^T + b_j, or (dx) dx = sum_j dy_j W_j
int linear_tiles(const LinArgs& a, bool dx, int dtype, hipStream_t st);
// Whether one launch takes a forward with one output and the packing beside it (an error for a bad packing), and that launch
int packs_beside(const LinArgs& a, const tgt_node_pack_args* pack, int dtype, bool& fits);
int linear_tiles_and_pack(const LinArgs& a, const tgt_node_pack_args& pack, int dtype, hipStream_t st);

struct GradWArgs {
    const void* x;         // [N, K]
    const void* dy[3];     // [N, M]
    float* partial;        // [workers][nw][M*K + M]
    int nw;
    int64_t N;
    int K, M;
};

// Every worker's dW_j = dy_j^T x and db_j = column sums of dy_j over its share of the rows
int gradw_tiles(const GradWArgs& a, int workers, int dtype, hipStream_t st);

}  // namespace tgt
