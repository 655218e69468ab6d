// Products of several tokens (split_product.hip) on the bf16 matrix cores with
// fp32 accuracy, and the row kernels that prepare their input.
#ifndef TLA_BATCH_H
#define TLA_BATCH_H

#include "tla_internal.h"

namespace tla {

enum ProductKind { kProductDirect, kProductResident, kProductTiled };

constexpr int kProductMaxNorm = 4096;  // columns of an rmsnorm inside the product, at most

// out[t][row] (+)= W[row] . x[t] for t < n and every format of the reference
// (F32 / F16 16-byte aligned, Q8_0 / Q4_0 4-byte, Q6_K 2-byte).  x is fp32
// rows or the bf16 planes that launch_split_rows / launch_norm_split_rows or
// a paired product wrote.
struct ProductParams {
    GemvSegment seg[kGemvMaxSeg];
    int n_seg;
    int total_rows;            // sum of seg[].rows
    int cols;                  // multiple of 64 (of 256 for Q6_K)
    long long row_bytes;
    int n;                     // tokens
    int add;                   // 1: out += W.x, 0: out = W.x
    const float* x;            // x[t * x_stride + col], 16-byte aligned rows (direct, planes = 0)
    long long x_stride;
    const float* norm_w;       // non-null (direct, planes = 0): x is replaced by rmsnorm(x, norm_w, eps)
    float eps;
    int planes;                // 1: x comes as planes (always for resident and tiled)
    const unsigned char* xs;   // the planes
    int pair;                  // 1: segments 0 and 1 are the gate and up matrices (equal rows, a
                               // multiple of 32): hs receives the planes of silu(gate) * up; a
                               // segment's out may be NULL (direct and resident)
    unsigned char* hs;
    // the plan (plan_product)
    int kind;
    int n_tiles;               // token tiles of 16 (tiled: a multiple of 4)
    int rows_per_group;        // 16-row subtiles per workgroup (tiled: per wave)
    int row_groups;
    int x_share;               // direct: consecutive blocks that share an x operand, 1, 2 or 4
    int shares;                // resident: workgroups per row group and K range, each a share of the tiles
    int k_splits;              // K cut into this many ranges of blk_per_split 32-column
    int blk_per_split;         // blocks (even); each range's sums go to part, and a
    float* part;               // second launch adds them in range order: [k_splits][n][total_rows]
    int defer_reduce;          // 1: that launch is left to the caller (launch_norm_split_rows,
                               // launch_reduce_rmsnorm_rows)
};
// Fills the plan from the shape (n, total_rows, cols, pair) for n_cu compute
// units; the options (0: per shape) are the row subtiles per workgroup, the
// token tiles per resident workgroup (at most) and the K ranges (at least).
// The first two leave every sum's order as it is.
void plan_product(int type, int n_cu, int opt_rows, int opt_tiles, int opt_k, ProductParams* p);
// Estimated microseconds of a resident or tiled plan, without the planes' launch.
double product_us(int type, int n_cu, const ProductParams& p);
hipError_t launch_product(int type, const ProductParams& p, hipStream_t s);

hipError_t load_product_code();  // as tla_internal.h's
size_t product_planes_bytes(int n, int cols);
size_t product_part_bytes(int n, int total_rows, int k_splits);
// The planes of n rows of x (gated: of silu(x[t][c]) * x[t][cols + c]).
hipError_t launch_split_rows(const float* x, long long x_stride, int n, int cols, bool gated, unsigned char* xs,
                             hipStream_t s);
// The planes of rmsnorm(x[t], w, eps) for n dense rows; with k_splits > 0, x[t]
// first takes a deferred product's range sums (and is written back).
hipError_t launch_norm_split_rows(float* x, const float* part, int k_splits, int n, int cols, const float* w, float eps,
                                  unsigned char* xs, hipStream_t s);

// x[t][c] += the K ranges' sums part[z][t][c] (z in order), then out[t] =
// rmsnorm(x[t]) * w (the rmsnorm rows' arithmetic): n_tok rows of size
// floats, one workgroup per row.  x, part, out 16-byte aligned, size a
// multiple of 4.
hipError_t launch_reduce_rmsnorm_rows(float* x, const float* part, int k_splits, float* out, const float* w,
                                      int n_tok, int size, float eps, hipStream_t s);

}  // namespace tla

#endif  // TLA_BATCH_H
