// What the two resident Mamba-3 steps (resident_m3_step.hip, resident_m3_row.hip) have in common.
#pragma once
#include "resident.hpp"
#include "m3_math.hpp"

namespace mrs {

constexpr int kMaxNc = 16, kMaxOc = 16, kMaxEx = 16, kMaxDs = 64;   // bounds of the fixed LDS areas and of a thread's work

// What a workgroup needs of a layer besides the two big weights (byte offsets): B and C norm weights, its head's B and C biases [ds]
// each, the next layer's norm weight for its columns [oc], D and dt bias of its head.
struct SmallBlock { int bnw, cnw, bb, cb, nw, D, dtb, bytes; };
__host__ __device__ inline SmallBlock small_block(int ds, int oc) {
    SmallBlock o;
    o.bnw = 0;
    o.cnw = ds * 4;
    o.bb = 2 * ds * 4;
    o.cb = 3 * ds * 4;
    o.nw = 4 * ds * 4;
    o.D = o.nw + oc * 4;
    o.dtb = o.D + 4;
    o.bytes = up1k(o.dtb + 4);
    return o;
}
// A workgroup's part of a layer in memory: in_proj columns x: nc | z: nc | shared: ex, out_proj columns, the small block, each padded to
// whole kilobytes.  The columns lie as the step reads them: [K / 8][columns][8], or with row_order [columns][K].
struct LayerBlock { int out, small, bytes; };
__host__ __device__ inline LayerBlock layer_block(int dm, int di, int cols, int oc, int ds) {
    LayerBlock o;
    o.out = up1k(cols * dm * 2);
    o.small = o.out + up1k(oc * di * 2);
    o.bytes = o.small + small_block(ds, oc).bytes;
    return o;
}

// The row-order step (resident_m3_row.hip): the kernel chain's sums, term by term, for one row.  d_model = 256 KI.
bool resident_m3_row_ok(const ResidentM3Args &a, int dtype);
size_t resident_m3_row_lds(const ResidentM3Args &a);
int launch_resident_m3_row(hipStream_t st, int dtype, const ResidentM3Args &a, const ResidentM3Args *dev, const TokenRows &rows);

}  // namespace mrs
