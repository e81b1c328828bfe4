// What the two resident Mamba-1 steps share: resident_step.hip (a group of workgroups per row) and resident_rows.hip (up to
// sixteen rows per group) take their weights in the same order.
#pragma once
#include "resident.hpp"

namespace mrs {

constexpr int kDs = 16, kDc = 4;           // states and conv taps of a channel
constexpr int kMaxNc = 24, kMaxOc = 16, kMaxXd = 96, kMaxDr = 64;   // bounds of the fixed LDS areas
// What a workgroup needs of a layer besides the two big weights, as one block (byte offsets): x_proj rows [nc / 8][xd][8], dt weights
// [nc][dr], A [nc][16], conv taps [nc][4], conv bias, D, dt bias [nc], the next layer's norm weight for its columns [oc].
struct SmallBlock { int xw, dtw, aneg, cw, cb, D, dtb, nw, bytes; };
__host__ __device__ constexpr SmallBlock small_block(int nc, int oc, int xd, int dr) {
    SmallBlock o{};
    o.xw = 0;
    o.dtw = o.xw + nc * xd * 2;
    o.aneg = o.dtw + nc * dr * 2;
    o.cw = o.aneg + nc * kDs * 4;
    o.cb = o.cw + nc * kDc * 4;
    o.D = o.cb + nc * 4;
    o.dtb = o.D + nc * 4;
    o.nw = o.dtb + nc * 4;
    o.bytes = up1k(o.nw + oc * 4);
    return o;
}
// A workgroup's part of a layer in memory: in_proj columns [dm / 8][2 nc][8], out_proj columns [di / 8][oc][8], the small block, each
// padded to whole kilobytes.
struct LayerBlock { int out, small, bytes; };
__host__ __device__ constexpr LayerBlock layer_block(int dm, int di, int nc, int oc, int xd, int dr) {
    LayerBlock o{};
    o.out = up1k(2 * nc * dm * 2);
    o.small = o.out + up1k(oc * di * 2);
    o.bytes = o.small + small_block(nc, oc, xd, dr).bytes;
    return o;
}

}  // namespace mrs
