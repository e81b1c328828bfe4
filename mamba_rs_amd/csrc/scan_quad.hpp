// The scan route with four lanes per channel (m1_scan_quad.hip), as m1_scan.hip dispatches to it.
#pragma once
#include "common.hpp"
#include <type_traits>

namespace mrs {

constexpr int kQuadLen = 128;   // longest chunk: its B and C rows lie in LDS as a whole (16 KB)
struct ScanQuadArgs {
    float *h;
    void *y;
    const void *delta, *u, *B, *C, *gate;
    int64_t bc_stride, gate_stride;
    const float *a_neg, *D;
    float *h0copy, *S, *sumd;   // [batch][16][di], [batch][nchunk - 1][16][di], [batch][nchunk - 1][di]; unused with one chunk
    int batch, Tlen, di, tiles, nchunk, len;
};
int launch_scan_quad(hipStream_t st, int dtype, int gate_mode, const ScanQuadArgs &a);

}  // namespace mrs
