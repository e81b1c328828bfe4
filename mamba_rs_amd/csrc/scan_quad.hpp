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
    int first = 0;   // the first chunk whose outputs are wanted
    // with dt_w (then delta is not read, 16-bit storage, one chunk of at most kQuadDtLen steps): the kernel forms delta = softplus(dt_in row . dt_w
    // row of the channel + dt_b) itself, in f32.  dt_in: rows of dr elements bc_stride apart, dt_w [di][dr]; dr a multiple of 8, both 16-byte aligned.
    const void *dt_in = nullptr, *dt_w = nullptr;
    const float *dt_b = nullptr;
    int dr = 0;
};
constexpr int kQuadDtLen = 64;
bool scan_quad_dt_ok(int dtype, int T, int dr, int64_t bc_stride, const void *dt_in, const void *dt_w);
int launch_scan_quad(hipStream_t st, int dtype, int gate_mode, const ScanQuadArgs &a);

}  // namespace mrs
