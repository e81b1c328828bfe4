// conv1d + SiLU and x_proj of a long prefill in one launch, 16-bit storage, d_conv 4.
//
// The reference runs the causal conv over the sequence and then a GEMM over its result (src/mamba_ssm/gpu/prefill.rs:777-845,
// kernels/conv1d.cu:209-315).  As two launches the conv moves x in and u out, and the GEMM, whose result is a few dozen columns, waits for u to
// come back.  Here a workgroup owns 32 or 64 steps of a sequence and all columns of the x_proj rows, and walks the channels 64 at a time.
//   * x (with the eight rows in front of the first step), x_proj's rows in matrix-operand order, taps, biases and the carried window go from memory straight to
//     LDS, three to five pieces of 64 channels ahead of their use.
//   * Sixteen waves: eight form u of a piece from x, two channels and a few steps a lane; four request the pieces to come and multiply the piece before by
//     x_proj's rows; four store it.  One barrier per piece: behind it u of the piece is there for the products and the stores, the next
//     piece's operands are in LDS, and the place of the piece before is free for a request.
//   * u lies in LDS as the matrix instructions take it, a row's 16-byte piece p at place p ^ (row / 2 % 8), so that neither their reads nor the
//     stores' meet on banks; its sums are the conv kernel's, term by term (and u its bits, but for one f16 value in 4000 that the compiler rounds by way of f32 here).
// Bound by the exponentials and divisions of SiLU (about 12 us of 16384 x 1536) and by x and u, 100 MB there (20 us at the rate of a copy).  16384 rows,
// two launches / this: d_inner 1536, 80 columns 23.0 + 23.2 / 28.3 us; 5120, 192 columns 72.7 + 69.8 / 114, where every unit takes in all of x_proj (2 MB).  As
// eight waves that all do everything, and so wait for their own LDS reads in front of each other's arithmetic: 39 at d_inner 1536.
#include "common.hpp"
#include "mfma_tiles.hpp"
#include "size_rules.hpp"

namespace mrs {
namespace {

constexpr int kConvWaves = 8, kMoveWaves = 4, kStoreWaves = 4, kConvThreads = 64 * (kConvWaves + kMoveWaves + kStoreWaves);
constexpr int kPiece = kConvPiece;   // channels of a piece

struct ConvXprojArgs {
    void *u, *xdbl;
    float *state;
    const void *x, *wp;
    const float *w, *bias;
    int64_t x_stride;
    int T, di, xd, tiles;   // tiles: of a sequence
    float *shares;          // with several slices of the channels: the products' shares, [slice][step][xd]
    int slices, pieces;     // pieces of a slice
    int64_t share_stride;
};

template <typename T> __device__ __forceinline__ void unpack2(unsigned v, float &a, float &b) {
    struct alignas(4) T2 { T v[2]; };
    const T2 t = __builtin_bit_cast(T2, v);
    a = Store<T>::ld(&t.v[0]); b = Store<T>::ld(&t.v[1]);
}

// ROWS: steps of a workgroup (32 or 64), NT: column tiles of x_proj, S: pieces in LDS
template <typename T, int ROWS, int NT, int S>
__global__ __launch_bounds__(kConvThreads) void conv_xproj_kernel(ConvXprojArgs g) {
    constexpr int kSteps = ROWS / 16;   // of a conv thread
    constexpr int kX = (ROWS + 8) * 128, kTaps = kX, kWin = kTaps + 1024, kBias = kWin + 1024, kW = kBias + 1024, kStage = kW + 2 * NT * 1024;
    constexpr int kReq = kStage / 1024, R = (kReq + kMoveWaves - 1) / kMoveWaves;   // requests of a piece, and of a wave
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int slice = blockIdx.x % g.slices, bt = blockIdx.x / g.slices, p0 = slice * g.pieces;
    const int b = bt / g.tiles, t0 = (bt - b * g.tiles) * ROWS, Tlen = g.T, di = g.di, np = min(g.pieces, di / kPiece - p0);
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    char *ut = smem + S * kStage;   // u of two pieces, 8 KB each
    const T *xs = (const T *)g.x + (int64_t)b * Tlen * g.x_stride + p0 * kPiece;   // (the slice's first channel)

    if (w < kConvWaves) {
        // ---- conv: channels 2 c and + 1, kSteps steps of the tile from kSteps r on
        const int c = tid & 31, r = tid >> 5;
        const bool front = t0 == 0 && kSteps * r < 3;
        const char *st = smem;
        char *out = ut;
        auto conv = [&]() {
            const float4 tap0 = *reinterpret_cast<const float4 *>(st + kTaps + 32 * c), tap1 = *reinterpret_cast<const float4 *>(st + kTaps + 32 * c + 16);
            const float2 bs = *reinterpret_cast<const float2 *>(st + kBias + 8 * c);
            float v0[kSteps + 3], v1[kSteps + 3];
#pragma unroll
            for (int k = 0; k < kSteps + 3; k++) unpack2<T>(*reinterpret_cast<const unsigned *>(st + (kSteps * r + 5 + k) * 128 + 4 * c), v0[k], v1[k]);
            if (front) {   // in front of the sequence: the carried window
                const float4 s0 = *reinterpret_cast<const float4 *>(st + kWin + 32 * c), s1 = *reinterpret_cast<const float4 *>(st + kWin + 32 * c + 16);
                if (r == 0) {
                    v0[0] = s0.y; v0[1] = s0.z; v0[2] = s0.w;
                    v1[0] = s1.y; v1[1] = s1.z; v1[2] = s1.w;
                } else {   // two steps a thread: the second's first is the step in front
                    v0[0] = s0.w; v1[0] = s1.w;
                }
            }
#pragma unroll
            for (int k = 0; k < kSteps; k++) {
                float o0 = fmaf(v0[k], tap0.x, bs.x), o1 = fmaf(v1[k], tap1.x, bs.y);
                o0 = fmaf(v0[k + 1], tap0.y, o0); o1 = fmaf(v1[k + 1], tap1.y, o1);
                o0 = fmaf(v0[k + 2], tap0.z, o0); o1 = fmaf(v1[k + 2], tap1.z, o1);
                o0 = fmaf(v0[k + 3], tap0.w, o0); o1 = fmaf(v1[k + 3], tap1.w, o1);
                struct alignas(4) T2 { T v[2]; } o;
                Store<T>::st(&o.v[0], silu(o0)); Store<T>::st(&o.v[1], silu(o1));
                const int row = kSteps * r + k;
                *reinterpret_cast<T2 *>(out + row * 128 + 16 * ((c >> 2) ^ ((row >> 1) & 7)) + 4 * (c & 3)) = o;
            }
            st = st == smem + (S - 1) * kStage ? smem : st + kStage;
            out = out == ut ? ut + ROWS * 128 : ut;
        };
        lds_barrier();
        conv();
        for (int p = 0; p < np; p++) {
            lds_barrier();   // u of piece p and the operands of p + 1 are there; everybody is done with piece p - 1
            if (p + 1 < np) conv();
        }
    } else if (w >= kConvWaves + kMoveWaves) {
        // ---- stores: u through a buffer resource that ends with the sequence.  By waves that wait for no loads: the counter of what is under way goes down in
        // the loads' order among themselves and the stores' among themselves only.
        const int mt = tid - 64 * (kConvWaves + kMoveWaves), srow = mt >> 3, sp = mt & 7, spl = 16 * (sp ^ ((srow >> 1) & 7));   // rows srow, srow + 32
        const __amdgpu_buffer_rsrc_t ures = __builtin_amdgcn_make_buffer_rsrc((T *)g.u + (int64_t)b * Tlen * di, 0, Tlen * di * 2, 0x00020000);
        const unsigned uoff = (unsigned)(t0 + srow) * (unsigned)di * 2u + 16u * (unsigned)sp;
        const char *uin = ut;
        lds_barrier();
        for (int p = 0; p < np; p++) {
            lds_barrier();   // (as above)
            typedef unsigned v4u __attribute__((ext_vector_type(4)));
            v4u o[ROWS / 32];
#pragma unroll
            for (int i = 0; i < ROWS / 32; i++) o[i] = *reinterpret_cast<const v4u *>(uin + (srow + 32 * i) * 128 + spl);
#pragma unroll
            for (int i = 0; i < ROWS / 32; i++) __builtin_amdgcn_raw_buffer_store_b128(o[i], ures, uoff + 64u * (unsigned)(i * di), (p0 + p) * (kPiece * 2), 0);
            uin = uin == ut ? ut + ROWS * 128 : ut;
        }
    } else {
        // ---- the waves that move: requests and products
        // Requests of a piece: 9 of eight rows of x, taps, window, biases, 2 NT of x_proj; a wave takes every fourth (past the end the last one again)
        const int mw = w - kConvWaves;
        const char *from[R];
        int step[R];
        unsigned voff[R], to[R];
#pragma unroll
        for (int i = 0; i < R; i++) {
            const int q = min(mw + kMoveWaves * i, kReq - 1);   // (the same for the wave)
            voff[i] = 16u * (unsigned)l;
            to[i] = lds0 + (unsigned)q * 1024u;
            if (q < kX / 1024) {
                const int t = min(max(t0 - 8 + 8 * q + (l >> 3), 0), Tlen - 1);
                from[i] = (const char *)xs; step[i] = kPiece * 2; voff[i] = (unsigned)t * (unsigned)g.x_stride * 2u + 16u * (unsigned)(l & 7);
            } else if (q == kTaps / 1024) {
                from[i] = (const char *)(g.w + p0 * kPiece * 4); step[i] = kPiece * 16;
            } else if (q == kWin / 1024) {   // (read by the first workgroup of a sequence alone)
                from[i] = (const char *)((t0 == 0 ? g.state + (int64_t)b * di * 4 : g.w) + p0 * kPiece * 4); step[i] = kPiece * 16;
            } else if (q == kBias / 1024) {
                from[i] = (const char *)(g.bias + p0 * kPiece); step[i] = kPiece * 4; voff[i] = 16u * (unsigned)min(l, 15);
            } else {
                const int j = q - kW / 1024;   // column tile j / 2, half j % 2 of the piece
                from[i] = (const char *)g.wp + ((int64_t)(j >> 1) * (di >> 5) + (j & 1) + 2 * p0) * 1024; step[i] = 2048;
            }
        }
        unsigned ring = 0;
        auto request = [&]() {
#pragma unroll
            for (int i = 0; i < R; i++) {
                dma_kb(__builtin_amdgcn_readfirstlane(to[i] + ring), from[i], voff[i]);
                from[i] += step[i];
            }
            ring = ring == (S - 1) * kStage ? 0 : ring + kStage;
        };
#pragma unroll
        for (int p = 0; p < S - 1; p++)
            if (p < np) request();

        // a wave has half of the row tiles and half of the column tiles (an odd last one is the first half's)
        constexpr int kM = ROWS / 32, kN = (NT + 1) / 2;
        const int lr = l & 15, lg = l >> 4, row0 = 16 * kM * (mw & 1) + lr, n0 = kN * (mw >> 1);
        v4f acc[kM][kN];
#pragma unroll
        for (int i = 0; i < kM; i++)
#pragma unroll
            for (int j = 0; j < kN; j++) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
        // until at most `newer` pieces' requests are under way (loads come back in order)
        auto wait_newer = [&](int newer) {
            if (newer >= S - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * R) : "memory");
            else if (newer == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * R) : "memory");
            else if (newer == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * R) : "memory");
            else if (newer == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        };
        static_assert(S >= 4 && S <= 6 && (S - 2) * R < 64, "the counts above");
        wait_newer(min(np, S - 1) - 1);
        lds_barrier();   // piece 0
        wait_newer(min(np, S - 1) - 2);
        const char *ws = smem, *uin = ut;
        for (int p = 0; p < np; p++) {
            lds_barrier();   // (as above)
            if (p + S - 1 < np) request();
            uint4 ua[kM][2];
#pragma unroll
            for (int i = 0; i < kM; i++)
#pragma unroll
                for (int kk = 0; kk < 2; kk++) ua[i][kk] = *reinterpret_cast<const uint4 *>(uin + (row0 + 16 * i) * 128 + 16 * ((4 * kk + lg) ^ ((lr >> 1) & 7)));
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int j = 0; j < kN; j++) {
                    const uint4 wf = *reinterpret_cast<const uint4 *>(ws + kW + (2 * min(n0 + j, NT - 1) + kk) * 1024 + 16 * l);
#pragma unroll
                    for (int i = 0; i < kM; i++) acc[i][j] = Mma32<T>::mma(wf, ua[i][kk], acc[i][j]);   // (transposed: a lane holds four columns of a row)
                }
            ws = ws == smem + (S - 1) * kStage ? smem : ws + kStage;
            uin = uin == ut ? ut + ROWS * 128 : ut;
            if (p + 2 < np) wait_newer(min(np, p + S) - (p + 3));   // the operands of piece p + 2
        }
#pragma unroll
        for (int i = 0; i < kM; i++) {
            const int t = t0 + row0 + 16 * i;
            T *out = (T *)g.xdbl + ((int64_t)b * Tlen + min(t, Tlen - 1)) * g.xd;
#pragma unroll
            for (int j = 0; j < kN; j++) {
                const int col = 16 * (n0 + j) + 4 * lg;
                if (t < Tlen && n0 + j < NT && col < g.xd) {
                    if (g.slices > 1) {
                        *reinterpret_cast<v4f *>(g.shares + slice * g.share_stride + ((int64_t)b * Tlen + t) * g.xd + col) = acc[i][j];
                        continue;
                    }
                    struct alignas(8) T4 { T v[4]; } o;
#pragma unroll
                    for (int e = 0; e < 4; e++) Store<T>::st(&o.v[e], acc[i][j][e]);
                    *reinterpret_cast<T4 *>(out + col) = o;
                }
            }
        }
    }
    // The sequence's last four inputs are the window from now on; the workgroup that read the old one writes it.
    if (t0 == 0) {
        float *sout = g.state + ((int64_t)b * di + p0 * kPiece) * 4;
        for (int ch = tid; ch < np * kPiece; ch += kConvThreads) {
            const T *px = xs + (int64_t)(Tlen - 4) * g.x_stride + ch;
            *reinterpret_cast<float4 *>(sout + 4 * ch) = make_float4(Store<T>::ld(px), Store<T>::ld(px + g.x_stride), Store<T>::ld(px + 2 * g.x_stride), Store<T>::ld(px + 3 * g.x_stride));
        }
    }
}

template <typename T, int ROWS, int NT>
int launch_conv_xproj_t(hipStream_t st, const ConvXprojArgs &g, int batch) {
    constexpr size_t stage = (ROWS + 8) * 128 + 3 * 1024 + 2 * NT * 1024, ut = 2 * ROWS * 128;
    constexpr int S = std::min<int>((160 * 1024 - ut) / stage, 6);
    constexpr size_t lds = S * stage + ut;
    static const hipError_t attr = hipFuncSetAttribute((const void *)conv_xproj_kernel<T, ROWS, NT, S>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "conv + x_proj: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((conv_xproj_kernel<T, ROWS, NT, S>), dim3((unsigned)(batch * g.tiles * g.slices)), dim3(kConvThreads), lds, st, g);
    return check_launch("conv_xproj_kernel");
}
template <typename T, int NT = kConvMinTiles>
int launch_conv_xproj_n(hipStream_t st, const ConvXprojArgs &g, int batch, int rows) {
    if constexpr (NT < kConvMaxTiles)
        if (conv_xproj_col_tiles(g.xd) > NT) return launch_conv_xproj_n<T, NT + 1>(st, g, batch, rows);
    return rows == 64 ? launch_conv_xproj_t<T, 64, NT>(st, g, batch) : launch_conv_xproj_t<T, 32, NT>(st, g, batch);
}

}  // namespace

bool conv_xproj_ok(int dtype, const void *u, const void *xdbl, const float *state, const void *x, int64_t x_stride, const void *wp, const float *w, const float *bias, int batch, int T,
                   int di, int dc, int xd) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && dc == 4 && di % kPiece == 0 && di >= 2 * kPiece && T >= 4 && conv_xproj_columns_ok(xd) && x_stride % 8 == 0 && wp &&
           x_stride >= di && (int64_t)T * x_stride < (int64_t)1 << 30 && (int64_t)batch * ((T + 31) / 32) < (int64_t)1 << 30 && aligned(u, 16) && aligned(xdbl, 8) && aligned(state, 16) &&
           aligned(x, 16) && aligned(wp, 16) && aligned(w, 16) && aligned(bias, 4);
}

int launch_conv_xproj(hipStream_t st, int dtype, void *u, void *xdbl, float *state, const void *x, int64_t x_stride, const void *wp, const float *w, const float *bias, int batch, int T,
                      int di, int xd) {
    if (!conv_xproj_ok(dtype, u, xdbl, state, x, x_stride, wp, w, bias, batch, T, di, 4, xd)) return fail(MRS_E_SHAPE, "conv + x_proj: shape outside the route (T=%d d_inner=%d columns=%d)", T, di, xd);
    const int rows = conv_xproj_rows(batch, T);
    const ConvXprojArgs g = {u, xdbl, state, x, wp, w, bias, x_stride, T, di, xd, (T + rows - 1) / rows, nullptr, 1, di / kPiece, 0};
    return dtype == MRS_BF16 ? launch_conv_xproj_n<bf16_t>(st, g, batch, rows) : launch_conv_xproj_n<f16_t>(st, g, batch, rows);
}

// Fewer rows: the channels in slices as well, whose products are summed in f32, in the order of the slices, by a second launch.  At 777 x 2048, 96 columns: conv 5.4, x_proj 8.0 us
// as two launches, here 6.2 + 3.3.
template <typename T> static __global__ __launch_bounds__(256) void conv_xproj_sum_kernel(T *__restrict__ out, const float *__restrict__ shares, int slices, int64_t n4) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const v4f *p = reinterpret_cast<const v4f *>(shares) + i;
    v4f v[kConvMaxSlices], s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kConvMaxSlices; k++) v[k] = p[min(k, slices - 1) * n4];   // all asked for at once
#pragma unroll
    for (int k = 0; k < kConvMaxSlices; k++)
        if (k < slices) s += v[k];
    struct alignas(4 * sizeof(T)) T4 { T v[4]; } o;
#pragma unroll
    for (int e = 0; e < 4; e++) Store<T>::st(&o.v[e], s[e]);
    reinterpret_cast<T4 *>(out)[i] = o;
}

int launch_conv_xproj_sliced(hipStream_t st, int dtype, void *u, void *xdbl, float *shares, float *state, const void *x, int64_t x_stride, const void *wp, const float *w, const float *bias,
                             int batch, int T, int di, int xd) {
    const int slices = conv_xproj_form(batch, T, di, xd);
    if (!conv_xproj_ok(dtype, u, xdbl, state, x, x_stride, wp, w, bias, batch, T, di, 4, xd) || slices < 2 || !aligned(shares, 16))
        return fail(MRS_E_SHAPE, "conv + x_proj in slices: shape outside the route (T=%d d_inner=%d columns=%d)", T, di, xd);
    const int pieces = (di / kPiece + slices - 1) / slices;
    const int64_t n = (int64_t)batch * T * xd;
    const ConvXprojArgs g = {u, xdbl, state, x, wp, w, bias, x_stride, T, di, xd, (T + 31) / 32, shares, (di / kPiece + pieces - 1) / pieces, pieces, n};
    const int rc = dtype == MRS_BF16 ? launch_conv_xproj_n<bf16_t>(st, g, batch, 32) : launch_conv_xproj_n<f16_t>(st, g, batch, 32);
    if (rc) return rc;
    const dim3 grid((unsigned)((n / 4 + 255) / 256));
    if (dtype == MRS_BF16) hipLaunchKernelGGL(conv_xproj_sum_kernel<bf16_t>, grid, dim3(256), 0, st, (bf16_t *)xdbl, shares, g.slices, n / 4);
    else hipLaunchKernelGGL(conv_xproj_sum_kernel<f16_t>, grid, dim3(256), 0, st, (f16_t *)xdbl, shares, g.slices, n / 4);
    return check_launch("conv_xproj_sum_kernel");
}

}  // namespace mrs
