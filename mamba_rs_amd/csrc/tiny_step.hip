// A whole Mamba-1 backbone step in one launch for small f32 models (d_inner <= 512: the reference's default
// configuration, d_model 128 x 3 layers, and the tiny CPU-runnable one).  The reference runs such a step as 4 GEMMs and
// 10 kernels per layer (GpuMambaBackbone::step, src/mamba_ssm/gpu/inference.rs:993-1252); at this size every one of them
// is a launch that moves a few kilobytes, so a step costs its launch count (3 layers: 21 launches, 50 us in a graph).
// The batch rows of a step never meet, and a row's activations (d_model + 2 d_inner + ... floats) fit in LDS many times
// over, so one workgroup walks one batch row through input projection, every layer and the final norm: products as
// matrix-vector sweeps over weights that sit in L2 (shared by all rows), the layer's conv window and SSM state read and
// written in place.  Arithmetic per element is that of the separate kernels (same softplus, SiLU, exp2 forms, f32
// accumulation); only the order of the dot-product sums differs, and it is fixed (same result on every run).
#include "tiny_rows.hpp"
#include "host_io.hpp"
#include "mfma_tiles.hpp"
#include <algorithm>
#include <type_traits>

namespace mrs {
namespace {

__global__ __launch_bounds__(kTinyThreads) void tiny_backbone_step_kernel(TinyStepArgs a) {
    extern __shared__ float lds[];
    const int dm = a.dm, di = a.di, ds = a.ds, dc = a.dc, dr = a.dr, xd = a.xd;
    const int xin_n = rup4(a.input_dim > dm ? a.input_dim : dm), di4 = rup4(di);
    float *res = lds;                   // [dm]      residual stream of this row
    float *xin = res + rup4(dm);        // [max(dm, input_dim)] operand of the product in flight (input row, normed row)
    float *proj = xin + xin_n;          // [2 di]    in_proj output: x half, gate half
    float *u = proj + rup4(2 * di);     // [di]      conv + SiLU output
    float *dl = u + di4;                // [di]      delta
    float *y = dl + di4;                // [di]      gated scan output
    float *xdbl = y + di4;              // [xd]      x_proj output: dt input, B, C
    float *part = xdbl + rup4(xd);      // [kTinyPart]
    float *red = part + kTinyPart;      // [waves]
    const int tid = threadIdx.x, b = blockIdx.x;
    const int lg = ds >> 2, rows_pp = kTinyThreads / lg;   // scan step: ds / 4 lanes per channel, one float4 of state each
    const int g = tid % lg, d0 = tid / lg;
    const bool now = a.host.out != nullptr;

    TinyStepLayer lnext = a.layers[0];
    // input row -> residual stream (identity or projection + bias)
    for (int i = tid; i < a.input_dim; i += kTinyThreads) {
        const float v = a.input[(int64_t)b * a.input_dim + i];
        xin[i] = v;
        if (a.input_copy) host_store(a.input_copy + (int64_t)b * a.input_dim + i, v);   // (the input came straight from host memory)
    }
    __syncthreads();
    if (a.in_w) {
        gemv_rows(a.in_w, a.input_dim, dm, xin, res, part, a.in_b);
    } else {
        for (int i = tid; i < dm; i += kTinyThreads) res[i] = xin[i];
        __syncthreads();
    }

    for (int l = 0; l < a.n_layers; l++) {
        // this layer's table entry was read a layer ago, the next one's is read now: the pointer fetch is off the critical path
        const TinyStepLayer lw = lnext;
        lnext = a.layers[min(l + 1, a.n_layers - 1)];
        // what the layer needs from memory whatever its input turns out to be is requested ahead of its use: the conv
        // window, taps and bias of channel tid and the norm weight now, the dt weights and the first two passes' float4s
        // of SSM state with their a_neg and D after in_proj
        float *cst = a.conv_state + ((int64_t)l * a.batch + b) * di * dc;
        float *hst = a.ssm_state + ((int64_t)l * a.batch + b) * di * ds;
        float cwin[8], ctap[8], cbias = 0.0f;
        const bool chan = tid < di;
        if (chan) {
            cbias = lw.conv_b[tid];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                cwin[k] = k < dc ? cst[(int64_t)tid * dc + k] : 0.0f;
                ctap[k] = k < dc ? lw.conv_w[(int64_t)tid * dc + k] : 0.0f;
            }
        }
        const float nw = tid < dm ? lw.norm_w[tid] : 0.0f;
        // RMSNorm of the residual stream
        float ss = 0.0f;
        for (int i = tid; i < dm; i += kTinyThreads) ss = fmaf(res[i], res[i], ss);
        const float inv = rms_inv(block_sum(ss, red), dm, a.eps);
        if (tid < dm) xin[tid] = res[tid] * inv * nw;
        for (int i = tid + kTinyThreads; i < dm; i += kTinyThreads) xin[i] = res[i] * inv * lw.norm_w[i];
        __syncthreads();
        gemv_rows(lw.in_proj, dm, 2 * di, xin, proj, part, nullptr);
        float dtb = 0.0f, dtw[8];
        if (chan) {
            dtb = lw.dt_b[tid];
#pragma unroll
            for (int k = 0; k < 8; k++) dtw[k] = lw.dt_w[(int64_t)min(k, dr - 1) * di + tid];
        }
        float4 hvp[kTinyPre], avp[kTinyPre];
        float Dp[kTinyPre];
#pragma unroll
        for (int p = 0; p < kTinyPre; p++) {
            const int d = d0 + p * rows_pp;
            hvp[p] = avp[p] = make_float4(0.f, 0.f, 0.f, 0.f);
            Dp[p] = 0.0f;
            if (d < di) {
                hvp[p] = *reinterpret_cast<const float4 *>(hst + (int64_t)d * ds + 4 * g);
                avp[p] = *reinterpret_cast<const float4 *>(lw.a_neg + (int64_t)d * ds + 4 * g);
                Dp[p] = lw.D[d];
            }
        }
        // conv1d step + SiLU on the x half (window slot k holds the input d_conv - k steps back; the new input goes last)
        if (chan) {
            float s = cbias;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (k < dc) {
                    const float v = k + 1 < dc ? cwin[k + 1 < 8 ? k + 1 : 7] : proj[tid];
                    s = fmaf(v, ctap[k], s);
                    leave(now, cst + (int64_t)tid * dc + k, v);
                }
            }
            u[tid] = silu(s);
        }
        __syncthreads();
        gemv_rows(lw.x_proj, di, xd, u, xdbl, part, nullptr);
        // dt_proj + bias + softplus
        if (chan) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) s = fmaf(j < dr ? xdbl[j] : 0.0f, dtw[j], s);
            for (int r0 = 8; r0 < dr; r0 += 8) {   // dt_rank beyond 8: eight weight loads in flight at a time
                float wv[8];
#pragma unroll
                for (int j = 0; j < 8; j++) wv[j] = lw.dt_w[(int64_t)min(r0 + j, dr - 1) * di + tid];
#pragma unroll
                for (int j = 0; j < 8; j++) s = fmaf(r0 + j < dr ? xdbl[r0 + j] : 0.0f, wv[j], s);
            }
            dl[tid] = softplus20(s + dtb);
        }
        __syncthreads();
        // scan step + D skip + SiLU gate (the arithmetic of ssm_step_kernel)
        for (int d = d0, pass = 0; d < di; d += rows_pp, pass++) {
            float4 hv, av;
            float Dd;
            if (pass == 0) { hv = hvp[0]; av = avp[0]; Dd = Dp[0]; }
            else if (pass == 1) { hv = hvp[kTinyPre - 1]; av = avp[kTinyPre - 1]; Dd = Dp[kTinyPre - 1]; }
            else {
                hv = *reinterpret_cast<const float4 *>(hst + (int64_t)d * ds + 4 * g);
                av = *reinterpret_cast<const float4 *>(lw.a_neg + (int64_t)d * ds + 4 * g);
                Dd = lw.D[d];
            }
            const float *Bv = xdbl + dr + 4 * g, *Cv = xdbl + dr + ds + 4 * g;
            const float du = dl[d] * u[d], x = dl[d] * kLog2e;
            hv.x = fmaf(fast_exp2(x * av.x), hv.x, du * Bv[0]);
            hv.y = fmaf(fast_exp2(x * av.y), hv.y, du * Bv[1]);
            hv.z = fmaf(fast_exp2(x * av.z), hv.z, du * Bv[2]);
            hv.w = fmaf(fast_exp2(x * av.w), hv.w, du * Bv[3]);
            leave4(now, hst, 4 * di * ds, 4u * (unsigned)(d * ds + 4 * g), hv);
            float acc = hv.x * Cv[0];
            acc = fmaf(hv.y, Cv[1], acc);
            acc = fmaf(hv.z, Cv[2], acc);
            acc = fmaf(hv.w, Cv[3], acc);
            for (int m = 1; m < lg; m <<= 1) acc += __shfl_xor(acc, m, kWave);
            if (g == 0) y[d] = fmaf(Dd, u[d], acc) * silu(proj[di + d]);
        }
        __syncthreads();
        gemv_rows(lw.out_proj, di, dm, y, xin, part, nullptr);
        for (int i = tid; i < dm; i += kTinyThreads) res[i] += xin[i];
        __syncthreads();
    }
    float ss = 0.0f;
    for (int i = tid; i < dm; i += kTinyThreads) ss = fmaf(res[i], res[i], ss);
    const float inv = rms_inv(block_sum(ss, red), dm, a.eps);
    for (int i = tid; i < dm; i += kTinyThreads) {
        const float v = res[i] * inv * a.norm_f[i];
        leave(now, a.temporal + (int64_t)b * dm + i, v);
        if (now) host_store(a.host.out + (int64_t)b * dm + i, v);
    }
    if (now) host_row_done(a.host, b);
}

// The same step with the weights streamed, for models of the default expand, d_state, d_conv and dt_rank; of those this route takes
// d_model 64 and 128 (x_proj's row is a multiple of four floats there), and each is an instance.  In the kernel above every product asks
// for its weights when its operand is ready: a layer of d_model 128 takes 10.4 us, while its 442 KB come in in 3.3 (one CU takes in at most
// 58 bytes a clock from L2, measured with 1 to 256 of them reading, however many loads are in flight).  Here the requests never stop:
// a thread holds its rows of the next layer's in_proj and x_proj in registers and those of out_proj in LDS, and each is asked for again
// behind its use, in portions that go out while the LDS reads of the chain are under way: all of them at once would hold the waves at
// their next instruction until the last is taken in (5.65 us against 5.3).  The chain is shorter as well: eight barriers a layer, the sum of squares
// taken by every wave for itself and applied behind in_proj, partial sums added by the thread that needs the column, the vectors brought
// by one request a wave.  A layer 5.3 us at d_model 128 and 2.25 at 64 (before: 10.4 and 8); the step of three layers, with the host's rows,
// 44.1 -> 28.4 us and 37.4 -> 20.5, 256 rows 82.7 -> 72.0, 1024 rows 321 -> 272.
// NOW: the host waits for flags (host_io.hpp), for which rows, windows and states are written all the way to memory; without them that costs a step 0.7 us and has the next one fetch its
// states from there (three layers of 128 queued one behind the other, every step written through / as here: 1 row 19.0 / 18.0 us, 128 rows 20.3 / 19.3; of 64 10.7 / 10.1, 11.2 / 10.9).
template <int DM, bool NOW> __global__ __launch_bounds__(kTinyThreads) void tiny_stream_step_kernel(TinyStepArgs a) {
    extern __shared__ float lds[];
    constexpr int di = 2 * DM, ds = 16, dr = DM / 16, xd = dr + 2 * ds;
    constexpr int lg = ds / 4, rows_pp = kTinyThreads / lg, passes = (di + rows_pp - 1) / rows_pp;   // scan step: a float4 of state per lane
    using In = Sweep<DM, 2 * di>;
    using Xp = Sweep<di, xd>;
    using Out = Sweep<di, DM>;
    static_assert(di % rows_pp == 0 && 4 * DM <= kTinyThreads && 8 * xd <= kTinyThreads && 2 * di <= kTinyThreads, "one thread each");
    float *part = lds;                  // [kTinyPart]
    float *res = part + kTinyPart;      // [DM]   residual stream of this row
    float *gate = res + DM;             // [di]   silu(gate half)
    float *u = gate + di;               // [di]   conv + SiLU output
    float *dl = u + di;                 // [di]   delta
    float *y = dl + di;                 // [di]   gated scan output
    float *xdbl = y + di;               // [xd]   x_proj output: dt input, B, C
    float *xin = xdbl + xd;             // [kStreamInput]  input row, then residual stream times norm weight
    float *vec = xin + kStreamInput;    // [8][256]   the layer's vectors: conv taps (four chunks of di floats), conv bias, dt bias, D, next norm weight
    float *dtl = vec + 2048;            // [dr][di]   dt_proj
    float *wo = dtl + (dr * di + 255) / 256 * 256;   // [Out::rows][threads] float4: out_proj's rows, each thread its own (last: the others are reached by constant offsets)
    const int tid = threadIdx.x, b = blockIdx.x;
    const Xp xp(tid);
    const bool now = NOW && a.host.out;   // (the stores as blocks of their own behind this branch: with the host 27.8 us, without it 28.2)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned wo_at = lds_address(wo) + 1024u * wave, vec_at = lds_address(vec) + 1024u * wave, dt_at = lds_address(dtl) + 1024u * wave;

    float4 wi[In::rows], wx[Xp::rows];
    auto ask_in = [&](const float *W, unsigned off, int j0, int n) {
#pragma unroll
        for (int j = j0; j < j0 + n; j++) wi[j] = ld4(global(W + j * 2 * di), off);
    };
    auto ask_x = [&](const float *W, unsigned off) {
#pragma unroll
        for (int j = 0; j < Xp::rows; j++) wx[j] = ld4(global(W + j * xd), off);
    };
    auto ask_out = [&](const float *W, unsigned off, int j0, int n) {
#pragma unroll
        for (int j = j0; j < j0 + n; j++) dma_kb(wo_at + (unsigned)j * (16u * kTinyThreads), W + j * DM, off);
    };

    TinyStepLayer lw = table_entry(a.layers), lnext = table_entry(a.layers + min(1, a.n_layers - 1));
    stream_input<DM>(a, lw.norm_w, xin, res, part, [&] {
        ask_in(lw.in_proj, In(tid).off, 0, In::rows);
        ask_x(lw.x_proj, own(xp.off));
    });

    auto layer = [&](auto last_layer, int l) {
        constexpr bool kLast = decltype(last_layer)::value;
        const int tid = (int)own(threadIdx.x), lane = tid & 63, cx = min(tid >> 3, xd - 1), co = min(tid >> 2, DM - 1);   // (not held over the layers)
        const In in(tid);
        const Out op(tid);
        // what the layer needs besides its products, and the norm weight of the next one
        float *cst = a.conv_state + ((int64_t)l * a.batch + b) * di * 4;
        float *hst = a.ssm_state + ((int64_t)l * a.batch + b) * di * ds;
        {   // One request a wave each, into LDS: a load of 4 bytes a lane takes as long as one of 16.
            const float *v = wave < 4 ? lw.conv_w + wave * di : wave == 4 ? lw.conv_b : wave == 5 ? lw.dt_b : wave == 6 ? lw.D : kLast ? a.norm_f : lnext.norm_w;
            dma_kb(vec_at, v, (16u * lane) & (wave == 7 ? 4u * DM - 1 : 4u * di - 1));   // (a shorter vector is read around)
            if (wave < dr * di / 256) dma_kb(dt_at, lw.dt_w + wave * 256, 16u * lane);
        }
        const unsigned ch16 = own(16u * min(tid, di - 1)), st4 = own(16u * tid);
        float4 win = make_float4(0.f, 0.f, 0.f, 0.f), hv[passes], av[passes];
        if (tid < di) win = ld4(global(cst), ch16);
#pragma unroll
        for (int p = 0; p < passes; p++) {
            hv[p] = ld4(global(hst + p * rows_pp * ds), st4);
            av[p] = ld4(global(lw.a_neg + p * rows_pp * ds), st4);
        }
        // the k-th eighth of the next layer's in_proj, asked for while the LDS reads before it are under way
        auto feed = [&](int k) {
            pin();
            if (!kLast) ask_in(lnext.in_proj, own(in.off), k * In::rows / 8, In::rows / 8);
            pin();
        };
        pin();
        // out_proj's rows: half of them during in_proj, a quarter each during the conv and x_proj
        constexpr int out_part = Out::rows * 2 / In::rows;
        auto feed_out = [&](int quarter) {
            pin();
            ask_out(lw.out_proj, op.off, quarter * Out::rows / 4, Out::rows / 4);
            pin();
        };
        // RMSNorm and in_proj: 1 / rms is a factor of every column
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        const float ss = lane_squares<DM>(res);
#pragma unroll
        for (int j = 0; j < In::rows; j += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(&xin[in.j * In::rows + j]);
            fma4(acc, x.x, wi[j]); fma4(acc, x.y, wi[j + 1]); fma4(acc, x.z, wi[j + 2]); fma4(acc, x.w, wi[j + 3]);
            pin(acc);
            ask_out(lw.out_proj, op.off, j / 4 * out_part, out_part);   // (the wave has read what these rows replace)
            pin();
        }
        const float inv = rms_inv(wave_sum(ss), DM, a.eps);
        if (in.on) *reinterpret_cast<float4 *>(&part[in.j * 2 * di + 4 * in.q]) = acc;
        // The vectors are in LDS: half of out_proj's requests are newer, and loads come back in order (stores that are still open only raise the count).  Of that half
        // a part is waited for as well: as fast as letting all of it be under way (the step of three layers, one row, 28.1 us both ways; five layers, 100 rows, 54.7 to 55.5).
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Out::rows / 4) : "memory");
        lds_barrier();
        // conv1d step + SiLU on the x half (window slot k holds the input d_conv - k steps back; the new input goes last), SiLU of the gate half
        const float4 tap = *reinterpret_cast<const float4 *>(&vec[min(tid, di - 1) / (di / 4) * 256 + min(tid, di - 1) % (di / 4) * 4]);
        const float cb = vec[4 * 256 + min(tid, di - 1)];
        const float p = inv * part_sum<2 * di, In::n, 1>(part, min(tid, 2 * di - 1), 0, [&] { feed_out(2); });
        if (tid < di) {
            float s = fmaf(win.y, tap.x, cb);
            s = fmaf(win.z, tap.y, s);
            s = fmaf(win.w, tap.z, s);
            s = fmaf(p, tap.w, s);
            win = make_float4(win.y, win.z, win.w, p);
            if (!kLast || !now) leave4(now, cst, 16 * di, ch16, win);
            u[tid] = silu(s);
        } else if (tid < 2 * di) {
            gate[tid - di] = silu(p);
        }
        lds_barrier();
        // x_proj
        acc = make_float4(0.f, 0.f, 0.f, 0.f);
        {
            float4 x[Xp::rows / 4];
#pragma unroll
            for (int j = 0; j < Xp::rows; j += 4) x[j / 4] = *reinterpret_cast<const float4 *>(&u[xp.j * Xp::rows + j]);
            feed_out(3);
#pragma unroll
            for (int j = 0; j < Xp::rows; j += 4) {
                fma4(acc, x[j / 4].x, wx[j]); fma4(acc, x[j / 4].y, wx[j + 1]); fma4(acc, x[j / 4].z, wx[j + 2]); fma4(acc, x[j / 4].w, wx[j + 3]);
            }
        }
        pin(acc);
        if (xp.on) *reinterpret_cast<float4 *>(&part[xp.j * xd + 4 * xp.q]) = acc;
        lds_barrier();
        const float xs = oct_sum(part_sum<xd, Xp::n, 8>(part, cx, tid & 7, [&] { feed(0); }));
        if ((tid & 7) == 0 && tid < 8 * xd) xdbl[cx] = xs;
        pin();
        if (!kLast) ask_x(lnext.x_proj, own(xp.off));
        pin();
        lds_barrier();
        // dt_proj + bias + softplus
        {
            float v[dr], w[dr], s = 0.0f;
            const int c = min(tid, di - 1);
#pragma unroll
            for (int j = 0; j < dr; j++) { v[j] = xdbl[j]; w[j] = dtl[j * di + c]; }
            const float dtb = vec[5 * 256 + c];
            feed(1);
            if (tid < di) {
#pragma unroll
                for (int j = 0; j < dr; j++) s = fmaf(v[j], w[j], s);
                dl[tid] = softplus20(s + dtb);
            }
        }
        lds_barrier();
        // scan step + D skip + gate (the arithmetic of ssm_step_kernel)
        if (kLast) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // out_proj's rows (ahead of the layer's stores)
        const int g = tid % lg;
        float Bv[4], Cv[4];
#pragma unroll
        for (int k = 0; k < 4; k++) { Bv[k] = xdbl[dr + 4 * g + k]; Cv[k] = xdbl[dr + ds + 4 * g + k]; }
#pragma unroll
        for (int p = 0; p < passes; p++) {
            const int d = tid / lg + p * rows_pp;
            const float dv = dl[d], uv = u[d], gv = gate[d], Dv = vec[6 * 256 + d];
            feed(2 + p);
            const float du = dv * uv, x = dv * kLog2e;
            float4 &h = hv[p];
            h.x = fmaf(fast_exp2(x * av[p].x), h.x, du * Bv[0]);
            h.y = fmaf(fast_exp2(x * av[p].y), h.y, du * Bv[1]);
            h.z = fmaf(fast_exp2(x * av[p].z), h.z, du * Bv[2]);
            h.w = fmaf(fast_exp2(x * av[p].w), h.w, du * Bv[3]);
            if (!now) leave4(false, hst + p * rows_pp * ds, 0, st4, h);
            float s = h.x * Cv[0];
            s = fmaf(h.y, Cv[1], s);
            s = fmaf(h.z, Cv[2], s);
            s = fmaf(h.w, Cv[3], s);
            s = quad_sum(s);
            if (g == 0) y[d] = fmaf(Dv, uv, s) * gv;
        }
        if (passes == 1) feed(3);
        // The wave's rows of out_proj are in LDS: half of in_proj's requests are newer (and, as above, a part of them is waited for).
        if (!kLast) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(In::rows / 4) : "memory");
        pin();
        // They take about a microsecond: behind the wait above, with out_proj in front of the next one, and in the last layer, whose wait is for everything, the window as well (three
        // layers of 128, one row, with the host: 27.8 us; the window where it is formed 28.2, the states in front of the wait and in halves 29.1).
        if (now) {
#pragma unroll
            for (int p = 0; p < passes; p++) host_store4(hst, 4 * di * ds, st4 + 4u * (unsigned)(p * rows_pp * ds), hv[p]);
            if (kLast && tid < di) host_store4(cst, 16 * di, ch16, win);
        }
        pin();
        lds_barrier();
        // out_proj and residual
        acc = stream_out_sweep(op, y, wo, [&](int turn) { feed(4 + turn); });
        pin(acc);
        if (op.on) *reinterpret_cast<float4 *>(&part[op.j * DM + 4 * op.q]) = acc;
        lds_barrier();
        const float os = quad_sum(part_sum<DM, Out::n, 4>(part, co, tid & 3, [&] { feed(7); }));
        if ((tid & 3) == 0 && tid < 4 * DM) {
            const float r = res[co] + os;
            res[co] = r;
            xin[co] = r * vec[7 * 256 + co];
        }
        lds_barrier();
    };
    for (int l = 0; l + 1 < a.n_layers; l++) {
        const TinyStepLayer after = table_entry(a.layers + min(l + 2, a.n_layers - 1));
        layer(std::false_type(), l);
        lw = lnext;
        lnext = after;
    }
    layer(std::true_type(), a.n_layers - 1);
    stream_output<DM>(a, now, xin, res);
}

template <int DM> bool tiny_stream_fits(const TinyStepArgs &a) {
    return a.dm == DM && a.di == 2 * DM && a.ds == 16 && a.dc == 4 && a.dr == DM / 16 && a.input_dim <= kStreamInput;
}
template <int DM, bool NOW> int launch_tiny_stream(hipStream_t st, const TinyStepArgs &a) {
    constexpr int dr = DM / 16, di = 2 * DM, xd = dr + 32;
    constexpr size_t lds = sizeof(float) * (kTinyPart + DM + 4 * di + xd + kStreamInput + 2048 + (dr * di + 255) / 256 * 256 + (size_t)Sweep<di, DM>::rows * 4 * kTinyThreads);
    static_assert(lds <= 160 * 1024, "LDS");
    static const hipError_t attr = hipFuncSetAttribute((const void *)tiny_stream_step_kernel<DM, NOW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "tiny backbone step: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((tiny_stream_step_kernel<DM, NOW>), dim3((unsigned)a.batch), dim3(kTinyThreads), lds, st, a);
    return check_launch("tiny_stream_step_kernel");
}

size_t tiny_lds_bytes(const TinyStepArgs &a) {
    const int xin_n = rup4(a.input_dim > a.dm ? a.input_dim : a.dm);
    return sizeof(float) * ((size_t)rup4(a.dm) + xin_n + rup4(2 * a.di) + 3 * (size_t)rup4(a.di) + rup4(a.xd) + kTinyPart + kTinyThreads / 64);
}

}  // namespace

bool tiny_step_ok(int dtype, int input_dim, int dm, int di, int ds, int dc, int dr, int xd) {
    if (input_dim < 1 || dm < 4 || di < 2 || xd < 4) return false;
    if (sweep_rounds(input_dim, dm) > kTinyMaxRounds || sweep_rounds(dm, 2 * di) > kTinyMaxRounds || sweep_rounds(di, xd) > kTinyMaxRounds ||
        sweep_rounds(di, dm) > kTinyMaxRounds)
        return false;
    return dtype == MRS_F32 && dm >= 4 && dm % 4 == 0 && dm <= 1024 && di % 4 == 0 && di >= 4 && di <= 512 && xd % 4 == 0 && xd >= 4 &&
           xd <= 1024 && (ds == 4 || ds == 8 || ds == 16 || ds == 32 || ds == 64) && dc >= 1 && dc <= 8 && dr >= 1 && input_dim >= 1 &&
           input_dim <= 4096 && xd == dr + 2 * ds;
}

int launch_tiny_step(hipStream_t st, const TinyStepArgs &a) {
    if (!tiny_step_ok(MRS_F32, a.input_dim, a.dm, a.di, a.ds, a.dc, a.dr, a.xd) || a.batch < 1 || a.n_layers < 1 || !a.layers || !a.input ||
        !a.conv_state || !a.ssm_state || !a.temporal || !a.norm_f)
        return fail(MRS_E_SHAPE, "tiny backbone step: shape outside the single-launch route (d_model=%d d_inner=%d d_state=%d xdbl=%d)", a.dm, a.di,
                    a.ds, a.xd);
    if (tiny_stream_fits<128>(a)) return a.host.out ? launch_tiny_stream<128, true>(st, a) : launch_tiny_stream<128, false>(st, a);
    if (tiny_stream_fits<64>(a)) return a.host.out ? launch_tiny_stream<64, true>(st, a) : launch_tiny_stream<64, false>(st, a);
    const size_t lds = tiny_lds_bytes(a);
    if (lds > 64 * 1024) return fail(MRS_E_SHAPE, "tiny backbone step: %zu bytes of LDS", lds);
    hipLaunchKernelGGL(tiny_backbone_step_kernel, dim3((unsigned)a.batch), dim3(kTinyThreads), lds, st, a);
    return check_launch("tiny_backbone_step_kernel");
}

}  // namespace mrs
