// A whole Mamba-3 SISO backbone step in one launch for small f32 models (the reference's default configuration:
// d_model 128, 4 layers, headdim 16, d_state 16).  GpuMamba3Backbone::step runs such a step as fourteen launches per
// layer (src/mamba3_siso/gpu/inference.rs:506-1000), the engine here as three; at this size each of them moves a few
// kilobytes and costs its launch.  One workgroup walks one batch row through input projection, every layer and the final
// norm: in_proj and out_proj as matrix-vector sweeps over weights that sit in L2, the layer step between them with the
// formulas of m3_layer_step_kernel (B/C RMSNorm + bias, angle accumulation in f64 and rotation, alpha / beta / gamma,
// the trapezoidal state update, D skip, SiLU gate or RMSNormGated), states updated in place.  Only the order of the
// dot-product sums differs from the kernel chain, and it is fixed.
#include "tiny_rows.hpp"
#include "host_io.hpp"
#include "m3_math.hpp"
#include "mfma_tiles.hpp"
#include <type_traits>

namespace mrs {
namespace {

__global__ __launch_bounds__(kTinyThreads) void tiny_m3_backbone_step_kernel(TinyM3StepArgs a) {
    extern __shared__ float lds[];
    const int dm = a.dm, di = a.di, nh = a.nh, hd = a.hd, ds = a.ds, ng = a.ng, nr = a.nr, ip = a.ip;
    const int xin_n = rup4(a.input_dim > dm ? a.input_dim : dm), di4 = rup4(di);
    float *res = lds;                   // [dm]       residual stream of this row
    float *xin = res + rup4(dm);        // [max(dm, input_dim)] operand of the product in flight
    float *proj = xin + xin_n;          // [ip]       in_proj output: z | x | B | C | dd_dt | dd_A | trap | angles
    float *kl = proj + rup4(ip);        // [nh ds]    K of every head (normalised, biased, rotated B)
    float *ql = kl + rup4(nh * ds);     // [nh ds]    Q of every head
    float *yr = ql + rup4(nh * ds);     // [di]       y before the gate
    float *yg = yr + di4;               // [di]       gated y: out_proj's operand
    float *ginv = yg + di4;             // [2 ng]     1 / rms of the raw B and C rows per group
    float *part = ginv + rup4(2 * ng);  // [kTinyPart]
    float *red = part + kTinyPart;      // [waves]
    const int tid = threadIdx.x, b = blockIdx.x;
    const int lg = ds >> 2, per_head = hd * lg, tasks = nh * per_head;   // one lane-task per float4 of SSM state
    const int na = nr > 0 ? nr : 1;

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

    TinyM3StepLayer lnext = a.layers[0];
    for (int l = 0; l < a.n_layers; l++) {
        const TinyM3StepLayer lw = lnext;
        lnext = a.layers[min(l + 1, a.n_layers - 1)];
        float *ssm = a.ssm + ((int64_t)l * a.batch + b) * nh * hd * ds;
        float *kst = a.kst + ((int64_t)l * a.batch + b) * nh * ds;
        float *vst = a.vst + ((int64_t)l * a.batch + b) * nh * hd;
        float *ang = a.angle + ((int64_t)l * a.batch + b) * nh * na;
        // RMSNorm of the residual stream, in_proj
        float ss = 0.0f;
        for (int i = tid; i < dm; i += kTinyThreads) ss = fmaf(res[i], res[i], ss);
        const float inv = rms_inv(block_sum(ss, red), dm, a.eps);
        for (int i = tid; i < dm; i += kTinyThreads) xin[i] = res[i] * inv * lw.norm_w[i];
        __syncthreads();
        gemv_rows(lw.in_proj, dm, ip, xin, proj, part, nullptr);
        const float *braw = proj + 2 * di, *craw = braw + ng * ds;
        const float *sc = proj + 2 * di + 2 * ng * ds;   // dd_dt | dd_A | trap | angles
        // B/C RMSNorm over d_state per group (bcnorm_fwd, ops/norms.rs:50-80)
        for (int grp = 0; grp < ng; grp++) {
            float sb = 0.0f, scs = 0.0f;
            for (int n = tid; n < ds; n += kTinyThreads) {
                sb = fmaf(braw[grp * ds + n], braw[grp * ds + n], sb);
                scs = fmaf(craw[grp * ds + n], craw[grp * ds + n], scs);
            }
            sb = block_sum(sb, red);
            scs = block_sum(scs, red);
            if (tid == 0) {
                ginv[2 * grp] = 1.0f / sqrtf(sb / (float)ds + a.eps);
                ginv[2 * grp + 1] = 1.0f / sqrtf(scs / (float)ds + a.eps);
            }
        }
        __syncthreads();
        // K and Q of every head: weight, per-head bias
        for (int i = tid; i < nh * ds; i += kTinyThreads) {
            const int h = i / ds, n = i - h * ds, grp = h / (nh / ng);
            kl[i] = braw[grp * ds + n] * ginv[2 * grp] * lw.bnw[n] + lw.b_bias[i];
            ql[i] = craw[grp * ds + n] * ginv[2 * grp + 1] * lw.cnw[n] + lw.c_bias[i];
        }
        __syncthreads();
        // angle accumulation (f64, wrapped to [0, 2 pi)) and rotation of the first 2 nr coordinates of K and Q
        for (int i = tid; i < nh * nr; i += kTinyThreads) {
            const int h = i / nr, r = i - h * nr;
            const float dtv = softplus20(sc[h] + lw.dt_bias[h]);
            const float delta = tanhf(sc[3 * nh + r]) * kPi * dtv;
            const float an = (float)wrap_2pi((double)ang[i] + (double)delta);
            ang[i] = an;
            float sn, cs;
            sincosf(an, &sn, &cs);
            float *kp2 = kl + h * ds + 2 * r, *qp2 = ql + h * ds + 2 * r;
            const float b0 = kp2[0], b1 = kp2[1], c0 = qp2[0], c1 = qp2[1];
            kp2[0] = cs * b0 - sn * b1; kp2[1] = sn * b0 + cs * b1;
            qp2[0] = cs * c0 - sn * c1; qp2[1] = sn * c0 + cs * c1;
        }
        __syncthreads();
        // trapezoidal update of one float4 of state per lane-task, y = H q + D x (lane-task = (head, row p, quad g))
        for (int t = tid; t < tasks; t += kTinyThreads) {
            const int h = t / per_head, rem = t - h * per_head, p = rem / lg, g = rem - p * lg;
            float *Hrow = ssm + ((int64_t)h * hd + p) * ds + 4 * g;
            float4 H = *reinterpret_cast<const float4 *>(Hrow);
            const float4 kp = *reinterpret_cast<const float4 *>(kst + h * ds + 4 * g);
            const float vp = vst[h * hd + p];
            const float xv = proj[di + h * hd + p];
            const float dtv = softplus20(sc[h] + lw.dt_bias[h]);
            const float a_val = fminf(-heavy_tail(sc[nh + h]), -a.a_floor);
            const float trap = sigmoidf_fast(sc[2 * nh + h]);
            const float al = fast_exp2(a_val * dtv * kLog2e);
            const float be = al * dtv * (1.0f - trap), ga = trap * dtv;
            const float4 kc = *reinterpret_cast<const float4 *>(&kl[h * ds + 4 * g]);
            const float4 qc = *reinterpret_cast<const float4 *>(&ql[h * ds + 4 * g]);
            const float bv = be * vp, gx = ga * xv;
            H.x = fmaf(al, H.x, fmaf(bv, kp.x, gx * kc.x));
            H.y = fmaf(al, H.y, fmaf(bv, kp.y, gx * kc.y));
            H.z = fmaf(al, H.z, fmaf(bv, kp.z, gx * kc.z));
            H.w = fmaf(al, H.w, fmaf(bv, kp.w, gx * kc.w));
            float acc = H.x * qc.x;
            acc = fmaf(H.y, qc.y, acc);
            acc = fmaf(H.z, qc.z, acc);
            acc = fmaf(H.w, qc.w, acc);
            for (int m = 1; m < lg; m <<= 1) acc += __shfl_xor(acc, m, kWave);
            *reinterpret_cast<float4 *>(Hrow) = H;
            if (g == 0) yr[h * hd + p] = fmaf(lw.D[h], xv, acc);
        }
        __syncthreads();   // every read of the previous k_state and v_state has returned
        for (int i = tid; i < nh * ds; i += kTinyThreads) kst[i] = kl[i];
        // gate: y * silu(z), or RMSNormGated over the head first (rmsnorm_gated_forward, ops/norms.rs:84-114)
        for (int i = tid; i < di; i += kTinyThreads) {
            const float xv = proj[di + i], zi = proj[i];
            vst[i] = xv;
            float o = yr[i] * silu(zi);
            if (a.outproj_norm) {
                const int h = i / hd;
                float sq = 0.0f;
                for (int p = 0; p < hd; p++) sq = fmaf(yr[h * hd + p], yr[h * hd + p], sq);
                o = yr[i] * (1.0f / sqrtf(sq / (float)hd + a.eps)) * lw.ngw[i] * silu(zi);
            }
            yg[i] = o;
        }
        __syncthreads();
        gemv_rows(lw.out_proj, di, dm, yg, xin, part, nullptr);
        for (int i = tid; i < dm; i += kTinyThreads) res[i] += xin[i];
        __syncthreads();
    }
    float ss = 0.0f;
    for (int i = tid; i < dm; i += kTinyThreads) ss = fmaf(res[i], res[i], ss);
    const float inv = rms_inv(block_sum(ss, red), dm, a.eps);
    for (int i = tid; i < dm; i += kTinyThreads) {
        const float v = res[i] * inv * a.norm_f[i];
        leave(a.host.out != nullptr, a.temporal + (int64_t)b * dm + i, v);
        if (a.host.out) host_store(a.host.out + (int64_t)b * dm + i, v);
    }
    if (a.host.out) host_row_done(a.host, b);
}

// The same step with the weights streamed (tiny_step.hip: why and how), for models of the default expand, headdim, d_state, groups and rope
// fraction without the norm in front of out_proj; of those this route takes d_model 64 and 128.  A thread holds its rows of the next layer's
// in_proj in registers, z and x columns and the narrow rest as two sweeps, and those of out_proj in LDS.  Six barriers a layer: partial sums of in_proj | its columns |
// rotations and the heads' coefficients, one lane each | state update, which takes its K and Q from in_proj's columns itself | out_proj | its sums.
// A layer 5.7 us at d_model 128 with 48 rows (before: 13.3; its 460 KB come in in 3.4); the step of four layers, with the host's rows, in a loop of steps 63.8 -> 41.3 us, one
// row 57.7 -> 35.0, 1024 rows 383 -> 282, d_model 64 with 16 rows 47.5 -> 26.3.
template <int DM> __global__ __launch_bounds__(kTinyThreads) void tiny_m3_stream_step_kernel(TinyM3StepArgs a) {
    extern __shared__ float lds[];
    constexpr int di = 2 * DM, ds = 16, hd = 16, nh = di / hd, nr = 4, ip = 2 * di + 2 * ds + 3 * nh + nr, rest = ip - 2 * di;
    constexpr int lg = ds / 4, rows_pp = kTinyThreads / lg, passes = di / rows_pp;   // state update: a float4 of state per lane
    using In = Sweep<DM, 2 * di, ip>;
    using Rest = Sweep<DM, rest, ip>;
    using Out = Sweep<di, DM>;
    static_assert(di % rows_pp == 0 && 4 * DM <= kTinyThreads && 4 * rest <= kTinyThreads && 2 * di <= kTinyThreads && nh * nr <= 64 && nh <= 64, "one thread each");
    float *part = lds;                  // [kTinyPart]  partial sums of z | x, of out_proj
    float *part2 = part + kTinyPart;    // [Rest::n][rest]
    float *res = part2 + Rest::n * rest;   // [DM]  residual stream of this row
    float *gate = res + DM;             // [di]   silu(z)
    float *xs = gate + di;              // [di]   x
    float *y = xs + di;                 // [di]   gated y
    float *cols = y + di;               // [rest] B | C | dd_dt | dd_A | trap | angles
    float *turn = cols + rest;          // [nh][nr][2]  cos, sin
    float *coef = turn + 2 * nh * nr;   // [nh][4]  alpha, beta, gamma
    float *xin = coef + 4 * nh;         // [kStreamInput]  input row, then residual stream times norm weight
    float *vec = xin + kStreamInput;    // [10][256]  B bias, C bias, next norm weight, dt bias, B norm, C norm, D, previous K; previous x, angles
    float *wo = vec + 2560;             // [Out::rows][threads] float4: out_proj's rows, each thread its own (last: the others are reached by constant offsets)
    const int tid = threadIdx.x, b = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned wo_at = lds_address(wo) + 1024u * wave, vec_at = lds_address(vec) + 1024u * wave;

    float4 wi[In::rows], wr[Rest::rows];
    auto ask_in = [&](const float *W, unsigned off, int j0, int n) {
#pragma unroll
        for (int j = j0; j < j0 + n; j++) wi[j] = ld4(global(W + j * ip), off);
    };
    auto ask_rest = [&](const float *W, unsigned off) {
#pragma unroll
        for (int j = 0; j < Rest::rows; j++) wr[j] = ld4(global(W + j * ip + 2 * di), off);
    };
    auto ask_out = [&](const float *W, unsigned off, int j0, int n) {
#pragma unroll
        for (int j = j0; j < j0 + n; j++) dma_kb(wo_at + (unsigned)j * (16u * kTinyThreads), W + j * DM, off);
    };
    TinyM3StepLayer lw = table_entry(a.layers), lnext = table_entry(a.layers + min(1, a.n_layers - 1));
    stream_input<DM>(a, lw.norm_w, xin, res, part, [&] {
        ask_in(lw.in_proj, In(tid).off, 0, In::rows);
        ask_rest(lw.in_proj, Rest(tid).off);
    });

    auto layer = [&](auto last_layer, int l) {
        constexpr bool kLast = decltype(last_layer)::value;
        const int tid = (int)own(threadIdx.x), lane = tid & 63, co = min(tid >> 2, DM - 1), cr = min(tid >> 2, rest - 1);   // (not held over the layers)
        const In in(tid);
        const Rest rp(tid);
        const Out op(tid);
        const int64_t row = (int64_t)l * a.batch + b;
        float *hst = a.ssm + row * di * ds, *kst = a.kst + row * nh * ds, *vst = a.vst + row * di, *ang = a.angle + row * nh * nr;
        {   // One or two requests a wave, into LDS: a load of 4 bytes a lane takes as long as one of 16.
            const float *v = wave == 0 ? lw.b_bias : wave == 1 ? lw.c_bias : wave == 2 ? (kLast ? a.norm_f : lnext.norm_w) : wave == 3 ? lw.dt_bias
                           : wave == 4 ? lw.bnw : wave == 5 ? lw.cnw : wave == 6 ? lw.D : kst;
            const int n = wave == 2 ? DM : wave == 3 || wave == 6 ? nh : wave == 4 || wave == 5 ? ds : di;
            dma_kb(vec_at, v, (16u * lane) & (4u * n - 1));   // (a shorter vector is read around)
            if (wave < 2) dma_kb(vec_at + 8 * 1024, wave ? ang : vst, (16u * lane) & (wave ? 4u * nh * nr - 1 : 4u * di - 1));
        }
        const unsigned st4 = own(16u * tid);
        float4 hv[passes];
#pragma unroll
        for (int p = 0; p < passes; p++) hv[p] = ld4(global(hst + p * rows_pp * ds), st4);
        // the k-th eighth of the next layer's in_proj, asked for while the LDS reads before it are under way
        auto feed = [&](int k) {
            pin();
            if (!kLast) ask_in(lnext.in_proj, own(in.off), k * In::rows / 8, In::rows / 8);
            pin();
        };
        // out_proj's rows: half of them during in_proj, a quarter each during its sums and the rotations
        constexpr int out_part = Out::rows * 2 / In::rows;
        auto feed_out = [&](int quarter) {
            pin();
            ask_out(lw.out_proj, op.off, quarter * Out::rows / 4, Out::rows / 4);
            pin();
        };
        pin();
        // RMSNorm and in_proj: 1 / rms is a factor of every column
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f), acr = acc;
        const float ss = lane_squares<DM>(res);
#pragma unroll
        for (int j = 0; j < In::rows; j += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(&xin[in.j * In::rows + j]);
            fma4(acc, x.x, wi[j]); fma4(acc, x.y, wi[j + 1]); fma4(acc, x.z, wi[j + 2]); fma4(acc, x.w, wi[j + 3]);
            pin(acc);
            ask_out(lw.out_proj, op.off, j / 4 * out_part, out_part);   // (the wave has read what these rows replace)
            pin();
        }
#pragma unroll
        for (int j = 0; j < Rest::rows; j += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(&xin[rp.j * Rest::rows + j]);
            fma4(acr, x.x, wr[j]); fma4(acr, x.y, wr[j + 1]); fma4(acr, x.z, wr[j + 2]); fma4(acr, x.w, wr[j + 3]);
        }
        pin(acr);
        const float inv = rms_inv(wave_sum(ss), DM, a.eps);
        if (in.on) *reinterpret_cast<float4 *>(&part[in.j * 2 * di + 4 * in.q]) = acc;
        if (rp.on) *reinterpret_cast<float4 *>(&part2[rp.j * rest + 4 * rp.q]) = acr;
        // The vectors are in LDS: half of out_proj's requests are newer, and loads come back in order (stores that are still open only raise the count).  Of that half
        // a part is waited for as well: as fast as letting all of it be under way (the step of four layers, 48 rows, 41.4 us both ways).
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Out::rows / 4) : "memory");
        lds_barrier();
        {
            const float r = inv * quad_sum(part_sum<rest, Rest::n, 4>(part2, cr, tid & 3, [] {}));
            const float p = inv * part_sum<2 * di, In::n, 1>(part, min(tid, 2 * di - 1), 0, [&] { feed_out(2); });
            if ((tid & 3) == 0 && tid < 4 * rest) cols[cr] = r;
            if (tid < di) gate[tid] = silu(p);
            else if (tid < 2 * di) xs[tid - di] = p;
        }
        lds_barrier();
        feed_out(3);
        pin();
        if (!kLast) ask_rest(lnext.in_proj, own(rp.off));
        pin();
        // the angles (f64, wrapped to [0, 2 pi)) by the first wave, a lane each; alpha, beta, gamma by the second, a lane per head
        const float *sc = cols + 2 * ds;   // dd_dt | dd_A | trap | angles
        if (wave == 0 && tid < nh * nr) {
            const int h = tid / nr;
            const float dtv = softplus20(sc[h] + vec[3 * 256 + h]);
            const float delta = tanhf(sc[3 * nh + tid % nr]) * kPi * dtv;
            const float an = (float)wrap_2pi((double)vec[9 * 256 + tid] + (double)delta);
            ang[tid] = an;
            float sn, cs;
            sincosf(an, &sn, &cs);
            turn[2 * tid] = cs; turn[2 * tid + 1] = sn;
        } else if (wave == 1 && lane < nh) {
            const float dtv = softplus20(sc[lane] + vec[3 * 256 + lane]);
            const float a_val = fminf(-heavy_tail(sc[nh + lane]), -a.a_floor);
            const float trap = sigmoidf_fast(sc[2 * nh + lane]);
            const float al = fast_exp2(a_val * dtv * kLog2e);
            coef[4 * lane] = al; coef[4 * lane + 1] = al * dtv * (1.0f - trap); coef[4 * lane + 2] = trap * dtv;
        }
        // B/C RMSNorm (bcnorm_fwd, ops/norms.rs:50-80), weight: what K and Q of every head have in common, this lane's four columns
        const int g = tid % lg;
        float kn[4], qn[4];
        {
            const float4 bv = *reinterpret_cast<const float4 *>(&cols[4 * g]), cv = *reinterpret_cast<const float4 *>(&cols[ds + 4 * g]);
            const float4 bw = *reinterpret_cast<const float4 *>(&vec[4 * 256 + 4 * g]), cw = *reinterpret_cast<const float4 *>(&vec[5 * 256 + 4 * g]);
            feed(0);
            const float sb = quad_sum(fmaf(bv.w, bv.w, fmaf(bv.z, bv.z, fmaf(bv.y, bv.y, bv.x * bv.x))));
            const float sq = quad_sum(fmaf(cv.w, cv.w, fmaf(cv.z, cv.z, fmaf(cv.y, cv.y, cv.x * cv.x))));
            const float ib = 1.0f / sqrtf(sb / (float)ds + a.eps), ic = 1.0f / sqrtf(sq / (float)ds + a.eps);
            kn[0] = bv.x * ib * bw.x; kn[1] = bv.y * ib * bw.y; kn[2] = bv.z * ib * bw.z; kn[3] = bv.w * ib * bw.w;
            qn[0] = cv.x * ic * cw.x; qn[1] = cv.y * ic * cw.y; qn[2] = cv.z * ic * cw.z; qn[3] = cv.w * ic * cw.w;
        }
        if (kLast) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // out_proj's rows (ahead of the state's stores)
        lds_barrier();
        // trapezoidal update of one float4 of state per lane and pass, y = H q + D x, gate
#pragma unroll
        for (int p = 0; p < passes; p++) {
            const int d = tid / lg + p * rows_pp, h = d / hd, c = 4 * g;
            const float4 kp = *reinterpret_cast<const float4 *>(&vec[7 * 256 + h * ds + c]), bb = *reinterpret_cast<const float4 *>(&vec[h * ds + c]);
            const float4 cb = *reinterpret_cast<const float4 *>(&vec[256 + h * ds + c]), cf = *reinterpret_cast<const float4 *>(&coef[4 * h]);
            const float4 tr = *reinterpret_cast<const float4 *>(&turn[2 * (h * nr + 2 * (g & 1))]);   // the pairs 2 g and 2 g + 1, if they turn
            const float vp = vec[8 * 256 + d], xv = xs[d], gv = gate[d], Dv = vec[6 * 256 + h];
            feed(1 + p);
            float4 k = make_float4(kn[0] + bb.x, kn[1] + bb.y, kn[2] + bb.z, kn[3] + bb.w), q = make_float4(qn[0] + cb.x, qn[1] + cb.y, qn[2] + cb.z, qn[3] + cb.w);
            if (c < 2 * nr) {   // the first 2 nr coordinates
                k = make_float4(tr.x * k.x - tr.y * k.y, tr.y * k.x + tr.x * k.y, tr.z * k.z - tr.w * k.w, tr.w * k.z + tr.z * k.w);
                q = make_float4(tr.x * q.x - tr.y * q.y, tr.y * q.x + tr.x * q.y, tr.z * q.z - tr.w * q.w, tr.w * q.z + tr.z * q.w);
            }
            const float bv = cf.y * vp, gx = cf.z * xv;
            float4 H = hv[p];
            H.x = fmaf(cf.x, H.x, fmaf(bv, kp.x, gx * k.x));
            H.y = fmaf(cf.x, H.y, fmaf(bv, kp.y, gx * k.y));
            H.z = fmaf(cf.x, H.z, fmaf(bv, kp.z, gx * k.z));
            H.w = fmaf(cf.x, H.w, fmaf(bv, kp.w, gx * k.w));
            *reinterpret_cast<float4 *>(reinterpret_cast<char *>(hst + p * rows_pp * ds) + st4) = H;
            if (d % hd == 0) *reinterpret_cast<float4 *>(kst + h * ds + c) = k;
            float s = H.x * q.x;
            s = fmaf(H.y, q.y, s);
            s = fmaf(H.z, q.z, s);
            s = fmaf(H.w, q.w, s);
            s = quad_sum(s);
            if (g == 0) y[d] = fmaf(Dv, xv, s) * gv;
        }
        if (tid < di) vst[tid] = xs[tid];
        if (passes == 1) feed(2);
        feed(3);
        // The wave's rows of out_proj are in LDS: half of in_proj's requests are newer (and, as above, a part of them is waited for).
        if (!kLast) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(In::rows / 4) : "memory");
        pin();
        lds_barrier();
        // out_proj and residual
        acc = stream_out_sweep(op, y, wo, [&](int turn) { feed(4 + turn); });
        if (op.on) *reinterpret_cast<float4 *>(&part[op.j * DM + 4 * op.q]) = acc;
        lds_barrier();
        const float os = quad_sum(part_sum<DM, Out::n, 4>(part, co, tid & 3, [&] { feed(7); }));
        if ((tid & 3) == 0 && tid < 4 * DM) {
            const float r = res[co] + os;
            res[co] = r;
            xin[co] = r * vec[2 * 256 + co];
        }
        lds_barrier();
    };
    for (int l = 0; l + 1 < a.n_layers; l++) {
        const TinyM3StepLayer after = table_entry(a.layers + min(l + 2, a.n_layers - 1));
        layer(std::false_type(), l);
        lw = lnext;
        lnext = after;
    }
    layer(std::true_type(), a.n_layers - 1);
    stream_output<DM>(a, a.host.out != nullptr, xin, res);
}

template <int DM> bool tiny_m3_stream_fits(const TinyM3StepArgs &a) {
    return a.dm == DM && a.di == 2 * DM && a.hd == 16 && a.ds == 16 && a.ng == 1 && a.nr == 4 && !a.outproj_norm && a.input_dim <= kStreamInput;
}
template <int DM> int launch_tiny_m3_stream(hipStream_t st, const TinyM3StepArgs &a) {
    constexpr int di = 2 * DM, nh = di / 16, rest = 36 + 3 * nh, ip = 2 * di + rest;
    constexpr size_t lds = sizeof(float) * (kTinyPart + Sweep<DM, rest, ip>::n * rest + DM + 3 * di + rest + 8 * nh + 4 * nh + kStreamInput + 2560 + (size_t)Sweep<di, DM>::rows * 4 * kTinyThreads);
    static_assert(lds <= 160 * 1024, "LDS");
    static const hipError_t attr = hipFuncSetAttribute((const void *)tiny_m3_stream_step_kernel<DM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "tiny Mamba-3 backbone step: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL(tiny_m3_stream_step_kernel<DM>, dim3((unsigned)a.batch), dim3(kTinyThreads), lds, st, a);
    return check_launch("tiny_m3_stream_step_kernel");
}

size_t tiny_m3_lds_bytes(int input_dim, int dm, int di, int nh, int ds, int ng, int ip) {
    const int xin_n = rup4(input_dim > dm ? input_dim : dm);
    return sizeof(float) * ((size_t)rup4(dm) + xin_n + rup4(ip) + 2 * (size_t)rup4(nh * ds) + 2 * (size_t)rup4(di) + rup4(2 * ng) + kTinyPart + kTinyThreads / 64);
}

}  // namespace

bool tiny_m3_step_ok(int dtype, int input_dim, int dm, int di, int nh, int hd, int ds, int ng, int nr, int ip) {
    if (dtype != MRS_F32 || input_dim < 1 || input_dim > 4096 || dm < 4 || dm % 4 != 0 || dm > 2048 || ip % 4 != 0 || ip > 2048 || di < 1 || di > 1024)
        return false;
    const int lg = ds / 4;
    if (ds % 4 != 0 || lg < 1 || lg > 64 || (lg & (lg - 1)) != 0 || nh < 1 || ng < 1 || nh % ng != 0 || nh * hd != di || nr < 0 || 2 * nr > ds) return false;
    if (ip != 2 * di + 2 * ng * ds + 3 * nh + nr) return false;
    if (sweep_rounds(input_dim, dm) > kTinyMaxRounds || sweep_rounds(dm, ip) > kTinyMaxRounds || sweep_rounds(di, dm) > kTinyMaxRounds) return false;
    return tiny_m3_lds_bytes(input_dim, dm, di, nh, ds, ng, ip) <= 64 * 1024;
}

int launch_tiny_m3_step(hipStream_t st, const TinyM3StepArgs &a) {
    if (!tiny_m3_step_ok(MRS_F32, a.input_dim, a.dm, a.di, a.nh, a.hd, a.ds, a.ng, a.nr, a.ip) || a.batch < 1 || a.n_layers < 1 || !a.layers ||
        !a.input || !a.ssm || !a.kst || !a.vst || !a.angle || !a.temporal || !a.norm_f)
        return fail(MRS_E_SHAPE, "tiny Mamba-3 backbone step: shape outside the single-launch route (d_model=%d d_inner=%d d_state=%d in_proj width=%d)",
                    a.dm, a.di, a.ds, a.ip);
    if (tiny_m3_stream_fits<128>(a)) return launch_tiny_m3_stream<128>(st, a);
    if (tiny_m3_stream_fits<64>(a)) return launch_tiny_m3_stream<64>(st, a);
    const size_t lds = tiny_m3_lds_bytes(a.input_dim, a.dm, a.di, a.nh, a.ds, a.ng, a.ip);
    hipLaunchKernelGGL(tiny_m3_backbone_step_kernel, dim3((unsigned)a.batch), dim3(kTinyThreads), lds, st, a);
    return check_launch("tiny_m3_backbone_step_kernel");
}

}  // namespace mrs
