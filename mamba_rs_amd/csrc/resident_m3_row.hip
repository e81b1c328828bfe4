// The resident Mamba-3 step (resident_m3_step.hip) for one row with the kernel chain's own sums: every product, every sum of squares and
// every rounding is the one that gemm_skinny.hip's row-wise route and m3_layer_step_kernel make, in their order, so that a model of any
// depth steps through one launch and keeps the bits, and with them the tokens, of the chain.
//
// A column's product is 32 or 64 lanes along its weight row (v_dot2), then a butterfly over them.  That needs no sum across waves: a wave
// that has finished a column of in_proj puts it into the exchange by itself, the shared ones first, and out_proj's eight columns are one
// for each wave.  The exchange of the residual row carries the f32 values, for everybody forms the 16-column sums of squares
// of the chain from them; the next operand is rounded where it arrives.
//
// What bounds it: the same three exchanges a layer as in resident_m3_step.hip, with less between them -- no sums across waves through LDS,
// and one barrier fewer before a result leaves.  Per step at one row, kernel chain / the matrix-core step / this: 24 layers of d_model 768
// 266 / 212 / 159 us, of 1024 328 / - / 196; four layers of 768 53 / 38 / 31, of 256 49 / 30 / 23 (bf16; f16 the same within 1 us).
#include "dot8.hpp"
#include "resident_m3.hpp"

namespace mrs {
namespace {

// Sums over the 32 lanes of each half and over the 64 lanes of a wave, in every lane, as v += shfl_xor(v, m) with m = 32 (64 lanes only),
// 16, 8, 4, 2, 1 makes them.
__device__ __forceinline__ float butterfly32(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return row16_sum(__uint_as_float(a[0]) + __uint_as_float(a[1]));
}
__device__ __forceinline__ float butterfly64(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return butterfly32(__uint_as_float(a[0]) + __uint_as_float(a[1]));
}
__device__ __forceinline__ float rounded(float v) { asm volatile("" : "+v"(v)); return v; }   // a product that is not to become part of an fma

// KI: d_model / 256 (d_inner twice that).  LPR lanes along a row of in_proj, CW columns of a wave at a time, PER pieces of a lane each.
template <int KI> struct RowOrder {
    static constexpr int dm = 256 * KI, di = 2 * dm, LPR = KI % 2 ? 32 : 64, CW = 64 / LPR, PER = dm / 8 / LPR, OPER = di / 8 / 64,
                         rounds = (2 * kMaxNc + kMaxEx + CW * kComputeWaves - 1) / (CW * kComputeWaves), tiles = dm / 16, words = (dm + kCompute - 1) / kCompute;
    static constexpr int part = 0, pre = part + 64 * 4, xz = pre + 16, kl = xz + 2 * kMaxNc * 4, ql = kl + kMaxDs * 4, coef = ql + kMaxDs * 4, xs = coef + 16,
                         ys = xs + dm * 2, small = ys + di * 2;   // LDS bytes
    __host__ __device__ static int wout(int small_bytes) { return small + 2 * small_bytes; }
    __host__ __device__ static int win(int small_bytes, int oc) { return wout(small_bytes) + up1k(oc * di * 2); }
    __host__ __device__ static int total(int small_bytes, int oc, int cols) { return win(small_bytes, oc) + up1k(cols * dm * 2); }
};

template <typename T, int KI>
__global__ __launch_bounds__(kResThreads) void resident_m3_row_kernel(const ResidentM3Args *args, TokenRows rows) {
    using S = RowOrder<KI>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int state;   // kRollCall, 0, or a ResidentFault
    const auto state_now = [] { return __hip_atomic_load(&state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    const auto *a = as_table(args);
    constexpr int dm = S::dm, di = S::di;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = a->G, src = blockIdx.x;
    const int nl = a->n_layers, nc = a->nc, oc = a->oc, ex = a->ex, ds = a->ds, nh = a->nh, hd = a->hd, ng = a->ng, nr = a->nr;
    const int c0 = src * nc, o0 = src * oc, cols = 2 * nc + ex;
    const SmallBlock sb = small_block(ds, oc);

    if (wave >= kComputeWaves) {
        const LayerBlock lb = layer_block(dm, di, cols, oc, ds);
        const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
        bring_weights({(const char *)a->weights + (size_t)src * lb.bytes, (size_t)G * lb.bytes, lds0 + S::win(sb.bytes, oc), lds0 + S::wout(sb.bytes),
                       lds0 + S::small, lb.out, lb.small, sb.bytes, a->cached}, wave, nl, state, {a->roll, a->broken, gridDim.x, a->wait, 0});
        return;
    }

    // ---- the waves that compute
    T *xs = (T *)(smem + S::xs);
    unsigned *ys = (unsigned *)(smem + S::ys);
    float *rl = (float *)ys;   // the last residual row, when y is no longer read
    static_assert(di * 2 >= dm * 4);
    const uint4 *win = (const uint4 *)(smem + S::win(sb.bytes, oc)), *wout = (const uint4 *)(smem + S::wout(sb.bytes));
    float *part = (float *)(smem + S::part), *pre = (float *)(smem + S::pre), *xz = (float *)(smem + S::xz), *kl = (float *)(smem + S::kl),
          *ql = (float *)(smem + S::ql), *coef = (float *)(smem + S::coef);
    const int shared = 2 * ng * ds + 3 * nh + nr;   // columns of in_proj behind z and x
    u64 *e1 = a->xch, *e2 = e1 + dm, *e3 = e2 + shared;
    const unsigned base = *a->epoch;
    const int lane = tid & 63, LG = ds >> 2;        // LG lanes per state row, four states each
    const int head = c0 / hd, grp = head / (nh / ng), na = max(nr, 1);
    const bool head_owner = c0 == head * hd;        // stores what a head's workgroups all form: k and the angles
    const int p = tid / LG, g = tid - p * LG;       // channel and lane of a state row: threads below nc * LG
    const bool scans = tid < nc * LG;
    float *hst = a->ssm + (size_t)c0 * ds, *kst = a->kst + (size_t)head * ds, *vst = a->vst + c0, *ast = a->angle + (size_t)head * na;
    const size_t hst_l = (size_t)di * ds, kst_l = (size_t)nh * ds, vst_l = di, ast_l = (size_t)nh * na;

    // layer 0's operand and sum of squares: 256 threads, as prenorm_rows_kernel
    float res = 0.0f;   // the residual stream: column o0 + wave, in every lane of the wave
    const int ow = min(wave, oc - 1);
    with_input_row<T>(a->input, rows, 0, dm, [&](auto in, bool taken) {
        const float *nw = a->norm_w;
        if (wave < 4) {
            float ss = 0.0f;
#pragma unroll
            for (int k = 0; k < KI; k++) {
                const float v = in(tid + 256 * k);
                ss = fmaf(v, v, ss);
                Store<T>::st(xs + tid + 256 * k, v * nw[tid + 256 * k]);
            }
            ss = butterfly64(ss);
            if (lane == 0) pre[wave] = ss;
        }
        res = in(o0 + ow);
        if (taken && lane == 0 && wave < oc) a->input[o0 + wave] = res;
    });
    lds_barrier();
    const float inv0 = inv_rms(pre[0] + pre[1] + pre[2] + pre[3], dm, a->eps);   // later row scales: from the tiles' sums

    uint4 wi[S::rounds][S::PER], wo[S::OPER];
    // columns from the last one down: the shared ones, which all wait for, come first
    const int ll = lane & (S::LPR - 1), half = S::LPR == 64 ? 0 : lane >> 5;
    const auto take_in = [&] {
#pragma unroll
        for (int r = 0; r < S::rounds; r++) {
            const int c = max(cols - 1 - (S::CW * (wave + kComputeWaves * r) + half), 0);
#pragma unroll
            for (int j = 0; j < S::PER; j++) wi[r][j] = win[(unsigned)(here(c) * (dm / 8) + ll + S::LPR * j)];
        }
    };
    take_in();

#pragma unroll 1
    for (int l = 0; l < nl; l++) {
        const unsigned tag = base + 1 + l;
        const bool more = l + 1 < nl;
        const char *small = smem + S::small + (l & 1) * sb.bytes;
        // the state, for after exchange 2
        float *Hrow = hst + l * hst_l + 4 * (scans ? here(tid) : 0), *vrow = vst + l * vst_l + (scans ? p : 0);
        float4 H = *reinterpret_cast<const float4 *>(Hrow);
        const float4 kp = *reinterpret_cast<const float4 *>(kst + l * kst_l + 4 * (scans ? g : 0));
        const float vp = *vrow;
        const int pair = min(here(lane) >> 1, na - 1);
        float ang = wave < 2 ? ast[l * ast_l + pair] : 0.0f;
        float nw[S::words];   // the next layer's norm weights
#pragma unroll
        for (int u = 0; u < S::words; u++) nw[u] = a->norm_rows[(size_t)(more ? l + 1 : l) * dm + min(here(tid) + kCompute * u, dm - 1)];
        // ---- in_proj
        {
            float sum[S::rounds];
            uint4 x[S::PER];
#pragma unroll
            for (int j = 0; j < S::PER; j++) x[j] = reinterpret_cast<const uint4 *>(xs)[ll + S::LPR * j];
            float inv = inv0;
            if (l > 0) inv = inv_rms(butterfly64(lane < S::tiles ? part[lane] : 0.0f), dm, a->eps);
#pragma unroll
            for (int r = 0; r < S::rounds; r++) {
                sum[r] = 0.0f;
#pragma unroll
                for (int j = 0; j < S::PER; j++) sum[r] = dot8<T>(x[j], wi[r][j], sum[r]);
                const float v = (S::LPR == 64 ? butterfly64(sum[r]) : butterfly32(sum[r])) * inv;
                const int q = S::CW * (wave + kComputeWaves * r) + here(half), c = cols - 1 - q;
                if (here(ll) == 0 && c >= 0) {
                    const int e = src * ex + c - 2 * nc;
                    if (c < 2 * nc) xz[c] = v;
                    else if (e < shared) xch_put(e2 + e, v, tag);
                }
            }
        }
        lds_barrier();   // 1
        bool ok = true;
        const auto tagged = [&](u64 w) { return (unsigned)(w >> 32) == tag; };
        if (wave < 2) {
            // ---- wave 0 forms k from B, wave 1 q from C: RMSNorm over d_state, the head's bias, the rotation of the first 2 nr coordinates by
            // the accumulated angle (f64, wrapped); a lane per coordinate
            const int n = min(here(lane), ds - 1), at = (wave == 0 ? grp : ng + grp) * ds + n, sc = 2 * ng * ds;
            u64 r[3];
            ok = xch_poll<3>(e2, [&](int u) { return (unsigned)(u == 0 ? at : u == 1 ? sc + head : nr > 0 ? sc + 3 * nh + pair : at); }, tagged, r, state_now);
            const float raw = __uint_as_float((unsigned)r[0]), val = here(lane) < ds ? raw : 0.0f;
            const float *nwp = reinterpret_cast<const float *>(small + (wave == 0 ? sb.bnw : sb.cnw)), *bias = reinterpret_cast<const float *>(small + (wave == 0 ? sb.bb : sb.cb));
            // lane 0's sum: the first step of the chain's butterfly is an fma, a lane's own square onto its partner's (right in the lower lanes here)
            const float sq = rounded(val * val);
            const auto hi = __builtin_amdgcn_permlane32_swap(__float_as_uint(sq), __float_as_uint(sq), false, false);
            const float tot = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(butterfly32(fmaf(val, val, __uint_as_float(hi[1]))))));
            const float scale = 1.0f / sqrtf(tot / (float)ds + a->eps);
            float v = fmaf(raw * scale, nwp[n], bias[n]);
            if (nr > 0) {
                const float dtv = softplus20(__uint_as_float((unsigned)r[1]) + *reinterpret_cast<const float *>(small + sb.dtb));
                const float delta = tanhf(__uint_as_float((unsigned)r[2])) * kPi * dtv;
                ang = (float)wrap_2pi((double)ang + (double)delta);
                float sn, cs;
                sincosf(ang, &sn, &cs);
                const float other = rounded(sn * __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xb1, 0xf, 0xf, true)));   // by the pair's other coordinate
                if (here(lane) < 2 * nr) v = fmaf(cs, v, (lane & 1) ? other : -other);
            }
            if (here(lane) < ds) (wave == 0 ? kl : ql)[here(lane)] = v;
        } else if (wave == 2) {
            // ---- alpha, beta, gamma of the head
            const int sc = 2 * ng * ds + head;
            u64 r[3];
            ok = xch_poll<3>(e2, [&](int u) { return (unsigned)(sc + u * nh); }, tagged, r, state_now);
            const float dtv = softplus20(__uint_as_float((unsigned)r[0]) + *reinterpret_cast<const float *>(small + sb.dtb));
            const float a_val = fminf(-heavy_tail(__uint_as_float((unsigned)r[1])), -a->a_floor), trap = sigmoidf_fast(__uint_as_float((unsigned)r[2]));
            const float al = fast_exp2(a_val * dtv * kLog2e);
            if (lane == 0) *reinterpret_cast<float4 *>(coef) = make_float4(al, al * dtv * (1.0f - trap), trap * dtv, 0.0f);
        }
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 2
        if (state) break;
        // ---- trapezoidal update of this lane's four states, y = H q + D x, SiLU gate
        float4 kc = make_float4(0.f, 0.f, 0.f, 0.f);
        if (scans) {
            const float4 co = *reinterpret_cast<const float4 *>(coef), qc = *reinterpret_cast<const float4 *>(ql + 4 * g);
            kc = *reinterpret_cast<const float4 *>(kl + 4 * g);
            const float xv = xz[p], zi = xz[nc + p], bv = co.y * vp, gx = co.z * xv;
            H.x = fmaf(co.x, H.x, fmaf(bv, kp.x, rounded(gx * kc.x)));
            H.y = fmaf(co.x, H.y, fmaf(bv, kp.y, rounded(gx * kc.y)));
            H.z = fmaf(co.x, H.z, fmaf(bv, kp.z, rounded(gx * kc.z)));
            H.w = fmaf(co.x, H.w, fmaf(bv, kp.w, rounded(gx * kc.w)));
            float acc = H.x * qc.x;
            acc = fmaf(H.y, qc.y, acc);
            acc = fmaf(H.z, qc.z, acc);
            acc = fmaf(H.w, qc.w, acc);
            // over the row's 4, 8 or 16 lanes
            acc += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0xb1, 0xf, 0xf, true));    // quad_perm [1,0,3,2]
            acc += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0x4e, 0xf, 0xf, true));    // quad_perm [2,3,0,1]
            const float o8 = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0x141, 0xf, 0xf, true));   // row_half_mirror
            acc = LG > 4 ? acc + o8 : acc;
            const float o16 = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0x140, 0xf, 0xf, true));  // row_mirror
            acc = LG > 8 ? acc + o16 : acc;
            const T yr = (T)(fmaf(*reinterpret_cast<const float *>(small + sb.D), xv, acc) * silu(zi));
            const float yn = __shfl_down(Store<T>::ld(&yr), LG, kWave);   // the next channel's
            if (g == 0 && (p & 1) == 0) xch_put_word(e3 + (unsigned)((c0 + p) >> 1), half_pair_word<T>(yr, (T)yn, tag));
            *reinterpret_cast<float4 *>(Hrow) = H;
            if (g == 0) *vrow = xv;
        }
        // ---- y of all channels
#pragma unroll
        for (int j = 0; j < S::OPER; j++) wo[j] = wout[(unsigned)(here(ow) * (di / 8) + lane + 64 * j)];   // while y is on its way
        ok = take_y(e3, di, tag, (T *)ys) && ok;
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 3
        if (state) break;
        // every workgroup of the head has used the previous k and angles for the y that is now here
        if (head_owner) {
            if (scans && p == 0) *reinterpret_cast<float4 *>(kst + l * kst_l + 4 * g) = kc;
            if (wave == 0 && (lane & 1) == 0 && (lane >> 1) < nr) ast[l * ast_l + (lane >> 1)] = ang;
        }
        // ---- out_proj, a column per wave; residual
        {
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j < S::OPER; j++) sum = dot8<T>(reinterpret_cast<const uint4 *>(ys)[here(lane) + 64 * j], wo[j], sum);
            const T o = (T)butterfly64(sum);
            res += Store<T>::ld(&o);
            if (here(lane) == 0 && wave < oc) xch_put(e1 + (unsigned)(o0 + wave), res, tag);
        }
        lds_barrier();   // 4
        if (more) take_in();   // while the residual row is on its way
        // ---- the residual row: the next operand, and the sums of squares of its tiles of 16 columns
        if (S::words > 1 || dm >= kCompute || wave < dm / 64) {
            const int t = here(tid);
            u64 r[S::words];
            ok = xch_poll<S::words>(e1, [&](int u) { return (unsigned)min(t + kCompute * u, dm - 1); }, tagged, r) && ok;
#pragma unroll
            for (int u = 0; u < S::words; u++) {
                const int i = t + kCompute * u;
                if (dm % kCompute != 0 && u == S::words - 1 && i >= dm) continue;   // whole waves
                const float v = __uint_as_float((unsigned)r[u]), s = row16_sum(rounded(v * v));
                if (more) Store<T>::st(xs + i, v * nw[u]);
                else rl[i] = v;
                if ((t & 15) == 0) part[i >> 4] = s;
            }
        }
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 5
        if (state) break;
    }
    // final norm of this wave's column: the sum of squares of 256 threads, as add_rmsnorm_kernel
    const bool lost = state != 0;
    if (wave < oc) {
        float q[4];
#pragma unroll
        for (int w = 0; w < 4; w++) {
            float ss = 0.0f;
#pragma unroll
            for (int k = 0; k < KI; k++) {
                const float v = rl[64 * w + lane + 256 * k];
                ss = fmaf(v, v, ss);
            }
            q[w] = butterfly64(ss);
        }
        const float inv = inv_rms(q[0] + q[1] + q[2] + q[3], dm, a->eps);
        if (lane == 0) {
            const float o = lost ? __uint_as_float(0x7fc00000u) : res * inv * a->norm_f[o0 + wave];
            a->temporal[o0 + wave] = o;
            Store<T>::st((T *)a->temporal_t + o0 + wave, o);
        }
    }
    if (tid == 0) {
        if (state == kStepLost) {
            __hip_atomic_store(a->roll, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a->broken, (unsigned)kStepLost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (src == 0) *a->epoch = base + nl;   // every workgroup has read it: each has published the last exchange
    }
}

template <typename T, int KI> int launch_t(hipStream_t st, const ResidentM3Args &a, const ResidentM3Args *dev, const TokenRows &rows) {
    static const hipError_t attr = hipFuncSetAttribute((const void *)resident_m3_row_kernel<T, KI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kResLdsMax);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "resident step: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((resident_m3_row_kernel<T, KI>), dim3((unsigned)a.G), dim3(kResThreads), resident_m3_row_lds(a), st, dev, rows);
    return check_launch("resident_m3_row_kernel");
}
template <typename T> int launch(hipStream_t st, const ResidentM3Args &a, const ResidentM3Args *dev, const TokenRows &rows) {
    switch (a.dm / 256) {
    case 1: return launch_t<T, 1>(st, a, dev, rows);
    case 2: return launch_t<T, 2>(st, a, dev, rows);
    case 3: return launch_t<T, 3>(st, a, dev, rows);
    default: return launch_t<T, 4>(st, a, dev, rows);
    }
}

}  // namespace

bool resident_m3_row_ok(const ResidentM3Args &a, int dtype) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && a.batch == 1 && a.dm % 256 == 0 && a.dm >= 256 && a.dm <= 1024 && a.di == 2 * a.dm;
}

size_t resident_m3_row_lds(const ResidentM3Args &a) {
    const int sb = small_block(a.ds, a.oc).bytes, cols = 2 * a.nc + a.ex;
    switch (a.dm / 256) {
    case 1: return (size_t)RowOrder<1>::total(sb, a.oc, cols);
    case 2: return (size_t)RowOrder<2>::total(sb, a.oc, cols);
    case 3: return (size_t)RowOrder<3>::total(sb, a.oc, cols);
    default: return (size_t)RowOrder<4>::total(sb, a.oc, cols);
    }
}

int launch_resident_m3_row(hipStream_t st, int dtype, const ResidentM3Args &a, const ResidentM3Args *dev, const TokenRows &rows) {
    if (!resident_m3_row_ok(a, dtype) || a.oc > kComputeWaves || !a.norm_rows) return fail(MRS_E_SHAPE, "resident Mamba-3 step: shape outside the row-order route");
    return dtype == MRS_BF16 ? launch<bf16_t>(st, a, dev, rows) : launch<f16_t>(st, a, dev, rows);
}

}  // namespace mrs
