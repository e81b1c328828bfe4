// A whole Mamba-1 backbone step in one resident launch, for one batch row (or a few, each on a group of workgroups of its own).
//
// The reference runs a decode step as 4 GEMMs and 10 kernels per layer (src/mamba_ssm/gpu/inference.rs:993-1252), the kernel
// chain of engine.hip as three or four; at a few rows each of those launches costs what the hand-over between dependent
// kernels costs (about 4 us), whatever it moves.  Here G workgroups stay on the chip for the whole step.  Workgroup s owns
// d_inner / G channels -- their columns of in_proj (both halves), conv windows, taps, x_proj rows, dt weights and SSM state
// -- and d_model / G columns of out_proj with the residual stream's elements there.  Per layer:
//   in_proj on the normed residual row (every workgroup holds the whole row), conv + SiLU of its own channels, their share of
//   the x_proj row           -> exchange 2: G shares of the x_proj row, added by every workgroup in the same order
//   dt_proj + softplus, state update, gate of its own channels -> exchange 3: y
//   out_proj, residual add   -> exchange 1: the next layer's operand round(residual * norm weight), and sums of squares
// A layer's weights go straight from memory to LDS, by waves that do nothing else, while the others wait for their neighbours.
// Values are rounded to the storage type where the kernel chain rounds them.
//
// The layer loop is kept small on purpose (products on the matrix cores, rolled loops, operands in LDS): every layer runs through it
// once, and code that does not stay in the instruction cache costs more than the work (the same step with the weights in
// registers and unrolled loops, 100 KB of code: 427 us for 24 layers of d_model 768; with vector dot products whose sizes are
// run-time values, 30 KB: 285 to 340 us).
#include "resident_m1.hpp"

namespace mrs {
namespace {

// Lines of exchange 2 per workgroup, a wave each.
__host__ __device__ constexpr int share_lines(int xd) { return (xd + kLineVals - 1) / kLineVals; }
static_assert(share_lines(kMaxXd) <= kComputeWaves, "");
constexpr int kInSteps = 4, kInTiles = 2 * kMaxNc / 16, kOutSteps = 8;      // k-steps of 32 per computing wave and 16-column tiles held in registers

struct Fix {   // LDS: what has a small bound lies at fixed offsets, the weights and rows behind it (bytes)
    static constexpr int pre = 0, pre2 = pre + kComputeWaves * 2 * kMaxNc * 4, us = pre2 + kComputeWaves * 16 * 4, zs = us + 64,
                         xdl = zs + 128, inv = xdl + kMaxXd * 4, xs = inv + 64;
};
struct ResLds { int ys, small, wout, win, total; };
__host__ __device__ inline ResLds res_lds(int dm, int di, int nc, int oc, int xd, int dr) {
    ResLds o;
    o.ys = Fix::xs + dm * 2;
    o.small = o.ys + di * 2;
    o.wout = o.small + 2 * small_block(nc, oc, xd, dr).bytes;   // (two small blocks in turn)
    o.win = o.wout + up1k(oc * di * 2);
    o.total = o.win + up1k(2 * nc * dm * 2);
    return o;
}

template <typename T>
__global__ __launch_bounds__(kResThreads) void resident_step_kernel(const ResidentArgs *args, TokenRows rows) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int state;   // kRollCall, 0, or a ResidentFault
    const auto state_now = [] { return __hip_atomic_load(&state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    const auto *a = as_table(args);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = a->G, b = blockIdx.x / G, src = blockIdx.x - b * G;
    const int dm = a->dm, di = a->di, nl = a->n_layers, nc = a->nc, oc = a->oc, xd = a->xd, dr = a->dr;
    const int c0 = src * nc, o0 = src * oc;
    const ResLds L = res_lds(dm, di, nc, oc, xd, dr);
    const SmallBlock sb = small_block(nc, oc, xd, dr);

    if (wave >= kComputeWaves) {
        const LayerBlock lb = layer_block(dm, di, nc, oc, xd, dr);
        const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
        bring_weights({(const char *)a->weights + (size_t)src * lb.bytes, (size_t)G * lb.bytes, lds0 + L.win, lds0 + L.wout, lds0 + L.small, lb.out, lb.small,
                       sb.bytes, a->cached}, wave, nl, state, {a->roll, a->broken, gridDim.x, a->wait, 0});
        return;
    }

    // ---- the waves that compute
    T *xs = (T *)(smem + Fix::xs), *ys = (T *)(smem + L.ys), *us = (T *)(smem + Fix::us);
    const T *win = (const T *)(smem + L.win), *wout = (const T *)(smem + L.wout);
    float *pre = (float *)(smem + Fix::pre), *pre2 = (float *)(smem + Fix::pre2), *zs = (float *)(smem + Fix::zs), *xdl = (float *)(smem + Fix::xdl),
          *invl = (float *)(smem + Fix::inv);
    const int lines = share_lines(xd);
    u64 *e2 = a->xch + (size_t)b * a->xch_stride, *e1 = e2 + (size_t)G * lines * 8, *e1s = e1 + (dm >> 1), *e3 = e1s + G;   // this row's buffers
    unsigned *epoch = a->epoch + 32 * b;
    const unsigned base = *epoch;
    const int lane = tid & 63, ct_in = (2 * nc) >> 4;
    const bool conv_wave = wave < lines;
    float *cst = a->conv_state + ((size_t)b * di + c0) * kDc, *hst = a->ssm_state + ((size_t)b * di + c0) * kDs;   // this workgroup's channels, layer 0
    const size_t cst_l = (size_t)a->batch * di * kDc, hst_l = (size_t)a->batch * di * kDs;                          // ... from a layer to the next

    float4 cwin = make_float4(0.f, 0.f, 0.f, 0.f);
    if (conv_wave) cwin = ld_off<float4>(cst, (unsigned)min(lane, nc - 1) * 16u);
    // the residual stream: columns o0 + 2 p and + 1 of thread p < oc / 2
    float res0 = 0.0f, res1 = 0.0f;
    const bool own = tid < (oc >> 1);
    float ss = 0.0f;
    with_input_row<T>(a->input, rows, b, dm, [&](auto in, bool taken) {
        const float *nw = a->norm_w;
        for (int i = tid; i < dm; i += kCompute) {
            const float v = in(i);
            ss = fmaf(v, v, ss);
            Store<T>::st(xs + i, v * nw[i]);
        }
        if (own) {
            res0 = in(o0 + 2 * tid); res1 = in(o0 + 2 * tid + 1);
            if (taken) *reinterpret_cast<float2 *>(a->input + (size_t)b * dm + o0 + 2 * tid) = make_float2(res0, res1);
        }
    });
    ss = wave_sum_last(ss);
    if (lane == 63) pre2[wave] = ss;
    lds_barrier();
    float inv0 = 0.0f;   // layer 0's row scale; later ones come through LDS
#pragma unroll
    for (int w = 0; w < kComputeWaves; w++) inv0 += pre2[w];
    inv0 = inv_rms(inv0, dm, a->eps);

    RowProduct<T, kInSteps, kInTiles> pin;
    RowProduct<T, kOutSteps, 1> pout;
    pin.take(win, 2 * nc, dm >> 5, ct_in);

#pragma unroll 1
    for (int l = 0; l < nl; l++) {
        const unsigned tag = base + 1 + l;
        const bool more = l + 1 < nl;
        // the scan step's state: channel tid / 16, state tid % 16
        float *hl = hst + l * hst_l;
        float hv = hl[min(here(tid), nc * kDs - 1)];
        const char *small = smem + L.small + (l & 1) * sb.bytes;
        // ---- in_proj
        const float inv = l == 0 ? inv0 : invl[0];
        pin.run(xs, dm >> 5, ct_in, pre);
        lds_barrier();   // 1
        float xnew = 0.0f;
        if (conv_wave) {
            // ---- conv step + SiLU, by every wave that needs the channels
            const int i = min(here(lane), nc - 1);
            const float4 tap = *reinterpret_cast<const float4 *>(small + sb.cw + i * 16);
            const float bias = *reinterpret_cast<const float *>(small + sb.cb + i * 4);
            const T xr = (T)(row_sum(pre, 2 * nc, i) * inv), zr = (T)(row_sum(pre, 2 * nc, nc + i) * inv);
            xnew = Store<T>::ld(&xr);
            float o = fmaf(cwin.y, tap.x, bias);
            o = fmaf(cwin.z, tap.y, o); o = fmaf(cwin.w, tap.z, o); o = fmaf(xnew, tap.w, o);
            us[i] = (T)silu(o);   // (the waves write the same values)
            zs[i] = Store<T>::ld(&zr);
            // ---- share of the x_proj row: a line of 14 entries per wave (the tile's last two columns are not used)
            const int n = here(lane) & 15, kg = here(lane) >> 4;
            uint4 ua = make_uint4(0, 0, 0, 0), wb = ua;
            if (kg * 8 < nc) {
                ua = *reinterpret_cast<const uint4 *>(us + kg * 8);
                wb = *reinterpret_cast<const uint4 *>(small + (kg * xd + min(wave * kLineVals + n, xd - 1)) * 16);
            }
            const v4f s = Mma32<T>::mma(ua, wb, (v4f){0.f, 0.f, 0.f, 0.f});
            const float nb = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(s[0]), 0xb1, 0xf, 0xf, true));   // the neighbour lane's
            const unsigned low = (unsigned)__ballot(__float_as_uint(s[0]) & 1u) & ((1u << kLineVals) - 1u);
            if (here(lane) < 16 && (n & 1) == 0)
                xch_put_word(e2 + (unsigned)((src * lines + wave) * 8 + (n >> 1)), n < kLineVals ? pair_word(s[0], nb, tag) : (u64)tag << 32 | low);
        }
        // ---- the whole x_proj row: a wave per line, eight neighbouring lanes for a workgroup's 64 bytes (with a word's eight workgroups in
        // neighbouring lanes instead, each of them in another line: 24 layers of d_model 768 179 us a step against 171, of 1024 266
        // against 252), the shares in workgroup order within a lane, then over the eight groups of lanes
        bool ok = true;
        {
            constexpr int KU = 8;
            const int q = here(tid) & 7, g = here(tid) >> 3 & 7;   // q 7: the line's low bits
            if (conv_wave) {
                float s0 = 0.0f, s1 = 0.0f;
                const unsigned see_lo = q == 7 ? 0u : 1u, see_hi = q == 7 ? ~0u : 1u;   // a pair's parity, or the tag
#pragma unroll 1
                for (int k0 = g; k0 < G; k0 += 8 * KU) {
                    u64 r[KU];
                    ok = ok && xch_poll<KU>(e2, [&](int u) { return (unsigned)((min(k0 + 8 * u, G - 1) * lines + wave) * 8 + q); },
                                            [&](u64 w) { return ((((unsigned)w ^ tag) & see_lo) | (((unsigned)(w >> 32) ^ tag) & see_hi)) == 0; }, r, state_now);
#pragma unroll
                    for (int u = 0; u < KU; u++) {
                        const unsigned in = k0 + 8 * u < G ? ~0u : 0u, low = last_of_8((unsigned)r[u]);
                        s0 += __uint_as_float(with_bit((unsigned)r[u], low, 2 * q) & in);
                        s1 += __uint_as_float(with_bit((unsigned)(r[u] >> 32), low, 2 * q + 1) & in);
                    }
                }
                const T r0 = (T)groups_sum(s0), r1 = (T)groups_sum(s1);
                const int e = wave * kLineVals + 2 * q;
                if (g == 0 && q < 7 && e < xd) *reinterpret_cast<float2 *>(xdl + e) = make_float2(Store<T>::ld(&r0), Store<T>::ld(&r1));
            }
        }
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 2
        if (state) break;
        // the window, by the first wave: all waves have theirs in registers, they have used it in front of the barrier
        if (wave == 0 && lane < nc) *reinterpret_cast<float4 *>(cst + l * cst_l + lane * kDc) = make_float4(cwin.y, cwin.z, cwin.w, xnew);
        // ---- dt_proj + softplus, state update, D skip, gate: sixteen lanes per channel, one state each
        if (here(tid) < nc * kDs) {
            const int t = here(tid), n = t & 15, cl = t >> 4;
            const float av = *reinterpret_cast<const float *>(small + sb.aneg + t * 4), dtb = *reinterpret_cast<const float *>(small + sb.dtb + cl * 4),
                        Dd = *reinterpret_cast<const float *>(small + sb.D + cl * 4), z = zs[cl];
            const T *wp = (const T *)(small + sb.dtw) + cl * dr;
            float wv[kMaxDr / 16], xv[kMaxDr / 16];
#pragma unroll
            for (int k = 0; k < kMaxDr / 16; k++) {
                const int kk = min(k * 16 + n, dr - 1);
                wv[k] = Store<T>::ld(wp + kk); xv[k] = k * 16 + n < dr ? xdl[kk] : 0.0f;
            }
            const float Bn = xdl[dr + n], Cn = xdl[dr + kDs + n], u = Store<T>::ld(us + cl);
            float td = 0.0f;
#pragma unroll
            for (int k = 0; k < kMaxDr / 16; k++) td = fmaf(xv[k], wv[k], td);
            const float delta = softplus20(row16_sum(td) + dtb);
            const float h = fmaf(fast_exp2(delta * kLog2e * av), hv, delta * u * Bn);
            const float acc = row16_sum(h * Cn);
            const T yr = (T)(fmaf(Dd, u, acc) * silu(z));
            const float yf = Store<T>::ld(&yr), yn = __shfl_down(yf, 16, kWave);   // the next channel's
            if (n == 0 && (cl & 1) == 0) xch_put_word(e3 + (unsigned)((c0 + cl) >> 1), half_pair_word<T>(yr, (T)yn, tag));
            hl[t] = h;
        }
        // ---- y of all channels
        pout.take(wout, oc, di >> 5, 1);   // while y is on its way
        ok = take_y(e3, di, tag, ys) && ok;
        if (!ok && state == 0) state = kStepLost;
        if (more && conv_wave) cwin = ld_off<float4>(cst + (l + 1) * cst_l, (unsigned)min(here(lane), nc - 1) * 16u);
        lds_barrier();   // 3
        if (state) break;
        // ---- out_proj, residual, the next operand
        pout.run(ys, di >> 5, 1, pre2);
        lds_barrier();   // 4
        put_operand<T>(pre2, oc, o0, src, more ? reinterpret_cast<const float *>(small + sb.nw) : nullptr, e1, e1s, tag, res0, res1);
        if (more) pin.take(win, 2 * nc, dm >> 5, ct_in);   // while the operand row is on its way
        ok = take_operand(e1, e1s, G, dm, a->eps, tag, more, xs, invl) && ok;
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 5
        if (state) break;
    }
    // final norm of this workgroup's columns: f32, and once more in the storage type for a head
    const bool lost = state != 0;
    if (own) {
        const float inv = invl[0];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int n = o0 + 2 * tid + k;
            const float o = lost ? __uint_as_float(0x7fc00000u) : (k ? res1 : res0) * inv * a->norm_f[n];
            a->temporal[(size_t)b * dm + n] = o;
            Store<T>::st((T *)a->temporal_t + (size_t)b * dm + n, o);
        }
    }
    if (tid == 0) {
        if (state == kStepLost) {
            __hip_atomic_store(a->roll, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a->broken, (unsigned)kStepLost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (src == 0) *epoch = base + nl;   // every workgroup of the row has read it: each has published the last exchange
    }
}

// A layer's weights in the order the workgroups bring them in: one block of layer_block() per workgroup.  in_t [2 di][dm], out_t [dm][di],
// dt_t [di][dr] transposed, x_proj [di][xd]; a thread writes 16 bytes of a block.
struct PackArgs {
    const uint16_t *in_t, *out_t, *x_proj, *dt_t;
    const float *a_neg, *conv_w, *conv_b, *D, *dt_b, *next_nw;
    int dm, di, xd, dr, nc, oc;
};
__global__ __launch_bounds__(256) void pack_layer_kernel(char *__restrict__ dst, PackArgs p) {
    const LayerBlock lb = layer_block(p.dm, p.di, p.nc, p.oc, p.xd, p.dr);
    const SmallBlock sb = small_block(p.nc, p.oc, p.xd, p.dr);
    const int s = blockIdx.y, c0 = s * p.nc, o0 = s * p.oc;
    const int at = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 16;
    if (at >= lb.bytes) return;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (at < lb.out) {
        const int i = at >> 4, c = i % (2 * p.nc), k8 = i / (2 * p.nc);
        if (k8 < p.dm >> 3) v = *reinterpret_cast<const uint4 *>(p.in_t + (size_t)(c < p.nc ? c0 + c : p.di + c0 + c - p.nc) * p.dm + k8 * 8);
    } else if (at < lb.small) {
        const int i = (at - lb.out) >> 4, c = i % p.oc, k8 = i / p.oc;
        if (k8 < p.di >> 3) v = *reinterpret_cast<const uint4 *>(p.out_t + (size_t)(o0 + c) * p.di + k8 * 8);
    } else {
        const int q = at - lb.small;
        unsigned w[4] = {0, 0, 0, 0};
        for (int k = 0; k < 4; k++) {   // (the parts start on 4-byte boundaries)
            const int o = q + 4 * k;
            const float *f = nullptr;
            if (o < sb.dtw) {
                const int e = o >> 1, c = (e >> 3) / p.xd * 8 + (e & 7), j = (e >> 3) % p.xd;
                w[k] = p.x_proj[(size_t)(c0 + c) * p.xd + j] | (unsigned)p.x_proj[(size_t)(c0 + c + 1) * p.xd + j] << 16;
            } else if (o < sb.aneg) w[k] = *reinterpret_cast<const unsigned *>(p.dt_t + (size_t)c0 * p.dr + ((o - sb.dtw) >> 1));
            else if (o < sb.cw) f = p.a_neg + (size_t)c0 * kDs + ((o - sb.aneg) >> 2);
            else if (o < sb.cb) f = p.conv_w + (size_t)c0 * kDc + ((o - sb.cw) >> 2);
            else if (o < sb.D) f = p.conv_b + c0 + ((o - sb.cb) >> 2);
            else if (o < sb.dtb) f = p.D + c0 + ((o - sb.D) >> 2);
            else if (o < sb.nw) f = p.dt_b + c0 + ((o - sb.dtb) >> 2);
            else if (o < sb.nw + p.oc * 4 && p.next_nw) f = p.next_nw + o0 + ((o - sb.nw) >> 2);
            if (f) w[k] = __float_as_uint(*f);
        }
        v = make_uint4(w[0], w[1], w[2], w[3]);
    }
    *reinterpret_cast<uint4 *>(dst + (size_t)s * lb.bytes + at) = v;
}

}  // namespace

static bool shape_ok(const ResidentArgs &a, int dtype) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && a.dm % 32 == 0 && a.di % 32 == 0 && a.dm <= 32 * kComputeWaves * kInSteps &&
           a.di <= 32 * kComputeWaves * kOutSteps && a.ds == kDs && a.dc == kDc && a.xd % 2 == 0 && a.xd >= 4 && a.xd <= kMaxXd && a.dr >= 2 &&
           a.dr % 2 == 0 && a.dr <= kMaxDr;
}
static bool plan_ok(const ResidentArgs &a) {
    return a.nc >= 8 && a.nc % 8 == 0 && a.nc <= kMaxNc && a.nc * a.G == a.di && a.oc >= 2 && a.oc % 2 == 0 && a.oc <= kMaxOc && a.oc * a.G == a.dm &&
           (size_t)res_lds(a.dm, a.di, a.nc, a.oc, a.xd, a.dr).total <= kResLdsMax;
}

// As few workgroups as the weights' buffers in LDS allow: an exchange among 64 takes 1.5 us, among 128 1.8 us, and the weights
// arrive in time from 64 compute units (d_model 768: 177 us per step with 64 workgroups, 215 with 96).
bool resident_plan(ResidentArgs &a, int dtype) {
    if (!shape_ok(a, dtype)) return false;
    for (a.nc = kMaxNc; a.nc >= 8; a.nc -= 8) {
        if (a.di % a.nc) continue;
        a.G = a.di / a.nc;
        a.oc = a.dm / a.G;
        if (!plan_ok(a)) continue;
        a.groups = a.batch; a.rows = 1; a.rows_buf = nullptr;
        a.xch_stride = ((size_t)a.G * share_lines(a.xd) * 8 + a.dm / 2 + a.G + a.di / 2 + 7) / 8 * 8;   // (lines of 64 bytes)
        return true;
    }
    return false;
}

size_t resident_layer_bytes(const ResidentArgs &a) { return (size_t)a.G * layer_block(a.dm, a.di, a.nc, a.oc, a.xd, a.dr).bytes; }

int launch_resident_pack(hipStream_t st, const ResidentArgs &a, void *dst, const ResidentLayer &w) {
    const PackArgs p = {(const uint16_t *)w.in_t, (const uint16_t *)w.out_t, (const uint16_t *)w.x_proj, (const uint16_t *)w.dt_t, w.a_neg, w.conv_w, w.conv_b,
                        w.D, w.dt_b, w.next_nw, a.dm, a.di, a.xd, a.dr, a.nc, a.oc};
    const int n16 = layer_block(a.dm, a.di, a.nc, a.oc, a.xd, a.dr).bytes / 16;
    hipLaunchKernelGGL(pack_layer_kernel, dim3((unsigned)((n16 + 255) / 256), (unsigned)a.G), dim3(256), 0, st, (char *)dst, p);
    return check_launch("pack_layer_kernel");
}

template <typename T>
static int launch_resident_t(hipStream_t st, const ResidentArgs &a, const ResidentArgs *dev, const TokenRows &rows) {
    static const hipError_t attr = hipFuncSetAttribute((const void *)resident_step_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kResLdsMax);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "resident step: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((resident_step_kernel<T>), dim3((unsigned)(a.G * a.batch)), dim3(kResThreads), (size_t)res_lds(a.dm, a.di, a.nc, a.oc, a.xd, a.dr).total, st, dev, rows);
    return check_launch("resident_step_kernel");
}

int launch_resident_step(hipStream_t st, int dtype, const ResidentArgs &a, const ResidentArgs *dev, const TokenRows &rows) {
    if (!shape_ok(a, dtype) || !plan_ok(a) || a.batch < 1 || a.G * a.batch > kRollMax || a.n_layers < 1 || !a.weights || !a.norm_w || !a.input || !a.xch || !a.epoch || !a.roll || !a.broken ||
        !a.temporal || !a.temporal_t || !dev)
        return fail(MRS_E_SHAPE, "resident step: shape outside the route (d_model=%d d_inner=%d d_state=%d workgroups=%d)", a.dm, a.di, a.ds, a.G);
    return dtype == MRS_BF16 ? launch_resident_t<bf16_t>(st, a, dev, rows) : launch_resident_t<f16_t>(st, a, dev, rows);
}

}  // namespace mrs
