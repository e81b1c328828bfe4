// A whole Mamba-3 SISO backbone step in one resident launch, for one batch row (or a few, each on a group of workgroups of its own):
// the Mamba-3 counterpart of resident_step.hip.
//
// The reference's step is fourteen launches per layer (src/mamba3_siso/gpu/inference.rs:506-1000), the kernel chain of
// m3_engine.hip three; at a few rows each of those costs what the hand-over between dependent kernels costs.  Here workgroup s
// of G owns d_inner / G channels of one head -- their columns of in_proj (z and x), their rows of the state -- d_model / G
// columns of out_proj, and an equal share of the columns that every head needs (B, C, dt, A, trap, angles).  Per layer:
//   in_proj on the normed residual row   -> exchange 2: the shared columns, f32
//   B/C norm, bias and rotation of the own head (every workgroup of a head forms them itself), state update, gate
//                                        -> exchange 3: y
//   out_proj, residual add               -> exchange 1: the next layer's operand and sums of squares
// Values are rounded to the storage type where the kernel chain rounds them: the operand rows, y and out_proj's result.
//
// What bounds it: three all-to-all exchanges and the chain between them, not the weights (7.4 MB a layer at d_model 768).
// Per bf16 step, kernel chain / this (routes of one build, steps queued): four layers of d_model 64 46 / 26 us at one row and 49 / 27 at
// 32; of d_model 256 50 / 33 at eight; of d_model 768 57 / 42 at two; 24 layers of 768 317 / 230 at two (kept on the chain all the same,
// kResidentM3Layers in m3_engine.hip says why).  One row of a width that is a multiple of 256 takes resident_m3_row.hip.
#include "resident_m3.hpp"

namespace mrs {
namespace {

constexpr int kInSteps = 4, kInTiles = (2 * kMaxNc + kMaxEx) / 16, kOutSteps = 8;   // k-steps of 32 per computing wave, 16-column tiles

struct Fix {   // LDS: what has a small bound lies at fixed offsets, the weights and rows behind it (bytes)
    static constexpr int pre = 0, pre2 = pre + kComputeWaves * 16 * kInTiles * 4, xz = pre2 + kComputeWaves * 16 * 4, kl = xz + 2 * kMaxNc * 4,
                         ql = kl + kMaxDs * 4, coef = ql + kMaxDs * 4, inv = coef + 16, xs = inv + 16;
};
struct ResLds { int ys, small, wout, win, total; };
__host__ __device__ inline ResLds res_lds(int dm, int di, int cols, int oc, int ds) {
    ResLds o;
    o.ys = Fix::xs + dm * 2;
    o.small = o.ys + di * 2;
    o.wout = o.small + 2 * small_block(ds, oc).bytes;   // (two small blocks in turn)
    o.win = o.wout + up1k(oc * di * 2);
    o.total = o.win + up1k(cols * dm * 2);
    return o;
}

template <typename T>
__global__ __launch_bounds__(kResThreads) void resident_m3_step_kernel(const ResidentM3Args *args, TokenRows rows) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int state;   // kRollCall, 0, or a ResidentFault
    const auto state_now = [] { return __hip_atomic_load(&state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    const auto *a = as_table(args);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = a->G, b = blockIdx.x / G, src = blockIdx.x - b * G;
    const int dm = a->dm, di = a->di, nl = a->n_layers, nc = a->nc, oc = a->oc, ex = a->ex, ds = a->ds, nh = a->nh, hd = a->hd, ng = a->ng, nr = a->nr;
    const int c0 = src * nc, o0 = src * oc, cols = 2 * nc + ex;
    const ResLds L = res_lds(dm, di, cols, oc, ds);
    const SmallBlock sb = small_block(ds, oc);

    if (wave >= kComputeWaves) {
        const LayerBlock lb = layer_block(dm, di, cols, oc, ds);
        const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
        bring_weights({(const char *)a->weights + (size_t)src * lb.bytes, (size_t)G * lb.bytes, lds0 + L.win, lds0 + L.wout, lds0 + L.small, lb.out, lb.small,
                       sb.bytes, a->cached}, wave, nl, state, {a->roll, a->broken, gridDim.x, a->wait, 0});
        return;
    }

    // ---- the waves that compute
    T *xs = (T *)(smem + Fix::xs), *ys = (T *)(smem + L.ys);
    const T *win = (const T *)(smem + L.win), *wout = (const T *)(smem + L.wout);
    float *pre = (float *)(smem + Fix::pre), *pre2 = (float *)(smem + Fix::pre2), *xz = (float *)(smem + Fix::xz), *kl = (float *)(smem + Fix::kl),
          *ql = (float *)(smem + Fix::ql), *coef = (float *)(smem + Fix::coef), *invl = (float *)(smem + Fix::inv);
    const int shared = 2 * ng * ds + 3 * nh + nr;   // columns of in_proj behind z and x
    u64 *e1 = a->xch + (size_t)b * a->xch_stride, *e1s = e1 + (dm >> 1), *e2 = e1s + G, *e3 = e2 + shared;   // this row's buffers
    unsigned *epoch = a->epoch + 32 * b;
    const unsigned base = *epoch;
    const int lane = tid & 63, ct_in = (cols + 15) >> 4, LG = ds >> 2;   // LG lanes per state row, four states each
    const int head = c0 / hd, grp = head / (nh / ng), na = max(nr, 1);
    const bool head_owner = c0 == head * hd;      // stores what a head's workgroups all form: k and the angles
    const int p = tid / LG, g = tid - p * LG;     // channel and lane of a state row: threads below nc * LG
    const bool scans = tid < nc * LG;
    // this row's states of layer 0, and from a layer to the next
    const size_t bh = (size_t)b * nh + head, heads = (size_t)a->batch * nh;
    float *hst = a->ssm + ((size_t)b * di + c0) * ds, *kst = a->kst + bh * ds, *vst = a->vst + (size_t)b * di + c0, *ast = a->angle + bh * na;
    const size_t hst_l = (size_t)a->batch * di * ds, kst_l = heads * ds, vst_l = (size_t)a->batch * di, ast_l = heads * na;

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
    pin.take(win, cols, dm >> 5, ct_in);

#pragma unroll 1
    for (int l = 0; l < nl; l++) {
        const unsigned tag = base + 1 + l;
        const bool more = l + 1 < nl;
        const char *small = smem + L.small + (l & 1) * sb.bytes;
        // the state, for after exchange 2
        float *Hrow = hst + l * hst_l + 4 * (scans ? here(tid) : 0), *vrow = vst + l * vst_l + (scans ? p : 0);
        float4 H = *reinterpret_cast<const float4 *>(Hrow);
        const float4 kp = *reinterpret_cast<const float4 *>(kst + l * kst_l + 4 * (scans ? g : 0));
        const float vp = *vrow;
        const int pair = min(here(lane) >> 1, na - 1);
        float ang = wave < 2 ? ast[l * ast_l + pair] : 0.0f;
        // ---- in_proj
        const float inv = l == 0 ? inv0 : invl[0];
        pin.run(xs, dm >> 5, ct_in, pre);
        lds_barrier();   // 1
        bool ok = true;
        const auto tagged = [&](u64 w) { return (unsigned)(w >> 32) == tag; };
        if (wave == kComputeWaves - 1) {
            const int e = src * ex + here(lane);   // this workgroup's share of the shared columns
            if (here(lane) < ex && e < shared) xch_put(e2 + e, row_sum(pre, 16 * ct_in, 2 * nc + here(lane)) * inv, tag);
        } else if (wave == kComputeWaves - 2) {
            if (here(lane) < 2 * nc) xz[here(lane)] = row_sum(pre, 16 * ct_in, here(lane)) * inv;
        } else if (wave < 2) {
            // ---- wave 0 forms k from B, wave 1 q from C: RMSNorm over d_state, the head's bias, the rotation of the first 2 nr coordinates by
            // the accumulated angle (f64, wrapped); a lane per coordinate
            const int n = min(here(lane), ds - 1), at = (wave == 0 ? grp : ng + grp) * ds + n, sc = 2 * ng * ds;
            u64 r[3];
            ok = xch_poll<3>(e2, [&](int u) { return (unsigned)(u == 0 ? at : u == 1 ? sc + head : nr > 0 ? sc + 3 * nh + pair : at); }, tagged, r, state_now);
            const float raw = __uint_as_float((unsigned)r[0]);
            const float *nw = reinterpret_cast<const float *>(small + (wave == 0 ? sb.bnw : sb.cnw)), *bias = reinterpret_cast<const float *>(small + (wave == 0 ? sb.bb : sb.cb));
            const float sq = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wave_sum_last(here(lane) < ds ? raw * raw : 0.0f)), 63));
            const float scale = 1.0f / sqrtf(sq / (float)ds + a->eps);
            float v = raw * scale * nw[n] + bias[n];
            if (nr > 0) {
                const float dtv = softplus20(__uint_as_float((unsigned)r[1]) + *reinterpret_cast<const float *>(small + sb.dtb));
                const float delta = tanhf(__uint_as_float((unsigned)r[2])) * kPi * dtv;
                ang = (float)wrap_2pi((double)ang + (double)delta);
                float sn, cs;
                sincosf(ang, &sn, &cs);
                const float other = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xb1, 0xf, 0xf, true));   // the pair's other coordinate
                if (here(lane) < 2 * nr) v = (lane & 1) ? sn * other + cs * v : cs * v - sn * other;
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
            H.x = fmaf(co.x, H.x, fmaf(bv, kp.x, gx * kc.x));
            H.y = fmaf(co.x, H.y, fmaf(bv, kp.y, gx * kc.y));
            H.z = fmaf(co.x, H.z, fmaf(bv, kp.z, gx * kc.z));
            H.w = fmaf(co.x, H.w, fmaf(bv, kp.w, gx * kc.w));
            float acc = H.x * qc.x;
            acc = fmaf(H.y, qc.y, acc);
            acc = fmaf(H.z, qc.z, acc);
            acc = fmaf(H.w, qc.w, acc);
            // over the row's 4, 8 or 16 lanes
            acc += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0xb1, 0xf, 0xf, true));    // quad_perm [1,0,3,2]
            acc += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0x4e, 0xf, 0xf, true));    // quad_perm [2,3,0,1]
            const float o8 = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0x141, 0xf, 0xf, true));   // row_half_mirror
            acc += LG > 4 ? o8 : 0.0f;
            const float o16 = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(acc), 0x140, 0xf, 0xf, true));  // row_mirror
            acc += LG > 8 ? o16 : 0.0f;
            const T yr = (T)(fmaf(*reinterpret_cast<const float *>(small + sb.D), xv, acc) * silu(zi));
            const float yn = __shfl_down(Store<T>::ld(&yr), LG, kWave);   // the next channel's
            if (g == 0 && (p & 1) == 0) xch_put_word(e3 + (unsigned)((c0 + p) >> 1), half_pair_word<T>(yr, (T)yn, tag));
            *reinterpret_cast<float4 *>(Hrow) = H;
            if (g == 0) *vrow = xv;
        }
        // ---- y of all channels
        pout.take(wout, oc, di >> 5, 1);   // while y is on its way
        ok = take_y(e3, di, tag, ys) && ok;
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 3
        if (state) break;
        // every workgroup of the head has used the previous k and angles for the y that is now here
        if (head_owner) {
            if (scans && p == 0) *reinterpret_cast<float4 *>(kst + l * kst_l + 4 * g) = kc;
            if (wave == 0 && (lane & 1) == 0 && (lane >> 1) < nr) ast[l * ast_l + (lane >> 1)] = ang;
        }
        // ---- out_proj, residual, the next operand
        pout.run(ys, di >> 5, 1, pre2);
        lds_barrier();   // 4
        put_operand<T>(pre2, oc, o0, src, more ? reinterpret_cast<const float *>(small + sb.nw) : nullptr, e1, e1s, tag, res0, res1);
        if (more) pin.take(win, cols, dm >> 5, ct_in);   // while the operand row is on its way
        ok = take_operand(e1, e1s, G, dm, a->eps, tag, more, xs, invl) && ok;
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // 5
        if (state) break;
    }
    // final norm of this workgroup's columns
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

// A layer's weights in the order the workgroups bring them in: one block of layer_block() per workgroup.  in_t [ip][dm] and out_t
// [dm][di] transposed; a thread writes 16 bytes of a block.
struct PackArgs {
    const uint16_t *in_t, *out_t;
    const float *bnw, *cnw, *b_bias, *c_bias, *D, *dt_bias, *next_nw;
    int dm, di, ip, ds, hd, nc, oc, ex, row_order;
};
__global__ __launch_bounds__(256) void pack_m3_layer_kernel(char *__restrict__ dst, PackArgs p) {
    const int cols = 2 * p.nc + p.ex;
    const LayerBlock lb = layer_block(p.dm, p.di, cols, p.oc, p.ds);
    const SmallBlock sb = small_block(p.ds, p.oc);
    const int s = blockIdx.y, c0 = s * p.nc, o0 = s * p.oc, head = c0 / p.hd;
    const int at = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 16;
    if (at >= lb.bytes) return;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (at < lb.out) {
        const int i = at >> 4, n8 = p.dm >> 3, c = p.row_order ? i / n8 : i % cols, k8 = p.row_order ? i % n8 : i / cols;
        // in_proj's columns are [z: di | x: di | shared]
        const int col = c < p.nc ? p.di + c0 + c : c < 2 * p.nc ? c0 + c - p.nc : 2 * p.di + s * p.ex + c - 2 * p.nc;
        if (k8 < n8 && c < cols && col < p.ip) v = *reinterpret_cast<const uint4 *>(p.in_t + (size_t)col * p.dm + k8 * 8);
    } else if (at < lb.small) {
        const int i = (at - lb.out) >> 4, n8 = p.di >> 3, c = p.row_order ? i / n8 : i % p.oc, k8 = p.row_order ? i % n8 : i / p.oc;
        if (k8 < n8 && c < p.oc) v = *reinterpret_cast<const uint4 *>(p.out_t + (size_t)(o0 + c) * p.di + k8 * 8);
    } else {
        const int q = at - lb.small;
        unsigned w[4] = {0, 0, 0, 0};
        for (int k = 0; k < 4; k++) {
            const int o = q + 4 * k;
            const float *f = nullptr;
            if (o < sb.cnw) f = p.bnw + (o >> 2);
            else if (o < sb.bb) f = p.cnw + ((o - sb.cnw) >> 2);
            else if (o < sb.cb) f = p.b_bias + (size_t)head * p.ds + ((o - sb.bb) >> 2);
            else if (o < sb.nw) f = p.c_bias + (size_t)head * p.ds + ((o - sb.cb) >> 2);
            else if (o < sb.D) f = p.next_nw ? p.next_nw + o0 + ((o - sb.nw) >> 2) : nullptr;
            else if (o == sb.D) f = p.D + head;
            else if (o == sb.dtb) f = p.dt_bias + head;
            if (f) w[k] = __float_as_uint(*f);
        }
        v = make_uint4(w[0], w[1], w[2], w[3]);
    }
    *reinterpret_cast<uint4 *>(dst + (size_t)s * lb.bytes + at) = v;
}

int shared_cols(const ResidentM3Args &a) { return 2 * a.ng * a.ds + 3 * a.nh + a.nr; }
bool shape_ok(const ResidentM3Args &a, int dtype) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && a.dm % 32 == 0 && a.di % 32 == 0 && a.dm <= 32 * kComputeWaves * kInSteps &&
           a.di <= 32 * kComputeWaves * kOutSteps && (a.ds == 16 || a.ds == 32 || a.ds == 64) && a.nr >= 0 && 2 * a.nr <= a.ds && a.nh * a.hd == a.di &&
           a.ng >= 1 && a.nh % a.ng == 0;
}
bool plan_ok(const ResidentM3Args &a) {
    return (a.nc == 8 || a.nc == 16) && a.hd % a.nc == 0 && a.nc * a.G == a.di && a.oc >= 2 && a.oc % 2 == 0 && a.oc <= kMaxOc && a.oc * a.G == a.dm &&
           a.ex >= 1 && a.ex <= kMaxEx && a.ex * a.G >= shared_cols(a) &&
           (a.row_order ? resident_m3_row_lds(a) : (size_t)res_lds(a.dm, a.di, 2 * a.nc + a.ex, a.oc, a.ds).total) <= kResLdsMax;
}

}  // namespace

// (a.row_order set: the plan of resident_m3_row.hip.)  A workgroup's channels belong to one head; as few workgroups as the plan allows, as in resident_plan().
bool resident_m3_plan(ResidentM3Args &a, int dtype) {
    if (!shape_ok(a, dtype) || (a.row_order && !resident_m3_row_ok(a, dtype))) return false;
    for (a.nc = kMaxNc; a.nc >= 8; a.nc -= 8) {
        if (a.di % a.nc) continue;
        a.G = a.di / a.nc;
        a.oc = a.dm / a.G;
        a.ex = (shared_cols(a) + a.G - 1) / a.G;
        if (!plan_ok(a)) continue;
        a.xch_stride = (size_t)((a.row_order ? a.dm : a.dm / 2 + a.G) + shared_cols(a) + a.di / 2);
        return true;
    }
    return false;
}

size_t resident_m3_layer_bytes(const ResidentM3Args &a) { return (size_t)a.G * layer_block(a.dm, a.di, 2 * a.nc + a.ex, a.oc, a.ds).bytes; }

int launch_resident_m3_pack(hipStream_t st, const ResidentM3Args &a, void *dst, const ResidentM3Layer &w) {
    const PackArgs p = {(const uint16_t *)w.in_t, (const uint16_t *)w.out_t, w.bnw, w.cnw, w.b_bias, w.c_bias, w.D, w.dt_bias, w.next_nw,
                        a.dm, a.di, 2 * a.di + shared_cols(a), a.ds, a.hd, a.nc, a.oc, a.ex, a.row_order};
    const int n16 = layer_block(a.dm, a.di, 2 * a.nc + a.ex, a.oc, a.ds).bytes / 16;
    hipLaunchKernelGGL(pack_m3_layer_kernel, dim3((unsigned)((n16 + 255) / 256), (unsigned)a.G), dim3(256), 0, st, (char *)dst, p);
    return check_launch("pack_m3_layer_kernel");
}

template <typename T>
static int launch_resident_m3_t(hipStream_t st, const ResidentM3Args &a, const ResidentM3Args *dev, const TokenRows &rows) {
    static const hipError_t attr = hipFuncSetAttribute((const void *)resident_m3_step_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kResLdsMax);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "resident step: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((resident_m3_step_kernel<T>), dim3((unsigned)(a.G * a.batch)), dim3(kResThreads),
                       (size_t)res_lds(a.dm, a.di, 2 * a.nc + a.ex, a.oc, a.ds).total, st, dev, rows);
    return check_launch("resident_m3_step_kernel");
}

int launch_resident_m3_step(hipStream_t st, int dtype, const ResidentM3Args &a, const ResidentM3Args *dev, const TokenRows &rows) {
    if (!shape_ok(a, dtype) || !plan_ok(a) || a.batch < 1 || a.G * a.batch > kRollMax || a.n_layers < 1 || !a.weights || !a.norm_w || !a.norm_f || !a.input || !a.xch || !a.epoch ||
        !a.roll || !a.broken || !a.temporal || !a.temporal_t || !a.ssm || !a.kst || !a.vst || !a.angle || !dev)
        return fail(MRS_E_SHAPE, "resident Mamba-3 step: shape outside the route (d_model=%d d_inner=%d d_state=%d workgroups=%d)", a.dm, a.di, a.ds, a.G);
    if (a.row_order) return launch_resident_m3_row(st, dtype, a, dev, rows);
    return dtype == MRS_BF16 ? launch_resident_m3_t<bf16_t>(st, a, dev, rows) : launch_resident_m3_t<f16_t>(st, a, dev, rows);
}

}  // namespace mrs
