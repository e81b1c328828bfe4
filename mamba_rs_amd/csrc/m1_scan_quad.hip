// Mamba-1 selective scan over short or few sequences (d_state 16): four lanes share a channel, four states each.
//
// m1_scan.hip gives a lane all sixteen states of a channel and a wave 64 channels; that fills the chip with the fewest instructions
// once there are some waves per SIMD.  Below one wave per SIMD it is a lone wave's serial walk that sets the time -- about 500
// clocks per step, sixteen of its instructions on the quarter-rate exponential unit.  Here a step is a quarter of that per
// wave, with four times the waves:
//   * a wave owns 16 channels, lane 4 c + g states 4 g .. 4 g + 3 of channel c; four waves (64 channels) share a workgroup and
//     the staged B / C rows of the chunk, which lie in LDS as f32 from the start;
//   * activations are loaded for four steps at a time, lane g the step t + g, and handed round the four lanes by DPP operands; in the
//     same way lane g keeps the output of step t + g, so that D u, the gate and the store happen once per four steps and lane.
//   * a prompt of up to 64 steps can bring dt_proj along: the wave's 16 channels x 64 steps are four tiles of the matrix cores, and delta stays in
//     f32 in LDS.  For a generation's prompt, which otherwise goes through steps that keep delta in f32; no faster than dt_proj with a
//     rounded delta in front (24 layers, 13 x 11 rows of d_model 1024 995 / 992 us, 48 of 768 888 / 899).
// The two passes and their workspace (chunk summaries, step sums) are those of m1_scan.hip; a short sequence is one pass.  What bounds
// it is the issue of about 35 instructions per step and wave, four of them exponentials: 8 us per million (row, channel) steps once
// the chip is full.  Both kernels timed: at the dispatch in m1_scan.hip.
#include "common.hpp"
#include "mfma_tiles.hpp"
#include "scan_quad.hpp"

namespace mrs {
namespace {

template <int K> __device__ __forceinline__ float quad_lane(float v) {   // lane K of the four
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), K * 0x55, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_sum(float v) {
    v += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xb1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
    return v + __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x4e, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
}

// four elements of a row whose pairs are dword-aligned (16-bit) or which is dword-aligned (f32)
template <typename T> __device__ __forceinline__ v4f row_quad(const T *p) {
    v4f o;
    if constexpr (sizeof(T) == 2) {
        struct alignas(4) P2 { T v[2]; };
        const P2 a = reinterpret_cast<const P2 *>(p)[0], b = reinterpret_cast<const P2 *>(p)[1];
        o = v4f{Store<T>::ld(&a.v[0]), Store<T>::ld(&a.v[1]), Store<T>::ld(&b.v[0]), Store<T>::ld(&b.v[1])};
    } else {
        o = v4f{p[0], p[1], p[2], p[3]};
    }
    return o;
}

// OUT false: pass A -- chunk c < nchunk - 1 from a zero state (chunk 0: the caller's, which it also copies), leaving its end state and
// sum of delta.  OUT true: pass B -- the entering state folded from the summaries before, then y; the last chunk leaves the state.
// DT: delta is formed here.
template <typename T, int GATE, bool OUT, bool DT = false>
__global__ __launch_bounds__(256) void scan_quad_kernel(ScanQuadArgs a) {
    constexpr int kLen = DT ? kQuadDtLen : kQuadLen;
    __shared__ alignas(16) float Bs[kLen][16], Cs[OUT ? kLen : 1][16];
    __shared__ float Ds[DT ? kLen : 1][80];   // [step][channel of the workgroup]
    const int tile = blockIdx.x % a.tiles, rest = blockIdx.x / a.tiles, b = rest % a.batch, c = (OUT ? a.first : 0) + rest / a.batch;
    const int tid = threadIdx.x, lane = tid & 63, g = lane & 3, di = a.di;
    const int d = tile * 64 + (tid >> 2);
    const bool live = d < di;
    const int dd = live ? d : di - 1;   // dead lanes shadow the last channel and store nothing
    const int t0 = c * a.len, ns = min(a.len, a.Tlen - t0), nq = (ns + 3) >> 2;
    const int64_t row0 = (int64_t)b * a.Tlen + t0;
    const T *dp = (const T *)a.delta + row0 * di + dd, *up = (const T *)a.u + row0 * di + dd, *gp = GATE ? (const T *)a.gate + row0 * a.gate_stride + dd : nullptr;

    // four groups of four steps at a time, the next ones requested before the current ones are worked on
    constexpr int NB = 4;
    T rd[NB], ru[NB], rg[NB], nd[NB], nu[NB], ng[NB];
    auto request = [&](T (&x)[NB], T (&w)[NB], T (&z)[NB], int q0) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int64_t t = min(4 * (q0 + i) + g, ns - 1);
            if (DT) x[i] = (T)0.0f; else x[i] = dp[t * di];
            w[i] = up[t * di];
            if (GATE) z[i] = gp[t * a.gate_stride];
        }
    };
    request(rd, ru, rg, 0);
    float a2[4], h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) a2[j] = a.a_neg[(int64_t)dd * 16 + 4 * g + j] * kLog2e;
    const float Dd = OUT ? a.D[dd] : 0.0f;
    float *hp = a.h + ((int64_t)b * di + dd) * 16 + 4 * g;
    const int64_t own = (int64_t)(4 * g) * di + dd;   // states 4 g .. of channel dd in a [16][di] block: + j di
    // the chunk's B and C rows; the rows that fill up the last group are zeros (their steps have delta u = 0)
    {
        const T *Bp = (const T *)a.B + row0 * a.bc_stride, *Cp = (const T *)a.C + row0 * a.bc_stride;
        for (int i = tid; i < 16 * nq; i += 256) {
            const int row = i >> 2, q = 4 * (i & 3);
            v4f bv = {0.f, 0.f, 0.f, 0.f}, cv = bv;
            if (row < ns) {
                bv = row_quad(Bp + row * a.bc_stride + q);
                if (OUT) cv = row_quad(Cp + row * a.bc_stride + q);
            }
            *reinterpret_cast<v4f *>(&Bs[row][q]) = bv;
            if (OUT) *reinterpret_cast<v4f *>(&Cs[row][q]) = cv;
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) h[j] = 0.0f;
    if (c == 0) {
        float *copy = a.h0copy + (int64_t)b * 16 * di + own;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            h[j] = OUT && a.nchunk > 1 ? copy[(int64_t)j * di] : hp[j];
            if (!OUT && live) copy[(int64_t)j * di] = h[j];
        }
    } else if (OUT) {
        // sum over k < c of exp(a sum of the delta sums between) S_k, as in m1_scan.hip; four chunks' summaries requested together
        const int64_t sbase = (int64_t)b * (a.nchunk - 1);
#pragma unroll
        for (int j = 0; j < 4; j++) h[j] = a.S[(sbase + c - 1) * 16 * di + own + (int64_t)j * di];
        float suffix = 0.0f;
        for (int k0 = c - 2; k0 >= 0; k0 -= 4) {
            float Sv[4][4], sm[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = max(k0 - i, 0);
                sm[i] = a.sumd[(sbase + k + 1) * di + dd];
#pragma unroll
                for (int j = 0; j < 4; j++) Sv[i][j] = a.S[(sbase + k) * 16 * di + own + (int64_t)j * di];
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (k0 - i >= 0) {
                    suffix += sm[i];
#pragma unroll
                    for (int j = 0; j < 4; j++) h[j] = fmaf(fast_exp2(suffix * a2[j]), Sv[i][j], h[j]);
                }
        }
    }
    if constexpr (DT) {
        // this wave's 16 channels: dt_proj on the matrix cores, step 16 m + 4 (l / 16) + i in register i of tile m
        const int n = lane & 15, kg = lane >> 4, ch = min(tile * 64 + (tid >> 6) * 16 + n, di - 1), mt = (ns + 15) >> 4;
        const T *wp = (const T *)a.dt_w + (int64_t)ch * a.dr, *xp = (const T *)a.dt_in + row0 * a.bc_stride;
        v4f td[kLen / 16];
#pragma unroll
        for (int m = 0; m < kLen / 16; m++) td[m] = v4f{0.f, 0.f, 0.f, 0.f};
        for (int k = 8 * kg; k - 8 * kg < a.dr; k += 32) {
            const bool in = k < a.dr;
            const uint4 none = make_uint4(0, 0, 0, 0);
            const uint4 w = in ? *reinterpret_cast<const uint4 *>(wp + k) : none;
#pragma unroll
            for (int m = 0; m < kLen / 16; m++)
                if (m < mt) td[m] = Mma32<T>::mma(in ? *reinterpret_cast<const uint4 *>(xp + (int64_t)min(16 * m + n, ns - 1) * a.bc_stride + k) : none, w, td[m]);
        }
        const float bias = a.dt_b[ch];
#pragma unroll
        for (int m = 0; m < kLen / 16; m++)
            if (m < mt)
#pragma unroll
                for (int i = 0; i < 4; i++) Ds[16 * m + 4 * kg + i][(tid >> 6) * 16 + n] = softplus20(td[m][i] + bias);
    }
    __syncthreads();
    float sd = 0.0f;
    for (int q0 = 0; q0 < nq; q0 += NB) {
        request(nd, nu, ng, q0 + NB);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int q = q0 + i, s = 4 * q + g;
            if (q < nq) {   // (uniform)
                const bool in = s < ns;
                const float dl = !in ? 0.0f : DT ? Ds[s][tid >> 2] : Store<T>::ld(&rd[i]), uu = Store<T>::ld(&ru[i]), du = in ? dl * uu : 0.0f;
                float y = 0.0f;
                auto step = [&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    const float dlk = quad_lane<k>(dl), duk = quad_lane<k>(du);
                    const v4f bv = *reinterpret_cast<const v4f *>(&Bs[4 * q + k][4 * g]);
#pragma unroll
                    for (int j = 0; j < 4; j++) h[j] = fmaf(fast_exp2(dlk * a2[j]), h[j], duk * bv[j]);
                    if constexpr (OUT) {
                        const v4f cv = *reinterpret_cast<const v4f *>(&Cs[4 * q + k][4 * g]);
                        float acc = h[0] * cv[0];
                        acc = fmaf(h[1], cv[1], acc);
                        acc = fmaf(h[2], cv[2], acc);
                        acc = quad_sum(fmaf(h[3], cv[3], acc));
                        y = g == k ? acc : y;
                    }
                };
                step(std::integral_constant<int, 0>());
                step(std::integral_constant<int, 1>());
                step(std::integral_constant<int, 2>());
                step(std::integral_constant<int, 3>());
                if constexpr (OUT) {
                    y = fmaf(Dd, uu, y);
                    if (GATE == 1) y *= Store<T>::ld(&rg[i]);
                    if (GATE == 2) y *= silu(Store<T>::ld(&rg[i]));
                    if (in && live) Store<T>::st((T *)a.y + (row0 + s) * di + d, y);
                } else {
                    sd += dl;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NB; i++) { rd[i] = nd[i]; ru[i] = nu[i]; if (GATE) rg[i] = ng[i]; }
    }
    if (!live) return;
    if constexpr (OUT) {
        if (c == a.nchunk - 1) {
#pragma unroll
            for (int j = 0; j < 4; j++) hp[j] = h[j];
        }
    } else {
        const int64_t sbase = (int64_t)b * (a.nchunk - 1) + c;
        sd = quad_sum(sd);
#pragma unroll
        for (int j = 0; j < 4; j++) a.S[sbase * 16 * di + own + (int64_t)j * di] = h[j];
        if (g == 0) a.sumd[sbase * di + d] = sd;
    }
}

template <typename T> int launch_quad_t(hipStream_t st, int gate_mode, const ScanQuadArgs &a) {
    const unsigned per = (unsigned)(a.tiles * a.batch);
    if (a.nchunk > 1) {
        hipLaunchKernelGGL((scan_quad_kernel<T, 0, false>), dim3(per * (unsigned)(a.nchunk - 1)), dim3(256), 0, st, a);
        const int rc = check_launch("scan_quad_kernel (states)");
        if (rc) return rc;
    }
    const dim3 grid(per * (unsigned)(a.nchunk - a.first));
    if constexpr (sizeof(T) == 2) {
        if (a.dt_w) {
            if (gate_mode != 2) return fail(MRS_E_SHAPE, "scan with dt_proj: gate mode %d", gate_mode);
            hipLaunchKernelGGL((scan_quad_kernel<T, 2, true, true>), grid, dim3(256), 0, st, a);
            return check_launch("scan_quad_kernel (dt_proj)");
        }
    }
    if (gate_mode == 0) hipLaunchKernelGGL((scan_quad_kernel<T, 0, true>), grid, dim3(256), 0, st, a);
    else if (gate_mode == 1) hipLaunchKernelGGL((scan_quad_kernel<T, 1, true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((scan_quad_kernel<T, 2, true>), grid, dim3(256), 0, st, a);
    return check_launch("scan_quad_kernel");
}

}  // namespace

bool scan_quad_dt_ok(int dtype, int T, int dr, int64_t bc_stride, const void *dt_in, const void *dt_w) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && T >= 1 && T <= kQuadDtLen && dr >= 8 && dr % 8 == 0 && bc_stride % 8 == 0 && bc_stride >= dr && dt_w && aligned(dt_in, 16) &&
           aligned(dt_w, 16);
}

int launch_scan_quad(hipStream_t st, int dtype, int gate_mode, const ScanQuadArgs &a) {
    if (a.dt_w && (!scan_quad_dt_ok(dtype, a.Tlen, a.dr, a.bc_stride, a.dt_in, a.dt_w) || a.nchunk != 1 || !a.dt_b))
        return fail(MRS_E_SHAPE, "scan with dt_proj: %d steps in %d chunks, dt_rank %d", a.Tlen, a.nchunk, a.dr);
    if (a.len < 1 || a.len > kQuadLen || a.nchunk < 1 || (int64_t)a.nchunk * a.len < a.Tlen || (int64_t)(a.nchunk - 1) * a.len >= a.Tlen || a.tiles * 64 < a.di || a.first < 0 || a.first >= a.nchunk)
        return fail(MRS_E_SHAPE, "scan: %d chunks of %d for %d steps", a.nchunk, a.len, a.Tlen);
    MRS_DISPATCH_DTYPE(dtype, T_, return launch_quad_t<T_>(st, gate_mode, a));
    return MRS_OK;
}

}  // namespace mrs
