// Building blocks of the single-launch backbone steps for small f32 models (tiny_step.hip, tiny_m3_step.hip): a workgroup
// walks one batch row through the whole network, its products are matrix-vector sweeps over weights that sit in L2.
#pragma once
#include "common.hpp"
#include "host_io.hpp"

namespace mrs {
namespace {

constexpr int kTinyThreads = 512;    // 8 waves: one float4 of SSM state per lane and pass at d_inner 256, d_state 16
constexpr int kTinyPre = 2;          // passes of the scan step whose state is requested at the top of the layer
constexpr int kTinySlices = 16;      // most k slices per product (their partial sums are added serially)
constexpr int kTinyPart = 2048;      // floats of k-slice partial sums: (N / 4 column quads) x (k slices) <= 512 threads x 4

// Every array carved out of the workgroup's LDS starts on a 16-byte boundary: some of them (the partial sums, K and Q of the
// Mamba-3 step) are read and written as float4, and an array in front of them whose length is not a multiple of four
// floats (an input row wider than d_model, an odd d_inner) would otherwise shift them off it.
__host__ __device__ constexpr int rup4(int n) { return (n + 3) & ~3; }

// out[n] = bias[n] + sum_k x[k] W[k][n] for n < N; W row-major [K][N] in global memory, x and out in LDS, N % 4 == 0 and
// N <= 2048.  A thread owns four consecutive columns over one slice of K (16-byte weight loads, consecutive lanes on
// consecutive quads, sixteen rows requested before the first multiply-add); the slices' partial sums meet in LDS and are
// added in slice order.
__device__ __forceinline__ void gemv_rows(const float *__restrict__ W, int K, int N, const float *x, float *out, float *part,
                                          const float *__restrict__ bias) {
    const int tid = threadIdx.x;
    const int nq = N >> 2;
    const int ks_n = min(kTinyThreads / nq, kTinySlices);   // k slices (>= 1)
    const int kper = (K + ks_n - 1) / ks_n;
    const int q = tid % nq, ks = tid / nq;
    if (ks < ks_n) {
        const int k0 = ks * kper, k1 = min(K, k0 + kper);
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        const float *wp = W + 4 * q;
        for (int kb = k0; kb < k1; kb += 16) {
            float4 w[16];
#pragma unroll
            for (int j = 0; j < 16; j++) w[j] = *reinterpret_cast<const float4 *>(wp + (int64_t)min(kb + j, k1 - 1) * N);   // rows past the slice re-read its last one
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const float xv = kb + j < k1 ? x[kb + j] : 0.0f;
                acc.x = fmaf(xv, w[j].x, acc.x); acc.y = fmaf(xv, w[j].y, acc.y); acc.z = fmaf(xv, w[j].z, acc.z); acc.w = fmaf(xv, w[j].w, acc.w);
            }
        }
        *reinterpret_cast<float4 *>(&part[ks * N + 4 * q]) = acc;
    }
    __syncthreads();
    for (int n = tid; n < N; n += kTinyThreads) {
        float s = bias ? bias[n] : 0.0f;
        for (int j = 0; j < ks_n; j++) s += part[j * N + n];
        out[n] = s;
    }
    __syncthreads();
}

// sum of v over the workgroup (every thread gets it); red: one float of LDS per wave
__device__ __forceinline__ float block_sum(float v, float *red) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < kTinyThreads / 64; i++) s += red[i];
    __syncthreads();
    return s;
}

__device__ __forceinline__ float rms_inv(float ss, int dm, float eps) {
    float rms = sqrtf(ss / (float)dm + eps);
    if (!isfinite(rms) || rms < 1e-20f) rms = 1.0f;   // the reference's finite guard (kernels/norms.cu:58-61)
    return 1.0f / rms;
}

// Rounds of sixteen weight rows a lane goes through in a [K][N] sweep (each is a dependent trip to L2); the routes built
// on these sweeps take a model only while every sweep stays within kTinyMaxRounds -- beyond that the kernel chains with
// their full-width GEMMs are faster (d_model 256 x d_inner 512: 16 rounds for in_proj, 264 us against 102 us per step).
constexpr int kTinyMaxRounds = 3;
inline int sweep_rounds(int K, int N) {
    if (N % 4 != 0 || N < 4 || N / 4 > kTinyThreads || K < 1) return 1 << 20;
    const int ks_n = kTinyThreads / (N / 4) < kTinySlices ? kTinyThreads / (N / 4) : kTinySlices;
    const int kper = (K + ks_n - 1) / ks_n;
    return (kper + 15) / 16;
}

// ---- the streamed form: a layer's weights are on their way before the layer begins ----

// A [K][N] product (rows LD floats apart) whose every thread owns four columns, 4 q .. 4 q + 3, of one of n slices of `rows` rows.
template <int K, int N, int LD = N> struct Sweep {
    static constexpr int most = kTinyThreads / (N / 4) < 32 ? kTinyThreads / (N / 4) : 32;
    static constexpr int rows = ((K + most - 1) / most + 3) / 4 * 4, n = K / rows;
    static_assert(N % 4 == 0 && LD % 4 == 0 && K % rows == 0 && n * N <= kTinyPart, "whole slices");
    int q, j;       // (a thread behind the last slice works on slice 0 and its sum goes nowhere)
    bool on;
    unsigned off;   // its first row's bytes
    __device__ explicit Sweep(int tid) : q(tid % (N / 4)), j(tid / (N / 4)), on(j < n) {
        if (!on) j = 0;
        off = 4u * (j * rows * LD + 4 * q);
        asm volatile("" : "+v"(off));   // (kept as 32 bits beside a scalar base)
    }
};

template <int CTRL> __device__ __forceinline__ float dpp_add(float v) {
    return v + __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float quad_sum(float v) { return dpp_add<0x4e>(dpp_add<0xb1>(v)); }   // quad_perm [1,0,3,2], [2,3,0,1]
__device__ __forceinline__ float oct_sum(float v) { return dpp_add<0x141>(quad_sum(v)); }          // row_half_mirror
// sum over the wave, the same in every lane
__device__ __forceinline__ float wave_sum(float v) {
    v = dpp_add<0x140>(oct_sum(v));
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1 and 3
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2 and 3
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), 63));
}

// Memory operations stay on their side of this line.
__device__ __forceinline__ void pin() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// ... and so do the sums so far: without this the compiler moves them to their one use, behind the requests into the registers they read.
__device__ __forceinline__ void pin(float4 &v) {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)::"memory");
    __builtin_amdgcn_sched_barrier(0);
}
// A table entry by scalar loads, and reads through the pointers it holds: they come out of memory, so the compiler has to be told
// that they point to global memory (a flat load would count as an LDS operation too, and every LDS wait would wait for it).
template <typename T> __device__ __forceinline__ T table_entry(const T *p) {
    constexpr int n = sizeof(T) / 8;
    union { T t; uint64_t w[n]; } v = {};
    const auto *q = (const __attribute__((address_space(4))) uint64_t *)(uintptr_t)p;
#pragma unroll
    for (int i = 0; i < n; i++) v.w[i] = q[i];
    return v.t;
}
using gbytes = const __attribute__((address_space(1))) char *;
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ gbytes global(const void *p) { return (gbytes)(uintptr_t)p; }
__device__ __forceinline__ float ld1(gbytes p, unsigned off) { return *(const __attribute__((address_space(1))) float *)(p + off); }
__device__ __forceinline__ float4 ld4(gbytes p, unsigned off) {
    const f32x4 v = *(const __attribute__((address_space(1))) f32x4 *)(p + off);
    return make_float4(v.x, v.y, v.z, v.w);
}
// A byte offset the compiler keeps as 32 bits beside a scalar base and computes where it is used.
__device__ __forceinline__ unsigned own(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ void fma4(float4 &acc, float x, float4 w) {
    acc.x = fmaf(x, w.x, acc.x); acc.y = fmaf(x, w.y, acc.y); acc.z = fmaf(x, w.z, acc.z); acc.w = fmaf(x, w.w, acc.w);
}
// column c of a product: the partial sums j0, j0 + STEP, .. of n; `meanwhile` runs while they come
template <int N, int NS, int STEP, typename F> __device__ __forceinline__ float part_sum(const float *part, int c, int j0, const F &meanwhile) {
    float v[(NS + STEP - 1) / STEP], s = 0.0f;
#pragma unroll
    for (int j = 0; j < NS; j += STEP) v[j / STEP] = part[(j0 + j) * N + c];
    meanwhile();
#pragma unroll
    for (int j = 0; j < NS; j += STEP) s += v[j / STEP];
    return s;
}

__device__ __forceinline__ unsigned lds_address(const float *p) { return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const float *)p; }

constexpr int kStreamInput = 512;   // widest input row

// Input row -> residual stream `res` (identity or projection + bias) and its product with the first layer's norm weight, `xin`
// (kStreamInput floats, which first hold the row).  The first eight rows of a slice of the projection are asked for ahead of `ahead`'s requests.
template <int DM, typename Args, typename F>
__device__ __forceinline__ void stream_input(const Args &a, const float *norm_w, float *xin, float *res, float *part, const F &ahead) {
    constexpr int nq = DM / 4, sn = kTinyThreads / nq < kTinySlices ? kTinyThreads / nq : kTinySlices;
    const int tid = threadIdx.x, b = blockIdx.x, co = min(tid >> 2, DM - 1);
    const int kper = (a.input_dim + sn - 1) / sn, q = tid % nq, s = tid / nq;
    const int k0 = min(s * kper, a.input_dim), k1 = min(a.input_dim, k0 + kper);
    float4 w[8];
    const float v0 = a.input[(int64_t)b * a.input_dim + min(tid, a.input_dim - 1)];
    auto ask = [&](int kb) {
#pragma unroll
        for (int j = 0; j < 8; j++) w[j] = ld4(global(a.in_w), 4u * (min(kb + j, a.input_dim - 1) * DM + 4 * q));
    };
    if (a.in_w) ask(k0);
    const float nw = ld1(global(norm_w), 4u * co), bias = a.in_w ? a.in_b[co] : 0.0f;
    pin();
    ahead();
    pin();
    if (tid < a.input_dim) {
        xin[tid] = v0;
        if (a.input_copy) host_store(a.input_copy + (int64_t)b * a.input_dim + tid, v0);   // (the input came straight from host memory)
    }
    lds_barrier();
    float r;
    if (a.in_w) {
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int kb = k0; kb < k1; kb += 8) {
            if (kb != k0) ask(kb);
#pragma unroll
            for (int j = 0; j < 8; j++) fma4(acc, kb + j < k1 ? xin[kb + j] : 0.0f, w[j]);
        }
        if (s < sn) *reinterpret_cast<float4 *>(&part[s * DM + 4 * q]) = acc;
        lds_barrier();
        r = bias + part_sum<DM, sn, 1>(part, co, 0, [] {});
    } else {
        r = xin[co];
        lds_barrier();   // xin is read before it is written again
    }
    if ((tid & 3) == 0 && tid < 4 * DM) { res[co] = r; xin[co] = r * nw; }
    lds_barrier();
}
// this lane's part of the residual stream's sum of squares (every wave takes all of it)
template <int DM> __device__ __forceinline__ float lane_squares(const float *res) {
    const int lane = threadIdx.x & 63;
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < DM; i += 64) ss = fmaf(res[i + lane], res[i + lane], ss);
    return ss;
}
// This thread's sum of out_proj's sweep: its rows are at wo[row][thread].  feed(0), feed(1) and feed(2) run while the LDS reads are under way.
template <typename S, typename F> __device__ __forceinline__ float4 stream_out_sweep(const S &op, const float *y, const float *wo, const F &feed) {
    constexpr int turns = S::rows / 4;
    const int tid = threadIdx.x;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f), x[2], w[2][4];
    auto take = [&](int t) {
        x[t % 2] = *reinterpret_cast<const float4 *>(&y[op.j * S::rows + 4 * t]);
#pragma unroll
        for (int k = 0; k < 4; k++) w[t % 2][k] = reinterpret_cast<const float4 *>(wo)[(4 * t + k) * kTinyThreads + tid];
    };
    take(0);
#pragma unroll
    for (int t = 0; t < turns; t++) {
        if (t + 1 < turns) take(t + 1);
        if (t < 3) feed(t);
        fma4(acc, x[t % 2].x, w[t % 2][0]); fma4(acc, x[t % 2].y, w[t % 2][1]); fma4(acc, x[t % 2].z, w[t % 2][2]); fma4(acc, x[t % 2].w, w[t % 2][3]);
    }
#pragma unroll
    for (int t = turns; t < 3; t++) feed(t);
    pin(acc);
    return acc;
}
// The final norm: xin holds the residual stream times norm_f.
template <int DM, typename Args> __device__ __forceinline__ void stream_output(const Args &a, bool now, const float *xin, const float *res) {
    const int tid = threadIdx.x, b = blockIdx.x;
    const float inv = rms_inv(wave_sum(lane_squares<DM>(res)), DM, a.eps);
    if (tid < DM) {
        const float v = xin[tid] * inv;
        leave(now, a.temporal + (int64_t)b * DM + tid, v);
        if (now) host_store(a.host.out + (int64_t)b * DM + tid, v);
    }
    if (now) host_row_done(a.host, b);
}

}  // namespace
}  // namespace mrs
