// Logits of a language model: logits[M][V] = hidden[M][K] . table[V][K]^T, 16-bit operands, f32 accumulate on the matrix cores, and each tile's part of the greedy pick.
//
// The reference sends the product to the vendor GEMM (src/mamba_ssm/gpu/blas.rs:709-740) and picks on the host.  It is one pass over the table, so the kernel is that stream:
//   * the table lies in tiles (tile_weight, gemm_wide.hip): a wave owns sixteen columns and streams their contiguous kilobytes, eight ahead, into registers;
//   * a workgroup holds the hidden rows in LDS in the order of the matrix operand, 32 K bytes for sixteen rows; eight waves, two workgroups to a compute unit, where that leaves room
//     for two, else sixteen waves.  Up to 136 KB of them (64 rows of K 1024); past that the vendor kernel has it;
//   * the table is read past the caches where a step touches more than they hold (step_outgrows_cache).
// Bound by memory: 2.8b shape, 16 rows, 257 MB in 42.9 us = 6.0 TB/s (through the caches 55.7; the vendor kernel 58.4); 130m shape, 77 MB, 1 row 15.4 us (vendor 15.4; the gain there
// is in the layers, whose weights now stay in the cache: 205 -> 201 us a step), 64 rows 22.3 (25.5).  From the row-major table through LDS, 64 columns to a workgroup: 14.2, 27.2, 61.0.
// The pick as a launch over the workgroups' maxima is 4.0 us whatever the rows, over the logits 3.9 at one row and 5.9 at 64; storing the logits as whole lines through LDS changed nothing.
#include "common.hpp"
#include "mfma_tiles.hpp"

namespace mrs {
namespace {

constexpr size_t kHeadLds = 136 * 1024;   // hidden rows held by a workgroup, at most

__device__ __forceinline__ unsigned long long pick_key(float best, int bi) {
    const unsigned bits = __float_as_uint(best + 0.0f);   // (the two zeros are equal)
    return (unsigned long long)((bits & 0x80000000u) ? ~bits : (bits | 0x80000000u)) << 32 | (unsigned)bi;
}

typedef unsigned u4 __attribute__((ext_vector_type(4)));
template <bool STREAM> __device__ __forceinline__ uint4 load_table(const uint4 *p) {
    if constexpr (STREAM) return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u4 *>(p)));
    else return *p;
}

template <typename T, int MT, int WAVES, bool STREAM>
__global__ __launch_bounds__(64 * WAVES) void lm_head_kernel(float *__restrict__ C, int64_t ldc, const T *__restrict__ A, const T *__restrict__ Wp, int M, int N, int K, int vocab,
                                                             unsigned long long *__restrict__ keys) {
    extern __shared__ __attribute__((aligned(1024))) uint4 hid[];   // [k-step][row tile][lane]
    __shared__ unsigned long long best_s[WAVES][16 * MT];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lg = l >> 4;
    const int nks = K >> 5, ntiles = N >> 4, tile = blockIdx.x * WAVES + w;
    const uint4 *wp = reinterpret_cast<const uint4 *>(Wp) + (int64_t)min(tile, ntiles - 1) * nks * 64 + l;
    constexpr int R = 8;   // k-steps of the table ahead
    uint4 wr[R];
#pragma unroll
    for (int r = 0; r < R; r++) wr[r] = load_table<STREAM>(wp + min(r, nks - 1) * 64);
    __builtin_amdgcn_sched_barrier(0);
    for (int p0 = tid; p0 < nks * MT * 64; p0 += 4 * 64 * WAVES) {
        uint4 h[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int p = min(p0 + q * 64 * WAVES, nks * MT * 64 - 1), t = p >> 6, ks = t / MT, row = min(16 * (t % MT) + (p & 15), M - 1);
            h[q] = *reinterpret_cast<const uint4 *>(A + (int64_t)row * K + 32 * ks + 8 * ((p >> 4) & 3));
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (p0 + q * 64 * WAVES < nks * MT * 64) hid[p0 + q * 64 * WAVES] = h[q];
    }
    lds_barrier();
    // Sums of four k-steps, which are added up: one chain over K of 768 to 2560 is 1.5 to 3.1e-7 off the sum in 64 bits (of their norm), the vendor kernels' 0.8 to 1.4e-7 (to 2.0e-7 at 64 rows), these 0.7 to 1.2e-7.
    // (A sum joins the others behind the next one's second step, when the matrix cores are done with it.)
    v4f acc[2][MT], sum[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) sum[i] = acc[1][i] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int kb = 0; kb < nks; kb += R) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int h = r / 4 % 2;
            if (r % 4 == 0) {
#pragma unroll
                for (int i = 0; i < MT; i++) acc[h][i] = (v4f){0.f, 0.f, 0.f, 0.f};
            }
            if (kb + r < nks) {
#pragma unroll
                for (int i = 0; i < MT; i++) acc[h][i] = Mma32<T>::mma(wr[r], hid[((kb + r) * MT + i) * 64 + l], acc[h][i]);   // (a lane holds four columns of a row)
            }
            wr[r] = load_table<STREAM>(wp + min(kb + r + R, nks - 1) * 64);
            __builtin_amdgcn_sched_barrier(0);   // each refill right behind its use
            if (r % 4 == 1) {
#pragma unroll
                for (int i = 0; i < MT; i++) sum[i] += acc[1 - h][i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++) sum[i] += acc[1][i];
    const int col = 16 * tile + 4 * lg;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = 16 * i + lr;
        if (row < M && tile < ntiles) *reinterpret_cast<float4 *>(C + (int64_t)row * ldc + col) = make_float4(sum[i][0], sum[i][1], sum[i][2], sum[i][3]);
        if (!keys) continue;
        float best = -INFINITY;
        int bi = 0;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (col + e < vocab && sum[i][e] >= best) { best = sum[i][e]; bi = col + e; }   // ascending: >= keeps the last maximum
        if (best == -INFINITY) bi = vocab - 1;   // the last of its equals where the row has nothing above it (NaN is passed over)
        unsigned long long key = pick_key(best, bi);
        key = max(key, (unsigned long long)__shfl_xor((long long)key, 16, kWave));
        key = max(key, (unsigned long long)__shfl_xor((long long)key, 32, kWave));
        if (lg == 0) best_s[w][row] = key;
    }
    if (!keys) return;
    lds_barrier();
    for (int r = tid; r < M; r += 64 * WAVES) {
        unsigned long long key = best_s[0][r];
#pragma unroll
        for (int q = 1; q < WAVES; q++) key = max(key, best_s[q][r]);
        keys[(int64_t)r * gridDim.x + blockIdx.x] = key;
    }
}

// The largest of a row's keys: its index is the token.
__global__ __launch_bounds__(256) void pick_kernel(int *__restrict__ tokens, const unsigned long long *__restrict__ keys, int n) {
    __shared__ unsigned long long part[4];
    const unsigned long long *k = keys + (int64_t)blockIdx.x * n;
    unsigned long long key = 0;
    for (int i0 = threadIdx.x; i0 < n; i0 += 4 * 256) {   // four at a time are under way
        unsigned long long v[4];
#pragma unroll
        for (int h = 0; h < 4; h++) v[h] = k[min(i0 + 256 * h, n - 1)];
        key = max(key, max(max(v[0], v[1]), max(v[2], v[3])));
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) key = max(key, (unsigned long long)__shfl_xor((long long)key, m, kWave));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = key;
    __syncthreads();
    if (threadIdx.x == 0) tokens[blockIdx.x] = (int)(unsigned)max(max(part[0], part[1]), max(part[2], part[3]));
}

template <typename T, int MT, int WAVES, bool STREAM>
int launch_head(hipStream_t st, float *C, int64_t ldc, const void *A, const void *Wp, int M, int N, int K, int vocab, unsigned long long *keys) {
    static const hipError_t attr = hipFuncSetAttribute((const void *)lm_head_kernel<T, MT, WAVES, STREAM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kHeadLds);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "lm head: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((lm_head_kernel<T, MT, WAVES, STREAM>), dim3((unsigned)((N / 16 + WAVES - 1) / WAVES)), dim3(64 * WAVES), (size_t)MT * 32 * K, st, C, ldc, (const T *)A,
                       (const T *)Wp, M, N, K, vocab, keys);
    return check_launch("lm_head_kernel");
}
// Waves of a workgroup, a tile of columns each: two workgroups to a compute unit where the hidden rows leave room for that.
int head_waves(int M, int K) { return (size_t)((M + 15) / 16) * 32 * K <= 76 * 1024 ? 8 : 16; }

template <typename T>
int launch_head_t(hipStream_t st, float *C, int64_t ldc, const void *A, const void *Wp, int M, int N, int K, int vocab, unsigned long long *keys, bool stream) {
#define MRS_HEAD(MT_)                                                                                                                                             \
    if (head_waves(M, K) == 8) return stream ? launch_head<T, MT_, 8, true>(st, C, ldc, A, Wp, M, N, K, vocab, keys) : launch_head<T, MT_, 8, false>(st, C, ldc, A, Wp, M, N, K, vocab, keys); \
    return stream ? launch_head<T, MT_, 16, true>(st, C, ldc, A, Wp, M, N, K, vocab, keys) : launch_head<T, MT_, 16, false>(st, C, ldc, A, Wp, M, N, K, vocab, keys)
    switch ((M + 15) / 16) {
        case 1: MRS_HEAD(1);
        case 2: MRS_HEAD(2);
        case 3: MRS_HEAD(3);
        default: MRS_HEAD(4);
    }
#undef MRS_HEAD
}

}  // namespace

size_t lm_head_keys(int M, int N, int K) { return (size_t)M * ((N / 16 + head_waves(M, K) - 1) / head_waves(M, K)); }

bool lm_head_ok(int dtype, int M, int N, int K) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && M >= 1 && M <= 64 && N >= 16 && N % 16 == 0 && K >= 32 && K % 32 == 0 && (size_t)((M + 15) / 16) * 32 * K <= kHeadLds;
}

int launch_lm_head(hipStream_t st, int dtype, float *C, int64_t ldc, const void *A, const void *Wp, int M, int N, int K, int vocab, unsigned long long *keys, bool stream) {
    if (!lm_head_ok(dtype, M, N, K) || vocab < 1 || vocab > N || ldc < N || ldc % 4 != 0 || !aligned(C, 16) || !aligned(A, 16) || !aligned(Wp, 16))
        return fail(MRS_E_SHAPE, "lm head: M=%d N=%d K=%d vocab=%d", M, N, K, vocab);
    if (dtype == MRS_BF16) return launch_head_t<bf16_t>(st, C, ldc, A, Wp, M, N, K, vocab, keys, stream);
    return launch_head_t<f16_t>(st, C, ldc, A, Wp, M, N, K, vocab, keys, stream);
}

int launch_pick(hipStream_t st, int *tokens, const unsigned long long *keys, int M, int N, int K) {
    hipLaunchKernelGGL(pick_kernel, dim3((unsigned)M), dim3(256), 0, st, tokens, keys, (int)(lm_head_keys(M, N, K) / M));
    return check_launch("pick_kernel");
}

}  // namespace mrs
