// Projections of a prefill of some hundred rows: C[M,N] = A[M,K] . Wt[N,K]^T, 16-bit operands, f32 accumulate on the matrix cores.
//
// The reference sends these to the vendor GEMM (src/mamba_ssm/gpu/blas.rs:1138-1163), and so does this library for larger ones.
// Here the product is a few microseconds of work, and a library call costs the host more than that: a prompt of 64 to 500 rows took
// the same time, the time of its launches.  The kernel:
//   * tiles of 64 x 64, four waves of a quarter each;
//   * both operands go from memory straight to LDS, three 64-wide k-steps ahead of their use, in four buffers with one barrier
//     per k-step.  A row of a k-step is 128 bytes, eight 16-byte pieces; piece p of row r lies at place p ^ (r % 8), so that the
//     rows a matrix operand takes the same piece of spread over the banks (the lanes fetch permuted pieces of the same line:
//     the copy itself writes in lane order);
//   * workgroups are numbered so that the units of one die (block index modulo 8) share column tiles: each die's L2 then takes in an
//     eighth of the weight instead of all of it;
//   * K may be cut into slices over the second grid dimension, which leave f32 products side by side.
// It is bound by what a compute unit takes in (about 34 bytes a clock).  In a bf16 prefill, vendor / this: 64 x 3072 x 768 7.6 / 6.1 us, 64 x 768 x 1536
// 7.8 / 8.5, 777 x 4096 x 1024 14.5 / 16.2, 777 x 1024 x 2048 12.9 / 11.1, 1500 x 768 x 1536 13.8 / 11.0, 300 x 2560 x 5120 27.2 / 26.0.  Also measured: more
// buffers (6, 8: fewer workgroups per unit, 24 us at 777 x 4096 x 1024), tiles of 128 x 128 (15.8 there, 23 at 777 x 1024 x 2048) and
// 64 x 128 (18.3 / 14.7), and the operands of the next k-step read from LDS under the products (no change).
#include "common.hpp"
#include "mfma_tiles.hpp"
#include "size_rules.hpp"
#include <algorithm>

namespace mrs {
namespace {

constexpr int kMidThreads = 256, kTile = kMidTile, kStepK = kMidStepK, kStages = 4;

template <typename T, typename TO>
__global__ __launch_bounds__(kMidThreads) void gemm_mid_kernel(TO *__restrict__ C, int64_t ldc, const T *__restrict__ A, int64_t lda, const T *__restrict__ Wt,
                                                               int M, int N, int K, int mtiles, int per) {
    constexpr int MT = kTile / 32, NT = kTile / 32;             // 16 x 16 tiles of a wave
    constexpr int kRows = 2 * kTile, kStage = kRows * 2 * kStepK;  // bytes of a k-step: A's rows, then Wt's
    constexpr int kLoads = kRows / 8 / 4;                      // 1 KB requests of a wave per k-step
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int total = gridDim.x, xcd = blockIdx.x & 7, each = total >> 3, rest = total & 7;
    const int p = xcd * each + min(xcd, rest) + (blockIdx.x >> 3);
    const int m0 = p % mtiles * kTile, n0 = p / mtiles * kTile, ks0 = blockIdx.y * per, nk = min(K / kStepK - ks0, per);   // this slice's k-steps
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;

    // request q of a wave: rows 8 (w + 4 q) .. + 7 of the stage, lane l row l / 8 and place l % 8; rows past the end repeat the last
    unsigned voff[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; q++) {
        const int r = 8 * (w + 4 * q) + (l >> 3), piece = (l & 7) ^ (l >> 3);
        const bool is_a = 8 * (w + 4 * q) < kTile;   // (the same for the wave)
        const unsigned row = is_a ? (unsigned)min(m0 + r, M - 1) * (unsigned)lda : (unsigned)min(n0 + r - kTile, N - 1) * (unsigned)K;
        voff[q] = (row + 8u * (unsigned)piece) * 2u + (unsigned)ks0 * (2u * kStepK);
    }
    auto request = [&](int kt) {
        const unsigned buf = lds0 + (unsigned)(kt % kStages) * kStage;
#pragma unroll
        for (int q = 0; q < kLoads; q++) {
            const T *base = 8 * (w + 4 * q) < kTile ? A : Wt;
            dma_kb(__builtin_amdgcn_readfirstlane(buf + (unsigned)(w + 4 * q) * 1024u), base, voff[q] + (unsigned)kt * (2u * kStepK));
        }
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; s++)
        if (s < nk) request(s);

    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
    const int wm = (w & 1) * (kTile / 2), wn = (w >> 1) * (kTile / 2), lr = l & 15, lg = l >> 4;
    for (int kt = 0; kt < nk; kt++) {
        // this k-step's requests of this wave are in (the younger ones may be under way), then everybody's; everybody is also done
        // with the k-step before, whose buffer the next request takes
        if (kt + kStages - 2 < nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads * (kStages - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        if (kt + kStages - 1 < nk) request(kt + kStages - 1);
        const char *sa = smem + (kt % kStages) * kStage, *sw = sa + kTile * 2 * kStepK;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            uint4 af[MT], wf[NT];
            const int place = 16 * ((4 * kk + lg) ^ (lr & 7));
#pragma unroll
            for (int i = 0; i < MT; i++) af[i] = *reinterpret_cast<const uint4 *>(sa + (wm + 16 * i + lr) * (2 * kStepK) + place);
#pragma unroll
            for (int j = 0; j < NT; j++) wf[j] = *reinterpret_cast<const uint4 *>(sw + (wn + 16 * j + lr) * (2 * kStepK) + place);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) acc[i][j] = Mma32<T>::mma(wf[j], af[i], acc[i][j]);   // (transposed: a lane holds four columns of a row)
        }
    }
    C += (int64_t)blockIdx.y * M * ldc;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int row = m0 + wm + 16 * i + lr;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int col = n0 + wn + 16 * j + 4 * lg;
            if (row < M && col < N) {
                struct alignas(4 * sizeof(TO)) T4 { TO v[4]; } o;
#pragma unroll
                for (int e = 0; e < 4; e++) Store<TO>::st(&o.v[e], acc[i][j][e]);
                *reinterpret_cast<T4 *>(C + (int64_t)row * ldc + col) = o;
            }
        }
    }
}

template <typename T, typename TO>
int launch_mid(hipStream_t st, void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int M, int N, int K, int slices = 1) {
    constexpr size_t lds = (size_t)kStages * 2 * kTile * 2 * kStepK;
    static const hipError_t attr = hipFuncSetAttribute((const void *)gemm_mid_kernel<T, TO>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "mid gemm: LDS size: %s", hipGetErrorString(attr));
    const int mt = (M + kTile - 1) / kTile, nt = (N + kTile - 1) / kTile;
    const int steps = K / kStepK, per = (steps + slices - 1) / slices;
    hipLaunchKernelGGL((gemm_mid_kernel<T, TO>), dim3((unsigned)(mt * nt), (unsigned)((steps + per - 1) / per)), dim3(kMidThreads), lds, st, (TO *)C, ldc, (const T *)A, lda,
                       (const T *)Wt, M, N, K, mt, per);
    return check_launch("gemm_mid_kernel");
}

}  // namespace

// Where the own kernel is ahead in a prefill: K no longer than a tile walks in about 9 us (the vendor kernels cut a longer one up), and either one
// round of tiles over the compute units or little enough work that the vendor kernels' larger tiles do not show.  A layer of a bf16
// prefill, vendor / this: 64 rows at d_model 768 72.8 / 59.5 us, 200 rows 70.9 / 59.9, 500 rows 77.7 / 68.3, 300 rows at 1024 76.8 / 67.2; from
// there out_proj alone, 1500 rows at 768 94.0 / 90.7, 2048 rows 113.9 / 111.7.
bool mid_gemm_wins(int64_t M, int N, int K) {
    const int64_t tiles = (M + kTile - 1) / kTile * ((N + kTile - 1) / kTile), steps = K / kStepK;
    return steps <= 40 && (tiles <= 256 || tiles * steps <= 10000);
}

bool mid_gemm_ok(int dtype, int out_f32, const void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && M >= 1 && N >= 4 && N % 4 == 0 && K >= kStepK && K % kStepK == 0 && lda % 8 == 0 && lda >= K && ldc % 4 == 0 &&
           ldc >= N && C && aligned(C, out_f32 ? 16 : 8) && in_pieces(A) && in_pieces(Wt) && M * lda < (int64_t)1 << 30 && (int64_t)N * K < (int64_t)1 << 30;
}

int launch_mid_gemm(hipStream_t st, int dtype, int out_f32, void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K) {
    if (!mid_gemm_ok(dtype, out_f32, C, ldc, A, lda, Wt, M, N, K))
        return fail(MRS_E_SHAPE, "mid gemm: 16-bit storage, N %% 4 == 0, K %% 64 == 0, 16-byte aligned operands (M=%lld N=%d K=%d)", (long long)M, N, K);
    if (dtype == MRS_BF16)
        return out_f32 ? launch_mid<bf16_t, float>(st, C, ldc, A, lda, Wt, (int)M, N, K) : launch_mid<bf16_t, bf16_t>(st, C, ldc, A, lda, Wt, (int)M, N, K);
    return out_f32 ? launch_mid<f16_t, float>(st, C, ldc, A, lda, Wt, (int)M, N, K) : launch_mid<f16_t, f16_t>(st, C, ldc, A, lda, Wt, (int)M, N, K);
}

int launch_mid_gemm_parts(hipStream_t st, int dtype, float *parts, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K, int slices) {
    if (!mid_gemm_ok(dtype, 1, parts, N, A, lda, Wt, M, N, K) || slices < 1 || slices > K / kStepK) return fail(MRS_E_SHAPE, "mid gemm: %d slices of M=%lld N=%d K=%d", slices, (long long)M, N, K);
    return dtype == MRS_BF16 ? launch_mid<bf16_t, float>(st, parts, N, A, lda, Wt, (int)M, N, K, slices) : launch_mid<f16_t, float>(st, parts, N, A, lda, Wt, (int)M, N, K, slices);
}

}  // namespace mrs
