// Projections of a long prefill: C[M,N] = A[M,K] . Wt[N,K]^T, 16-bit operands, f32 accumulate on the matrix cores.
//
// The reference sends these to the vendor GEMM (src/mamba_ssm/gpu/blas.rs:1138-1163), and so does this library where that one's tiles come out
// even.  Its kernels take 256 x 256 tiles, and where those leave the last round over the 256 compute units partly empty the product
// pays for the whole round and more (16384 x 2560 x 5120, 640 tiles: 425-460 us, and 16384 x 10240 x 2560 with four times the tiles
// 565).  Here a tile is 256 rows and 192 or 320 columns, whichever needs less time in whole rounds.  The kernel:
//   * eight waves, four down and two across, each with a quarter of the rows of both halves of the tile and half of the columns;
//   * both operands go from memory straight to LDS, one 64-wide k-step in use and the next under way.  A row of a k-step is 128 bytes,
//     eight 16-byte pieces; piece p of row r lies at place p ^ (r / 2 % 8), so that sixteen rows' pieces cover all banks once
//     (the lanes fetch permuted pieces of the same line: the copy itself writes in lane order);
//   * a k-step is four quarters of the tile.  The waves are two groups, one barrier apart: while one group's four waves, one per SIMD, multiply a
//     quarter, the other's read the operands of theirs from LDS and request what the step after next needs in the places both have read.
// Over a long K it is bound by the clock that the card holds under it: 16384 x 2560 x 5120 in a prefill runs at 1.72 to 1.85 GHz, where the kernels beside it have 2.0 to 2.3, with the matrix cores
// busy 74 % of the cycles at least.  Over a short one the ends of the rounds count: 16384 x 3288 x 768, 2.75 rounds of twelve k-steps, 41 to 46 %.  Alone, bf16, the
// library's (torch's copy) / this: 16384 x 2560 x 5120 425 / 284 us, 8000 x 2560 x 5120 161 / 142, 4000 x 10240 x 2560 242 / 149, 2000 x 10240 x 2560 102 / 76,
// 6000 x 3072 x 768 48 / 28, 12000 x 3072 x 768 79 / 54; but 16384 x 10240 x 2560 561 / 598, 16384 x 3072 x 768 67 / 70, 8192 cubed 694 / 738.
// Also measured, at 16384 x 3072 x 768 and 8192 cubed with tiles of 256 columns (this: 71, 738): two halves per k-step instead of four quarters 71, 755; the halves of A in turn, which evens
// out the LDS reads 72, 765; one workgroup per unit that walks its tiles with the next one's requests under the stores 69, 743; 32 x 32
// matrix instructions 96, 867.  With the residual add, the next norm's operand and the row's sum of squares in out_proj's epilogue a layer of a
// prefill gained 2 us of 330 (all workgroups come to their epilogues together, and nothing runs under that traffic), so the products stay plain.
#include "common.hpp"
#include "mfma_tiles.hpp"
#include <stdlib.h>

namespace mrs {
namespace {

constexpr int kBigThreads = 512, kTileM = 256, kStepK = 64;

#define MRS_BAR() asm volatile("s_barrier" ::: "memory")
#define MRS_LGKM0() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
#define MRS_PIN() __builtin_amdgcn_sched_barrier(0)

// rows 1 and 3 (of sixteen lanes) of a trade places with rows 0 and 2 of b
__device__ __forceinline__ void swap16(unsigned &a, unsigned &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
template <typename T> __device__ __forceinline__ unsigned pack2(float a, float b) {
    struct alignas(4) T2 { T v[2]; } o;
    Store<T>::st(&o.v[0], a); Store<T>::st(&o.v[1], b);
    return __builtin_bit_cast(unsigned, o);
}

// SPLIT: columns from n1 on (a multiple of 16) leave as f32 in C2, n1 columns to the left
template <typename T, int NB, bool SPLIT>
__global__ __launch_bounds__(kBigThreads, 2) void gemm_big_kernel(T *__restrict__ C, int64_t ldc, const T *__restrict__ A, int64_t lda, const T *__restrict__ Wt,
                                                                  int M, int N, int K, int mtiles, int ntiles, BigSplit split) {
    constexpr int BN = 64 * NB, kA = kTileM * 128, kStage = kA + BN * 128;   // bytes of a k-step: A's rows, then Wt's
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int nk = K / kStepK;
    // the units of one die (block index modulo 8) share tiles of eight row blocks
    const int total = gridDim.x, xcd = blockIdx.x & 7;
    const int p = xcd * (total >> 3) + min(xcd, total & 7) + (blockIdx.x >> 3);
    const int grp = p / (8 * ntiles), q0 = p - grp * 8 * ntiles, gm = min(8, mtiles - grp * 8);
    const int m0 = (grp * 8 + q0 % gm) * kTileM, n0 = q0 / gm * BN;
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;

    // request q of a wave: eight rows of 128 bytes, lane l row l / 8 and place l % 8; rows past the end repeat the last
    const int lrow = l >> 3;
    unsigned va[4], vb[NB];
#pragma unroll
    for (int i = 0; i < 4; i++) {   // i = 2 h + q: half h of A's rows
        const int r = (i >> 1) * 128 + 8 * (2 * w + (i & 1)) + lrow;
        va[i] = ((unsigned)min(r, M - 1 - m0) * (unsigned)lda + 8u * (unsigned)((l & 7) ^ ((r >> 1) & 7))) * 2u;
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int r = 8 * (NB * w + i) + lrow;
        vb[i] = ((unsigned)min(r, N - 1 - n0) * (unsigned)K + 8u * (unsigned)((l & 7) ^ ((r >> 1) & 7))) * 2u;
    }
    const T *Ab = A + (int64_t)m0 * lda, *Wb = Wt + (int64_t)n0 * K;
    auto req_a = [&](int kt, int h) {
        const unsigned buf = lds0 + (unsigned)(kt & 1) * kStage + (unsigned)h * 16384u;
#pragma unroll
        for (int q = 0; q < 2; q++) dma_kb(__builtin_amdgcn_readfirstlane(buf + (unsigned)(2 * w + q) * 1024u), Ab + kt * kStepK, va[2 * h + q]);
    };
    auto req_b = [&](int kt) {
        const unsigned buf = lds0 + (unsigned)(kt & 1) * kStage + kA;
#pragma unroll
        for (int q = 0; q < NB; q++) dma_kb(__builtin_amdgcn_readfirstlane(buf + (unsigned)(NB * w + q) * 1024u), Wb + kt * kStepK, vb[q]);
    };
    req_a(0, 0); req_a(0, 1); req_b(0);
    req_a(1, 0); req_a(1, 1); req_b(1);   // (K is at least two steps)

    const int lr = l & 15, lg = l >> 4, wm = w >> 1, wn = w & 1;   // four waves down, two across
    v4f acc[2][2][2][NB];   // [half of the rows][16 rows][half of the columns][16 columns]
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[a][i][b][j] = (v4f){0.f, 0.f, 0.f, 0.f};
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 + NB) : "memory");
    MRS_BAR();
    if (w >= 4) MRS_BAR();   // from here on the second four waves are one barrier behind the first

    uint4 af[2][2][2], wf[NB][2];
    const int pl0 = 16 * (lg ^ ((lr >> 1) & 7)), pl1 = pl0 ^ 64;
    for (int kt = 0; kt < nk; kt++) {
        const char *sa = smem + (kt & 1) * kStage + (wm * 32 + lr) * 128, *sb = smem + (kt & 1) * kStage + kA + (wn * 16 * NB + lr) * 128;
        auto read_a = [&](int h) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                af[h][i][0] = *reinterpret_cast<const uint4 *>(sa + h * 16384 + i * 2048 + pl0);
                af[h][i][1] = *reinterpret_cast<const uint4 *>(sa + h * 16384 + i * 2048 + pl1);
            }
        };
        auto read_b = [&](int h) {
#pragma unroll
            for (int j = 0; j < NB; j++) {
                wf[j][0] = *reinterpret_cast<const uint4 *>(sb + h * (32 * NB * 128) + j * 2048 + pl0);
                wf[j][1] = *reinterpret_cast<const uint4 *>(sb + h * (32 * NB * 128) + j * 2048 + pl1);
            }
        };
        auto mul = [&](int a, int b) {   // (transposed: a lane holds four columns of a row)
            MRS_PIN();
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int kk = 0; kk < 2; kk++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++) acc[a][i][b][j] = Mma32<T>::mma(wf[j][kk], af[a][i][kk], acc[a][i][b][j]);
            __builtin_amdgcn_s_setprio(0);
            MRS_PIN();
        };
        // a request takes the place of what both groups of waves have read before the last barrier
        const bool more = kt + 2 < nk;
        read_b(0); read_a(0);
        MRS_PIN(); MRS_LGKM0(); MRS_BAR(); mul(0, 0); MRS_BAR();
        read_a(1);
        if (more) req_a(kt + 2, 0);
        MRS_PIN(); MRS_LGKM0(); MRS_BAR(); mul(1, 0); MRS_BAR();
        read_b(1);
        if (more) req_a(kt + 2, 1);
        MRS_PIN(); MRS_LGKM0(); MRS_BAR(); mul(1, 1); MRS_BAR();
        if (more) { req_b(kt + 2); asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 + NB) : "memory"); }   // the next step is in
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        MRS_PIN(); MRS_BAR(); mul(0, 1); MRS_BAR();
    }
    if (w < 4) MRS_BAR();

    // Out.  Two lanes trade halves of their pieces so that a lane stores sixteen bytes: of tiles x and y, lanes of even row group get x's columns, of odd y's.
    auto out_pair = [&](const v4f &x, const v4f &y, int row, int col) {
        unsigned x0 = pack2<T>(x[0], x[1]), x1 = pack2<T>(x[2], x[3]), y0 = pack2<T>(y[0], y[1]), y1 = pack2<T>(y[2], y[3]);
        swap16(x0, y0); swap16(x1, y1);
        if (row < M && col < (SPLIT ? split.n1 : N)) *reinterpret_cast<uint4 *>(C + (int64_t)row * ldc + col) = make_uint4(x0, x1, y0, y1);
    };
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int row = m0 + a * 128 + wm * 32 + lr, col = n0 + b * 32 * NB + wn * 16 * NB + 8 * (lg >> 1);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j + 1 < NB; j += 2) out_pair(acc[a][i][b][j], acc[a][i][b][j + 1], row + 16 * i, col + 16 * (j + (lg & 1)));
            if constexpr (SPLIT) {
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++) {
                        const int c = n0 + b * 32 * NB + wn * 16 * NB + 16 * j;   // (the same for the wave)
                        if (c >= split.n1 && row + 16 * i < M && c + 4 * lg < N)
                            *reinterpret_cast<v4f *>(split.C2 + (int64_t)(row + 16 * i) * split.ldc2 + (c + 4 * lg - split.n1)) = acc[a][i][b][j];
                    }
            }
            if constexpr (NB & 1) out_pair(acc[a][0][b][NB - 1], acc[a][1][b][NB - 1], row + 16 * (lg & 1), col + 16 * (NB - 1));
        }
}

template <typename T, int NB, bool SPLIT = false>
int launch_big(hipStream_t st, void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int M, int N, int K, const BigSplit &split = {}) {
    constexpr size_t lds = 2 * (kTileM + 64 * NB) * 128;
    static const hipError_t attr = hipFuncSetAttribute((const void *)gemm_big_kernel<T, NB, SPLIT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "big gemm: LDS size: %s", hipGetErrorString(attr));
    const int mt = (M + kTileM - 1) / kTileM, nt = (N + 64 * NB - 1) / (64 * NB);
    hipLaunchKernelGGL((gemm_big_kernel<T, NB, SPLIT>), dim3((unsigned)(mt * nt)), dim3(kBigThreads), lds, st, (T *)C, ldc, (const T *)A, lda, (const T *)Wt, M, N, K, mt, nt, split);
    return check_launch("gemm_big_kernel");
}

template <typename T>
int launch_big_type(hipStream_t st, int nb, void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int M, int N, int K) {
    return nb == 3 ? launch_big<T, 3>(st, C, ldc, A, lda, Wt, M, N, K) : launch_big<T, 5>(st, C, ldc, A, lda, Wt, M, N, K);
}

struct BigPlan { int nb; double us; };
// Columns of a tile over 64 for the less time in whole rounds over the compute units: a k-step of 64 nb columns takes about 0.2 + 0.31 nb us, and a
// round 3 + 0.5 nb around its steps (from the figures above and 19 other shapes, all within 10 %).
BigPlan big_plan(int64_t M, int N, int K) {
    BigPlan best = {0, 0.0};
    for (int nb = 3; nb <= 5; nb += 2) {   // (256 columns are the library's own, and it is ahead with them)
        const int64_t tiles = (M + kTileM - 1) / kTileM * ((N + 64 * nb - 1) / (64 * nb));
        const double us = (double)((tiles + 255) / 256) * (K / kStepK * (0.2 + 0.31 * nb) + 3.0 + 0.5 * nb);
        if (!best.nb || us < best.us) best = {nb, us};
    }
    return best;
}

}  // namespace

// Where the own kernel is ahead of the library's.  Up to one round of the library's 256 x 256 tiles it is not (its smaller tiles then fill the chip:
// 5000 x 768 x 1536 17 us, this 26), nor where its rounds are full.  A round costs it 1.24 us a k-step + 4, and a last one less than half full a
// tenth more on all of them (5000 x 10240 x 2560, 3.1 rounds: 250, this 200; 10000, 6.25: 394 / 365), a fuller one next to nothing (6000, 3.75: 227 /
// 220 alone, and in a prefill 2560 / 2586 for four layers; 10000 x 3072 x 768, 1.9: 44 / 46).
bool big_gemm_wins(int64_t M, int N, int K) {
    const int64_t tiles = (M + 255) / 256 * ((N + 255) / 256), rest = tiles % 256;
    return tiles > 256 && rest && big_plan(M, N, K).us < (rest <= 128 ? 1.1 : 1.04) * (double)((tiles + 255) / 256) * (K / kStepK * 1.24 + 4.0);
}

bool big_gemm_ok(int dtype, const void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K) {
    return (dtype == MRS_BF16 || dtype == MRS_F16) && M >= 1 && M < (int64_t)1 << 30 && N >= 8 && N % 8 == 0 && K >= 2 * kStepK && K % kStepK == 0 && lda % 8 == 0 && lda >= K &&
           lda < 1 << 22 && K < 1 << 22 && ldc % 8 == 0 && ldc >= N && aligned(C, 16) && aligned(A, 16) && aligned(Wt, 16) &&
           (M + kTileM - 1) / kTileM * ((N + 191) / 192) < (int64_t)1 << 28;
}

int launch_big_gemm(hipStream_t st, int dtype, void *C, int64_t ldc, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K) {
    if (!big_gemm_ok(dtype, C, ldc, A, lda, Wt, M, N, K))
        return fail(MRS_E_SHAPE, "big gemm: 16-bit storage, N %% 8 == 0, K %% 64 == 0 from 128 up, 16-byte aligned operands (M=%lld N=%d K=%d)", (long long)M, N, K);
    const int nb = big_plan(M, N, K).nb;
    return dtype == MRS_BF16 ? launch_big_type<bf16_t>(st, nb, C, ldc, A, lda, Wt, (int)M, N, K) : launch_big_type<f16_t>(st, nb, C, ldc, A, lda, Wt, (int)M, N, K);
}

bool big_gemm_split_ok(int dtype, const void *C, int64_t ldc, const BigSplit &split, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K) {
    return big_gemm_ok(dtype, C, ldc, A, lda, Wt, M, split.n1, K) && split.n1 % 16 == 0 && N > split.n1 && N % 4 == 0 && split.ldc2 % 4 == 0 && split.ldc2 >= N - split.n1 &&
           aligned(split.C2, 16) && (M + kTileM - 1) / kTileM * ((N + 191) / 192) < (int64_t)1 << 28;
}

static double split_us(int64_t M, int N, int K) { return (double)(((M + kTileM - 1) / kTileM * ((N + 319) / 320) + 255) / 256) * (K / kStepK * 1.75 + 5.5); }

// One launch over all columns, 320 to a tile, against the first n1 on whichever kernel big_gemm_wins() names and the rest on the library's (5 us and what it moves at
// 3 TB/s: 16384 x 216 x 768 18.4).  The rest often rides in rounds that the first columns leave partly empty.  Four layers of a bf16 Mamba-3 prefill, d_model 768
// (3072 + 216 columns), two products / one: 2000 rows 487 / 492, 3000 540 / 533, 5000 723 / 678, 6000 792 / 845, 10000 1054 / 1011, 12000
// 1185 / 1232, 16384 1249 / 1219.
bool big_gemm_split_wins(int64_t M, int n1, int N, int K) {
    const int64_t tiles = (M + 255) / 256 * ((n1 + 255) / 256);
    const double first = big_gemm_wins(M, n1, K) ? big_plan(M, n1, K).us : 1.1 * (double)((tiles + 255) / 256) * (K / kStepK * 1.24 + 4.0);
    return M >= 2560 && split_us(M, N, K) < first + 5.0 + (double)M * (2.0 * K + 4.0 * (N - n1)) / 3e6;
}

int launch_big_gemm_split(hipStream_t st, int dtype, void *C, int64_t ldc, const BigSplit &split, const void *A, int64_t lda, const void *Wt, int64_t M, int N, int K) {
    if (!big_gemm_split_ok(dtype, C, ldc, split, A, lda, Wt, M, N, K))
        return fail(MRS_E_SHAPE, "big gemm: columns %d of %d in f32 (M=%lld K=%d)", N - split.n1, N, (long long)M, K);
    return dtype == MRS_BF16 ? launch_big<bf16_t, 5, true>(st, C, ldc, A, lda, Wt, (int)M, N, K, split) : launch_big<f16_t, 5, true>(st, C, ldc, A, lda, Wt, (int)M, N, K, split);
}

}  // namespace mrs
