// Host rows in, host rows out: how the engines' step() hands a step's input to the GPU and takes its result back.
//
// The rows travel through one block of pinned, coherent host memory the engine owns: the GPU reads the input from it and writes
// the result into it, each row followed by the step's number in that row's flag, and the host waits for the flags.  Against a
// pageable hipMemcpyAsync each way and a stream synchronisation -- about 32 us around a 38 us step of the default
// configuration -- that leaves a launch, the trips over the bus and nothing else: 8 us around the same step.
#pragma once
#include "common.hpp"
#include <chrono>
#include <string.h>

namespace mrs {

// A flag has a line of host memory to itself: the host reads it over and over while the GPU's writes come in, and with sixteen rows' flags in a line every one
// of those writes takes the line away from it.  Flags apart, rows and states written past the caches (host_store below), a step of three f32 layers, before / now, us:
// d_model 64 1 row 20.2 / 19.2, 48 rows 27.2 / 21.3, 128 rows 38.9 / 21.9; 128 28.3 / 27.4, 36.4 / 29.7, 48.6 / 31.5; Mamba-3, four layers of 128, 35.3 / 33.3, 42.0 / 34.6, 54.4 / 36.3.
constexpr int kHostFlag = 16;

struct HostIo {
    char *block = nullptr;
    float *in = nullptr, *out = nullptr;   // [rows][input_dim], [rows][dm]
    unsigned *done = nullptr;              // [rows][kHostFlag]: the number of the last step whose row is complete
    unsigned seq = 0;
    int rows = 0;
};

inline int host_io_create(HostIo *io, int rows, int input_dim, int dm) {
    auto up = [](size_t n) { return (n + 255) / 256 * 256; };
    const size_t a = up((size_t)rows * input_dim * 4), b = up((size_t)rows * dm * 4), c = up((size_t)rows * kHostFlag * 4);
    const hipError_t e = hipHostMalloc((void **)&io->block, a + b + c, hipHostMallocMapped | hipHostMallocCoherent);
    if (e != hipSuccess) return fail(MRS_E_HIP, "pinned rows: %s", hipGetErrorString(e));
    io->in = (float *)io->block; io->out = (float *)(io->block + a); io->done = (unsigned *)(io->block + a + b);
    memset(io->done, 0, c);
    io->seq = 0; io->rows = rows;
    return MRS_OK;
}
inline void host_io_destroy(HostIo *io) { if (io->block) hipHostFree(io->block); io->block = nullptr; }

// Waits until every row of step io->seq is there.  A step that takes longer than a few milliseconds is left to the runtime's own wait.
inline int host_io_wait(HostIo *io, hipStream_t st) {
    volatile unsigned *done = io->done;
    int first = 0;   // the rows before it are complete
    auto complete = [&]() {
        constexpr int kAtOnce = 8;   // flags whose lines are asked for together
        for (; first < io->rows; first += kAtOnce) {
            unsigned open = 0;
            for (int r = first; r < io->rows && r < first + kAtOnce; r++) open |= done[(size_t)r * kHostFlag] ^ io->seq;
            if (open) return false;
        }
        return true;
    };
    const auto t0 = std::chrono::steady_clock::now();
    for (unsigned n = 1; !complete(); n++) {
        __builtin_ia32_pause();
        if ((n & 255) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(4)) {
            const hipError_t e = hipStreamSynchronize(st);
            if (e != hipSuccess) return fail(MRS_E_HIP, "step: %s", hipGetErrorString(e));
            if (!complete()) return fail(MRS_E_HIP, "step: the GPU finished without delivering the rows");
        }
    }
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
    return MRS_OK;
}

// A float of the result, written past the caches, and one row's flag behind all of them: every thread of the workgroup that wrote the row calls host_row_done.
// Nothing but these floats has to be out before the flag is, so each wave waits for its own stores and that is all.  (A fence for the whole system writes
// back every changed line of the die's L2 first, once for each row.)  A single-launch step writes its final rows and the copy of its input rows on the device in the same way, and the
// Mamba-1 ones their states: the flags let the caller go on before the launch has ended, and another stream of the caller's may use what temporal_ptr(), input_ptr() and state_ptrs() give.
__device__ __forceinline__ void host_store(float *p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }
// Four of them, `off` bytes (a multiple of 16) into a block of `bytes` that all lanes share.
__device__ __forceinline__ void host_store4(float *block, int bytes, unsigned off, float4 v) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    constexpr int kSystem = 1 | 16;   // sc0, sc1: what the stores above have
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), __builtin_amdgcn_make_buffer_rsrc(block, 0, bytes, 0x00020000), off, 0, kSystem);
}
// What a single-launch step leaves on the device.  now: flags will say so (above).  Without them the launch's end brings it out, and the next step finds it in the L2.
__device__ __forceinline__ void leave(bool now, float *p, float v) {
    if (now) host_store(p, v);
    else *p = v;
}
__device__ __forceinline__ void leave4(bool now, float *block, int bytes, unsigned off, float4 v) {
    if (now) host_store4(block, bytes, off, v);
    else *reinterpret_cast<float4 *>(reinterpret_cast<char *>(block) + off) = v;
}
__device__ __forceinline__ void host_row_done(const HostRows &h, int row) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(h.done + (size_t)row * kHostFlag, h.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

static __global__ __launch_bounds__(256) void host_in_kernel(float *__restrict__ dst, const float *__restrict__ src, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}
// A step's input projection: out[row][n] = bias[n] + sum_k in[row][k] W[k][n], W [K][N] row-major, N a multiple of 4, and the row once more into `copy` (or null): it may come
// straight from host memory.  A workgroup has a row: a thread four consecutive columns over one slice of K, its first eight weight rows on their way while the row is, and the
// slices' sums meet in LDS.  Bound by its trips to memory.  As a kernel for the bias, the library's product (about 5 us for one row) and, from host memory, a copy in front, they
// were three launches: a step of four bf16 layers of d_model 128, 1 row 51 us, this 41 (48 rows 85 / 78); Mamba-3 53 / 41 and 73 / 68; four f32 layers of 192, 48 rows, 120 / 111.
constexpr int kProjThreads = 512, kProjMaxK = 4096;
inline bool project_rows_ok(int64_t rows, int K, int N) { return rows >= 1 && rows <= 128 && K >= 1 && K <= kProjMaxK && N >= 4 && N % 4 == 0 && N <= 4 * kProjThreads; }
static __global__ __launch_bounds__(kProjThreads) void project_rows_kernel(float *__restrict__ out, float *__restrict__ copy, const float *__restrict__ in, const float *__restrict__ W,
                                                                            const float *__restrict__ bias, int K, int N) {
    extern __shared__ float proj_x[];   // [slices][rows of a slice, in whole rounds], zeros behind K
    __shared__ float4 part[kProjThreads];
    constexpr int kRound = 8;
    const int tid = threadIdx.x, nq = N >> 2, slices = kProjThreads / nq, per = (K + slices - 1) / slices, padded = (per + kRound - 1) / kRound * kRound;
    const int q = tid % nq, s = min(tid / nq, slices - 1), k0 = s * per;   // (threads behind the last slice repeat it)
    const int64_t row = blockIdx.x;
    float4 w[kRound];
    auto ask = [&](int j0) {
#pragma unroll
        for (int j = 0; j < kRound; j++) w[j] = *reinterpret_cast<const float4 *>(W + (int64_t)min(k0 + j0 + j, K - 1) * N + 4 * q);
    };
    ask(0);
    for (int i = tid; i < slices * padded; i += kProjThreads) {
        const int sl = i / padded, j = i - sl * padded, k = sl * per + j;
        float v = 0.0f;
        if (j < per && k < K) {
            v = in[row * K + k];
            if (copy) copy[row * K + k] = v;
        }
        proj_x[i] = v;
    }
    __syncthreads();
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int j0 = 0; j0 < per; j0 += kRound) {
        if (j0) ask(j0);
#pragma unroll
        for (int j = 0; j < kRound; j++) {
            const float x = proj_x[s * padded + j0 + j];
            acc.x = fmaf(x, w[j].x, acc.x); acc.y = fmaf(x, w[j].y, acc.y); acc.z = fmaf(x, w[j].z, acc.z); acc.w = fmaf(x, w[j].w, acc.w);
        }
    }
    part[tid] = acc;
    __syncthreads();
    if (tid < nq) {
        float4 o = *reinterpret_cast<const float4 *>(bias + 4 * tid);
        for (int t = 0; t < slices; t++) {
            const float4 p = part[t * nq + tid];
            o.x += p.x; o.y += p.y; o.z += p.z; o.w += p.w;
        }
        *reinterpret_cast<float4 *>(out + row * N + 4 * tid) = o;
    }
}
inline int launch_project_rows(hipStream_t st, float *out, float *copy, const float *in, const float *W, const float *bias, int rows, int K, int N) {
    const int slices = kProjThreads / (N / 4), per = (K + slices - 1) / slices;
    hipLaunchKernelGGL(project_rows_kernel, dim3((unsigned)rows), dim3(kProjThreads), (size_t)slices * ((per + 7) / 8 * 8) * 4, st, out, copy, in, W, bias, K, N);
    return check_launch("project_rows_kernel");
}

static __global__ __launch_bounds__(256) void host_out_kernel(HostRows h, const float *__restrict__ rows, int dm) {
    const int r = blockIdx.x;
    for (int i = threadIdx.x; i < dm; i += 256) host_store(h.out + (size_t)r * dm + i, rows[(size_t)r * dm + i]);
    host_row_done(h, r);
}

}  // namespace mrs
