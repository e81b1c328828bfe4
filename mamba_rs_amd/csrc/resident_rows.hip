// A whole Mamba-1 backbone step in one resident launch, for up to sixteen batch rows per group of workgroups.
//
// resident_step.hip gives every row a group of G workgroups, so four rows of d_model 768 fill the chip.  Here a group takes up to
// sixteen rows, the rows of one matrix instruction: the weights come in once for all of them.  Ownership is the same (workgroup s:
// d_inner / G channels, d_model / G columns of out_proj with the residual there), so is the order of the weights in memory.  Per layer:
//   in_proj on the normed residual rows, conv + SiLU of the own channels -> exchange 2f: u, to the few workgroups that form a column
//                                         tile of the x_proj rows each    -> exchange 2: those rows, to all
//   dt_proj + softplus, state update, gate of the own channels          -> exchange 3: y
//   out_proj, residual add                                              -> exchange 1: the next operand, and sums of squares
// (Shares of x_proj added up by every workgroup, as one row's are, would be 650 KB read by each at sixteen rows; added up in two steps they
// took 7.9 us a layer at 64 rows of d_model 768 where this takes 4.)
//
// Operand rows are plain memory, written through to where all dies see them and followed by a flag; every layer has rows of its own, so
// that their readers can take them through their die's cache (words that carry their tag, polled by 64 workgroups of four groups:
// 605 us a step at 64 rows of d_model 768, flags 517 in the same state of this file).  They lie in matrix-core order: with K split over
// the computing waves a wave loads its k-steps straight into the registers they are used from.
//
// What bounds it: four exchanges a layer of 0.5 us per hand-over -- store, flag, rows: ten of them -- and the chains of a few hundred
// instructions between them; at full groups the states as well (12 MB a layer).  Per step, kernel chain / this (bf16, steps queued): 24
// layers of d_model 768 at 5, 16, 32, 64 rows 311 / 240, 362 / 247, 409 / 273, 512 / 314 us; of 1024 at 2, 13, 32 407 / 286, 432 / 306, 495 / 336;
// eight of 512 at 64 134 / 91; four of 256 at 128 68 / 41.
#include "resident_m1.hpp"
#include <type_traits>

namespace mrs {
namespace {

constexpr int kRows = kResidentRows;   // of a group: the rows of a matrix instruction
static_assert(kRows == 16, "");
// The shapes: d_model a multiple of 256 (KI: k-steps of in_proj per computing wave), expand 2 and the rank of dt that goes with the
// width.  All sizes are constants: with run-time sizes the layer loop was 2 200 instructions a wave, a third of them address arithmetic and
// reloads of scalars, and that is time: a phase is a chain of a few hundred instructions on two waves a SIMD.
constexpr int kLineWords = 16;   // exchange words of a cache line
template <int KI> struct RowsShape {
    static constexpr int dm = 256 * KI, di = 2 * dm, dr = dm / 16, xd = dr + 2 * kDs, nc = KI == 3 ? 24 : 16, G = di / nc, oc = dm / G;
    static constexpr int iks = dm / 32, oks = di / 32;                    // k-steps of 32
    static constexpr int ct = 2 * nc / 16, tiles = (nc + 15) / 16, xt = xd / 16;   // column tiles of in_proj, channel tiles, column tiles of x_proj: a workgroup of the group for each
    static constexpr SmallBlock sb = small_block(nc, oc, 0, dr);
    static constexpr LayerBlock lb = layer_block(dm, di, nc, oc, 0, dr);
    // a layer's weights: the workgroups' blocks, and behind them x_proj as [tile][k-step][lane][8]
    static constexpr unsigned x_bytes = (unsigned)(xt * oks) * 1024u;
    static constexpr size_t layer_bytes = (size_t)G * lb.bytes + x_bytes;
    // LDS (bytes): the in_proj weights at 0, and once they are in registers the waves' shares of its product
    static constexpr int xdp = xd + 4, xdtp = 32 * ((dr + 31) / 32) + 8;   // rows of f32, of the storage type
    static constexpr int win = up1k(2 * nc * dm * 2), pre = kComputeWaves * ct * 1024, wout = win > pre ? win : pre, small = wout + up1k(oc * di * 2),
                         pre2 = small + 2 * sb.bytes, xdl = pre2 + kComputeWaves * 1024, xdt = xdl + kRows * xdp * 4, sqs = xdt + kRows * xdtp * 2,
                         spare = sqs + kComputeWaves * kRows * 4, lds = spare + 256;
    // A group's exchange words.  2f and 3f, the flags of u and y: [workgroup][16], the first of them used; 2, the x_proj rows: [tile][row][8]; 1,
    // the sums of squares: [workgroup][row].  No two workgroups write to one cache line: a line that every die is reading is taken from
    // all of them at each write.  (Flags side by side: 24 layers of d_model 768 at 64 rows 403 us a step, as they are 374.)
    static constexpr unsigned e2f = 0, e3f = kLineWords * G, e2 = 2 * kLineWords * G, e1 = e2 + xt * kRows * 8, words = e1 + kRows * G;
    // ... and its operand rows: per layer u, y and the next layer's operand, in matrix-core order ([k-step][lane][8])
    static constexpr unsigned u_bytes = di * kRows * 2, rows_bytes = (2 * di + dm) * kRows * 2;
    static_assert(kRows * nc * kDs * 4 / 128 <= 192 && kRows * nc * kDc * 4 / 128 <= 64 && nc * kDc * 4 % 128 == 0, "a request per wave for the states' lines");
    static_assert(xd % 16 == 0 && xd <= kMaxXd && dr <= kMaxDr && nc % 8 == 0 && nc <= kMaxNc && oc % 2 == 0 && oc <= kMaxOc && nc * G == di && oc * G == dm &&
                  xt <= G && G % 8 == 0 && G <= 128 && (size_t)lds <= kResLdsMax && kRows == kLineWords, "");
};

// The waves that bring weights, as in resident.hpp, for the barriers of this kernel.  A layer has, behind the taking of in_proj's weights into
// registers, T (their buffer becomes the shares'), then A behind in_proj, B behind the conv, X behind x_proj (the buffer is free), C
// behind exchange 2, D when y is there and E behind out_proj.  The four waves ask for out_proj's weights and a part of the next
// in_proj's while x_proj's rows are waited for, and for the rest while y is: where the exchanges need the memory least.
struct RowsFeed {
    const char *blk;              // this workgroup's block of layer 0
    size_t next;                  // ... to that of the next layer
    unsigned win, wout, small;    // LDS byte addresses; the small blocks of two layers lie one after the other
    // This workgroup's states in layer 1: their lines are asked for a phase before they are loaded (into `spare`: 256 bytes of LDS nobody
    // reads).  At full groups they are 12 MB a layer, mostly from memory, and a wave's polls stand behind its own loads.
    const char *conv, *ssm;
    size_t conv_next, ssm_next;   // ... to those of the next layer
    int rows;
    unsigned spare;
    int cached;                   // layers whose weights come through the last cache; the others' are read past it
    bool hurry;                   // the workgroup forms x_proj rows: it does not wait for them, but for u, a barrier earlier
};
// One request: a lane asks for a line, number `first` + lane of `lines` of 128 bytes per row.
template <int LINES, int ROW_BYTES> __device__ __forceinline__ void touch_lines(unsigned spare, const char *at, int rows, int first) {
    const int n = min(first + (int)(threadIdx.x & 63), rows * LINES - 1), r = n / LINES;
    const unsigned voff = (unsigned)(r * ROW_BYTES + (n - r * LINES) * 128);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(spare), "v"(voff), "s"(at) : "m0", "memory");
}
template <class S> __device__ __forceinline__ void bring_rows_weights(const RowsFeed f, int wave, int nl, int &state, RollCall call) {
    constexpr int in_pieces = S::lb.out >> 10, out_pieces = (S::lb.small - S::lb.out) >> 10, small_pieces = S::sb.bytes >> 10, early = in_pieces / 2;
    const char *blk = f.blk;
    const bool first = (threadIdx.x & 63) == 0, roll_wave = wave == 10;
    const int w = wave - kComputeWaves;
    if (roll_wave) {
        const int s = call.answer();
        if (first) state = s;
    }
    dma_to_lds(f.win, blk, w, in_pieces, 4);
    dma_to_lds(f.small, blk + S::lb.small, w, small_pieces, 4);
    dma_wait();
    // The roll call's outcome is taken while the workgroup's first wait for others goes on, that is in front of the same barrier: behind it,
    // the wait would have no end where the others are called off (xch_poll does not count while `state` is kRollCall).
    const auto take_outcome = [&] {
        if (roll_wave && state == kRollCall) {
            const int s = call.outcome();
            if (first) state = s;
        }
    };
    lds_barrier();   // layer 0's weights are there
    lds_barrier();   // T
#pragma unroll 1
    for (int l = 0; l < nl; l++) {
        const bool more = l + 1 < nl;
        const char *next = blk + f.next, *ssm = f.ssm + l * f.ssm_next, *conv = f.conv + l * f.conv_next;   // the next layer's
        if (state > 0) return;   // (called off before it began, or lost)
        lds_barrier();   // A
        if (l == 0 && f.hurry) take_outcome();
        lds_barrier();   // B
        lds_barrier();   // X
        const auto early_part = [&](auto sleep) {
            constexpr int Z = decltype(sleep)::value;
            dma_to_lds<Z>(f.wout, blk + S::lb.out, w, out_pieces, 4, l >= f.cached);
            if (more) {
                dma_to_lds<Z>(f.small + ((l + 1) & 1) * S::sb.bytes, next + S::lb.small, w, small_pieces, 4);
                dma_to_lds<Z>(f.win, next, w, early, 4, l + 1 >= f.cached);
            }
        };
        if (f.hurry) early_part(std::integral_constant<int, 1>());
        else early_part(std::integral_constant<int, 2>());
        if (l == 0 && !f.hurry) take_outcome();
        lds_barrier();   // C
        if (state) return;
        dma_wait();   // out_proj's weights are there
        if (more) {
            if (w < 3) touch_lines<S::nc * kDs * 4 / 128, S::di * kDs * 4>(f.spare, ssm, f.rows, w * 64);
            else touch_lines<S::nc * kDc * 4 / 128, S::di * kDc * 4>(f.spare, conv, f.rows, 0);
            dma_to_lds<1>(f.win, next, early + w, in_pieces, 4, l + 1 >= f.cached);
        }
        blk = next;
        lds_barrier();   // D
        if (state) return;
        dma_wait();
        lds_barrier();   // E
        lds_barrier();   // T
    }
}

// This wave's k-steps (wave, wave + 8, ...) of operand rows in matrix-core order.  Whoever wrote them has said so, and nobody on this die can
// have read them before in this launch: every layer has rows of its own.
template <int KS>
__device__ __forceinline__ void take_frags(const char *rows, uint4 (&a)[KS]) {
    asm volatile("" ::: "memory");   // not before the flags
    const unsigned at = (unsigned)here(threadIdx.x) * 16u;
#pragma unroll
    for (int s = 0; s < KS; s++) a[s] = ld_off<uint4>(rows + s * (kComputeWaves * 1024), at);
}
__device__ __forceinline__ void put_pair(char *rows, unsigned bytes, unsigned pair) {
    __hip_atomic_store(reinterpret_cast<unsigned *>(rows + bytes), pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// where channel c of a row (or its place) lies in operand rows
__device__ __forceinline__ unsigned operand_at(int c, int row) { return (unsigned)(((c >> 3) * kRows + row) * 16 + (c & 7) * 2); }
// u's and y's rows lie in the order 0 4 8 12 1 5 ...: the four a wave has are neighbours.
__device__ __forceinline__ int y_place(int row) { return (row & 3) * 4 + (row >> 2); }
// By each of n waves when it has put its part of u or y out: the last of them raises the workgroup's flag.
__device__ __forceinline__ void say(u64 *flag, unsigned tag, unsigned *count, unsigned n) {
    dma_wait();
    if ((here(threadIdx.x) & 63) == 0 && __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) % n == n - 1) xch_put(flag, 0.0f, tag);
}
template <typename T> __device__ __forceinline__ unsigned half_pair(T a, T b) {
    return (unsigned)__builtin_bit_cast(uint16_t, b) << 16 | __builtin_bit_cast(uint16_t, a);
}
// This wave's k-steps of a weight in LDS, [K / 8][COLS][8], in column tiles.
template <int KS, int COLS> struct RowsWeight {
    static constexpr int CT = (COLS + 15) / 16;
    uint4 w[KS][CT];
    __device__ __forceinline__ void take(const void *wl) {
        const int t = here(threadIdx.x), n = t & 15, at = (t >> 4) * COLS;
#pragma unroll
        for (int c = 0; c < CT; c++) {
            const uint4 *wp = reinterpret_cast<const uint4 *>(wl) + at + (COLS % 16 && c == CT - 1 ? min(c * 16 + n, COLS - 1) : c * 16 + n);
#pragma unroll
            for (int s = 0; s < KS; s++) w[s][c] = wp[s * (kComputeWaves * 4 * COLS)];
        }
    }
};
// A wave's share of a 16 x 16 tile: [register][lane], so that those who read one register's rows find them side by side.
__device__ __forceinline__ void put_share(float *out, int l, v4f v) {
#pragma unroll
    for (int i = 0; i < 4; i++) out[i * 64 + l] = v[i];
}
template <typename T, int KS, int COLS>
__device__ __forceinline__ void rows_product(const RowsWeight<KS, COLS> &w, const uint4 (&a)[KS], float *out) {
    constexpr int CT = RowsWeight<KS, COLS>::CT;
    const int t = here(threadIdx.x);
    v4f acc[CT];
#pragma unroll
    for (int c = 0; c < CT; c++) acc[c] = Mma32<T>::mma(a[0], w.w[0][c], (v4f){0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int s = 1; s < KS; s++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[c] = Mma32<T>::mma(a[s], w.w[s][c], acc[c]);
#pragma unroll
    for (int c = 0; c < CT; c++) put_share(out + ((t >> 6) * CT + c) * 256, t & 63, acc[c]);
}
// entry (row, column) of a product, its waves' shares added in wave order
template <int CT> __device__ __forceinline__ float rows_sum(const float *out, int row, int c) {
    const float *p = out + ((c >> 4) * 256 + (row & 3) * 64 + (row >> 2) * 16 + (c & 15));
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kComputeWaves; w++) v += p[w * CT * 256];
    return v;
}
// v[k] of lane 4 m + j becomes v[j] of lane 4 m + k: four lanes' sixteen states as four whole 64-byte lines.
__device__ __forceinline__ float quad_other(float v, int ctrl1) { return __uint_as_float(ctrl1 ? __builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xb1, 0xf, 0xf, true) : __builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x4e, 0xf, 0xf, true)); }
__device__ __forceinline__ void quad_turn(float4 (&v)[4]) {
    const bool odd = here(threadIdx.x) & 1, high = here(threadIdx.x) & 2;
    const auto swap = [](float &a, float &b, bool up, int ctrl1) {   // a of the upper lanes for b of the lower ones
        const float x = quad_other(up ? a : b, ctrl1);
        a = up ? x : a;
        b = up ? b : x;
    };
    const auto swap4 = [&](float4 &a, float4 &b, bool up, int ctrl1) {
        swap(a.x, b.x, up, ctrl1); swap(a.y, b.y, up, ctrl1); swap(a.z, b.z, up, ctrl1); swap(a.w, b.w, up, ctrl1);
    };
    swap4(v[0], v[1], odd, 1); swap4(v[2], v[3], odd, 1);
    swap4(v[0], v[2], high, 0); swap4(v[1], v[3], high, 0);
}
template <typename V> __device__ __forceinline__ void st_off(void *base, unsigned bytes, V v) { *reinterpret_cast<V *>(reinterpret_cast<char *>(base) + bytes) = v; }
__device__ __forceinline__ float neighbour(float v) { return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xb1, 0xf, 0xf, true)); }   // lane ^ 1's
__device__ __forceinline__ float sum_of_8(float v) {
    v += neighbour(v);
    v += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x4e, 0xf, 0xf, true));    // lane ^ 2
    return v + __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0x141, 0xf, 0xf, true));   // row_half_mirror
}
// Over the four rows of 16 lanes: the sum of the lanes 16 apart, in every lane.
__device__ __forceinline__ float quarters_sum(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <typename T, int KI>
__global__ __launch_bounds__(kResThreads) void resident_rows_kernel(const ResidentArgs *args, TokenRows rows) {
    using S = RowsShape<KI>;
    constexpr int dm = S::dm, di = S::di, nc = S::nc, oc = S::oc, G = S::G, dr = S::dr, KO = 2 * KI;
    constexpr SmallBlock sb = S::sb;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int state;   // kRollCall, 0, or a ResidentFault
    __shared__ unsigned put[2];   // waves that have put their u, y out
    const auto state_now = [] { return __hip_atomic_load(&state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    const auto *a = as_table(args);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = blockIdx.x / G, src = blockIdx.x % G, nl = a->n_layers;

    // this group's rows, this workgroup's channels and columns of out_proj
    const size_t cst_l = (size_t)a->batch * di * kDc, hst_l = (size_t)a->batch * di * kDs;   // states of a layer
    const int share = a->batch / a->groups, rest = a->batch - share * a->groups, nr = share + (grp < rest ? 1 : 0), r0 = grp * share + min(grp, rest);
    const int c0 = src * nc, o0 = src * oc;
    if (wave >= kComputeWaves) {
        const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
        bring_rows_weights<S>({(const char *)a->weights + (size_t)src * S::lb.bytes, S::layer_bytes, lds0, lds0 + S::wout, lds0 + S::small, (const char *)(a->conv_state + cst_l + (size_t)(r0 * di + c0) * kDc),
                               (const char *)(a->ssm_state + hst_l + (size_t)(r0 * di + c0) * kDs), cst_l * 4, hst_l * 4, nr, lds0 + S::spare, a->cached, src < S::xt}, wave, nl, state,
                              {a->roll, a->broken, gridDim.x, a->wait, 0});
        return;
    }

    // ---- the waves that compute
    const T *wout = (const T *)(smem + S::wout);
    float *pre = (float *)smem, *pre2 = (float *)(smem + S::pre2), *xdl = (float *)(smem + S::xdl), *sqs = (float *)(smem + S::sqs);
    T *xdt = (T *)(smem + S::xdt);
    char *orows = (char *)a->rows_buf + (size_t)grp * nl * S::rows_bytes;   // this layer's u; y and the next operand behind it
    u64 *xb = a->xch + (size_t)grp * a->xch_stride;
    unsigned *epoch = a->epoch + 32 * grp;
    const unsigned base = *epoch;
    const int lane = tid & 63;
    // conv and scan step: a (row, channel) per lane, as the matrix instructions leave a tile's rows i, i + 4, ... in register i
    const int ri = wave & 3, ctile = wave >> 2, row = 4 * (lane >> 4) + ri, cl = ctile * 16 + (lane & 15), c = min(cl, nc - 1);
    const bool tile_wave = ctile < S::tiles, mine = tile_wave && row < nr && cl < nc;
    const bool x_group = src < S::xt;   // this workgroup forms the group's x_proj column tile `src`
    const unsigned cell = (unsigned)((r0 + min(row, nr - 1)) * di + c0 + c);   // in a layer's states
    float *cst = a->conv_state, *hst = a->ssm_state;   // this layer's
    const char *xweights = (const char *)a->weights + (size_t)G * S::lb.bytes + (x_group ? src * (S::oks * 1024) : 0) + wave * 1024;
    // residual stream: row tid / 8, columns o0 + 2 (tid % 8) and + 1
    const int orow = (tid >> 3) & 15, op = tid & 7;
    const bool own = tid < 8 * kRows && orow < nr && op < (oc >> 1);

    RowsWeight<KI, 2 * nc> pin;
    uint4 fa[KI];
    float4 cwin, hv[4];
    float res0 = 0.0f, res1 = 0.0f;
    {
        const float *nw = a->norm_w;
        float sq = 0.0f;
        const auto operand = [&](int s, auto in) {
            const int k = (wave + kComputeWaves * s) * 32 + (lane >> 4) * 8;
            T v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float p = in(k + j);
                sq = fmaf(p, p, sq);
                v[j] = (T)(p * nw[k + j]);
            }
            fa[s] = __builtin_bit_cast(uint4, v);
            asm volatile("" : "+v"(fa[s].x), "+v"(fa[s].y), "+v"(fa[s].z), "+v"(fa[s].w)::"memory");   // a k-step's loads at a time
        };
        with_input_row<T>(a->input, rows, r0 + min(lane & 15, nr - 1), dm, [&](auto in, bool) {
#pragma unroll
            for (int s = 0; s < KI; s++) operand(s, in);
        });
        sq = quarters_sum(sq);
        if (tid < 2) put[tid] = 0;
        if (lane < kRows) sqs[wave * kRows + lane] = sq;
        if (own)
            with_input_row<T>(a->input, rows, r0 + orow, dm, [&](auto in, bool taken) {
                res0 = in(o0 + 2 * op); res1 = in(o0 + 2 * op + 1);
                if (taken) *reinterpret_cast<float2 *>(a->input + (size_t)(r0 + orow) * dm + o0 + 2 * op) = make_float2(res0, res1);
            });
        for (int i = tid; i < kRows * S::xdtp; i += kCompute) xdt[i] = (T)0.0f;   // (what lies behind dt_rank stays zero)
    }
    lds_barrier();
    pin.take(smem);
    if (tile_wave) {
        cwin = ld_off<float4>(cst, cell * (kDc * 4));
#pragma unroll
        for (int k = 0; k < 4; k++) hv[k] = ld_off<float4>(hst, cell * (kDs * 4) + 16 * k);
    }
    constexpr int GW = (G + 63) / 64;
    const auto find = [&](unsigned first, int k) { return first + (unsigned)((G % 64 ? min(here(lane), G - 1) : here(lane)) + 64 * k) * kLineWords; };
    // The workgroups' sums of squares, this wave's eighth of the workgroups: rows 2 (lane % 8) and + 1 of one of them in a lane.  When
    // they are there, so are the operand's columns.
    const auto take_sums = [&](unsigned tag) {
        constexpr int GL = G / 64 ? G / 64 : 1;   // workgroups per lane
        const int p = here(lane) & 7, g = here(lane) >> 3;
        u64 x[2 * GL];
        const bool ok = xch_poll<2 * GL>(xb, [&](int k) {
            return S::e1 + (unsigned)((wave * (G / 8) + (G < 64 ? min(g, G / 8 - 1) : g + 8 * (k >> 1))) * kLineWords + min(2 * p + (k & 1), nr - 1));
        }, [&](u64 w) { return (unsigned)(w >> 32) == tag; }, x);
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int k = 0; k < GL; k++) { s0 += __uint_as_float((unsigned)x[2 * k]); s1 += __uint_as_float((unsigned)x[2 * k + 1]); }
        if (G < 64 && g >= G / 8) s0 = s1 = 0.0f;
        s0 = groups_sum(s0); s1 = groups_sum(s1);
        if (here(lane) < 8) *reinterpret_cast<float2 *>(sqs + wave * kRows + 2 * p) = make_float2(s0, s1);
        if (!ok && state == 0) state = kStepLost;
    };
    const auto scale_of = [&](int r) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kComputeWaves; w++) s += sqs[w * kRows + r];
        return inv_rms(s, dm, a->eps);
    };
    lds_barrier();   // T

#pragma unroll 1
    for (int l = 0; l < nl; l++) {
        const unsigned tag = base + 1 + l;
        const bool more = l + 1 < nl;
        const char *small = smem + S::small + (l & 1) * sb.bytes;
        const auto tagged = [&](u64 w) { return (unsigned)(w >> 32) == tag; };
        if (l > 0) take_frags<KI>(orows - dm * kRows * 2, fa);
        const float inv = scale_of(row);   // while they are on their way
        // ---- in_proj
        rows_product<T>(pin, fa, pre);
        uint4 xw[KO];
        if (x_group) {
#pragma unroll
            for (int s = 0; s < KO; s++) xw[s] = ld_off<uint4>(xweights + s * (kComputeWaves * 1024), (unsigned)here(lane) * 16u);
        } else {
#pragma unroll
            for (int s = 0; s < KO; s++) xw[s] = make_uint4(0, 0, 0, 0);
        }
        xweights += S::layer_bytes;
        if (state > 0) break;   // (called off before it began, or lost)
        lds_barrier();   // A
        // ---- conv step + SiLU
        float xnew = 0.0f, z = 0.0f, u = 0.0f;
        if (tile_wave) {
            const float4 tap = *reinterpret_cast<const float4 *>(small + sb.cw + c * 16);
            const float bias = *reinterpret_cast<const float *>(small + sb.cb + c * 4);
            const T xr = (T)(rows_sum<S::ct>(pre, row, c) * inv), zr = (T)(rows_sum<S::ct>(pre, row, nc + c) * inv);
            xnew = Store<T>::ld(&xr); z = Store<T>::ld(&zr);
            float o = fmaf(cwin.y, tap.x, bias);
            o = fmaf(cwin.z, tap.y, o); o = fmaf(cwin.w, tap.z, o); o = fmaf(xnew, tap.w, o);
            const T ur = (T)silu(o);
            u = Store<T>::ld(&ur);
            const float un = neighbour(u);
            const int ch = c0 + cl;
            if (mine && (cl & 1) == 0) put_pair(orows, operand_at(ch, y_place(row)), half_pair<T>(ur, (T)un));
            say(xb + S::e2f + (unsigned)src * kLineWords, tag, &put[0], 4 * S::tiles);
        }
        // ---- x_proj: the tile's workgroup takes u of all channels
        bool ok = true;
        if (x_group && wave == 0) {
            u64 r[GW];
            ok = xch_poll<GW>(xb, [&](int k) { return find(S::e2f, k); }, tagged, r, state_now);
        }
        lds_barrier();   // B
        if (x_group) {
            uint4 fu[KO];
            take_frags<KO>(orows, fu);
            v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KO; s++) acc = Mma32<T>::mma(fu[s], xw[s], acc);
            put_share(pre2 + wave * 256, here(lane), acc);
        }
        lds_barrier();   // X
        if (x_group && wave < 4) {
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < kComputeWaves; w++) v += pre2[(w * 4 + wave) * 64 + here(lane)];
            const float vn = neighbour(v);
            const int xr = (here(lane) >> 4) + 4 * wave, n = here(lane) & 15;   // (the rows lie in y's order: register i of quarter q is row 4 i + q)
            if (xr < nr && (n & 1) == 0) xch_put_word(xb + S::e2 + (unsigned)((src * kRows + xr) * 8 + (n >> 1)), half_pair_word<T>((T)v, (T)vn, tag));
        }
        // ---- the x_proj rows: word tid % 8 of row tid / 8 % 16 of tile tid / 128, and of tile 4 + tid / 128
        {
            constexpr int XW = (S::xt + 3) / 4;
            const int t0 = here(tid), xr = (t0 >> 3) & 15;
            const auto tile = [&](int k) { return min((t0 >> 7) + 4 * k, S::xt - 1); };
            u64 r[XW];
            if (xr < nr) ok = xch_poll<XW>(xb, [&](int k) { return S::e2 + (unsigned)(tile(k) * (kRows * 8) + (t0 & 127)); }, tagged, r, state_now) && ok;
#pragma unroll
            for (int k = 0; k < XW; k++) {
                const int col = tile(k) * 16 + 2 * (t0 & 7);
                const unsigned pair = (unsigned)r[k];
                const uint16_t b0 = (uint16_t)pair, b1 = (uint16_t)(pair >> 16);
                const T v0 = __builtin_bit_cast(T, b0), v1 = __builtin_bit_cast(T, b1);
                if (xr < nr) {
                    *reinterpret_cast<float2 *>(xdl + xr * S::xdp + col) = make_float2(Store<T>::ld(&v0), Store<T>::ld(&v1));
                    if (col < dr) *reinterpret_cast<unsigned *>(xdt + xr * S::xdtp + col) = pair;
                }
            }
        }
        if (!ok && state == 0) state = kStepLost;
        lds_barrier();   // C
        if (state) break;
        char *yrows = orows + S::u_bytes, *onext = yrows + S::u_bytes;
        if (tile_wave) {
            // ---- dt_proj + softplus
            const int n = here(lane) & 15, kg = here(lane) >> 4;
            v4f td = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < (dr + 31) / 32; s++) {
                const int k = 32 * s + 8 * kg;
                const uint4 xa = *reinterpret_cast<const uint4 *>(xdt + n * S::xdtp + k);
                uint4 wb = make_uint4(0, 0, 0, 0);
                if (32 * s + 32 <= dr || k < dr) wb = *reinterpret_cast<const uint4 *>(small + sb.dtw + (c * dr + k) * 2);
                td = Mma32<T>::mma(xa, wb, td);
            }
            const float t01 = ri & 1 ? td[1] : td[0], t23 = ri & 1 ? td[3] : td[2], tdv = ri & 2 ? t23 : t01;
            const float delta = softplus20(tdv + *reinterpret_cast<const float *>(small + sb.dtb + c * 4));
            // ---- state update, D skip, gate
            const float dl = delta * kLog2e, du = delta * u;
            const float4 *av = reinterpret_cast<const float4 *>(small + sb.aneg + c * (kDs * 4)), *Bv = reinterpret_cast<const float4 *>(xdl + row * S::xdp + dr);
            float acc = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 an = av[k];
                const float2 b0 = reinterpret_cast<const float2 *>(Bv)[2 * k], b1 = reinterpret_cast<const float2 *>(Bv)[2 * k + 1],
                             q0 = reinterpret_cast<const float2 *>(Bv)[8 + 2 * k], q1 = reinterpret_cast<const float2 *>(Bv)[8 + 2 * k + 1];
                hv[k].x = fmaf(fast_exp2(dl * an.x), hv[k].x, du * b0.x); acc = fmaf(hv[k].x, q0.x, acc);
                hv[k].y = fmaf(fast_exp2(dl * an.y), hv[k].y, du * b0.y); acc = fmaf(hv[k].y, q0.y, acc);
                hv[k].z = fmaf(fast_exp2(dl * an.z), hv[k].z, du * b1.x); acc = fmaf(hv[k].z, q1.x, acc);
                hv[k].w = fmaf(fast_exp2(dl * an.w), hv[k].w, du * b1.y); acc = fmaf(hv[k].w, q1.y, acc);
            }
            const float yv = fmaf(*reinterpret_cast<const float *>(small + sb.D + c * 4), u, acc) * silu(z), yn = neighbour(yv);
            const int ch = c0 + cl;
            if (mine && (cl & 1) == 0) put_pair(yrows, operand_at(ch, y_place(row)), half_pair<T>((T)yv, (T)yn));
            say(xb + S::e3f + (unsigned)src * kLineWords, tag, &put[1], 4 * S::tiles);
        }
        // The states go back while y is on its way (those of the wave that looks for it, later: its polls would stand behind them).
        const auto put_states = [&] {
            if (mine) st_off(cst, cell * (kDc * 4), make_float4(cwin.y, cwin.z, cwin.w, xnew));
            if (tile_wave) {
                quad_turn(hv);
                const unsigned at = (unsigned)((r0 + min(row, nr - 1)) * di + c0 + (cl & ~3)) * (kDs * 4) + 16 * (here(lane) & 3);
                if (mine) {
#pragma unroll
                    for (int k = 0; k < 4; k++) st_off(hst, at + k * (kDs * 4), hv[k]);
                }
            }
        };
        if (wave != 0) put_states();
        // ---- y of all channels: one wave looks for the flags
        if (wave == 0) {
            u64 r[GW];
            ok = xch_poll<GW>(xb, [&](int k) { return find(S::e3f, k); }, tagged, r);
            if (!ok && state == 0) state = kStepLost;
        }
        lds_barrier();   // D
        if (state) break;
        uint4 fy[KO];
        RowsWeight<KO, oc> pout;
        take_frags<KO>(yrows, fy);
        pout.take(wout);
        // ---- out_proj
        rows_product<T>(pout, fy, pre2);
        lds_barrier();   // E
        // ---- the residual; the next operand and the sums of squares of this workgroup's columns go out
        if (tid < 8 * kRows) {
            float sq = 0.0f;
            if (own) {
                const T a0 = (T)rows_sum<1>(pre2, y_place(orow), 2 * op), a1 = (T)rows_sum<1>(pre2, y_place(orow), 2 * op + 1);
                res0 += Store<T>::ld(&a0); res1 += Store<T>::ld(&a1);
                sq = fmaf(res0, res0, res1 * res1);
                if (more) {
                    const float2 nw = *reinterpret_cast<const float2 *>(small + sb.nw + 8 * op);
                    const int c = o0 + 2 * op;
                    put_pair(onext, operand_at(c, orow), half_pair<T>((T)(res0 * nw.x), (T)(res1 * nw.y)));
                }
            }
            sq = sum_of_8(sq);
            dma_wait();   // the sum says that the wave's columns are there
            if (op == 0 && orow < nr) xch_put(xb + S::e1 + (unsigned)(src * kRows + orow), sq, tag);
        }
        if (wave == 0) put_states();
        pin.take(smem);   // while the operand rows are on their way
        if (more) {
            cst += cst_l; hst += hst_l;
            if (tile_wave) {
                cwin = ld_off<float4>(cst, cell * (kDc * 4));
#pragma unroll
                for (int k = 0; k < 4; k++) hv[k] = ld_off<float4>(hst, cell * (kDs * 4) + 16 * k);
            }
        }
        take_sums(tag);
        orows += S::rows_bytes;
        lds_barrier();   // T
    }
    lds_barrier();
    // final norm of this workgroup's columns: f32, and once more in the storage type for a head
    const bool lost = state != 0;
    if (own) {
        const float inv = scale_of(orow);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int n = o0 + 2 * op + k;
            const float o = lost ? __uint_as_float(0x7fc00000u) : (k ? res1 : res0) * inv * a->norm_f[n];
            a->temporal[(size_t)(r0 + orow) * dm + n] = o;
            Store<T>::st((T *)a->temporal_t + (size_t)(r0 + orow) * dm + n, o);
        }
    }
    if (tid == 0) {
        if (state == kStepLost) {
            __hip_atomic_store(a->roll, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a->broken, (unsigned)kStepLost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (src == 0) *epoch = base + nl;   // every workgroup of the group has read it: each has published the last exchange
    }
}

// x_proj [di][xd] as [tile][k-step][lane][8], columns past xd zero; a thread writes 16 bytes.
__global__ __launch_bounds__(256) void pack_x_kernel(uint4 *__restrict__ dst, const uint16_t *__restrict__ x_proj, int di, int xd, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int lane = i & 63, ks = (i >> 6) % (di / 32), col = (i >> 6) / (di / 32) * 16 + (lane & 15), k = ks * 32 + 8 * (lane >> 4);
    unsigned w[4] = {0, 0, 0, 0};
    if (col < xd)
        for (int j = 0; j < 4; j++) w[j] = x_proj[(size_t)(k + 2 * j) * xd + col] | (unsigned)x_proj[(size_t)(k + 2 * j + 1) * xd + col] << 16;
    dst[i] = make_uint4(w[0], w[1], w[2], w[3]);
}

}  // namespace

// f<KI>() for the shape's KI, or `no`
template <typename F> static auto rows_shape(const ResidentArgs &a, F f, decltype(f(RowsShape<1>())) no) {
    if (a.dm % 256 || a.di != 2 * a.dm || a.ds != kDs || a.dc != kDc || a.dr != a.dm / 16 || a.xd != a.dr + 2 * kDs) return no;
    switch (a.dm / 256) {
        case 1: return f(RowsShape<1>());
        case 2: return f(RowsShape<2>());
        case 3: return f(RowsShape<3>());
        case 4: return f(RowsShape<4>());
        default: return no;
    }
}

// Eight rows to a group while there are places for the groups (24 layers of d_model 768, rows in 1, 2 and 4 groups: 8 rows 242 / 247 / 253 us a
// step, 16 rows 250 / 247 / 257, 32 rows - / 278 / 273).
constexpr int kRowsWanted = 8;
bool resident_rows_plan(ResidentArgs &a, int dtype) {
    if (dtype != MRS_BF16 && dtype != MRS_F16) return false;
    return rows_shape(a, [&](auto s) {
        using S = decltype(s);
        a.nc = S::nc; a.G = S::G; a.oc = S::oc;
        a.groups = (a.batch + kRowsWanted - 1) / kRowsWanted;
        if (a.groups > kRollMax / S::G) a.groups = kRollMax / S::G;
        a.rows = (a.batch + a.groups - 1) / a.groups;
        a.xch_stride = (S::words + kLineWords - 1) / kLineWords * kLineWords;
        return a.rows <= kRows;
    }, false);
}

size_t resident_rows_bytes(const ResidentArgs &a) { return rows_shape(a, [&](auto s) { return (size_t)a.groups * a.n_layers * decltype(s)::rows_bytes; }, 0); }
size_t resident_rows_layer_bytes(const ResidentArgs &a) { return rows_shape(a, [&](auto s) { return (size_t)decltype(s)::layer_bytes; }, 0); }
int launch_resident_rows_pack(hipStream_t st, const ResidentArgs &a, void *dst, const ResidentLayer &w) {
    ResidentArgs blocks = a;
    blocks.xd = 0;
    if (const int rc = launch_resident_pack(st, blocks, dst, w)) return rc;
    const int n = a.xd / 16 * (a.di / 32) * 64;
    hipLaunchKernelGGL(pack_x_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (uint4 *)((char *)dst + (size_t)a.G * layer_block(a.dm, a.di, a.nc, a.oc, 0, a.dr).bytes),
                       (const uint16_t *)w.x_proj, a.di, a.xd, n);
    return check_launch("pack_x_kernel");
}

template <typename T, int KI>
static int launch_rows_k(hipStream_t st, const ResidentArgs &a, const ResidentArgs *dev, const TokenRows &rows) {
    static const hipError_t attr = hipFuncSetAttribute((const void *)resident_rows_kernel<T, KI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kResLdsMax);
    if (attr != hipSuccess) return fail(MRS_E_HIP, "resident step: LDS size: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((resident_rows_kernel<T, KI>), dim3((unsigned)(RowsShape<KI>::G * a.groups)), dim3(kResThreads), (size_t)RowsShape<KI>::lds, st, dev, rows);
    return check_launch("resident_rows_kernel");
}

int launch_resident_rows(hipStream_t st, int dtype, const ResidentArgs &a, const ResidentArgs *dev, const TokenRows &rows) {
    ResidentArgs plan = a;
    const bool ok = resident_rows_plan(plan, dtype) && plan.G == a.G && a.groups >= 1 && a.groups <= a.batch && a.groups * a.G <= kRollMax &&
                    a.rows == (a.batch + a.groups - 1) / a.groups && a.rows <= kRows && a.xch_stride == plan.xch_stride && a.n_layers >= 1 && a.weights && a.norm_w && a.input &&
                    a.xch && a.epoch && a.roll && a.broken && a.temporal && a.temporal_t && a.rows_buf && dev;
    if (!ok) return fail(MRS_E_SHAPE, "resident step: shape outside the route (d_model=%d d_inner=%d d_state=%d workgroups=%d rows=%d)", a.dm, a.di, a.ds, a.G, a.rows);
    return rows_shape(a, [&](auto s) {
        constexpr int KI = decltype(s)::dm / 256;
        return dtype == MRS_BF16 ? launch_rows_k<bf16_t, KI>(st, a, dev, rows) : launch_rows_k<f16_t, KI>(st, a, dev, rows);
    }, MRS_E_SHAPE);
}

}  // namespace mrs
