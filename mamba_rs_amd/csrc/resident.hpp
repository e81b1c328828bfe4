// Building blocks of the resident decode steps (resident_step.hip, resident_rows.hip, resident_m3_step.hip, resident_m3_row.hip): one launch walks
// the whole network, G workgroups share every layer's columns, and what a layer's phases need from each other travels through memory while the workgroups stay
// on the chip.
//
// Exchange: a value and the number of the layer it belongs to (its tag) are one 64-bit word, stored and polled with relaxed
// agent-scope atomics.  The word is its own flag, so a phase costs one store and one load to the coherence point of the
// chip -- no counter, no fence, no cache write-back.  Measured for all-to-all exchanges of 768 values, two workgroup
// barriers included: 1.3 us among 32 workgroups, 1.5 among 64, 1.8 among 128, 2.4 among 256 (a counter barrier over 256
// workgroups: 2.3 to 3.7 us and the data still to be fetched; a kernel boundary in a graph: about 4 us).
// A layer's exchanges form a cycle (residual -> x_proj shares -> y -> residual), and a workgroup writes its words of the next layer only
// behind the last of them, the residual, which everybody takes from everybody and puts out after its last read of the others: one buffer
// per exchange is enough, also for one that only a few workgroups read (resident_rows.hip: u).
//
// A launch begins with a roll call (RollCall): no workgroup stores anything but exchange words and operand rows before all of them are on
// the chip; states and output rows it does not touch.
// Ordinary kernels that hold the compute units delay it.  If the units do not come free within the wait the caller set, the launch is
// called off as a whole: the states are what they were, the output rows become NaN, `broken` (host memory) is raised, and launches
// queued behind it leave at once.  After the roll call a wait is over when its neighbours have done their part; those waits are
// bounded as well (kSpinLimit polls, about two seconds), and a workgroup that gives up there leaves the states unfinished.
#pragma once
#include "common.hpp"
#include "mfma_tiles.hpp"

namespace mrs {

typedef unsigned long long u64;
constexpr unsigned kSpinLimit = 1u << 21;

// The roll call, by one of the waves that bring weights.  roll[0]: a launch was called off or lost, its successors do not begin;
// roll[1]: number of the launch; roll[2 + its parity]: the ruling; behind kRollHead words, one per workgroup: the number of the last
// launch it has answered, plus one.  A workgroup goes on when it has seen all answers and, after that, no ruling against it.  One that has
// waited `wait` polls (one to two microseconds each) in vain first puts kDoubt there and then looks at the answers again: whoever went on
// without seeing the doubt had seen all of them before it, so they are all there now and it goes on as well; otherwise the launch
// is called off.  So all workgroups take the same way, also those that get a place only when others have left.  A wait of 0 calls off
// without an answer.
// The answers are read while the first exchange is waited for: a step takes about a microsecond longer for it (four layers of
// d_model 256 at eight rows 30.8 -> 31.5 us, of d_model 64 at 32 25.8 -> 27.0; 24 layers of d_model 768 within what builds differ by).
// As a count on one word, added to and polled by 256 workgroups: 4 to 11 us.
constexpr int kRollCall = -1;   // a workgroup's state: the roll call, 0 under way, or a ResidentFault
constexpr unsigned kDoubt = 1, kGo = 2, kOff = 3;
struct RollCall {
    unsigned *roll, *broken;
    unsigned all, wait, number;
    static __device__ __forceinline__ unsigned get(const unsigned *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    static __device__ __forceinline__ void put(unsigned *p, unsigned v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    static __device__ __forceinline__ void done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }   // what was asked for before is there, what is asked for next comes after
    __device__ __forceinline__ int answer() {
        const u64 head = __hip_atomic_load(reinterpret_cast<u64 *>(roll), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        number = __builtin_amdgcn_readfirstlane((unsigned)(head >> 32));
        if (__builtin_amdgcn_readfirstlane((unsigned)head)) return kStepCalledOff;
        if (wait && (threadIdx.x & 63) == 0) put(roll + kRollHead + blockIdx.x, number + 1u);
        return kRollCall;
    }
    __device__ __forceinline__ bool answered() const {
        bool have = true;
        unsigned r[kRollMax / 64];
#pragma unroll
        for (int k = 0; k < kRollMax / 64; k++) r[k] = get(roll + kRollHead + min((unsigned)(k * 64) + (threadIdx.x & 63u), all - 1u));
#pragma unroll
        for (int k = 0; k < kRollMax / 64; k++) have = have && r[k] == number + 1u;
        const bool yes = __all(have);
        done();
        return yes;
    }
    __device__ __forceinline__ int outcome() const {
        unsigned *ruling = roll + 2 + (number & 1u);
        const bool first = (threadIdx.x & 63) == 0;
#pragma unroll 1
        for (unsigned spins = 0;; spins++) {
            const bool yes = answered();
            const unsigned v = __builtin_amdgcn_readfirstlane(get(ruling));
            if (v == kOff) return kStepCalledOff;
            if (yes && v != kDoubt) break;
            if (v == 0 && spins >= wait) {
                unsigned none = 0;
                const bool mine = first && __hip_atomic_compare_exchange_strong(ruling, &none, kDoubt, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (!__any(mine)) continue;
                done();
                const bool go = answered();
                if (first) {
                    if (!go) {
                        put(roll, 1u);
                        __hip_atomic_store(broken, (unsigned)kStepCalledOff, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
                    put(ruling, go ? kGo : kOff);
                }
                if (go) break;
                return kStepCalledOff;
            }
            __builtin_amdgcn_s_sleep(4);
        }
        if (blockIdx.x == 0 && first) {   // everybody has read the number: the next launch's
            put(roll + 2 + ((number + 1u) & 1u), 0u);
            put(roll + 1, number + 1u);
        }
        return 0;
    }
};

__device__ __forceinline__ void xch_put(u64 *p, float v, unsigned tag) {
    __hip_atomic_store(p, ((u64)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 xch_get(const u64 *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ __forceinline__ int here_s(int v) { asm volatile("" : "+s"(v)); return v; }   // the same for a value all lanes share

// A table that no kernel writes, read through the scalar cache.
template <typename V> using scalar_table = const __attribute__((address_space(4))) V *;
template <typename V> __device__ __forceinline__ scalar_table<V> as_table(const V *p) { return (scalar_table<V>)(uintptr_t)p; }

// What a step's row starts from, for the prologues: begin(in, taken) with in(i) its element i, from the input buffer, or (taken) from the embedding table.
// The table's row is one more load to wait for, about 1.5 us where a kernel in front that gathers the rows is 4.9 in a graph.
template <typename T, class F> __device__ __forceinline__ void with_input_row(const float *input, const TokenRows &t, int row, int dm, F begin) {
    if (t.embed) {
        const bool zero = t.finished && t.finished[row];
        const T *e = (const T *)t.embed + (size_t)min(max(t.tokens[row], 0), t.vocab - 1) * dm;
        begin([=](int i) { const float v = Store<T>::ld(e + i); return zero ? 0.0f : v; }, true);
    } else {
        const float *in = input + (size_t)row * dm;
        begin([=](int i) { return in[i]; }, false);
    }
}

// Sum over the 16 lanes of a DPP row, in every lane of it.
__device__ __forceinline__ float row16_sum(float v) {
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x128, 0xf, 0xf, false));   // row_ror:8
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x124, 0xf, 0xf, false));
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x122, 0xf, 0xf, false));
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x121, 0xf, 0xf, false));
    return v;
}

// Keeps what is computed from v inside the scope it is used in: a layer loop's many lane-dependent addresses would otherwise all
// be hoisted out of it, and spilled.
__device__ __forceinline__ int here(int v) { asm volatile("" : "+v"(v)); return v; }

// base (the same for the whole wave) + a 32-bit lane offset in bytes: one scalar base and one vector register per access
template <typename V> __device__ __forceinline__ V ld_off(const void *base, unsigned bytes) {
    return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + bytes);
}

// One wave copies the 1 KB pieces first, first + step, ... below `pieces` of contiguous memory to LDS byte address `to` (both 16-byte
// aligned) without passing through registers.  The compiler's wait counting does not see it: dma_wait() by the same wave and a
// workgroup barrier come before the data is read.  Requests are spaced (s_sleep: 64 clocks each): a compute unit's requests are
// served in order, and a burst of them would stand in front of the exchange's stores and polls.
template <int SLEEP = 1> __device__ __forceinline__ void dma_to_lds(unsigned to, const void *from, int first, int pieces, int step, bool stream = false) {
    const u64 at = (u64)(uintptr_t)from;   // the same for the whole wave
    const u64 src = (u64)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)at) | (u64)(unsigned)__builtin_amdgcn_readfirstlane((unsigned)(at >> 32)) << 32;
    const unsigned lane16 = (unsigned)(threadIdx.x & 63) * 16u, dst0 = __builtin_amdgcn_readfirstlane(to);
    if (stream) {
#pragma unroll 1
        for (int i = first; i < pieces; i += step) {
            const unsigned voff = (unsigned)i * 1024u + lane16, dst = dst0 + (unsigned)i * 1024u;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_sleep %3" ::"s"(dst), "v"(voff), "s"(src), "n"(SLEEP) : "m0", "memory");
        }
        return;
    }
#pragma unroll 1
    for (int i = first; i < pieces; i += step) {
        const unsigned voff = (unsigned)i * 1024u + lane16, dst = dst0 + (unsigned)i * 1024u;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_sleep %3" ::"s"(dst), "v"(voff), "s"(src), "n"(SLEEP) : "m0", "memory");
    }
}
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Over the eight groups of eight lanes: the sum of the lanes 8 apart, in every lane.
__device__ __forceinline__ float groups_sum(float v) {
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x128, 0xf, 0xf, false));   // row_ror:8
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);   // rows 0 0 2 2 and 1 1 3 3
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);   // the lower half twice and the upper half twice
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
// Lane 7's value of the eight lanes this one belongs to.
__device__ __forceinline__ unsigned last_of_8(unsigned v) {
    const unsigned q = __builtin_amdgcn_mov_dpp(v, 0xff, 0xf, 0xf, true);           // quad_perm [3,3,3,3]: in the upper four
    return __builtin_amdgcn_update_dpp(q, q, 0x141, 0xf, 0x5, false);               // row_half_mirror into the lower four (banks 0 and 2)
}

// Sum over a wave, in lane 63.
__device__ __forceinline__ float wave_sum_last(float v) {
    v = row16_sum(v);
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1 and 3
    v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2 and 3
    return v;
}

constexpr int kComputeWaves = 8, kCompute = 64 * kComputeWaves;
constexpr int kResThreads = kCompute + 4 * 64;   // eight waves compute, four bring weights
__host__ __device__ constexpr int up1k(int n) { return (n + 1023) & ~1023; }
constexpr size_t kResLdsMax = 160 * 1024 - 256;

// Fourteen f32 in a line of eight exchange words: seven words of two each, where the lowest mantissa bit carries the parity of the layer's
// tag (a line is rewritten every layer, so what is not of this layer is of the one before), and one of those bits with the tag.
// The values arrive whole, infinities and NaN as well.  (Two whole f32 per word with a "not there" value that its writer puts back, so
// that every word is written twice a layer: 24 layers of d_model 1024 9 to 14 us slower.)
constexpr int kLineVals = 14;
__device__ __forceinline__ u64 pair_word(float a, float b, unsigned tag) {
    const unsigned x = (__float_as_uint(a) & ~1u) | (tag & 1u), y = (__float_as_uint(b) & ~1u) | (tag & 1u);
    return (u64)y << 32 | x;
}
__device__ __forceinline__ unsigned with_bit(unsigned half, unsigned bits, int at) { return (half & ~1u) | (bits >> at & 1u); }
// Two 16-bit values and the tag.
template <typename T> __device__ __forceinline__ u64 half_pair_word(T a, T b, unsigned tag) {
    return (u64)tag << 32 | (unsigned)__builtin_bit_cast(uint16_t, b) << 16 | __builtin_bit_cast(uint16_t, a);
}
__device__ __forceinline__ void xch_put_word(u64 *p, u64 w) { __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Polls the KU words base[idx(0)] .. base[idx(KU - 1)] until ready(word) holds for all of them.  False when the wait was given up; a
// step's first exchange (state() its workgroup's) waits as long as the roll call is not over.
struct NoRollCall { __device__ __forceinline__ int operator()() const { return 0; } };
template <int KU, class IDX, class READY, class STATE = NoRollCall>
__device__ __forceinline__ bool xch_poll(const u64 *base, IDX idx, READY ready, u64 (&r)[KU], STATE state = STATE()) {
    for (unsigned spins = 0; spins <= kSpinLimit; spins++) {
        bool have = true;
#pragma unroll
        for (int u = 0; u < KU; u++) r[u] = xch_get(base + idx(u));
#pragma unroll
        for (int u = 0; u < KU; u++) have &= ready(r[u]);   // (no branch per word)
        if (have) return true;
        if ((spins & 63u) == 63u) {
            const int s = state();
            if (s > 0) return false;
            if (s == kRollCall) spins = 0;
        }
    }
    return false;
}

// One row's product on the matrix cores, K split over the computing waves in steps of 32 (step wave, wave + 8, ...; at most KS per wave):
// the weight in LDS as [K / 8][cols][8], 16 CT columns of it (columns past `cols` repeat the last one), x in LDS.  take() brings this
// wave's pieces of the weight into registers, which can be done while x is still on its way; run() leaves this wave's share of
// column c in out[wave * 16 CT + c].  Only one of the sixteen rows of a matrix instruction is used: what the product costs is
// bringing the weights from LDS.
template <typename T, int KS, int CT> struct RowProduct {
    uint4 w[KS][CT];
    __device__ __forceinline__ void take(const T *wl, int cols, int ksteps, int ct) {
        const int t = here(threadIdx.x), l = t & 63, n = l & 15, kg = l >> 4, w0 = __builtin_amdgcn_readfirstlane(t >> 6);
        const uint4 *wp = reinterpret_cast<const uint4 *>(wl);
#pragma unroll
        for (int c = 0; c < CT; c++)
            if (c < ct) {
                const int col = min(c * 16 + n, cols - 1);
#pragma unroll
                for (int s = 0; s < KS; s++)
                    if (w0 + kComputeWaves * s < ksteps) w[s][c] = wp[(unsigned)(((w0 + kComputeWaves * s) * 4 + kg) * cols + col)];
            }
    }
    __device__ __forceinline__ void run(const T *x, int ksteps, int ct, float *out) const {
        const int t = here(threadIdx.x), l = t & 63, kg = l >> 4, w0 = __builtin_amdgcn_readfirstlane(t >> 6);
        v4f acc[CT];
#pragma unroll
        for (int c = 0; c < CT; c++) acc[c] = (v4f){0.f, 0.f, 0.f, 0.f};
        uint4 a[KS];
#pragma unroll
        for (int s = 0; s < KS; s++)
            if (w0 + kComputeWaves * s < ksteps) a[s] = reinterpret_cast<const uint4 *>(x)[(w0 + kComputeWaves * s) * 4 + kg];   // the same for all rows
#pragma unroll
        for (int s = 0; s < KS; s++)
            if (w0 + kComputeWaves * s < ksteps) {
#pragma unroll
                for (int c = 0; c < CT; c++) acc[c] = Mma32<T>::mma(a[s], w[s][c], acc[c]);
            }
        if (l < 16) {   // row 0, column l % 16 is register 0 of lanes 0 to 15
#pragma unroll
            for (int c = 0; c < CT; c++)
                if (c < ct) out[w0 * 16 * ct + c * 16 + l] = acc[c][0];
        }
    }
};
// the waves' shares of column c, added in wave order
__device__ __forceinline__ float row_sum(const float *out, int cols16, int c) {
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kComputeWaves; w++) v += out[w * cols16 + c];
    return v;
}

// The waves that bring weights: wave 10 out_proj's, the others in_proj's, 11 the small block as well.  Each buffer is refilled as
// soon as the phase that reads it is over and is there before the barrier in front of its next use; requests go out
// where the computing waves wait for their neighbours (a wave that is still issuing them holds up a barrier).  A layer has five
// barriers, behind: 1 in_proj, 2 the second exchange, 3 y, 4 out_proj, 5 the next operand.
struct WeightFeed {
    const char *blk;              // this workgroup's block of layer 0: in_proj part, out_proj part, small block, each of whole kilobytes
    size_t next;                  // ... to that of the next layer
    unsigned win, wout, small;    // LDS byte addresses; the small blocks of two layers lie one after the other
    int out, small_at, small_bytes;   // offsets in the block
    int cached;                   // layers whose weights come through the last cache; the others' are read past it
};
__device__ __forceinline__ void bring_weights(const WeightFeed f, int wave, int nl, int &state, RollCall call) {
    const char *blk = f.blk;
    const bool first = (threadIdx.x & 63) == 0, out_wave = wave == 10, small_wave = wave == 11;
    const int iw = wave == 11 ? 2 : wave - 8, cached = f.cached, in_pieces = f.out >> 10, in_mid = in_pieces / 2, out_pieces = (f.small_at - f.out) >> 10;
    auto bring_in = [&](const char *p, int l, int from, int to) { dma_to_lds(f.win, p, from + iw, to, 3, l >= cached); };
    auto bring_out = [&](const char *p, int l) { dma_to_lds(f.wout, p + f.out, 0, out_pieces, 1, l >= cached); };
    auto bring_small = [&](const char *p, int l) { dma_to_lds(f.small + (l & 1) * f.small_bytes, p + f.small_at, 0, f.small_bytes >> 10, 1); };
    if (out_wave) {
        const int s = call.answer();
        if (first) state = s;
        bring_out(blk, 0);
    } else bring_in(blk, 0, 0, in_pieces);
    if (small_wave) bring_small(blk, 0);
    if (!out_wave) dma_wait();
    lds_barrier();   // layer 0's row is there
#pragma unroll 1
    for (int l = 0; l < nl; l++) {
        const bool more = l + 1 < nl;
        blk += f.next;   // the next layer's
        lds_barrier();   // 1
        if (small_wave && more) bring_small(blk, l + 1);
        if (!out_wave && more) bring_in(blk, l + 1, 0, in_mid);
        if (out_wave) {
            if (l == 0 && state == kRollCall) {
                const int s = call.outcome();
                if (first) state = s;
            }
            dma_wait();
        }
        lds_barrier();   // 2
        if (state) return;
        if (!out_wave && more) bring_in(blk, l + 1, in_mid, in_pieces);
        lds_barrier();   // 3
        if (state) return;
        if (!out_wave) dma_wait();
        lds_barrier();   // 4
        if (out_wave && more) bring_out(blk, l + 1);
        lds_barrier();   // 5
        if (state) return;
    }
}

// The parts of a layer that both networks share.
__device__ __forceinline__ float inv_rms(float s, int dm, float eps) {
    float rms = sqrtf(s / (float)dm + eps);
    if (!isfinite(rms) || rms < 1e-20f) rms = 1.0f;   // the reference's finite guard (kernels/norms.cu:58-61)
    return 1.0f / rms;
}

// y of all channels (exchange 3) to LDS.
template <typename T> __device__ __forceinline__ bool take_y(const u64 *e3, int di, unsigned tag, T *ys) {
    bool ok = true;
#pragma unroll 1
    for (int i0 = 0; i0 < di >> 1; i0 += 2 * kCompute) {
        const int t = i0 + here(threadIdx.x), n3 = di >> 1;
        if (t < n3) {
            u64 r[2];
            ok = ok && xch_poll<2>(e3, [&](int u) { return (unsigned)(u == 1 && t + kCompute < n3 ? t + kCompute : t); },
                                   [&](u64 w) { return (unsigned)(w >> 32) == tag; }, r);
            *reinterpret_cast<unsigned *>(ys + 2 * t) = (unsigned)r[0];
            if (t + kCompute < n3) *reinterpret_cast<unsigned *>(ys + 2 * (t + kCompute)) = (unsigned)r[1];
        }
    }
    return ok;
}

// out_proj's columns join the residual stream (thread p holds columns o0 + 2 p and + 1); the next layer's operand (next_nw: its norm
// weight for these columns, null behind the last layer) and the workgroup's sum of squares go out.
template <typename T>
__device__ __forceinline__ void put_operand(const float *pre2, int oc, int o0, int src, const float *next_nw, u64 *e1, u64 *e1s, unsigned tag, float &res0, float &res1) {
    if (here(threadIdx.x) >= 16) return;
    const int p = here(threadIdx.x);
    float sq = 0.0f;
    if (p < oc >> 1) {
        const T a0 = (T)row_sum(pre2, 16, 2 * p), a1 = (T)row_sum(pre2, 16, 2 * p + 1);
        res0 += Store<T>::ld(&a0); res1 += Store<T>::ld(&a1);
        sq = fmaf(res0, res0, res1 * res1);
        if (next_nw) {
            const float2 nw = *reinterpret_cast<const float2 *>(next_nw + 2 * p);
            xch_put_word(e1 + (unsigned)((o0 >> 1) + p), half_pair_word<T>((T)(res0 * nw.x), (T)(res1 * nw.y), tag));
        }
    }
    sq = row16_sum(sq);
    if (p == 0) xch_put(e1s + src, sq, tag);
}

// Exchange 1: the next operand row to xs (if there is one), the row's scale to *inv.
template <typename T>
__device__ __forceinline__ bool take_operand(const u64 *e1, const u64 *e1s, int G, int dm, float eps, unsigned tag, bool more, T *xs, float *inv) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const auto tagged = [&](u64 w) { return (unsigned)(w >> 32) == tag; };
    bool ok = true;
    if (wave == kComputeWaves - 1) {
        // the workgroups' sums of squares: this wave, in workgroup order within a lane
        float s = 0.0f;
#pragma unroll 1
        for (int g = here(lane); g < G; g += 64) {
            u64 r[1];
            ok = ok && xch_poll<1>(e1s, [&](int) { return (unsigned)g; }, tagged, r);
            s += __uint_as_float((unsigned)r[0]);
        }
        s = wave_sum_last(s);
        if (lane == 63) *inv = inv_rms(s, dm, eps);
    }
    if (more) {
#pragma unroll 1
        for (int t = here(threadIdx.x); t < dm >> 1; t += kCompute) {
            u64 r[1];
            ok = ok && xch_poll<1>(e1, [&](int) { return (unsigned)t; }, tagged, r);
            *reinterpret_cast<unsigned *>(xs + 2 * t) = (unsigned)r[0];
        }
    }
    return ok;
}

}  // namespace mrs
