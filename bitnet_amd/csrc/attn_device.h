// Device parts of the attention kernels: bf16 helpers, and the decode step's work on one block of
// cache rows, on the waves' results and on the splits' records.  Shared, so that the attention of a
// decode step gives the same bits from every kernel that contains it.
#ifndef BITNET_AMD_ATTN_DEVICE_H
#define BITNET_AMD_ATTN_DEVICE_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "bitlinear_device.h"

namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kHeadDim = 128;

__device__ __forceinline__ float bf16f(uint32_t bits16) { return __uint_as_float(bits16 << 16); }
// fp32 -> bf16, round to nearest even, NaN kept
__device__ __forceinline__ uint16_t to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) { return f32x2_to_bf16x2(lo, hi); }
// of lane ^ 16 and lane ^ 32 as well: a value from all four rows of 16 lanes, without a trip through LDS
template <class Op>
__device__ __forceinline__ float over_rows(float v, Op op) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

constexpr int kDfRecUnits = kHeadDim + 2;  // record of one (sequence, kv head, split, head): 128 outputs, maximum, sum,
                                            // each an 8-byte unit (value, tag of the call that wrote it)
constexpr int kDfSpinLimit = 1 << 16;       // polls of the merging workgroup before it gives up
constexpr int kDfMaxSplits = 16;
constexpr int kDfMaxWaves = 8;
// Cache policy of a poll: sc1 alone, device scope.  (sc0 and sc1 together, system scope, which is also what a volatile
// access becomes, has been seen to give a line that this XCD wrote earlier in the launch although another XCD had
// written it since.)  These loads are ordinary ones for the compiler, which takes them out of a loop that writes
// nothing: poll_again() in front of them keeps them in.
constexpr int kPollPolicy = 16;
__device__ __forceinline__ void poll_again() { asm volatile("" ::: "memory"); }
constexpr float kDfScale = 0.08838834764831845f;            // 128^-0.5
constexpr float kDfC2 = kDfScale * 1.4426950408889634f;     // * log2(e): the softmax runs in base 2

// A wave's running softmax over its blocks: for head c = lane % 16, unnormalised outputs
// 32 g4 + 8 j + t in o_acc[t][j] (g4 = lane / 16), maximum in raw score units, and this lane's share of the sum.
struct DfState {
    v4f o_acc[8];
    float m_run = -INFINITY, l_run = 0.0f;
    __device__ __forceinline__ DfState() {
#pragma unroll
        for (int t = 0; t < 8; ++t) o_acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
};

// What follows is bound by the number of instructions of one wave, not by memory: V rows are turned where a caller waits
// anyway, masks and the new row only in the block that needs them, results stored as the registers hold them, and the
// caller's own record added behind the others without selects (a step of 12 sequences at 512 positions, where
// attn_decode_flash_kernel runs 30 times: 1440 -> 1348 us).

// A block of 32 cache rows (positions 32 blk ..) as loaded: kb[bi][kk], dims 32 kk + 8 g4 .. of row 16 bi + c; vb[jj], dims
// 8 c .. of row 4 g4 + (jj & 3) + 16 (jj >> 2).  df_block wants the V rows turned (df_turn); in the block of the new
// token's position p the rows behind p are cleared in front of that, and row p, which is not in the cache yet, is put in:
// k by df_new_key, v (dims 8 c ..) by df_block.

// V rows behind the position: their probability is zero, but whatever the cache holds there (it may never have been
// written) must not reach the product as 0 x NaN
__device__ __forceinline__ void df_clear(v4u (&vb)[8], int p, int lane) {
    const int last = (p & 31) - 4 * (lane >> 4);
#pragma unroll
    for (int jj = 0; jj < 8; ++jj)
        if ((jj & 3) + (jj >> 2) * 16 > last) vb[jj] = v4u{0u, 0u, 0u, 0u};
}
// vb[t] becomes the operand of output dims 8 j + t of P.V: eight rows of one dim per lane
__device__ __forceinline__ void df_turn(v4u (&vb)[8]) {
    v4u va[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
        va[t].x = __builtin_amdgcn_perm(vb[1][t >> 1], vb[0][t >> 1], sel);
        va[t].y = __builtin_amdgcn_perm(vb[3][t >> 1], vb[2][t >> 1], sel);
        va[t].z = __builtin_amdgcn_perm(vb[5][t >> 1], vb[4][t >> 1], sel);
        va[t].w = __builtin_amdgcn_perm(vb[7][t >> 1], vb[6][t >> 1], sel);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) vb[t] = va[t];
}

// Row p of K, from LDS
__device__ __forceinline__ void df_new_key(v4u (&kb)[2][4], const uint16_t* knew, int p, int lane) {
    const int c = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
        if (bi * 16 + c == (p & 31)) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) kb[bi][kk] = *(const v4u*)(knew + kk * 32 + g4 * 8);
        }
}
// Row p of V: of turned rows it is a half-word of one of four words, in the operands of a quarter of the lanes.  All words
// are permuted, by selectors that leave the others as they are: branches on the word copy registers.
__device__ __forceinline__ void df_new_value(v4u (&va)[8], const v4u& vn, int p, int lane) {
    const int r = p & 31;
    const bool mine = lane >> 4 == ((r >> 2) & 3);
    const uint32_t even = r & 1 ? 0x05040100u : 0x03020504u, odd = r & 1 ? 0x07060100u : 0x03020706u, as_it_is = 0x03020100u;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const bool here = w == ((r & 3) + (r >> 4) * 4) >> 1;
        const uint32_t sel[2] = {mine ? (here ? even : as_it_is) : as_it_is, mine ? (here ? odd : as_it_is) : as_it_is};
#pragma unroll
        for (int t = 0; t < 8; ++t) va[t][w] = __builtin_amdgcn_perm(vn[t >> 1], va[t][w], sel[t & 1]);
    }
}

// Scores, softmax and P.V of one block for the heads in the columns of qa
__device__ __forceinline__ void df_block(const v4u (&kb)[2][4], v4u (&va)[8], const v4u& vn, const v8bf (&qa)[4], int blk, int p, int lane,
                                         DfState& st) {
    const int g4 = lane >> 4;
    float sc[8];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi) {
        v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, kb[bi][kk]), qa[kk], acc, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[bi * 4 + j] = acc[j];
    }
    if (blk == p >> 5) {  // (every other block is in the cache, and visible, as a whole)
        df_new_value(va, vn, p, lane);  // (while the matrix pipe has the scores)
        const int last = (p & 31) - 4 * g4;
#pragma unroll
        for (int i = 0; i < 8; ++i) sc[i] = (i & 3) + (i >> 2) * 16 <= last ? sc[i] : -INFINITY;
    }
    float mx = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7])));
    mx = over_rows(mx, [](float a, float b) { return fmaxf(a, b); });
    const float m_new = fmaxf(st.m_run, mx);  // finite: the block's first row is visible (32 blk <= p)
    const float m2 = m_new * kDfC2;
    float pr[8], psum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        pr[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], kDfC2, -m2));
        psum += pr[i];
    }
    // (nothing to rescale before the wave's first block)
    if (__builtin_amdgcn_ballot_w64(m_new != st.m_run && st.m_run > -INFINITY) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(__builtin_fmaf(st.m_run, kDfC2, -m2));
        st.l_run *= alpha;
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) st.o_acc[t][j] *= alpha;
    }
    st.m_run = m_new;
    st.l_run += psum;
    v4u pw;
    pw.x = pack_bf16x2(pr[0], pr[1]);
    pw.y = pack_bf16x2(pr[2], pr[3]);
    pw.z = pack_bf16x2(pr[4], pr[5]);
    pw.w = pack_bf16x2(pr[6], pr[7]);
    const v8bf pb = __builtin_bit_cast(v8bf, pw);
#pragma unroll
    for (int t = 0; t < 8; ++t) st.o_acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, va[t]), pb, st.o_acc[t], 0, 0, 0);
}

// A head's outputs of one wave in LDS: output 32 g4 + 8 j + t at 32 g4 + 4 t + j, as a lane has them in registers; the rows
// four banks apart, so that the heads' stores do not meet in one
constexpr int kDfOutRow = kHeadDim + 4;
// The wave's result for head c (lanes c < G) -> LDS: maximum (-inf, with a sum of 0, for a wave without visible
// positions), sum over its positions, 32 outputs per lane
template <int G>
__device__ __forceinline__ void df_wave_result(const DfState& st, int lane, float (*part_o)[kDfOutRow], float* part_m,
                                               float* part_l) {
    const int c = lane & 15, g4 = lane >> 4;
    const float l_tot = over_rows(st.l_run, [](float a, float b) { return a + b; });
    if (c < G) {
        if (g4 == 0) {
            part_m[c] = st.m_run;
            part_l[c] = l_tot;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) *(v4f*)&part_o[c][32 * g4 + 4 * t] = st.o_acc[t];
    }
}

// Outputs 2 lane and 2 lane + 1 of one head, unnormalised, with the maximum and the sum of exponentials
struct DfPartial {
    float o0, o1, mx, l;
};

// One head over the results of N waves, of which the first n are there (ALL: every one)
template <int G, int N, bool ALL>
__device__ __forceinline__ DfPartial df_combine(const float (*part_o)[G][kDfOutRow], const float (*part_m)[G],
                                                const float (*part_l)[G], int hh, int n, int lane) {
    DfPartial h = {0.0f, 0.0f, -INFINITY, 0.0f};
    static_assert(N == 4 || N == 8, "one or two batches");
    const int at0 = 32 * (lane >> 4) + 8 * (lane & 3) + ((lane >> 2) & 3);  // of output 2 lane; 2 lane + 1 four behind
    float m[N], l[N], o0[N], o1[N];
    // all values are requested together: left to itself the compiler waits for one wave's before the next one's.
    // A wave without visible positions adds nothing (by selects: branches cost more than what they skip).
    auto request = [&](int k0) {
#pragma unroll
        for (int k = k0; k < k0 + 4; ++k) {
            const int at = ALL || k < n ? k : 0;
            m[k] = part_m[at][hh];
            l[k] = part_l[at][hh];
            o0[k] = part_o[at][hh][at0];
            o1[k] = part_o[at][hh][at0 + 4];
        }
#pragma unroll
        for (int k = k0; k < k0 + 4; ++k) {
            asm volatile("" : "+v"(m[k]), "+v"(l[k]), "+v"(o0[k]), "+v"(o1[k]));
            h.mx = fmaxf(h.mx, m[k]);
        }
    };
    auto add = [&](int k0) {
#pragma unroll
        for (int k = k0; k < k0 + 4; ++k) {
            const float w = (ALL || k < n) && l[k] > 0.0f ? __builtin_amdgcn_exp2f((m[k] - h.mx) * kDfC2) : 0.0f;
            h.l += l[k] * w;
            h.o0 += w * o0[k];
            h.o1 += w * o1[k];
        }
    };
    request(0);
    if (N > 4) request(4);
    add(0);
    if (N > 4) add(4);
    return h;
}

// A split's record of one head; the maximum is kept in units of the scaled scores
__device__ __forceinline__ void df_store_record(unsigned long long* r, unsigned long long tag, const DfPartial& h, int lane) {
    // two units a store, past the L2 (16-byte stores, device scope)
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(r, 0, kDfRecUnits * 8, 0x00020000);
    const unsigned t = (unsigned)(tag >> 32);
    __builtin_amdgcn_raw_buffer_store_b128(v4u{__float_as_uint(h.o0), t, __float_as_uint(h.o1), t}, rsrc, lane * 16, 0, kPollPolicy);
    if (lane == 0)
        __builtin_amdgcn_raw_buffer_store_b128(v4u{__float_as_uint(h.mx * kDfScale), t, __float_as_uint(h.l), t}, rsrc, kHeadDim * 8, 0, kPollPolicy);
}

// One head over the splits' records rec[split][G][kDfRecUnits], eight splits at a time: all units of a batch are
// requested together and requested again while one of them still carries another tag, at most spin_limit times.  The
// last split's record is `own`, the caller's: it is not stored at all (loads wait for the acknowledgement of stores in
// front of them, 1.3 us).
template <int G>
__device__ __forceinline__ DfPartial df_merge(const unsigned long long* rec, int nact, int hh, unsigned long long tag,
                                              const DfPartial& own, int lane, int spin_limit, bool& gave_up) {
    constexpr int kBatch = 8;
    DfPartial h = {0.0f, 0.0f, -INFINITY, 0.0f};
    // device-coherent 16-byte loads (two units each; a unit is whole, whatever the other holds) with scalar offsets
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)rec, 0, nact * G * kDfRecUnits * 8, 0x00020000);
    const unsigned want = (unsigned)(tag >> 32);
    for (int k0 = 0; k0 < nact; k0 += kBatch) {
        v4u ml[kBatch], oo[kBatch];  // (maximum, tag, sum, tag), (output 2 lane, tag, output 2 lane + 1, tag)
#pragma unroll
        for (int k = 0; k < kBatch; ++k) ml[k] = oo[k] = v4u{0u, 0u, 0u, 0u};
        bool complete = false;
        for (int spin = 0; spin < spin_limit; ++spin) {
            poll_again();
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int at = ((k0 + k < nact - 1 ? k0 + k : 0) * G + hh) * (kDfRecUnits * 8);
                ml[k] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, kHeadDim * 8, at, kPollPolicy);
                oo[k] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane * 16, at, kPollPolicy);
            }
            unsigned other = 0;
#pragma unroll
            for (int k = 0; k < kBatch; ++k) other |= (ml[k].y ^ want) | (ml[k].w ^ want) | (oo[k].y ^ want) | (oo[k].w ^ want);
            asm("" : "+v"(other));  // (as one word: 32 compares of their own take 500 cycles)
            if (__builtin_amdgcn_ballot_w64(other != 0) == 0) {
                complete = true;
                break;
            }
        }
        gave_up = gave_up || !complete;
        // records here (those behind them repeat the first split's, which does not change a maximum); then, in the
        // last batch, the caller's
        const int there = nact - 1 - k0;
        const float own_mx = own.mx * kDfScale;
        float bm = there < kBatch ? fmaxf(h.mx, own_mx) : h.mx;
#pragma unroll
        for (int k = 0; k < kBatch; ++k) bm = fmaxf(bm, __uint_as_float(ml[k].x));
        if (k0) {
            const float wold = h.l > 0.0f ? __expf(h.mx - bm) : 0.0f;
            h.l *= wold;
            h.o0 *= wold;
            h.o1 *= wold;
        }
        h.mx = bm;
        float w[kBatch + 1];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) w[k] = __uint_as_float(ml[k].z) > 0.0f ? __expf(__uint_as_float(ml[k].x) - bm) : 0.0f;
        w[kBatch] = own.l > 0.0f ? __expf(own_mx - bm) : 0.0f;
        auto add = [&](float l, float o0, float o1, float w) {
            h.l += l * w;
            h.o0 += w * o0;
            h.o1 += w * o1;
        };
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
            if (k < there) add(__uint_as_float(ml[k].z), __uint_as_float(oo[k].x), __uint_as_float(oo[k].z), w[k]);
        if (there < kBatch) add(own.l, own.o0, own.o1, w[kBatch]);
    }
    return h;
}

}  // namespace

#endif
