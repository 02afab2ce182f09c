// Nucleus sampling of the next token (gpu/sample_utils.py:9-33 and gpu/generate.py:270-277 of the
// reference: softmax of logits / temperature, cut to the top_p nucleus, one draw) from the LM head's
// logits, which carry bf16 values.
//
// The draw is the exponential race over the sorted distribution: the rank r with the largest
// p[r] / noise[r] wins.  Written as sort, cumulative sum and race over the whole vocabulary that is some
// twenty passes over 128256 values (330 us a step at one sequence).  bf16 logits take only a few thousand
// different values, though, and tokens of one value are sorted by index, so the sorted distribution is
// known from a histogram alone: rank r belongs to the value whose cumulative counts enclose it, and only
// the winner's rank is turned into a token.  Three launches, 32 us together, bound by chains of LDS and
// memory latencies (one row of 128256 logits; at four rows the same):
//   1. histograms of 16 pieces of the vocabulary, 5 us
//   2. their sum, its masses and the nucleus's end; the race over one piece of the ranks per workgroup, 18 us
//   3. the winner: value and place among the tokens of that value -> piece -> token, 9 us
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "bitlinear_device.h"
#include "bitnet_decoder_ops.h"

namespace {

constexpr int kSpPieces = 16;
constexpr int kSpThreads = 1024;
// Levels of a magnitude: 0 for all below the bf16 bits `low` (zero included), then one per bf16 value, the last one for
// all from 64 powers of two above on.  Buckets in the order of the ranks: positive values downwards, level 0, negative
// ones.  `low` follows the temperature (sp_low): values below 2^-24 of it have the probability of zero, to half a unit
// in the last place of a float, and two different ones of 2^40 of it and more are so far apart that the lower one's
// probability is zero, so of an outermost bucket only the largest value counts (SpPiece).  All buckets of bf16, 65281,
// are more than the LDS holds.
constexpr int kSpLevels = 64 << 7;
constexpr int kSpBuckets = 2 * kSpLevels + 1;
constexpr int kSpRow = (kSpBuckets + 7) & ~7;

struct SpPiece {
    int first, last;  // its buckets in use (last < first: none)
    int key, count;   // the largest value (as sp_key) and how often it is there, where `first` is an outermost bucket
};
struct SpWinner {
    float v;
    int r, bucket, place;
};
static_assert(sizeof(SpWinner) == 16 && sizeof(SpPiece) == 16, "one 16-byte store");

// bf16 bits of the power of two at least 2^-25 and less than 2^-24 of the temperature; 1, above zero alone, for the smallest
int sp_low(float temperature) {
    int e;
    frexpf(temperature, &e);  // 2^(e - 1) <= temperature < 2^e
    const int low = (127 + e - 1 - 24) << 7;
    return low < 1 ? 1 : low;
}
__device__ __forceinline__ int sp_bucket(float logit, int low) {
    const int b = (int)(__float_as_uint(logit) >> 16), mag = b & 0x7fff;
    const int level = mag < low ? 0 : min(mag - low + 1, kSpLevels);
    return b & 0x8000 ? kSpLevels + level : kSpLevels - level;
}
// (an outermost bucket's value of least magnitude)
__device__ __forceinline__ float sp_value(int bucket, int low) {
    const int d = bucket - kSpLevels, level = d < 0 ? -d : d;
    const float m = level ? __uint_as_float((unsigned)(low + level - 1) << 16) : 0.0f;
    return d > 0 ? -m : m;
}
__device__ __forceinline__ bool sp_outermost(int bucket) { return bucket == 0 || bucket == kSpBuckets - 1; }
// order of bf16 values within a bucket of several, larger first
__device__ __forceinline__ int sp_key(float logit) {
    const int b = (int)(__float_as_uint(logit) >> 16), mag = b & 0x7fff;
    return b & 0x8000 ? 0x7fff + mag : 0x7fff - mag;  // both zeros: 0x7fff
}
__device__ __forceinline__ float sp_value_of_key(int key) {
    return key > 0x7fff ? -__uint_as_float((unsigned)(key - 0x7fff) << 16) : __uint_as_float((unsigned)(0x7fff - key) << 16);
}
__device__ __forceinline__ int sp_piece_size(int V) { return ((V + kSpPieces - 1) / kSpPieces + 3) & ~3; }

__global__ __launch_bounds__(kSpThreads) void sample_count_kernel(const float* __restrict__ logits, uint16_t* __restrict__ counts,
                                                                  SpPiece* __restrict__ pieces, int* __restrict__ error, int low, int V) {
    __shared__ __attribute__((aligned(16))) unsigned hist[kSpRow];
    __shared__ int first, last, top_key, top_count;
    const int tid = threadIdx.x, piece = blockIdx.x, row = blockIdx.y;
    for (int i = tid; i < kSpRow / 4; i += kSpThreads) ((v4u*)hist)[i] = v4u{0u, 0u, 0u, 0u};
    if (tid == 0) first = kSpBuckets, last = -1, top_key = 0xffff, top_count = 0;
    __syncthreads();
    const int size = sp_piece_size(V), lo = piece * size, hi = min(V, lo + size);
    const float* x = logits + (size_t)row * V;
    int mn = kSpBuckets, mx = -1;
    bool bad = false;
    for (int i = lo + tid; i < hi; i += kSpThreads) {
        const float v = x[i];
        bad = bad || !(v < INFINITY);  // a NaN or an infinite logit: no distribution
        const int b = sp_bucket(v, low);
        mn = min(mn, b);
        mx = max(mx, b);
        atomicAdd(&hist[b], 1u);
    }
#pragma unroll
    for (int off = 32; off; off >>= 1) {
        mn = min(mn, __shfl_xor(mn, off));
        mx = max(mx, __shfl_xor(mx, off));
    }
    if ((tid & 63) == 0) {
        atomicMin(&first, mn);
        atomicMax(&last, mx);
    }
    if (bad) __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __syncthreads();
    if (sp_outermost(first)) {  // rare; the same for all threads
        for (int i = lo + tid; i < hi; i += kSpThreads)
            if (sp_bucket(x[i], low) == first) atomicMin(&top_key, sp_key(x[i]));
        __syncthreads();
        for (int i = lo + tid; i < hi; i += kSpThreads)
            if (sp_key(x[i]) == top_key) atomicAdd(&top_count, 1);
        __syncthreads();
    }
    if (tid == 0) pieces[row * kSpPieces + piece] = SpPiece{first, last, top_key, top_count};
    uint32_t* to = (uint32_t*)(counts + (size_t)(row * kSpPieces + piece) * kSpRow);
    for (int i = (first >> 1) + tid; 2 * i <= last; i += kSpThreads) to[i] = hist[2 * i] | hist[2 * i + 1] << 16;
}

__global__ __launch_bounds__(kSpThreads) void sample_race_kernel(const uint16_t* __restrict__ counts, const SpPiece* __restrict__ pieces,
                                                                 const float* __restrict__ noise, SpWinner* __restrict__ winners,
                                                                 int* __restrict__ error, float inv_t, float top_p, int low, int V) {
    __shared__ __attribute__((aligned(16))) unsigned before[kSpRow];  // counts, then ranks in front of a bucket
    __shared__ __attribute__((aligned(16))) float odds[kSpRow];       // exp(its logit - the largest)
    __shared__ double wave_mass[kSpThreads / 64];
    __shared__ unsigned wave_count[kSpThreads / 64];
    __shared__ SpWinner best[kSpThreads / 64];
    __shared__ int kept;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, piece = blockIdx.x, row = blockIdx.y;
    SpPiece p[kSpPieces];
    int first = kSpBuckets, last = -1;
#pragma unroll
    for (int k = 0; k < kSpPieces; ++k) {
        p[k] = pieces[row * kSpPieces + k];
        first = min(first, p[k].first);
        last = max(last, p[k].last);
    }
    // of an outermost bucket the largest value's tokens are in the draw, as its first ranks, and no other token is
    int key = 0xffff, largest_count = 0;
    if (sp_outermost(first)) {
#pragma unroll
        for (int k = 0; k < kSpPieces; ++k) key = min(key, p[k].first == first ? p[k].key : 0xffff);
#pragma unroll
        for (int k = 0; k < kSpPieces; ++k) largest_count += p[k].first == first && p[k].key == key ? p[k].count : 0;
    }
    const float m = sp_value(first, low) * inv_t;
    const uint32_t* c = (const uint32_t*)(counts + (size_t)row * kSpPieces * kSpRow);
    const int base = first & ~1, n = last + 1 - base;
    for (int i = tid; 2 * i < n; i += kSpThreads) {
        const int at = base + 2 * i;
        unsigned lo = 0, hi = 0;
        uint32_t v[kSpPieces];  // all requested together, whatever a piece wrote: behind conditions they came one by one, 33 us
#pragma unroll
        for (int k = 0; k < kSpPieces; ++k) v[k] = c[(size_t)k * (kSpRow / 2) + (at >> 1)];
#pragma unroll
        for (int k = 0; k < kSpPieces; ++k) {
            const bool used = at + 1 >= p[k].first && at <= p[k].last;
            lo += used ? v[k] & 0xffffu : 0u;
            hi += used ? v[k] >> 16 : 0u;
        }
        before[2 * i] = lo;
        before[2 * i + 1] = hi;
        odds[2 * i] = at < first ? 0.0f : expf(sp_value(at, low) * inv_t - m);  // (a value above the largest: infinite)
        odds[2 * i + 1] = expf(sp_value(at + 1, low) * inv_t - m);
    }
    if (tid == 0) {
        kept = largest_count ? largest_count : V;
        // the largest logit over the temperature is no number: all are -inf, or it overflows
        const float largest = (largest_count ? sp_value_of_key(key) : sp_value(first, low)) * inv_t;
        if (!(fabsf(largest) < INFINITY)) __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
    if (largest_count) {
        if (tid == 0) before[first - base] = (unsigned)largest_count;
        __syncthreads();
    }
    // every thread a run of buckets
    const int per = (n + kSpThreads - 1) / kSpThreads, at0 = min(n, tid * per), at1 = min(n, at0 + per);
    unsigned count = 0;
    double mass = 0.0;
    for (int i = at0; i < at1; ++i) {
        const unsigned k = before[i];
        count += k;
        mass += (double)k * (double)odds[i];
    }
    unsigned count_in = count;
    double mass_in = mass;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned oc = __shfl_up(count_in, off);
        const double om = __shfl_up(mass_in, off);
        if (lane >= off) {
            count_in += oc;
            mass_in += om;
        }
    }
    if (lane == 63) {
        wave_count[wave] = count_in;
        wave_mass[wave] = mass_in;
    }
    __syncthreads();
    unsigned ranks = count_in - count;
    double sum = mass_in - mass, total = 0.0;
#pragma unroll
    for (int w = 0; w < kSpThreads / 64; ++w) {
        const unsigned wc = wave_count[w];
        const double wm = wave_mass[w];
        ranks += w < wave ? wc : 0u;
        sum += w < wave ? wm : 0.0;
        total += wm;
    }
    // A rank stays while the mass in front of it is at most top_p: the first one that does not ends the nucleus
    const double limit = (double)top_p * total;
    int end = V;
    for (int i = at0; i < at1; ++i) {
        const unsigned k = before[i];
        before[i] = ranks;
        const double e = (double)odds[i], behind = sum + (double)k * e;
        if (end == V && k && behind > limit) {
            const double stay = sum > limit ? 0.0 : floor((limit - sum) / e) + 1.0;
            if (stay < (double)k) end = (int)(ranks + (unsigned)stay);
        }
        sum = behind;
        ranks += k;
    }
#pragma unroll
    for (int off = 32; off; off >>= 1) end = min(end, __shfl_xor(end, off));
    if (lane == 0) atomicMin(&kept, end);
    __syncthreads();
    const int size = sp_piece_size(V), lo = piece * size, hi = min(kept, lo + size);
    const float* q = noise + (size_t)row * V;
    int top = 1;
    while (2 * top < n) top *= 2;
    float bv = -1.0f;
    int br = 0x7fffffff, bb = -1;  // value, rank, bucket (less base)
    // the last bucket with at most r ranks in front of it, for four ranks at a time: the steps depend on each other
    constexpr int kU = 4;
    for (int r0 = lo + tid; r0 < hi; r0 += kU * kSpThreads) {
        float z[kU];
        int a[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            z[u] = q[min(r0 + u * kSpThreads, V - 1)];
            a[u] = 0;
        }
        for (int step = top; step; step >>= 1) {
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int at = a[u] + step;
                const int in_front = (int)before[min(at, n - 1)];  // (not behind a condition: a branch per step and rank)
                a[u] = (at < n) & (in_front <= r0 + u * kSpThreads) ? at : a[u];
            }
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const float v = odds[a[u]] / z[u];
            if (r0 + u * kSpThreads < hi && v > bv) {
                bv = v;
                br = r0 + u * kSpThreads;
                bb = a[u];
            }
        }
    }
    auto reduce = [&](int lanes) {
        for (int off = lanes / 2; off; off >>= 1) {
            const float v = __shfl_xor(bv, off);
            const int r = __shfl_xor(br, off), k = __shfl_xor(bb, off);
            if (v > bv || (v == bv && r < br)) {
                bv = v;
                br = r;
                bb = k;
            }
        }
    };
    reduce(64);
    if (lane == 0) best[wave] = SpWinner{bv, br, bb, 0};
    __syncthreads();
    if (wave) return;
    const SpWinner w = best[lane & (kSpThreads / 64 - 1)];
    bv = w.v;
    br = w.r;
    bb = w.bucket;
    reduce(kSpThreads / 64);
    if (lane == 0) {
        SpWinner out = {bv, br, -1, 0};
        if (bv >= 0.0f) {
            out.bucket = base + bb;
            out.place = br - (int)before[bb];
        }
        winners[row * kSpPieces + piece] = out;
    }
}

// The token at `place` (by index) among those of [lo, hi) that `is` accepts -> *found.  A wave takes a run of them,
// 64 at a time and eight loads together (a thread's own run of eight is eight loads one after another).
template <class Is>
__device__ __forceinline__ void sp_pick(const float* x, int lo, int hi, int place, int* wave_count, int* found, Is is) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per = (hi - lo + kSpThreads - 1) / kSpThreads * 64, at0 = lo + wave * per, at1 = min(hi, at0 + per);
    constexpr int kU = 8;
    auto masks = [&](int at, unsigned long long (&m)[kU]) {
        float v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) v[u] = x[max(0, min(at + u * 64 + lane, hi - 1))];
#pragma unroll
        for (int u = 0; u < kU; ++u) m[u] = __builtin_amdgcn_ballot_w64(is(v[u]) & (at + u * 64 + lane < at1));
    };
    unsigned long long m[kU];
    int count = 0;
    for (int at = at0; at < at1; at += kU * 64) {
        masks(at, m);
#pragma unroll
        for (int u = 0; u < kU; ++u) count += __popcll(m[u]);
    }
    if (lane == 0) wave_count[wave] = count;
    __syncthreads();
    int from = 0;
#pragma unroll
    for (int w = 0; w < kSpThreads / 64; ++w) from += w < wave ? wave_count[w] : 0;
    if (place >= from && place < from + count) {
        for (int at = at0; at < at1; at += kU * 64) {
            if (per > kU * 64) masks(at, m);
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int before = from + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m[u] >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m[u], 0u));
                if (((m[u] >> lane) & 1u) && before == place) *found = at + u * 64 + lane;
                from += __popcll(m[u]);
            }
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(kSpThreads) void sample_token_kernel(const float* __restrict__ logits, const uint16_t* __restrict__ counts,
                                                                  const SpPiece* __restrict__ pieces, const SpWinner* __restrict__ winners,
                                                                  int64_t* __restrict__ token_out, int64_t* __restrict__ next_input,
                                                                  int64_t* __restrict__ positions, int64_t* __restrict__ history_row,
                                                                  int* __restrict__ error, int low, int V) {
    __shared__ int wave_count[kSpThreads / 64];
    __shared__ unsigned hist[256];
    __shared__ int found;
    const int tid = threadIdx.x, row = blockIdx.x;
    SpWinner w = winners[row * kSpPieces];
#pragma unroll
    for (int k = 1; k < kSpPieces; ++k) {
        const SpWinner o = winners[row * kSpPieces + k];
        if (o.v > w.v) w = o;  // (ties: the lower ranks come first)
    }
    if (tid == 0) found = -1;
    const float* x = logits + (size_t)row * V;
    int place = w.place;
    __syncthreads();
    if (w.bucket >= 0 && !sp_outermost(w.bucket) && w.bucket != kSpLevels) {  // tokens of one value
        const int size = sp_piece_size(V);
        unsigned n[kSpPieces];
#pragma unroll
        for (int k = 0; k < kSpPieces; ++k) {
            const SpPiece p = pieces[row * kSpPieces + k];
            n[k] = w.bucket >= p.first && w.bucket <= p.last ? counts[(size_t)(row * kSpPieces + k) * kSpRow + w.bucket] : 0u;
        }
        int piece = kSpPieces;
#pragma unroll
        for (int k = 0; k < kSpPieces; ++k)
            if (piece == kSpPieces) {
                if (place < (int)n[k]) piece = k;
                else place -= (int)n[k];
            }
        const int lo = min(V, piece * size);
        sp_pick(x, lo, min(V, lo + size), place, wave_count, &found, [&](float v) { return sp_bucket(v, low) == w.bucket; });
    } else if (w.bucket >= 0) {
        // a bucket of several values: the value by its high byte and then its low one, over the whole row (rare)
        int prefix = 0, mask = 0;
        for (int shift = 8; shift >= 0; shift -= 8) {
            if (tid < 256) hist[tid] = 0;
            __syncthreads();
            for (int i = tid; i < V; i += kSpThreads) {
                const int key = sp_key(x[i]);
                if (sp_bucket(x[i], low) == w.bucket && ((key ^ prefix) & mask) == 0) atomicAdd(&hist[(key >> shift) & 255], 1u);
            }
            __syncthreads();
            int digit = 0;
            while (digit < 255 && place >= (int)hist[digit]) place -= (int)hist[digit++];
            prefix |= digit << shift;
            mask |= 255 << shift;
            __syncthreads();
        }
        sp_pick(x, 0, V, place, wave_count, &found, [&](float v) { return sp_bucket(v, low) == w.bucket && sp_key(v) == prefix; });
    }
    if (tid == 0) {
        const int64_t token = found >= 0 ? found : 0;
        if (found < 0) __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        token_out[row] = token;
        if (next_input) next_input[row] = token;
        if (positions) positions[row] += 1;
        if (history_row) history_row[row] = token;
    }
}

size_t up16(size_t v) { return (v + 15) & ~(size_t)15; }

}  // namespace

extern "C" {

long long bitnet_top_p_workspace_bytes(int B, int V) {
    if (B < 1 || B > 65535 || V < 1 || V > 65535 * kSpPieces - 64) return -1;
    return (long long)(up16((size_t)B * kSpPieces * kSpRow * 2) + up16((size_t)B * kSpPieces * sizeof(SpPiece)) +
                       (size_t)B * kSpPieces * sizeof(SpWinner));
}

int bitnet_top_p_sample(const float* logits, const float* noise, void* workspace, float temperature, float top_p,
                        int64_t* token_out, int64_t* next_input, int64_t* positions, int64_t* history_row, int* error, int B, int V,
                        void* stream) {
    const float inv_t = 1.0f / temperature;
    const int low = sp_low(temperature);
    if (bitnet_top_p_workspace_bytes(B, V) < 0 || !(inv_t > 0.0f) || !(inv_t < INFINITY) || !(top_p >= 0.0f)) return 1;
    if (!logits || !noise || !workspace || !token_out || !error) return 2;
    if ((uintptr_t)workspace & 15u) return 1;
    unsigned char* ws = (unsigned char*)workspace;
    uint16_t* counts = (uint16_t*)ws;
    ws += up16((size_t)B * kSpPieces * kSpRow * 2);
    SpPiece* pieces = (SpPiece*)ws;
    SpWinner* winners = (SpWinner*)(ws + up16((size_t)B * kSpPieces * sizeof(SpPiece)));
    const hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(sample_count_kernel, dim3(kSpPieces, B), dim3(kSpThreads), 0, s, logits, counts, pieces, error, low, V);
    hipLaunchKernelGGL(sample_race_kernel, dim3(kSpPieces, B), dim3(kSpThreads), 0, s, counts, pieces, noise, winners, error, inv_t, top_p, low, V);
    hipLaunchKernelGGL(sample_token_kernel, dim3(B), dim3(kSpThreads), 0, s, logits, counts, pieces, winners, token_out, next_input,
                       positions, history_row, error, low, V);
    return hipGetLastError() == hipSuccess ? 0 : 3;
}

}  // extern "C"
