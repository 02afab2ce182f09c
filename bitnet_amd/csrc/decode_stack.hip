// The decoder layers of one decode step (gpu/model.py:214-245 of the reference, one new token per
// sequence, every layer) in ONE kernel.
//
// What bounds a decode step as a chain of launches is the boundary between two of them, not bytes: at
// one sequence of the 2B decoder a layer is 17 MB of weights, 3.4 us at the card's copy rate, and five
// dependent kernels, 26 us -- each pays for its launch (1.6 us, empty), for the trip of the activations
// to memory and back (1.2 us) and for the weights' latency that nothing before it could hide.  Here one
// workgroup per CU stays for the whole step.  A product's weights are in LDS before its activations
// exist, and outputs go to their readers directly: every value is written through to memory once, and
// readers poll for the values themselves.  Nobody waits for an acknowledgement, a counter or a launch;
// such a hand-over measures 1.4 us, readers' barrier included.  30 layers at 512 positions, us:
//   sequences            1     2     3     4     8
//   launches           755   875  1000  1070  1060
//   this kernel        462   569   634   662   724
// (the launches with the attention's earlier instructions.)  What is left of a phase (of a layer's 15 us at one sequence the
// five take about 2.7, 3.9, 2, 3.5 and 2.9): 1 to 1.3 us from the arrival of a task's inputs to its outputs (the exchange between
// the waves 0.3, norm and quantizer 0.3 to 0.5, products 0.1 to 0.3, the epilogue 0.3), the hand-over, and the last workgroup
// being late; the weights are not waited for.  Polls are as dense as pays: two in flight cost 7 %, a pause of 0.2 us behind
// each 1 %; outputs stored as 4 or 16 bytes a lane instead of two 1 %.
// Up to two tokens every workgroup of a product normalises and quantizes the rows by itself, between their
// arrival and its matrix instructions.  That part grows with the tokens (three: 1120 us).  Beyond two, one
// task per token does it for all and publishes int8 rows, which are the matrix instructions' operand as they
// lie in memory: one more hand-over, but a product's own work hardly depends on the tokens.  The rows stand
// with 64 values of every token side by side, so that one 16-byte load of a wave covers 16 / tokens k-steps
// of all of them and its lines are whole, and the first complete read may hit the XCD's L2 (eight sequences:
// 816 us with a row per token and every read past L2).
//
// Hand-over buffers.  Every (layer, step) has buffers of its own, in two sets that alternate between
// launches; a launch fills the other set with a value that no result can have (bf16 0xffff, a NaN that
// results are kept from having), so "not that value" means "written".  No buffer is reused within a
// launch, so nothing has to be protected from being overwritten.
//
// Tasks.  A layer is a list of tasks in dependency order -- 32 output rows of wqkv, or one (sequence,
// kv head, split) of the attention, or 32 gated outputs of w13 ... -- and all layers are one long list.
// A task needs only tasks in front of it.  Workgroups take the next task of the list whenever they
// finish one ("ticket mode"): every task in front of a taken one is finished or in the hands of a
// running workgroup, so the kernel ends with any number of workgroups resident, whatever else occupies
// the GPU.  Taking tickets costs one contended atomic per task; once all workgroups of the grid have
// been seen to run (each takes its first ticket from the counter, and the one that takes ticket
// grid - 1 says so), no counter is needed: ticket t + grid follows ticket t ("static mode").  Exactly
// one of the modes is decided per launch, by compare-and-swap; who waits for the decision longer than
// some 50 us decides for ticket mode.
//
// Waves.  Between the arrival of its inputs and its outputs a task is bound by the instructions that its
// SIMDs issue and by chains of dependent ones, so there is ONE computing wave per SIMD: a second one
// repeats every step that is not per element (reductions, scales, addresses), and eight waves of 320
// values took 1.9 us where four of 640 take 1.3.  A fifth wave takes the tickets, looks up what a task
// consists of and brings its weights into LDS, in pieces of 1 KB without a register in between, up to
// two tasks ahead; its waits for memory hold up nobody.  Loads of 4 bytes per lane, the width in which
// MFMA operands unpack, cost an instruction each and took 2-3 us a task when the computing waves did
// them.  The waves tell each other what they have done by numbers in LDS: the hardware's barrier would
// have to include the wave that fetches.
//
// The arithmetic is that of the kernels a step consists of otherwise, value for value (the shared
// definitions are in bitlinear_device.h and attn_device.h): both give the same bits.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <type_traits>

#include "attn_device.h"
#include "bitlinear_device.h"
#include "bitlinear_hip.h"
#include "bitlinear_probes.h"
#include "bitnet_decoder_ops.h"
#include "host_util.h"

namespace {

constexpr int kStWaves = 4;
constexpr int kStLanes = kStWaves * 64;   // of the computing waves
constexpr int kStThreads = kStLanes + 64;  // and the wave that fetches
// 64-wide k-steps per wave of a product over the model width (up to 2560) and over the feed-forward width (up to 6912).
// The registers set them: a w13 task keeps four row blocks of 10 steps as expanded operands, 160 of the 256 that
// one computing wave per SIMD has next to the wave that fetches, and a w2 task one block of 27 and its slice of the input.
// Narrower models take the same steps, multiplied with zeros: the exchanges and hand-overs, which are what a phase
// costs, do not get shorter with them.  Wider ones and more than kStMaxTokens take the kernels per layer.
constexpr int kStUpwD = 10;
constexpr int kStUpwF = 27;
constexpr int kStDirect = 2;      // tokens up to which every product task quantizes its input (see above)
constexpr int kStMaxTokens = 8;
constexpr int kStMaxG = 8;        // query heads per kv head
constexpr int kStSpinLimit = 1 << 19;   // polls (0.7 us each) before a wait gives up
constexpr int kStModePolls = 64;        // polls before the mode is decided without all workgroups
constexpr int kSc1 = kPollPolicy;       // device-coherent accesses
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef int v2i __attribute__((ext_vector_type(2)));
// Four int8 of quantized rows that mean "not written": as an int the least there is, so that the minimum of a lane's words
// shows whether one of them is that.  Its last byte, -128, comes only where the row's maximum is not finite: a finite one leaves
// |x| * scale below 127.5, an infinite one makes the scale 0, codes of 0 and, of infinity * 0, -128, and beside a NaN
// finite values are clamped.  A slice of such a row says in its record that it is written (kComplete).
constexpr int kUnsetBytes = INT32_MIN;
constexpr unsigned kComplete = 1u << 30;
constexpr int kLookEvery = 32;          // polls between two looks at that, a power of two
constexpr int kBeyond = 0x7ffffff0;     // an offset behind every descriptor: reads as zero, no access

// one product of one layer
struct StackEntry {
    const uint32_t* w;
    const uint16_t* norm;  // of the RMSNorm in front
    const uint16_t* ws;
    uint16_t* ck;  // entry 0: the layer's cache
    uint16_t* cv;
    float eps;
    int slot_rows;  // weight-scale runs, as bitlinear_scale_runs gives them
    uint32_t slot_map;
    int pad[3];
};
static_assert(sizeof(StackEntry) == 64, "the host writes eight 8-byte words per entry");

// control words, each on a 128-byte line of its own
struct StackControl {
    unsigned counter, pad0[31];  // next ticket; back to zero at the end of a launch
    unsigned mode, pad1[31];     // (launch + 1) * 2 + (1: ticket mode), once decided
    unsigned done, pad2[31];     // workgroups that have finished; back to zero at the end
    unsigned launch, pad3[31];   // launches so far
    int error, pad4[31];
};

struct StackArgs {
    const __attribute__((address_space(4))) StackEntry* entries;  // [layer][4]: wqkv, wo, w13, w2
    unsigned char* ws;
    // The first layer's input: sequence m's row of h_in is m, or, with tokens, its token's; the rotation's factors likewise: in
    // row m or the position's of cos and sin, whose rows are `factors` apart.  Against a kernel that collects them in front of
    // this one (4.6 us, most of them launch) a step of one sequence takes 578 us instead of 583 at 512 positions, of eight 843
    // instead of 848: the lookups and a row from memory stay.
    const uint16_t* h_in;
    uint16_t* h_out;
    const __attribute__((address_space(4))) int64_t* positions;
    const __attribute__((address_space(4))) int64_t* tokens;
    const float *cos, *sin;
    int in_rows, factors;
    int n_layers, B, dim, ffn, n_heads, n_kv, group, S, n_splits, attn_waves, spin_limit;  // group: query heads per kv head
    int ends[9];  // cumulative task counts of a layer's phases
    // a set: bytes per layer and offsets in it; behind the bf16 values of all layers (set_values bytes) the quantized rows
    int f_layer, f_o, f_ha, f_g, f_hb, f_rec;
    int f_bytes;  // quantized rows per layer
    int set_values, set_bytes;
    long long sets;     // offset of the first set in the workspace
    long long records;  // offset of the attention records
    float inv_dim, inv_ffn;  // correctly rounded reciprocals
};
typedef const __attribute__((address_space(4))) StackArgs* StackArgsPtr;  // the kernel's argument block

// wqkv (two 16-row blocks a task), attention, wo (one block), w13 (two pairs of blocks, gated), w2 (one block); in front
// of each product, beyond kStDirect tokens, its input rows normalised and quantized, one token a task
enum Phase { kQ1 = 0, kP1, kAttn, kQ3, kP3, kQ4, kP4, kQ5, kP5 };

struct Work {
    int layer, ph, first, idx;  // idx: the task's number in its phase, whose first task is number `first` of the layer
};

// A wave's share of a row: UPW 64-wide k-steps, 64 lanes x 8 consecutive values per 512, and what is left of the
// share as T values per lane
template <int UPW>
struct Slice {
    static constexpr int kValues = UPW * 64;
    static constexpr int kFull = kValues / 512;
    static constexpr int kRest = kValues % 512;
    static constexpr int T = kRest == 0 ? 0 : kRest <= 128 ? 2 : kRest <= 256 ? 4 : 8;
    static constexpr int kVec = kFull + (T ? 1 : 0);
};
constexpr int kStMaxVec = Slice<kStUpwF>::kVec;
static_assert(Slice<kStUpwF>::kVec == 4 && Slice<kStUpwD>::kVec == 2, "registers below");

constexpr int kStWordBytes = 40 * 1024;  // a task's packed words: at most four row blocks of 2560, or one of 6912
constexpr int kStBuffers = 3;

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

struct Waiter {
    int limit;
    int* error;
    bool dead;  // a wait gave up: nothing is waited for any more, so that the grid drains
    __device__ __forceinline__ bool give_up(int spin) {
        if (spin + 1 < limit &&
            ((spin & 1023) != 1023 || uniform(__hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0))
            return false;
        if ((threadIdx.x & 63) == 0) __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        dead = true;
        return true;
    }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00020000);
}
// both halves of a packed bf16 pair, in the upper half-word: the larger tells whether one is 0xffff
__device__ __forceinline__ unsigned unset_max(unsigned m, unsigned d) { return max(m, max(d, d << 16)); }
__device__ __forceinline__ bool is_unset(unsigned m) { return m >= 0xffff0000u; }
__device__ __forceinline__ void publish16(uint16_t* p, uint16_t v) {
    __hip_atomic_store(p, v < 0xfffeu ? v : (uint16_t)0xfffeu, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ unsigned lds_address(const void* p) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// LDS words that one wave writes while another looks: as LDS accesses (a volatile access through a generic pointer
// stays a flat one, and waits for all of the wave's memory loads as well)
template <class T>
__device__ __forceinline__ T lds_look(const T& v) {
    return *(const volatile __attribute__((address_space(3))) T*)&v;
}
template <class T>
__device__ __forceinline__ void lds_put(T& to, T v) {
    *(volatile __attribute__((address_space(3))) T*)&to = v;
}
// 16 bytes per lane straight into LDS, lane l's at `to` + 16 l.  In assembly, so that the compiler does not hold it
// against every later LDS access (it would wait for the load in front of the next one): what makes the words
// visible is that the fetching wave waits for its loads before it says in LDS that they are there.  The compiler does
// not look into the string for hazards, so the wait state between a write of m0 and a load that takes its LDS address
// from it is in it; a vector instruction's write of the descriptor needs five in front of the first load (settled).
__device__ __forceinline__ void load_to_lds(v4u rsrc, unsigned to, int voffset, int soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :
                 : "s"(to), "v"(voffset), "s"(rsrc), "s"(soffset)
                 : "memory");  // (m0 is the compiler's scratch: it sets it in front of each use of its own)
}
__device__ __forceinline__ void settled(v4u& rsrc) { asm volatile("s_nop 4" : "+s"(rsrc)); }
// The results of the IEEE operations they replace, bit for bit, from the hardware's approximations and one correction step
// each, at a third of the instructions.  Not on all arguments (compared one by one by decode_stack_math_kernel): 1 / x
// from 2^-126 to 2^126, which holds every maximum that leaves the scale's reciprocal a normal number; 1 / sqrt(x) from
// 2^-102 on, below which no caller's eps lies; x / width from 2^-115 on, below which the quotient vanishes next to such an eps;
// a sum over a scale as long as its first approximation does not overflow, scales of 2^-108 and more.  NaNs stay NaNs.
__device__ __forceinline__ float quotient(float x, float by, float inv) {  // inv: 1 / by, correctly rounded
    const float q = x * inv;
    return __builtin_fmaf(__builtin_fmaf(-q, by, x), inv, q);
}
__device__ __forceinline__ float divide(float x, float by, float inv) {
    const float q = x * inv;
    return q < INFINITY ? quotient(x, by, inv) : q;
}
__device__ __forceinline__ float reciprocal(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return x == INFINITY ? 0.0f : __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ float reciprocal_sqrt(float x) {  // 1 / sqrt(x), both rounded
    const float y = __builtin_amdgcn_rsqf(x);
    const float s0 = x * y;
    const float s = __builtin_fmaf(__builtin_fmaf(-s0, s0, x), 0.5f * y, s0);
    return x == INFINITY ? 0.0f : reciprocal(s);
}
// reductions that leave the wave's result in lane 63: rows of 16 by lane permutes, then row 0 into 1 and 2 into 3,
// then those two
template <class T, class Op>
__device__ __forceinline__ T wave_reduce_last(T v, Op op) {
    auto step = [&](auto ctrl, auto rows) {
        constexpr int C = decltype(ctrl)::value, R = decltype(rows)::value;
        if constexpr (sizeof(T) == 8) {
            const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
            const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, C, R, 0xF, R == 0xF);
            const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), C, R, 0xF, R == 0xF);
            v = op(v, __builtin_bit_cast(T, (unsigned long long)hi << 32 | lo));
        } else {
            v = op(v, __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), C, R, 0xF, R == 0xF)));
        }
    };
    step(std::integral_constant<int, 0xB1>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, 0x4E>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, 0x141>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, 0x140>{}, std::integral_constant<int, 0xF>{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});  // row_bcast15
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});  // row_bcast31
    return v;
}
// a packed pair of bf16 at a time: what sumsq8 and norm8 do for four
__device__ __forceinline__ double sumsq2(uint32_t d) {
    const float lo = __uint_as_float(d << 16), hi = __uint_as_float(d & 0xffff0000u);
    return (double)(lo * lo) + (double)(hi * hi);
}
__device__ __forceinline__ uint32_t norm2(uint32_t d, uint32_t w, float rstd) {
    return f32x2_to_bf16x2(__uint_as_float(d << 16) * rstd * __uint_as_float(w << 16),
                           __uint_as_float(d & 0xffff0000u) * rstd * __uint_as_float(w & 0xffff0000u));
}
// the larger of `top` and the magnitudes of a pair's products with its weights
__device__ __forceinline__ float product_max2(uint32_t d, uint32_t w, float top) {
    return fmaxf(fmaxf(fabsf(__uint_as_float(d << 16) * __uint_as_float(w << 16)),
                       fabsf(__uint_as_float(d & 0xffff0000u) * __uint_as_float(w & 0xffff0000u))), top);
}
__device__ __forceinline__ uint32_t quant2(uint32_t d, float s) {  // two bytes
    return __builtin_amdgcn_perm(quant_low_byte<0>(d & 0xffff0000u, s), quant_low_byte<0>(d << 16, s), 0x0c0c0400u);
}

// A quantized row's scale (bf16 bits) and a word for each of its four waves' slices: a set top bit is "not written",
// kComplete "the whole slice is in memory, also where it looks unset"
struct RowRecord {
    unsigned slice[4];
    unsigned scale, pad[3];
};
static_assert(sizeof(RowRecord) == 32 && kStWaves == 4, "one 16-byte and one 4-byte load");

// what the waves of an attention task found, in the task's words buffer
struct WaveResults {
    float o[kDfMaxWaves][kStMaxG][kDfOutRow];
    float m[kDfMaxWaves][kStMaxG], l[kDfMaxWaves][kStMaxG];
};
static_assert(sizeof(WaveResults) <= kStWordBytes, "");
constexpr int kStRow = kHeadDim + 8;  // so that the heads' pieces of 16 bytes do not meet in one bank

template <int MT>
struct Shared {
    static constexpr int TQ = MT <= kStDirect ? MT : 1;  // rows that a task normalises
    // packed words of this task and the next two (an attention task keeps its waves' outputs in its buffer)
    __attribute__((aligned(16))) uint8_t words[kStBuffers][kStWordBytes];
    __attribute__((aligned(16))) int8_t q[kStWaves][TQ][MT <= kStDirect ? kStUpwF * 64 + 80 : 16];  // a wave's quantized slices (reads go one step past)
    // the waves' partial sums: [row block][wave][token][row].  Twice where nothing else keeps a wave from writing the
    // next task's while another still reads
    int red[MT <= kStDirect ? 1 : 2][4][kStWaves][MT][16];
    // each wave's copy of an attention task's new rows: the q heads of the group, k, v
    __attribute__((aligned(16))) uint16_t rows[kStWaves][kStMaxG + 2][kStRow];
    // exchanges between the computing waves: values with the number of the exchange
    // (the first in two buffers: a wave may be a task ahead of one that has not looked yet, not two)
    __attribute__((aligned(16))) v4i sumsq[2][TQ][kStWaves];
    __attribute__((aligned(16))) v2i amax[TQ][kStWaves];
    __attribute__((aligned(16))) int met[kStWaves];
    // between them and the wave that fetches: counts of tasks
    __attribute__((aligned(16))) int consumed[kStWaves];
    int claimed, ready;
    __attribute__((aligned(16))) v4i tasks[4][4];  // what the computing waves have to know about a task (Task)
    uint16_t scales[4][2][32];                     // weight scales of its output rows
};

// A task as the fetching wave describes it: the computing waves find everything they would have to look up or work
// out in LDS (their own way through arguments and tables took a microsecond between two tasks)
struct Task {
    int layer, ph, idx;
    float eps;
    const uint16_t *src, *res;  // attention: the published q | k | v rows; the cache's k.  Quantizers: res = the row's record
    uint16_t *dst, *aux;        // attention: the published outputs; the cache's v.  Products: aux = the norm's weights, or,
                                // where src are quantized rows, their records
    int K, n_out;               // attention: kv head, sequence
    float inv_k;                // attention: split
    int flags;                  // 1: src is published, 2: dst is, 4: res is, 8: the rows of src or res are input_row()'s.
                                // Attention: the position
};

// a lane's values of one token's slice
template <int UPW>
struct Values {
    uint4 full[Slice<UPW>::kFull];
    uint32_t rest[Slice<UPW>::T / 2];
};
template <int MT>
struct Got {
    v4i e[4 * kStUpwD];     // the weights as MFMA operands: [row block][k-step], or the 27 steps of one block
    Values<kStUpwF> f[Shared<MT>::TQ];  // (the first members serve the shorter slices)
    uint4 g[kStMaxVec];     // norm weights of this lane's values
    float wild;             // infinity if one of them is 2^20 or more or not a number, otherwise 0
    uint16_t res;
};

template <int MT>
struct Stack {
    static constexpr int TQ = Shared<MT>::TQ;
    static constexpr bool kDirect = MT <= kStDirect;
    StackArgsPtr a;
    Shared<MT>& sh;
    Waiter wt;
    unsigned char* set;  // this launch's hand-over buffers
    unsigned launch;
    int tid, lane, wave;
    int exchange;  // exchanges so far: the same in all computing waves
    int turn;      // which part of `red`
    int side;      // ... of `sumsq`

    // Makes the compiler compute what follows from the thread's place and the arguments anew from here on: kept
    // over the whole loop of tasks, the addresses of all phases together do not fit the registers.
    __device__ __forceinline__ void forget() {
        asm volatile("" : "+v"(tid), "+v"(lane), "+s"(wave), "+s"(a));
    }

    // --- where things are ------------------------------------------------------------------------
    __device__ __forceinline__ unsigned char* layer_set(int layer) const { return set + (size_t)layer * a->f_layer; }
    __device__ __forceinline__ uint16_t* qkv(int layer) const { return (uint16_t*)layer_set(layer); }
    __device__ __forceinline__ uint16_t* o(int layer) const { return (uint16_t*)(layer_set(layer) + a->f_o); }
    __device__ __forceinline__ uint16_t* ha(int layer) const { return (uint16_t*)(layer_set(layer) + a->f_ha); }
    __device__ __forceinline__ uint16_t* gate(int layer) const { return (uint16_t*)(layer_set(layer) + a->f_g); }
    __device__ __forceinline__ uint16_t* hb(int layer) const { return (uint16_t*)(layer_set(layer) + a->f_hb); }
    // the residual stream in front of the attention block of `layer`
    // (of one sequence its row, of more the first row of what the first layer reads by input_row())
    __device__ __forceinline__ const uint16_t* h_before(int layer) const {
        return layer == 0 ? a->h_in + (MT == 1 ? (size_t)input_row(0) * a->dim : 0) : hb(layer - 1);
    }
    __device__ __forceinline__ int input_row(int m) const {
        if (!a->tokens) return m;
        const int64_t t = a->tokens[m];
        return t < 0 ? 0 : t >= (int64_t)a->in_rows ? a->in_rows - 1 : (int)t;  // nothing outside the table is read
    }
    __device__ __forceinline__ int input_bytes() const { return a->in_rows * a->dim * 2; }

    __device__ __forceinline__ Work locate(int layer, int r) const {
        Work w;
        while (r >= a->ends[8]) {
            r -= a->ends[8];
            ++layer;
        }
        int ph = 0, base = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (r >= a->ends[i]) {
                ph = i + 1;
                base = a->ends[i];
            }
        w.layer = layer;
        w.ph = ph;
        w.first = base;
        w.idx = r - base;
        return w;
    }
    // product of a phase: 0 wqkv, 1 wo, 2 w13, 3 w2
    static __device__ __forceinline__ int product_of(int ph) { return ph <= kAttn ? 0 : (ph - 1) >> 1; }

    __device__ __forceinline__ int batch() const { return MT == 1 ? 1 : a->B; }

    // output slot of this thread within a task: row of a 16-row block, token, and -- where a task has two rows of
    // blocks -- which
    __device__ __forceinline__ int out_row() const { return tid & 15; }
    template <int RPW>
    __device__ __forceinline__ int out_tb() const { return RPW == 1 ? 0 : (tid >> 4) & 1; }
    template <int RPW>
    __device__ __forceinline__ int out_token() const { return RPW == 1 ? tid >> 4 : tid >> 5; }

    // --- between the waves of a workgroup ------------------------------------------------------------
    // (LDS operations of a wave are carried out in order, so a number written behind a value vouches for it; the
    // hardware's barrier would have to include the wave that fetches)
    __device__ __forceinline__ void arrive() {
        ++exchange;
        if (lane == 0) lds_put(sh.met[wave], exchange);
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void await() const {
        for (;;) {
            asm volatile("" ::: "memory");
            const v4i m = lds_look(*(const v4i*)sh.met);
            if (uniform(min(min(m.x, m.y), min(m.z, m.w)) - exchange) >= 0) break;
        }
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void meet() {
        arrive();
        await();
    }

    // --- the wave that fetches -----------------------------------------------------------------------
    // distance in LDS of the two runs of row blocks that a w13 task multiplies with (and in expand())
    __device__ __forceinline__ int run_stride() const { return (a->dim * 8 + 4095) & ~4095; }
    __device__ __forceinline__ void describe(const Work& wk, const __attribute__((address_space(4))) StackEntry* e, v4i* to) const {
        const int l = wk.layer;
        const bool last = l + 1 >= a->n_layers;
        uint64_t src, res = 0, dst, aux = (uint64_t)e->norm;
        int K = a->dim, n_out = a->dim, flags = 3;
        float inv_k = a->inv_dim;
        // quantized rows of product i of the layer, 64 values of every token side by side, and their records
        auto bytes = [&](int i) { return (uint64_t)(set + a->set_values + (size_t)l * a->f_bytes + (size_t)i * a->B * a->dim); };
        auto record = [&](int i) { return (uint64_t)(layer_set(l) + a->f_rec) + (uint64_t)(i * a->B) * sizeof(RowRecord); };
        const int i = product_of(wk.ph);
        if (wk.ph == kAttn) {
            src = (uint64_t)qkv(l), dst = (uint64_t)o(l), res = (uint64_t)e->ck, aux = (uint64_t)e->cv;
            const int rest = wk.idx / a->n_kv;
            K = wk.idx % a->n_kv, n_out = rest / a->n_splits, inv_k = __uint_as_float((unsigned)(rest % a->n_splits));
            const int64_t p = a->positions[n_out];
            flags = p < 0 ? 0 : (p >= (int64_t)a->S ? a->S - 1 : (int)p);
        } else {
            src = (uint64_t)(i == 0 ? h_before(l) : i == 1 ? o(l) : i == 2 ? ha(l) : gate(l));
            if (i == 0 && l == 0) flags = (flags & ~1) | (MT == 2 ? 8 : 0);
            if (i == 3) K = a->ffn, inv_k = a->inv_ffn;
            if (wk.ph == kP1 || wk.ph == kP3 || wk.ph == kP4 || wk.ph == kP5) {
                if (!kDirect) src = bytes(i), aux = record(i);
                dst = (uint64_t)(i == 0 ? qkv(l) : i == 1 ? ha(l) : i == 2 ? gate(l) : last ? a->h_out : hb(l));
                if (i == 0) n_out = (a->n_heads + 2 * a->n_kv) * kHeadDim;
                if (i == 1) res = (uint64_t)h_before(l), flags |= l == 0 ? (MT == 1 ? 0 : 8) : 4;  // (the caller's values may be any)
                if (i == 2) n_out = a->ffn;
                if (i == 3) res = (uint64_t)ha(l), flags |= 4;
                if (i == 3 && last) flags &= ~2;
            } else {
                src += (uint64_t)(i == 0 && l == 0 ? input_row(wk.idx) : wk.idx) * K * 2;
                dst = bytes(i) + (uint64_t)wk.idx * 64;
                res = record(i) + (uint64_t)wk.idx * sizeof(RowRecord);
            }
        }
        if (lane == 0) {
            lds_put(to[0], v4i{l < a->n_layers ? l : -1, wk.ph, wk.idx, (int)__float_as_uint(e->eps)});
            lds_put(to[1], v4i{(int)src, (int)(src >> 32), (int)res, (int)(res >> 32)});
            lds_put(to[2], v4i{(int)dst, (int)(dst >> 32), (int)aux, (int)(aux >> 32)});
            lds_put(to[3], v4i{K, n_out, (int)__float_as_uint(inv_k), flags});
        }
    }
    // the weight scale of output row lane % 32 of a task, of w13's second half in the upper lanes
    __device__ __forceinline__ uint16_t scale_of(const Work& wk, const __attribute__((address_space(4))) StackEntry* e) const {
        const int first = wk.ph == kP1 || wk.ph == kP4 ? 2 * wk.idx : wk.idx;
        const int n = first * 16 + (lane & 31) + (lane >> 5) * a->ffn;
        int run = 0;
#pragma unroll
        for (int j = 1; j < 8; ++j) run += n >= j * e->slot_rows ? 1 : 0;
        return e->ws[(e->slot_map >> (3 * run)) & 7u];
    }
    // the packed words of a task into LDS, in pieces of 1 KB
    __device__ __forceinline__ void fetch(const Work& wk, const uint32_t* w, int buffer) const {
        if (wk.ph != kP1 && wk.ph != kP3 && wk.ph != kP4 && wk.ph != kP5) return;
        const int K = wk.ph == kP5 ? a->ffn : a->dim;
        const int half = a->ffn >> 4;  // row blocks of one half of w13
        const bool pairs = wk.ph == kP1 || wk.ph == kP4;
        const int first = pairs ? 2 * wk.idx : wk.idx;
        const int bytes = uniform((!pairs || (wk.ph == kP4 && first + 1 >= half) ? 1 : 2) * K * 4);
        for (int i = 0; i < (wk.ph == kP4 ? 2 : 1); ++i) {
            const uintptr_t from = (uintptr_t)w + (size_t)(i * half + first) * K * 4;
            v4u r = {(unsigned)uniform((int)from), (unsigned)uniform((int)(from >> 32)) & 0xffffu, (unsigned)bytes, 0x00020000u};
            settled(r);
            const unsigned to = lds_address(&sh.words[buffer][i ? run_stride() : 0]);
#pragma nounroll
            for (int at = 0; at < bytes; at += 1024) load_to_lds(r, to + at, lane * 16, at);
        }
    }

    // --- a product -----------------------------------------------------------------------------------
    // the norm's weights for this lane's values
    template <int UPW>
    __device__ __forceinline__ void norm_weights(const uint16_t* norm, int K, Got<MT>& got) const {
        typedef Slice<UPW> S;
        const __amdgpu_buffer_rsrc_t r = make_rsrc(norm, K * 2);
        int off[S::kVec];
        slice_offsets<UPW>(K * 2, off);
#pragma unroll
        for (int i = 0; i < S::kFull; ++i) got.g[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off[i], 0, 0));
        if (S::T == 2) got.g[S::kFull].x = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off[S::kFull], 0, 0);
        if (S::T == 4) {
            const v2u t = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(r, off[S::kFull], 0, 0));
            got.g[S::kFull].x = t.x;
            got.g[S::kFull].y = t.y;
        }
    }
    // (behind the loads' way to memory, in front of the wait for the activations)
    template <int UPW>
    __device__ __forceinline__ void look_at_weights(Got<MT>& got) const {
        typedef Slice<UPW> S;
        uint32_t most = 0;
#pragma unroll
        for (int i = 0; i < S::kFull; ++i) most = absmax_bits8(got.g[i], most);
        if (S::T) most = absmax_bits8(make_uint4(got.g[S::kFull].x, S::T == 4 ? got.g[S::kFull].y : 0u, 0u, 0u), most);
        got.wild = most >= 0x4980u ? INFINITY : 0.0f;  // 2^20
        asm volatile("" : "+v"(got.wild));
    }
    // byte offsets of this lane's values in a row of row_bytes, kBeyond past its end
    template <int UPW>
    __device__ __forceinline__ void slice_offsets(int row_bytes, int (&off)[Slice<UPW>::kVec]) const {
        typedef Slice<UPW> S;
        const int first = wave * S::kValues * 2;
#pragma unroll
        for (int i = 0; i < S::kFull; ++i) {
            const int at = first + i * 1024 + lane * 16;
            off[i] = at < row_bytes ? at : kBeyond;
        }
        if (S::T) {
            const int at = first + S::kFull * 1024 + lane * (S::T * 2);
            off[S::kFull] = lane * S::T < S::kRest && at < row_bytes ? at : kBeyond;
        }
    }
    // The packed words of a task, in LDS, -> MFMA operands.  In front of the wait for the activations, where nothing
    // else is to be done.
    template <int UPW, int RPW>
    __device__ __forceinline__ void expand(int K, int buffer, Got<MT>& got) {
        const int p = lane & 15, g = lane >> 4;
        const int lane_word = (g >> 1) * 32 + (p >> 3) * 16 + (g & 1) * 8 + (p & 7);
        const uint8_t* words = &sh.words[buffer][wave * (UPW * 256) + lane_word * 4];
        const int stride2 = RPW == 4 ? (K * 8 + 4095) & ~4095 : 0;
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
            for (int j = 0; j < UPW; ++j) {
                // (past the end of K: whatever follows, times activations that are zero)
                const uint32_t w = *(const uint32_t*)(words + (i >> 1) * stride2 + (i & 1) * K * 4 + j * 256);
                // bytes that read 64 times the weight (two-bit fields at the top, less the codes' 2): sums need no correction
                v4i& e = got.e[i * kStUpwD + j];
                const uint32_t c = w ^ 0xaaaaaaaau;
                e.x = (int)(c << 6 & 0xc0c0c0c0u);
                e.y = (int)(c << 4 & 0xc0c0c0c0u);
                e.z = (int)(c << 2 & 0xc0c0c0c0u);
                e.w = (int)(c & 0xc0c0c0c0u);
            }
        // now, not where they are used: the compiler would put this work behind the wait, next to the products
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
            for (int j = 0; j < UPW; ++j) asm volatile("" : "+v"(got.e[i * kStUpwD + j]));
    }
    // the slices of the tokens' rows and, RES, this thread's value of a row that was complete before them
    template <int UPW, bool RES>
    __device__ __forceinline__ void gather_slices(const Task& tk, Got<MT>& got) {
        typedef Slice<UPW> S;
        const int K = tk.K, B = TQ == 1 ? 1 : a->B;
        int off[S::kVec];
        slice_offsets<UPW>(K * 2, off);
        const bool by_token = MT > 1 && kDirect && (tk.flags & 8) != 0;
        const __amdgpu_buffer_rsrc_t rows = make_rsrc(tk.src, by_token && !RES ? input_bytes() : B * K * 2);
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(RES ? tk.res : tk.src, RES ? (by_token ? input_bytes() : B * tk.n_out * 2) : 0);
        int row_at[TQ], res_row = out_token<1>();
#pragma unroll
        for (int t = 0; t < TQ; ++t) row_at[t] = (t < B ? t : B - 1) * K * 2;  // tokens beyond the batch repeat the last one
        if (by_token) {
            if (RES) {
                res_row = input_row(res_row < B ? res_row : 0);
            } else {
#pragma unroll
                for (int t = 0; t < TQ; ++t) row_at[t] = input_row(t < B ? t : B - 1) * K * 2;
            }
        }
        const int res_off = RES && out_token<1>() < B ? (res_row * tk.n_out + tk.idx * 16 + out_row()) * 2 : kBeyond;
        const bool published = (tk.flags & 1) != 0;
        for (int spin = 0;; ++spin) {
            poll_again();
            if (RES) got.res = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, res_off, 0, kSc1);
            unsigned m = RES && (tk.flags & 4) ? (unsigned)got.res << 16 : 0u;
#pragma unroll
            for (int t = 0; t < TQ; ++t) {
                Values<kStUpwF>& v = got.f[t];
                const int at = row_at[t];
#pragma unroll
                for (int i = 0; i < S::kFull; ++i) v.full[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, off[i], at, kSc1));
                if (S::T == 2) v.rest[0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rows, off[S::kFull], at, kSc1);
                if (S::T == 4) {
                    const v2u r = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(rows, off[S::kFull], at, kSc1));
                    v.rest[0] = r.x;
                    v.rest[1] = r.y;
                }
            }
#pragma unroll
            for (int t = 0; t < TQ; ++t) {
                const Values<kStUpwF>& v = got.f[t];
#pragma unroll
                for (int i = 0; i < S::kFull; ++i) m = unset_max(unset_max(unset_max(unset_max(m, v.full[i].x), v.full[i].y), v.full[i].z), v.full[i].w);
#pragma unroll
                for (int i = 0; i < S::T / 2; ++i) m = unset_max(m, v.rest[i]);
            }
            if (__builtin_amdgcn_ballot_w64(is_unset(m)) == 0 || !published || wt.dead || wt.give_up(spin)) break;
        }
    }

    // Norm and quantizer of the wave's slices: the scales, and the bytes by put8 (8 of them, a 512-value piece's) and
    // put_rest (S::T of them).  Whether one of the rows has a value that is not finite.
    // The waves meet once for both of a row's reductions.  The quantizer needs the largest of the normalised values
    // bf16((h r) g), and r the sum of squares; but each of those is |h g| r within two roundings, so the largest lies
    // between max |h g| r (1 - 2^-21) and the same with a plus, and where both ends round to the same bf16 that is it
    // (all but one row in some 4000, and rows of very small, very large or missing numbers, for which the maximum is
    // exchanged as well).  Products of bf16 are exact in fp32; `wild`: a weight of 2^20 or more, beyond which what
    // underflows in h r could matter.  30 layers 513 -> 497 us at one sequence, 630 -> 597 at two.
    template <int UPW, class Put8, class PutRest>
    __device__ __forceinline__ bool quantize(const Task& tk, Got<MT>& got, float (&s)[TQ], Put8 put8, PutRest put_rest) {
        typedef Slice<UPW> S;
        side ^= 1;
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            const Values<kStUpwF>& v = got.f[t];
            double sq = 0.0;  // lanes without a value hold zeros
            float top = got.wild;
#pragma unroll
            for (int i = 0; i < S::kFull; ++i) {
                sq += sumsq8(v.full[i]);
                top = product_max2(v.full[i].x, got.g[i].x, product_max2(v.full[i].y, got.g[i].y, top));
                top = product_max2(v.full[i].z, got.g[i].z, product_max2(v.full[i].w, got.g[i].w, top));
            }
#pragma unroll
            for (int i = 0; i < S::T / 2; ++i) {
                sq += sumsq2(v.rest[i]);
                top = product_max2(v.rest[i], i == 0 ? got.g[S::kFull].x : got.g[S::kFull].y, top);
            }
            sq = wave_reduce_last(sq, [](double x, double y) { return x + y; });
            const int high = wave_reduce_last(__float_as_int(top), [](int x, int y) { return max(x, y); });
            const v2i bits = __builtin_bit_cast(v2i, sq);
            if (lane == 63) lds_put(sh.sumsq[side][t][wave], v4i{bits.x, bits.y, exchange + 1, high});
        }
        ++exchange;
        uint32_t am[TQ];
        bool known = true;
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            Values<kStUpwF>& v = got.f[t];
            v4i x[kStWaves];
            for (;;) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int k = 0; k < kStWaves; ++k) x[k] = lds_look(sh.sumsq[side][t][k]);
                if (uniform(min(min(x[0].z, x[1].z), min(x[2].z, x[3].z)) - exchange) >= 0) break;
            }
            double total = 0.0;
#pragma unroll
            for (int k = 0; k < kStWaves; ++k) total += __builtin_bit_cast(double, v2i{x[k].x, x[k].y});
            const float rstd = reciprocal_sqrt(divide((float)total, (float)tk.K, tk.inv_k) + tk.eps);
            const float top = __int_as_float(max(max(x[0].w, x[1].w), max(x[2].w, x[3].w))) * rstd;
            const uint32_t ends = f32x2_to_bf16x2(__builtin_fmaf(top, -0x1p-21f, top), __builtin_fmaf(top, 0x1p-21f, top));
            am[t] = ends & 0xffffu;
            known = known && top >= 0x1p-60f && top <= 0x1p60f && am[t] == ends >> 16;
#pragma unroll
            for (int i = 0; i < S::kFull; ++i) v.full[i] = norm8(v.full[i], got.g[i], rstd);
            if (S::T) {
                v.rest[0] = norm2(v.rest[0], got.g[S::kFull].x, rstd);
                if (S::T == 4) v.rest[1] = norm2(v.rest[1], got.g[S::kFull].y, rstd);
            }
        }
        bool nonfinite = false;
        if (!uniform(known)) nonfinite = exchange_maxima<UPW>(tk, got, am);
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            const Values<kStUpwF>& v = got.f[t];
            // quant_scale<0>
            s[t] = bf16_to_f32(f32_to_bf16_rne(reciprocal(fmaxf(__uint_as_float(am[t] << 16), 1e-5f)) * 127.0f));
#pragma unroll
            for (int i = 0; i < S::kFull; ++i) put8(t, i, quant_vec8<0>(v.full[i], s[t]));
            if (S::T) {
                uint32_t r = quant2(v.rest[0], s[t]);
                if (S::T == 4) r |= quant2(v.rest[1], s[t]) << 16;
                put_rest(t, r);
            }
        }
        return nonfinite;
    }
    // The rows' maxima from the normalised values themselves; whether one of them is infinite or a NaN
    template <int UPW>
    __device__ __forceinline__ bool exchange_maxima(const Task& tk, Got<MT>& got, uint32_t (&am)[TQ]) {
        typedef Slice<UPW> S;
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            const Values<kStUpwF>& v = got.f[t];
            uint32_t m = 0;
#pragma unroll
            for (int i = 0; i < S::kFull; ++i) m = absmax_bits8(v.full[i], m);
            if (S::T) m = absmax_bits8(make_uint4(v.rest[0], S::T == 4 ? v.rest[1] : 0u, 0u, 0u), m);
            m = wave_reduce_last(m, [](uint32_t x, uint32_t y) { return max(x, y); });
            if (lane == 63) lds_put(sh.amax[t][wave], v2i{(int)m, exchange + 1});
        }
        ++exchange;
        bool nonfinite = false;
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
            Values<kStUpwF>& v = got.f[t];
            v4i x[2];
            for (;;) {
                asm volatile("" ::: "memory");
                x[0] = lds_look(*(const v4i*)&sh.amax[t][0]);
                x[1] = lds_look(*(const v4i*)&sh.amax[t][2]);
                if (uniform(min(min(x[0].y, x[0].w), min(x[1].y, x[1].w)) - exchange) >= 0) break;
            }
            am[t] = (uint32_t)max(max(x[0].x, x[0].z), max(x[1].x, x[1].z));
            if (uniform((int)am[t]) >= 0x7f80) {  // 0 times a NaN: the values past the end of K have to be zeros again
                nonfinite = true;
#pragma unroll
                for (int i = 0; i < S::kFull; ++i)
                    if (wave * S::kValues + i * 512 + lane * 8 >= tk.K) v.full[i] = make_uint4(0u, 0u, 0u, 0u);
                if (S::T && (lane * S::T >= S::kRest || wave * S::kValues + S::kFull * 512 + lane * S::T >= tk.K)) {
                    v.rest[0] = 0u;
                    if (S::T == 4) v.rest[1] = 0u;
                }
            }
        }
        return nonfinite;
    }

    // norm + quantizer of the wave's slices, products, outputs.  RPW 1, 2: row blocks; 4: two pairs (x1, x3), gated
    template <int UPW, int RPW, bool RES>
    __device__ __forceinline__ void product(const Task& tk, int k, Got<MT>& got) {
        typedef Slice<UPW> S;
        float s[MT];
        quantize<UPW>(
            tk, got, s, [&](int t, int i, uint2 v) { *(uint2*)(sh.q[wave][t] + i * 512 + lane * 8) = v; },
            [&](int t, uint32_t r) {
                if (lane * S::T < S::kRest) {
                    if (S::T == 2) *(uint16_t*)(sh.q[wave][t] + S::kFull * 512 + lane * 2) = (uint16_t)r;
                    if (S::T == 4) *(uint32_t*)(sh.q[wave][t] + S::kFull * 512 + lane * 4) = r;
                }
            });
        // the same wave wrote its slices and reads them: LDS operations of a wave complete in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int p = lane & 15, g = lane >> 4;
        // The products' columns beyond the tokens carry the same tokens at other k-steps: one read serves SP steps (a
        // read per step, of which the columns take the same bytes 16 / MT times, bounds this part: 66 cycles a step),
        // step s is multiplied into accumulator s, and of that the columns of step s count.
        constexpr int SP = RPW == 4 ? 2 : 4;
        const int step = (p / MT) % SP;
        const int8_t* brow = &sh.q[wave][p % MT][step * 64 + g * 16];
        v4i acc[RPW][SP];
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
            for (int c = 0; c < SP; ++c) acc[i][c] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < UPW; j += SP) {
            const v4i b = *(const v4i*)(brow + j * 64);  // (steps past the slice: not multiplied)
#pragma unroll
            for (int c = 0; c < SP; ++c)
                if (j + c < UPW) {
#pragma unroll
                    for (int i = 0; i < RPW; ++i)
                        acc[i][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(got.e[i * kStUpwD + j + c], b, acc[i][c], 0, 0, 0);
                }
        }
        // lane (p, g) holds token p, rows 4 g ..
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            v4i v = acc[i][0];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int c = 1; c < SP; ++c) v[r] = step == c ? acc[i][c][r] : v[r];
                v[r] += __builtin_amdgcn_update_dpp(0, v[r], 0x120 + MT, 0xF, 0xF, true);  // row_ror
                if (SP == 4) v[r] += __builtin_amdgcn_update_dpp(0, v[r], 0x120 + 2 * MT, 0xF, 0xF, true);
            }
            if (p < MT) *(v4i*)&sh.red[turn][i][wave][p][4 * g] = v;
        }
        float sm = s[0];
#pragma unroll
        for (int t = 1; t < MT; ++t) sm = out_token<RPW>() == t ? s[t] : sm;
        finish<RPW, RES>(tk, k, sm, got.res);
    }
    // The outputs, by the first waves, from the waves' sums in LDS: sm is the scale of this thread's token (out_token)
    template <int RPW, bool RES>
    __device__ __forceinline__ void finish(const Task& tk, int k, float sm, uint16_t res) {
        arrive();
        if (kDirect && wave * 64 >= (RPW == 1 ? 16 : 32) * MT) return;
        // (what does not need the sums, while they come)
        const int m = out_token<RPW>(), tb = out_tb<RPW>(), row = out_row();
        const int n = ((RPW == 1 ? tk.idx : 2 * tk.idx + tb) * 16) + row;
        const uint16_t* ws = &sh.scales[k & 3][0][RPW == 1 ? tid & 15 : tid & 31];
        const float inv_s = reciprocal(sm), w1 = bf16_to_f32(ws[0]), w3 = RPW == 4 ? bf16_to_f32(ws[32]) : 0.0f;
        await();
        if (m < batch() && m < MT && n < tk.n_out) {
            auto value = [&](int i, float w) {
                int sum = 0;
#pragma unroll
                for (int k = 0; k < kStWaves; ++k) sum += sh.red[turn][i][k][m][row];
                return f32_to_bf16_rne(quotient((float)(sum >> 6), sm, inv_s) * w);  // (64 times the sum)
            };
            uint16_t v = value(tb, w1);
            if (RPW == 4) {
                const uint16_t x3 = value(2 + tb, w3);
                const float r = fmaxf(bf16_to_f32(v), 0.0f);
                v = f32_to_bf16_rne(bf16_to_f32(f32_to_bf16_rne(r * r)) * bf16_to_f32(x3));
            }
            if (RES) v = f32_to_bf16_rne(bf16_to_f32(res) + bf16_to_f32(v));
            uint16_t* to = tk.dst + (size_t)m * tk.n_out + n;
            if (tk.flags & 2)
                publish16(to, v);
            else
                *to = v;
        }
    }

    // --- beyond kStDirect tokens: a token's row quantized, once for all workgroups ----------------------
    template <int UPW>
    __device__ __forceinline__ void quantizer_task(const Task& tk, int k) {
        typedef Slice<UPW> S;
        Got<MT> got;
        norm_weights<UPW>(tk.aux, tk.K, got);
        wait_ready(k);
        consume(k);
        look_at_weights<UPW>(got);
        gather_slices<UPW, false>(tk, got);
        float s[TQ];
        const int first = wave * S::kValues, step = batch() * 64;
        const __amdgpu_buffer_rsrc_t to = make_rsrc(tk.dst, ((tk.K >> 6) - 1) * step + 64);
        auto place = [&](int at) { return (at >> 6) * step + (at & 63); };
        // (4 bytes at least a store: a word is there or not; values past the end of K are not stored)
        const bool nonfinite = quantize<UPW>(
            tk, got, s,
            [&](int, int i, uint2 v) {
                const int at = first + i * 512 + lane * 8;
                __builtin_amdgcn_raw_buffer_store_b64(v2u{v.x, v.y}, to, at < tk.K ? place(at) : kBeyond, 0, kSc1);
            },
            [&](int, uint32_t r) {
                int at = first + S::kFull * 512 + lane * S::T;
                bool mine = lane * S::T < S::kRest && at < tk.K;
                if (S::T == 2) {  // with the neighbour's
                    r = (r & 0xffffu) | (unsigned)__builtin_amdgcn_update_dpp(0, (int)r, 0xB1, 0xF, 0xF, true) << 16;
                    mine = mine && (lane & 1) == 0;
                }
                __builtin_amdgcn_raw_buffer_store_b32(r, to, mine ? place(at) : kBeyond, 0, kSc1);
            });
        RowRecord* rec = (RowRecord*)tk.res;
        if (nonfinite) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // readers cannot tell from the words that they are there
        if (lane == 0) {
            __hip_atomic_store(&rec->slice[wave], nonfinite ? kComplete : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (wave == 0) __hip_atomic_store(&rec->scale, (unsigned)f32_to_bf16_rne(s[0]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // a product of quantized rows: they are the MFMAs' column operand as they lie in memory
    template <int UPW, int RPW, bool RES>
    __device__ __forceinline__ void bytes_task(const Task& tk, int k) {
        Got<MT> got;
        wait_ready(k);
        expand<UPW, RPW>(tk.K, k % kStBuffers, got);
        consume(k);
        const int p = lane & 15, g = lane >> 4, B = batch(), K = tk.K;
        const int first = wave * (UPW * 64);
        const int live = K - first < 0 ? 0 : (K - first) >> 6;  // k-steps of the slice in front of the end of K
        const int m = out_token<RPW>() < B ? out_token<RPW>() : B - 1;
        // column p is token p % MT at the k-step p / MT of SP that one load covers (as in product())
        constexpr int SP = 16 / MT, kLoads = (UPW + SP - 1) / SP;
        const int ps = p / MT, pt = p % MT;
        const unsigned step = B * 64;
        const unsigned base = pt < B ? (first + ps * 64) * B + pt * 64 + g * 16 : kBeyond;  // (no such token: zeros, no access)
        const __amdgpu_buffer_rsrc_t rows = make_rsrc(tk.src, B * K), recs = make_rsrc(tk.aux, B * (int)sizeof(RowRecord));
        const bool by_token = RES && (tk.flags & 8) != 0;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(RES ? tk.res : tk.src, RES ? (by_token ? input_bytes() : B * tk.n_out * 2) : 0);
        const int res_off = RES ? ((by_token ? input_row(m) : m) * tk.n_out + tk.idx * 16 + out_row()) * 2 : kBeyond;
        v4i b[kLoads], sums;
        unsigned scale = 0;
        auto recorded = [&] { return (int)(sums.x | sums.y | sums.z | sums.w | (int)scale) >= 0; };
        auto lowest = [](int m, v4i v) { return min(min(min(m, v.x), min(v.y, v.z)), v.w); };
        int unset = kUnsetBytes;  // of this lane's values; 1, which none has, once its slice is known to be in memory
        auto incomplete = [&] {
            int low = 0;
#pragma unroll
            for (int j = 0; j < kLoads; ++j) low = lowest(low, b[j]);
            return __builtin_amdgcn_ballot_w64(low == unset || !recorded() || (RES && (tk.flags & 4) && got.res == 0xffffu)) != 0;
        };
        // Whether this lane's slice is in memory, whatever it looks like: what is read behind this is what was written.
        // Asked for seldom: with the answer in every poll eight sequences took 4 % more time.
        auto vouched = [&] {
            poll_again();
            unsigned held = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(
                recs, pt < B ? pt * (int)sizeof(RowRecord) + wave * 4 : kBeyond, 0, kSc1);
            asm volatile("" : "+v"(held));
            return (int)held >= 0 && (held & kComplete) != 0;
        };
        // one piece until it is there, then all: all workgroups asking for all rows all the time fill the fabric, and so
        // do all asking for the same piece
        const int turns = live / SP;  // loads of which every column is in front of the end of K
        const unsigned probe = turns > 0 ? base + (tk.idx % turns) * (SP * step) : ps < live ? base : (unsigned)kBeyond;
        for (int spin = 0;; ++spin) {
            poll_again();
            const v4i v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rows, probe, 0, kSc1));
            if (__builtin_amdgcn_ballot_w64(lowest(0, v) == kUnsetBytes) == 0 || wt.dead || wt.give_up(spin)) break;
            if ((spin & (kLookEvery - 1)) == kLookEvery - 1 && __builtin_amdgcn_ballot_w64(vouched()) != 0) break;
        }
        auto get = [&](auto policy) {
            poll_again();
            if (RES) got.res = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, res_off, 0, kSc1);
            sums = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(recs, m * (int)sizeof(RowRecord), 0, decltype(policy)::value));
            scale = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(recs, m * (int)sizeof(RowRecord) + 16, 0, decltype(policy)::value);
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                b[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                                   rows, j * SP + ps < live ? base + j * (SP * step) : (unsigned)kBeyond, 0, decltype(policy)::value));
        };
        get(std::integral_constant<int, 0>{});
        for (int spin = 0; incomplete() && !wt.dead && !wt.give_up(spin); ++spin) {
            if ((spin & (kLookEvery - 1)) == 3) unset = vouched() ? 1 : kUnsetBytes;
            get(std::integral_constant<int, kSc1>{});
        }
        v4i acc[RPW][SP];
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
            for (int c = 0; c < SP; ++c) acc[i][c] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < UPW; ++j)
#pragma unroll
            for (int i = 0; i < RPW; ++i)
                acc[i][j % SP] = __builtin_amdgcn_mfma_i32_16x16x64_i8(got.e[i * kStUpwD + j], b[j / SP], acc[i][j % SP], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < RPW; ++i) {
            v4i v = acc[i][0];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int c = 1; c < SP; ++c) v[r] = ps == c ? acc[i][c][r] : v[r];
                v[r] += __builtin_amdgcn_update_dpp(0, v[r], 0x120 + MT, 0xF, 0xF, true);  // row_ror
                if (SP == 4) v[r] += __builtin_amdgcn_update_dpp(0, v[r], 0x120 + 2 * MT, 0xF, 0xF, true);
            }
            if (p < MT) *(v4i*)&sh.red[turn][i][wave][p][4 * g] = v;
        }
        finish<RPW, RES>(tk, k, bf16_to_f32((uint16_t)scale), got.res);
        turn ^= 1;
    }

    // --- attention: rope, cache write and one split of one (sequence, kv head) ------------------------
    // (attn_decode_flash_kernel's work on published rows; the last active split merges)
    struct Place {
        int G, kvh, sp, b, p, pblk, nact, busy, n_heads, n_kv, nsplit, attn_waves;
        unsigned tag;              // of this task's records
        unsigned long long *rec, *own;  // of its (sequence, kv head), and of its split
        uint32_t* out;
    };
    __device__ __forceinline__ Place attention_place(const Task& tk) const {
        Place w;
        w.G = a->group;
        w.n_heads = a->n_heads;
        w.n_kv = a->n_kv;
        w.nsplit = a->n_splits;
        w.attn_waves = a->attn_waves;
        w.kvh = tk.K;
        w.b = tk.n_out;
        w.sp = (int)__float_as_uint(tk.inv_k);
        w.p = tk.flags;
        w.pblk = w.p >> 5;
        w.nact = w.pblk + 1 < w.nsplit ? w.pblk + 1 : w.nsplit;
        // the split's blocks are dealt to attn_waves waves in turn: this many of them have one
        const int blocks = uniform((w.pblk - w.sp) / w.nsplit) + 1;
        w.busy = blocks < w.attn_waves ? blocks : w.attn_waves;
        w.tag = launch * (unsigned)a->n_layers + (unsigned)tk.layer + 1u;
        w.rec = (unsigned long long*)(a->ws + a->records) + ((size_t)(w.b * w.n_kv + w.kvh) * w.nsplit) * kStMaxG * kDfRecUnits;
        w.own = w.rec + (size_t)w.sp * kStMaxG * kDfRecUnits;
        w.out = (uint32_t*)(tk.dst + (size_t)w.b * a->dim + (size_t)w.kvh * w.G * kHeadDim);
        // (looked up here, not where they are used: a scalar load behind the task's inputs is waited for)
        asm volatile("" : "+s"(w.tag), "+s"(w.rec), "+s"(w.own), "+s"(w.out), "+s"(w.G), "+s"(w.busy), "+s"(w.nact), "+s"(w.nsplit));
        return w;
    }
    // Up to the waves' results in LDS.  From the arrival of the token's row on a task is bound by the number of its instructions
    // (one wave per SIMD), so everything that does not need the row is in registers before: the first block's cache rows, V
    // turned, the rotation's factors, who has the new row, all of Place.  Every wave rotates the q heads for itself, eight
    // values a lane, so the waves meet only once, over the results.  From the row to the split's record 2.5 us -> 1.3 (the split
    // with the new row 2.9 -> 1.6; blocks and products where the compiler put them, and two meetings), one sequence at
    // 512 positions 613 -> 587 us a step, two 720 -> 690, eight 870 -> 856.
    // fresh, has_new: the cache's row p, k in lanes 0 .. 15 and v in those behind, for its caller to store.
    __device__ __forceinline__ void attend(const Task& wk, const Place& at, WaveResults& res, v4u& fresh, bool& has_new) {
        if (wave >= at.busy) {
            df_wave_result<kStMaxG>(DfState(), lane, res.o[wave], res.m[wave], res.l[wave]);
            return;
        }
        const int G = at.G, nsplit = at.nsplit, kvh = at.kvh, sp = at.sp, b = at.b, p = at.p, pblk = at.pblk, n_kv = at.n_kv;
        const int c = lane & 15, g4 = lane >> 4;
        const int row_elems = (at.n_heads + 2 * n_kv) * kHeadDim;
        uint16_t* ck = (uint16_t*)wk.res + ((size_t)b * a->S * n_kv + kvh) * kHeadDim;
        uint16_t* cv = wk.aux + ((size_t)b * a->S * n_kv + kvh) * kHeadDim;
        const int row_bytes = n_kv * kHeadDim * 2;
        const int cache_bytes = (a->S - 1) * row_bytes + kHeadDim * 2;
        const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(ck, cache_bytes), v_rsrc = make_rsrc(cv, cache_bytes);
        const int blk_stride = nsplit * at.attn_waves;  // this wave takes the blocks of waves wave, wave + kStWaves, ...
        v4u kb[2][4], vb[8];
        auto request_rows = [&](int blk) {
            const int base = blk * 32 * row_bytes;
#pragma unroll
            for (int bi = 0; bi < 2; ++bi) {
                const int off = base + (bi * 16 + c) * row_bytes + g4 * 16;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) kb[bi][kk] = __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, off + kk * 64, 0, 0);
            }
#pragma unroll
            for (int jj = 0; jj < 8; ++jj)
                vb[jj] = __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, base + ((jj & 3) + (jj >> 2) * 16 + 4 * g4) * row_bytes + c * 16, 0, 0);
        };
        auto turn_rows = [&](int blk) {
            if (blk == pblk) df_clear(vb, p, lane);
            df_turn(vb);
        };
        request_rows(sp + nsplit * wave);
        // the factors of pairs 4 c ..
        const size_t factors = (size_t)(a->tokens ? p : b) * a->factors;
        v4u cs = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(a->cos + factors, kHeadDim * 2), c * 16, 0, 0);
        v4u sn = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(a->sin + factors, kHeadDim * 2), c * 16, 0, 0);
        const int turn = uniform(pblk / nsplit);
        has_new = uniform(pblk - turn * nsplit == sp && (turn % at.attn_waves) % kStWaves == wave);

        // heads 4 u + g4 of the group, dims 8 c .. (lanes beyond the last head repeat it); where it is wanted k by lanes
        // 0 .. 15 and v by the others
        constexpr int kRounds = kStMaxG / 4;
        const __amdgpu_buffer_rsrc_t row = make_rsrc(wk.src + (size_t)b * row_elems, row_elems * 2);
        v4u raw[kRounds] = {};
        int head[kRounds];
#pragma unroll
        for (int u = 0; u < kRounds; ++u) head[u] = 4 * u + g4 < G ? 4 * u + g4 : G - 1;
        const int new_head = lane < 16 ? at.n_heads + kvh : at.n_heads + n_kv + kvh;
        auto request_token = [&]() {
            poll_again();
#pragma unroll
            for (int u = 0; u < kRounds; ++u)
                if (4 * u < G) raw[u] = __builtin_amdgcn_raw_buffer_load_b128(row, ((kvh * G + head[u]) * kHeadDim + 8 * c) * 2, 0, kSc1);
            if (has_new) fresh = __builtin_amdgcn_raw_buffer_load_b128(row, (new_head * kHeadDim + 8 * c) * 2, 0, kSc1);
        };
        // Where wqkv's and the attention's tasks together are more than the workgroups (280 of 256 at four sequences, 360 at
        // eight), some come here from a wqkv task: the token's row is there by the time that the cache rows are, 1.5 us later,
        // and a poll behind those is another 0.4.  So the row is requested along with them and looked at once they are turned: four
        // sequences 784 -> 775 us a step at 512 positions, five 798 -> 783, eight 853 -> 845.  (With the cache rows brought into
        // the L2 by the wave that fetches it is there 0.5 us earlier, and wo's phase takes 0.8 longer.)  Up to two sequences
        // everybody waits for the row, and an early look costs 0.5 %.
        if constexpr (!kDirect) request_token();
        turn_rows(sp + nsplit * wave);
        DfState st;
        // (kept in front of the polls)
#pragma unroll
        for (int t = 0; t < 8; ++t) asm volatile("" : "+v"(st.o_acc[t]), "+v"(vb[t]), "+v"(kb[t >> 2][t & 3]));
        asm volatile("" : "+v"(cs), "+v"(sn));
        for (int spin = 0;; ++spin) {
            if (kDirect || spin > 0) request_token();
            unsigned m = 0;
            auto look = [&](const v4u& v) { m = unset_max(unset_max(unset_max(unset_max(m, v.x), v.y), v.z), v.w); };
#pragma unroll
            for (int u = 0; u < kRounds; ++u)
                if (4 * u < G) look(raw[u]);
            look(fresh);
            if (__builtin_amdgcn_ballot_w64(is_unset(m)) == 0 || wt.dead || wt.give_up(spin)) break;
        }
        // rope on adjacent pairs, fp32, rounded to bf16
        auto rotated = [&](const v4u& v) {
            auto pair = [](unsigned d, unsigned cs, unsigned sn) {
                const float x = bf16f(d), y = __uint_as_float(d & 0xffff0000u), k = __uint_as_float(cs), s = __uint_as_float(sn);
                return pack_bf16x2(x * k - y * s, x * s + y * k);
            };
            return v4u{pair(v.x, cs.x, sn.x), pair(v.y, cs.y, sn.y), pair(v.z, cs.z, sn.z), pair(v.w, cs.w, sn.w)};
        };
        uint16_t(*rows)[kStRow] = sh.rows[wave];
#pragma unroll
        for (int u = 0; u < kRounds; ++u)
            if (4 * u < G) *(v4u*)&rows[head[u]][8 * c] = rotated(raw[u]);
        if (has_new) {
            const v4u r = rotated(fresh);
            fresh = lane < 16 ? r : fresh;
            *(v4u*)&rows[lane < 16 ? kStMaxG : kStMaxG + 1][8 * c] = fresh;
        }
        v4u vn = {0u, 0u, 0u, 0u};
        auto new_row = [&]() {
            df_new_key(kb, rows[kStMaxG], p, lane);
            vn = *(const v4u*)&rows[kStMaxG + 1][8 * c];
        };
        int blk = sp + nsplit * wave;
        if (blk == pblk) new_row();
        // q^T as the B operand: column c = head c (columns beyond the group repeat its heads and are not looked at)
        v8bf qa[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) qa[kk] = __builtin_bit_cast(v8bf, *(const v4u*)&rows[c & (G - 1)][kk * 32 + g4 * 8]);
        auto later_block = [&]() {
            request_rows(blk);
            turn_rows(blk);
            if (blk == pblk) new_row();
            df_block(kb, vb, vn, qa, blk, p, lane, st);
        };
        // (the first block stands by itself: nothing that a loop over the others needs is in its way)
        df_block(kb, vb, vn, qa, blk, p, lane, st);
        while ((blk += blk_stride) <= pblk) later_block();
        df_wave_result<kStMaxG>(st, lane, res.o[wave], res.m[wave], res.l[wave]);
        if (at.busy <= kStWaves) return;
        st = DfState();
        const int w = wave + kStWaves;
        for (blk = sp + nsplit * w; blk <= pblk && w < at.attn_waves; blk += blk_stride) later_block();
        df_wave_result<kStMaxG>(st, lane, res.o[w], res.m[w], res.l[w]);
    }
    // the waves' results over the workgroup, then over the splits
    __device__ __forceinline__ void attention_outputs(const Place& at, const WaveResults& res) {
        const int G = at.G, sp = at.sp, nact = at.nact;
        const unsigned long long tag = (unsigned long long)at.tag << 32;
        meet();
        for (int hh = wave; hh < G; hh += kStWaves) {
            DfPartial h = at.busy <= kStWaves ? df_combine<kStMaxG, 4, true>(res.o, res.m, res.l, hh, 4, lane)
                                              : df_combine<kStMaxG, 8, true>(res.o, res.m, res.l, hh, 8, lane);
            if (sp < nact - 1) {
                df_store_record(at.own + hh * kDfRecUnits, tag, h, lane);
                continue;
            }
            bool gave_up = false;
            if (nact > 1) h = df_merge<kStMaxG>(at.rec, nact, hh, tag, h, lane, wt.dead ? 1 : wt.limit, gave_up);
            if (uniform(gave_up)) {
                if (lane == 0) __hip_atomic_store(wt.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                wt.dead = true;
            }
            const float is = gave_up ? __builtin_nanf("") : 1.0f / h.l;
            __hip_atomic_store(at.out + hh * (kHeadDim / 2) + lane, (uint32_t)to_bf16(h.o0 * is) | ((uint32_t)to_bf16(h.o1 * is) << 16),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // to_bf16 gives no 0xffff
        }
    }

    // --- one task --------------------------------------------------------------------------------------
    template <int UPW, int RPW, bool RES>
    __device__ __forceinline__ void product_task(const Task& tk, int k) {
        Got<MT> got;
        norm_weights<UPW>(tk.aux, tk.K, got);
        wait_ready(k);
        expand<UPW, RPW>(tk.K, k % kStBuffers, got);
        consume(k);
        look_at_weights<UPW>(got);
        gather_slices<UPW, RES>(tk, got);
        product<UPW, RPW, RES>(tk, k, got);
    }
    // task k's words are in its buffer
    __device__ __forceinline__ void wait_ready(int k) const {
        while (uniform(lds_look(sh.ready)) <= k) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
    }
    // task k's buffer is free again
    __device__ __forceinline__ void consume(int k) {
        asm volatile("" ::: "memory");
        if (lane == 0) lds_put(sh.consumed[wave], k + 1);
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void run(const Task& tk, int k) {
        if (tk.ph == kAttn) {
            WaveResults& res = *(WaveResults*)sh.words[k % kStBuffers];
            wait_ready(k);
            const Place at = attention_place(tk);
            if (at.sp < at.nact) {  // (else no visible rows in this split)
                v4u fresh = {0u, 0u, 0u, 0u};
                bool has_new = false;
                attend(tk, at, res, fresh, has_new);
                attention_outputs(at, res);
                // the cache's row p, k in lanes 0 .. 15 and v in those behind: nothing in this launch reads it
                if (has_new && lane < 32)
                    *(v4u*)((lane < 16 ? (uint16_t*)tk.res : tk.aux) + (((size_t)at.b * a->S + at.p) * at.n_kv + at.kvh) * kHeadDim + 8 * (lane & 15)) = fresh;
            }
            consume(k);
        } else if constexpr (kDirect) {
            switch (tk.ph) {
                case kP1: product_task<kStUpwD, 2, false>(tk, k); break;
                case kP3: product_task<kStUpwD, 1, true>(tk, k); break;
                case kP4: product_task<kStUpwD, 4, false>(tk, k); break;
                default: product_task<kStUpwF, 1, true>(tk, k); break;
            }
        } else {
            switch (tk.ph) {
                case kP1: bytes_task<kStUpwD, 2, false>(tk, k); break;
                case kP3: bytes_task<kStUpwD, 1, true>(tk, k); break;
                case kP4: bytes_task<kStUpwD, 4, false>(tk, k); break;
                case kP5: bytes_task<kStUpwF, 1, true>(tk, k); break;
                case kQ5: quantizer_task<kStUpwF>(tk, k); break;
                default: quantizer_task<kStUpwD>(tk, k); break;
            }
        }
    }
};

template <int MT>
__global__ __launch_bounds__(kStThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void decode_stack_kernel(const StackArgs a) {
    __shared__ Shared<MT> sh;
    StackControl* ctl = (StackControl*)a.ws;
    const int tid = threadIdx.x;
    // changes only when every workgroup of this launch is done; written past the writer's L2, so read past this one
    const unsigned launch = (unsigned)uniform((int)__hip_atomic_load(&ctl->launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    Stack<MT> st{(StackArgsPtr)__builtin_amdgcn_kernarg_segment_ptr(), sh, Waiter{a.spin_limit, &ctl->error, false},
                 a.ws + a.sets + (size_t)(launch & 1u) * a.set_bytes, launch, tid, tid & 63, uniform(tid >> 6), 0, 0, 0};
    if (tid < kStWaves) sh.met[tid] = sh.consumed[tid] = 0;
    if (tid < 2 * Shared<MT>::TQ * kStWaves) ((v4i*)sh.sumsq)[tid] = v4i{0, 0, 0, 0};
    if (tid < Shared<MT>::TQ * kStWaves) ((v2i*)sh.amax)[tid] = v2i{0, 0};
    if (tid == 0) sh.claimed = sh.ready = 0;
    {
        // the other set, for the next launch
        const __amdgpu_buffer_rsrc_t other = make_rsrc(a.ws + a.sets + (size_t)((launch & 1u) ^ 1u) * a.set_bytes, a.set_bytes);
        for (int at = (blockIdx.x * kStThreads + tid) * 16; at < a.set_bytes; at += gridDim.x * kStThreads * 16) {
            const unsigned u = at < a.set_values ? ~0u : (unsigned)kUnsetBytes;
            __builtin_amdgcn_raw_buffer_store_b128(v4u{u, u, u, u}, other, at, 0, kSc1);
        }
    }
    __syncthreads();
    Work cur = st.locate(0, 0);
    if (st.wave == kStWaves) {
        // The wave that fetches: takes tickets and brings the tasks' words into LDS, up to two tasks ahead of the
        // computing waves.  Its waits for memory hold up nobody (loads of one wave return in order).
        const unsigned grid = gridDim.x, undecided = (launch + 1u) << 1;
        auto decide = [&](unsigned mode) {
            unsigned seen = __hip_atomic_load(&ctl->mode, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while (((seen ^ undecided) >> 1) != 0) {
                if (__hip_atomic_compare_exchange_strong(&ctl->mode, &seen, undecided | mode, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT))
                    break;
            }
        };
        auto claim = [&] {
            unsigned t = 0;
            if (st.lane == 0) t = __hip_atomic_fetch_add(&ctl->counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return uniform((int)t);
        };
        int mode = -1;  // 0 static, 1 tickets
        int at = 0;     // ticket of cur
        for (int k = 0;; ++k) {
            int t;
            if (k == 0) {
                t = claim();
                if (t == (int)grid - 1 && st.lane == 0) decide(0u);
            } else {
                if (mode < 0) {
                    unsigned seen = 0;
                    for (int spin = 0; spin < kStModePolls; ++spin) {
                        seen = (unsigned)uniform((int)__hip_atomic_load(&ctl->mode, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                        if (((seen ^ undecided) >> 1) == 0) break;
                    }
                    if (((seen ^ undecided) >> 1) != 0) {
                        if (st.lane == 0) decide(1u);
                        seen = (unsigned)uniform((int)__hip_atomic_load(&ctl->mode, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                    }
                    mode = (int)(seen & 1u);
                }
                t = mode == 0 ? at + (int)grid : claim();
            }
            cur = st.locate(cur.layer, cur.first + cur.idx + (t - at));
            at = t;
            const bool end = cur.layer >= a.n_layers;
            const auto* e = a.entries + ((end ? 0 : cur.layer) * 4 + st.product_of(cur.ph));
            st.describe(cur, e, sh.tasks[k & 3]);
            if (st.lane == 0) lds_put(sh.claimed, k + 1);
            asm volatile("" ::: "memory");
            if (end) break;
            // task k - kStBuffers has left this buffer
            for (;;) {
                asm volatile("" ::: "memory");
                const v4i c = lds_look(*(const v4i*)sh.consumed);
                if (uniform(min(min(c.x, c.y), min(c.z, c.w))) >= k + 1 - kStBuffers) break;
                __builtin_amdgcn_s_sleep(2);
            }
            const uint16_t scale = st.scale_of(cur, e);
            st.fetch(cur, e->w, k % kStBuffers);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            sh.scales[k & 3][st.lane >> 5][st.lane & 31] = scale;
            asm volatile("" ::: "memory");
            if (st.lane == 0) lds_put(sh.ready, k + 1);
            asm volatile("" ::: "memory");
        }
        return;
    }
    for (int k = 0;; ++k) {
        st.forget();
        while (uniform(lds_look(sh.claimed)) <= k) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
        v4i task[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) task[i] = lds_look(sh.tasks[k & 3][i]);
        auto word = [&](int i) { return uniform(task[i >> 2][i & 3]); };
        auto address = [&](int i) { return (uint64_t)(unsigned)word(i + 1) << 32 | (unsigned)word(i); };
        Task tk;
        tk.layer = word(0), tk.ph = word(1), tk.idx = word(2);
        if (tk.layer < 0) break;
        tk.eps = __uint_as_float((unsigned)word(3));
        tk.src = (const uint16_t*)address(4);
        tk.res = (const uint16_t*)address(6);
        tk.dst = (uint16_t*)address(8);
        tk.aux = (uint16_t*)address(10);
        tk.K = word(12), tk.n_out = word(13), tk.flags = word(15);
        tk.inv_k = __uint_as_float((unsigned)word(14));
        st.run(tk, k);
    }
    if (tid == 0) {
        const unsigned e = __hip_atomic_fetch_add(&ctl->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
        if (e == gridDim.x) {  // every workgroup has taken its last ticket
            __hip_atomic_store(&ctl->done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&ctl->counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&ctl->launch, launch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// A fresh workspace: zero control words and records, both sets unset
__global__ __launch_bounds__(256) void decode_stack_reset_kernel(v4u* ws, long long n, long long sets, long long set_units,
                                                                 long long value_units) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const bool in = i >= sets && i < sets + 2 * set_units;
        const unsigned fill = !in ? 0u : (i - sets) % set_units < value_units ? ~0u : (unsigned)kUnsetBytes;
        ws[i] = v4u{fill, fill, fill, fill};
    }
}

// The short forms above against the IEEE operations in their place: how many of n arguments give other bits, and the
// lowest and the highest of them (found[0..2])
__global__ __launch_bounds__(256) void decode_stack_math_kernel(int what, float by, unsigned first, unsigned n, unsigned* found) {
    unsigned wrong = 0, low = ~0u, high = 0;
    const float inv = 1.0f / by;
    for (unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (unsigned long long)gridDim.x * 256) {
        const unsigned at = first + (unsigned)i;
        const float x = what == 3 ? (float)(int)at : __uint_as_float(at);
        float a, b;
        switch (what) {
            case 0: a = reciprocal(x), b = 1.0f / x; break;
            case 1: a = reciprocal_sqrt(x), b = 1.0f / __builtin_sqrtf(x); break;
            case 2: a = divide(x, by, inv), b = x / by; break;
            default: a = quotient(x, by, inv), b = x / by; break;
        }
        const bool same = __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
        if (!same) {
            ++wrong;
            low = min(low, at);
            high = max(high, at);
        }
    }
    if (wrong) {
        atomicAdd(&found[0], wrong);
        atomicMin(&found[1], low);
        atomicMax(&found[2], high);
    }
}

long long up256(long long v) { return (v + 255) & ~255ll; }

// Fills in everything that follows from the sizes; false: not a shape these kernels take
bool stack_plan(StackArgs& a, long long* bytes) {
    const int nqkv = (a.n_heads + 2 * a.n_kv) * kHeadDim;
    if (a.B < 1 || a.B > kStMaxTokens || a.n_layers < 1 || a.n_layers > 4096 || a.n_heads < 1 || a.n_kv < 1) return false;
    if (a.n_heads % a.n_kv || a.n_heads * kHeadDim != a.dim || a.S < 1) return false;
    const int g = a.n_heads / a.n_kv;
    if (g != 1 && g != 2 && g != 4 && g != 8) return false;
    a.group = g;
    if (a.dim % 64 || a.dim > kStWaves * kStUpwD * 64 || a.ffn < 64 || a.ffn % 64 || a.ffn > kStWaves * kStUpwF * 64) return false;
    if (a.n_splits < 1 || a.n_splits > kDfMaxSplits) return false;
    const int nq = a.B <= kStDirect ? 0 : a.B;
    const int counts[9] = {nq, nqkv / 32, a.n_kv * a.n_splits * a.B, nq, a.dim / 16, nq, (a.ffn / 16 + 1) / 2, nq, a.dim / 16};
    int sum = 0;
    for (int i = 0; i < 9; ++i) a.ends[i] = sum += counts[i];
    if ((long long)sum * a.n_layers > (1ll << 30)) return false;
    long long f = up256((long long)a.B * nqkv * 2);
    a.f_o = (int)f;
    f = up256(f + (long long)a.B * a.dim * 2);
    a.f_ha = (int)f;
    f = up256(f + (long long)a.B * a.dim * 2);
    a.f_g = (int)f;
    f = up256(f + (long long)a.B * a.ffn * 2);
    a.f_hb = (int)f;
    f = up256(f + (long long)a.B * a.dim * 2);
    a.f_rec = (int)f;
    if (nq) f = up256(f + 4ll * a.B * (long long)sizeof(RowRecord));
    a.f_layer = (int)f;
    const long long rows = nq ? up256((long long)a.B * (3ll * a.dim + a.ffn)) : 0;
    if ((f + rows) * a.n_layers > (1ll << 30)) return false;
    a.f_bytes = (int)rows;
    a.set_values = (int)(f * a.n_layers);
    a.set_bytes = (int)((f + rows) * a.n_layers);
    a.sets = up256(sizeof(StackControl));
    a.records = a.sets + 2ll * a.set_bytes;
    a.inv_dim = 1.0f / (float)a.dim;
    a.inv_ffn = 1.0f / (float)a.ffn;
    *bytes = up256(a.records + (long long)a.B * a.n_kv * a.n_splits * kStMaxG * kDfRecUnits * 8);
    return true;
}

}  // namespace

// in decoder_ops.hip: threads the attention kernel of this shape runs with; 0: a shape it does not take
int bitnet_attn_decode_threads(int B, int S, int n_heads, int n_kv_heads, int n_splits);

static int stack_launch(StackArgs a, const void* entries, void* workspace, uint16_t* h_out, const int64_t* positions, int n_layers, int B, int S, int dim, int ffn,
                        int n_heads, int n_kv_heads, int n_splits, int workgroups, int spin_limit, void* stream) {
    a.n_layers = n_layers, a.B = B, a.S = S, a.dim = dim, a.ffn = ffn, a.n_heads = n_heads, a.n_kv = n_kv_heads, a.n_splits = n_splits;
    long long bytes = 0;
    if (!stack_plan(a, &bytes)) return 1;
    const int threads = bitnet_attn_decode_threads(B, S, n_heads, n_kv_heads, n_splits);
    if (!threads) return 1;
    if (!entries || !workspace || !a.h_in || !h_out || !positions || !a.cos || !a.sin) return 2;
    if (((uintptr_t)entries & 63u) || ((uintptr_t)workspace & 255u) || ((uintptr_t)a.h_in & 15u) || ((uintptr_t)h_out & 15u)) return 1;
    a.entries = (const __attribute__((address_space(4))) StackEntry*)entries;
    a.ws = (unsigned char*)workspace;
    a.h_out = h_out;
    a.positions = (const __attribute__((address_space(4))) int64_t*)positions;
    a.attn_waves = threads / 64;
    a.spin_limit = spin_limit > 0 ? spin_limit : kStSpinLimit;
    int grid = workgroups;
    if (grid <= 0) {  // one per CU
        static int cus[bitnet_host::kMaxDevices];
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= bitnet_host::kMaxDevices) return 3;
        if (!cus[dev]) {
            int n = 0;
            if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) return 3;
            cus[dev] = n;
        }
        grid = cus[dev];
    }
#define BITNET_STACK(MT) hipLaunchKernelGGL(decode_stack_kernel<MT>, dim3(grid), dim3(kStThreads), 0, (hipStream_t)stream, a)
    if (B == 1) BITNET_STACK(1);
    else if (B == 2) BITNET_STACK(2);
    else if (B <= 4) BITNET_STACK(4);
    else BITNET_STACK(8);
#undef BITNET_STACK
    return hipGetLastError() == hipSuccess ? 0 : 3;
}

extern "C" {

long long bitnet_decode_stack_workspace_bytes(int n_layers, int B, int S, int dim, int ffn, int n_heads, int n_kv_heads,
                                              int n_splits) {
    StackArgs a = {};
    a.n_layers = n_layers, a.B = B, a.S = S, a.dim = dim, a.ffn = ffn, a.n_heads = n_heads, a.n_kv = n_kv_heads, a.n_splits = n_splits;
    long long bytes = 0;
    if (!stack_plan(a, &bytes) || !bitnet_attn_decode_threads(B, S, n_heads, n_kv_heads, n_splits)) return -1;
    return bytes;
}

int bitnet_decode_stack_reset(void* workspace, int n_layers, int B, int S, int dim, int ffn, int n_heads, int n_kv_heads,
                              int n_splits, void* stream) {
    StackArgs a = {};
    a.n_layers = n_layers, a.B = B, a.S = S, a.dim = dim, a.ffn = ffn, a.n_heads = n_heads, a.n_kv = n_kv_heads, a.n_splits = n_splits;
    long long bytes = 0;
    if (!stack_plan(a, &bytes)) return 1;
    if (!workspace) return 2;
    if ((uintptr_t)workspace & 255u) return 1;
    hipLaunchKernelGGL(decode_stack_reset_kernel, dim3(1024), dim3(256), 0, (hipStream_t)stream, (v4u*)workspace, bytes >> 4, a.sets >> 4,
                       (long long)a.set_bytes >> 4, (long long)a.set_values >> 4);
    return hipGetLastError() == hipSuccess ? 0 : 3;
}

int bitnet_decode_stack_error_offset(void) { return (int)offsetof(StackControl, error); }

int bitnet_decode_stack(const void* entries, void* workspace, const uint16_t* h_in, uint16_t* h_out, const int64_t* positions,
                        const float* rope_rows, int n_layers, int B, int S, int dim, int ffn, int n_heads, int n_kv_heads,
                        int n_splits, int workgroups, int spin_limit, void* stream) {
    StackArgs a = {};
    a.h_in = h_in, a.in_rows = B;
    a.cos = rope_rows, a.sin = rope_rows ? rope_rows + kHeadDim / 2 : nullptr, a.factors = kHeadDim;
    return stack_launch(a, entries, workspace, h_out, positions, n_layers, B, S, dim, ffn, n_heads, n_kv_heads, n_splits, workgroups,
                        spin_limit, stream);
}

int bitnet_decode_stack_step(const void* entries, void* workspace, const int64_t* tokens, const uint16_t* emb, const float* cos_table,
                             const float* sin_table, uint16_t* h_out, const int64_t* positions, int V, int n_layers, int B, int S,
                             int dim, int ffn, int n_heads, int n_kv_heads, int n_splits, int workgroups, int spin_limit,
                             void* stream) {
    if (V < 1 || dim < 1 || (long long)V * dim * 2 > kBeyond) return 1;  // 32-bit byte offsets into the embedding
    if (!tokens) return 2;
    StackArgs a = {};
    a.h_in = emb, a.in_rows = V;
    a.tokens = (const __attribute__((address_space(4))) int64_t*)tokens;
    a.cos = cos_table, a.sin = sin_table, a.factors = kHeadDim / 2;
    return stack_launch(a, entries, workspace, h_out, positions, n_layers, B, S, dim, ffn, n_heads, n_kv_heads, n_splits, workgroups,
                        spin_limit, stream);
}

int bitlinear_probe_stack_math(int what, float by, uint32_t first, uint32_t n, uint32_t* found, void* stream) {
    if (what < 0 || what > 3 || !(by > 0.0f) || !n) return BITLINEAR_ERR_ARG;
    if (!found) return BITLINEAR_ERR_NULL;
    hipLaunchKernelGGL(decode_stack_math_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, what, by, first, n, found);
    return hipGetLastError() == hipSuccess ? BITLINEAR_OK : BITLINEAR_ERR_LAUNCH;
}

}  // extern "C"
