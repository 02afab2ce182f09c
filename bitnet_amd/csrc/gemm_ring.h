// Prefill GEMM whose operands both travel through LDS (included by bitlinear_hip.hip): int8 activation rows and packed
// weight words come by direct-to-LDS loads into a ring of S stages of CK k each.
//
// For outputs of about one tile per CU.  A tile is then alone on its CU, and what the other kernels leave to the next
// workgroup to hide is in the open: their loops request a chunk or two ahead and stop at every wait (512 x 3840 x 2560,
// 240 tiles of 64 x 128: 9.4 us, of which the matrix instructions are 2.2).  Measured here, on a lone tile (cycles of
// one CU at 2.4 GHz):
//  * loads bring 54 to 60 bytes a cycle into a CU whatever they are, so a tile's bytes are worth as much attention as its
//    multiplications (64 x 128: 96 bytes per k, 1.9 us at K = 2560).  Two thirds of LDS is ring.
//  * the first stages are there some 2000 cycles behind the start, of which half is the trip to memory.  So three stages are
//    requested, two waited for, and the ring is filled up beside the first two chunks: with S - 1 stages in front of
//    the first wait it ended after 3050 cycles (512 x 2560 x 2560 7.95 -> 7.6 us).  The instance without loader waves
//    requests S - 1 stages at once, and waits for the first two alone: a weight scale that is converted where it is
//    loaded makes the wave wait for all its requests there, at K = 2560 for all of K.
//  * a request behind the end of K costs what any other does (its zeros are written into LDS), so there are none: the last
//    S - 1 chunks wait for fewer and fewer stages.  Both together: 101 x 3840 x 2560 5.35 -> 4.9 us, 60 x 2560 x 640 4.3 -> 3.8.
//  * what the epilogue reads from memory (residual, scales, angles) is requested in front of the exchange of the sums
//    (norm, wo and residual of 512 tokens 12.9 -> 12.5 us, norm, w2 and residual 20.9 -> 20.0).
//  * a wave that issues a load waits while the path is taken by others, and does not multiply meanwhile.  So LW further
//    waves do nothing but load (512 x 3840 x 2560: 9.2 -> 8.6 us); the 32 x 64 tile's eight computing waves issue their
//    few loads between the MFMAs instead (5.6 against 6.2 us).
//  * an MFMA hides about four vector instructions of its SIMD and every further one takes 2.5 to 4 cycles, two waves or
//    one, so a wave's tile is 64 x 64 where it can be (expanding a word is eight instructions, here for two MFMAs).
//  * LDS reads run at 220 bytes a cycle without conflicts (rows swizzled so that 16 rows at one piece fall on 16
//    different slots of the 256 bytes that the banks span), writes at 76: with KG groups of waves that split the k-steps
//    of a stage, sums go through LDS once, and with KG = 1 not at all (512 x 13824 x 2560: 21.2 -> 20.2 us).
//  * two loader waves instead of four: the 64 x 64 tile's loop 2.46 -> 3.06 us per 2560 k.  So where a stage's loads do not divide by
//    four some of those waves have one load less (64 x 96 tiles 13.6 -> 12.5 us at 512 x 2560 x 6912).
// One barrier per stage: behind it the next stage is complete for every wave, so the first operands of a stage are read
// while the one in front is still being multiplied, and the stage before that is free for the loaders.  (Behind the last
// chunk operands are read from a stage that was not requested; nothing multiplies them.)
// Beyond a tile's start and end it is the matrix instructions: 512 x 13824 x 2560 in 128 x 256 tiles is 13.3 us per 2560 k and
// 7.4 us besides, 11.0 on zeros (what the pipe's clock makes of the operands), and the same with half the expansions and two
// thirds of the LDS reads (a wave's tile 128 x 64), with seven instructions a word instead of eight, and with two k-groups.
// Codes are expanded to bytes that read 64 w, as in gemm_i2_prefill_dma_kernel, which also defines the interleaved column
// tiles of a wave.  K % 128 == 0.
#ifndef BITNET_AMD_GEMM_RING_H
#define BITNET_AMD_GEMM_RING_H

// A wave's tile is 32 MT x 32 NT; WM x WN waves side by side, KG of them one behind the other in k; LW loading waves (0:
// the computing ones load)
template <int MT, int NT, int WM, int WN, int KG, int CK, int S, int LW>
struct Ring {
    static constexpr int WAVES = WM * WN * KG;  // that compute
    static constexpr int LWAVES = LW ? LW : WAVES;  // that load
    static constexpr int TM = 32 * MT * WM, TN = 32 * NT * WN;
    static constexpr int KSTEPS = CK / 32;       // 32-k MFMA steps per stage
    static constexpr int KPW = KSTEPS / KG;      // ... of which a wave takes this many
    static constexpr int PPR = CK / 16;          // 16-byte pieces per activation row and stage
    static constexpr int RPI = 64 / PPR;         // activation rows one load instruction of a wave covers
    static constexpr int SWZ_SHIFT = PPR == 8 ? 1 : 0, SWZ = PPR == 8 ? 7 : 15;
    static constexpr int A_BYTES = TM * CK, W_BYTES = TN * CK / 4, STAGE = A_BYTES + W_BYTES;
    static constexpr int AR = A_BYTES / 1024 / LWAVES, WR = (W_BYTES / 1024 + LWAVES - 1) / LWAVES, LOADS = AR + WR;
    static constexpr int WX = W_BYTES / 1024 % LWAVES;  // not zero: that many loading waves have the last load of a stage, the others not
    static constexpr int OUT_ROW = TN * 4 + 16;  // bytes of a row of sums: 16 rows at one column fall on 16 different 16-byte slots
    static constexpr int RED = KG > 1 ? KG * TM * OUT_ROW : 0;
    static constexpr int LDS = S * STAGE > RED ? S * STAGE : RED;
    static constexpr int THREADS = 64 * (WAVES + LW);
    static constexpr int WGS = 2 * (LDS + TM * 8 + 64) <= 160 * 1024 ? 2 : 1;  // workgroups per CU
    static_assert(AR * LWAVES * 1024 == A_BYTES && W_BYTES % 1024 == 0 && (LW || WX == 0), "whole load instructions per wave");
    static_assert(KPW >= 2 && KPW % 2 == 0 && KPW * KG == KSTEPS, "operand registers alternate");
    static_assert(S >= 4 && (S - 1) * LOADS <= 63, "loads in flight are counted in six bits");
    static_assert(LDS + TM * 8 + 64 <= 160 * 1024, "LDS of a CU");
};
// What becomes of the outputs: what follows a prompt's product is a launch and a trip of its rows through memory less (in a
// layer of a 512-token prompt rope and cache write 5.8 us beside the GEMM's 8.4, together 9.5; the gate's output is half of
// what w13 wrote, 22 -> 20.9, and the norm behind it reads half, 6.0 -> 5.4).  RingPlain: rows of `out`, with the residual added if there is one.
struct RingPlain {
    static constexpr bool kGate = false, kRope = false;
};
// RingGate: the weight's rows are two halves, x1 and x3, and out = bf16(bf16(relu(x1)^2) * x3), half as wide.  A wave's two
// column tiles are the same columns of either half.
struct RingGate {
    static constexpr bool kGate = true, kRope = false;
};
// RingRope: the columns are heads of 128: q heads are rotated into q_out, k heads rotated and v heads copied into the cache
// rows of the tokens' positions (what rope_cache_tokens_kernel does with the rows, value for value)
struct RingRope {
    static constexpr bool kGate = false, kRope = true;
    const int64_t* positions;
    const float *cos_t, *sin_t;
    uint16_t *cache_k, *cache_v, *q_out;
    int T, S, n_heads, n_kv;
};
// N words, two to four
template <int N>
struct RingWords {
    typedef uint32_t type __attribute__((ext_vector_type(N)));
};
// a token's position, and the angles of N neighbouring pairs there
template <int N>
struct RingTurn {
    typedef float angles __attribute__((ext_vector_type(N)));
    int p;
    angles cs, sn;
};
constexpr int kRingBeyond = 0x7ffffff0;  // an offset behind every descriptor: nothing is fetched, zeros arrive

template <int MT, int NT, int WM, int WN, int KG, int CK, int S, int LW, class Epi>
__global__ __launch_bounds__(64 * (WM * WN * KG + LW)) __attribute__((amdgpu_waves_per_eu((WM * WN * KG + LW) * Ring<MT, NT, WM, WN, KG, CK, S, LW>::WGS / 4)))
void gemm_i2_prefill_kernel(
    const int8_t* __restrict__ act, const uint32_t* __restrict__ wq, int M, int N, int K, int flags,
    int row_tiles, int col_tiles, unsigned magic, const uint16_t* __restrict__ s, uint16_t* __restrict__ out, int32_t* __restrict__ acc_out,
    const uint16_t* __restrict__ ws, ScaleMap smap, const uint16_t* __restrict__ residual, const Epi epi) {
    typedef Ring<MT, NT, WM, WN, KG, CK, S, LW> R;
    constexpr int QR = 8 / NT;
    constexpr int COLS = Epi::kGate ? R::TN / 2 : R::TN;  // output columns of a tile
    // a wave's column tiles lie 32 columns (of the gate: half the rows) apart; otherwise they interleave, and their words are one read
    constexpr bool kApart = Epi::kGate || NT == 3;
    static_assert(NT != 3 || KG > 1, "outputs straight from the registers are those of interleaved column tiles");
    static_assert(!Epi::kGate || NT == 2, "a column tile of either half");
    extern __shared__ __attribute__((aligned(1024))) int8_t lds_x[];

    int row_tile, col_tile;
    if (!tile_of_workgroup(blockIdx.x, row_tiles, col_tiles, magic, row_tile, col_tile)) return;
    const bool has_out = flags != 0;  // repeats out != nullptr

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
    const int nl = lane & 31, kc = lane >> 5;
    const int m0 = row_tile * R::TM, n_base = col_tile * COLS;
    const int n_out = Epi::kGate ? N >> 1 : N;
    const int nchunks = (K + CK - 1) / CK;

    const int rows_here = (M - m0) < R::TM ? (M - m0) : R::TM;
    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc((void*)(act + (size_t)m0 * K), 0, rows_here * K, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)wq, 0, (N >> 2) * K, 0x00020000);

    const int lw = LW ? wave - R::WAVES : wave;  // (negative: a wave that does not load)
    // activation requests: rows XOR-swizzled in 16-byte pieces (by choice of the piece a lane fetches)
    int a_voff[R::AR], a_k[R::AR];
#pragma unroll
    for (int r = 0; r < R::AR; ++r) {
        const int row = (r * R::LWAVES + lw) * R::RPI + lane / R::PPR;
        a_k[r] = ((lane % R::PPR) ^ ((row >> R::SWZ_SHIFT) & R::SWZ)) * 16;
        a_voff[r] = row * K + a_k[r];
    }
    // weight requests: [k-step][row block][128 bytes] in the stage
    int w_voff[R::WR], w_k[R::WR];
#pragma unroll
    for (int r = 0; r < R::WR; ++r) {
        const int q = (r * R::LWAVES + lw) * 64 + lane;
        constexpr int per_step = R::TN / 16 * 8;
        const int ks = q / per_step;
        int blk = (q % per_step) / 8;
        if (Epi::kGate) {  // of a wave's four blocks two are x1's, two x3's
            const int half = (blk >> 1) & 1;
            blk = (n_base >> 4) + (blk >> 2) * 2 + (blk & 1);
            blk = (blk < (n_out >> 4) ? blk : (n_out >> 4) - 1) + half * (n_out >> 4);
        } else {
            blk += n_base >> 4;
            blk = blk < (N >> 4) ? blk : (N >> 4) - 1;  // (row blocks behind the last are never stored)
        }
        w_k[r] = ks * 32;
        w_voff[r] = blk * K * 4 + ks * 128 + (q & 7) * 16;
    }
    // part p of P of a stage's requests, `loads` a wave
    auto issue = [&](int c, int st, int p, int P, auto loads) {
        const int left = K - c * CK;  // k in front of the end of the rows
        int8_t* to = lds_x + st * R::STAGE;
#pragma unroll
        for (int r = 0; r < loads.value; ++r) {
            if (r * P / R::LOADS != p) continue;
            if (r < R::AR) {
                load16_to_lds(a_rsrc, to + (r * R::LWAVES + lw) * 1024, a_k[r] < left ? a_voff[r] : kRingBeyond, c * CK);
            } else {
                const int i = r - R::AR;
                load16_to_lds(w_rsrc, to + R::A_BYTES + (i * R::LWAVES + lw) * 1024, w_k[i] < left ? w_voff[i] : kRingBeyond, c * (CK * 4));
            }
        }
    };
    // all of a wave's requests have arrived but those of its last `stages` stages
    auto wait_all_but = [](auto stages, auto loads) {
        constexpr int n = decltype(stages)::value * decltype(loads)::value;
        __builtin_amdgcn_s_waitcnt(0x0f70 | (n & 15) | (n >> 4 << 14));
    };
    constexpr std::integral_constant<int, 0> none{};
    constexpr std::integral_constant<int, 1> one_stage{};
    constexpr std::integral_constant<int, 2> two_stages{};
    constexpr std::integral_constant<int, S - 3> full{};  // the ring's stages behind the two that are in use
    auto meet = [&] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    constexpr int kFirst = LW ? 3 : S - 1;  // stages requested in front of the first wait
    constexpr std::integral_constant<int, R::LOADS> all_loads{};
    auto first_stages = [&](auto loads) {
#pragma unroll
        for (int c = 0; c < kFirst; ++c)
            if (c < nchunks) issue(c, c, 0, 1, loads);
    };
    // what a loading wave does: at the end of chunk c stage c + 2 has to be there
    auto load_stages = [&](auto loads) {
        first_stages(loads);
        if (nchunks <= S) {  // all of K fits the ring
            wait_all_but(none, loads);
            meet();
            for (int c = kFirst; c < nchunks; ++c) issue(c, c, 0, 1, loads);
            wait_all_but(none, loads);
            for (int c = 0; c < nchunks; ++c) meet();
        } else {
            wait_all_but(one_stage, loads);
            meet();
            int c = 0, st = kFirst % S;
            auto next_stage = [&](int i) {
                issue(i, st, 0, 1, loads);
                st = st + 1 == S ? 0 : st + 1;
            };
            if constexpr (S > 4) {  // two stages at a time until S - 1 are on their way
                static_assert(S == 6, "two chunks of two stages");
                next_stage(3);
                next_stage(4);
                wait_all_but(two_stages, loads);
                meet();
                next_stage(5);
                next_stage(6);
                wait_all_but(full, loads);
                meet();
                c = 2;
            }
            for (; c + S - 1 < nchunks; ++c) {
                next_stage(c + S - 1);
                wait_all_but(full, loads);
                meet();
            }
            if constexpr (S > 4) {
                wait_all_but(two_stages, loads);
                meet();
                wait_all_but(one_stage, loads);
                meet();
            }
            wait_all_but(none, loads);
            for (int i = 0; i < 3; ++i) meet();
        }
        meet();
        lds_barrier();
    };
    if (LW && lw >= 0) {
        if constexpr (R::WX != 0) {
            if (lw >= R::WX) {
                load_stages(std::integral_constant<int, R::LOADS - 1>{});
                return;
            }
        }
        load_stages(all_loads);
        return;
    }
    if (!LW) first_stages(all_loads);

    // the outputs that go through LDS: eight of a row per thread, four where there are fewer
    constexpr int CPT = KG > 1 && R::TM * COLS < R::WAVES * 64 * 8 ? 4 : 8;
    constexpr int PER_ROW = COLS / CPT;            // threads that share a row
    constexpr int ROWS = R::WAVES * 64 / PER_ROW;  // rows that the threads cover at a time
    constexpr int TIMES = (R::TM + ROWS - 1) / ROWS;
    const int pr = threadIdx.x / PER_ROW < ROWS ? threadIdx.x / PER_ROW : R::TM, pc = threadIdx.x % PER_ROW * CPT, n = n_base + pc;
    // the scales, for the epilogue
    __shared__ float sval[R::TM], rinv[R::TM], wsv[kMaxSeg];
    uint32_t s_raw = 0, ws_raw = 0;
    if (has_out) {
        const int m = m0 + (int)threadIdx.x;
        if (threadIdx.x < R::TM) s_raw = s[m < M ? m : M - 1];
        if (threadIdx.x < kMaxSeg) ws_raw = ws[(int)threadIdx.x < smap.nseg ? threadIdx.x : 0];
    }
    auto put_scales = [&] {
        asm volatile("" : "+v"(s_raw), "+v"(ws_raw));  // (converted here and not where they are loaded, see the top)
        if (threadIdx.x < R::TM) {
            const float sv = bf16_to_f32((uint16_t)s_raw);
            sval[threadIdx.x] = sv;
            rinv[threadIdx.x] = 1.0f / sv;
        }
        if (threadIdx.x < kMaxSeg) wsv[threadIdx.x] = bf16_to_f32((uint16_t)ws_raw);
    };
    // with loader waves while the first stages are on their way (in the instances without k-groups behind the loop measures 0.3 us less)
    if (LW && KG > 1) put_scales();
    // ... as are the positions of this thread's outputs
    int64_t at[KG > 1 ? TIMES : MT] = {};
    if constexpr (Epi::kRope) {
#pragma unroll
        for (int i = 0; i < (KG > 1 ? TIMES : MT); ++i) {
            const int m = m0 + (KG > 1 ? i * ROWS + pr : (wm * MT + i) * 32 + nl);
            at[i] = epi.positions[m < M ? m : M - 1];
        }
    }

    v16i acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0;

    // where the lane's operands are within a stage
    typedef typename RingWords<NT>::type wvec_t;
    int a_rd[R::KPW];
#pragma unroll
    for (int j = 0; j < R::KPW; ++j)
        a_rd[j] = (wm * MT * 32 + nl) * CK + ((((grp * R::KPW + j) * 2 + kc) ^ ((nl >> R::SWZ_SHIFT) & R::SWZ)) * 16);
    const int w_rd = R::A_BYTES + grp * R::KPW * (R::TN * 8) +
                     (kApart ? (wn * NT * 2 + (nl >> 4)) * 128 + ((nl >> 3 & 1) * 16 + kc * 8 + (nl & 7)) * 4
                             : (wn * NT * 2 + nl / (2 * QR)) * 128 + (((nl % (2 * QR)) / QR) * 16 + kc * 8 + NT * (nl % QR)) * 4);
    auto expand = [&](uint32_t wd) -> v4i {
        const uint32_t x = wd ^ 0xAAAAAAAAu;
        v4i r;
        r.x = (int)((x << 6) & 0xC0C0C0C0u);
        r.y = (int)((x << 4) & 0xC0C0C0C0u);
        r.z = (int)((x << 2) & 0xC0C0C0C0u);
        r.w = (int)(x & 0xC0C0C0C0u);
        return r;
    };
    auto read_a = [&](const int8_t* stage, int j, v4i(&a)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[mt] = *(const v4i*)(stage + a_rd[j] + mt * 32 * CK);
    };
    auto read_w = [&](const int8_t* stage, int j) -> wvec_t {
        const int8_t* from = stage + w_rd + j * (R::TN * 8);
        if constexpr (kApart) {
            wvec_t w;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) w[nt] = *(const uint32_t*)(from + nt * 256);
            return w;
        } else {
            return *(const wvec_t*)from;
        }
    };
    // stages 0 and 1 are there (every wave waits for its own requests, then all meet)
    if (!LW) {
        if (nchunks < S - 1) wait_all_but(none, all_loads);
        else wait_all_but(full, all_loads);
    }
    meet();

    v4i aop[2][MT], bop[2][NT];
    wvec_t wraw[2];
    read_a(lds_x, 0, aop[0]);
    wraw[0] = read_w(lds_x, 0);
    wraw[1] = read_w(lds_x, 1);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) bop[0][nt] = expand(wraw[0][nt]);

    int st = 0;
    // chunk c; `load`: and part by part the requests of stage c + S - 1, into the stage in front of this one, which was read in
    // the chunk before and every wave has left
    auto chunk = [&](int c, auto load) {
        const int8_t* here = lds_x + st * R::STAGE;
        const int st1 = st + 1 == S ? 0 : st + 1;
        const int8_t* next = lds_x + st1 * R::STAGE;
        constexpr int SLOTS = MT * NT;
#pragma unroll
        for (int j = 0; j < R::KPW; ++j) {
            const int cur = j & 1, nxt = cur ^ 1;
#pragma unroll
            for (int slot = 0; slot < SLOTS; ++slot) {
                const int mt = slot / NT, nt = slot % NT;
                acc[mt][nt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bop[cur][nt], aop[cur][mt], acc[mt][nt], 0, 0, 0);
                if (slot == 0) {
                    if (j + 1 < R::KPW) read_a(here, j + 1, aop[nxt]);
                    else read_a(next, 0, aop[nxt]);
                    wraw[cur] = j + 2 < R::KPW ? read_w(here, j + 2) : read_w(next, j + 2 - R::KPW);
                }
#pragma unroll
                for (int i = 0; i < NT; ++i)
                    if ((i * SLOTS / NT + (SLOTS > NT ? 1 : 0)) % SLOTS == slot) bop[nxt][i] = expand(wraw[nxt][i]);
                if (load.value && slot == SLOTS - 1) issue(c + S - 1, st == 0 ? S - 1 : st - 1, j, R::KPW, all_loads);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        st = st1;
    };
    if constexpr (LW > 0) {
        for (int c = 0; c < nchunks; ++c) {
            chunk(c, std::false_type{});
            meet();
        }
    } else {
        for (int c = 0; c + S - 1 < nchunks; ++c) {
            chunk(c, std::true_type{});
            wait_all_but(full, all_loads);  // the chunk behind the next one has to be there before the next one ends
            meet();
        }
        auto last = [&](auto behind) {  // ... that has `behind` chunks behind it
            constexpr int n = decltype(behind)::value;
            if (nchunks <= n) return;
            chunk(0, std::false_type{});
            wait_all_but(std::integral_constant<int, (n > 2 ? n - 2 : 0)>{}, all_loads);
            meet();
        };
        static_assert(S == 6, "S - 1 chunks without requests");
        last(std::integral_constant<int, 4>{});
        last(std::integral_constant<int, 3>{});
        last(std::integral_constant<int, 2>{});
        last(std::integral_constant<int, 1>{});
        last(std::integral_constant<int, 0>{});
    }

    // the reference's epilogue (the bits of the IEEE divide by the token's scale from its reciprocal and one correction
    // step, as in gemm_i2_prefill_kernel): two neighbouring sums -> packed bf16
    auto result2 = [](int x, int y, float sv, float ri, float w) {
        const float a = (float)x, b = (float)y;
        const float p0 = a * ri, q0 = b * ri;
        return f32x2_to_bf16x2(__builtin_fmaf(__builtin_fmaf(-p0, sv, a), ri, p0) * w, __builtin_fmaf(__builtin_fmaf(-q0, sv, b), ri, q0) * w);
    };
    auto low = [](uint32_t d) { return __uint_as_float(d << 16); };
    auto high = [](uint32_t d) { return __uint_as_float(d & 0xffff0000u); };
    // two gated outputs (glu8's arithmetic)
    auto gate2 = [&](uint32_t x1, uint32_t x3) {
        const float r0 = fmaxf(low(x1), 0.0f), r1 = fmaxf(high(x1), 0.0f);
        const uint32_t sq = f32x2_to_bf16x2(r0 * r0, r1 * r1);
        return f32x2_to_bf16x2(low(sq) * low(x3), high(sq) * high(x3));
    };
    constexpr int PAIRS = CPT / 2;  // of neighbouring outputs, a word each
    typedef typename RingWords<PAIRS>::type words_t;
    typedef RingTurn<PAIRS> turn_t;
    auto turn_of = [&](int64_t at, int n) {
        turn_t t = {};
        if constexpr (Epi::kRope) {
            t.p = at < 0 ? 0 : (at >= (int64_t)epi.S ? epi.S - 1 : (int)at);  // nothing outside the buffers is touched
            t.cs = *(const typename turn_t::angles*)(epi.cos_t + (size_t)t.p * 64 + (n & 127) / 2);
            t.sn = *(const typename turn_t::angles*)(epi.sin_t + (size_t)t.p * 64 + (n & 127) / 2);
        }
        return t;
    };
    // CPT consecutive outputs of one token from their sums
    auto store = [&](int m, int n, const int(&x)[CPT], float sv, float ri, float w, const turn_t& turn, auto residual_here) {
        const size_t o = (size_t)m * N + n;
        if (!Epi::kRope && acc_out) {
#pragma unroll
            for (int i = 0; i < CPT; i += 4) *(v4i*)(acc_out + o + i) = v4i{x[i], x[i + 1], x[i + 2], x[i + 3]};
        }
        if (!has_out) return;
        words_t ob;
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) ob[i] = result2(x[2 * i], x[2 * i + 1], sv, ri, w);
        if constexpr (Epi::kRope) {
            const int head = n >> 7, in = n & 127;
            uint16_t* to = epi.q_out + ((size_t)m * epi.n_heads + head) * 128 + in;
            if (head >= epi.n_heads) {
                const int kv = head - epi.n_heads;
                to = (kv < epi.n_kv ? epi.cache_k : epi.cache_v) +
                     (((size_t)(m / epi.T) * epi.S + turn.p) * epi.n_kv + (kv < epi.n_kv ? kv : kv - epi.n_kv)) * 128 + in;
            }
            if (head < epi.n_heads + epi.n_kv) {
#pragma unroll
                for (int i = 0; i < PAIRS; ++i)
                    ob[i] = f32x2_to_bf16x2(low(ob[i]) * turn.cs[i] - high(ob[i]) * turn.sn[i], low(ob[i]) * turn.sn[i] + high(ob[i]) * turn.cs[i]);
            }
            *(words_t*)to = ob;
        } else {
            if (residual) {  // out = bf16(residual + bf16(result))
                const words_t res = residual_here(o);
#pragma unroll
                for (int i = 0; i < PAIRS; ++i) ob[i] = f32x2_to_bf16x2(low(res[i]) + low(ob[i]), high(res[i]) + high(ob[i]));
            }
            *(words_t*)(out + o) = ob;
        }
    };
    meet();
    if (!LW || KG == 1) put_scales();
    if constexpr (KG == 1) {
        // every wave holds its sums whole: 4 NT consecutive columns per register quad, stored straight from the registers
        lds_barrier();
        const int nw = n_base + wn * (COLS / WN);
        const int n_last = nw + COLS / WN - 1 < n_out ? nw + COLS / WN - 1 : n_out - 1;
        const int n_first = nw < n_out ? nw : n_out - 1;
        const int slot_first = scale_slot(smap, n_first);
        const int slot3 = Epi::kGate ? scale_slot(smap, n_out + n_first) : 0;
        const bool one_slot = slot_first == scale_slot(smap, n_last) && (!Epi::kGate || slot3 == scale_slot(smap, n_out + n_last));
        const float w1 = wsv[slot_first], w3 = wsv[slot3];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int row = (wm * MT + mt) * 32 + nl, m = m0 + row;
            const float sv = sval[row], ri = rinv[row];
            auto column = [&](int g4) {  // the first of a register quad's columns
                const int ridx = g4 * 8 + kc * 4;
                return Epi::kGate ? nw + ridx : nw + 16 * (ridx / (2 * QR)) + 8 * ((ridx % (2 * QR)) / QR) + NT * (ridx % QR);
            };
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int n = column(g4);
                if (m >= M || n >= n_out) continue;
                int x[4 * NT];
                if constexpr (Epi::kGate) {
                    const float wa = one_slot ? w1 : wsv[scale_slot(smap, n)], wb = one_slot ? w3 : wsv[scale_slot(smap, n_out + n)];
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] = acc[mt][i >> 2][g4 * 4 + (i & 3)] >> 6;
                    *(uint2*)(out + (size_t)m * n_out + n) =
                        make_uint2(gate2(result2(x[0], x[1], sv, ri, wa), result2(x[4], x[5], sv, ri, wb)),
                                   gate2(result2(x[2], x[3], sv, ri, wa), result2(x[6], x[7], sv, ri, wb)));
                } else {
#pragma unroll
                    for (int i = 0; i < 4 * NT; ++i) x[i] = acc[mt][i % NT][g4 * 4 + i / NT] >> 6;
                    turn_t turn = {};
                    if constexpr (Epi::kRope) turn = turn_of(at[mt], n);
                    store(m, n, x, sv, ri, one_slot ? w1 : wsv[scale_slot(smap, n)], turn, [&](size_t o) { return *(const words_t*)(residual + o); });
                }
            }
        }
        return;
    }
    // requested in front of the exchange
    turn_t turn[TIMES] = {};
    words_t res[TIMES] = {};
#pragma unroll
    for (int i = 0; i < TIMES; ++i) {
        if constexpr (Epi::kRope) turn[i] = turn_of(at[i], n);
    }
    if (!Epi::kGate && !Epi::kRope && residual) {
#pragma unroll
        for (int i = 0; i < TIMES; ++i) {
            const int row = i * ROWS + pr, m = m0 + row;
            if (row < R::TM && m < M && n < N) res[i] = *(const words_t*)(residual + (size_t)m * N + n);
        }
    }
    // The sums go through LDS, which adds the groups' shares and turns a lane's pieces of 32 rows into whole runs of a
    // row.  (A lane holds token nl; register quad g4 of its NT column tiles is 4 NT consecutive columns.)
    {
        int8_t* to = lds_x + (grp * R::TM + wm * MT * 32 + nl) * R::OUT_ROW + wn * (COLS / WN) * 4;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int ridx = g4 * 8 + kc * 4;
                const int n = kApart ? ridx : 16 * (ridx / (2 * QR)) + 8 * ((ridx % (2 * QR)) / QR) + NT * (ridx % QR);
#pragma unroll
                for (int v = 0; v < NT; ++v) {
                    v4i t;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int i = 4 * v + j;  // column n + i: register i / NT of the quad, column tile i % NT (apart: of tile v)
                        t[j] = kApart ? acc[mt][v][g4 * 4 + j] : acc[mt][i % NT][g4 * 4 + i / NT];
                    }
                    *(v4i*)(to + mt * 32 * R::OUT_ROW + (n + v * (Epi::kGate ? COLS : kApart ? 32 : 4)) * 4) = t;
                }
            }
    }
    const int slot = scale_slot(smap, n), slot3 = Epi::kGate ? scale_slot(smap, n_out + n) : 0;
    lds_barrier();
    const float w = wsv[slot], w3 = wsv[slot3];
    // (exact: the accumulators are 64 * sum(w * a))
    auto sums = [&](const int8_t* from, int(&x)[CPT]) {
#pragma unroll
        for (int i = 0; i < CPT; i += 4) {
            v4i t = *(const v4i*)(from + i * 4);
#pragma unroll
            for (int g = 1; g < KG; ++g) t += *(const v4i*)(from + g * R::TM * R::OUT_ROW + i * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[i + e] = t[e] >> 6;
        }
    };
#pragma unroll
    for (int p = 0; p < TIMES; ++p) {
        const int row = p * ROWS + pr, m = m0 + row;
        if (row >= R::TM || m >= M || n >= n_out) continue;  // N % 16 == 0: the columns are in or out together
        const int8_t* from = lds_x + row * R::OUT_ROW + pc * 4;
        const float sv = sval[row], ri = rinv[row];
        int x[CPT];
        sums(from, x);
        if constexpr (Epi::kGate) {
            int y[CPT];
            sums(from + COLS * 4, y);
            words_t ob;
#pragma unroll
            for (int i = 0; i < PAIRS; ++i)
                ob[i] = gate2(result2(x[2 * i], x[2 * i + 1], sv, ri, w), result2(y[2 * i], y[2 * i + 1], sv, ri, w3));
            *(words_t*)(out + (size_t)m * n_out + n) = ob;
        } else {
            store(m, n, x, sv, ri, w, turn[p], [&](size_t) { return res[p]; });
        }
    }
}

#endif
