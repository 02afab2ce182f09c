// Weight layout converters on the device: ternary int8 [N, K] <-> the packed int8 [N, K / 4] of the
// reference packer (gpu/pack_weight.py:76-98; the closed form is spelled out in
// bitnet_amd/pack_weight.py).  Both directions move every byte once and compute on whole words.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bitlinear_hip.h"
#include "host_util.h"

namespace {

// HBM-bound: N * K bytes on one side, N * K / 4 on the other.  One packed word is 16 consecutive k of
// one row, a 16-row x 32-k tile is 32 words, and tiles of a row block are contiguous, so a lane takes
// four rows x 16 k: four 16-byte pieces of the ternary matrix and one 16-byte piece of the packed one.
// A wave takes 16 rows x 256 k (eight tiles): 256 contiguous bytes per row on the one side, 1 KB on
// the other.  As a chain of torch operations (13 passes and two host round trips for the range check)
// packing 13824 x 2560 took 265 us, now 20 (the copy of its 44 MB takes 9; the rest is the host waiting).
constexpr int kPackThreads = 256;
constexpr int kPackTiles = 8;  // tiles per wave

struct PackPlace {
    size_t w_off;    // first of the lane's four pieces in the ternary matrix, in 16-byte units
    size_t p_off;    // the lane's piece of the packed matrix, in 16-byte units
    int row_pieces;  // distance of the four pieces
    bool valid;
};

__device__ __forceinline__ PackPlace pack_place(int row_blocks, int tiles) {
    const int lane = threadIdx.x & 63;
    const int groups = (tiles + kPackTiles - 1) / kPackTiles;
    const long long wave = (long long)blockIdx.x * (kPackThreads / 64) + (threadIdx.x >> 6);
    const long long nb = wave / groups;
    const int h = lane & 1, kb = (int)(wave - nb * groups) * kPackTiles + ((lane >> 1) & 7);
    const int quad = lane >> 4;  // rows 4 quad .. 4 quad + 3 of the block: r_hi = quad / 2, r_lo = 4 (quad % 2) + i
    PackPlace p;
    p.valid = nb < row_blocks && kb < tiles;
    p.row_pieces = tiles * 2;
    p.w_off = ((size_t)nb * 16 + quad * 4) * p.row_pieces + (size_t)kb * 2 + h;
    p.p_off = ((size_t)nb * tiles + kb) * 8 + (quad >> 1) * 4 + h * 2 + (quad & 1);
    return p;
}

// Four ternary bytes -> their two-bit codes (w + 2), each in the low bits of its byte.  `bad` collects
// the bits in which a byte differs from all of -1, 0 and 1.
__device__ __forceinline__ uint32_t codes4(uint32_t d, uint32_t& bad) {
    const uint32_t neg = ((d >> 7) & 0x01010101u) * 0xffu;
    bad |= (d ^ neg) & (0xfefefefeu | neg);
    return (d & 0x03030303u) ^ 0x02020202u;
}

__global__ __launch_bounds__(kPackThreads) void pack_int2_kernel(const uint4* __restrict__ w, uint4* __restrict__ packed,
                                                                 int* bad_flag, int row_blocks, int tiles) {
    const PackPlace p = pack_place(row_blocks, tiles);
    if (!p.valid) return;
    uint4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = w[p.w_off + (size_t)i * p.row_pieces];
    uint32_t out[4], bad = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)  // byte e % 4 of the word, bits 2 (e / 4): the four dwords side by side
        out[i] = codes4(v[i].x, bad) | (codes4(v[i].y, bad) << 2) | (codes4(v[i].z, bad) << 4) | (codes4(v[i].w, bad) << 6);
    packed[p.p_off] = make_uint4(out[0], out[1], out[2], out[3]);
    if (bad) __hip_atomic_store(bad_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A word's codes at bits 2 S of every byte -> four bytes code - 2
template <int S>
__device__ __forceinline__ uint32_t ternary4(uint32_t word) {
    const uint32_t x = ((word >> (2 * S)) & 0x03030303u) ^ 0x02020202u;  // two-bit two's complement
    return x | (((x >> 1) & 0x01010101u) * 0xfcu);
}

__global__ __launch_bounds__(kPackThreads) void unpack_int2_kernel(const uint4* __restrict__ packed, uint4* __restrict__ w,
                                                                   int row_blocks, int tiles) {
    const PackPlace p = pack_place(row_blocks, tiles);
    if (!p.valid) return;
    const uint4 v = packed[p.p_off];
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i)
        w[p.w_off + (size_t)i * p.row_pieces] = make_uint4(ternary4<0>(d[i]), ternary4<1>(d[i]), ternary4<2>(d[i]), ternary4<3>(d[i]));
}

// the launch's grid; 0 for a shape the layout does not have
unsigned pack_grid(int N, int K) {
    if (N <= 0 || K <= 0 || N % 16 || K % 32) return 0;
    const long long waves = (long long)(N / 16) * ((K / 32 + kPackTiles - 1) / kPackTiles);
    const long long blocks = (waves + kPackThreads / 64 - 1) / (kPackThreads / 64);
    return blocks < (1ll << 31) ? (unsigned)blocks : 0;
}

}  // namespace

extern "C" {

int bitlinear_pack_int2(const int8_t* ternary, int8_t* packed, int32_t* bad_flag, int N, int K, void* stream) {
    const unsigned grid = pack_grid(N, K);
    if (!grid) return BITLINEAR_ERR_SHAPE;
    if (!ternary || !packed || !bad_flag) return BITLINEAR_ERR_NULL;
    if ((((uintptr_t)ternary) | ((uintptr_t)packed)) & 15u) return BITLINEAR_ERR_ARG;
    hipLaunchKernelGGL(pack_int2_kernel, dim3(grid), dim3(kPackThreads), 0, (hipStream_t)stream, (const uint4*)ternary,
                       (uint4*)packed, bad_flag, N / 16, K / 32);
    return hipGetLastError() == hipSuccess ? BITLINEAR_OK : BITLINEAR_ERR_LAUNCH;
}

int bitlinear_unpack_int2(const int8_t* packed, int8_t* ternary, int N, int K, void* stream) {
    const unsigned grid = pack_grid(N, K);
    if (!grid) return BITLINEAR_ERR_SHAPE;
    if (!ternary || !packed) return BITLINEAR_ERR_NULL;
    if ((((uintptr_t)ternary) | ((uintptr_t)packed)) & 15u) return BITLINEAR_ERR_ARG;
    hipLaunchKernelGGL(unpack_int2_kernel, dim3(grid), dim3(kPackThreads), 0, (hipStream_t)stream, (const uint4*)packed,
                       (uint4*)ternary, N / 16, K / 32);
    return hipGetLastError() == hipSuccess ? BITLINEAR_OK : BITLINEAR_ERR_LAUNCH;
}

}  // extern "C"
