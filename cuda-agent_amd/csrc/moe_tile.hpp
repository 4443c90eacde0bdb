// Device helpers shared by the MoE GEMMs whose workgroups stage weight rows and pair rows of one expert in LDS
// (moe_gemm_tiled.hip, moe_gemm_narrow.hip): operand types, global -> LDS loads, and the mapping of workgroups to tiles.
#pragma once
#include "lds_load.hpp"
#include "moe_common.hpp"

namespace moe {

typedef int intx8 __attribute__((ext_vector_type(8)));
typedef int intx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef const __attribute__((address_space(3))) uint8_t* lds_bytes;
typedef const __attribute__((address_space(3))) intx4* lds_x4;

constexpr int SUPER_ROWS = 4;   // row tiles and pair tiles of the block of workgroups that
constexpr int SUPER_PAIRS = 8;  // run together on one XCD and share its L2

// (one part of the tiles per XCD: find_tile)
inline int tiled_grid(int row_tiles, int max_pair_tiles) { return (row_tiles * max_pair_tiles + 7) / 8 * 8; }

template <int N>
struct IntConstant {
    static constexpr int value = N;
};

__device__ __forceinline__ intx8 join(intx4 lo, intx4 hi) {
    return intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// 8 e4m3 codes (two dwords) -> 8 bf16, exactly (every e4m3 value is a bf16 value)
__device__ __forceinline__ bf16x8 e4m3x8_to_bf16(int lo, int hi) {
    const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
    const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
    const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
    const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

__device__ __forceinline__ void wait_all_loads() {
    __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));  // vmcnt(0)
    asm volatile("" ::: "memory");
}

using lds::dma16;  // (completion is awaited once per block, before the barrier)
using lds::dma16_once;

// The tile of a workgroup: row tile `rb` of expert `e`, pair tile number `pt` of the table (see
// moe_tiled_prepare_kernel), which is tile `in_expert` of that expert's. False if there is none. Consecutive workgroup
// ids go round-robin to the 8 XCDs, each with its own L2: every XCD takes as many tiles as any other, to within
// one, in an order in which the 32 workgroups that run together on it are mostly a 4 x 8 block of (row tile, pair tile): they
// share 4 weight tiles and 8 activation tiles through that L2 instead of pulling 18 different ones. Neighbouring blocks go to
// different XCDs, since experts with many pairs stand together with others in no XCD's favour. (Whole blocks dealt out, one
// XCD could have one more than another, and where the row tiles are not a multiple of 4 every second or third block was
// partly empty, always on the same XCDs: 8192 tokens of 128 experts of 2048 x 768
// 0.71 ms, 0.88 dealt like that; of 64 experts of 4096 x 1536 1.03, 1.06; of 256 of 7168 x 2048 4.26, 4.31. In eight runs of neighbours, one each: 3 to 7 % slower where a sixteenth
// of 256 experts is chosen e^2 times as readily.)
__device__ __forceinline__ bool find_tile(const int* __restrict__ tile_start, int n_experts, int row_tiles, int& rb,
                                          int& e, int& in_expert) {
    const int total_tiles = tile_start[n_experts];
    const int n = total_tiles * row_tiles;
    const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
    const int dealt = n / 256 * 32;  // tiles that every XCD gets in runs of 32; what is left is cut into eight parts
    int at;
    if (turn < dealt) {
        at = turn / 32 * 256 + xcd * 32 + turn % 32;
    } else {
        const int left = n - dealt * 8;
        at = dealt * 8 + left * xcd / 8 + (turn - dealt);
        if (at >= dealt * 8 + left * (xcd + 1) / 8) return false;
    }
    const int group = at / (row_tiles * SUPER_PAIRS);  // of 8 pair tiles, the last of what is left
    const int pairs = min(SUPER_PAIRS, total_tiles - group * SUPER_PAIRS);
    at -= group * row_tiles * SUPER_PAIRS;
    const int block = at / (SUPER_ROWS * pairs);  // of 4 row tiles, the last of what is left
    const int rows = min(SUPER_ROWS, row_tiles - block * SUPER_ROWS);
    at -= block * SUPER_ROWS * pairs;
    rb = block * SUPER_ROWS + at % rows;
    const int pt = group * SUPER_PAIRS + at / rows;
    int lo = 0, hi = n_experts;  // largest slot with tile_start[slot] <= pt
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (tile_start[mid] <= pt) lo = mid; else hi = mid;
    }
    e = tile_start[n_experts + 1 + lo];  // the expert in that slot of the dispatch order
    in_expert = pt - tile_start[lo];
    return true;
}

}  // namespace moe
