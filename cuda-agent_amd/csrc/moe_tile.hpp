// Device helpers shared by the MoE GEMMs whose workgroups stage weight rows and pair rows of one expert in LDS
// (moe_gemm_tiled.hip, moe_gemm_narrow.hip): operand types, global -> LDS loads, and the mapping of workgroups to tiles.
#pragma once
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
constexpr int SUPER_PAIRS = 8;  // share one XCD's L2

inline int tiled_grid(int row_tiles, int max_pair_tiles) {
    const int supers = ((row_tiles + SUPER_ROWS - 1) / SUPER_ROWS) * ((max_pair_tiles + SUPER_PAIRS - 1) / SUPER_PAIRS);
    return ((supers + 7) / 8) * 8 * SUPER_ROWS * SUPER_PAIRS;
}

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

// 64 lanes x 16 bytes, global -> LDS (lds_base + lane*16); asm so that the compiler does not
// make every later LDS read wait for it: completion is awaited once per block, before the barrier.
__device__ __forceinline__ void dma16(const void* base, uint32_t lane_byte_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_byte_offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}

// The same with the non-temporal hint, for bytes that this launch reads once.
__device__ __forceinline__ void dma16_once(const void* base, uint32_t lane_byte_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                 :
                 : "v"(lane_byte_offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}

// The tile of a workgroup: row tile `rb` of expert `e`, pair tile number `pt` of the table (see
// moe_tiled_prepare_kernel), which is tile `in_expert` of that expert's. False if there is none. Consecutive workgroup
// ids go round-robin to the 8 XCDs, each with its own L2, so the 32 workgroups that run together on one XCD are given
// a 4 x 8 block of (row tile, pair tile): they share 4 weight tiles and 8 activation tiles through that L2 instead of
// pulling 18 different ones.
__device__ __forceinline__ bool find_tile(const int* __restrict__ tile_start, int n_experts, int row_tiles, int& rb,
                                          int& e, int& in_expert) {
    const int total_tiles = tile_start[n_experts];
    const int row_blocks4 = (row_tiles + SUPER_ROWS - 1) / SUPER_ROWS;
    const int linear = blockIdx.x;
    const int super = ((linear >> 3) / (SUPER_ROWS * SUPER_PAIRS)) * 8 + (linear & 7);
    const int within = (linear >> 3) % (SUPER_ROWS * SUPER_PAIRS);
    rb = (super % row_blocks4) * SUPER_ROWS + within % SUPER_ROWS;
    const int pt = (super / row_blocks4) * SUPER_PAIRS + within / SUPER_ROWS;
    if (rb >= row_tiles || pt >= total_tiles) return false;
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
