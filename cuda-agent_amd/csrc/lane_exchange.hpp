// Sums and maxima across lanes on the vector ALU: v_permlane32_swap and v_permlane16_swap between the halves and the rows of 16
// lanes, DPP rotations inside a row. Every result is that of the butterfly `for (off = FROM; off >= TO; off /= 2) v = op(v,
// __shfl_xor(v, off))` bit for bit, whose every step is a trip through the LDS crossbar of about 100 cycles (us, with those and
// with these: a GDN layer step of 37 requests 34.2, 31.4; sparse attention of 64 requests over 32768 rows 166, 161). They are not the
// faster ones everywhere: where a chip full of wavefronts is bound by memory, those that finish sooner can be in the way of the
// others' loads (gdn_decode.hip, moe_quant.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lanes {

// v of the lower and of the upper half of the wavefront, in both halves
__device__ __forceinline__ void both_halves(float v, float& lower, float& upper) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    lower = __uint_as_float(r[0]), upper = __uint_as_float(r[1]);
}

// v of lane l ^ 32
__device__ __forceinline__ float other_half(float v) {
    float lower, upper;
    both_halves(v, lower, upper);
    return (threadIdx.x & 32) != 0 ? lower : upper;
}

__device__ __forceinline__ float max_of_halves(float v) {
    float lower, upper;
    both_halves(v, lower, upper);
    return fmaxf(lower, upper);
}

__device__ __forceinline__ float sum_of_halves(float v) {
    float lower, upper;
    both_halves(v, lower, upper);
    return lower + upper;
}

// v of lane (l + N) % 16 of the row
template <int N>
__device__ __forceinline__ float row_rotated(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x120 + N, 0xf, 0xf, false));
}

// op over the lanes that differ in the bits FROM, FROM/2 .. TO of their number. All lanes of a row that takes part are active, and
// of two rows, or halves, that exchange. (Once the lanes 8 apart have the same value, a rotation by 4 brings that of
// lane ^ 4, and so on down.)
template <int FROM, int TO, typename Op>
__device__ __forceinline__ float butterfly(float v, Op op) {
    static_assert(FROM == 8 || FROM == 16 || FROM == 32, "starts between the lanes, rows or halves");
    if constexpr (FROM == 32) {
        float lower, upper;
        both_halves(v, lower, upper);
        v = op(lower, upper);
    }
    if constexpr (FROM >= 16 && TO <= 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    if constexpr (TO <= 8) v = op(v, row_rotated<8>(v));
    if constexpr (TO <= 4) v = op(v, row_rotated<4>(v));
    if constexpr (TO <= 2) v = op(v, row_rotated<2>(v));
    if constexpr (TO <= 1) v = op(v, row_rotated<1>(v));
    return v;
}

template <int FROM, int TO = 1>
__device__ __forceinline__ float butterfly_sum(float v) {
    return butterfly<FROM, TO>(v, [](float a, float b) { return a + b; });
}

template <int FROM, int TO = 1>
__device__ __forceinline__ float butterfly_max(float v) {
    return butterfly<FROM, TO>(v, [](float a, float b) { return fmaxf(a, b); });
}

// Inclusive prefix sum over the lanes of a wavefront: running sums inside each row of 16 lanes on DPP row
// shifts (vector ALU; the __shfl_up form is six dependent trips through the LDS crossbar), then the totals of
// the rows before a lane's own, read as scalars.
__device__ __forceinline__ int inclusive_sum(int v, int lane) {
#define ROW_SHR_ADD(n) v += __builtin_amdgcn_update_dpp(0, v, 0x110 + (n), 0xf, 0xf, false);
    ROW_SHR_ADD(1)
    ROW_SHR_ADD(2)
    ROW_SHR_ADD(4)
    ROW_SHR_ADD(8)
#undef ROW_SHR_ADD
    const int r0 = __builtin_amdgcn_readlane(v, 15);
    const int r1 = __builtin_amdgcn_readlane(v, 31);
    const int r2 = __builtin_amdgcn_readlane(v, 47);
    const int row = lane >> 4;
    return v + (row >= 1 ? r0 : 0) + (row >= 2 ? r1 : 0) + (row >= 3 ? r2 : 0);
}

}  // namespace lanes
