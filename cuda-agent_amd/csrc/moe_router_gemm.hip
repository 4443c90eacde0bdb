// Router projection of a MoE layer: logits[t, e] = sum_h x[t, h] * w[e, h], fp32.
//
// x is the layer's bf16 (or fp32) input, w the fp32 router weight [n_experts, hidden]; both are
// taken to fp32 exactly and multiplied on the fp32 matrix cores (v_mfma_f32_32x32x2_f32), or, a bf16 x
// of 64 tokens or more, as three exact products on the bf16 matrix cores (moe_router_gemm_long_kernel). So the
// result differs from an fp32 reference only by the order of the additions: the routing that
// follows compares these logits with each other, and a lower-precision product would move
// experts across the top-k boundary.
//
// A wavefront owns a 32-token x 32-expert tile of the output. The MFMA pairs lane l's A value
// (token l % 32) with lane l's B value (expert l % 32) as one k of the dot product, and any
// assignment of k to (lane half, step) works as long as A and B agree. So for every 64 values of
// k lane (row, half) reads the 32 consecutive values [64c + 32*half, +32) of its row: whole
// 128-byte lines of w, 64-byte pieces of bf16 x, straight from global memory into the operand
// registers (at 64 cycles per MFMA the loads are a small fraction of the time and need no LDS
// staging). 4 wavefronts of a workgroup cover 64 tokens x 64 experts.
//
// Few tokens: K is cut into n_splits ranges (grid z) so that the weight matrix is streamed by
// many CUs; partial sums go to a caller-provided scratch and a second kernel adds them in
// ascending split order, so the result does not depend on timing.
//
// Split-weight form (moe_router_split_weight_launcher + moe_router_logits_split_launcher): an fp32
// weight is the exact sum of three bf16 numbers (its 24 significand bits cut into 8 + 8 + 8; from 2^-110 on), and a
// product of two bf16 numbers is exact in fp32. With the weight stored once as those three planes the
// projection of a bf16 x runs on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16: 8 times the rate of
// the fp32 shape, three products per weight) and still differs from an fp32 reference by the order of the
// additions only. At that rate the operand loads are what matters: rows are fetched as whole lines into LDS, where the
// wavefronts of a workgroup share them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch_status.hpp"
#include "lds_load.hpp"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int K_CHUNK = 64;

// 32 consecutive values of a row as fp32
__device__ __forceinline__ void load32(float (&dst)[32], const float* p) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const floatx4 v = reinterpret_cast<const floatx4*>(p)[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[4 * i + j] = v[j];
    }
}
__device__ __forceinline__ void load32(float (&dst)[32], const uint16_t* p) {  // bf16 bits
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const u32x4 v = reinterpret_cast<const u32x4*>(p)[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            dst[8 * i + 2 * j] = __uint_as_float(v[j] << 16);
            dst[8 * i + 2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u);
        }
    }
}

// Sums of chunks [chunk_begin, chunk_end) for 32 tokens x 32 experts on the fp32 matrix cores: lane (row, half) has the
// `half` 32 values of a chunk of its token's and of its expert's row, from xp and wp on. Register i of a lane: token
// 8*(i/4) + 4*half + i%4, expert `row`.
template <typename X>
__device__ __forceinline__ floatx16 fp32_tile(const X* __restrict__ xp, const float* __restrict__ wp, int chunk_begin,
                                              int chunk_end) {
    floatx16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // two register sets: the loads of chunk c+1 are in flight while the MFMAs of chunk c run
    float a0[32], b0[32], a1[32], b1[32];
    if (chunk_begin < chunk_end) {
        load32(a0, xp + (size_t)chunk_begin * K_CHUNK);
        load32(b0, wp + (size_t)chunk_begin * K_CHUNK);
    }
    for (int c = chunk_begin; c < chunk_end; c += 2) {
        // (past the end the last chunk is read again and not used)
        const int c1 = c + 1 < chunk_end ? c + 1 : c;
        load32(a1, xp + (size_t)c1 * K_CHUNK);
        load32(b1, wp + (size_t)c1 * K_CHUNK);
#pragma unroll
        for (int s = 0; s < 32; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[s], b0[s], acc, 0, 0, 0);
        if (c + 1 >= chunk_end) break;
        const int c2 = c + 2 < chunk_end ? c + 2 : c + 1;
        load32(a0, xp + (size_t)c2 * K_CHUNK);
        load32(b0, wp + (size_t)c2 * K_CHUNK);
#pragma unroll
        for (int s = 0; s < 32; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[s], b1[s], acc, 0, 0, 0);
    }
    return acc;
}

// grid: x = 64-token tiles, y = 64-expert tiles, z = K split. out is logits (n_splits == 1) or
// the partial sums [split][tokens][n_experts].
template <typename X>
__global__ __launch_bounds__(256) void moe_router_gemm_kernel(const X* __restrict__ x,
                                                              const float* __restrict__ w,
                                                              float* __restrict__ out, int tokens,
                                                              int hidden, int n_experts,
                                                              int chunks_per_split) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row = lane & 31;
    const int half = lane >> 5;
    const int t0 = blockIdx.x * 64 + (wave & 1) * 32;
    const int e0 = blockIdx.y * 64 + (wave >> 1) * 32;
    if (t0 >= tokens || e0 >= n_experts) return;  // (no barrier in this kernel)
    // rows beyond the end read the last valid row; their results are not stored
    const int t = t0 + row < tokens ? t0 + row : tokens - 1;
    const int e = e0 + row < n_experts ? e0 + row : n_experts - 1;
    const int chunk_begin = blockIdx.z * chunks_per_split;
    int chunk_end = chunk_begin + chunks_per_split;
    const int n_chunks = hidden / K_CHUNK;
    if (chunk_end > n_chunks) chunk_end = n_chunks;
    const floatx16 acc = fp32_tile(x + (size_t)t * hidden + 32 * half, w + (size_t)e * hidden + 32 * half, chunk_begin, chunk_end);
    // result register i of a lane: token 8*(i/4) + 4*half + i%4 of the tile, expert `row`
    float* dst = out + (size_t)blockIdx.z * tokens * n_experts;
    if (e0 + row < n_experts) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int tt = t0 + 8 * (i / 4) + 4 * half + (i % 4);
            if (tt < tokens) dst[(size_t)tt * n_experts + e0 + row] = acc[i];
        }
    }
}

// ---- split-weight form ---------------------------------------------------------------------------------

// w [n] fp32 -> planes [3][n] bf16 with hi + mid + lo == w exactly: hi = the upper 16 bits of w, mid the upper
// 16 bits of w - hi, lo = w - hi - mid (at most 8 significant bits are left, so it is a bf16 number)
__global__ __launch_bounds__(256) void moe_router_split_kernel(const float* __restrict__ w,
                                                               uint16_t* __restrict__ planes, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float v = w[i];
    const uint32_t hi = __float_as_uint(v) & 0xffff0000u;
    const float r1 = v - __uint_as_float(hi);
    const uint32_t mid = __float_as_uint(r1) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(mid);
    planes[i] = (uint16_t)(hi >> 16);
    planes[n + i] = (uint16_t)(mid >> 16);
    planes[2 * n + i] = (uint16_t)(__float_as_uint(r2) >> 16);
}

typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef const __attribute__((address_space(3))) uint8_t* lds_bytes;

// grid: x = 64-token tiles, y = 32-expert tiles, z = K split; out as in moe_router_gemm_kernel
// A workgroup owns 64 tokens x 32 experts of one K split; wavefronts 0 and 1 multiply 32 tokens each, all four fetch. What
// bounds it is the latency of its loads: a split is a few chunks of 64 values of k, and up to FETCHED_CHUNKS of them (64 rows of x and
// 3 x 32 of the planes, 128 bytes each = 20 KB) are on their way into LDS before the first is waited for. (8 lanes fetch the line of
// a row, whose chunk p lies in slot p ^ ((row >> 1) & 7); a lane (row, half) of an operand holds values [32*half, +32) of its row, 8
// per MFMA step.)
// us of the projection, one chunk ahead through registers and 64 experts a workgroup, and this: 64 tokens of 7168 x 256 11.0, 8.8;
// 100 11.2, 10.0; 250 of 4096 x 128 10.2, 9.1; 1500 of 4096 x 64 15.3, 13.9; 1400 of 1024 x 256 14.0, 12.7.
template <int FETCHED_CHUNKS>
__global__ __launch_bounds__(256) void moe_router_gemm_split_kernel(const uint16_t* __restrict__ x,
                                                                    const uint16_t* __restrict__ planes,
                                                                    float* __restrict__ out, int tokens,
                                                                    int hidden, int n_experts,
                                                                    int chunks_per_split) {
    constexpr int LOADS = 5;  // load instructions of a wavefront per chunk
    constexpr int X_BYTES = 64 * K_CHUNK * 2, PLANE_BYTES = 32 * K_CHUNK * 2, CHUNK_BYTES = X_BYTES + 3 * PLANE_BYTES;
    __shared__ __attribute__((aligned(16))) uint8_t s_chunk[FETCHED_CHUNKS * CHUNK_BYTES];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 31;
    const int half = lane >> 5;
    const int t0 = blockIdx.x * 64;
    const int e0 = blockIdx.y * 32;
    const int chunk_begin = blockIdx.z * chunks_per_split;
    const int n = min(chunks_per_split, hidden / K_CHUNK - chunk_begin);  // (not positive: this split is empty)

    // fill side: a wavefront fetches 8 rows of x twice, and 8 of every plane (rows past the end repeat the last)
    const int ld_row = 8 * wave + (lane >> 3);
    const size_t ld_piece = (size_t)chunk_begin * K_CHUNK + 8 * ((lane & 7) ^ ((ld_row >> 1) & 7));
    const uint16_t* src[3] = {x + (size_t)min(t0 + ld_row, tokens - 1) * hidden + ld_piece,
                              x + (size_t)min(t0 + 32 + ld_row, tokens - 1) * hidden + ld_piece,
                              planes + (size_t)min(e0 + ld_row, n_experts - 1) * hidden + ld_piece};
    const size_t plane = (size_t)n_experts * hidden;
    const uint32_t lds0 = (uint32_t)(size_t)((lds_void_ptr)s_chunk) + wave * 1024;
    auto fetch = [&](int c) {
        const uint32_t at = lds0 + (c % FETCHED_CHUNKS) * CHUNK_BYTES;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const uint16_t* from = src[i < 2 ? i : 2] + (i < 2 ? 0 : (i - 2) * plane) + (size_t)c * K_CHUNK;
            lds::dma16_ptr(from, at + i * 4096);
        }
    };
    floatx16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < FETCHED_CHUNKS && c < n; ++c) fetch(c);
    const bool multiplies = wave < 2 && t0 + 32 * wave < tokens;
    for (int c = 0; c < n; ++c) {
        // chunk c has arrived (those behind it may be in flight)
        static_assert(FETCHED_CHUNKS <= 4, "at most three chunks behind");
        const int behind = min(FETCHED_CHUNKS - 1, n - 1 - c);
        if (behind == 3) __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (15 << 8));
        else if (behind == 2) __builtin_amdgcn_s_waitcnt(10 | (7 << 4) | (15 << 8));
        else if (behind == 1) __builtin_amdgcn_s_waitcnt(5 | (7 << 4) | (15 << 8));
        else __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (multiplies) {
            const lds_bytes st = (lds_bytes)s_chunk + (c % FETCHED_CHUNKS) * CHUNK_BYTES;
            auto operand = [&](int r, int s) {
                return *(const __attribute__((address_space(3))) bf16x8*)(st + (r * 8 + ((4 * half + s) ^ ((row >> 1) & 7))) * 16);
            };
            bf16x8 op[4][4];  // x, planes
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int s = 0; s < 4; ++s) op[m][s] = operand(m == 0 ? 32 * wave + row : 64 + 32 * (m - 1) + row, s);
            // smallest terms first
#pragma unroll
            for (int p = 3; p >= 1; --p)
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[0][s], op[p][s], acc, 0, 0, 0);
        }
        if (c + FETCHED_CHUNKS < n) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();  // chunk c has been read everywhere
            asm volatile("" ::: "memory");
            fetch(c + FETCHED_CHUNKS);
        }
    }
    if (!multiplies) return;
    float* dst = out + (size_t)blockIdx.z * tokens * n_experts;
    if (e0 + row < n_experts) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int tt = t0 + 32 * wave + 8 * (i / 4) + 4 * half + (i % 4);
            if (tt < tokens) dst[(size_t)tt * n_experts + e0 + row] = acc[i];
        }
    }
}

// The same product for many tokens: a workgroup of 4 wavefronts owns 128 tokens x 64 experts and shares its operand
// tiles through LDS (per 64 values of k: 128 rows of x and 3 x 64 rows of planes, 128 bytes each = 40 KB). With a
// tile of 32 x 32 per wavefront a CU's L1 is asked for 170 bytes per clock at the bf16 MFMA rate; here for 52.
//
// One wavefront per SIMD is all there is at 8192 tokens x 256 experts, so everything that takes time is requested
// early: global -> LDS loads into a ring of three stages, two of them in flight, and the operands of chunk c+1 are read
// into registers while the 24 MFMAs (768 cycles) of chunk c run. With one stage in flight through registers and the
// operand reads in front of the MFMAs a chunk took 2600 cycles (137 us for the 8192 x 256 logits
// of hidden 7168); this takes 83 us, 1.1 PFLOP/s of bf16 products (with the norm's output of that
// moment still to be written back, as in a layer, 87 to 98). With K split it also serves fewer tokens: 4096 tokens
// 85 us on the kernel above, 49 here; 1000: 24.7 and 21.5; 200: 14.6 and 12.5, the reduction included.
constexpr int BIG_TOKENS = 128;
constexpr int BIG_EXPERTS = 64;
constexpr int BIG_STAGE = (BIG_TOKENS + 3 * BIG_EXPERTS) * K_CHUNK * 2;  // bytes (40 KB)
constexpr int BIG_STAGES = 3;
constexpr int BIG_LOADS = BIG_STAGE / 1024 / 4;  // load instructions of a wavefront per stage

using lds::dma16;  // (completion is awaited once per chunk)

template <int N>
struct IntConstant {
    static constexpr int value = N;
};

// grid: x = 128-token tiles, y = 64-expert tiles, z = K split; out as in moe_router_gemm_kernel
__global__ __launch_bounds__(256, 1) void moe_router_gemm_split_tiled_kernel(const uint16_t* __restrict__ x,
                                                                             const uint16_t* __restrict__ planes,
                                                                             float* __restrict__ out, int tokens,
                                                                             int hidden, int n_experts,
                                                                             int chunks_per_split) {
    __shared__ __attribute__((aligned(16))) uint8_t s_stage[BIG_STAGES * BIG_STAGE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 31;
    const int half = lane >> 5;
    const int t0 = blockIdx.x * BIG_TOKENS;
    const int e0 = blockIdx.y * BIG_EXPERTS;
    const int chunk_begin = blockIdx.z * chunks_per_split;
    const int n = min(chunks_per_split, hidden / K_CHUNK - chunk_begin);  // (not positive: this split is empty)

    // fill side: instruction wave + 4*i (i < 10) covers 8 rows of the stage, lane -> row lane/8, chunk
    // (lane%8) ^ ((row >> 1) & 7): i < 4 rows of x, then two instructions per plane. Rows past the end repeat the last.
    const int ld_row = lane >> 3;
    const uint32_t ld_chunk = 16u * ((lane & 7) ^ (ld_row >> 1) ^ (4 * (wave & 1)));
    const uint16_t* base[4];  // x tile, planes
    base[0] = x + (size_t)t0 * hidden + (size_t)chunk_begin * K_CHUNK;
#pragma unroll
    for (int p = 0; p < 3; ++p)
        base[1 + p] = planes + ((size_t)p * n_experts + e0) * hidden + (size_t)chunk_begin * K_CHUNK;
    uint32_t off[6];  // bytes from the tile's first row: the four instructions of x, the two of any plane
#pragma unroll
    for (int i = 0; i < 4; ++i)
        off[i] = (uint32_t)min((wave + 4 * i) * 8 + ld_row, tokens - 1 - t0) * (uint32_t)hidden * 2u + ld_chunk;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        off[4 + i] = (uint32_t)min((wave + 4 * i) * 8 + ld_row, n_experts - 1 - e0) * (uint32_t)hidden * 2u + ld_chunk;
    const uint32_t stage_base = (uint32_t)(size_t)((lds_void_ptr)s_stage);
    auto issue = [&](int c, int i) {
        const int m = i < 4 ? 0 : 1 + (i - 4) / 2;
        dma16(base[m] + (size_t)c * K_CHUNK, off[i < 4 ? i : 4 + (i & 1)],
              stage_base + (c % BIG_STAGES) * BIG_STAGE + (wave + 4 * i) * 1024);
    };

    // read side: wavefront (wave & 1) takes tokens [64*(wave&1), +64), (wave >> 1) experts [32*(wave>>1), +32);
    // lane (row, half) holds values [32*half, +32) of its row, 8 per MFMA step
    const int a_row = 64 * (wave & 1) + row;
    const int b_row = BIG_TOKENS + 32 * (wave >> 1) + row;
    const int swizzle = (row >> 1) & 7;
    bf16x8 op[2][5][4];  // [chunk parity][two tiles of x, three planes][step]
    auto read_operands = [&](int c, bf16x8 (&dst)[5][4]) {
        const lds_bytes st = (lds_bytes)s_stage + (c % BIG_STAGES) * BIG_STAGE;
#pragma unroll
        for (int m = 0; m < 5; ++m)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int r = m < 2 ? a_row + 32 * m : b_row + BIG_EXPERTS * (m - 2);
                dst[m][s] = *(const __attribute__((address_space(3))) bf16x8*)(st + (r * 8 + ((4 * half + s) ^ swizzle)) * 16);
            }
    };
    floatx16 acc[2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
        acc[a] = floatx16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // MORE: chunk c+3 exists, and with it c+1 and c+2
    auto chunk = [&](int c, auto parity_tag, auto more_tag) {
        constexpr int P = decltype(parity_tag)::value;
        constexpr bool MORE = decltype(more_tag)::value != 0;
        // stage c+1 has arrived (that of c+2 may be in flight), and this wavefront holds its operands of chunk c
        if (MORE || c + 2 < n) __builtin_amdgcn_s_waitcnt(BIG_LOADS | (7 << 4) | (0 << 8));
        else __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (0 << 8));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();  // ... in every wavefront: stage c may be filled again
        asm volatile("" ::: "memory");
        if (MORE || c + 1 < n) read_operands(c + 1, op[P ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 2; p >= 0; --p) {  // smallest terms first
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[P][0][s], op[P][2 + p][s], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[P][1][s], op[P][2 + p][s], acc[1], 0, 0, 0);
                if constexpr (MORE) {
                    // (a load holds the wavefront until the memory pipeline has taken it: one per two MFMAs)
                    if ((2 - p) * 4 + s < BIG_LOADS) issue(c + 3, (2 - p) * 4 + s);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    if (n > 0) {
#pragma unroll
        for (int c = 0; c < BIG_STAGES; ++c)
            if (c < n)
#pragma unroll
                for (int i = 0; i < BIG_LOADS; ++i) issue(c, i);
        if (n > 2) __builtin_amdgcn_s_waitcnt(((2 * BIG_LOADS) & 15) | ((2 * BIG_LOADS) >> 4 << 14) | (7 << 4) | (15 << 8));
        else __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read_operands(0, op[0]);
        int c = 0;
        for (; c + 4 < n; c += 2) {
            chunk(c, IntConstant<0>{}, IntConstant<1>{});
            chunk(c + 1, IntConstant<1>{}, IntConstant<1>{});
        }
        // at most four chunks are left; the first may have one more to request
        for (; c < n; c += 2) {
            if (c + 3 < n) chunk(c, IntConstant<0>{}, IntConstant<1>{});
            else chunk(c, IntConstant<0>{}, IntConstant<0>{});
            if (c + 1 < n) chunk(c + 1, IntConstant<1>{}, IntConstant<0>{});
        }
    }
    float* dst = out + (size_t)blockIdx.z * tokens * n_experts;
    const int e = e0 + 32 * (wave >> 1) + row;
    if (e < n_experts) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int tt = t0 + 64 * (wave & 1) + 32 * a + 8 * (i / 4) + 4 * half + (i % 4);
                if (tt < tokens) dst[(size_t)tt * n_experts + e] = acc[a][i];
            }
    }
}

// Long sums on the bf16 matrix cores, for many tokens: a workgroup of 8 wavefronts owns 128 tokens x 64 experts. What
// bounds the kernel above is the LDS port (128 bytes a clock): a chunk of 64 values of k is 768 cycles of MFMA per SIMD, 320
// cycles of LDS writes by the DMA and, with the tile cut into four pieces of 64 x 32, one per wavefront, 640 of operand
// reads. So here the wavefronts share K instead: each holds the whole 128 x 64 tile (128 accumulator registers) and takes
// every eighth step of 16 values, which reads every operand once per workgroup (320 cycles). Wavefronts 0-3 take the even
// chunks, 4-7 the odd ones, half a period apart, so that a SIMD has one wavefront in the middle of its 24 MFMAs while the
// other one waits for a barrier or for its operands. Chunks come by global -> LDS loads into a ring of four stages, three of
// them in flight. The eight partial tiles are added through LDS at the end, in a fixed order (about 1.5 us, which few
// chunks do not make up for).
//
// 8192 x 256 logits of hidden 7168: 80 us = 1.1 PFLOP/s of bf16 products (379 on the fp32 matrix cores). Against float64
// the relative error is 3.2e-7 (1.5e-6 on the fp32 matrix cores).
//
// W, 64 rows of 256 bytes a chunk, is cut into the three bf16 numbers in registers, 112 VALU instructions under the 24 MFMAs.
// Over the planes themselves the same kernel took 75.5 us where the one above takes 81.6, and is not used there: its sums
// differ from that one's by 1e-6, which for one in four batches of 8192 tokens puts some token across the boundary
// between two groups of experts.
struct LongTile {
    static constexpr int X_BYTES = BIG_TOKENS * K_CHUNK * 2;  // 16 KB
    static constexpr int STAGE = X_BYTES + BIG_EXPERTS * K_CHUNK * 4;
    static constexpr int STAGES = 4;
    static constexpr int LOADS = STAGE / 1024 / 4;  // load instructions of a wavefront per stage (half of them fill one)
};

// The last bit of a bf16 number is 2^-133 at the least (the matrix core takes subnormal ones as they are), and that of a
// weight from 2^-110 on, so that its three parts are the weight. Magnitudes as doubled bit patterns less one, which puts zero
// above all others.
constexpr uint32_t SPLIT_SMALLEST = ((127u - 110u) << 24) - 1u;

// 8 consecutive values of fp32 weights as three operands (see moe_router_split_kernel); the smallest magnitude among
// them goes into `smallest`
__device__ __forceinline__ void split_weights(bf16x8 (&planes)[3], const floatx4 (&w)[2], uint32_t& smallest) {
    uint32_t out[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v[2] = {w[i / 2][2 * (i & 1)], w[i / 2][2 * (i & 1) + 1]};
        smallest = min(smallest, min((__float_as_uint(v[0]) << 1) - 1u, (__float_as_uint(v[1]) << 1) - 1u));
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            // (the upper halves of both side by side)
            out[p][i] = __builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u);
#pragma unroll
            for (int j = 0; j < 2; ++j) v[j] -= __uint_as_float(__float_as_uint(v[j]) & 0xffff0000u);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) planes[p] = __builtin_bit_cast(bf16x8, u32x4{out[p][0], out[p][1], out[p][2], out[p][3]});
}

// grid: x = 128-token tiles, y = 64-expert tiles, z = K split; out as in moe_router_gemm_kernel
__global__ __launch_bounds__(512, 2) void moe_router_gemm_long_kernel(const uint16_t* __restrict__ x,
                                                                      const float* __restrict__ w, float* __restrict__ out,
                                                                      int tokens, int hidden, int n_experts,
                                                                      int chunks_per_split) {
    typedef LongTile T;
    __shared__ __attribute__((aligned(16))) uint8_t s_stage[4 * 32 * 1024 > T::STAGES * T::STAGE ? 4 * 32 * 1024 : T::STAGES * T::STAGE];
    __shared__ int s_small[BIG_EXPERTS];  // whether an expert has a weight that is not the sum of its parts
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 31;
    const int half = lane >> 5;
    const int piece = wave & 3;
    const int parity = wave >> 2;
    const int t0 = blockIdx.x * BIG_TOKENS;
    const int e0 = blockIdx.y * BIG_EXPERTS;
    const int chunk_begin = blockIdx.z * chunks_per_split;
    const int n = min(chunks_per_split, hidden / K_CHUNK - chunk_begin);  // (not positive: this split is empty)

    // fill side: the wavefronts of one parity fill a stage, a kilobyte per instruction, rows past the end repeating the
    // last. Instruction piece + 4*i: i < 4 8 rows of x, lane -> row lane/8, chunk (lane%8) ^ ((row >> 1) & 7); then
    // four of 4 rows of the weight, lane -> row lane/16, chunk (lane%16) ^ (row & 15).
    const int ld_row = lane >> 3;
    const uint32_t ld_chunk = 16u * ((lane & 7) ^ (ld_row >> 1) ^ (4 * (piece & 1)));
    const uint16_t* x_base = x + (size_t)t0 * hidden + (size_t)chunk_begin * K_CHUNK;
    const float* w_base = w + (size_t)e0 * hidden + (size_t)chunk_begin * K_CHUNK;
    uint32_t x_off[4], w_off[4];  // bytes from the tile's first row
#pragma unroll
    for (int i = 0; i < 4; ++i)
        x_off[i] = (uint32_t)min((piece + 4 * i) * 8 + ld_row, tokens - 1 - t0) * (uint32_t)hidden * 2u + ld_chunk;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        w_off[i] = (uint32_t)min((piece + 4 * i) * 4 + (lane >> 4), n_experts - 1 - e0) * (uint32_t)hidden * 4u +
                   16u * ((lane & 15) ^ (4 * piece + (lane >> 4)));
    const uint32_t stage_base = (uint32_t)(size_t)((lds_void_ptr)s_stage);
    auto issue = [&](int c) {
        const uint32_t st = stage_base + (c % T::STAGES) * T::STAGE + piece * 1024;
#pragma unroll
        for (int i = 0; i < 4; ++i) dma16(x_base + (size_t)c * K_CHUNK, x_off[i], st + i * 4096);
#pragma unroll
        for (int i = 0; i < T::LOADS - 4; ++i)
            dma16(w_base + (size_t)c * K_CHUNK, w_off[i], st + T::X_BYTES + i * 4096);
    };

    // read side: values [16*piece, +16) of the chunks of this parity; lane (row, half) the 8 values of `half` of its row
    // in every block of 32 rows: four of x, then two of the weight
    const uint32_t read_off = (uint32_t)(row * 8 + ((2 * piece + half) ^ ((row >> 1) & 7))) * 16u;
    const uint32_t w_read[2] = {(uint32_t)(row * 16 + ((4 * piece + 2 * half) ^ (row & 15))) * 16u,
                                (uint32_t)(row * 16 + ((4 * piece + 2 * half + 1) ^ (row & 15))) * 16u};
    typedef const __attribute__((address_space(3))) bf16x8* lds_bf16x8;
    typedef const __attribute__((address_space(3))) floatx4* lds_floatx4;
    bf16x8 a[4], b[2][3];
    floatx4 raw[2][2];
    uint32_t smallest[2] = {0xffffffffu, 0xffffffffu};  // of this lane's experts
    if (threadIdx.x < BIG_EXPERTS) s_small[threadIdx.x] = 0;
    floatx16 acc[4][2];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int g = 0; g < 2; ++g)
            acc[m][g] = floatx16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // the 12 products of 32 experts, smallest terms first
    auto products = [&](int g) {
        split_weights(b[g], raw[g], smallest[g]);
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[m][g] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m], b[g][p], acc[m][g], 0, 0, 0);
    };
    auto barrier = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // Barrier c: chunk c has arrived and the operands of chunk c-1 are in registers, so stage c-1 may be filled again.
    // The wavefronts of the other parity than c requested chunk c (and c+2 after it) and read chunk c-1.
    auto other_barrier = [&](int c) {
        if (c + 2 < n) __builtin_amdgcn_s_waitcnt(T::LOADS | (7 << 4) | (0 << 8));
        else __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (0 << 8));
        barrier();
    };
    if (n > 0) {
        if (parity == 1) {
            issue(0);
            if (n > 2) issue(2);
            other_barrier(0);
        } else {
            if (n > 1) issue(1);
        }
        for (int c = parity; c < n; c += 2) {
            barrier();
            const lds_bytes st = (lds_bytes)s_stage + (c % T::STAGES) * T::STAGE;
#pragma unroll
            for (int m = 0; m < 4; ++m) a[m] = *(lds_bf16x8)(st + read_off + m * 4096);
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int j = 0; j < 2; ++j) raw[g][j] = *(lds_floatx4)(st + T::X_BYTES + g * 8192 + w_read[j]);
            __builtin_amdgcn_sched_barrier(0);
            if (c + 3 < n) issue(c + 3);
            products(0);
            if (c + 1 < n) other_barrier(c + 1);
            products(1);
        }
    }
    // Sum of the eight tiles: 4-7 leave theirs for 0-3 (32 KB each, 4 registers of a lane side by side), and all eight add
    // the four sums, an eighth each: register quad q of a lane holds tokens 32*(q/8) + 8*(q%4) + 4*half + [0, 4) of
    // expert 32*(q/4%2) + row.
    floatx4* tile = reinterpret_cast<floatx4*>(s_stage) + piece * 2048 + lane;
    auto quad = [&](int q) {
        const floatx16& v = acc[q / 8][q / 4 % 2];
        return floatx4{v[4 * (q & 3)], v[4 * (q & 3) + 1], v[4 * (q & 3) + 2], v[4 * (q & 3) + 3]};
    };
    const bool small = __syncthreads_or(min(smallest[0], smallest[1]) < SPLIT_SMALLEST);
    if (small) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
            if (smallest[g] < SPLIT_SMALLEST) s_small[32 * g + row] = 1;
    }
    if (parity == 1) {
#pragma unroll
        for (int q = 0; q < 32; ++q) tile[q * 64] = quad(q);
    }
    __syncthreads();
    if (parity == 0) {
#pragma unroll
        for (int q = 0; q < 32; ++q) {
            tile[q * 64] = tile[q * 64] + quad(q);
            if (q % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
    float* dst = out + (size_t)blockIdx.z * tokens * n_experts;
    const floatx4* sums = reinterpret_cast<const floatx4*>(s_stage) + lane;
    // (quads 4*wave + [0, 4): 32 tokens x 32 experts)
    const int tile_t0 = t0 + 32 * (wave / 2), tile_e0 = e0 + 32 * (wave % 2);
    const int e = tile_e0 + row;
    float v[16];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int q = 4 * wave + k;
        const floatx4 sum = (sums[q * 64] + sums[2048 + q * 64]) + (sums[4096 + q * 64] + sums[6144 + q * 64]);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[4 * k + i] = sum[i];
    }
    auto token_of = [&](int i) { return tile_t0 + 8 * (i / 4) + 4 * half + i % 4; };
    // What the three products don't give is taken from the fp32 matrix cores, as a tile of moe_router_gemm_kernel: the sums of
    // an expert with too small a weight, and sums that are no number. (An infinite weight leaves infinity - infinity
    // behind, and an infinite x times a part that is zero is no number either.)
    // us, 8192 tokens of 7168 x 256, 85 as a rule: with one weight of 2^-120 420, with an infinity in one token 261, with a
    // NaN in one token 86, in all of them 240 (the fp32 matrix cores for all sums: 400).
    uint32_t again = 0;  // bit i: v[i]
#pragma unroll
    for (int i = 0; i < 16; ++i)
        if (e < n_experts && token_of(i) < tokens && v[i] != v[i]) again |= 1u << i;
    if (__ballot(again != 0) != 0) {
        // ... but a token whose own values hold a NaN, as those of padding may, keeps it
        const uint16_t* x_part = x + (size_t)chunk_begin * K_CHUNK + lane * 8;
        for (int i = 0; i < 16; ++i) {
            const uint64_t lanes = __ballot(again >> i & 1);
            for (int h = 0; h < 2; ++h) {
                if ((uint32_t)(lanes >> (32 * h)) == 0) continue;
                const uint16_t* at = x_part + (size_t)(tile_t0 + 8 * (i / 4) + 4 * h + i % 4) * hidden;
                bool nan = false;
                for (int c = lane * 8; c < n * K_CHUNK; c += 512, at += 512) {
                    const u32x4 pairs = *reinterpret_cast<const u32x4*>(at);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        nan |= (pairs[j] & 0x7fffu) > 0x7f80u || (pairs[j] & 0x7fff0000u) > 0x7f800000u;
                }
                if (__ballot(nan) != 0 && half == h) again &= ~(1u << i);
            }
        }
    }
    if (small && s_small[e - e0]) again = 0xffff;
    if (__ballot(again != 0) != 0) {
        const floatx16 exact = fp32_tile(x + (size_t)min(tile_t0 + row, tokens - 1) * hidden + 32 * half,
                                         w + (size_t)min(e, n_experts - 1) * hidden + 32 * half, chunk_begin, chunk_begin + n);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = again >> i & 1 ? exact[i] : v[i];
    }
    if (e < n_experts) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (token_of(i) < tokens) dst[(size_t)token_of(i) * n_experts + e] = v[i];
    }
}

// Few tokens and the split weight, in one launch: a workgroup owns 16 tokens x 5 experts over all of K, its 8 wavefronts take
// the chunks of K in turn, and the 16 columns of an MFMA (16 x 16 x 32) are the three planes of the five experts. What bounds
// so small a product is the start and end of its launches and the latency of its loads, so there is no second kernel to add
// partial sums, and a wavefront requests 7 chunks at once (224 KB of loads in flight on a CU). Rows are loaded by consecutive
// lanes and turned into operands through LDS: with the operand's own 16 rows side by side in a load a CU took one lane a
// clock, 16 bytes (16 tokens of 7168 x 256, the same weight every time: 13.8 us instead of 6.9).
// Sums: per wavefront, column and token, then over the wavefronts in ascending order, then lo + mid + hi; relative error
// against float64 1.8e-7 (7168 x 256), as with splits of K.
//
// us, with K split over workgroups and so, six weights in turn: 16 tokens of 7168 x 256 9.1, 8.4; 48 10.0, 9.3; 64 of 2048 x 128
// 6.1, 4.4; 64 of 4096 x 256 8.6, 7.3; 192 of 7168 x 64 9.6, 8.9. The same weight every time: 7.9, 7.2; 8.8, 8.8; 5.8, 3.8; 7.8,
// 6.3; 8.7, 7.3.
constexpr int FEW_TOKENS = 16;
constexpr int FEW_EXPERTS = 5;
constexpr int FEW_WAVES = 8;

__global__ __launch_bounds__(64 * FEW_WAVES) void moe_router_gemm_few_kernel(const uint16_t* __restrict__ x,
                                                                             const uint16_t* __restrict__ planes,
                                                                             float* __restrict__ logits, int tokens,
                                                                             int hidden, int n_experts) {
    constexpr int AHEAD = 7;  // chunks of a wavefront whose loads are in flight
    __shared__ __attribute__((aligned(16))) float s_part[FEW_WAVES][16 * FEW_TOKENS];  // [wavefront][column][token]
    __shared__ float s_sum[16 * FEW_TOKENS];
    // (private to a wavefront, whose LDS operations execute in order)
    __shared__ u32x4 s_turn[FEW_WAVES][4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15;  // of the operands: token, and column
    const int quarter = lane >> 4;
    const int t0 = blockIdx.x * FEW_TOKENS;
    const int e0 = blockIdx.y * FEW_EXPERTS;
    const int n_chunks = hidden / K_CHUNK;
    // fill side: a load instruction takes 64 bytes of 16 rows, lane -> row lane/4, 16-byte piece lane%4 (tokens, experts and
    // the column beyond the end repeat the last one; their results are not stored)
    const int ld_row = lane >> 2;
    const int t = min(t0 + ld_row, tokens - 1);
    const int used = min(ld_row, 3 * FEW_EXPERTS - 1);
    const int e = min(e0 + used / 3, n_experts - 1);
    const u32x4* xp = reinterpret_cast<const u32x4*>(x + (size_t)t * hidden) + (lane & 3);
    const u32x4* wp = reinterpret_cast<const u32x4*>(planes + ((size_t)(used % 3) * n_experts + e) * hidden) + (lane & 3);
    // piece p of row r waits in slot 4*r + (p ^ (r / 4)), which keeps the reads of 16 rows off each other's banks
    const int slot_in = 4 * ld_row + ((lane & 3) ^ (ld_row >> 2));
    const int slot_out = 4 * col + (quarter ^ (col >> 2));
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = wave; c0 < n_chunks; c0 += FEW_WAVES * AHEAD) {
        u32x4 raw[AHEAD][4];  // x, planes: first and second half of the chunk
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            const int c = c0 + FEW_WAVES * j;
            if (c < n_chunks) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    raw[j][2 + s] = wp[c * (K_CHUNK * 2 / 16) + 4 * s];
                    raw[j][s] = xp[c * (K_CHUNK * 2 / 16) + 4 * s];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            if (c0 + FEW_WAVES * j < n_chunks) {
                bf16x8 op[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) s_turn[wave][i][slot_in] = raw[j][i];
#pragma unroll
                for (int i = 0; i < 4; ++i) op[i] = __builtin_bit_cast(bf16x8, s_turn[wave][i][slot_out]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[0], op[2], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[1], op[3], acc, 0, 0, 0);
            }
        }
    }
    // result register i of a lane: token 4*quarter + i, column `col`
    *reinterpret_cast<floatx4*>(&s_part[wave][col * FEW_TOKENS + 4 * quarter]) = acc;
    __syncthreads();
    if (threadIdx.x < 16 * FEW_TOKENS) {
        float sum = s_part[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < FEW_WAVES; ++w) sum += s_part[w][threadIdx.x];
        s_sum[threadIdx.x] = sum;
    }
    __syncthreads();
    const int token = t0 + (int)(threadIdx.x % FEW_TOKENS);
    const int k = threadIdx.x / FEW_TOKENS;
    if (k < FEW_EXPERTS && e0 + k < n_experts && token < tokens) {
        const float* sums = s_sum + 3 * k * FEW_TOKENS + threadIdx.x % FEW_TOKENS;
        logits[(size_t)token * n_experts + e0 + k] = (sums[2 * FEW_TOKENS] + sums[FEW_TOKENS]) + sums[0];
    }
}

// logits = partial[0] + partial[1] + ... in that order. A chain of memory latencies: BATCH partial sums are requested at once.
template <int BATCH>
__global__ __launch_bounds__(256) void moe_router_reduce_kernel(const float* __restrict__ partial,
                                                                float* __restrict__ logits,
                                                                size_t count, int n_splits) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    float sum = 0.f;
    for (int s0 = 0; s0 < n_splits; s0 += BATCH) {
        float v[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; ++j) v[j] = partial[(size_t)(s0 + j < n_splits ? s0 + j : 0) * count + i];
#pragma unroll
        for (int j = 0; j < BATCH; ++j)
            if (s0 + j < n_splits) sum = (s0 + j == 0) ? v[j] : sum + v[j];
    }
    logits[i] = sum;
}

void launch_reduce(const void* partial, float* logits, size_t count, int n_splits, hipStream_t stream) {
    const auto kernel = n_splits <= 2    ? moe_router_reduce_kernel<2>
                        : n_splits <= 8  ? moe_router_reduce_kernel<8>
                        : n_splits <= 16 ? moe_router_reduce_kernel<16>
                                         : moe_router_reduce_kernel<32>;
    // Few logits are latency: one wavefront a workgroup spreads them over the CUs (500 tokens of 256 experts, the whole router
    // 27.6 us, with 256 threads 27.7). Many are dealt out faster in fewer workgroups (5000 tokens 124.2 -> 122.2, 3001 82.1 ->
    // 81.9; 1023 alike, where the line is).
    const unsigned threads = count <= 1024 * 256 ? 64 : 256;
    kernel<<<(unsigned)((count + threads - 1) / threads), threads, 0, stream>>>(static_cast<const float*>(partial), logits,
                                                                                count, n_splits);
}

int pick_router_splits(int tokens, int hidden, int n_experts) {
    const long tiles = (long)((tokens + 63) / 64) * ((n_experts + 63) / 64);
    const int n_chunks = hidden / K_CHUNK;
    int splits = 1;
    // Aims at two tiles of 64 x 64 per CU (the split weight's kernel for few workgroups has tiles of 64 x 32, twice as many). Splits
    // of ceil(n_chunks / splits) chunks, two at least; where the division leaves a remainder the last ones have fewer or none: 112
    // chunks in 32 splits are 28 of four and 4 that store zeros, which the reduction adds like any others.
    while (tiles * splits < 512 && splits * 2 * 2 <= n_chunks) splits *= 2;
    return splits;
}

}  // namespace

// K splits the launcher uses for these sizes (1 = no scratch needed)
extern "C" int moe_router_logits_num_splits(int tokens, int hidden, int n_experts) {
    if (tokens <= 0 || hidden <= 0 || n_experts <= 0 || hidden % K_CHUNK != 0) return 0;
    return pick_router_splits(tokens, hidden, n_experts);
}

// bytes of scratch moe_router_logits_launcher needs (0 when K is not split)
extern "C" size_t moe_router_logits_workspace_bytes(int tokens, int hidden, int n_experts) {
    const int splits = moe_router_logits_num_splits(tokens, hidden, n_experts);
    return splits <= 1 ? 0 : (size_t)splits * tokens * n_experts * sizeof(float);
}

// logits [tokens, n_experts] fp32 = x [tokens, hidden] (x_dtype 0 = fp32, 1 = bf16) times
// w [n_experts, hidden] fp32, transposed. hidden a multiple of 64; x and w 16-byte aligned.
// workspace: moe_router_logits_workspace_bytes(...) bytes of device scratch (may be null if 0).
extern "C" void moe_router_logits_launcher(float* logits, const void* x, const float* w,
                                           void* workspace, size_t workspace_bytes, int tokens,
                                           int hidden, int n_experts, int x_dtype, int config,
                                           hipStream_t stream) {
    if (tokens <= 0 || n_experts <= 0) return;
    if (hidden <= 0 || hidden % K_CHUNK != 0 || (x_dtype != 0 && x_dtype != 1) ||
        (tokens + 63) / 64 > 0x7fffffff / 64 || (n_experts + 63) / 64 > 65535) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
                           reinterpret_cast<uintptr_t>(workspace);
    if (!logits || !x || !w || (bits & 15u) != 0) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    const int splits = pick_router_splits(tokens, hidden, n_experts);
    const size_t need = splits <= 1 ? 0 : (size_t)splits * tokens * n_experts * sizeof(float);
    if (need > 0 && (!workspace || workspace_bytes < need)) {
        caa::set_status(CAA_WORKSPACE_TOO_SMALL);
        return;
    }
    const int n_chunks = hidden / K_CHUNK;
    const int chunks_per_split = (n_chunks + splits - 1) / splits;
    float* out = splits > 1 ? static_cast<float*>(workspace) : logits;
    const dim3 grid((tokens + 63) / 64, (n_experts + 63) / 64, splits);
    // A bf16 x: the weight cut into bf16 parts on the way to the matrix core, wherever a tile has enough to do (config 3 forces
    // it, 1 the fp32 matrix core; us, fp32 and bf16 matrix core: 64 tokens of 7168 x 256 14.1, 12.2; 512: 34.3, 16.6; 8192: 379,
    // 80; with two chunks of K a split only where the tiles fill the chip: 1000 of 2048 x 128 18.8, 13.6, but 512 of it, 64
    // workgroups, 11.2, 11.4; 17 of 7168 x 384 11.9, 12.2).
    const dim3 tiles((tokens + BIG_TOKENS - 1) / BIG_TOKENS, (n_experts + BIG_EXPERTS - 1) / BIG_EXPERTS, splits);
    const bool enough = tokens >= 64 && (chunks_per_split >= 3 || (long)tiles.x * tiles.y * splits >= 144);
    if (x_dtype == 1 && hidden <= (1 << 23) && (config == 3 || (config != 1 && enough))) {
        moe_router_gemm_long_kernel<<<tiles, 512, 0, stream>>>(static_cast<const uint16_t*>(x), w, out, tokens, hidden,
                                                                      n_experts, chunks_per_split);
    } else if (x_dtype == 0) {
        moe_router_gemm_kernel<float><<<grid, 256, 0, stream>>>(
            static_cast<const float*>(x), w, out, tokens, hidden, n_experts, chunks_per_split);
    } else {
        moe_router_gemm_kernel<uint16_t><<<grid, 256, 0, stream>>>(
            static_cast<const uint16_t*>(x), w, out, tokens, hidden, n_experts, chunks_per_split);
    }
    if (splits > 1) {
        launch_reduce(workspace, logits, (size_t)tokens * n_experts, splits, stream);
    }
}

// planes [3, n_experts, hidden] bf16 (written) from w [n_experts, hidden] fp32: the three bf16 numbers whose
// sum is the weight, for moe_router_logits_split_launcher. Done once per weight.
extern "C" void moe_router_split_weight_launcher(void* planes, const float* w, int n_experts, int hidden,
                                                 hipStream_t stream) {
    if (n_experts <= 0 || hidden <= 0) return;
    if (!planes || !w) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    const size_t n = (size_t)n_experts * hidden;
    moe_router_split_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(w, static_cast<uint16_t*>(planes), n);
}

// moe_router_logits_launcher for a bf16 x and a weight given as the planes above: the same logits up to the
// order of the fp32 additions, on the bf16 matrix cores. Sizes, scratch (moe_router_logits_workspace_bytes)
// and limits as there; x and planes 16-byte aligned, hidden a multiple of 64.
extern "C" void moe_router_logits_split_launcher(float* logits, const void* x, const void* planes,
                                                 void* workspace, size_t workspace_bytes, int tokens,
                                                 int hidden, int n_experts, int config, hipStream_t stream) {
    if (tokens <= 0 || n_experts <= 0) return;
    if (hidden <= 0 || hidden % K_CHUNK != 0 || (tokens + 63) / 64 > 0x7fffffff / 64 ||
        (n_experts + 63) / 64 > 65535) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(planes) |
                           reinterpret_cast<uintptr_t>(workspace);
    if (!logits || !x || !planes || (bits & 15u) != 0) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    const int splits = pick_router_splits(tokens, hidden, n_experts);
    const size_t need = splits <= 1 ? 0 : (size_t)splits * tokens * n_experts * sizeof(float);
    if (need > 0 && (!workspace || workspace_bytes < need)) {
        caa::set_status(CAA_WORKSPACE_TOO_SMALL);
        return;
    }
    // One launch where a round of workgroups does and what they fetch, each its 31 rows, is little enough for the
    // memory-side cache (norm, projection and routing in a row over changing inputs, us, K split and one launch: 48 tokens of
    // 7168 x 256, 69 MB, 18.2, 17.4; 56 of it, 92 MB, 18.5, 20.0; 96 of 7168 x 128, 69 MB, 17.8, 17.1; 112 of it, 81 MB, 18.0, 19.9;
    // 192 of 7168 x 64, 69 MB, 17.1, 16.3; 208 of it, 75 MB, 17.6, 18.9, but 176, 64 MB, 17.0, 17.8; 64 of 4096 x 256, 208
    // workgroups, 15.9, 14.5; 80 of it, 260, 17.0, 19.8). Config 4 forces it.
    const dim3 few((tokens + FEW_TOKENS - 1) / FEW_TOKENS, (n_experts + FEW_EXPERTS - 1) / FEW_EXPERTS);
    const long few_wgs = (long)few.x * few.y;
    const long few_bytes = few_wgs * (FEW_TOKENS + 3 * FEW_EXPERTS) * hidden * 2;
    if (hidden <= (1 << 24) && few.y <= 65535 && (config == 4 || (config == 0 && few_wgs <= 256 && few_bytes <= 72000000))) {
        moe_router_gemm_few_kernel<<<few, 64 * FEW_WAVES, 0, stream>>>(
            static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(planes), logits, tokens, hidden, n_experts);
        return;
    }
    const int n_chunks = hidden / K_CHUNK;
    const int chunks_per_split = (n_chunks + splits - 1) / splits;
    // Enough 128 x 64 tiles and splits to fill the chip: the workgroup-tiled kernel (config 2 forces it, 1 the other one).
    // It has one workgroup on a CU, so that a part of a second round costs a whole one, which few chunks of K do not make up
    // for, all the less where each has little to share (us, tiled and not; 1500 tokens of 4096 x 64, 384 workgroups of 2
    // chunks: 16.7, 13.7; 1400 of 1024 x 256, 352 of 2: 15.3, 12.7; one tile of experts, 1200 of 7168 x 64, 320 of 4: 18.1,
    // 16.2; a third of the rows padding, 160 of 7168 x 384, 384 of 4: 17.7, 16.7; but 300 of 7168 x 256, 384 of 4: 18.4, 20.1).
    const long token_tiles = (tokens + BIG_TOKENS - 1) / BIG_TOKENS;
    const long big_wgs = token_tiles * ((n_experts + BIG_EXPERTS - 1) / BIG_EXPERTS) * splits;
    const bool part_of_second_round = big_wgs > 256 && big_wgs < 512;
    const bool few_chunks = chunks_per_split <= 2 ||
                            (chunks_per_split <= 4 && splits >= 16 && big_wgs < 448 &&
                             (n_experts <= BIG_EXPERTS || 3L * tokens < 2 * BIG_TOKENS * token_tiles));
    const bool wide = n_experts > 32 * 65535;  // (more than a grid has tiles of 32 experts for)
    const bool tiled = hidden <= (1 << 24) && (config == 2 || wide || (config != 1 && big_wgs >= 192 && tokens >= BIG_TOKENS &&
                                                              !(part_of_second_round && few_chunks)));
    float* out = splits > 1 ? static_cast<float*>(workspace) : logits;
    const int tile_tokens = tiled ? BIG_TOKENS : 64;
    const dim3 grid((tokens + tile_tokens - 1) / tile_tokens, tiled ? (n_experts + 63) / 64 : (n_experts + 31) / 32, splits);
    // Four chunks ahead are 80 KB of LDS, two workgroups to a CU; with more workgroups than that two chunks and four workgroups are
    // faster (us, the projection alone with four and two: 100 tokens of 7168 x 384, 768 workgroups, 13.8, 12.6; 1200 of 7168 x 64
    // 19.1, 16.2; 160 of 7168 x 384 18.1, 16.6), and two chunks in all need no more.
    const bool two_ahead = chunks_per_split <= 2 || (long)grid.x * grid.y * grid.z > 512;
    const auto kernel = tiled       ? moe_router_gemm_split_tiled_kernel
                        : two_ahead ? moe_router_gemm_split_kernel<2>
                                    : moe_router_gemm_split_kernel<4>;
    kernel<<<grid, 256, 0, stream>>>(static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(planes), out, tokens,
                                     hidden, n_experts, chunks_per_split);
    if (splits > 1) {
        launch_reduce(workspace, logits, (size_t)tokens * n_experts, splits, stream);
    }
}
