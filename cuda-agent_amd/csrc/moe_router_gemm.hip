// Router projection of a MoE layer: logits[t, e] = sum_h x[t, h] * w[e, h], fp32.
//
// x is the layer's bf16 (or fp32) input, w the fp32 router weight [n_experts, hidden]; both are
// taken to fp32 exactly and multiplied on the fp32 matrix cores (v_mfma_f32_32x32x2_f32), so the
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
// weight is the exact sum of three bf16 numbers (its 24 significand bits cut into 8 + 8 + 8), and a
// product of two bf16 numbers is exact in fp32. With the weight stored once as those three planes the
// projection of a bf16 x runs on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16: 8 times the rate of
// the fp32 shape, three products per weight) and still differs from an fp32 reference by the order of the
// additions only. At that rate the operand loads are what matters: rows are fetched as whole lines and
// turned into the operand layout through a small LDS buffer private to the wavefront.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch_status.hpp"

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
    const X* xp = x + (size_t)t * hidden + 32 * half;
    const float* wp = w + (size_t)e * hidden + 32 * half;

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

// grid as moe_router_gemm_kernel. A wavefront owns 32 tokens x 32 experts; per 64 values of k it fetches
// four tiles of 32 rows x 128 bytes (x and the three weight planes), each with 4 load instructions of whole
// lines (lane l: 16-byte chunk l % 8 of row 8*j + l / 8), and passes them one after the other through its
// 4 KB LDS buffer (chunk c of row r at slot c ^ ((r >> 1) & 7)) into the operand layout: lane (row, half)
// holds values [32*half, +32) of its row, 8 per MFMA step. No barrier: the buffer is private and the LDS
// operations of a wavefront execute in order.
__global__ __launch_bounds__(256) void moe_router_gemm_split_kernel(const uint16_t* __restrict__ x,
                                                                    const uint16_t* __restrict__ planes,
                                                                    float* __restrict__ out, int tokens,
                                                                    int hidden, int n_experts,
                                                                    int chunks_per_split) {
    __shared__ u32x4 s_tile[4][32 * 8];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row = lane & 31;
    const int half = lane >> 5;
    const int t0 = blockIdx.x * 64 + (wave & 1) * 32;
    const int e0 = blockIdx.y * 64 + (wave >> 1) * 32;
    if (t0 >= tokens || e0 >= n_experts) return;  // (no barrier in this kernel)
    u32x4* tile = s_tile[wave];
    const int chunk_begin = blockIdx.z * chunks_per_split;
    int chunk_end = chunk_begin + chunks_per_split;
    const int n_chunks = hidden / K_CHUNK;
    if (chunk_end > n_chunks) chunk_end = n_chunks;
    const size_t plane = (size_t)n_experts * hidden;

    // fill side: rows 8*j + lane/8 of the tile, chunk lane%8 (rows beyond the end repeat the last valid one)
    const u32x4* src[4][4];  // [x, hi, mid, lo][instruction]
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 8 * j + (lane >> 3);
        const int t = t0 + r < tokens ? t0 + r : tokens - 1;
        const int e = e0 + r < n_experts ? e0 + r : n_experts - 1;
        src[0][j] = reinterpret_cast<const u32x4*>(x + (size_t)t * hidden) + (lane & 7);
#pragma unroll
        for (int p = 0; p < 3; ++p)
            src[1 + p][j] = reinterpret_cast<const u32x4*>(planes + p * plane + (size_t)e * hidden) + (lane & 7);
    }
    u32x4 raw[4][4];
    auto load_chunk = [&](int c) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j) raw[m][j] = src[m][j][(size_t)c * (K_CHUNK * 2 / 16)];
    };
    // operand of matrix m: through the buffer
    bf16x8 op[4][4];
    auto stage = [&](int m) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 8 * j + (lane >> 3);
            tile[r * 8 + ((lane & 7) ^ ((r >> 1) & 7))] = raw[m][j];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
            op[m][s] = __builtin_bit_cast(bf16x8, tile[row * 8 + ((4 * half + s) ^ ((row >> 1) & 7))]);
    };

    floatx16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (chunk_begin < chunk_end) load_chunk(chunk_begin);
    for (int c = chunk_begin; c < chunk_end; ++c) {
#pragma unroll
        for (int m = 0; m < 4; ++m) stage(m);
        if (c + 1 < chunk_end) load_chunk(c + 1);  // in flight under the MFMAs below
        // smallest terms first
#pragma unroll
        for (int p = 3; p >= 1; --p)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[0][s], op[p][s], acc, 0, 0, 0);
    }
    float* dst = out + (size_t)blockIdx.z * tokens * n_experts;
    if (e0 + row < n_experts) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int tt = t0 + 8 * (i / 4) + 4 * half + (i % 4);
            if (tt < tokens) dst[(size_t)tt * n_experts + e0 + row] = acc[i];
        }
    }
}

// The same product for many tokens: a workgroup of 4 wavefronts owns 128 tokens x 64 experts and shares its operand
// tiles through LDS (per 64 values of k: 128 rows of x and 3 x 64 rows of planes, 128 bytes each = 40 KB). The per-wavefront
// kernel above asks its CU's L1 for 170 bytes per clock at the bf16 MFMA rate; this one for 52.
//
// One wavefront per SIMD is all there is at 8192 tokens x 256 experts, so everything that takes time is requested
// early: global -> LDS loads into a ring of three stages, two of them in flight, and the operands of chunk c+1 are read
// into registers while the 24 MFMAs (768 cycles) of chunk c run. With one stage in flight through registers and the
// operand reads in front of the MFMAs a chunk took 2600 cycles (137 us for the 8192 x 256 logits
// of hidden 7168); this takes 83 us, 1.1 PFLOP/s of bf16 products (with the norm's output of that
// moment still to be written back, as in a layer, 87 to 98). With K split it also serves fewer tokens: 4096 tokens
// 86 us on the per-wavefront kernel, 49 here; 1000: 27.7 and 21.9; 200: 15.5 and 13.2, the reduction included.
constexpr int BIG_TOKENS = 128;
constexpr int BIG_EXPERTS = 64;
constexpr int BIG_STAGE = (BIG_TOKENS + 3 * BIG_EXPERTS) * K_CHUNK * 2;  // bytes (40 KB)
constexpr int BIG_STAGES = 3;
constexpr int BIG_LOADS = BIG_STAGE / 1024 / 4;  // load instructions of a wavefront per stage

typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef const __attribute__((address_space(3))) uint8_t* lds_bytes;

// 64 lanes x 16 bytes, global -> LDS (lds_base + lane*16). asm, so that later LDS reads are not made to wait for it: its
// completion is awaited once per chunk.
__device__ __forceinline__ void dma16(const void* base, uint32_t lane_byte_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_byte_offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}

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

// logits = partial[0] + partial[1] + ... in that order
__global__ __launch_bounds__(256) void moe_router_reduce_kernel(const float* __restrict__ partial,
                                                                float* __restrict__ logits,
                                                                size_t count, int n_splits) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    // eight loads at a time are in flight; the additions stay in ascending split order
    float sum = 0.f;
    for (int s0 = 0; s0 < n_splits; s0 += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = s0 + j < n_splits ? partial[(size_t)(s0 + j) * count + i] : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (s0 + j < n_splits) sum = (s0 + j == 0) ? v[j] : sum + v[j];
    }
    logits[i] = sum;
}

int pick_router_splits(int tokens, int hidden, int n_experts) {
    const long tiles = (long)((tokens + 63) / 64) * ((n_experts + 63) / 64);
    const int n_chunks = hidden / K_CHUNK;
    int splits = 1;
    // aim at about two workgroups per CU; every split keeps at least 2 chunks
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
    (void)config;
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
    if (x_dtype == 0) {
        moe_router_gemm_kernel<float><<<grid, 256, 0, stream>>>(
            static_cast<const float*>(x), w, out, tokens, hidden, n_experts, chunks_per_split);
    } else {
        moe_router_gemm_kernel<uint16_t><<<grid, 256, 0, stream>>>(
            static_cast<const uint16_t*>(x), w, out, tokens, hidden, n_experts, chunks_per_split);
    }
    if (splits > 1) {
        const size_t count = (size_t)tokens * n_experts;
        moe_router_reduce_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(
            static_cast<const float*>(workspace), logits, count, splits);
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
    const int n_chunks = hidden / K_CHUNK;
    const int chunks_per_split = (n_chunks + splits - 1) / splits;
    // Enough 128 x 64 tiles and splits to fill the chip: the workgroup-tiled kernel (config 2 forces it, 1 the other one).
    // It has one workgroup on a CU, so that a part of a second round costs a whole one, which few chunks of K do not make up
    // for, all the less where each has little to share (us, tiled and not; 1500 tokens of 4096 x 64, 384 workgroups of 2
    // chunks: 17.3, 15.4; 1400 of 1024 x 256, 352 of 2: 15.9, 14.0; one tile of experts, 1200 of 7168 x 64, 320 of 4: 18.7,
    // 17.9; a third of the rows padding, 160 of 7168 x 384, 384 of 4: 18.1, 17.0; but 300 of 7168 x 256, 384 of 4: 19.2, 20.7).
    const long token_tiles = (tokens + BIG_TOKENS - 1) / BIG_TOKENS;
    const long big_wgs = token_tiles * ((n_experts + BIG_EXPERTS - 1) / BIG_EXPERTS) * splits;
    const bool part_of_second_round = big_wgs > 256 && big_wgs < 512;
    const bool few_chunks = chunks_per_split <= 2 ||
                            (chunks_per_split <= 4 && splits >= 16 && big_wgs < 448 &&
                             (n_experts <= BIG_EXPERTS || 3L * tokens < 2 * BIG_TOKENS * token_tiles));
    const bool tiled = hidden <= (1 << 24) && (config == 2 || (config != 1 && big_wgs >= 192 && tokens >= BIG_TOKENS &&
                                                              !(part_of_second_round && few_chunks)));
    float* out = splits > 1 ? static_cast<float*>(workspace) : logits;
    const int tile_tokens = tiled ? BIG_TOKENS : 64;
    const dim3 grid((tokens + tile_tokens - 1) / tile_tokens, (n_experts + 63) / 64, splits);
    const auto kernel = tiled ? moe_router_gemm_split_tiled_kernel : moe_router_gemm_split_kernel;
    kernel<<<grid, 256, 0, stream>>>(static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(planes), out, tokens,
                                     hidden, n_experts, chunks_per_split);
    if (splits > 1) {
        const size_t count = (size_t)tokens * n_experts;
        moe_router_reduce_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(
            static_cast<const float*>(workspace), logits, count, splits);
    }
}
