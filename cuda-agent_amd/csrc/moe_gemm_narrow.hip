// Grouped FP8 GEMMs of the MoE layer, narrow tiles: a few to about a hundred pairs per expert.
//
// With that many pairs the layer is still bound by the stream of its weights. The streaming form (moe_gemm.hip) goes
// over an expert's weights once per 16 or 32 pairs, and the 256-pair tiles (moe_gemm_tiled.hip) run one workgroup per
// CU, so that nothing is loaded while a workgroup starts and ends. Here a workgroup of 4 wavefronts computes 256 weight
// rows (gate/up: 128 gate rows and the matching 128 up rows) x up to 62 pairs of one expert, in 80 KB of LDS and 256
// registers, which is what lets two of them share a CU: one streams while the other starts, ends or waits.
//
// Per 128-block of K a stage holds 32 KB of weights and 64 rows of activations, the last two of which are not rows: they
// hold the block's pair scales (hence 62). Two stages; a wavefront copies its operands of a block into registers, and
// after a barrier the stage is filled with the block after the next, so that two blocks are in flight all the time.
// Each wavefront loads the 64 weight rows it multiplies itself, and a quarter of the activations. The weights of an
// expert with one tile carry the non-temporal hint (256 experts of 7168 x 2048, 31 pairs each: 1.92 ms a layer, 2.13
// without it; 47: 2.02 and 2.18); those of an expert with several do not (with it on all weights, 64 pairs: 2.81 ms
// instead of 2.54).
//
// Measured, 7168 x 2048 x 256 experts, 8 pairs each: gate/up 1.08 ms = 7.0 TB/s of weights, the read rate of this card;
// down 0.62 ms = 6.0 TB/s (16 K blocks a tile: starting and ending weigh more). The whole layer of 1000 tokens takes
// 1.90 ms (streaming 2.48, 256-pair tiles 2.24), of 1500 tokens 1.98 (3.72, 2.34). HBM reads of the layer of 1500 tokens with
// a shared expert: 8.00 GB in gate/up, 4.02 GB in down, for 7.55 and 3.77 GB of weights.
//
// Operand layout, LDS swizzle (slot of 16-byte chunk c of row r: r*8 + (c ^ ((r >> 1) & 7))) and the folding of the block
// scales are those of moe_gemm_tiled.hip. The gate/up GEMM converts the codes to bf16 in registers and multiplies on
// the bf16 matrix core, as the streaming form does and for its reason: the requantised h agrees with an fp32 evaluation
// (1500 pairs of 7168 x 2048: 29 of 3.07 million codes are not those of a float64 evaluation, as in the streaming form;
// 4624 with the 256-pair tiles, which repair the large ones).
#include "lane_exchange.hpp"
#include "launch_status.hpp"
#include "moe_tile.hpp"

namespace {

using namespace moe;

constexpr int ROWS = 256;              // weight rows of a tile
constexpr int PAIRS = 62;              // pairs of a tile
constexpr int PAIR_COLS = 64;          // columns of the result (the last two belong to no pair)
constexpr int STAGE_A = ROWS * GROUP;  // 32 KB
constexpr int SCALES_AT = STAGE_A + PAIRS * GROUP;
constexpr int STAGE_BYTES = STAGE_A + PAIR_COLS * GROUP;
constexpr int WAVE_A = 64 * GROUP;     // one wavefront's weight rows of a stage
static_assert((PAIR_COLS - PAIRS) * GROUP == PAIR_COLS * (int)sizeof(float), "two rows hold the scales of all columns");

__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }

// Y_F32 (down only): y as fp32 rows; otherwise fp16 with a power of two per pair and 256 columns (y_scale).
template <bool GATE_UP, bool Y_F32>
__global__ __launch_bounds__(256, 2) void moe_narrow_gemm_kernel(
    const uint8_t* __restrict__ w_q, const float* __restrict__ w_s, const uint8_t* __restrict__ a_q,
    const float* __restrict__ as_t, const int* __restrict__ sorted_pairs, const int* __restrict__ expert_offsets,
    const int* __restrict__ tile_start, uint8_t* __restrict__ h_q, float* __restrict__ h_s, float* __restrict__ hs_t,
    void* __restrict__ y, float* __restrict__ y_scale, int K, int n_rows, int inter, int top_k, int n_experts,
    int scale_stride, bool pow2) {
    __shared__ __attribute__((aligned(16))) uint8_t s_stage[2 * STAGE_BYTES];

    int rb, e, in_expert;
    if (!find_tile(tile_start, n_experts, GATE_UP ? inter / GROUP : n_rows / ROWS, rb, e, in_expert)) return;
    // an expert's tiles are of equal size
    const int expert_begin = expert_offsets[e];
    const int expert_pairs = expert_offsets[e + 1] - expert_begin;
    const int tiles = (expert_pairs + PAIRS - 1) / PAIRS;
    const int per_tile = (expert_pairs + tiles - 1) / tiles;
    const int begin = expert_begin + in_expert * per_tile;
    const int cnt = min(per_tile, expert_pairs - in_expert * per_tile);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int KB = K / GROUP;
    const int row_blocks = n_rows / GROUP;
    const int r32 = lane & 31;
    const int half = lane >> 5;

    // ---- fill side: a load instruction covers 8 rows, lane -> row lane/8, chunk (lane%8) ^ ((row >> 1) & 7) ----
    const uint32_t ld_row = lane >> 3;
    const uint32_t ld_chunk = (lane & 7) ^ (ld_row >> 1);  // (instructions of odd number: ^ 4)
    const uint32_t ld_off_even = ld_row * (uint32_t)K + 16 * ld_chunk;
    const uint32_t ld_off_odd = ld_row * (uint32_t)K + 16 * (ld_chunk ^ 4);
    // this wavefront's 64 rows are two runs of 32: MFMA tiles 0 and 1
    const int row0 = GATE_UP ? rb * GROUP + wave * 32 : rb * ROWS + wave * 64;
    const uint8_t* run0 = w_q + ((size_t)e * n_rows + row0) * K;
    const uint8_t* run1 = run0 + (size_t)(GATE_UP ? inter : 32) * K;
    uint32_t b_off[2];
    bool b_row[2];
    int in_flight = 8 + (wave == 0 ? 1 : 0);  // load instructions of this wavefront per block
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int p = (2 * wave + i) * 8 + (int)ld_row;
        b_row[i] = p < cnt;  // (rows of no pair keep what LDS holds: they feed columns that are not stored)
        const int pos = begin + (b_row[i] ? p : 0);
        const int arow = GATE_UP ? sorted_pairs[pos] / top_k : pos;
        b_off[i] = (uint32_t)arow * (uint32_t)K + 16 * (ld_chunk ^ (4 * i));
        in_flight += (2 * wave + i) * 8 < cnt ? 1 : 0;
    }
    const float* s_src = as_t + begin;  // + kb*scale_stride; 64 floats, the tail is other pairs' or padding
    const float* ws0;
    const float* ws1;
    if (GATE_UP) {
        ws0 = w_s + ((size_t)e * row_blocks + rb) * KB;
        ws1 = w_s + ((size_t)e * row_blocks + inter / GROUP + rb) * KB;
    } else {
        ws0 = w_s + ((size_t)e * row_blocks + rb * 2 + (wave >> 1)) * KB;
        ws1 = ws0;
    }
    const bool once = tiles == 1;  // these weights are read by no other workgroup
    const uint32_t stage_base = (uint32_t)(size_t)((lds_void_ptr)s_stage);
    // load n (0..10) of block kb: pair scales, two row groups of activations, eight of weights
    constexpr int LOADS = 11;
    auto issue_load = [&](int kb, int n) {
        const uint32_t st = stage_base + (kb & 1) * STAGE_BYTES;
        if (n == 0) {
            if (wave == 0 && lane < 16) dma16(s_src + (size_t)kb * scale_stride, lane * 16, st + SCALES_AT);
        } else if (n < 3) {
            if (b_row[n - 1]) dma16(a_q + (size_t)kb * GROUP, b_off[n - 1], st + STAGE_A + (2 * wave + n - 1) * 1024);
        } else {
            const int i = n - 3;
            const uint8_t* src = (i < 4 ? run0 : run1) + (size_t)(8 * (i & 3)) * K + (size_t)kb * GROUP;
            const uint32_t off = (i & 1) ? ld_off_odd : ld_off_even;
            if (once) dma16_once(src, off, st + wave * WAVE_A + i * 1024);
            else dma16(src, off, st + wave * WAVE_A + i * 1024);
        }
    };

    // ---- read side: operand of k-step s, 16-byte piece j: chunk 4s + 2*half + j of row r32 (+32*tile) ----
    const uint32_t rd = (r32 * 8 + ((2 * half) ^ ((r32 >> 1) & 7))) * 16;
    const lds_bytes stage_ptr = (lds_bytes)s_stage;

    floatx16 acc[2][2];  // [weight rows 32*a][pairs 32*b]
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = floatx16{0};

    // One block of K for NB tiles of 32 pairs; MORE: there is a block kb+2 to request.
    auto block = [&](auto nb_tag, auto more_tag, int kb) {
        constexpr int NB = decltype(nb_tag)::value;
        constexpr bool MORE = decltype(more_tag)::value != 0;
        const lds_bytes st = stage_ptr + (kb & 1) * STAGE_BYTES;
        const float w[2] = {ws0[kb], ws1[kb]};
        auto operand = [&](lds_bytes row0_ptr, int s) {
            return join(*(lds_x4)(row0_ptr + (rd ^ (64 * s))), *(lds_x4)(row0_ptr + (rd ^ (64 * s) ^ 16)));
        };
        intx8 A[2][2], B[NB][2];  // [tile][k-step]
        float bs[NB];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int a = 0; a < 2; ++a) A[a][s] = operand(st + wave * WAVE_A + a * 32 * GROUP, s);
#pragma unroll
            for (int b = 0; b < NB; ++b) B[b][s] = operand(st + STAGE_A + b * 32 * GROUP, s);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
            bs[b] = *(const __attribute__((address_space(3))) float*)(st + SCALES_AT + (b * 32 + r32) * 4);
        if constexpr (MORE) {
            // every wavefront holds its operands: the stage may be filled again
            __builtin_amdgcn_s_waitcnt((63 & 15) | ((63 >> 4) << 14) | (7 << 4) | (0 << 8));  // lgkmcnt(0)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        // the loads of block kb+2, spread over the products (a load holds the wavefront until the memory pipeline
        // has taken it)
        constexpr int SLOTS = 2 * NB;
        auto loads = [&](int slot) {
            if constexpr (MORE) {
#pragma unroll
                for (int n = 0; n < LOADS; ++n)
                    if (n * SLOTS / LOADS == slot) issue_load(kb + 2, n);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if constexpr (GATE_UP) {
            // A lane's 32 operand bytes of a k-step, eight at a time, are the operands of four bf16 MFMAs (A and B
            // take the same bytes of their lanes, so the products pair up the same k).
            bf16x8 Ab[2][8];
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    Ab[a][u] = e4m3x8_to_bf16(A[a][u >> 2][2 * (u & 3)], A[a][u >> 2][2 * (u & 3) + 1]);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                bf16x8 Bb[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    Bb[u] = e4m3x8_to_bf16(B[b][u >> 2][2 * (u & 3)], B[b][u >> 2][2 * (u & 3) + 1]);
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    floatx16 p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Ab[a][0], Bb[0], floatx16{0}, 0, 0, 0);
#pragma unroll
                    for (int u = 1; u < 8; ++u) p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Ab[a][u], Bb[u], p, 0, 0, 0);
                    loads(2 * b + a);
                    acc[a][b] += p * (bs[b] * w[a]);
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    floatx16 p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[a][0], B[b][0], floatx16{0}, 0, 0, 0, 0, 0, 0);
                    p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[a][1], B[b][1], p, 0, 0, 0, 0, 0, 0);
                    loads(2 * b + a);
                    acc[a][b] += p * (bs[b] * w[a]);
                }
            }
        }
    };
    // at the top of block kb: its loads are complete, those of block kb+1 may be in flight
    auto await_block = [&](bool last) {
        switch (last ? 0 : in_flight) {
            case 8: __builtin_amdgcn_s_waitcnt(8 | (7 << 4) | (15 << 8)); break;
            case 9: __builtin_amdgcn_s_waitcnt(9 | (7 << 4) | (15 << 8)); break;
            case 10: __builtin_amdgcn_s_waitcnt(10 | (7 << 4) | (15 << 8)); break;
            case 11: __builtin_amdgcn_s_waitcnt(11 | (7 << 4) | (15 << 8)); break;
            default: __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8)); break;
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    wait_all_loads();  // (nothing of the compiler's is in flight when the counted loads start)
#pragma unroll
    for (int n = 0; n < LOADS; ++n) issue_load(0, n);
    if (KB > 1) {
#pragma unroll
        for (int n = 0; n < LOADS; ++n) issue_load(1, n);
    }
    auto k_loop = [&](auto nb_tag) {
        for (int kb = 0; kb < KB - 2; ++kb) {
            await_block(false);
            block(nb_tag, IntConstant<1>{}, kb);
            asm volatile("" ::: "memory");
        }
        for (int kb = KB > 1 ? KB - 2 : 0; kb < KB; ++kb) {
            await_block(kb + 1 == KB);
            block(nb_tag, IntConstant<0>{}, kb);
            asm volatile("" ::: "memory");
        }
    };
    if (cnt > 32) k_loop(IntConstant<2>{});
    else k_loop(IntConstant<1>{});
    __syncthreads();  // the stages are free: the epilogue transposes through them

    // result layout: register i of acc[a][b] is row 8*(i/4) + 4*half + i%4 of run a, pair b*32 + r32
    if constexpr (GATE_UP) {
        float* s_amax = reinterpret_cast<float*>(s_stage);  // [4 wavefronts][64 pairs]
        constexpr int CODE_ROW = GROUP + 16;                // bytes per pair row of codes
        uint8_t* s_codes = s_stage + 4 * PAIR_COLS * sizeof(float);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float m = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                acc[0][b][i] = silu(acc[0][b][i]) * acc[1][b][i];
                m = fmaxf(m, fabsf(acc[0][b][i]));
            }
            m = lanes::max_of_halves(m);
            if (half == 0) s_amax[wave * PAIR_COLS + b * 32 + r32] = m;
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int pl = b * 32 + r32;
            const float m = fmaxf(fmaxf(s_amax[pl], s_amax[PAIR_COLS + pl]),
                                  fmaxf(s_amax[2 * PAIR_COLS + pl], s_amax[3 * PAIR_COLS + pl]));
            const float scale = group_scale(m, pow2);
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                float q[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    q[r] = fminf(fmaxf(acc[0][b][4 * qd + r] / scale, -E4M3_MAX), E4M3_MAX);
                int packed = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
                packed = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], packed, true);
                *reinterpret_cast<int*>(s_codes + pl * CODE_ROW + wave * 32 + 8 * qd + 4 * half) = packed;
            }
            if (wave == 0 && half == 0 && pl < cnt) {
                const size_t pos = (size_t)begin + pl;
                h_s[pos * (inter / GROUP) + rb] = scale;
                hs_t[(size_t)rb * scale_stride + pos] = scale;
            }
        }
        __syncthreads();
        // 8 lanes write the 128 codes of one pair
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int pl = (wave * 2 + it) * 8 + (lane >> 3);
            if (pl < cnt) {
                const size_t at = ((size_t)begin + pl) * inter + rb * GROUP + (lane & 7) * 16;
                *reinterpret_cast<intx4*>(h_q + at) = *reinterpret_cast<const intx4*>(s_codes + pl * CODE_ROW + (lane & 7) * 16);
            }
        }
    } else if constexpr (Y_F32) {
        constexpr int Y_ROW = ROWS + 4;  // floats per staged pair row
        float* s_y = reinterpret_cast<float*>(s_stage);
        static_assert(PAIR_COLS * Y_ROW * sizeof(float) <= 2 * STAGE_BYTES, "epilogue LDS");
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int qd = 0; qd < 4; ++qd)
                    *reinterpret_cast<floatx4*>(s_y + (b * 32 + r32) * Y_ROW + wave * 64 + a * 32 + 8 * qd + 4 * half) =
                        floatx4{acc[a][b][4 * qd], acc[a][b][4 * qd + 1], acc[a][b][4 * qd + 2], acc[a][b][4 * qd + 3]};
        __syncthreads();
        // a wavefront writes the 1 KB of one pair per instruction
#pragma unroll 4
        for (int pl = wave; pl < cnt; pl += 4)
            *reinterpret_cast<floatx4*>(static_cast<float*>(y) + ((size_t)begin + pl) * n_rows + rb * ROWS + lane * 4) =
                *reinterpret_cast<const floatx4*>(s_y + pl * Y_ROW + lane * 4);
    } else {
        // fp16 of y / 2^e, 2^e the power of two above the largest magnitude of the pair's 256 values of this tile, as
        // moe_gemm_tiled.hip stores it
        typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));
        constexpr int Y_ROW = ROWS + 8;  // halfs per staged pair row
        _Float16* s_y = reinterpret_cast<_Float16*>(s_stage);
        float* s_max = reinterpret_cast<float*>(s_stage + PAIR_COLS * Y_ROW * sizeof(_Float16));  // [4 wavefronts][64 pairs]
        static_assert(PAIR_COLS * Y_ROW * sizeof(_Float16) + 4 * PAIR_COLS * sizeof(float) <= 2 * STAGE_BYTES, "epilogue LDS");
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float m = 0.f;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int i = 0; i < 16; ++i) m = fmaxf(m, fabsf(acc[a][b][i]));
            m = lanes::max_of_halves(m);
            if (half == 0) s_max[wave * PAIR_COLS + b * 32 + r32] = m;
        }
        __syncthreads();
        auto pair_exponent = [&](int pl) {  // biased exponent of 2^e
            const float m = fmaxf(fmaxf(s_max[pl], s_max[PAIR_COLS + pl]),
                                  fmaxf(s_max[2 * PAIR_COLS + pl], s_max[3 * PAIR_COLS + pl]));
            const uint32_t e_bits = ((__float_as_uint(m) >> 23) & 255u) + 1u;
            return m > 0.f ? (e_bits > 253u ? 253u : e_bits) : 127u;
        };
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const float inv = __uint_as_float((254u - pair_exponent(b * 32 + r32)) << 23);
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int qd = 0; qd < 4; ++qd)
                    *reinterpret_cast<halfx4*>(s_y + (b * 32 + r32) * Y_ROW + wave * 64 + a * 32 + 8 * qd + 4 * half) =
                        halfx4{(_Float16)(acc[a][b][4 * qd] * inv), (_Float16)(acc[a][b][4 * qd + 1] * inv),
                               (_Float16)(acc[a][b][4 * qd + 2] * inv), (_Float16)(acc[a][b][4 * qd + 3] * inv)};
        }
        __syncthreads();
        // 32 lanes write the 512 bytes of one pair
#pragma unroll 4
        for (int pl = 2 * wave + half; pl < cnt; pl += 8) {
            const size_t row = (size_t)begin + pl;
            *reinterpret_cast<intx4*>(static_cast<_Float16*>(y) + row * n_rows + rb * ROWS + r32 * 8) =
                *reinterpret_cast<const intx4*>(s_y + pl * Y_ROW + r32 * 8);
            if (r32 == 0) y_scale[row * (n_rows / ROWS) + rb] = __uint_as_float(pair_exponent(pl) << 23);
        }
    }
}

bool sizes_ok(unsigned long long a_bytes, int hidden, int inter) {
    return hidden > 0 && inter > 0 && hidden % ROWS == 0 && inter % GROUP == 0 && a_bytes < (1ull << 32);  // 32-bit offsets
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

// Pairs of one tile: what moe_tiled_prepare_launcher numbers the tiles for.
extern "C" int moe_narrow_tile_pairs() { return PAIRS; }

// As moe_gate_up_tiled_launcher with the exact requantisation.
extern "C" void moe_gate_up_narrow_launcher(void* h_q, float* h_s, float* hs_t, const void* x_q, const float* xs_t,
                                            const void* w13_q, const float* w13_s, const int* sorted_pairs,
                                            const int* expert_offsets, const int* tile_start, int tokens, int hidden,
                                            int inter, int n_experts, int top_k, int scale_stride, int ue8m0,
                                            hipStream_t stream) {
    if (tokens <= 0) return;
    if (!sizes_ok((unsigned long long)tokens * hidden, hidden, inter)) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    if (!h_q || !h_s || !hs_t || !x_q || !xs_t || !w13_q || !w13_s || !sorted_pairs || !expert_offsets || !tile_start ||
        !aligned16(h_q) || !aligned16(x_q) || !aligned16(w13_q)) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    const dim3 grid(tiled_grid(inter / GROUP, (int)((long)tokens * top_k / PAIRS) + n_experts));
    moe_narrow_gemm_kernel<true, false><<<grid, 256, 0, stream>>>(
        static_cast<const uint8_t*>(w13_q), w13_s, static_cast<const uint8_t*>(x_q), xs_t, sorted_pairs, expert_offsets,
        tile_start, static_cast<uint8_t*>(h_q), h_s, hs_t, nullptr, nullptr, hidden, 2 * inter, inter, top_k, n_experts,
        scale_stride, ue8m0 != 0);
}

// y as moe_down_tiled_launcher stores it, or, y_scale null, as moe_down_launcher does (fp32 rows).
extern "C" void moe_down_narrow_launcher(float* y, float* y_scale, const void* h_q, const float* hs_t, const void* w2_q,
                                         const float* w2_s, const int* expert_offsets, const int* tile_start, int tokens,
                                         int hidden, int inter, int n_experts, int top_k, int scale_stride,
                                         hipStream_t stream) {
    if (tokens <= 0) return;
    if (!sizes_ok((unsigned long long)tokens * top_k * inter, hidden, inter)) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    if (!y || !h_q || !hs_t || !w2_q || !w2_s || !expert_offsets || !tile_start || !aligned16(y) || !aligned16(h_q) ||
        !aligned16(w2_q)) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    const dim3 grid(tiled_grid(hidden / ROWS, (int)((long)tokens * top_k / PAIRS) + n_experts));
    const auto kernel = y_scale ? moe_narrow_gemm_kernel<false, false> : moe_narrow_gemm_kernel<false, true>;
    kernel<<<grid, 256, 0, stream>>>(static_cast<const uint8_t*>(w2_q), w2_s, static_cast<const uint8_t*>(h_q), hs_t,
                                     nullptr, expert_offsets, tile_start, nullptr, nullptr, nullptr, y, y_scale, inter,
                                     hidden, inter, top_k, n_experts, scale_stride, false);
}
