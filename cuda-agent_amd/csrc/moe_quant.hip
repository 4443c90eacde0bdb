// Activation quantisation: bf16 rows -> e4m3 codes with one fp32 scale per 128-wide group.
//   scale = max(amax, 1e-12) * fp32(1/448);  code = e4m3_rne(clamp(v / scale, -448, 448))
//   (or, on request, scale = the smallest power of two >= max(amax, 1e-12) / 448)
// One wavefront per (row, group), two elements per lane. The division is IEEE fp32 so that the
// codes are bit-identical to a CPU evaluation of the same formula; v_cvt_pk_fp8_f32 rounds to
// nearest even but does not saturate (465 -> NaN), hence the clamp.
#include <hip/hip_bf16.h>

#include "lane_exchange.hpp"
#include "launch_status.hpp"
#include "moe_common.hpp"

namespace {

using namespace moe;

__global__ __launch_bounds__(256) void moe_quant_bf16_kernel(const __hip_bfloat16* __restrict__ x,
                                                             uint8_t* __restrict__ q,
                                                             float* __restrict__ scales,
                                                             long n_groups, bool pow2) {
    const int lane = threadIdx.x & 63;
    const long g = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (g >= n_groups) return;
    const unsigned raw = *reinterpret_cast<const unsigned*>(x + g * GROUP + 2 * lane);
    const float v0 = __uint_as_float(raw << 16);
    const float v1 = __uint_as_float(raw & 0xffff0000u);
    float amax = fmaxf(fabsf(v0), fabsf(v1));
    amax = lanes::butterfly_max<32>(amax);
    const float scale = group_scale(amax, pow2);
    const float a = fminf(fmaxf(v0 / scale, -E4M3_MAX), E4M3_MAX);
    const float b = fminf(fmaxf(v1 / scale, -E4M3_MAX), E4M3_MAX);
    const int packed = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    *reinterpret_cast<uint16_t*>(q + g * GROUP + 2 * lane) = (uint16_t)(packed & 0xffff);
    if (lane == 0) scales[g] = scale;
}

// Same result with 16 lanes per group: a lane loads 8 values (16 bytes) and stores 8 codes.
template <bool SHUFFLED>
__global__ __launch_bounds__(256) void moe_quant_bf16_vec_kernel(const __hip_bfloat16* __restrict__ x,
                                                                 uint8_t* __restrict__ q,
                                                                 float* __restrict__ scales,
                                                                 long n_groups, bool pow2) {
    const long g = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (g < n_groups) quantise_group16<SHUFFLED>(x, q, scales, g, threadIdx.x & 15, pow2);
}

}  // namespace

// q [rows, cols] e4m3 codes and scales [rows, cols/128] fp32 from x [rows, cols] bf16.
// config bit 32: power-of-two scales (the smallest power of two >= amax / 448).
extern "C" void moe_quant_bf16_launcher(void* q, float* scales, const void* x, int rows, int cols,
                                        int config, hipStream_t stream) {
    const bool pow2 = (config & CONFIG_UE8M0) != 0;
    if (rows <= 0 || cols <= 0) return;
    if (cols % GROUP != 0) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    if (!q || !scales || !x || (reinterpret_cast<uintptr_t>(x) & 3u) ||
        (reinterpret_cast<uintptr_t>(q) & 1u)) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    const long n_groups = (long)rows * (cols / GROUP);
    if (!(reinterpret_cast<uintptr_t>(x) & 15u) && !(reinterpret_cast<uintptr_t>(q) & 7u)) {
        // The maximum of a group through the LDS crossbar where the workgroups are five to thirty to a CU: wavefronts that wait
        // for it leave the vector ALU to those that have yet to request their values. us on the vector ALU and so, x in the caches,
        // and not: 24000 groups 3.5, 3.5 and 4.2, 4.1; 32768 4.0, 3.9 and 4.8, 4.6; 40000 5.1, 4.9 and 5.6, 5.5; 64000 6.9, 6.6 and 7.6,
        // 7.5; 80000 7.9, 7.5 and 8.7 either way; 112000 9.7, 9.4 and 11.3 either way; but 16000 2.9, 2.9 and 3.5, 3.5; 168000 12.9, 12.8
        // and 15.2, 15.7.
        const bool shuffled = n_groups > 16 * 5 * 256 && n_groups <= 16 * 30 * 256;
        const auto kernel = shuffled ? moe_quant_bf16_vec_kernel<true> : moe_quant_bf16_vec_kernel<false>;
        kernel<<<dim3((unsigned)((n_groups + 15) / 16)), 256, 0, stream>>>(
            static_cast<const __hip_bfloat16*>(x), static_cast<uint8_t*>(q), scales, n_groups, pow2);
        return;
    }
    const long blocks = (n_groups + 3) / 4;
    moe_quant_bf16_kernel<<<dim3((unsigned)blocks), 256, 0, stream>>>(
        static_cast<const __hip_bfloat16*>(x), static_cast<uint8_t*>(q), scales, n_groups, pow2);
}

namespace {

__device__ __forceinline__ void unpack_bf16x8(float (&v)[8], const unsigned (&raw)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = __uint_as_float(raw[j] << 16);
        v[2 * j + 1] = __uint_as_float(raw[j] & 0xffff0000u);
    }
}

// one run of a row: v its values, w their weights, `at` its place in x, group16 the lane's number among the 16 of its group.
// STREAM: the codes carry the non-temporal hint
template <bool STREAM>
__device__ __forceinline__ void normalise_run(float (&v)[8], const float (&w)[8], float rinv, size_t at, int group16,
                                              __hip_bfloat16* __restrict__ y, uint8_t* __restrict__ q,
                                              float* __restrict__ scale_at, bool pow2) {
    typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
    typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
    float amax = 0.f;
    unsigned packed_y[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float n = __bfloat162float(__float2bfloat16(v[j] * rinv));  // the norm's result in bf16
        const __hip_bfloat16 yb = __float2bfloat16(w[j] * n);            // times the weight, in bf16
        v[j] = __bfloat162float(yb);
        amax = fmaxf(amax, fabsf(v[j]));
        const unsigned bits = (unsigned)(__float_as_uint(v[j]) >> 16);
        if (j & 1) packed_y[j >> 1] |= bits << 16; else packed_y[j >> 1] = bits;
    }
    if (y != nullptr) *reinterpret_cast<uintx4*>(y + at) = uintx4{packed_y[0], packed_y[1], packed_y[2], packed_y[3]};
    amax = lanes::butterfly_max<8>(amax);
    const float scale = group_scale(amax, pow2);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = fminf(fmaxf(v[j] / scale, -E4M3_MAX), E4M3_MAX);
    uintx2 packed;
    int lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
    int hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], 0, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], hi, true);
    packed[0] = (unsigned)lo;
    packed[1] = (unsigned)hi;
    if constexpr (STREAM) __builtin_nontemporal_store(packed, reinterpret_cast<uintx2*>(q + at));
    else *reinterpret_cast<uintx2*>(q + at) = packed;
    if (group16 == 0) *scale_at = scale;
}

// RMS normalisation of a row followed by the activation quantisation of the result, one workgroup per row (cols <=
// 8192): y = w * bf16(x * rsqrt(mean(x^2) + eps)) rounded to bf16 (the two roundings of a bf16 norm layer), then per
// 128-wide group of y the scale and the e4m3 codes of moe_quant_bf16. A lane owns runs of 8 consecutive values (16 lanes
// per group), 8 * LANES apart; the row is read once and y, the codes and the scales are written once.
// LANES: 1024 lanes with one run each finish a row soonest, which is what counts while every row has a workgroup's place
// to itself; with more rows what counts is how many of them are in flight, and a CU holds six workgroups of 256 lanes
// against two of 1024. The shorter the row, the sooner lanes without a run outweigh what the others gain.
// STREAM (256 lanes): x and the codes carry the non-temporal hint.
// Both forms add the squares in the same order: within a run, over the 64 lanes of 512 consecutive values, then these
// sums in ascending order.
template <int LANES, bool STREAM>
__global__ __launch_bounds__(LANES) void moe_rmsnorm_quant_kernel(const __hip_bfloat16* __restrict__ x,
                                                                  const __hip_bfloat16* __restrict__ weight,
                                                                  __hip_bfloat16* __restrict__ y,
                                                                  uint8_t* __restrict__ q,
                                                                  float* __restrict__ scales, int cols,
                                                                  float eps, bool pow2) {
    typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
    constexpr int RUNS = 1024 / LANES;
    __shared__ float s_part[16];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const size_t row = blockIdx.x;
    auto load = [&](unsigned (&raw)[4], const __hip_bfloat16* src) {
        const uintx4 r = *reinterpret_cast<const uintx4*>(src);
        raw[0] = r.x, raw[1] = r.y, raw[2] = r.z, raw[3] = r.w;
    };
    // the squares of 512 consecutive values, number `part` of the row
    auto add_squares = [&](float ss, int part) {
        ss = lanes::butterfly_sum<32>(ss);
        if (lane == 0) s_part[part] = ss;
    };
    auto row_rinv = [&]() {
        __syncthreads();
        float total = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) total += s_part[i];
        return 1.f / sqrtf(total / (float)cols + eps);  // correctly rounded, as a CPU evaluation
    };
    auto finish = [&](float (&v)[8], const float (&w)[8], float rinv, int c0) {
        normalise_run<STREAM>(v, w, rinv, row * cols + c0, tid & 15, y, q, scales + row * (cols / GROUP) + c0 / GROUP, pow2);
    };
    if constexpr (RUNS == 1) {
        const int c0 = tid * 8;
        const bool live = c0 < cols;
        float v[8], w[8];
        float ss = 0.f;
        if (live) {
            unsigned raw[4], wraw[4];
            load(raw, x + row * cols + c0);
            load(wraw, weight + c0);
            unpack_bf16x8(v, raw);
            unpack_bf16x8(w, wraw);
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = fmaf(v[j], v[j], ss);
        }
        add_squares(ss, wave);
        const float rinv = row_rinv();
        if (live) finish(v, w, rinv, c0);
    } else {
        // (four runs stay packed until they are used: 78 registers, six workgroups on a CU)
        unsigned raw[RUNS][4], wraw[RUNS][4];
#pragma unroll
        for (int r = 0; r < RUNS; ++r) {
            const int c0 = (r * LANES + tid) * 8;
#pragma unroll
            for (int j = 0; j < 4; ++j) raw[r][j] = wraw[r][j] = 0u;
            if (c0 < cols) {
                if constexpr (STREAM) {
                    const uintx4 xr = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(x + row * cols + c0));
                    raw[r][0] = xr.x, raw[r][1] = xr.y, raw[r][2] = xr.z, raw[r][3] = xr.w;
                } else {
                    load(raw[r], x + row * cols + c0);
                }
                load(wraw[r], weight + c0);
            }
        }
#pragma unroll
        for (int r = 0; r < RUNS; ++r) {
            float v[8], ss = 0.f;
            unpack_bf16x8(v, raw[r]);
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = fmaf(v[j], v[j], ss);
            add_squares(ss, r * (LANES / 64) + wave);
        }
        const float rinv = row_rinv();
#pragma unroll
        for (int r = 0; r < RUNS; ++r) {
            const int c0 = (r * LANES + tid) * 8;
            if (c0 >= cols) return;
            float v[8], w[8];
            unpack_bf16x8(v, raw[r]);
            unpack_bf16x8(w, wraw[r]);
            finish(v, w, rinv, c0);
        }
    }
}

}  // namespace

// The norm in front of the layer fused with the layer's activation quantiser:
//   y [rows, cols] bf16 (or null) = weight * bf16(x * rsqrt(mean(x^2) + eps)), rounded to bf16
//   q [rows, cols] e4m3 codes and scales [rows, cols/128] fp32: moe_quant_bf16_launcher applied to y
// x [rows, cols] bf16, weight [cols] bf16; cols a multiple of 128, at most 8192; x, weight, y 16-byte and
// q 8-byte aligned. config bit 32: power-of-two scales.
extern "C" void moe_rmsnorm_quant_launcher(void* q, float* scales, void* y, const void* x,
                                           const void* weight, float eps, int rows, int cols,
                                           int config, hipStream_t stream) {
    const bool pow2 = (config & CONFIG_UE8M0) != 0;
    if (rows <= 0 || cols <= 0) return;
    if (cols % GROUP != 0 || cols > 8192) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                           reinterpret_cast<uintptr_t>(y);
    if (!q || !scales || !x || !weight || (bits & 15u) || (reinterpret_cast<uintptr_t>(q) & 7u)) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
    // us with 1024 lanes and with 256: 7168 columns 1400 rows 13.8 and 14.3, 1700: 16.0, 15.4, 8192: 68.4, 55.9 (4.9 TB/s, 60 %
    // of them writes); 4096: 1536 rows 9.5 and 10.0, 2000: 11.9, 11.8; 2048: 600 rows 4.6 and 4.8, 1000: 5.6, 5.3; 1024: 513 rows
    // 3.6 and 3.8, 768: 4.5, 4.1
    const bool many = rows > (cols > 2048 ? 1600 : cols > 1024 ? 768 : 576);
    // x and the codes past the caches where they and y don't fit the memory-side one (256 MB) together, so that y is there for
    // the router projection. us, through the caches and so: 8192 rows of 7168 (294 MB) alone 67.8, 59.0; with projection and
    // routing 157.4, 149.7, with a pass over the codes behind these 169.3, 162.0, with an addition to x 210.2, 206.9; norm and
    // gate/up GEMM of 256 experts of 2048, 8 a token 11748, 11749 (but 2427, 2480 of 8 experts of 128, one a token); 8192 of 4096
    // (168 MB) 35.6, 36.3; 94.9, 94.7; 107.2, 104.4; 126.5, 124.7; 3000 of 7168 (108 MB) 23.8, 26.1; 79.6, 79.7; 86.2,
    // 88.2; 100.4, 100.3; 8192 of 2048 (84 MB) 23.7, 25.7; 54.1, 53.8; 60.3, 60.1; 69.8, 71.2.
    const bool past_caches = many && y && (size_t)rows * cols * 5 > (256u << 20);
    const auto kernel = past_caches ? moe_rmsnorm_quant_kernel<256, true>
                        : many        ? moe_rmsnorm_quant_kernel<256, false>
                                      : moe_rmsnorm_quant_kernel<1024, false>;
    kernel<<<rows, many ? 256 : 1024, 0, stream>>>(
        static_cast<const __hip_bfloat16*>(x), static_cast<const __hip_bfloat16*>(weight),
        static_cast<__hip_bfloat16*>(y), static_cast<uint8_t*>(q), scales, cols, eps, pow2);
}
