// Top-k selection of index scores: the step that produces the row indices sparse-MLA decode
// gathers. Per request, the k largest of n fp32 scores, ties going to the lower index, listed in
// ascending index order; everything is integer work on the scores' bit patterns, so the result
// is exact.
//
//   key(x)  = the 32-bit pattern of x mapped monotonically to an unsigned integer (-0 = +0;
//             NaN maps to 0, below every number, so a NaN is chosen only when nothing else is left)
//   T       = the k-th largest key
//   chosen  = keys > T, plus the first (k - #greater) keys == T in index order
//
// One workgroup of 1024 lanes per request: nothing outside the outputs can be written, so the CUs of the chip cannot
// share a row. What bounds it is the vector ALU of that one CU (64 lanes a clock: one instruction per entry of a row
// of 65536 is 0.43 us) and the chain of barriers, so an entry is touched by as few instructions as possible:
//
//   pivot    an eighth of the row (spread evenly) goes into a histogram of 4096 key ranges; the rank in it that leaves
//            1.5 times the wanted entries plus four standard deviations of an independent sample gives a lower bound
//   collect  entries >= pivot, compared as floats, are appended to a list in LDS (about 3700 for k = 2048)
//   select   the list's keys are counted by their distance from the pivot, 2^13 keys to a bin; the few keys in the
//            bin of the k-th largest are sorted out bit by bit. Chosen entries become bits of a bitmap of the row,
//            whose words are placed in the output by a workgroup-wide scan
//
// If the sample says that the list would be too long, or it turns out shorter than k or too long (rows of few distinct
// values, a sample that misled), and for rows of up to 8192 or more than 262144 entries (the bitmaps' size) or k above
// 3072, the whole row is searched instead: a radix select with digits of 11, 11 and 10 bits, most significant first,
// which stops as soon as all keys of a digit's bin are wanted or the first digit's bin holds a single key.
//
// Rows of up to 65536 scores are held in registers, in words of 64 consecutive entries (a load instruction fetches
// 256 consecutive bytes; with 16-byte pieces of 64 different lines, as each lane owning consecutive entries asks for,
// the row came through L1 eight times). Longer rows are read again by each step. The output never depends on timing.
//
// Measured (us; one row unless stated, k = 2048; radix select over four 8-bit digits before): n = 8192 7.1 -> 6.1,
// 16384 10.3 -> 7.4, 32768 19.5 -> 9.9, 64 rows of it 20.0 -> 10.3; 65536 115 -> 13.8; 131072 221 -> 20.4. Rows that the
// whole-row search takes: one value, n = 8192 9.1 -> 5.9, 16384 14.0 -> 11.0, 32768 26 -> 18; two values 8.4 -> 6.6,
// 12.9 -> 11.5, 24.4 -> 18.9; 95 % masked 9.3 -> 7.0, 14.4 -> 12.9, 27 -> 21. Slower than before: rows that have k
// entries left unmasked but fewer than the sample's rank asks for, for which the sample is for nothing (95 % of 16384
// masked, k = 512: 10.8 -> 12.3), and 64 rows of 8192 in some 50 values (7.6 -> 7.9).
//
// Entries beyond a request's valid length (lengths[b], optional) are not candidates; if fewer
// than k candidates exist the remaining outputs are -1, which the attention treats as padding.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lane_exchange.hpp"
#include "launch_status.hpp"

namespace {

constexpr int SELECT_THREADS = 1024;
constexpr int SELECT_WAVES = SELECT_THREADS / 64;

template <int N>
struct IntConstant {
    static constexpr int value = N;
};

__device__ __forceinline__ uint32_t score_key(float x) {
    if (x != x) return 0u;
    x += 0.f;  // -0 -> +0
    const uint32_t u = __float_as_uint(x);
    // monotone in the float order; the smallest number (-inf) maps to 0x007fffff, above NaN's 0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// the score with the smallest key that is at least `key` (key above that of -inf)
__device__ __forceinline__ float key_score(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

// Sum of the entries of `sums` before entry `wave` (uniform). The 16 entries are scanned by the lanes of a row.
__device__ __forceinline__ int sum_before(const int* sums, int wave, int lane) {
    static_assert(SELECT_WAVES == 16, "one row of 16 lanes");
    int v = sums[lane & 15];
#define ROW_SHR_ADD(n) v += __builtin_amdgcn_update_dpp(0, v, 0x110 + (n), 0xf, 0xf, false);
    ROW_SHR_ADD(1)
    ROW_SHR_ADD(2)
    ROW_SHR_ADD(4)
    ROW_SHR_ADD(8)
#undef ROW_SHR_ADD
    const int before = __builtin_amdgcn_readlane(v, wave == 0 ? 0 : wave - 1);
    return wave == 0 ? 0 : before;
}

constexpr int DIGIT_BINS = 2048;    // the digits of a key are 11, 11 and 10 bits
constexpr int SAMPLE_BITS = 12;     // of the histogram of the sample
constexpr int MAX_CANDIDATES = 6144;
constexpr int MAX_FILTER_WANT = 3072;   // (1.5 times it and the margin of the sample stay below MAX_CANDIDATES)
constexpr int MAX_FILTER_ROW = 262144;  // entries the two bitmaps of the filter can be made for

// Of a word of 32 or 64 flags keep the `take` lowest that are set (take < number set)
template <typename Word>
__device__ __forceinline__ Word lowest_set(Word w, int take) {
    int low = 0;  // the most bits of the word that hold at most `take` flags
#pragma unroll
    for (int step = 4 * sizeof(Word); step >= 1; step >>= 1)
        if (__popcll(w & (((Word)1 << (low + step)) - 1)) <= take) low += step;
    return w & (((Word)1 << low) - 1);
}

// Adds N words of 64 bins to a histogram of COPIES interleaved copies. LDS does additions to one address one after the
// other, so that where the bin of lane 0 or 32 of the first word is that of more than 16 of its lanes (of a masked row
// one of the two may hold an entry that is not masked), that bin and one of those left over are added as one number each.
template <int N, int COPIES>
__device__ __forceinline__ void count_words(int* hist, const uint32_t (&bin)[N], int lane) {
    const unsigned long long same0 = __ballot(bin[0] == (uint32_t)__builtin_amdgcn_readlane(bin[0], 0));
    const unsigned long long same32 = __ballot(bin[0] == (uint32_t)__builtin_amdgcn_readlane(bin[0], 32));
    bool on[N];
#pragma unroll
    for (int j = 0; j < N; ++j) on[j] = true;
    if (__popcll(same0) > 16 || __popcll(same32) > 16) {
        unsigned long long same = __popcll(same0) > 16 ? same0 : same32;
        const unsigned long long rest = ~same;
        for (int probe = 0; probe < 2; ++probe) {
            const uint32_t b = __builtin_amdgcn_readlane(bin[0], __builtin_ctzll(same));
            int n = 0;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const bool add = on[j] && bin[j] == b;
                n += __popcll(__ballot(add));
                on[j] = on[j] && !add;
            }
            if (lane == 0) atomicAdd(&hist[b * COPIES], n);
            if (n == 64 * N) return;
            if (rest == 0ull) break;
            same = rest;
        }
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
        if (on[j]) atomicAdd(&hist[bin[j] * COPIES + (lane & (COPIES - 1))], 1);
}

// P words of 64 entries per wavefront; the row is taken in chunks of CHUNK = 1024 * P entries. RESIDENT: one chunk
// holds the whole row and stays in registers; else the row is read again by every step.
template <int P, bool RESIDENT>
__global__ __launch_bounds__(SELECT_THREADS) void topk_select_kernel(
    const float* __restrict__ scores, const int* __restrict__ lengths, int* __restrict__ idx_out,
    int n, int k) {
    constexpr int CHUNK = SELECT_THREADS * P;
    constexpr int GROUP = P < 8 ? P : 8;  // words handled under one test of the row's end
    constexpr bool FILTER = P >= 16;
    constexpr int HIST_COPIES = FILTER ? 2 : 4;  // of the first digit's histogram
    __shared__ __attribute__((aligned(16))) int s_hist[DIGIT_BINS * HIST_COPIES];  // [bin][copy]
    // (without the filter there is room to give the later digits histograms of their own, cleared with the first: a
    // barrier and a clear less for each)
    __shared__ __attribute__((aligned(16))) int s_hist_later[FILTER ? 4 : 2 * DIGIT_BINS];
    __shared__ int s_wave_sum[2][SELECT_WAVES];
    __shared__ int s_bin, s_above, s_in_bin, s_count, s_near_count, s_differ;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x;
    const float* row = scores + (size_t)b * n;
    int valid = lengths != nullptr ? lengths[b] : n;
    valid = valid < 0 ? 0 : (valid > n ? n : valid);
    const int want = k < valid ? k : valid;  // entries that will be chosen
    int* dst = idx_out + (size_t)b * k;
    for (int j = want + tid; j < k; j += SELECT_THREADS) dst[j] = -1;
    if (want == 0) return;

    // Word j of this wavefront in chunk c: entries first + 64*j .. first + 64*j + 63, one per lane, with
    // first = c*CHUNK + span. `left` entries of the wavefront's span exist (uniform); lanes past the end hold NaN. A row in
    // registers is dealt out in as many words (whole groups) per wavefront as it needs, not P: of rows that are shorter
    // than the kernel's CHUNK, by their lengths or because n lies above a power of two, the first wavefronts would have all
    // (us: 24 rows of 33024 with 8250 to 33024 valid entries 12.1 -> 10.4, in few values 23.2 -> 19.8; one row of 40000 12.3 ->
    // 10.6; 200 of 10000 10.6 -> 10.3).
    const int per_wave = RESIDENT ? GROUP * ((valid + SELECT_THREADS * GROUP - 1) / (SELECT_THREADS * GROUP)) : P;
    const int span = wave * 64 * per_wave;
    auto left_from = [&](int c0) {
        const int left = valid - c0 - span;
        return RESIDENT && left > 64 * per_wave ? 64 * per_wave : left;
    };
    auto load_chunk = [&](float (&val)[P], int first, int left) {
        const float* src = row + first;
        if (left >= 64 * P) {
#pragma unroll
            for (int j = 0; j < P; ++j) val[j] = src[64 * j + lane];
        } else {
#pragma unroll
            for (int g = 0; g < P; g += GROUP) {
#pragma unroll
                for (int j = g; j < g + GROUP; ++j) val[j] = __builtin_nanf("");
                if (64 * (g + GROUP) <= left) {
#pragma unroll
                    for (int j = g; j < g + GROUP; ++j) val[j] = src[64 * j + lane];
                } else if (64 * g < left) {
#pragma unroll
                    for (int j = g; j < g + GROUP; ++j) {
                        const int i = 64 * j + lane;
                        const float v = src[i < left ? i : 0];
                        val[j] = i < left ? v : __builtin_nanf("");
                    }
                }
            }
        }
    };
    // f(g) for the groups of words g .. g + GROUP - 1 of the span that hold entries of the row
    auto for_groups = [&](int left, auto f) {
#pragma unroll
        for (int g = 0; g < P; g += GROUP)
            if (64 * g < left) f(g);
    };
    auto clear_hist = [&](int* hist, int words) {
        for (int i = tid; i < words / 4; i += SELECT_THREADS) reinterpret_cast<int4*>(hist)[i] = make_int4(0, 0, 0, 0);
    };
    // In the histogram of 2^BITS bins x COPIES: the bin in which the rank-th largest key lies (counting from the top
    // bin down), the keys in bins above it and in it; s_bin as it was if there are fewer than `rank` keys.
    auto find_bin = [&](const int* hist, auto bits_tag, auto copies_tag, int rank, int& bin, int& above_bin, int& in_bin) {
        constexpr int BINS = 1 << decltype(bits_tag)::value;
        constexpr int COPIES = decltype(copies_tag)::value;
        constexpr int PER = BINS / SELECT_THREADS;  // bins of a lane
        __syncthreads();  // the counts are complete
        int c[PER];
        int mine = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            c[j] = 0;
#pragma unroll
            for (int h = 0; h < COPIES; ++h) c[j] += hist[(BINS - 1 - (PER * tid + j)) * COPIES + h];
            mine += c[j];
        }
        const int upto = lanes::inclusive_sum(mine, lane);
        if (lane == 63) s_wave_sum[0][wave] = upto;
        __syncthreads();
        int above = upto - mine + sum_before(s_wave_sum[0], wave, lane);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            if (above < rank && above + c[j] >= rank) {  // one bin of the workgroup
                s_bin = BINS - 1 - (PER * tid + j);
                s_above = above;
                s_in_bin = c[j];
            }
            above += c[j];
        }
        __syncthreads();
        bin = s_bin, above_bin = s_above, in_bin = s_in_bin;
    };
    // The want-th largest key (`threshold`) and how many of the keys equal to it are chosen, most significant digit
    // first; if all keys of a digit's bin are wanted the digits below do not matter and the threshold is the bin's
    // lowest key. first(hist) adds all keys to the histogram of the upper 11 bits, later(hist, threshold, shift, above)
    // those that are threshold from bit `above` up to that of the bits from `shift` up. one_key(threshold): whether all
    // keys of the first digit's bin are the same, and if so that key; asked where the bin is so full that they may be
    // (masked entries, rows of a few values): additions to one address are done one after the other, so that two more
    // digits over 8192 masked entries took 12 us. Not expected, to keep its code out of the others' way: a workgroup
    // alone on its CU waits for the instructions it fetches, and a few dozen more in line cost 5 % of a short row.
    auto radix_select = [&](auto copies_tag, auto first, auto later, auto one_key, uint32_t& threshold, int& need_eq) {
        clear_hist(s_hist, DIGIT_BINS * decltype(copies_tag)::value);
        if constexpr (!FILTER) clear_hist(s_hist_later, 2 * DIGIT_BINS);
        if (tid == 0) s_differ = 0;
        __syncthreads();
        first(s_hist);
        int bin, above, in_bin;
        find_bin(s_hist, IntConstant<11>{}, copies_tag, want, bin, above, in_bin);
        threshold = (uint32_t)bin << 21;
        int remaining = want - above;
        if (__builtin_expect(in_bin != remaining && in_bin >= valid / 4, 0) && one_key(threshold)) {
            need_eq = remaining;
            return;
        }
#pragma unroll
        for (int shift = 10; in_bin != remaining && shift >= 0; shift -= 10) {
            int* hist = FILTER ? s_hist : s_hist_later + (shift == 10 ? 0 : DIGIT_BINS);
            if constexpr (FILTER) {
                clear_hist(hist, DIGIT_BINS);
                __syncthreads();
            }
            later(hist, threshold, shift, shift == 10 ? 21 : 10);
            find_bin(hist, IntConstant<11>{}, IntConstant<1>{}, remaining, bin, above, in_bin);
            threshold |= (uint32_t)bin << shift;
            remaining -= above;
        }
        need_eq = in_bin == remaining ? valid : remaining;
    };

    float val[P];
    if (RESIDENT) load_chunk(val, span, left_from(0));

    if constexpr (FILTER) {
        constexpr int BITMAP = (RESIDENT ? CHUNK : MAX_FILTER_ROW) / 32;
        __shared__ uint2 s_list[MAX_CANDIDATES];  // (score bits, index), in no particular order
        __shared__ uint32_t s_gt[BITMAP], s_eq[BITMAP];
        if (want <= MAX_FILTER_WANT && want < valid && (RESIDENT || valid <= MAX_FILTER_ROW)) {
            // An eighth of the row, spread evenly: lane l takes word g + l % 8 of every group of words.
            clear_hist(s_hist, 1 << SAMPLE_BITS);
            if (tid == 0) s_count = s_near_count = 0, s_bin = -1;
            const int words = (valid + 31) / 32;
            for (int i = tid; i < words; i += SELECT_THREADS) s_gt[i] = s_eq[i] = 0u;
            __syncthreads();
            for (int c0 = 0; c0 < valid; c0 += CHUNK) {
                const int left = left_from(c0);
                if constexpr (RESIDENT) {
                    for_groups(left, [&](int g) {
                        float v = val[g];
#pragma unroll
                        for (int j = 1; j < 8; ++j) {
                            v = (lane & 7) == j ? val[g + j] : v;
                            asm("" : "+v"(v));  // (a chain of selects, not an array in memory with an index)
                        }
                        if (v == v) atomicAdd(&s_hist[score_key(v) >> (32 - SAMPLE_BITS)], 1);
                    });
                    break;
                } else {
                    float v[P / 8];
#pragma unroll
                    for (int g = 0; g < P; g += 8) {
                        const int i = 64 * (g + (lane & 7)) + lane;
                        v[g / 8] = i < left ? row[c0 + span + i] : __builtin_nanf("");
                    }
#pragma unroll
                    for (int g = 0; g < P / 8; ++g)
                        if (v[g] == v[g]) atomicAdd(&s_hist[score_key(v[g]) >> (32 - SAMPLE_BITS)], 1);
                }
            }
            // The pivot: the rank in the sample that leaves half as many entries again as are wanted, plus four
            // standard deviations of an independent sample and a few.
            const float expect = 0.125f * (float)want;
            const int rank = (int)(1.5f * expect + 4.f * __builtin_sqrtf(expect)) + 16;
            int bin, above, in_bin;
            find_bin(s_hist, IntConstant<SAMPLE_BITS>{}, IntConstant<1>{}, rank, bin, above, in_bin);
            const uint32_t pivot_key = (uint32_t)bin << (32 - SAMPLE_BITS);
            // (a number: NaN and -inf are below it; and no list that is sure to be too long, as of rows of few values)
            if (bin > 0 && pivot_key > 0x007fffffu && 8 * (above + in_bin) <= MAX_CANDIDATES + 1024) {
                const float pivot = key_score(pivot_key);
                // (a lane appends its own entries one after the other: what a word costs is VALU time, of which one CU
                // has 64 lanes a clock)
                auto collect = [&](const float (&v)[P], int first, int left) {
                    int mine = 0;
                    for_groups(left, [&](int g) {
#pragma unroll
                        for (int j = g; j < g + GROUP; ++j) mine += v[j] >= pivot ? 1 : 0;
                    });
                    const int upto = lanes::inclusive_sum(mine, lane);
                    const int total = __builtin_amdgcn_readlane(upto, 63);
                    if (total == 0) return;
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&s_count, total);
                    at = __builtin_amdgcn_readfirstlane(at);
                    if (at + total > MAX_CANDIDATES) return;  // (the count says that the list is not complete)
                    uint2* to = s_list + at + upto - mine;
                    const uint32_t index = (uint32_t)(first + lane);
                    for_groups(left, [&](int g) {
#pragma unroll
                        for (int j = g; j < g + GROUP; ++j) {
                            if (v[j] >= pivot) {
                                *to = make_uint2(__float_as_uint(v[j]), index + 64u * j);
                                ++to;
                            }
                        }
                    });
                };
                if constexpr (RESIDENT) {
                    collect(val, span, left_from(0));
                } else {
                    float next[P];
                    load_chunk(val, span, valid - span);
                    for (int c0 = 0; c0 < valid; c0 += CHUNK) {
                        const int c1 = c0 + CHUNK;
                        if (c1 < valid) load_chunk(next, c1 + span, valid - c1 - span);
                        collect(val, c0 + span, valid - c0 - span);
#pragma unroll
                        for (int j = 0; j < P; ++j) val[j] = next[j];
                    }
                }
                __syncthreads();
                const int count = s_count;
                if (count >= want && count <= MAX_CANDIDATES) {
                    constexpr int PER = MAX_CANDIDATES / SELECT_THREADS;
                    uint32_t lkey[PER], lidx[PER];
#pragma unroll
                    for (int r = 0; r < PER; ++r) {
                        lkey[r] = lidx[r] = 0u;  // (key 0 is below every candidate's)
                        const int i = tid + r * SELECT_THREADS;
                        if (i < count) {
                            const uint2 e = s_list[i];
                            lkey[r] = score_key(__uint_as_float(e.x));
                            lidx[r] = e.y;
                        }
                    }
                    // The threshold among the candidates. Keys are counted by their distance from the pivot, 2^13 keys to
                    // a bin (1/1024 of an octave): few share a bin, and those of the threshold's bin, if at most 64, are
                    // sorted out bit by bit by one wavefront. A threshold four octaves above the pivot lands in
                    // the last bin with everything beyond it: then digit by digit.
                    constexpr int NEAR_BITS = 13;
                    auto near_bin = [&](uint32_t x) {
                        const uint32_t d = (x - pivot_key) >> NEAR_BITS;
                        return d < (1u << SAMPLE_BITS) ? d : (1u << SAMPLE_BITS) - 1u;
                    };
                    uint32_t threshold = 0u;
                    int need_eq = valid;
                    clear_hist(s_hist, 1 << SAMPLE_BITS);
                    __syncthreads();
#pragma unroll
                    for (int r = 0; r < PER; ++r)
                        if (lkey[r] != 0u) atomicAdd(&s_hist[near_bin(lkey[r])], 1);
                    int tbin, tabove, tin;
                    find_bin(s_hist, IntConstant<SAMPLE_BITS>{}, IntConstant<1>{}, want, tbin, tabove, tin);
                    if (tin == want - tabove) {
                        threshold = pivot_key + ((uint32_t)tbin << NEAR_BITS);
                    } else if (tin <= 64 && tbin < (1 << SAMPLE_BITS) - 1) {
#pragma unroll
                        for (int r = 0; r < PER; ++r)
                            if (lkey[r] != 0u && near_bin(lkey[r]) == (uint32_t)tbin)
                                s_hist[atomicAdd(&s_near_count, 1)] = (int)(lkey[r] - pivot_key);
                        __syncthreads();
                        if (wave == 0) {
                            const uint32_t x = lane < tin ? (uint32_t)s_hist[lane] : 0u;
                            unsigned long long alive = tin == 64 ? ~0ull : (1ull << tin) - 1ull;
                            int remaining = want - tabove;
                            uint32_t t = (uint32_t)tbin << NEAR_BITS;
#pragma unroll
                            for (int bit = NEAR_BITS - 1; bit >= 0; --bit) {
                                const unsigned long long ones = alive & __ballot((x >> bit) & 1u);
                                const int n_ones = __popcll(ones);
                                if (n_ones >= remaining) {
                                    alive = ones;
                                    t |= 1u << bit;
                                } else {
                                    alive &= ~ones;
                                    remaining -= n_ones;
                                }
                            }
                            if (lane == 0) s_bin = (int)(pivot_key + t), s_above = remaining;
                        }
                        __syncthreads();
                        threshold = (uint32_t)s_bin;
                        need_eq = s_above;
                    } else {
                        // Rows of few values have many equal keys there (not in the last bin, with everything beyond it).
                        bool differs = tbin == (1 << SAMPLE_BITS) - 1;
                        if (!differs) {
#pragma unroll
                            for (int r = 0; r < PER; ++r)
                                if (lkey[r] != 0u && near_bin(lkey[r]) == (uint32_t)tbin) s_hist[0] = (int)lkey[r];
                            __syncthreads();  // (the counts have been read: any of the bin's keys)
                            threshold = (uint32_t)s_hist[0];
                            need_eq = want - tabove;
#pragma unroll
                            for (int r = 0; r < PER; ++r)
                                differs = differs || (lkey[r] != 0u && near_bin(lkey[r]) == (uint32_t)tbin && lkey[r] != threshold);
                            if (__ballot(differs) != 0ull && lane == 0) s_near_count = 1;
                            __syncthreads();
                            differs = s_near_count != 0;
                        }
                        if (differs) {
                            radix_select(IntConstant<1>{}, [&](int* hist) {
#pragma unroll
                                for (int r = 0; r < PER; ++r)
                                    if (lkey[r] != 0u) atomicAdd(&hist[lkey[r] >> 21], 1);
                            }, [&](int* hist, uint32_t prefix, int shift, int above) {
                                const uint32_t mask = (1u << (above - shift)) - 1u;
#pragma unroll
                                for (int r = 0; r < PER; ++r)
                                    if (lkey[r] != 0u && (lkey[r] ^ prefix) >> above == 0u) atomicAdd(&hist[(lkey[r] >> shift) & mask], 1);
                            }, [](uint32_t&) { return false; }, threshold, need_eq);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < PER; ++r) {
                        const uint32_t flag = 1u << (lidx[r] & 31);
                        if (lkey[r] > threshold) atomicOr(&s_gt[lidx[r] >> 5], flag);
                        if (lkey[r] == threshold) atomicOr(&s_eq[lidx[r] >> 5], flag);
                    }
                    __syncthreads();
                    // the words of a lane are consecutive; their places come from a workgroup-wide scan
                    const int per = (words + SELECT_THREADS - 1) / SELECT_THREADS;
                    const int w0 = tid * per, w1 = w0 + per < words ? w0 + per : words;
                    int n_gt = 0, n_eq = 0;
                    for (int w = w0; w < w1; ++w) n_gt += __popc(s_gt[w]), n_eq += __popc(s_eq[w]);
                    // (at most MAX_CANDIDATES of either: one scan of the packed pair)
                    const int upto = lanes::inclusive_sum(n_gt | (n_eq << 16), lane);
                    if (lane == 63) s_wave_sum[0][wave] = upto;
                    __syncthreads();
                    const int before = upto - (n_gt | (n_eq << 16)) + sum_before(s_wave_sum[0], wave, lane);
                    int gt_at = before & 0xffff, eq_at = before >> 16;
                    for (int w = w0; w < w1; ++w) {
                        uint32_t word = s_gt[w], ties = s_eq[w];
                        int at = gt_at + (eq_at < need_eq ? eq_at : need_eq);
                        gt_at += __popc(word);
                        const int n_ties = __popc(ties), take = need_eq > eq_at ? need_eq - eq_at : 0;
                        eq_at += n_ties;
                        if (take < n_ties) ties = lowest_set(ties, take);
                        for (word |= ties; word != 0u; word &= word - 1u) dst[at++] = 32 * w + __builtin_ctz(word);
                    }
                    return;
                }
            }
            __syncthreads();  // the shared words are used again below
        }
    }

    // The whole row, digit by digit
    uint32_t key[P];
    auto make_keys = [&]() {
#pragma unroll
        for (int j = 0; j < P; ++j) key[j] = score_key(val[j]);
    };
    // (entries past the end hold the smallest key: they land in the lowest bin of every digit and can only be among
    // the ties of key 0, from which the emission takes entries of the row alone)
    if (RESIDENT) make_keys();
    uint32_t threshold = 0u;
    int need_eq = valid;
    if (want < valid) {
        // f(g) for the groups of words of the whole row
        auto for_row = [&](auto f) {
            for (int c0 = 0; c0 < valid; c0 += CHUNK) {
                const int left = left_from(c0);
                if constexpr (!RESIDENT) {
                    load_chunk(val, c0 + span, left);
                    make_keys();
                }
                for_groups(left, f);
                if (RESIDENT) break;
            }
        };
        radix_select(IntConstant<HIST_COPIES>{}, [&](int* hist) {
            for_row([&](int g) {
                uint32_t bin[GROUP];
#pragma unroll
                for (int j = 0; j < GROUP; ++j) bin[j] = key[g + j] >> 21;
                count_words<GROUP, HIST_COPIES>(hist, bin, lane);
            });
        }, [&](int* hist, uint32_t prefix, int shift, int above) {
            const uint32_t mask = (1u << (above - shift)) - 1u;  // (fewer than a quarter of the row, or of several keys)
            for_row([&](int g) {
#pragma unroll
                for (int j = g; j < g + GROUP; ++j)
                    if ((key[j] ^ prefix) >> above == 0u) atomicAdd(&hist[(key[j] >> shift) & mask], 1);
            });
        }, [&](uint32_t& prefix) {
            auto in_bin = [&](uint32_t x) { return (x ^ prefix) >> 21 == 0u; };
            bool any = false, differs = false;
            uint32_t mine = 0u;
            for_row([&](int g) {
#pragma unroll
                for (int j = g; j < g + GROUP; ++j) {
                    any = any || in_bin(key[j]);
                    mine = in_bin(key[j]) ? key[j] : mine;
                }
            });
            if (any) s_hist[0] = (int)mine;  // (its counts have been read: any key of the bin)
            __syncthreads();
            const uint32_t one = (uint32_t)s_hist[0];
            for_row([&](int g) {
#pragma unroll
                for (int j = g; j < g + GROUP; ++j) differs = differs || (in_bin(key[j]) && key[j] != one);
            });
            if (__ballot(differs) != 0ull && lane == 0) s_differ = 1;
            __syncthreads();
            if (s_differ != 0) return false;
            prefix = one;
            return true;
        }, threshold, need_eq);
    }

    // Emission. Lane j of a wavefront holds word j of the span as two masks (keys above / equal to the threshold);
    // a scan of their counts gives every word its place in the output.
    int gt_before = 0, eq_before = 0;  // in earlier chunks
    for (int c0 = 0; c0 < valid; c0 += CHUNK) {
        const int left = left_from(c0);
        if constexpr (!RESIDENT) {
            load_chunk(val, c0 + span, left);
            make_keys();
        }
        uint32_t gt_lo = 0u, gt_hi = 0u, eq_lo = 0u, eq_hi = 0u;
        for_groups(left, [&](int g) {
#pragma unroll
            for (int j = g; j < g + GROUP; ++j) {
                const unsigned long long gt = __ballot(key[j] > threshold);
                const unsigned long long eq = __ballot(key[j] == threshold);
                gt_lo = lane == j ? (uint32_t)gt : gt_lo;
                gt_hi = lane == j ? (uint32_t)(gt >> 32) : gt_hi;
                eq_lo = lane == j ? (uint32_t)eq : eq_lo;
                eq_hi = lane == j ? (uint32_t)(eq >> 32) : eq_hi;
            }
        });
        unsigned long long word = ((unsigned long long)gt_hi << 32) | gt_lo;
        unsigned long long ties = ((unsigned long long)eq_hi << 32) | eq_lo;
        const int in_word = left - 64 * lane;  // entries of the row in this lane's word
        ties &= in_word >= 64 ? ~0ull : in_word <= 0 ? 0ull : (1ull << in_word) - 1ull;
        const int n_gt = __popcll(word), n_eq = __popcll(ties);
        const int gt_upto = lanes::inclusive_sum(n_gt, lane), eq_upto = lanes::inclusive_sum(n_eq, lane);
        if (c0 > 0) __syncthreads();  // the sums of the chunk before have been read
        if (lane == 63) {
            s_wave_sum[0][wave] = gt_upto;
            s_wave_sum[1][wave] = eq_upto;
        }
        __syncthreads();
        int gt_at = gt_before + gt_upto - n_gt, eq_at = eq_before + eq_upto - n_eq;
#pragma unroll
        for (int w = 0; w < SELECT_WAVES; ++w) {
            const int g = s_wave_sum[0][w], e = s_wave_sum[1][w];
            gt_at += w < wave ? g : 0;
            eq_at += w < wave ? e : 0;
            gt_before += g;
            eq_before += e;
        }
        // the ties of this word that are still wanted: its lowest ones
        const int take = need_eq > eq_at ? need_eq - eq_at : 0;
        if (take < n_eq) ties = lowest_set(ties, take);
        word |= ties;
        int at = gt_at + (eq_at < need_eq ? eq_at : need_eq);
        // Words of many entries are written by all lanes together, one word after the other; where the words outnumber the
        // entries of the fullest, every lane writes its own word's.
        const unsigned long long full = __ballot(word != 0ull);
        if (P <= 8 || __ballot(__popcll(word) > __popcll(full)) != 0ull) {
#pragma unroll
            for (int j = 0; j < P; ++j) {
                if (P > 8 && !((full >> j) & 1ull)) continue;
                const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)word, j);
                const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(word >> 32), j);
                const int place = __builtin_amdgcn_readlane(at, j) + __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
                if (((((unsigned long long)hi << 32) | lo) >> lane) & 1ull) dst[place] = c0 + span + 64 * j + lane;
            }
        } else {
            const int first = c0 + span + 64 * lane;
            for (; word != 0ull; word &= word - 1ull) dst[at++] = first + __builtin_ctzll(word);
        }
        if (RESIDENT) break;
    }
}

}  // namespace

// idx_out [batch, k] int32: per request the indices of the k largest scores among the first
// lengths[b] (or n, if lengths is null) entries of scores [batch, n] fp32; ties go to the lower
// index; listed in ascending index order; -1 where fewer than k candidates exist.
// config is accepted for the launcher pattern and has one value.
extern "C" void topk_select_launcher(int* idx_out, const float* scores, const int* lengths,
                                     int batch, int n, int k, int config, hipStream_t stream) {
    (void)config;
    if (batch <= 0 || k <= 0) return;
    if (n <= 0) {
        caa::set_status(CAA_UNSUPPORTED_SHAPE);
        return;
    }
    if (!idx_out || !scores) {
        caa::set_status(CAA_BAD_ARGUMENT);
        return;
    }
#define TOPK_LAUNCH(P, RESIDENT) \
    topk_select_kernel<P, RESIDENT><<<batch, SELECT_THREADS, 0, stream>>>(scores, lengths, idx_out, n, k)
    if (n <= 4 * SELECT_THREADS) {
        TOPK_LAUNCH(4, true);
    } else if (n <= 8 * SELECT_THREADS) {
        TOPK_LAUNCH(8, true);
    } else if (n <= 16 * SELECT_THREADS) {
        TOPK_LAUNCH(16, true);
    } else if (n <= 32 * SELECT_THREADS) {
        TOPK_LAUNCH(32, true);
    } else if (n <= 64 * SELECT_THREADS) {
        TOPK_LAUNCH(64, true);
    } else {
        TOPK_LAUNCH(32, false);
    }
#undef TOPK_LAUNCH
}
