// Int8 attention without scores in memory: one launch takes every (image, head)'s queries through
// the scores, the exponentials, their quantization and the weighted values (attention::attend,
// blocks/src/attention.rs:81-214), with the bits of the step-by-step kernels in attention.hip.
//
// A wave owns 32 queries of one head. The scores are formed transposed, keys by queries
// (v_mfma_i32_32x32x32_i8 with the keys as the first operand): lane l then holds query l % 32
// against keys 8j + 4(l / 32) + i of a block of 32 keys, j and i in 0..3. That layout is what the
// rest needs:
//   * the reference adds the exponentials into eight sums by key mod 8 (scalar.rs:117-126): key
//     mod 8 is 4(l / 32) + i, so a lane's four running sums take its values in key order, one add
//     per score and no exchange until the end;
//   * a row's group of 32 weights (one quantization group) is a lane's sixteen values and its
//     partner's in the other half: one lane swap per group;
//   * the sixteen levels are the second operand of the values' product in place, as long as the
//     values are stored with their keys in the same order (an integer dot does not depend on it).
// The row's maximum comes first, from a pass that forms the scores and keeps only that: forming
// them twice costs a fifth of the arithmetic, keeping them 128 MiB of memory traffic per head
// of 4096 x 4096.
//
// The keys and values of a (image, key head) are kept as one record per block of 32 keys: key
// levels [block of channels][half][key][16], key scales [block of channels][key], value levels
// [32 channels][half][channel][16 keys in the lane's order], value scales [channel]. A workgroup
// of four waves (128 queries) brings two records at a time into LDS, double-buffered.
//
// Bound: instruction issue. Additions and multiplications take 2.4 cycles a wave with two waves on the
// SIMD, fused multiply-adds, maxima and byte permutes 4.2, so totals are converted by subtraction
// (unbiased) and exponents taken from an addition's low bits (exp_by_additions): 4096 x 4096, 16 heads of
// 72, in 342 us at its fastest dispatch and 369 on average, 365 a call with the keys' and values'
// preparation in a loop of calls (452 with conversion instructions), against 941 unit by unit. 16 queries a
// wave (16 x 16 products, four waves a SIMD) took 560 a call where 32 took 452: the same arithmetic with
// twice the instructions around it.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attention.h"
#include "common.h"
#include "proj.h"

namespace fg {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

// One record's parts, for PB blocks of 32 channels the last of which holds 8 TJ of them.
template <int PB, int TJ>
struct Record {
    static constexpr int kChannels = 32 * (PB - 1) + 8 * TJ;
    static constexpr int kKeyScales = PB * 1024;
    static constexpr int kKeyBytes = kKeyScales + PB * 128;
    static constexpr int kValues = kKeyBytes;
    static constexpr int kValueScales = kValues + kChannels * 32;
    static constexpr int kBytes = kValueScales + kChannels * 4;
};

struct FusedParams {
    const float *query, *key, *value;
    size_t query_stride, query_offset, key_stride, key_offset, value_stride, value_offset;
    int heads, kv_heads, group, queries, keys, hd, nkb;
    char *records;       // [image · kv_heads + kh][nkb] records
    float *mean;         // [image · kv_heads + kh][hd]
    float *out;
    size_t out_stride;
    int out_aligned;     // out's rows allow 16-byte stores
    int keys_aligned;    // the keys' rows allow 16-byte loads
    int tiles, items;    // query tiles per (image, head), and all of them
    float scale;
};

constexpr int kMeanThreads = 256, kMeanChannels = 16, kMeanKeys = 512;

// The keys' mean (attention.rs:104-110): per channel of an image's key row a sum over the keys in
// order. A workgroup takes 16 neighbouring channels: its waves bring 512 keys at a time into LDS, a
// thread four neighbouring keys of a channel as one 16-byte run, with the next two chunks in
// flight, and a lane of the first wave adds each channel's. The chain of additions (2.8 ns each) is
// the bound, as long as enough CUs share the reading: 4096 keys of 1152 channels 25 us in 72
// workgroups, of which the chain is 11.5 (30 us in 18 workgroups of 64 channels: about 50 GB/s a CU).
__device__ __forceinline__ void key_means(const FusedParams &p, int image, int c0)
{
    extern __shared__ __align__(16) v4f chunk[];  // [2][kMeanKeys / 4][kMeanChannels]
    constexpr int C = kMeanChannels, kSlots = kMeanThreads / C;
    constexpr int kRuns = kMeanKeys / 4 / kSlots;  // runs of four keys a thread brings of a chunk
    const int width = p.kv_heads * p.hd, channel = threadIdx.x % C, slot = threadIdx.x / C;
    const float *src = p.key + size_t(image) * size_t(p.keys) * p.key_stride + p.key_offset + min(c0 + channel, width - 1);
    float s = 0.0f;
    auto load = [&](v4f (&r)[kRuns], int k0) {
#pragma unroll
        for (int u = 0; u < kRuns; u++) {
#pragma unroll
            for (int e = 0; e < 4; e++) r[u][e] = src[size_t(min(k0 + 4 * (slot + kSlots * u) + e, p.keys - 1)) * p.key_stride];
        }
    };
    auto step = [&](v4f (&r)[kRuns], int k0, v4f *buf) {
#pragma unroll
        for (int u = 0; u < kRuns; u++) buf[(slot + kSlots * u) * C + channel] = r[u];
        __syncthreads();
        if (k0 + 2 * kMeanKeys < p.keys) load(r, k0 + 2 * kMeanKeys);
        if (threadIdx.x >= C) return;
        // runs of 32 keys in two register sets in turn: a run's reads go out before the additions of
        // the one before it
        const int n = min(kMeanKeys, p.keys - k0), runs = n / 32;
        v4f x[2][8];
        auto fetch = [&](v4f (&v)[8], int run) {
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = buf[(run * 8 + u) * C + channel];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](const v4f (&v)[8]) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
#pragma unroll
                for (int e = 0; e < 4; e++) s = s + v[u][e];
            }
        };
        if (runs > 0) fetch(x[0], 0);
        for (int run = 0; run < runs; run += 2) {
            fetch(x[1], min(run + 1, runs - 1));
            add(x[0]);
            fetch(x[0], min(run + 2, runs - 1));
            if (run + 1 < runs) add(x[1]);
        }
        for (int k = runs * 32; k < n; k++) s = s + buf[k / 4 * C + channel][k % 4];
    };
    v4f even[kRuns], odd[kRuns];
    load(even, 0);
    load(odd, kMeanKeys);
    for (int k0 = 0; k0 < p.keys; k0 += 2 * kMeanKeys) {
        step(even, k0, chunk);
        if (k0 + kMeanKeys < p.keys) step(odd, k0 + kMeanKeys, chunk + kMeanKeys / 4 * C);
    }
    if (slot == 0 && c0 + channel < width) p.mean[size_t(image) * width + c0 + channel] = s / float(p.keys);
}

// The values' half of the records (Scratch::transpose, attention.rs:119-137): one thread per
// (table, block of keys, channel), the channel's 32 keys quantized as one Q7b32 block, channels
// fastest so neighbouring threads read neighbouring values.
template <int PB, int TJ>
__device__ __forceinline__ void value_record(const FusedParams &p, unsigned id, unsigned n)
{
    using R = Record<PB, TJ>;
    if (id >= n) return;
    const unsigned c = id % unsigned(R::kChannels), tb = id / unsigned(R::kChannels);
    const unsigned kb = tb % unsigned(p.nkb), t = tb / unsigned(p.nkb);
    const unsigned image = t / unsigned(p.kv_heads), kh = t % unsigned(p.kv_heads);
    char *rec = p.records + size_t(tb) * R::kBytes;
    const int tile = int(c) / 32, row = int(c) % 32, rows = tile == PB - 1 ? 8 * TJ : 32;
    int4 *dst = reinterpret_cast<int4 *>(rec + R::kValues + tile * 1024);
    float *scale = reinterpret_cast<float *>(rec + R::kValueScales) + c;
    if (int(c) >= p.hd) {
        dst[row] = dst[rows + row] = make_int4(0, 0, 0, 0);
        *scale = 0.0f;
        return;
    }
    const float *src = p.value + size_t(image) * unsigned(p.keys) * p.value_stride + p.value_offset + size_t(kh) * p.hd + c;
    float x[32];
#pragma unroll
    for (int i = 0; i < 32; i++) {
        const int k = 32 * int(kb) + i;
        x[i] = k < p.keys ? src[size_t(k) * p.value_stride] : 0.0f;
    }
    int w[8];
    *scale = q7_block(x, w);
    dst[row] = make_int4(w[0], w[2], w[4], w[6]);          // keys 8j + 0..3
    dst[rows + row] = make_int4(w[1], w[3], w[5], w[7]);   // keys 8j + 4..7
}

// The keys' means and, in the workgroups after theirs, the values' halves of the records: neither
// needs the other, and the means are a few workgroups' chains of additions.
template <int PB, int TJ>
__global__ __launch_bounds__(kMeanThreads) void mean_and_values_kernel(FusedParams p, int mean_blocks, int mean_groups,
                                                                       unsigned values)
{
    const int b = int(blockIdx.x);
    if (b < mean_blocks) {
        key_means(p, b / mean_groups, b % mean_groups * kMeanChannels);
        return;
    }
    value_record<PB, TJ>(p, unsigned(b - mean_blocks) * kMeanThreads + threadIdx.x, values);
}

// The keys' half of the records (attention.rs:110-118): each key less the mean as Q7b32 blocks,
// zeros past the channels; keys past the last are zero levels with a zero scale. Eight lanes per
// (table, key, block of channels), four channels each.
template <int PB, int TJ>
__global__ __launch_bounds__(256) void key_record_kernel(FusedParams p, unsigned groups)
{
    using R = Record<PB, TJ>;
    const unsigned lid = blockIdx.x * 256u + threadIdx.x, sub = lid & 7u;
    const unsigned g = min(lid >> 3, groups - 1);  // past the end: the last group again, never stored
    const unsigned key = g % 32u, b = g / 32u % unsigned(PB), tb = g / (32u * PB);  // eight keys of a block per wave
    const unsigned t = tb / unsigned(p.nkb), row = (tb - t * unsigned(p.nkb)) * 32u + key;
    const unsigned image = t / unsigned(p.kv_heads), kh = t % unsigned(p.kv_heads);
    const bool live = int(row) < p.keys;
    const float *src = p.key + (size_t(image) * unsigned(p.keys) + min(int(row), p.keys - 1)) * p.key_stride + p.key_offset +
                       size_t(kh) * p.hd;
    const float *mu = p.mean + size_t(t) * p.hd;
    const int d0 = 32 * int(b) + 4 * int(sub);  // whole quads: all four channels or none
    float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (d0 < p.hd) {
        if (p.keys_aligned) {
            const v4f k = *reinterpret_cast<const v4f *>(src + d0), m = *reinterpret_cast<const v4f *>(mu + d0);
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = k[j] - m[j];
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = src[d0 + j] - mu[d0 + j];
        }
    }
    float amax = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
    amax = max8(fmaxf(0.0f, amax));
    const float d = group_scale(amax, 63.0f);
    const int packed = q7_levels4(x, d);
    if ((lid >> 3) >= groups) return;
    char *rec = p.records + size_t(tb) * R::kBytes;
    const unsigned half = sub / 4;
    *reinterpret_cast<int *>(rec + b * 1024 + (half * 32 + key) * 16 + (sub & 3) * 4) = live ? packed : 0;
    if (sub == 0) *reinterpret_cast<float *>(rec + R::kKeyScales + b * 128 + key * 4) = live ? d : 0.0f;
}

// ref_exp and ref_exp_fast by additions: that of 1.5 · 2^23 rounds to an integer, ties to even, and
// leaves it in the low bits, where rint, the conversion and the shifted sum issue at half the rate.
// Same bits; a longer chain, so not for kernels of one wave a SIMD.
template <bool FAST>
__device__ __forceinline__ float exp_by_additions(float x)
{
    x = FAST ? fmaxf(x, -87.0f) : x < -87.0f ? -87.0f : (x > 88.0f ? 88.0f : x);
    const float rounded = x * 1.44269504088896340736f + 12582912.0f;
    const float n = rounded - 12582912.0f;
    float poly;
    if (FAST) {
        const float r = __builtin_fmaf(-n, 0.693147180559945309417f, x);
        poly = 1.0f / 24.0f;
        poly = __builtin_fmaf(poly, r, 1.0f / 6.0f);
        poly = __builtin_fmaf(poly, r, 0.5f);
        poly = __builtin_fmaf(poly, r, 1.0f);
        poly = __builtin_fmaf(poly, r, 1.0f);
    } else {
        const float r = x - n * 0.6933594f - n * -2.1219444e-4f;
        poly = 1.9875691e-4f;
        poly = poly * r + 1.3981999e-3f;
        poly = poly * r + 8.333452e-3f;
        poly = poly * r + 4.1665796e-2f;
        poly = poly * r + 0.16666666f;
        poly = poly * r + 0.5f;
        poly = poly * r * r + r + 1.0f;
    }
    return poly * __uint_as_float((__float_as_uint(rounded) << 23) + 0x3F800000u);
}

// The low bytes of four dwords as one.
__device__ __forceinline__ int low_bytes(unsigned a, unsigned b, unsigned c, unsigned d)
{
    return int(__builtin_amdgcn_perm(b, a, 0x0c0c0400u) | __builtin_amdgcn_perm(d, c, 0x04000c0cu));
}

// A lane's half (16 of 32) of a quantization group of values >= 0 (or NaN): the group's largest.
__device__ __forceinline__ float group_peak(const float (&e)[16])
{
    float a = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) a = fmaxf(a, e[r]);
    const float2 h = half_pair(a);
    return fmaxf(h.x, h.y);
}
// Where the shared reciprocal gives the IEEE quotients (quantize_groups).
__device__ __forceinline__ bool in_range(float a) { return a >= 0x1p-52f && a <= 0x1p66f; }
// The group's scale and the half's sixteen levels where its largest is in range. rint and the
// conversion are one addition of 1.5 · 2^23, whose sum rounds to the quotient's nearest integer,
// ties to even, in its low bits (a NaN's low byte is the level 0).
__device__ __forceinline__ float quantize_half(float a, const float (&e)[16], v4i &levels)
{
    float c = 127.0f;
    asm("" : "+v"(c));  // the divisor's reciprocal from v_rcp_f32 at run time, as the expansion takes it
    const float d = corrected_quotient(a, c, refined_reciprocal(c));
    const float r = refined_reciprocal(d);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        unsigned l[4];
#pragma unroll
        for (int i = 0; i < 4; i++) l[i] = __float_as_uint(corrected_quotient(e[4 * j + i], d, r) + 12582912.0f);
        levels[j] = low_bytes(l[0], l[1], l[2], l[3]);
    }
    return d;
}
// ... and elsewhere, by the IEEE division
__device__ __forceinline__ float quantize_half_far(float a, const float (&e)[16], v4i &levels)
{
    const float d = a == 0.0f ? 1.0f : a / 127.0f;
#pragma unroll
    for (int j = 0; j < 4; j++)
        levels[j] = pack4(level_of(e[4 * j] / d), level_of(e[4 * j + 1] / d), level_of(e[4 * j + 2] / d),
                          level_of(e[4 * j + 3] / d));
    return d;
}

template <int PB, int TJ, bool FAST>
__global__ __launch_bounds__(256, 2) void attend_fused_kernel(FusedParams p)
{
    using R = Record<PB, TJ>;
    constexpr int kRounds = (2 * R::kBytes / 16 + 255) / 256;
    __shared__ __align__(16) char buffers[2][2 * R::kBytes];
    // workgroup i runs on XCD i % 8: each XCD takes a contiguous run of (image, head) query tiles,
    // so a head's records are read through few L2s
    const int band = (p.items + 7) / 8, item = int(blockIdx.x & 7u) * band + int(blockIdx.x >> 3);
    if (item >= p.items) return;
    const int u = item / p.tiles, tile = item - u * p.tiles;
    const int image = u / p.heads, head = u - image * p.heads, t = image * p.kv_heads + head / p.group;
    const int tid = int(threadIdx.x), lane = tid & 63, l31 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q0 = tile * 128 + wave * 32;
    const bool active = q0 < p.queries;
    const int query = min(q0 + l31, p.queries - 1);
    const char *records = p.records + size_t(t) * p.nkb * R::kBytes;

    // the query's levels: this lane's sixteen channels of each block
    v4i ql[PB];
    float qs[PB];
    {
        const float *row = p.query + (size_t(image) * p.queries + query) * p.query_stride + p.query_offset + size_t(head) * p.hd;
#pragma unroll
        for (int b = 0; b < PB; b++) {
            float x[16], a = 0.0f;
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const int c = 32 * b + 16 * half + k;
                x[k] = c < p.hd ? row[c] : 0.0f;
                a = fmaxf(a, fabsf(x[k]));
            }
            const float2 h = half_pair(a);
            const float d = group_scale(fmaxf(h.x, h.y), 127.0f);
            qs[b] = d;
#pragma unroll
            for (int j = 0; j < 4; j++)
                ql[b][j] = pack4(quantize_level(x[4 * j], d), quantize_level(x[4 * j + 1], d), quantize_level(x[4 * j + 2], d),
                                 quantize_level(x[4 * j + 3], d));
        }
    }

    // two records (their first `bytes` bytes) from global memory to registers, then to LDS
    v4i staged[kRounds];
    auto load = [&](int stage, int bytes) {
        const int per = bytes / 16;
#pragma unroll
        for (int r = 0; r < kRounds; r++) {
            const int i = min(tid + 256 * r, 2 * per - 1), second = i >= per;
            const int kb = min(2 * stage + second, p.nkb - 1);
            staged[r] = reinterpret_cast<const v4i *>(records + size_t(kb) * R::kBytes)[i - second * per];
        }
    };
    auto store = [&](int at, int bytes) {
        const int per = bytes / 16;
#pragma unroll
        for (int r = 0; r < kRounds; r++) {
            const int i = tid + 256 * r, second = i >= per;
            if (i < 2 * per) reinterpret_cast<v4i *>(buffers[at] + second * R::kBytes)[i - second * per] = staged[r];
        }
    };
    // both of a stage's blocks at once where their registers allow
    constexpr bool kTogether = PB < 4 && !(PB == 3 && TJ == 3);
    const v16i biased = biased_zero<v16i>();
    // N blocks' scores before their scaling, the reference's order over the channel blocks (its
    // first addition, to +0, is left out: a term of -0 gives the same exponential). The scale
    // products of two (key block, channel block) pairs come from one f32 outer product
    // (v_mfma_f32_32x32x1_2b, a lane per key and query and pair, each rounded once): one 4-byte
    // LDS read per lane where the scales in the product's layout are four of 16 bytes.
    auto scores = [&](const char *rec, auto count, auto &s) {
        constexpr int N = decltype(count)::value, F = N * PB;
        const v32f zero32 = {};
#pragma unroll
        for (int f = 0; f < F; f += 2) {
            const int g = f + 1 < F ? f + 1 : f;
            const int fo = f / PB * R::kBytes + f % PB * 128, go = g / PB * R::kBytes + g % PB * 128;
            const float ks = *reinterpret_cast<const float *>(rec + R::kKeyScales + l31 * 4 + (half ? go : fo));
            const v32f scale = __builtin_amdgcn_mfma_f32_32x32x1f32(ks, half ? qs[g % PB] : qs[f % PB], zero32, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                if (f + e >= F) break;
                const int n = (f + e) / PB, b = (f + e) % PB;
                const v4i k = *reinterpret_cast<const v4i *>(rec + n * R::kBytes + b * 1024 + lane * 16);
                const v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(k, ql[b], biased, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float term = unbiased(d[r]) * scale[16 * e + r];
                    s[n][r] = b == 0 ? term : s[n][r] + term;
                }
            }
        }
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    const int pairs = p.keys / 64;  // stages of two whole blocks; at most one more follows
    const int stages = (p.nkb + 1) / 2;

    // the row's maximum. Scaling by a positive factor keeps the order of rounded values, so the
    // maximum is scaled instead of every score.
    float peak = -INFINITY;
    load(0, R::kKeyBytes);
    for (int st = 0; st < stages; st++) {
        store(st & 1, R::kKeyBytes);
        __syncthreads();
        if (st + 1 < stages) load(st + 1, R::kKeyBytes);
        if (!active) continue;
        const char *buf = buffers[st & 1];
        if (st < pairs) {
            float s[2][16];
            scores(buf, Two{}, s);
#pragma unroll
            for (int r = 0; r < 16; r++) peak = fmaxf(fmaxf(peak, s[0][r]), s[1][r]);
        } else {
            for (int blk = 0; blk < 2 && 2 * st + blk < p.nkb; blk++) {
                float s[1][16];
                scores(buf + blk * R::kBytes, One{}, s);
                const int left = p.keys - 32 * (2 * st + blk);
#pragma unroll
                for (int r = 0; r < 16; r++)
                    peak = fmaxf(peak, 8 * (r / 4) + 4 * half + r % 4 < left ? s[0][r] : -INFINITY);
            }
        }
    }
    {
        const float2 h = half_pair(peak);
        peak = fmaxf(h.x, h.y) * p.scale;
    }
    __syncthreads();

    float sums[4] = {0.0f, 0.0f, 0.0f, 0.0f}, rest[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    v16f acc[PB];
#pragma unroll
    for (int c = 0; c < PB; c++) acc[c] = v16f{};
    // N blocks of keys (`left` keys from the first of them on, when MASKED): their exponentials and
    // sums, their levels, then their weighted values. The levels' rare division is one branch for
    // all of them, so that the arithmetic before and after it stays in one block each.
    auto weigh = [&](const char *rec, auto count, auto masked, int left) {
        constexpr int N = decltype(count)::value;
        constexpr bool MASKED = decltype(masked)::value;
        float s[N][16], a[N], d[N];
        v4i levels[N];
        bool fast = true;
        scores(rec, count, s);
#pragma unroll
        for (int n = 0; n < N; n++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float x = s[n][r] * p.scale - peak;
                s[n][r] = exp_by_additions<FAST>(x);
                if (MASKED && 8 * (r / 4) + 4 * half + r % 4 >= left) s[n][r] = 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (!MASKED || 8 * j + 8 <= left)
                        sums[i] = sums[i] + s[n][4 * j + i];
                    else if (8 * j < left)
                        rest[i] = s[n][4 * j + i];  // the last run, of fewer than eight keys
                }
            }
            a[n] = group_peak(s[n]);
            d[n] = quantize_half(a[n], s[n], levels[n]);
            fast = fast && in_range(a[n]);
        }
        if (!__all(fast)) {
#pragma unroll
            for (int n = 0; n < N; n++)
                if (!in_range(a[n])) d[n] = quantize_half_far(a[n], s[n], levels[n]);
        }
        // their scale products as the scores': whole tiles of 32 channels by outer products, two to
        // one, a short last tile by multiplications
        constexpr int W = TJ > 2 ? PB : PB - 1, F = N * W;
        const v32f zero32 = {};
        auto dots = [&](int n, int c) {
            const int rows = c == PB - 1 ? 8 * TJ : 32;
            const char *values = rec + n * R::kBytes + R::kValues + c * 1024;
            const v4i v = *reinterpret_cast<const v4i *>(values + (half * rows + min(l31, rows - 1)) * 16);
            return __builtin_amdgcn_mfma_i32_32x32x32_i8(v, levels[n], biased, 0, 0, 0);
        };
#pragma unroll
        for (int f = 0; f < F; f += 2) {
            const int g = f + 1 < F ? f + 1 : f;
            auto offset = [&](int x) {
                const int n = x / max(W, 1), c = x % max(W, 1);
                return n * R::kBytes + R::kValueScales + (32 * c + (c == PB - 1 ? min(l31, 8 * TJ - 1) : l31)) * 4;
            };
            const float vs = *reinterpret_cast<const float *>(rec + (half ? offset(g) : offset(f)));
            const v32f scale = __builtin_amdgcn_mfma_f32_32x32x1f32(vs, half ? d[g / max(W, 1)] : d[f / max(W, 1)], zero32, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                if (f + e >= F) break;
                const int n = (f + e) / max(W, 1), c = (f + e) % max(W, 1);
                const v16i t = dots(n, c);
#pragma unroll
                for (int r = 0; r < (c == PB - 1 ? 4 * TJ : 16); r++) acc[c][r] = acc[c][r] + unbiased(t[r]) * scale[16 * e + r];
            }
        }
        if (W < PB) {
#pragma unroll
            for (int n = 0; n < N; n++) {
                const v16i t = dots(n, PB - 1);
#pragma unroll
                for (int j = 0; j < TJ; j++) {
                    const v4f vs = *reinterpret_cast<const v4f *>(rec + n * R::kBytes + R::kValueScales + (32 * (PB - 1) + 8 * j + 4 * half) * 4);
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[PB - 1][4 * j + i] = acc[PB - 1][4 * j + i] + unbiased(t[4 * j + i]) * (vs[i] * d[n]);
                }
            }
        }
    };
    load(0, R::kBytes);
    for (int st = 0; st < stages; st++) {
        store(st & 1, R::kBytes);
        __syncthreads();
        if (st + 1 < stages) load(st + 1, R::kBytes);
        if (!active) continue;
        const char *buf = buffers[st & 1];
        if (st < pairs) {
            if (kTogether) {
                weigh(buf, Two{}, std::false_type{}, 64);
            } else {
#pragma unroll 1
                for (int blk = 0; blk < 2; blk++) weigh(buf + blk * R::kBytes, One{}, std::false_type{}, 32);
            }
        } else {
            for (int blk = 0; blk < 2 && 2 * st + blk < p.nkb; blk++)
                weigh(buf + blk * R::kBytes, One{}, std::true_type{}, p.keys - 32 * (2 * st + blk));
        }
    }

    // the row's total: the keys past the whole runs of eight in order, then the eight sums in order
    float total = -0.0f;
    float lo[8], hi[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float2 r = half_pair(rest[i]), s = half_pair(sums[i]);
        lo[i] = r.x;
        lo[4 + i] = r.y;
        hi[i] = s.x;
        hi[4 + i] = s.y;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) total = total + lo[i];
#pragma unroll
    for (int i = 0; i < 8; i++) total = total + hi[i];
    if (q0 + l31 >= p.queries) return;
    float *row = p.out + (size_t(image) * p.queries + query) * p.out_stride + size_t(head) * p.hd;
#pragma unroll
    for (int c = 0; c < PB; c++) {
#pragma unroll
        for (int j = 0; j < (c == PB - 1 ? TJ : 4); j++) {
            const int first = 32 * c + 8 * j + 4 * half;  // whole quads: all four channels or none
            if (first < p.hd) {
                v4f o;
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = acc[c][4 * j + i] / total;
                if (p.out_aligned) {
                    *reinterpret_cast<v4f *>(row + first) = o;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++) row[first + i] = o[i];
                }
            }
        }
    }
}

template <int PB, int TJ>
int launch_as(FusedParams p, int images, bool fast, hipStream_t s)
{
    using R = Record<PB, TJ>;
    const int tables = images * p.kv_heads;
    const int groups = (p.kv_heads * p.hd + kMeanChannels - 1) / kMeanChannels, means = images * groups;
    const unsigned values = unsigned(tables) * unsigned(p.nkb) * unsigned(R::kChannels);
    const size_t lds = size_t(2) * kMeanKeys * kMeanChannels * 4;
    mean_and_values_kernel<PB, TJ><<<unsigned(means) + (values + kMeanThreads - 1) / kMeanThreads, kMeanThreads, lds, s>>>(
        p, means, groups, values);
    FG_HIP(hipGetLastError());
    const unsigned kgroups = unsigned(tables) * unsigned(p.nkb) * 32u * unsigned(PB);
    key_record_kernel<PB, TJ><<<(kgroups + 31) / 32, 256, 0, s>>>(p, kgroups);
    FG_HIP(hipGetLastError());
    const unsigned grid = unsigned((p.items + 7) / 8) * 8;
    if (fast)
        attend_fused_kernel<PB, TJ, true><<<grid, 256, 0, s>>>(p);
    else
        attend_fused_kernel<PB, TJ, false><<<grid, 256, 0, s>>>(p);
    FG_HIP(hipGetLastError());
    return FG_OK;
}

template <int PB>
int launch_tail(const FusedParams &p, int tail, int images, bool fast, hipStream_t s)
{
    switch (tail) {
    case 1: return launch_as<PB, 1>(p, images, fast, s);
    case 2: return launch_as<PB, 2>(p, images, fast, s);
    case 3: return launch_as<PB, 3>(p, images, fast, s);
    default: return launch_as<PB, 4>(p, images, fast, s);
    }
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }
size_t record_bytes(const fg_attention *c)
{
    const size_t pb = (c->head_dim + 31) / 32, channels = (c->head_dim + 7) / 8 * 8;
    return pb * 1152 + channels * 36;
}

}  // namespace

size_t attend_fused_bytes(const fg_attention *c)
{
    const size_t tables = c->images * c->kv_heads;
    return align256(tables * ((c->keys + 31) / 32) * record_bytes(c)) + align256(tables * c->head_dim * 4);
}

int launch_attend_fused(const fg_attention *c, float *out, void *workspace, hipStream_t s)
{
    FusedParams p{};
    p.query = c->query;
    p.key = c->key;
    p.value = c->value;
    p.query_stride = c->query_stride;
    p.query_offset = c->query_offset;
    p.key_stride = c->key_stride;
    p.key_offset = c->key_offset;
    p.value_stride = c->value_stride;
    p.value_offset = c->value_offset;
    p.heads = int(c->heads);
    p.kv_heads = int(c->kv_heads);
    p.group = int(c->heads / c->kv_heads);
    p.queries = int(c->queries);
    p.keys = int(c->keys);
    p.hd = int(c->head_dim);
    p.nkb = int((c->keys + 31) / 32);
    p.records = static_cast<char *>(workspace);
    p.mean = reinterpret_cast<float *>(p.records + align256(c->images * c->kv_heads * size_t(p.nkb) * record_bytes(c)));
    p.out = out;
    p.out_stride = c->heads * c->head_dim;
    p.out_aligned = reinterpret_cast<uintptr_t>(out) % 16 == 0;  // head_dim is whole quads
    p.keys_aligned = reinterpret_cast<uintptr_t>(p.key) % 16 == 0 && p.key_stride % 4 == 0 && p.key_offset % 4 == 0;
    p.tiles = (p.queries + 127) / 128;
    p.items = int(c->images * c->heads * size_t(p.tiles));
    p.scale = 1.0f / sqrtf(float(p.hd));
    const int images = int(c->images), pb = (p.hd + 31) / 32, tail = (p.hd - 32 * (pb - 1) + 7) / 8;
    const bool fast = c->exponentials == FG_EXP_FAST;
    switch (pb) {
    case 1: return launch_tail<1>(p, tail, images, fast, s);
    case 2: return launch_tail<2>(p, tail, images, fast, s);
    case 3: return launch_tail<3>(p, tail, images, fast, s);
    default: return launch_tail<4>(p, tail, images, fast, s);
    }
}

}  // namespace fg
