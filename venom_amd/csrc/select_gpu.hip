// Magnitude selector on the GPU: for every (V-row block, m-column group) the subset of 4 (3 in a three-column tail) columns that
// maximises the sum over the block's rows of the two largest magnitudes (group_n_m2 / func, end2end/grouped_nmv_tensor.py:81-343),
// and, in the same launch where four groups of a block fit the LDS, the V:N:M encoding of that choice (to_sparse_sr_nm / func2,
// :345-560; the storage map is in vnm_format.cpp).  The totals are accumulated exactly as the host code does it (fp32, row by
// row, largest then second largest, no fused operations), subsets are ranked in lexicographic order and only a strictly larger
// total replaces the best one, so the winner is the host's winner bit for bit.
//
// What bounds it: vector instructions.  A subset's total is a serial chain of 2 V additions (their order is part of the result),
// so the additions cannot be shared; everything around them can.  A lane owns a triple a < b < c of a group and runs the subsets
// {a, b, c, d > c}, up to five at a time: the two largest of the triple once per row, then per subset the two largest of three
// values (max, min, max) and the two additions.  fp16 magnitudes stay fp16: two rows per packed max / min (exact) and
// v_fma_mix_f32 with a factor of one as the addition (it widens the half it is told to and rounds once, like the fp32 addition):
// 7 instructions per subset and row pair and 5 per triple, 18 when every subset was taken by itself on fp32 magnitudes.
// Triples go in colex order (c, b, a), so the lanes of a wave have runs of nearly the same length; waves draw 64 at a time, the
// longest runs first.  Magnitudes sit in LDS column by column (16-byte reads of eight rows); columns and groups are an odd number
// of 16-byte units apart, so that sixteen lanes on sixteen groups or columns read different banks.
// Measured, search and encoding (before: fp32 magnitudes, every subset by itself, a second launch for the encoding): 4096 x 1024 at
// 64:2:8 16 us (38), 64:2:10 31 (56), 64:2:16 78 (173), 64:2:32 668 (1413); 768 x 768 at 32:2:8 7 (19), 128:2:16 46 (64).  At m = 4,
// one subset, 12 us are left: a workgroup's loads, barriers and stores.  A packed maximum and v_fma_mix_f32 take 4.8 clocks of a SIMD,
// so 64:2:16 is at 80 % of what its instructions need.  (16-byte loads and an LDS copy of the block for the encoding: level or slower.)

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <algorithm>

#include "spmm_kernels.h"

namespace spatha {

namespace {
constexpr int kMaxGroups = 32;          // groups of a workgroup, a power of two
constexpr int kThreads = 512;
constexpr int kRun = 5;                 // subsets of one triple that a lane totals at a time
constexpr size_t kLdsLimit = 150 * 1024;

// (magnitudes are canonical - `magnitude` made them so -: without the quieting instruction that fmaxf / fminf put in front of every
// operand that comes from memory)
__device__ __forceinline__ float max2(float a, float b) { float d; asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b)); return d; }
__device__ __forceinline__ float min2(float a, float b) { float d; asm("v_min_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b)); return d; }
__device__ __forceinline__ float max3(float a, float b, float c) {
    float d;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

// Magnitudes as whole numbers: without a NaN among them they are ordered alike, and the compiler sees instructions it can place (an asm
// result may not be read by the very next vector instruction: every second one had an s_nop in front).  One row of fp32, two of fp16.
typedef unsigned short Pair __attribute__((ext_vector_type(2)));
typedef _Float16 HalfPair __attribute__((ext_vector_type(2)));

// total + largest + second, row by row, for N subsets side by side; one: 1.0f that the compiler does not know, so that widening and
// addition are one v_fma_mix_f32 (rounds once, like the addition)
template <int N>
__device__ __forceinline__ void add_rows(float (&total)[N], const uint32_t (&largest)[N], const uint32_t (&second)[N], float) {
#pragma unroll
    for (int k = 0; k < N; k++) total[k] = __fadd_rn(total[k], __builtin_bit_cast(float, largest[k]));
#pragma unroll
    for (int k = 0; k < N; k++) total[k] = __fadd_rn(total[k], __builtin_bit_cast(float, second[k]));
}
template <int N>
__device__ __forceinline__ void add_rows(float (&total)[N], const Pair (&largest)[N], const Pair (&second)[N], float one) {
#pragma unroll
    for (int row = 0; row < 2; row++) {
#pragma unroll
        for (int k = 0; k < N; k++) total[k] = __builtin_fmaf((float)__builtin_bit_cast(HalfPair, largest[k])[row], one, total[k]);
#pragma unroll
        for (int k = 0; k < N; k++) total[k] = __builtin_fmaf((float)__builtin_bit_cast(HalfPair, second[k])[row], one, total[k]);
    }
}
// the middle one of three, and of low <= high and x
__device__ __forceinline__ uint32_t middle(uint32_t low, uint32_t high, uint32_t x) {
    return __builtin_elementwise_max(__builtin_elementwise_min(low, high), __builtin_elementwise_min(__builtin_elementwise_max(low, high), x));
}
__device__ __forceinline__ Pair middle(Pair low, Pair high, Pair x) {
    return __builtin_elementwise_max(__builtin_elementwise_min(high, x), low);
}

__device__ __forceinline__ float magnitude(float x) { return __builtin_canonicalizef(__builtin_fabsf(x)); }
__device__ __forceinline__ uint16_t magnitude(__half x) {
    const uint16_t b = __half_as_ushort(x) & 0x7fffu;
    return b > 0x7c00u ? (uint16_t)(b | 0x200u) : b;            // (a NaN quiet, as every use of it as a number makes it)
}
__device__ __forceinline__ bool is_nan(float x) { return x != x; }
__device__ __forceinline__ bool is_nan(uint16_t x) { return x > 0x7c00u; }
__device__ __forceinline__ float widen(float x) { return x; }
__device__ __forceinline__ float widen(uint16_t x) { return __half2float(__ushort_as_half(x)); }
__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(__half x) { return __half2float(x); }
__device__ __forceinline__ uint16_t to_bits(float x) { return __half_as_ushort(__float2half_rn(x)); }
__device__ __forceinline__ uint16_t to_bits(__half x) { return __half_as_ushort(x); }

// how a magnitude is stored in LDS, and what one 32-bit word of a column holds (Word: one row in fp32, two rows in fp16)
template <class T> struct Stored;
template <> struct Stored<float> { using Type = float; using Word = uint32_t; };
template <> struct Stored<__half> { using Type = uint16_t; using Word = Pair; };

// triples out of n (a block's magnitudes fit the LDS, so a group has at most 1200 columns: 32 bits are enough)
__device__ __forceinline__ unsigned triples_of(int n) { return n < 3 ? 0u : (unsigned)n * (unsigned)(n - 1) / 2u * (unsigned)(n - 2) / 3u; }

struct Best {
    float total;
    uint64_t order;             // a, b, c, d in 16 bits each: lexicographic
    __device__ __forceinline__ void take(float t, uint64_t o) {
        if (t > total || (t == total && o < order)) {
            total = t;
            order = o;
        }
    }
};
__device__ __forceinline__ uint64_t order_of(int a, int b, int c, int d) {
    return ((uint64_t)a << 48) | ((uint64_t)b << 32) | ((uint64_t)c << 16) | (uint64_t)d;
}

// The totals of {a, b, c, d0 + k}, k < N; a d beyond `width` stands for the last one (a total twice, no harm done).
// units: 16-byte units of a column; base, pitch: the group's first column and the distance of two columns in such units
template <class T, int N>
__device__ __forceinline__ void run_triple(const uint4* base, int pitch, int units, int a, int b, int c, int d0, int width, float one,
                                           Best& best) {
    using Word = typename Stored<T>::Word;
    const uint4 *pa = base + a * pitch, *pb = base + b * pitch, *pc = base + c * pitch;
    const uint4* pd[N];
    float total[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        pd[k] = base + (d0 + k < width ? d0 + k : width - 1) * pitch;
        total[k] = 0.f;
    }
#pragma unroll 2
    for (int r = 0; r < units; r++) {
        const uint4 A = pa[r], B = pb[r], C = pc[r];
        uint4 D[N];
#pragma unroll
        for (int k = 0; k < N; k++) D[k] = pd[k][r];
        auto word = [&](uint32_t wa, uint32_t wb, uint32_t wc, auto member) {
            const Word x = __builtin_bit_cast(Word, wa), y = __builtin_bit_cast(Word, wb), z = __builtin_bit_cast(Word, wc);
            const Word h = __builtin_elementwise_max(x, y), l = __builtin_elementwise_min(x, y), t1 = __builtin_elementwise_max(h, z),
                       t2 = middle(l, h, z);
            Word largest[N], second[N];
#pragma unroll
            for (int k = 0; k < N; k++) {
                const Word d = __builtin_bit_cast(Word, member(D[k]));
                largest[k] = __builtin_elementwise_max(t1, d);
                second[k] = middle(t2, t1, d);
            }
            add_rows<N>(total, largest, second, one);
        };
        word(A.x, B.x, C.x, [](const uint4& v) { return v.x; });
        word(A.y, B.y, C.y, [](const uint4& v) { return v.y; });
        word(A.z, B.z, C.z, [](const uint4& v) { return v.z; });
        word(A.w, B.w, C.w, [](const uint4& v) { return v.w; });
    }
#pragma unroll
    for (int k = 0; k < N; k++) best.take(total[k], order_of(a, b, c, d0 + k < width ? d0 + k : width - 1));
}

// One subset as two pairs: which of the values a NaN hides depends on the order of the comparisons, and this one is the format's.
// take 3: the subset without d.
template <class T>
__device__ float total_of_pairs(const uint4* base, int pitch, int v, int a, int b, int c, int d, int take) {
    using S = typename Stored<T>::Type;
    const S *pa = (const S*)(base + a * pitch), *pb = (const S*)(base + b * pitch), *pc = (const S*)(base + c * pitch),
            *pd = (const S*)(base + d * pitch);
    float total = 0.f;
    for (int r = 0; r < v; r++) {
        const float x = widen(pa[r]), y = widen(pb[r]), z = widen(pc[r]);
        const float h1 = max2(x, y), l1 = min2(x, y);
        if (take == 4) {
            const float w = widen(pd[r]), h2 = max2(z, w), l2 = min2(z, w);
            total = __fadd_rn(total, max2(h1, h2));
            total = __fadd_rn(total, max3(min2(h1, h2), l1, l2));
        } else {
            total = __fadd_rn(total, max2(h1, z));
            total = __fadd_rn(total, max2(min2(h1, z), l1));
        }
    }
    return total;
}

// All subsets of the `here` groups of `width` columns at `base`, group_pitch apart: lane l works on group l % stride (stride a power
// of two, here <= stride; lanes without a group of their own repeat the last one's work).  counter: 0 on entry.
template <class T>
__device__ __forceinline__ void search(const uint4* base, int group_pitch, int pitch, int v, int stride_log2, int here, int width, bool nans,
                                       float one, unsigned* counter, Best& best) {
    const int lane = threadIdx.x & 63, units = v * (int)sizeof(typename Stored<T>::Type) / 16;
    const int mine = lane & ((1 << stride_log2) - 1), group = mine < here ? mine : here - 1;
    const uint4* cols0 = base + group * group_pitch;
    const unsigned triples = triples_of(width - 1);
    while (true) {
        unsigned batch = 0;
        if (lane == 0) batch = atomicAdd(counter, 1u);
        batch = __builtin_amdgcn_readfirstlane(batch);
        const unsigned first = batch << (6 - stride_log2);
        if (first >= triples) break;
        unsigned t = first + (unsigned)(lane >> stride_log2);
        if (t >= triples) t = triples - 1;
        int c = 2, b = 1;                    // c (c - 1) / 2 triples have c as their largest member, b of those b in the middle
        for (unsigned with_c = 1; t >= with_c; c++) {
            t -= with_c;
            with_c += (unsigned)c;
        }
        for (; t >= (unsigned)b; b++) t -= (unsigned)b;
        const int a = (int)t;
        // (c does not fall from lane to lane: the first lane has the longest run)
        const int longest = __builtin_amdgcn_readfirstlane(width - 1 - c);
        if (nans) {
            for (int k = 0; k < longest; k++) {
                const int d = c + 1 + k < width ? c + 1 + k : width - 1;
                best.take(total_of_pairs<T>(cols0, pitch, v, a, b, c, d, 4), order_of(a, b, c, d));
            }
            continue;
        }
        const int pieces = (longest + kRun - 1) / kRun, n = (longest + pieces - 1) / pieces;
        for (int p = 0; p < pieces; p++) {
            const int d0 = c + 1 + p * n < width ? c + 1 + p * n : width - 1;
            switch (n) {
                case 1: run_triple<T, 1>(cols0, pitch, units, a, b, c, d0, width, one, best); break;
                case 2: run_triple<T, 2>(cols0, pitch, units, a, b, c, d0, width, one, best); break;
                case 3: run_triple<T, 3>(cols0, pitch, units, a, b, c, d0, width, one, best); break;
                case 4: run_triple<T, 4>(cols0, pitch, units, a, b, c, d0, width, one, best); break;
                default: run_triple<T, 5>(cols0, pitch, units, a, b, c, d0, width, one, best); break;
            }
        }
    }
}

// What row `src` (of one group) keeps of its columns c: the two largest magnitudes, the lower column among equals.
// kept: the two values' bits, the lower position in the low half; returns the two positions, two bits each.
template <class T>
__device__ __forceinline__ uint32_t keep_two(const T* src, const int4& c4, int take, uint32_t& kept) {
    const int c[4] = {c4.x, c4.y, c4.z, c4.w};
    T x[4];
    float a[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        x[i] = src[c[i]];        // (a fourth column that is not there reads the first again)
        a[i] = __builtin_fabsf(to_float(x[i]));
    }
    int i1 = 0, i2 = -1;
    float a1 = a[0], a2 = 0.f;
#pragma unroll
    for (int i = 1; i < 4; i++)
        if (i < take && a[i] > a1) { i1 = i; a1 = a[i]; }
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (i < take && i != i1 && (i2 < 0 || a[i] > a2)) { i2 = i; a2 = a[i]; }
    const int lo = i1 < i2 ? i1 : i2, hi = i1 < i2 ? i2 : i1;
    kept = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (i == lo) kept |= to_bits(x[i]);
        if (i == hi) kept |= (uint32_t)to_bits(x[i]) << 16;
    }
    return (uint32_t)(lo | (hi << 2));
}

// The same for group g, whose columns in one row are at `src`, whatever it is: searched ones by their winner, a tail of one or two columns whole, zeros beyond the matrix.
template <class T>
__device__ __forceinline__ uint32_t encode_group(const T* src, int g, int full, int rem, const int4& c4, uint32_t& kept) {
    kept = 0;
    if (g < full || (g == full && rem >= 3)) {
        // (positions 0 and 1: what a group without a winner stores)
        return c4.y != 0 ? keep_two(src, c4, g == full && rem == 3 ? 3 : 4, kept) : 4u;
    }
    if (g == full && rem > 0) {
        kept = to_bits(src[0]);
        if (rem == 2) kept |= (uint32_t)to_bits(src[1]) << 16;
        return rem == 2 ? 4u : 0u;
    }
    return 0u;
}

struct Conversion {
    int rows, cols, m, v, full, rem;
    int group_log2, wgs_per_block;      // groups per workgroup, workgroups per V block
    int pitch, group_pitch;             // of columns and groups in LDS, 16-byte units
    int4* columns;                      // winners, `columns_pitch` groups per V block
    int64_t columns_pitch;
    int ksp;                            // ENCODE: values, metadata
    uint16_t* values;
    uint32_t* metadata;
    float one;                          // 1 (add_rows)
};
}  // namespace

// Workgroup = 1 << group_log2 adjacent groups of one V block.  Without ENCODE the searched groups alone (the full ones, then a tail
// of three or more columns); with ENCODE all groups of the padded row, and values, metadata and column-loc of them are written.
template <class T, bool ENCODE>
__global__ __launch_bounds__(kThreads) void select_kernel(const T* __restrict__ dense, Conversion p) {
    using S = typename Stored<T>::Type;
    extern __shared__ uint4 tile[];                 // [group][column][units]
    __shared__ unsigned best_bits[kMaxGroups], counters[2], any_nan;
    __shared__ unsigned long long best_order[kMaxGroups];
    __shared__ int4 winners[kMaxGroups];
    const int tid = threadIdx.x, m = p.m, v = p.v;
    const int b = blockIdx.x / p.wgs_per_block, first = (blockIdx.x - b * p.wgs_per_block) << p.group_log2;
    const int searched = p.full + (p.rem >= 3 ? 1 : 0);
    const int here = p.full - first < (1 << p.group_log2) ? p.full - first : 1 << p.group_log2;        // full groups (may be <= 0)
    const bool has_tail = p.rem >= 3 && p.full >= first && p.full < first + (1 << p.group_log2);
    const T* base = dense + (int64_t)b * v * p.cols + (int64_t)first * m;
    if (tid < kMaxGroups) {
        best_bits[tid] = 0u;
        best_order[tid] = ~0ull;
        if (tid < 2) counters[tid] = 0u;
        if (tid == 2) any_nan = 0u;
    }
    __syncthreads();
    // magnitudes, transposed: two rows of a column at a time
    const int w = (here > 0 ? here * m : 0) + (has_tail ? p.rem : 0);
    bool nan = false;
    const int across = w < kThreads ? w : kThreads, pairs_at_once = w > 0 ? kThreads / across : 1, r0 = w > 0 ? tid / across : 0;
    if (r0 < pairs_at_once) {
        for (int c = tid - r0 * across; c < w; c += across) {
            const int g = c / m;
            S* column = (S*)(tile + g * p.group_pitch + (c - g * m) * p.pitch);
#pragma unroll 4
            for (int r = r0 * 2; r < v; r += pairs_at_once * 2) {
                const S x = magnitude(base[(int64_t)r * p.cols + c]), y = magnitude(base[(int64_t)(r + 1) * p.cols + c]);
                nan |= is_nan(x) | is_nan(y);
                if constexpr (sizeof(S) == 2) {
                    *(uint32_t*)(column + r) = (uint32_t)x | ((uint32_t)y << 16);
                } else {
                    *(float2*)(column + r) = make_float2(x, y);
                }
            }
        }
    }
    if (nan) any_nan = 1u;
    __syncthreads();
    const bool nans = any_nan != 0u;
    // the largest total of a group (positive floats order like their bits), then the first subset that reaches it
    auto settle = [&](const Best& best, int slot, bool mine) {
        const unsigned bits = mine && best.total > 0.f ? __builtin_bit_cast(unsigned, best.total) : 0u;
        if (bits) atomicMax(&best_bits[slot], bits);
        __syncthreads();
        if (bits && bits == best_bits[slot]) atomicMin(&best_order[slot], (unsigned long long)best.order);
    };
    if (here > 0) {
        Best best = {0.f, ~0ull};
        search<T>(tile, p.group_pitch, p.pitch, v, p.group_log2, here, m, nans, p.one, &counters[0], best);
        const int slot = tid & ((1 << p.group_log2) - 1);
        settle(best, slot < here ? slot : here - 1, true);
    }
    if (has_tail) {
        const int slot = p.full - first;
        const uint4* cols0 = tile + slot * p.group_pitch;
        Best best = {0.f, ~0ull};
        if (p.rem == 3) {
            if (tid == 0) best.take(total_of_pairs<T>(cols0, p.pitch, v, 0, 1, 2, 0, 3), order_of(0, 1, 2, 0));
        } else {
            search<T>(cols0, 0, p.pitch, v, 0, 1, p.rem, nans, p.one, &counters[1], best);
        }
        settle(best, slot, true);
    }
    __syncthreads();
    if (tid < 1 << p.group_log2) {
        const int g = first + tid;
        int4 pick = make_int4(0, 0, 0, 0);
        if (best_bits[tid]) {
            const unsigned long long o = best_order[tid];
            pick = make_int4((int)(o >> 48), (int)(o >> 32) & 0xffff, (int)(o >> 16) & 0xffff, (int)o & 0xffff);
        }
        if (ENCODE && g == p.full && (p.rem == 1 || p.rem == 2)) pick = make_int4(0, 1, 2, 3);
        winners[tid] = pick;
        if (g < (ENCODE ? p.ksp >> 1 : searched)) p.columns[(int64_t)b * p.columns_pitch + g] = pick;
    }
    if constexpr (ENCODE) {
        // a wave per 16 rows x 4 groups: lane = row / 4, group, row / 2 % 2, row % 2 (from the top), which is the order of the values
        __syncthreads();
        const int lane = tid & 63, q = lane >> 4, u = (lane >> 2) & 3, pr = (lane >> 1) & 1, s = lane & 1;
        const int quads = ((p.ksp >> 1) - first < (1 << p.group_log2) ? (p.ksp >> 1) - first : 1 << p.group_log2) >> 2;
        for (int i = tid >> 6; i < (v >> 4) * quads; i += kThreads / 64) {
            const int r16 = i / quads, t = i - r16 * quads, g = first + t * 4 + u;
            const int64_t row = (int64_t)b * v + r16 * 16 + q * 4 + pr * 2 + s;
            uint32_t kept;
            uint32_t word = encode_group(dense + row * p.cols + (int64_t)g * m, g, p.full, p.rem, winners[t * 4 + u], kept) << (s * 16 + u * 4);
            const int64_t tg = (first >> 2) + t;
            *(uint32_t*)(p.values + (row >> 4) * 16 * (int64_t)p.ksp + tg * 128 + lane * 2) = kept;
            word |= (uint32_t)__shfl_xor((int)word, 1);
            word |= (uint32_t)__shfl_xor((int)word, 4);
            word |= (uint32_t)__shfl_xor((int)word, 8);
            if (s == 0 && u == 0)
                p.metadata[(row >> 5) * (int64_t)(p.ksp >> 3) * 16 + tg * 16 + ((row >> 4) & 1) * 8 + q * 2 + pr] = word;
        }
    }
}

// The encoding by itself, behind a search whose workgroups hold fewer than four groups.  Thread id = (32-row block * tiles + tile) *
// 16 + row pair of the block: the index of its metadata word.
template <class T>
__global__ __launch_bounds__(256) void encode_winners_kernel(const T* __restrict__ dense, int rows, int cols, int m, int v, int ksp,
                                                             uint16_t* __restrict__ values, uint32_t* __restrict__ metadata,
                                                             int4* __restrict__ columns) {
    const int tiles = ksp >> 3, ngroups = ksp >> 1;
    const int full = cols / m, rem = cols - full * m, searched = full + (rem >= 3 ? 1 : 0);
    const int64_t total = (int64_t)(rows >> 1) * tiles;
    for (int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; id < total; id += (int64_t)gridDim.x * blockDim.x) {
        const int pair = (int)(id & 15);
        const int64_t bt = id >> 4;
        const int64_t rb = bt / tiles;
        const int t = (int)(bt - rb * tiles);
        const int64_t row = rb * 32 + pair * 2;
        const int64_t b = row / v;
        const bool leader = row == b * v;            // fills the columns that the search has not
        uint16_t* out = values + (row >> 4) * 16 * (int64_t)ksp + (int64_t)t * 128 + ((pair >> 1) & 3) * 32 + (pair & 1) * 4;
        uint32_t word = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int g = t * 4 + u;
            int4 c4 = make_int4(0, 0, 0, 0);
            if (g < searched) {
                c4 = columns[b * ngroups + g];
            } else {
                if (g == full && rem > 0) c4 = make_int4(0, 1, 2, 3);
                if (leader) columns[b * ngroups + g] = c4;
            }
            uint2 packed;
            word |= encode_group(dense + row * cols + (int64_t)g * m, g, full, rem, c4, packed.x) << (u * 4);
            word |= encode_group(dense + (row + 1) * cols + (int64_t)g * m, g, full, rem, c4, packed.y) << (16 + u * 4);
            *(uint2*)(out + u * 8) = packed;
        }
        metadata[id] = word;
    }
}

namespace {
// LDS of a workgroup of 1 << log2 groups, and the pitches in it: a column an odd number of 16-byte units from the next, and a group
// too; without the spare units (last resort) everything close together.
size_t lay_out(Conversion& p, int value_bytes, int log2, bool spare) {
    const int units = p.v * value_bytes / 16;
    p.group_log2 = log2;
    p.pitch = units + (spare ? 1 : 0);
    const int widest = p.full > 0 ? p.m : p.rem;
    p.group_pitch = widest * p.pitch;
    if (spare && p.group_pitch % 2 == 0) p.group_pitch++;
    return (size_t)std::min(1 << log2, std::max(p.full + (p.rem >= 3 ? 1 : 0), 1)) * p.group_pitch * 16;
}

// Groups per workgroup, as a power of two: the count with the shortest time by a fit to 400 timings (six matrices of 768 x 768 to
// 4096 x 1024, V = 32, 64, 128, m = 4 to 32, every count).  Rounds of workgroups over the CUs cost 0.16 ns per triple and row, 0.21 where
// a CU has one workgroup only (two waves per SIMD), and a workgroup's loads, barriers and stores 2 us of its CU.  The larger count
// where two are level, within 72 KB of LDS so that two workgroups share a CU.  Fewer than four groups cost the encoding a launch of
// its own (6 us; metadata words hold four).
template <class T>
int groups_log2(Conversion& p, int groups, int cus) {
    const double triple_rows = (double)(p.m - 1) * (p.m - 2) * (p.m - 3) / 6 * p.v;
    int best = -1;
    double least = 0;
    for (int log2 = 5; log2 >= 0; log2--) {
        if (lay_out(p, (int)sizeof(T), log2, log2 > 0) > (log2 > 2 ? 72 * 1024 : kLdsLimit)) continue;
        const int64_t wgs = (int64_t)(p.rows / p.v) * ((groups + (1 << log2) - 1) >> log2), rounds = (wgs + cus - 1) / cus;
        const double cost = (double)rounds * (1 << log2) * triple_rows * (rounds == 1 ? 0.21e-3 : 0.16e-3) + 2. * (double)wgs / cus +
                            (p.values && log2 < 2 ? 6. : 0.);
        if (best < 0 || cost < least) {
            least = cost;
            best = log2;
        }
    }
    return best < 0 ? 0 : best;
}

template <class T>
Conversion conversion_of(const T* dense, int rows, int cols, int m, int v, int32_t* columns, int64_t columns_pitch) {
    Conversion p = {};
    p.rows = rows; p.cols = cols; p.m = m; p.v = v; p.full = cols / m; p.rem = cols % m;
    p.columns = (int4*)columns;
    p.columns_pitch = columns_pitch;
    p.one = 1.f;
    return p;
}

template <class T, bool ENCODE>
hipError_t launch_select(const T* dense, Conversion p, int groups, int log2, hipStream_t stream) {
    size_t lds = lay_out(p, (int)sizeof(T), log2, true);
    if (lds > kLdsLimit) lds = lay_out(p, (int)sizeof(T), log2, false);
    if (lds > kLdsLimit) return hipErrorInvalidValue;
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)select_kernel<T, ENCODE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    p.wgs_per_block = (groups + (1 << log2) - 1) >> log2;
    hipLaunchKernelGGL((select_kernel<T, ENCODE>), dim3((unsigned)((int64_t)(p.rows / p.v) * p.wgs_per_block)), dim3(kThreads), lds, stream,
                       dense, p);
    return hipGetLastError();
}

template <class T>
hipError_t launch_convert_t(const T* dense, int rows, int cols, int m, int v, int ksp, int cus, uint16_t* values, uint32_t* metadata,
                            int32_t* columns, hipStream_t stream) {
    Conversion p = conversion_of<T>(dense, rows, cols, m, v, columns, ksp / 2);
    p.ksp = ksp;
    p.values = values;
    p.metadata = metadata;
    const int log2 = groups_log2<T>(p, ksp / 2, cus > 0 ? cus : 256), searched = p.full + (p.rem >= 3 ? 1 : 0);
    if (log2 >= 2) return launch_select<T, true>(dense, p, ksp / 2, log2, stream);
    const hipError_t e = searched ? launch_select<T, false>(dense, p, searched, log2, stream) : hipSuccess;
    if (e != hipSuccess) return e;
    const int64_t blocks = ((int64_t)(rows / 2) * (ksp / 8) + 255) / 256;
    hipLaunchKernelGGL((encode_winners_kernel<T>), dim3((unsigned)std::min<int64_t>(blocks, 65535 * 8)), dim3(256), 0, stream, dense, rows,
                       cols, m, v, ksp, values, metadata, (int4*)columns);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_select_winners_f32(const float* dense_dev, int rows, int cols, int m, int v, int cus, int32_t* out_dev,
                                     int64_t out_pitch, hipStream_t stream) {
    Conversion p = conversion_of<float>(dense_dev, rows, cols, m, v, out_dev, out_pitch);
    const int groups = p.full + (p.rem >= 3 ? 1 : 0);
    if ((rows / v) * (int64_t)groups == 0) return hipSuccess;
    return launch_select<float, false>(dense_dev, p, groups, groups_log2<float>(p, groups, cus > 0 ? cus : 256), stream);
}

hipError_t launch_convert(const void* dense_dev, int value_bits, int rows, int cols, int m, int v, int ksp, int cus, uint16_t* values,
                          uint32_t* metadata, int32_t* columns, hipStream_t stream) {
    return value_bits == 16 ? launch_convert_t<__half>((const __half*)dense_dev, rows, cols, m, v, ksp, cus, values, metadata, columns, stream)
                            : launch_convert_t<float>((const float*)dense_dev, rows, cols, m, v, ksp, cus, values, metadata, columns, stream);
}

}  // namespace spatha
