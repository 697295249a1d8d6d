// Magnitude selector, search phase on the GPU: for every (V-row block, m-column group) the subset of 4 (3 in a
// three-column tail) columns that maximises the sum over the block's rows of the two largest magnitudes
// (group_n_m2 / func, end2end/grouped_nmv_tensor.py:81-343).  The totals are accumulated exactly as the host code
// does it (fp32, row by row, largest then second largest, no fused operations), subsets are ranked in lexicographic
// order and only a strictly larger total replaces the best one, so the winner is the host's winner bit for bit.
//
// What bounds it: a subset's total is a serial chain of 2 V additions (their order is part of the result), so the work is
// V x subsets x (7 comparisons + 2 additions + 16 bytes of LDS reads), spread over independent (task, subset) chains.  A
// workgroup takes `groups` adjacent column groups of one V block, `lanes` threads each, every thread a contiguous range of
// subset ranks: with one group per workgroup (the form before this one) m = 8 kept 70 of 256 threads busy.  Magnitudes sit
// in LDS column by column (pitch V + 4 words: 16-byte reads of four rows at a time, sixteen different columns on different
// banks).
// 4096 x 1024 at 64:2:8 (8192 groups of 70 subsets): 28 us, 1024 x 1024 14.5; 4096 x 1024 at 64:2:16 (1820 subsets) 161.  With the
// encoder behind it (format_gpu.hip, 7.2 us) the first conversion takes 37.5 us, 6.3 ms when magnitudes, masks and arrays went
// through the host.

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <algorithm>

#include "spmm_kernels.h"

namespace spatha {

namespace {
__host__ __device__ __forceinline__ unsigned long long binom(int n, int k) {      // k <= 4
    if (k < 0 || n < k) return 0ull;
    unsigned long long r = 1ull;
    for (int i = 0; i < k; i++) r = r * (unsigned long long)(n - i) / (unsigned long long)(i + 1);
    return r;
}

// the rank-th subset of {0..width-1} of size `take` in lexicographic order
__device__ __forceinline__ void unrank(unsigned long long left, int width, int take, int (&pick)[4]) {
    if (binom(width, take) >> 31) {
        int c = 0;
        for (int i = 0; i < take; i++) {
            while (true) {
                const unsigned long long below = binom(width - 1 - c, take - 1 - i);   // subsets that keep c at position i
                if (left < below) break;
                left -= below;
                c++;
            }
            pick[i] = c++;
        }
        return;
    }
    // the same in 32 bits (every count fits), without divisions by a variable
    uint32_t l = (uint32_t)left;
    int c = 0;
    for (int i = 0; i < take; i++) {
        while (true) {
            const uint32_t n = (uint32_t)(width - 1 - c);
            const int k = take - 1 - i;
            uint32_t below = 1u;
            if (k == 1) below = n;
            else if (k == 2) below = n * (n - 1u) / 2u;
            else if (k == 3) below = n * (n - 1u) / 2u * (n - 2u) / 3u;
            if (l < below) break;
            l -= below;
            c++;
        }
        pick[i] = c++;
    }
}

// (operands are canonical - `magnitude` made them so -: without the quieting instruction that fmaxf / fminf put in front of every
// operand that comes from memory, 9 instructions a row and subset instead of 14)
__device__ __forceinline__ float max2(float a, float b) { float d; asm("v_max_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b)); return d; }
__device__ __forceinline__ float min2(float a, float b) { float d; asm("v_min_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b)); return d; }
__device__ __forceinline__ float max3(float a, float b, float c) {
    float d;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

__device__ __forceinline__ float magnitude(float x) { return __builtin_canonicalizef(__builtin_fabsf(x)); }
__device__ __forceinline__ float magnitude(__half x) { return __builtin_canonicalizef(__builtin_fabsf(__half2float(x))); }
}  // namespace

// Full groups: workgroup = `groups` adjacent groups of one V block, `lanes` threads per group (groups * lanes <= 256).
// The tail group (take_tail > 0, width = cols % m): a workgroup of its own per V block, behind the full ones, 256 threads.
// out: int4 per (V block, group), out_pitch entries per block; zeros where no subset has a positive total.
template <class T>
__global__ __launch_bounds__(256) void select_winners_kernel(const T* __restrict__ dense, int cols, int m, int v, int full,
                                                             int rem, int groups, int lanes, int wgs_per_block, int take_tail,
                                                             int pitch, int4* __restrict__ out, int64_t out_pitch) {
    extern __shared__ float4 tile4[];               // [column][pitch / 4]
    __shared__ unsigned best_bits[256];
    __shared__ unsigned long long best_rank[256];
    float* tile = (float*)tile4;
    const int tid = threadIdx.x;
    const int b = blockIdx.x / wgs_per_block, wg = blockIdx.x - b * wgs_per_block;
    const bool is_tail = take_tail > 0 && wg == wgs_per_block - 1;
    const int first = is_tail ? full : wg * groups;
    const int here = is_tail ? 1 : (full - first < groups ? full - first : groups);
    const int width = is_tail ? rem : m, take = is_tail ? take_tail : 4;
    const int per = is_tail ? 256 : lanes;
    const int w = here * width;
    const T* base = dense + (int64_t)b * v * cols + (int64_t)first * m;
    best_bits[tid] = 0u;
    best_rank[tid] = ~0ull;
    if (w <= 256) {
        const int rows_at_once = 256 / w, r0 = tid / w, c = tid - r0 * w;
        if (r0 < rows_at_once)
            for (int r = r0; r < v; r += rows_at_once) tile[c * pitch + r] = magnitude(base[(int64_t)r * cols + c]);
    } else {
        for (int r = 0; r < v; r++)
            for (int c = tid; c < w; c += 256) tile[c * pitch + r] = magnitude(base[(int64_t)r * cols + c]);
    }
    __syncthreads();
    const int mine = tid / per, sub = tid - mine * per;
    const unsigned long long nsub = binom(width, take);
    const unsigned long long chunk = (nsub + (unsigned)per - 1) / (unsigned)per;
    unsigned long long rank = chunk * (unsigned)sub;
    const unsigned long long end = rank + chunk < nsub ? rank + chunk : nsub;
    float best = 0.f;
    unsigned long long best_at = ~0ull;
    if (mine < here && rank < nsub) {
        int pick[4] = {0, 0, 0, 0};
        unrank(rank, width, take, pick);
        const float* cols0 = tile + (int64_t)mine * width * pitch;
        for (; rank < end; rank++) {
            float total = 0.f;
            const float4* t0 = (const float4*)(cols0 + pick[0] * pitch);
            const float4* t1 = (const float4*)(cols0 + pick[1] * pitch);
            const float4* t2 = (const float4*)(cols0 + pick[2] * pitch);
            if (take == 4) {
                const float4* t3 = (const float4*)(cols0 + pick[3] * pitch);
                auto row = [&total](float a, float bb, float c, float d) {
                    const float h1 = max2(a, bb), l1 = min2(a, bb), h2 = max2(c, d), l2 = min2(c, d);
                    total = __fadd_rn(total, max2(h1, h2));
                    total = __fadd_rn(total, max3(min2(h1, h2), l1, l2));
                };
#pragma unroll 4
                for (int r = 0; r < v / 4; r++) {
                    const float4 a = t0[r], bb = t1[r], c = t2[r], d = t3[r];
                    row(a.x, bb.x, c.x, d.x);
                    row(a.y, bb.y, c.y, d.y);
                    row(a.z, bb.z, c.z, d.z);
                    row(a.w, bb.w, c.w, d.w);
                }
            } else {
                auto row = [&total](float a, float bb, float c) {
                    const float h1 = max2(a, bb), l1 = min2(a, bb);
                    total = __fadd_rn(total, max2(h1, c));
                    total = __fadd_rn(total, max2(min2(h1, c), l1));
                };
                for (int r = 0; r < v / 4; r++) {
                    const float4 a = t0[r], bb = t1[r], c = t2[r];
                    row(a.x, bb.x, c.x);
                    row(a.y, bb.y, c.y);
                    row(a.z, bb.z, c.z);
                    row(a.w, bb.w, c.w);
                }
            }
            if (total > best) {
                best = total;
                best_at = rank;
            }
            // next subset in lexicographic order
            int i = take - 1;
            while (i >= 0 && pick[i] == width - take + i) i--;
            if (i >= 0) {
                pick[i]++;
                for (int k = i + 1; k < take; k++) pick[k] = pick[k - 1] + 1;
            }
        }
    }
    // the largest total of the group (positive floats order like their bits), then the lowest rank that reaches it
    const unsigned bits = best_at != ~0ull ? __builtin_bit_cast(unsigned, best) : 0u;
    if (bits) atomicMax(&best_bits[mine], bits);
    __syncthreads();
    if (bits && bits == best_bits[mine]) atomicMin(&best_rank[mine], best_at);
    __syncthreads();
    if (tid < here) {
        int pick[4] = {0, 0, 0, 0};
        if (best_bits[tid]) unrank(best_rank[tid], width, take, pick);
        out[(int64_t)b * out_pitch + first + tid] = make_int4(pick[0], pick[1], pick[2], pick[3]);
    }
}

template <class T>
hipError_t launch_select_winners(const T* dense_dev, int rows, int cols, int m, int v, int cus, int32_t* out_dev,
                                 int64_t out_pitch, hipStream_t stream) {
    const int blocks = rows / v, full = cols / m, rem = cols % m;
    const int take_tail = rem >= 3 ? (rem == 3 ? 3 : 4) : 0;
    if (blocks * (int64_t)(full + (take_tail ? 1 : 0)) == 0) return hipSuccess;
    if (cus <= 0) cus = 256;
    // Groups per workgroup: the count with the least (rounds of four workgroups per CU) x (subsets per thread), within 48 KB of
    // LDS; more threads per group only shorten the chains until a thread holds one subset.
    const int pitch_pad = v + 4;
    int groups = 1;
    double least = 0;
    for (int g = 1; g <= 64 && g <= std::max(full, 1); g++) {
        if (g > 1 && (size_t)g * m * pitch_pad * sizeof(float) > 48 * 1024) break;
        const double chunk = (double)((binom(m, 4) + 256 / g - 1) / (256 / g));
        const int64_t wgs = (int64_t)blocks * ((full + g - 1) / g), rounds = (wgs + 4 * cus - 1) / (4 * cus);
        const double cost = (double)rounds * (chunk + 0.25 * g * m / 16);      // (+ the loads of the block's rows)
        if (g == 1 || cost < least) {
            least = cost;
            groups = g;
        }
    }
    const int widest = std::max(full > 0 ? groups * m : 0, take_tail ? rem : 0);
    int pitch = pitch_pad;
    if ((size_t)widest * pitch * sizeof(float) > 150 * 1024) pitch = v;
    const size_t lds = (size_t)widest * pitch * sizeof(float);
    if (lds > 150 * 1024) return hipErrorInvalidValue;
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)select_winners_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const int wgs_per_block = (full + groups - 1) / groups + (take_tail ? 1 : 0);
    hipLaunchKernelGGL((select_winners_kernel<T>), dim3((unsigned)((int64_t)blocks * wgs_per_block)), dim3(256), lds, stream, dense_dev,
                       cols, m, v, full, rem, groups, 256 / groups, wgs_per_block, take_tail, pitch, (int4*)out_dev, out_pitch);
    return hipGetLastError();
}

hipError_t launch_select_winners_f32(const float* dense_dev, int rows, int cols, int m, int v, int cus, int32_t* out_dev,
                                     int64_t out_pitch, hipStream_t stream) {
    return launch_select_winners<float>(dense_dev, rows, cols, m, v, cus, out_dev, out_pitch, stream);
}
hipError_t launch_select_winners_f16(const uint16_t* dense_dev, int rows, int cols, int m, int v, int cus, int32_t* out_dev,
                                     int64_t out_pitch, hipStream_t stream) {
    return launch_select_winners<__half>((const __half*)dense_dev, rows, cols, m, v, cus, out_dev, out_pitch, stream);
}

}  // namespace spatha
