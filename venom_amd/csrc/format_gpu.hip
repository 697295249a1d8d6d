// V:N:M encoding and decoding on the GPU: the same entries in the same places as the host builder (vnm_format.cpp, which holds the
// storage map), from and to matrices that live in device memory (to_sparse_sr_nm / func2 and to_dense / func3,
// end2end/grouped_nmv_tensor.py:345-675).  Both kernels only move data; one thread owns one metadata word (two rows, four groups)
// or eight adjacent entries of a dense row, so that the compressed side and the dense side are each written in whole words.
// Encoding 4096 x 1024 at 64:2:8: 7.2 us; decoding 1024 x 4096 at 128:2:16: 6.8 us (a call of to_dense 32 us, most of it the wait for
// the flag of the offset check; 870 us when the arrays were decoded on the host).

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "spmm_kernels.h"

namespace spatha {

namespace {
__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(__half x) { return __half2float(x); }
__device__ __forceinline__ uint16_t to_bits(float x) { return __half_as_ushort(__float2half_rn(x)); }
__device__ __forceinline__ uint16_t to_bits(__half x) { return __half_as_ushort(x); }
}  // namespace

// Thread id = (32-row block * tiles + tile) * 16 + row pair of the block: the index of its metadata word.  Groups below `searched`
// keep, per row, the two largest magnitudes of the four winners (the lower column among equals); a tail of one or two columns is
// kept whole; groups beyond the matrix store zeros at position 0.
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
            uint16_t kept[4] = {0, 0, 0, 0};
            uint32_t nib[2] = {0u, 0u};
            if (g < searched) {
                const int4 c4 = columns[b * ngroups + g];
                const int c[4] = {c4.x, c4.y, c4.z, c4.w};
                const int take = (g == full && rem == 3) ? 3 : 4;
                nib[0] = nib[1] = 4u;                // positions 0 and 1: what a group without a winner stores
                if (c4.y != 0) {
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        const T* src = dense + (row + s) * cols + (int64_t)g * m;
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
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if (i == lo) kept[2 * s] = to_bits(x[i]);
                            if (i == hi) kept[2 * s + 1] = to_bits(x[i]);
                        }
                        nib[s] = (uint32_t)(lo | (hi << 2));
                    }
                }
            } else if (g == full && rem > 0) {
                if (rem == 2) nib[0] = nib[1] = 4u;
#pragma unroll
                for (int s = 0; s < 2; s++)
                    for (int j = 0; j < rem; j++) kept[2 * s + j] = to_bits(dense[(row + s) * cols + (int64_t)g * m + j]);
                if (leader) columns[b * ngroups + g] = make_int4(0, 1, 2, 3);
            } else if (leader) {
                columns[b * ngroups + g] = make_int4(0, 0, 0, 0);
            }
            uint2 packed;
            packed.x = kept[0] | ((uint32_t)kept[1] << 16);
            packed.y = kept[2] | ((uint32_t)kept[3] << 16);
            *(uint2*)(out + u * 8) = packed;
            word |= (nib[0] << (u * 4)) | (nib[1] << (16 + u * 4));
        }
        metadata[id] = word;
    }
}

__global__ __launch_bounds__(256) void decode_kernel(const uint16_t* __restrict__ values, const uint32_t* __restrict__ metadata,
                                                     const uint32_t* __restrict__ columns, int rows, int cols, int m, int v, int ksp,
                                                     uint16_t* __restrict__ dense, uint32_t* __restrict__ bad) {
    const int ngroups = ksp >> 1, per_row = (cols + 7) / 8;
    const int64_t start = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t n_columns = (int64_t)(rows / v) * ngroups * 4;
    for (int64_t i = start; i < n_columns; i += stride)
        if (columns[i] >= (uint32_t)m) *bad = 1u;
    for (int64_t id = start; id < (int64_t)rows * per_row; id += stride) {
        const int64_t r = id / per_row;
        const int c0 = (int)(id - r * per_row) * 8;
        const int64_t b = r / v;
        const uint16_t* vrow = values + (r >> 4) * 16 * (int64_t)ksp + ((r >> 2) & 3) * 32 + ((r >> 1) & 1) * 4 + (r & 1) * 2;
        const uint32_t* mrow = metadata + (r >> 5) * (int64_t)(ksp >> 3) * 16 + ((r & 31) >> 1);
        uint32_t out[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        const int stop = c0 + 8 < cols ? c0 + 8 : cols;
        for (int g = c0 / m; g * (int64_t)m < stop; g++) {
            const int t = g >> 2, u = g & 3;
            const uint32_t nib = (mrow[(int64_t)t * 16] >> ((int)(r & 1) * 16 + u * 4)) & 0xfu;
            const uint32_t two = *(const uint32_t*)(vrow + (int64_t)t * 128 + u * 8);
            const uint32_t* cl = columns + (b * ngroups + g) * 4;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t loc = cl[(nib >> (2 * j)) & 3u];
                const int64_t at = (int64_t)g * m + loc - c0;
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (loc < (uint32_t)m && at == k) out[k] = j ? two >> 16 : two & 0xffffu;
            }
        }
        uint16_t* dst = dense + r * cols + c0;
        if ((cols & 7) == 0) {
            *(uint4*)dst = make_uint4(out[0] | (out[1] << 16), out[2] | (out[3] << 16), out[4] | (out[5] << 16), out[6] | (out[7] << 16));
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (c0 + k < cols) dst[k] = (uint16_t)out[k];
        }
    }
}

static unsigned blocks_for(int64_t threads) {
    const int64_t blocks = (threads + 255) / 256;
    return (unsigned)(blocks < 65535 * 8 ? blocks : 65535 * 8);
}

hipError_t launch_encode_winners(const void* dense_dev, int value_bits, int rows, int cols, int m, int v, int ksp, uint16_t* values,
                                 uint32_t* metadata, int32_t* columns, hipStream_t stream) {
    const dim3 grid(blocks_for((int64_t)(rows / 2) * (ksp / 8))), block(256);
    if (value_bits == 16)
        hipLaunchKernelGGL((encode_winners_kernel<__half>), grid, block, 0, stream, (const __half*)dense_dev, rows, cols, m, v, ksp, values,
                           metadata, (int4*)columns);
    else
        hipLaunchKernelGGL((encode_winners_kernel<float>), grid, block, 0, stream, (const float*)dense_dev, rows, cols, m, v, ksp, values,
                           metadata, (int4*)columns);
    return hipGetLastError();
}

hipError_t launch_decode_f16(const uint16_t* values, const uint32_t* metadata, const uint32_t* columns, int rows, int cols, int m,
                             int v, int ksp, uint16_t* dense, uint32_t* bad, hipStream_t stream) {
    const dim3 grid(blocks_for((int64_t)rows * ((cols + 7) / 8))), block(256);
    hipLaunchKernelGGL(decode_kernel, grid, block, 0, stream, values, metadata, columns, rows, cols, m, v, ksp, dense, bad);
    return hipGetLastError();
}

}  // namespace spatha
