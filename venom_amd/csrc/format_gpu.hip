// V:N:M decoding on the GPU: the same entries in the same places as the host builder (vnm_format.cpp, which holds the storage map), to
// matrices that live in device memory (to_dense / func3, end2end/grouped_nmv_tensor.py:563-675).  The kernel only moves data; one
// thread owns eight adjacent entries of a dense row, so that the dense side is written in whole words.
// A call of to_dense on 1024 x 4096 at 128:2:16 takes 19.4 us, of which launching and waiting for the flag of the offset check are 13
// (26.3 with the flag and the arrays handled in Python, and a 64-bit division per thread here; 870 when the host decoded).

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "spmm_kernels.h"

namespace spatha {

// Workgroup = four rows of 64 pieces of eight entries; the offsets are looked over by the first workgroups, one each per thread.
__global__ __launch_bounds__(256) void decode_kernel(const uint16_t* __restrict__ values, const uint32_t* __restrict__ metadata,
                                                     const uint32_t* __restrict__ columns, int rows, int cols, int m, int v, int ksp,
                                                     uint16_t* __restrict__ dense, uint32_t* __restrict__ bad) {
    const int ngroups = ksp >> 1;
    const int64_t n_columns = (int64_t)(rows / v) * ngroups * 4, threads = (int64_t)gridDim.x * gridDim.y * 256;
    for (int64_t i = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x; i < n_columns; i += threads)
        if (columns[i] >= (uint32_t)m) *bad = 1u;
    // (rows and columns go up to 2^31 - 1: the counters beyond the last ones need a bit more)
    const uint32_t first = (blockIdx.x * 64u + (threadIdx.x & 63u)) * 8u;
    if (first >= (uint32_t)cols) return;
    const int c0 = (int)first, stop = cols - c0 > 8 ? c0 + 8 : cols, g0 = c0 / m;
    for (int64_t row = (int64_t)blockIdx.y * 4 + (threadIdx.x >> 6); row < rows; row += (int64_t)gridDim.y * 4) {
        const int r = (int)row;
        const uint16_t* vrow = values + (int64_t)(r >> 4) * 16 * ksp + ((r >> 2) & 3) * 32 + ((r >> 1) & 1) * 4 + (r & 1) * 2;
        const uint32_t* mrow = metadata + (int64_t)(r >> 5) * (ksp >> 3) * 16 + ((r & 31) >> 1);
        const uint32_t* crow = columns + (int64_t)(r / v) * ngroups * 4;
        uint32_t out[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int g = g0; g * (int64_t)m < stop; g++) {
            const int t = g >> 2, u = g & 3;
            const uint32_t nib = (mrow[(int64_t)t * 16] >> ((r & 1) * 16 + u * 4)) & 0xfu;
            const uint32_t two = *(const uint32_t*)(vrow + (int64_t)t * 128 + u * 8);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t loc = crow[g * (int64_t)4 + ((nib >> (2 * j)) & 3u)];
                const int64_t at = (int64_t)g * m + loc - c0;
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (loc < (uint32_t)m && at == k) out[k] = j ? two >> 16 : two & 0xffffu;
            }
        }
        uint16_t* dst = dense + (int64_t)r * cols + c0;
        if ((cols & 7) == 0) {
            *(uint4*)dst = make_uint4(out[0] | (out[1] << 16), out[2] | (out[3] << 16), out[4] | (out[5] << 16), out[6] | (out[7] << 16));
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (k < cols - c0) dst[k] = (uint16_t)out[k];
        }
    }
}

hipError_t launch_decode_f16(const uint16_t* values, const uint32_t* metadata, const uint32_t* columns, int rows, int cols, int m,
                             int v, int ksp, uint16_t* dense, uint32_t* bad, hipStream_t stream) {
    const int across = (int)(((int64_t)cols + 511) / 512);
    const dim3 grid((unsigned)across, (unsigned)((rows + 3) / 4 < 65535 ? (rows + 3) / 4 : 65535)), block(256);
    hipLaunchKernelGGL(decode_kernel, grid, block, 0, stream, values, metadata, columns, rows, cols, m, v, ksp, dense, bad);
    return hipGetLastError();
}

}  // namespace spatha
