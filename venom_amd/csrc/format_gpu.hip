// V:N:M decoding on the GPU: the same entries in the same places as the host builder (vnm_format.cpp, which holds the storage map), to
// matrices that live in device memory (to_dense / func3, end2end/grouped_nmv_tensor.py:563-675).  The kernel only moves data; one
// thread owns eight adjacent entries of a dense row, so that the dense side is written in whole words.
// 1024 x 4096 at 128:2:16: 6.8 us (a call of to_dense 27-30 us, most of it the wait for the flag of the offset check; 870 us when the
// arrays were decoded on the host).

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "spmm_kernels.h"

namespace spatha {

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

hipError_t launch_decode_f16(const uint16_t* values, const uint32_t* metadata, const uint32_t* columns, int rows, int cols, int m,
                             int v, int ksp, uint16_t* dense, uint32_t* bad, hipStream_t stream) {
    const dim3 grid(blocks_for((int64_t)rows * ((cols + 7) / 8))), block(256);
    hipLaunchKernelGGL(decode_kernel, grid, block, 0, stream, values, metadata, columns, rows, cols, m, v, ksp, dense, bad);
    return hipGetLastError();
}

}  // namespace spatha
