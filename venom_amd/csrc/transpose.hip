// out[c][r] = in[r][c] for fp16 matrices: the `dense.contiguous()` of a transposed activation that the
// PyTorch layer performs before every SpMM (reference: end2end/bert_pytorch.py:85-87, :130-134).
// A generic strided-copy kernel moves 2 bytes per lane on one side; this one moves 16 bytes per lane on
// both sides through a 64 x 64 LDS tile.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "spmm_kernels.h"

namespace spatha {

typedef uint32_t tr_u32x4 __attribute__((ext_vector_type(4)));

constexpr int TT = 64;            // tile edge
constexpr int TP = TT + 2;        // LDS pitch in halfs (odd number of 32-bit words: conflict-free column reads)

__global__ __launch_bounds__(256) void transpose_f16_kernel(const uint16_t* __restrict__ in, int rows, int cols,
                                                            uint16_t* __restrict__ out, int pitch) {
    __shared__ uint16_t tile[TT * TP];
    const int tid = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.y * TT, c0 = (int64_t)blockIdx.x * TT;
    const bool vec_in = (cols % 8 == 0), vec_out = (pitch % 8 == 0);
    // load: 8 lanes x 16 B per row, 32 rows per pass
#pragma unroll
    for (int pass = 0; pass < 2; pass++) {
        const int r = pass * 32 + (tid >> 3), c = (tid & 7) * 8;
        uint16_t v[8];
        if (r0 + r < rows) {
            const uint16_t* src = in + (r0 + r) * cols + c0 + c;
            if (vec_in && c0 + c + 8 <= cols) {
                *(tr_u32x4*)v = *(const tr_u32x4*)src;
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = (c0 + c + k < cols) ? src[k] : (uint16_t)0;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = 0;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) tile[r * TP + c + k] = v[k];
    }
    __syncthreads();
    // store: output row = input column; 8 lanes x 16 B per output row
#pragma unroll
    for (int pass = 0; pass < 2; pass++) {
        const int c = pass * 32 + (tid >> 3), r = (tid & 7) * 8;
        if (c0 + c >= cols) continue;
        uint16_t v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = tile[(r + k) * TP + c];
        uint16_t* dst = out + (c0 + c) * pitch + r0 + r;
        if (vec_out && r0 + r + 8 <= pitch) {        // (rows beyond the matrix are zeros in the tile)
            *(tr_u32x4*)dst = *(const tr_u32x4*)v;
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (r0 + r + k < pitch) dst[k] = v[k];
        }
    }
}

// out[c][r], rows of `pitch` entries (rows <= pitch, and below the next multiple of 8 where that is not rows itself): zeros behind
// the last column, so that a ragged activation arrives in the 16-byte row pieces that the SpMM reads
hipError_t launch_transpose_f16(const uint16_t* in, int rows, int cols, uint16_t* out, int pitch, hipStream_t stream) {
    dim3 grid((cols + TT - 1) / TT, (rows + TT - 1) / TT);
    hipLaunchKernelGGL(transpose_f16_kernel, grid, dim3(256), 0, stream, in, rows, cols, out, pitch);
    return hipGetLastError();
}

namespace {
struct __attribute__((packed, aligned(2))) Unaligned16 {
    tr_u32x4 v;
};
}  // namespace

// out[r][c] = in[r][c] for c < cols, rows in_pitch and out_pitch apart.  PAD: zeros from cols to out_pitch, a multiple of 8 (the padded copy of
// a right-hand side whose column count is no multiple of 8); else in_pitch is one, and the ragged rows of a result are cut out.  A
// thread takes one 16-byte piece, and the ragged side goes by one access at whatever alignment its row has.  Bound by launch and
// latency at most sizes: 1280 x 1037 2.85 us padded, 3.1 with two rows a thread, of which an empty launch is 2.4; cutting 3072 x 2785
// 7.5 us, 9.6 as a strided copy.
// Index counts pieces: 32 bits wherever they suffice, a 64-bit division by a variable is a subroutine.
template <bool PAD, typename Index>
__global__ __launch_bounds__(256) void repitch_f16_kernel(const uint16_t* __restrict__ in, int rows, int cols, int in_pitch,
                                                          uint16_t* __restrict__ out, int out_pitch) {
    const uint32_t pieces = (uint32_t)(cols + 7) >> 3;
    const Index total = (Index)rows * pieces;
    for (Index id = (Index)blockIdx.x * 256 + threadIdx.x; id < total; id += (Index)gridDim.x * 256) {
        const uint32_t r = (uint32_t)(id / pieces);
        const int c = (int)(id - (Index)r * pieces) * 8;
        const uint16_t* src = in + (int64_t)r * in_pitch + c;
        uint16_t* dst = out + (int64_t)r * out_pitch + c;
        tr_u32x4 v;
        if (!PAD) {
            v = *(const tr_u32x4*)src;
        } else if (c + 8 <= cols) {
            v = ((const Unaligned16*)src)->v;
        } else {
            uint16_t e[8];
#pragma unroll
            for (int i = 0; i < 8; i++) e[i] = c + i < cols ? src[i] : (uint16_t)0;
            v = (tr_u32x4){e[0] | ((uint32_t)e[1] << 16), e[2] | ((uint32_t)e[3] << 16), e[4] | ((uint32_t)e[5] << 16),
                           e[6] | ((uint32_t)e[7] << 16)};
        }
        if (PAD) {
            *(tr_u32x4*)dst = v;
        } else if (c + 8 <= cols) {
            ((Unaligned16*)dst)->v = v;
        } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (c + i < cols) dst[i] = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
        }
    }
}

template <bool PAD>
static hipError_t launch_repitch(const uint16_t* in, int rows, int cols, int in_pitch, uint16_t* out, int out_pitch, hipStream_t stream) {
    const int64_t pieces = (int64_t)rows * ((cols + 7) / 8), blocks = (pieces + 255) / 256;
    const unsigned grid = (unsigned)(blocks < 65535 * 8 ? blocks : 65535 * 8);
    // (a thread's next piece must not wrap either: a stride of 2^27 pieces at most below 2^31)
    auto kern = pieces < (1ll << 31) ? repitch_f16_kernel<PAD, uint32_t> : repitch_f16_kernel<PAD, uint64_t>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, stream, in, rows, cols, in_pitch, out, out_pitch);
    return hipGetLastError();
}
hipError_t launch_pad_columns_f16(const uint16_t* in, int rows, int cols, uint16_t* out, int pitch, hipStream_t stream) {
    return launch_repitch<true>(in, rows, cols, cols, out, pitch, stream);
}
hipError_t launch_cut_columns_f16(const uint16_t* in, int rows, int cols, int pitch, uint16_t* out, hipStream_t stream) {
    return launch_repitch<false>(in, rows, cols, pitch, out, cols, stream);
}

}  // namespace spatha
