// Attention of an encoder layer, softmax(scale Q K^T) V over every sequence and head of a batch, without a mask, for heads of 64
// features: what the models' attention modules compute between the query / key / value projections and the output projection
// (reference harness: end2end/bert_pytorch.py:170-219 runs the stock module).  The result is written feature-major, the layout
// that the output projection reads as its right-hand side, so that no transposed copy of it is made.
//
// A workgroup takes 128 queries of one head, 32 per wave, and walks the keys 64 at a time: K and V rows come into LDS by DMA, two
// buffers, one barrier a tile.  The wave multiplies S^T = K Q^T (v_mfma_f32_32x32x16_f16): a lane holds one query's scores of 32
// keys, so the row maximum and sum are in-lane but for one exchange between the wave's halves, and the probabilities are the
// other product's operand as they lie: O^T = V^T P^T takes the keys of a 16-key step in the order in which S^T leaves them (0-3,
// 8-11 in the lower lanes, 4-7, 12-15 in the upper ones), and two transposing LDS reads fetch V in that same order.  Scores,
// maxima, exponentials, sums and the output are fp32; probabilities are rounded to fp16 for the second product, as in the kernel
// that this replaces.  (The running maximum follows every new maximum: letting it lag by up to 2^8 spares most rescalings of O, but
// the largest probability is then no longer exactly one, and at 512 keys the result was 6 % further from the exact one.)
//
// What bounds it: vector instructions, 20 clocks of a SIMD per 64 scores (exponential 8, fma, addition 3 each, maximum and rounding
// about 2.3 each) against 16 of matrix instructions, which the other waves of the SIMD issue meanwhile.

#include <algorithm>

#include "spmm_device.h"

namespace spatha {

typedef float float16_t __attribute__((ext_vector_type(16)));

namespace {
constexpr int kKeys = 64, kQueries = 128, kHead = 64;
constexpr int kRowBytes = kHead * 2, kTileBytes = kKeys * kRowBytes;
constexpr int kOutPitch = kQueries + 8;          // halfs between two features of the finished tile in LDS

__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32, 64); }

// values of the keys behind a sequence's end (they have probability zero, and zero times an infinity is NaN)
__device__ const uint4 kNoValues = {0u, 0u, 0u, 0u};
}  // namespace

struct AttentionParams {
    const uint16_t *q, *k, *v;      // [batch * seq] rows, `pitch` halfs apart; head h at column 64 h
    uint16_t* out;                  // [heads * 64][out_pitch], column = token
    int64_t pitch, out_pitch;
    int seq, heads, groups, q_tiles;     // groups = batch * heads
    int pad;                        // columns behind the last token, below eight, that are set to zero
    float scale_log2;               // scale * log2(e)
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void attention_kernel(AttentionParams p) {
    __shared__ __attribute__((aligned(16))) char smem[4 * kTileBytes];      // K, V, K, V; then the finished tile
    static_assert(kHead * kOutPitch * 2 <= 4 * kTileBytes, "the finished tile fits");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the query tiles of a head on one XCD: its L2 reads K and V once
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int group = (local / p.q_tiles) * 8 + xcd, q_tile = local % p.q_tiles;
    if (group >= p.groups) return;
    const int batch = group / p.heads, head = group - batch * p.heads;
    const int seq = p.seq, tiles = (seq + kKeys - 1) / kKeys;
    const int64_t token0 = (int64_t)batch * seq;
    const uint16_t* k_base = p.k + token0 * p.pitch + head * kHead;
    const uint16_t* v_base = p.v + token0 * p.pitch + head * kHead;
    const uint32_t smem_base = (uint32_t)(uintptr_t)LDS_PTR(char, smem);
    const int half = lane >> 5, col = lane & 31;

    // a DMA instruction brings eight rows; 16-byte piece c of row r goes to place c ^ (r % 8) (whole rows are what lanes read at once)
    const int dma_row = lane >> 3, dma_piece = (lane & 7) ^ dma_row;
    auto load_tile = [&](int t) {
        const uint32_t dst = smem_base + (t & 1) * 2 * kTileBytes;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = wave * 16 + i * 8, key = t * kKeys + row + dma_row;
            const int64_t at = (int64_t)(key < seq ? key : seq - 1) * p.pitch + dma_piece * 8;
            dma_b128(k_base + at, dst + row * kRowBytes);
            dma_b128(key < seq ? (const void*)(v_base + at) : (const void*)&kNoValues, dst + kTileBytes + row * kRowBytes);
        }
    };
    load_tile(0);

    const int query = q_tile * kQueries + wave * 32 + col;
    const bool wave_on = q_tile * kQueries + wave * 32 < seq;
    half8_t q[4];
    {
        const uint16_t* src = p.q + (token0 + (query < seq ? query : seq - 1)) * p.pitch + head * kHead + half * 8;
#pragma unroll
        for (int s = 0; s < 4; s++) q[s] = *(const half8_t*)(src + s * 16);
    }
    int k_off[4], v_off[2];
#pragma unroll
    for (int s = 0; s < 4; s++) k_off[s] = col * kRowBytes + ((2 * s + half) ^ (lane & 7)) * 16;
    {
        const int e = 4 * half + ((lane & 15) >> 2);
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
            v_off[mb] = kTileBytes + e * kRowBytes + ((mb * 4 + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) ^ e) * 16 + (lane & 1) * 8;
    }
    float16_t o[2];
#pragma unroll
    for (int mb = 0; mb < 2; mb++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[mb][i] = 0.f;
    // of the scaled scores (in powers of two; finite from the start, so that a first tile of scores -inf adds exp2(-inf) = 0); this lane's
    // share of the sum
    float peak = -__FLT_MAX__, sum = 0.f;
    const float c = p.scale_log2;

    for (int t = 0; t < tiles; t++) {
        wait_vmcnt<0>();
        __syncthreads();            // tile t is there, tile t - 1 has been read
        if (t + 1 < tiles) load_tile(t + 1);
        if (!wave_on) continue;
        const char* st = smem + (t & 1) * 2 * kTileBytes;
        float16_t s[2];
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[kb][i] = 0.f;
#pragma unroll
            for (int d = 0; d < 4; d++)
                s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const half8_t*)(st + kb * 32 * kRowBytes + k_off[d]), q[d], s[kb], 0, 0, 0);
        }
        if (t == tiles - 1 && seq % kKeys) {
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (t * kKeys + kb * 32 + (i & 3) + 8 * (i >> 2) + 4 * half >= seq) s[kb][i] = -__builtin_inff();
        }
        float top = s[0][0];
#pragma unroll
        for (int i = 1; i < 32; i++) top = fmaxf(top, s[i >> 4][i & 15]);
        top = fmaxf(top, other_half(top)) * c;
        if (__any(top > peak)) {
            const float now = fmaxf(peak, top), fade = __builtin_amdgcn_exp2f(peak - now);
            peak = now;
            sum *= fade;
#pragma unroll
            for (int mb = 0; mb < 2; mb++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[mb][i] *= fade;
        }
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            half8_t prob[2];
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float e = __builtin_amdgcn_exp2f(fmaf(s[kb][i], c, -peak));
                sum += e;
                prob[i >> 3][i & 7] = (_Float16)e;
            }
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int mb = 0; mb < 2; mb++) {
                    const char* src = st + v_off[mb] + (kb * 32 + ks * 16) * kRowBytes;
                    const half4_t lo = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4_t, src)));
                    const half4_t hi = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(short4_t, src + 8 * kRowBytes)));
                    const half8_t vt = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    o[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vt, prob[ks], o[mb], 0, 0, 0);
                }
        }
    }
    __syncthreads();        // the last tile has been read
    uint16_t* tile = (uint16_t*)smem;
    if (wave_on) {
        sum += other_half(sum);
        const float inverse = 1.f / sum;
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const _Float16 h = (_Float16)(o[mb][i] * inverse);
                tile[(mb * 32 + (i & 3) + 8 * (i >> 2) + 4 * half) * kOutPitch + wave * 32 + col] = __builtin_bit_cast(uint16_t, h);
            }
    }
    __syncthreads();
    struct __attribute__((packed, aligned(2))) Piece { u32x4 v; };        // (a sequence may start at any token)
    uint16_t* out = p.out + (int64_t)head * kHead * p.out_pitch + token0;
    const bool last = token0 + seq == (int64_t)p.groups / p.heads * seq && q_tile == p.q_tiles - 1;
    const int limit = last ? seq + p.pad : seq, pieces = kQueries / 8 + (last ? 1 : 0);
    for (int i = tid; i < kHead * pieces; i += 256) {
        const int f = i / pieces, x = (i - f * pieces) * 8, first = q_tile * kQueries + x;
        const uint16_t* src = tile + f * kOutPitch + x;
        uint16_t* dst = out + (int64_t)f * p.out_pitch + first;
        if (first + 8 <= seq && x < kQueries) {
            ((Piece*)dst)->v = *(const u32x4*)src;
        } else if (x < kQueries || last) {
            for (int j = 0; first + j < limit && j < 8; j++) dst[j] = first + j < seq ? src[j] : (uint16_t)0;
        }
    }
}

hipError_t launch_attention_f16(const uint16_t* q, const uint16_t* k, const uint16_t* v, int64_t pitch, int batch, int seq, int heads,
                                float scale, uint16_t* out, int64_t out_pitch, hipStream_t stream) {
    const int64_t tokens = (int64_t)batch * seq;
    AttentionParams p = {};
    p.q = q; p.k = k; p.v = v; p.out = out;
    p.pitch = pitch; p.out_pitch = out_pitch;
    p.seq = seq; p.heads = heads; p.groups = batch * heads;
    p.q_tiles = (seq + kQueries - 1) / kQueries;
    p.pad = (int)std::min<int64_t>((8 - tokens % 8) % 8, out_pitch - tokens);
    p.scale_log2 = scale * 1.44269504088896340736f;
    const int64_t grid = (int64_t)(p.groups + 7) / 8 * 8 * p.q_tiles;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(attention_kernel, dim3((unsigned)grid), dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace spatha
