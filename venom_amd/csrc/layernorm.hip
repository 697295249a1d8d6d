// out = LayerNorm(x + residual) over the last dimension of a [tokens, hidden] fp16 matrix, in one pass over memory:
// the two elementwise kernels (addition, normalisation) that follow the attention-output and FFN-down projections of
// every encoder layer in the end-to-end models (reference harness: end2end/bert_pytorch.py:170-219 runs the stock
// BertSelfOutput / BertOutput modules, `LayerNorm(dropout(dense(h)) + input)`).
// Numerics follow the two kernels they replace: the sum is rounded to fp16 first (packed fp16 addition = one rounding of
// the exact sum), then mean, biased variance, 1/sqrt(var + eps) and the affine map are evaluated in fp32 and the result
// is rounded to fp16 once.
// The embedding of an encoder (the stock BertEmbeddings: three table rows a token, two additions, LayerNorm) is the same kernel with
// three gathered rows in place of x and the residual; its six launches took 87 us for 16384 x 1024 (lookups 27, additions 31, norm 29).
// One wave per token: a lane holds the token's 8-value chunks lane, lane + 64, ... in registers (two passes over
// registers for mean and variance, no re-read), wave-wide sums through DPP-style lane exchanges.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "spmm_kernels.h"

namespace spatha {

typedef uint32_t ln_u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 ln_half2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ ln_half2 as_half2(uint32_t w) { return __builtin_bit_cast(ln_half2, w); }
__device__ __forceinline__ uint32_t as_u32(ln_half2 h) { return __builtin_bit_cast(uint32_t, h); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// What is normalised: x + residual (may be null), row by row, or (EMB) the table rows (x[ids] + residual[types]) + third[positions], each sum
// rounded to fp16.  (Kernel arguments: what a norm needs fills one line of 64 bytes; with the embedding's behind it every norm took
// 0.2 us longer.)
struct LnArgs {
    float eps;
    int tokens, hidden;
    int out_t_pitch;             // tokens, or the next multiple of 8: the columns behind the last token are zeroed
};
struct EmbeddingArgs : LnArgs {
    const uint16_t* third;
    const int64_t *ids, *types, *positions;      // per token; per token, (types_stride 0) per position or (types_row) per position id; per position
    int64_t types_stride, types_row;             // types_row: entries of `types` where that is looked up at the position ids, else 0
    int seq;
    int64_t n_x, n_residual, n_third;            // table rows
};
template <bool EMB>
using Args = std::conditional_t<EMB, EmbeddingArgs, LnArgs>;

// an index outside its table ends the kernel, as it does in the lookups that this replaces
__device__ __forceinline__ int64_t table_row(int64_t index, int64_t rows) {
    if ((uint64_t)index >= (uint64_t)rows) __builtin_trap();
    return index;
}

template <bool EMB>
struct LnRows {
    const uint16_t *x, *residual, *third;
    __device__ __forceinline__ LnRows(const Args<EMB>& a, const uint16_t* x0, const uint16_t* residual0, int64_t token) {
        if constexpr (EMB) {
            const int64_t b = token / a.seq, s = token - b * a.seq;
            const int64_t position = a.positions[s], at = a.types_row ? table_row(position, a.types_row) : b * a.types_stride + s;
            x = x0 + table_row(a.ids[token], a.n_x) * a.hidden;
            residual = residual0 + table_row(a.types[at], a.n_residual) * a.hidden;
            third = a.third + table_row(position, a.n_third) * a.hidden;
        } else {
            x = x0 + token * a.hidden;
            residual = residual0 + token * a.hidden;         // (read only where there is one)
            third = nullptr;
        }
    }
};

__device__ __forceinline__ ln_u32x4 add_halves(ln_u32x4 a, ln_u32x4 b) {
    // (vector elements go through scalars: a bit cast applied to an indexed vector element reads element 0)
    const uint32_t p[4] = {a.x, a.y, a.z, a.w}, q[4] = {b.x, b.y, b.z, b.w};
    uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const ln_half2 t = as_half2(p[k]) + as_half2(q[k]);
        r[k] = as_u32(t);
    }
    return (ln_u32x4){r[0], r[1], r[2], r[3]};
}

// One token of `hidden` features: its 8-feature pieces lane, lane + 64, ... from `get`(j, piece), the normalised ones through `put`(piece, words).
// (get is called where a piece is converted: with the pieces fetched ahead into registers 4096 x 4096 took 17.4 us in place of 16.7)
template <int NJ, class Get, class Put>
__device__ __forceinline__ void normalise(const LnArgs& a, const uint16_t* __restrict__ gamma,
                                          const uint16_t* __restrict__ beta, int lane, Get&& get, Put&& put) {
    const int chunks = a.hidden >> 3;
    float s[NJ][8];
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        if (lane + 64 * j < chunks) {
            const ln_u32x4 in = get(j, lane + 64 * j);
            const uint32_t w[4] = {in.x, in.y, in.z, in.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const ln_half2 t = as_half2(w[k]);
                s[j][2 * k] = (float)t[0];
                s[j][2 * k + 1] = (float)t[1];
                sum += s[j][2 * k] + s[j][2 * k + 1];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) s[j][k] = 0.f;
        }
    }
    const float mean = wave_sum(sum) / (float)a.hidden;
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        if (lane + 64 * j < chunks) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float d = s[j][k] - mean;
                sq += d * d;
            }
        }
    }
    const float rstd = rsqrtf(wave_sum(sq) / (float)a.hidden + a.eps);
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int c = lane + 64 * j;
        if (c < chunks) {
            const ln_u32x4 gv = *(const ln_u32x4*)(gamma + c * 8);
            const ln_u32x4 bv = *(const ln_u32x4*)(beta + c * 8);
            const uint32_t g[4] = {gv.x, gv.y, gv.z, gv.w}, b[4] = {bv.x, bv.y, bv.z, bv.w};
            uint32_t ow[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const ln_half2 g2 = as_half2(g[k]), b2 = as_half2(b[k]);
                ln_half2 y;
                y[0] = (_Float16)((s[j][2 * k] - mean) * rstd * (float)g2[0] + (float)b2[0]);
                y[1] = (_Float16)((s[j][2 * k + 1] - mean) * rstd * (float)g2[1] + (float)b2[1]);
                ow[k] = as_u32(y);
            }
            put(c, (ln_u32x4){ow[0], ow[1], ow[2], ow[3]});
        }
    }
}

template <int NJ, bool EMB>
__global__ __launch_bounds__(256) void add_layernorm_f16_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ residual,
                                                                const uint16_t* __restrict__ gamma, const uint16_t* __restrict__ beta,
                                                                uint16_t* __restrict__ out, Args<EMB> a) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t token = (int64_t)blockIdx.x * 4 + wave;
    if (token >= a.tokens) return;
    const LnRows<EMB> rows(a, x, residual, token);
    normalise<NJ>(
        a, gamma, beta, lane,
        [&](int, int c) {
            ln_u32x4 v = *(const ln_u32x4*)(rows.x + c * 8);
            if (EMB || residual) v = add_halves(v, *(const ln_u32x4*)(rows.residual + c * 8));
            if (EMB) v = add_halves(v, *(const ln_u32x4*)(rows.third + c * 8));
            return v;
        },
        [&](int c, ln_u32x4 o) { *(ln_u32x4*)(out + token * a.hidden + c * 8) = o; });
}

// The same normalisation, written twice: row-major as above and FEATURE-MAJOR, out_t[hidden][tokens] - the layout the next
// V:N:M projection takes as its right-hand side (the reference's layer makes that copy with `x.T.contiguous()` in front of
// every SpMM, end2end/bert_pytorch.py:87, :130-134).  A workgroup of eight waves normalises TOK tokens (TOK / 8 per wave),
// leaves the fp16 results in an LDS tile [TOK][hidden + 4] (8-byte writes; the pitch of 2 (mod 64) words keeps the column
// reads below free of bank conflicts) and then writes the tile out by columns: a lane gathers the 8 tokens of one feature
// and stores them as 16 bytes, four (TOK = 32) lanes side by side covering 64 contiguous bytes of a feature's row.
template <int NJ, int TOK, bool EMB, bool XCD>
__global__ __launch_bounds__(512) void add_layernorm_f16_t_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ residual,
                                                                  const uint16_t* __restrict__ gamma, const uint16_t* __restrict__ beta,
                                                                  uint16_t* __restrict__ out, uint16_t* __restrict__ out_t, Args<EMB> a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t ln_tile[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int chunks = a.hidden >> 3;
    const int pitch = a.hidden + 4;                    // halfs
    // an XCD owns a contiguous range of tokens: adjacent pieces of a feature's row meet in its L2
    const int64_t tok0 = (XCD ? (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : (int64_t)blockIdx.x) * TOK;
    if (XCD && tok0 >= a.tokens) return;
    constexpr int PER_WAVE = TOK / 8;
    // all of the wave's tokens are fetched before the first one is reduced: 2 * PER_WAVE * NJ loads of 16 bytes in flight per lane
    ln_u32x4 xa[PER_WAVE][NJ], xb[PER_WAVE][NJ], xc[EMB ? PER_WAVE : 1][NJ];
#pragma unroll
    for (int t = 0; t < PER_WAVE; t++) {
        const int64_t token = tok0 + wave * PER_WAVE + t;
        const bool live = token < a.tokens;
        const LnRows<EMB> rows(a, x, residual, !EMB || live ? token : 0);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = lane + 64 * j;
            const ln_u32x4 zero = {0u, 0u, 0u, 0u};
            xa[t][j] = (live && c < chunks) ? *(const ln_u32x4*)(rows.x + c * 8) : zero;
            xb[t][j] = (live && c < chunks && (EMB || residual)) ? *(const ln_u32x4*)(rows.residual + c * 8) : zero;
            if (EMB) xc[EMB ? t : 0][j] = (live && c < chunks) ? *(const ln_u32x4*)(rows.third + c * 8) : zero;
        }
    }
#pragma unroll
    for (int t = 0; t < PER_WAVE; t++) {
        const int local = wave * PER_WAVE + t;
        const int64_t token = tok0 + local;
        if (token >= a.tokens) break;
        normalise<NJ>(
            a, gamma, beta, lane,
            [&](int j, int) {
                // (x + 0 would not be the identity for -0: the addition runs only with a residual)
                ln_u32x4 v = xa[t][j];
                if (EMB || residual) v = add_halves(v, xb[t][j]);
                if (EMB) v = add_halves(v, xc[EMB ? t : 0][j]);
                return v;
            },
            [&](int c, ln_u32x4 o) {
                *(ln_u32x4*)(out + token * a.hidden + c * 8) = o;
                uint32_t* dst = (uint32_t*)(ln_tile + local * pitch + c * 8);      // 8-byte aligned: pitch % 4 == 0
                *(uint2*)dst = make_uint2(o.x, o.y);
                *(uint2*)(dst + 2) = make_uint2(o.z, o.w);
            });
    }
    if (tok0 + TOK > a.tokens) {            // rows behind the last token
        for (int i = (int)(a.tokens - tok0) * pitch + threadIdx.x * 4; i < TOK * pitch; i += 512 * 4) *(uint2*)(ln_tile + i) = make_uint2(0u, 0u);
    }
    __syncthreads();
    // by columns: item = (feature f, piece p of 8 tokens)
    constexpr int PIECES = TOK / 8;
    const int items = a.hidden * PIECES;
    for (int idx = threadIdx.x; idx < items; idx += 512) {
        const int p = idx % PIECES, f = idx / PIECES;
        const int64_t token = tok0 + p * 8;
        if (token >= a.tokens) continue;                // (a piece with a token in it is all there: rows up to the pitch are zeros)
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t lo = ln_tile[(p * 8 + 2 * k) * pitch + f], hi = ln_tile[(p * 8 + 2 * k + 1) * pitch + f];
            w[k] = lo | (hi << 16);
        }
        const ln_u32x4 o = {w[0], w[1], w[2], w[3]};
        *(ln_u32x4*)(out_t + (int64_t)f * a.out_t_pitch + token) = o;
    }
}

struct LnOperands {
    const uint16_t *x, *residual, *gamma, *beta;
    uint16_t *out, *out_t;
};

template <int NJ, int TOK, bool EMB, bool XCD = false>
static hipError_t launch_ln_t(const Args<EMB>& a, const LnOperands& o, hipStream_t stream) {
    const int lds = TOK * (a.hidden + 4) * 2;
    auto kern = add_layernorm_f16_t_kernel<NJ, TOK, EMB, XCD>;
    if (lds > 48 * 1024) {
        static bool raised[16] = {};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (!raised[dev & 15]) {
            e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, TOK * (NJ * 512 + 4) * 2);
            if (e != hipSuccess) return e;
            raised[dev & 15] = true;
        }
    }
    const int blocks = (a.tokens + TOK - 1) / TOK;
    hipLaunchKernelGGL(kern, dim3(XCD ? (blocks + 7) / 8 * 8 : blocks), dim3(512), lds, stream, o.x, o.residual, o.gamma, o.beta,
                       o.out, o.out_t, a);
    return hipGetLastError();
}

// hidden <= 1024: 32 tokens per workgroup (66 KB of LDS), 16 where 32 would leave half of the CUs without one (4096 x 1024 10.9 -> 8.6 us, up
// to 1024 tokens 9.3 -> 6.5, of which 6.3 are the call; 8192 tokens level, 16384 23.2 against 25.0); <= 2048: 16; <= 4096: 8
template <bool EMB>
static hipError_t launch_norm(const Args<EMB>& a, const LnOperands& o, hipStream_t stream) {
    const int nj = (a.hidden / 8 + 63) / 64;
    if (o.out_t) {
        if (nj <= 1) return a.tokens <= 4096 ? launch_ln_t<1, 16, EMB, true>(a, o, stream) : launch_ln_t<1, 32, EMB>(a, o, stream);
        if (nj <= 2) return a.tokens <= 4096 ? launch_ln_t<2, 16, EMB, true>(a, o, stream) : launch_ln_t<2, 32, EMB>(a, o, stream);
        if (nj <= 4) return launch_ln_t<4, 16, EMB>(a, o, stream);
        return launch_ln_t<8, 8, EMB>(a, o, stream);
    }
    auto kern = nj <= 1 ? add_layernorm_f16_kernel<1, EMB> : nj <= 2 ? add_layernorm_f16_kernel<2, EMB>
                : nj <= 4 ? add_layernorm_f16_kernel<4, EMB> : add_layernorm_f16_kernel<8, EMB>;
    hipLaunchKernelGGL(kern, dim3((a.tokens + 3) / 4), dim3(256), 0, stream, o.x, o.residual, o.gamma, o.beta, o.out, a);
    return hipGetLastError();
}

hipError_t launch_add_layernorm_f16(const uint16_t* x, const uint16_t* residual, const uint16_t* gamma, const uint16_t* beta,
                                    float eps, int tokens, int hidden, uint16_t* out, uint16_t* out_t, hipStream_t stream) {
    LnArgs a = {};
    a.eps = eps; a.tokens = tokens; a.hidden = hidden; a.out_t_pitch = (tokens + 7) / 8 * 8;
    return launch_norm<false>(a, {x, residual, gamma, beta, out, out_t}, stream);
}

hipError_t launch_embed_layernorm_f16(const EmbeddingTables& t, const int64_t* ids, const int64_t* types, int64_t types_stride,
                                      int64_t types_row, const int64_t* positions, int batch, int seq, const uint16_t* gamma,
                                      const uint16_t* beta, float eps, uint16_t* out, uint16_t* out_t, hipStream_t stream) {
    EmbeddingArgs a = {};
    a.eps = eps; a.tokens = batch * seq; a.hidden = t.hidden; a.out_t_pitch = (a.tokens + 7) / 8 * 8;
    a.third = t.position;
    a.n_x = t.words; a.n_residual = t.types; a.n_third = t.positions;
    a.ids = ids; a.types = types; a.types_stride = types_stride; a.types_row = types_row; a.positions = positions; a.seq = seq;
    return launch_norm<true>(a, {t.word, t.type, gamma, beta, out, out_t}, stream);
}

}  // namespace spatha
