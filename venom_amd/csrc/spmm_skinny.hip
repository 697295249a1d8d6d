// Kernels without LDS staging of the operands: few columns of B (N <= 64), and small products of any width.

#include "spmm_device.h"

namespace spatha {

// ---------------------------------------------------------------------------
// One workgroup per 64-row tile (32 rows where V is a multiple of 32 only: half of a packed 64-row block, which is all that one
// gathered set of B rows serves) and 16 * NB columns; its W waves split the k-steps (wave w takes steps w, w + W, ...) and add
// their fp32 partial tiles through LDS at the end in a fixed order.  No LDS staging of B: a lane fetches the 16 elements of its
// B fragment straight from global memory through a buffer descriptor whose bounds check returns the zeros of padding rows and
// of columns beyond N.  Operands of a wave's next step and the row table of the one after are requested before a step is
// multiplied.
// NB = 1, 2 or 4 column blocks of 16.  Column block nb holds the columns NB * j + nb (j = 0 .. 15), not 16 * nb + j: lane j of
// a block then needs NB ADJACENT columns of every gathered row, one load of 2 * NB bytes instead of NB loads of 2 bytes - 16
// vector-memory instructions per k-step whatever NB.  N is a multiple of 8, so the NB columns of a lane lie all inside N or all
// outside; RAGGED: any N, B (rows b_pitch apart) and C addressed at whatever alignment their rows have, so that a ragged token count
// needs no padded copies (spatha_spmm_run_ragged: 4096 x 1024 at 64:2:8 and 301 tokens with GELU, row-major, 9.5 us, 23.0 with a
// launch for each copy).  Instances of their own: one for all counts took 2-5 % longer at multiples of 8 (768 x 3072 x 760 at 128:2:8
// 8.7 -> 8.9 us, 768 x 768 x 48 at 64:2:40 3.1 -> 3.3).
// What bounds it: with few tiles the trip to memory that a k-step's loads take (four waves a tile left 16 .. 192 of 256 CUs with
// one wave per SIMD and fewer than two steps in flight: 12288 x 12288 at 64:2:8 and 8 tokens 25.1 us for 101 MB; sixteen waves:
// 16.0); with many, the 12.8 KB of loads per 64 x 64 block and k-step through the L1 (0.8-1.2 ns a block and step over the chip).
// It has no pipeline to fill and no stage to share, so small products end sooner than on the staged tiles: 1024 x 4096 at
// 64:2:16 and 304 tokens 5.0 us (64 x 256 tiles 14.4), 1280 x 5120 at 32:2:16 and 304 tokens 6.2 us (staged half tiles 24.7).
// ---------------------------------------------------------------------------
// LEAN (four column blocks only): see the main loop.  (The lean form is compiled for three waves per SIMD - three workgroups
// of four waves per CU - which it reaches with 158 registers.)
// halfs between two tokens in LDS: odd in 32-bit words, so that the sixteen tokens of a fragment row sit on different banks
__host__ __device__ constexpr int token_pitch_halfs(int cols) { return (((cols + 7) / 8 * 4) | 1) * 2; }

// adjacent columns of C; ANYWHERE: at whatever alignment
template <bool ANYWHERE, class Columns>
__device__ __forceinline__ void store_columns(uint16_t* dst, Columns v) {
    struct __attribute__((packed, aligned(2))) Piece { Columns v; };
    if (ANYWHERE) ((Piece*)dst)->v = v;
    else *(Columns*)dst = v;
}

template <int NB, int W, bool HALF, bool LEAN>
struct DirectCfg {
    static constexpr int MB = HALF ? 2 : 4;                                     // instruction-row blocks per tile
    // partial tiles are added up PB row blocks at a time, CB adjacent columns per lane
    static constexpr int LDS_KB = LEAN ? 32 : 64;
    static constexpr int PB = W * MB * NB <= LDS_KB ? MB : W * 2 * NB <= LDS_KB ? 2 : 1;
    static constexpr int CB = W > 4 && NB > 2 ? 2 : NB;
    static constexpr int UNITS = PB * (NB / CB);
    static constexpr int WAVES_PER_EU = NB == 4 ? (LEAN || HALF ? 3 : 2) : NB == 2 ? 3 : 4;
    static_assert(W * PB * NB <= 64, "partial tiles exceed 64 KB");
};

template <int NB, int OUT_LAYOUT, int W, bool HALF, bool LEAN, bool TOKEN_MAJOR, bool RAGGED>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu((DirectCfg<NB, W, HALF, LEAN>::WAVES_PER_EU))))
void spmm_direct_kernel(SpmmParams p) {
    using Cfg = DirectCfg<NB, W, HALF, LEAN>;
    constexpr int MB = Cfg::MB, PB = Cfg::PB, CB = Cfg::CB;
    static_assert(NB == 1 || NB == 2 || NB == 4, "column blocks per tile");
    typedef float4_t Red[PB][NB][64];
    __shared__ Red fixed_red[TOKEN_MAJOR ? 1 : W];
    extern __shared__ __attribute__((aligned(16))) char dyn[];      // TOKEN_MAJOR: the tokens, then the partial tiles
    Red* red = TOKEN_MAJOR ? (Red*)dyn : fixed_red;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = p.S, N = p.N;
    int b_pitch = RAGGED ? p.b_pitch : N;
    uint32_t b_bytes = p.b_bytes;
    // (read at the start: left to the compiler, the first load of B waits for them, 0.1 us)
    if constexpr (RAGGED) asm volatile("" : "+s"(b_pitch), "+s"(b_bytes));
    // an XCD owns a contiguous range of tiles, row tile after row tile (the packed A of a row tile enters one L2 only) or, with
    // walk_group 1, column tile after column tile (the same for a column of B)
    const int tiles = p.tiles_m * p.tiles_n, chunk = (tiles + 7) >> 3;
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, id = xcd * chunk + local;
    if (local >= chunk || id >= tiles) return;
    const int minor = p.walk_group ? p.tiles_m : p.tiles_n, major = id / minor;
    const int tile = p.walk_group ? id - major * minor : major, tile_n = p.walk_group ? major : id - major * minor;
    const int half = HALF ? tile & 1 : 0;
    const int64_t block = HALF ? tile >> 1 : tile;                              // packed 64-row block
    const int li = lane & 15, kb = lane >> 4;
    const int64_t vb = ((int64_t)tile * (16 * MB)) / p.v;
    const char* a_tile = (const char*)p.apack + block * S * APACK_BLOCK;
    const uint32_t* rt_block = p.rowtab + vb * S * 64;
    __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)p.B, 0, (int)b_bytes, 0x00020000);
    const uint32_t row_bytes = (uint32_t)b_pitch * 2u;

    float4_t acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[a][b] = (float4_t){0.f, 0.f, 0.f, 0.f};

    struct Set {
        half8_t a[MB];
        uint32_t ix[MB / 2];
    };
    auto load_rt = [&](int st, u32x4 (&rt)[4]) {
        const uint32_t* q = rt_block + (int64_t)st * 64 + 4 * kb;
#pragma unroll
        for (int fb = 0; fb < 4; fb++) rt[fb] = *(const u32x4*)(q + 16 * fb);
    };
    auto load_a = [&](int st, Set& x) {
        const char* q = a_tile + (int64_t)st * APACK_BLOCK;
#pragma unroll
        for (int mb = 0; mb < MB; mb++) x.a[mb] = *(const half8_t*)(q + (half * 2 + mb) * 1024 + lane * 16);
#pragma unroll
        for (int d = 0; d < MB / 2; d++) x.ix[d] = *(const uint32_t*)(q + 4096 + (half + d) * 256 + lane * 4);
    };
    // This lane's NB columns, col0 + nb.  Where ragged rows of B have no padding that the last lane's could reach into, that lane moves down.
    const int lane_col = (tile_n * 16 + li) * NB;
    const int col0 = RAGGED && b_pitch % NB != 0 && lane_col > N - NB ? N - NB : lane_col;
    // (lanes beyond a ragged N fetch nothing in groups of four; single ones fetch what the last lane does: four lanes of which some are out
    // of the descriptor's range take the load a third longer - 49152 x 12288 at 64:2:4 and 18 tokens 170 against 132 us)
    const bool fetches = lane_col < (N + 4 * NB - 1) / (4 * NB) * (4 * NB), stores = lane_col < N;
    const uint32_t fetch_col = (uint32_t)(!RAGGED || lane_col < N ? col0 : b_pitch % NB != 0 ? N - NB : (N - 1) / NB * NB);
    const int token_pitch = token_pitch_halfs(p.cols);
    if constexpr (TOKEN_MAJOR) {
        // x [N][cols] -> LDS as it lies; columns N .. 15 of the tile are never stored, they multiply token 0
        const int pieces = (p.cols + 7) >> 3;
        for (int i = tid; i < N * pieces; i += W * 64) {
            const int t = i / pieces, c = (i - t * pieces) * 8;
            const uint16_t* src = p.B + (int64_t)t * p.cols + c;
            uint32_t* dst = (uint32_t*)((uint16_t*)dyn + t * token_pitch + c);       // 4-byte aligned: the pitch is even
            if ((p.cols & 7) == 0) {
                const u32x4 v = *(const u32x4*)src;
#pragma unroll
                for (int k = 0; k < 4; k++) dst[k] = v[k];
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (c + k < p.cols) ((uint16_t*)dst)[k] = src[k];
            }
        }
        __syncthreads();
    }
    const uint16_t* token = (const uint16_t*)dyn + (li < N ? li : 0) * token_pitch;
    auto load_b = [&](const u32x4 (&rt)[4], half16_t (&bf)[NB]) {
#pragma unroll
        for (int fb = 0; fb < 4; fb++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t row = rt[fb][j];
                if constexpr (TOKEN_MAJOR) {
                    const uint16_t h = token[row != 0xFFFFFFFFu ? row : 0u];
                    bf[0][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)(row != 0xFFFFFFFFu ? h : 0));
                    continue;
                }
                const uint32_t voff = (row != 0xFFFFFFFFu && (RAGGED ? fetches : col0 < N)) ? row * row_bytes + fetch_col * 2u : 0xF0000000u;
                if constexpr (NB == 1) {
                    const uint16_t h = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc_b, (int)voff, 0, 0);
                    bf[0][fb * 4 + j] = __builtin_bit_cast(_Float16, h);
                } else if constexpr (NB == 2) {
                    const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, (int)voff, 0, 0);
                    bf[0][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)w);
                    bf[1][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
                } else {
                    const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(rsrc_b, (int)voff, 0, 0);
                    bf[0][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)w.x);
                    bf[1][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)(w.x >> 16));
                    bf[2][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)w.y);
                    bf[3][fb * 4 + j] = __builtin_bit_cast(_Float16, (uint16_t)(w.y >> 16));
                }
            }
    };
    auto multiply = [&](const Set& x, const half16_t (&b)[NB]) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                if (mb & 1) acc[mb][nb] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(x.a[mb], b[nb], acc[mb][nb], (int)x.ix[mb >> 1], 0, 1);
                else acc[mb][nb] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(x.a[mb], b[nb], acc[mb][nb], (int)x.ix[mb >> 1], 0, 0);
            }
    };
    // (every condition below is uniform over the wave: `wave` and S sit in scalar registers)
    auto clamp_step = [&](int s) { return s < S ? s : S - 1; };
    int st = wave;
    if (st < S) {
        if constexpr (!LEAN) {
            u32x4 rt1[4], rt2[4];
            Set x0, x1;
            half16_t b0[NB], b1[NB];
            load_rt(st, rt1);
            load_a(st, x0);
            load_b(rt1, b0);
            load_rt(clamp_step(st + W), rt1);
            for (; st + W < S; st += W) {
                load_rt(clamp_step(st + 2 * W), rt2);
                load_a(st + W, x1);
                load_b(rt1, b1);
                multiply(x0, b0);
                x0 = x1;
#pragma unroll
                for (int k = 0; k < 4; k++) rt1[k] = rt2[k];
#pragma unroll
                for (int nb = 0; nb < NB; nb++) b0[nb] = b1[nb];
            }
            multiply(x0, b0);
        } else {
            // Four column blocks with every operand double-buffered need 192 registers: two workgroups per CU.  With more than two
            // 64-row tiles per CU (GPT-3 FFN matrix: three) this form runs instead: only B is double-buffered, the A operands and
            // the row table of the next step are requested behind this step's matrix instructions, into the registers those have
            // just read; three workgroups per CU, whose loads cover one another's waits (38 against 40.5 us there; with one tile
            // per CU or less and long k-loops it is the slower form, 33.5 against 31.2 us on 12288 x 12288 at 64:2:8; with a wave's
            // share of the k-loop at four steps or less its shorter prologue wins again: 5.4 against 5.7 us on 4096 x 1024).
            u32x4 rt1[4];
            Set x;
            half16_t b0[NB], b1[NB];
            load_rt(st, rt1);
            load_a(st, x);
            load_b(rt1, b0);
            load_rt(clamp_step(st + W), rt1);
            for (; st + W < S; st += W) {
                load_b(rt1, b1);
                multiply(x, b0);
                load_a(st + W, x);
                load_rt(clamp_step(st + 2 * W), rt1);
#pragma unroll
                for (int nb = 0; nb < NB; nb++) b0[nb] = b1[nb];
            }
            multiply(x, b0);
        }
    }
    if constexpr (TOKEN_MAJOR) __syncthreads();      // the tokens have been read: the partial tiles take their place
    // Unit u of a pass: row block mb = pass + u % PB (rows 16 * ib + 4 * mb + r of a 64-row tile, 8 * ib + 4 * mb + r of a 32-row
    // one), columns col0 + (u / PB) * CB + c
    const int ib = kb;
#pragma unroll
    for (int pass = 0; pass < MB; pass += PB) {
        if (pass) __syncthreads();      // the pass before has been read
#pragma unroll
        for (int pb = 0; pb < PB; pb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++) red[wave][pb][nb][lane] = acc[pass + pb][nb];
        __syncthreads();
        for (int u = wave; u < Cfg::UNITS; u += W) {
            const int pb = u % PB, nb0 = (u / PB) * CB, mb = pass + pb;
            const int64_t row0 = (int64_t)tile * (16 * MB) + (HALF ? 8 : 16) * ib + 4 * mb;
            half4_t h4[CB];
            half4_t bias4 = {(_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
            if (p.bias) bias4 = *(const half4_t*)(p.bias + row0);
#pragma unroll
            for (int c = 0; c < CB; c++) {
                float4_t sum = red[0][pb][nb0 + c][lane];
#pragma unroll
                for (int w = 1; w < W; w++) sum = sum + red[w][pb][nb0 + c][lane];
#pragma unroll
                for (int r = 0; r < 4; r++) h4[c][r] = (_Float16)sum[r];
                if (OUT_LAYOUT == SPATHA_OUT_TRANSPOSED || p.fuse) h4[c] = p.bias ? h4[c] + bias4 : h4[c];
            }
            if (p.act == SPATHA_ACT_GELU) {
#pragma unroll
                for (int c = 0; c < CB; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) h4[c][r] = (_Float16)act_gelu_erf((float)h4[c][r]);
            } else if (p.act == SPATHA_ACT_GELU_TANH) {
#pragma unroll
                for (int c = 0; c < CB; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) h4[c][r] = (_Float16)act_gelu_tanh((float)h4[c][r]);
            }
            const int col = col0 + nb0;
            if ((RAGGED ? !stores : col >= N) || SPATHA_KNOB(2)) continue;
            if (OUT_LAYOUT == SPATHA_OUT_TRANSPOSED) {
#pragma unroll
                for (int c = 0; c < CB; c++)
                    if (!RAGGED || CB == 1 || col + c < N) *(half4_t*)(p.C + (int64_t)(col + c) * p.rows + row0) = h4[c];
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    uint16_t* dst = p.C + (row0 + r) * N + col;
                    if constexpr (CB == 1) {
                        *(_Float16*)dst = h4[0][r];
                    } else if (!RAGGED || col + CB <= N) {
                        if constexpr (CB == 4) store_columns<RAGGED>(dst, (half4_t){h4[0][r], h4[1][r], h4[2][r], h4[3][r]});
                        else store_columns<RAGGED>(dst, (half2_t){h4[0][r], h4[1][r]});
                    } else {
#pragma unroll
                        for (int c = 0; c < CB; c++)
                            if (col + c < N) *((_Float16*)dst + c) = h4[c][r];
                    }
                }
            }
        }
    }
}

template <int NB, int OUT_LAYOUT, int W, bool HALF, bool LEAN = false>
static hipError_t launch_direct(SpmmParams p, hipStream_t stream) {
    p.tiles_m = p.rows / (HALF ? 32 : 64);
    p.tiles_n = (p.N + 16 * NB - 1) / (16 * NB);
    // The operand whose tiles are walked inside the other's enters every L2: the smaller one.  (1024 x 4096 x 2048 at 32:2:16, A 1.2 MB,
    // B 17 MB: 13.4 us column after column, 20.7 row after row; 1280 x 5120 x 104 at 64:2:8, A 3.7, B 1.1 MB: 8.9 against 7.2.)
    p.walk_group = p.b_bytes > p.apack_bytes ? 1 : 0;
    const int tiles = p.tiles_m * p.tiles_n;
    auto kern = p.N % 8 == 0 && p.b_pitch == p.N ? spmm_direct_kernel<NB, OUT_LAYOUT, W, HALF, LEAN, false, false>
                                                 : spmm_direct_kernel<NB, OUT_LAYOUT, W, HALF, LEAN, false, true>;
    hipLaunchKernelGGL(kern, dim3((tiles + 7) / 8 * 8), dim3(W * 64), 0, stream, p);
    return hipGetLastError();
}

// Columns (16 * nb) and waves per tile
struct DirectForm {
    int nb, w;
    bool lean;
};

static DirectForm direct_form(int rows, int N, int S, bool half, int64_t cus) {
    // The narrowest tile whose tiles still find a CU each, its k-steps over as many waves as they
    // feed; with more tiles than CUs fewer waves, so that several workgroups share a CU.  (Every form on ten layer shapes from
    // 768 x 3072 to 49152 x 12288, V = 32 / 64 / 128, m = 8 / 16 / 32, 8 .. 2048 tokens, both layouts: this choice is 1.1 %
    // behind the best form on the geometric mean.  12288 x 49152 at 128:2:16 and 8 tokens, 192 tiles of 192 k-steps: 28.8 us
    // with sixteen waves, 50.3 with four; 1024 x 4096 at 64:2:16 and 512 tokens: 5.2 us on 64 x 32 tiles of eight waves, 6.4 on
    // 64 x 64 ones.)
    const int64_t rows_tiles = rows / (half ? 32 : 64);
    auto tiles = [&](int nb) { return rows_tiles * ((N + 16 * nb - 1) / (16 * nb)); };
    DirectForm f = {1, 4, false};
    if (tiles(1) <= cus) {
        f.w = S > 12 ? 16 : S > 4 || N > 16 ? 8 : 4;
    } else if (N <= 16) {
        f.w = tiles(1) <= 2 * cus && S > 4 ? 8 : 4;
    } else if (tiles(2) <= cus) {
        f.nb = 2;
        f.w = S > 4 ? 8 : 4;
    } else if (N <= 32 || (S <= 4 && tiles(2) <= 3 * cus)) {
        f.nb = 2;
    } else {
        f.nb = 4;
        // (eight waves against four at 130 .. 256 tiles, 1080 products, both layouts: 64-row tiles 0.90-0.98 of the speed at five to
        // fourteen k-steps, 0.97-1.00 at sixteen, 1.03-1.06 at twenty, 1.13 at 48, whatever the number of tiles; 32-row tiles 0.95-1.03
        // up to eight, 1.02 at ten, 1.01-1.06 at fourteen, 1.16 at 48)
        if (tiles(4) <= cus && S > (half ? 8 : 16)) f.w = 8;
        f.lean = f.w == 4 && tiles(4) > cus && (S > 2 || tiles(4) > 2 * cus);
    }
    return f;
}

// place of a form in the tables below, < 0: not compiled
static int form_index(const DirectForm& f) {
    switch (f.nb * 100 + f.w) {
        case 104: return 0;
        case 108: return 1;
        case 116: return 2;
        case 204: return 3;
        case 208: return 4;
        case 404: return f.lean ? 6 : 5;
        case 408: return 7;
        default: return -1;
    }
}

template <int OUT_LAYOUT, bool HALF>
static hipError_t launch_direct_family(const SpmmParams& p, hipStream_t stream) {
    switch (form_index(direct_form(p.rows, p.N, p.S, HALF, p.cus))) {
        case 0: return launch_direct<1, OUT_LAYOUT, 4, HALF>(p, stream);
        case 1: return launch_direct<1, OUT_LAYOUT, 8, HALF>(p, stream);
        case 2: return launch_direct<1, OUT_LAYOUT, 16, HALF>(p, stream);
        case 3: return launch_direct<2, OUT_LAYOUT, 4, HALF>(p, stream);
        case 4: return launch_direct<2, OUT_LAYOUT, 8, HALF>(p, stream);
        case 5: return launch_direct<4, OUT_LAYOUT, 4, HALF>(p, stream);
        case 6: return launch_direct<4, OUT_LAYOUT, 4, HALF, true>(p, stream);
        case 7: return launch_direct<4, OUT_LAYOUT, 8, HALF>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

#define SPATHA_DIRECT_NAMES(prefix)                                                                                                   \
    {prefix "x16_splitk4", prefix "x16_splitk8", prefix "x16_splitk16", prefix "x32_splitk4", prefix "x32_splitk8", prefix "x64_splitk4", \
     prefix "x64_splitk4_lean", prefix "x64_splitk8"}
const char* spmm_direct_name(int variant, int rows, int N, int S, int cus) {
    static const char* const names[3][8] = {SPATHA_DIRECT_NAMES("smfmac16x16x64_skinny_tile64"),
                                            SPATHA_DIRECT_NAMES("smfmac16x16x64_direct_tile64"),
                                            SPATHA_DIRECT_NAMES("smfmac16x16x64_halftile_direct_tile32")};
    const int kind = variant == SPMM_VARIANT_SKINNY ? 0 : variant == SPMM_VARIANT_DIRECT64 ? 1 : variant == SPMM_VARIANT_HDIRECT32 ? 2 : -1;
    if (kind < 0) return nullptr;
    const int form = form_index(direct_form(rows, N, S, kind == 2, cus));
    return form < 0 ? nullptr : names[kind][form];
}
#undef SPATHA_DIRECT_NAMES

// A few tokens as they lie, x [N][cols] with N <= 16 (any count), transposed output: what the transposed copy ahead of the product
// would hold is read from LDS, where every workgroup puts the tokens first.
// (A layer of 1024 x 1024 at 64:2:8 on 8 tokens, whole call: 7.1 us, 12.1 with a transposing kernel ahead of the product.)
template <int W, bool HALF>
static hipError_t launch_token_major(SpmmParams p, hipStream_t stream) {
    using Cfg = DirectCfg<1, W, HALF, false>;
    p.tiles_m = p.rows / (HALF ? 32 : 64);
    p.tiles_n = 1;
    p.walk_group = 0;
    const size_t tokens = (size_t)p.N * token_pitch_halfs(p.cols) * 2, partial = (size_t)W * Cfg::PB * 64 * sizeof(float4_t);
    const size_t lds = ((tokens > partial ? tokens : partial) + 15) / 16 * 16;
    auto kern = spmm_direct_kernel<1, SPATHA_OUT_TRANSPOSED, W, HALF, false, true, false>;
    if (lds > 48 * 1024) {
        bool& attr_set = lds_attr_flag((const void*)kern);
        if (!attr_set) {
            hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
            if (e != hipSuccess) return e;
            attr_set = true;
        }
    }
    hipLaunchKernelGGL(kern, dim3((p.tiles_m + 7) / 8 * 8), dim3(W * 64), lds, stream, p);
    return hipGetLastError();
}

// (one workgroup a CU where the tokens take more than half of its LDS: not with more row tiles than CUs)
bool token_major_fits(int rows, int cols, int tokens, bool half_tiles, int cus) {
    return tokens <= 16 && (size_t)tokens * token_pitch_halfs(cols) * 2 <= 128 * 1024 && rows / (half_tiles ? 32 : 64) <= cus;
}

hipError_t launch_token_major(const SpmmParams& p, bool half_tiles, hipStream_t stream) {
    if (half_tiles) return p.S > 12 ? launch_token_major<16, true>(p, stream) : launch_token_major<8, true>(p, stream);
    return p.S > 12 ? launch_token_major<16, false>(p, stream) : launch_token_major<8, false>(p, stream);
}

hipError_t launch_skinny_family(int variant, int out_layout, const SpmmParams& p, hipStream_t stream) {
    const bool transposed = out_layout == SPATHA_OUT_TRANSPOSED;
    switch (variant) {
        case SPMM_VARIANT_SKINNY:
        case SPMM_VARIANT_DIRECT64:
            return transposed ? launch_direct_family<SPATHA_OUT_TRANSPOSED, false>(p, stream)
                              : launch_direct_family<SPATHA_OUT_ROW_MAJOR, false>(p, stream);
        case SPMM_VARIANT_HDIRECT32:
            return transposed ? launch_direct_family<SPATHA_OUT_TRANSPOSED, true>(p, stream)
                              : launch_direct_family<SPATHA_OUT_ROW_MAJOR, true>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace spatha
