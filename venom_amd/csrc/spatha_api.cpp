// C ABI of the library (see include/spatha.h): argument checking, plan
// management and kernel selection.  No torch types, no exceptions across the
// boundary, no exit().

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "../../include/spatha.h"
#include "spmm_kernels.h"
#include "vnm_format.h"

#include "spatha_internal.h"

namespace {
thread_local int g_last_hip_error = 0;

inline int hip_fail(hipError_t e) {
    g_last_hip_error = (int)e;
    return SPATHA_ERR_HIP;
}

// compute units of the current device (0 where the runtime does not say)
int device_cus() {
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return 0;
    return cus;
}

// kernels whose write-out can apply bias and activation ahead of either output layout
bool variant_has_fused_writeout(int variant) {
    using namespace spatha;
    switch (variant) {
        case SPMM_VARIANT_P128x128_S3: case SPMM_VARIANT_P64x256_S2: case SPMM_VARIANT_R64x256_S3:
        case SPMM_VARIANT_W128x128_S3: case SPMM_VARIANT_W128x256_S3: case SPMM_VARIANT_W64x256_S3:
        case SPMM_VARIANT_T128x256_S3: case SPMM_VARIANT_DS256x128_S3_C8: case SPMM_VARIANT_DSH256x128_S3_C8:
        case SPMM_VARIANT_UP512x128_S3: case SPMM_VARIANT_DU512x128_M16: case SPMM_VARIANT_WS128x128_S3:
        case SPMM_VARIANT_WS64x256_S3: case SPMM_VARIANT_OH192x256: case SPMM_VARIANT_H64x256_S2: case SPMM_VARIANT_H64x128_S3: case SPMM_VARIANT_H64x128_S2:
        case SPMM_VARIANT_DIRECT64: case SPMM_VARIANT_HDIRECT32:
            return true;
        default:
            return false;
    }
}

// kernels that address B, the packed operands and the tables through buffer descriptors (32-bit offsets)
bool variant_uses_buffer_descriptors(int variant) {
    using namespace spatha;
    switch (variant) {
        case SPMM_VARIANT_128x128: case SPMM_VARIANT_64x256: case SPMM_VARIANT_P128x128_S3: case SPMM_VARIANT_P64x256_S2:
            return false;
        default:
            return true;
    }
}

bool variant_ok(const spatha_spmm_plan* plan, int N, int variant, bool fused = false) {
    using namespace spatha;
    if (variant <= 0 || (variant >= SPMM_VARIANT_COUNT && variant != SPMM_VARIANT_HDIRECT32)) return false;
    if (fused && !variant_has_fused_writeout(variant)) return false;
    const int bm = spmm_variant_bm(variant);
    if (bm == 0) return false;
    const bool half_variant = variant == SPMM_VARIANT_H64x256_S2 || variant == SPMM_VARIANT_H64x128_S3 ||
                              variant == SPMM_VARIANT_H64x128_S2 || variant == SPMM_VARIANT_DSH256x128_S3_C8 ||
                              variant == SPMM_VARIANT_HDIRECT32;
    if (half_variant != (plan->half_tiles != 0)) return false;       // the packed operand order differs
    const uint64_t b_bytes = (uint64_t)plan->geo.cols * (uint64_t)N * 2u;
    if (variant == SPMM_VARIANT_DSH256x128_S3_C8) {
        if (plan->geo.m > 8 || plan->geo.rows % 256 != 0 || !plan->gtab) return false;
        return b_bytes < 0xE0000000ull && plan->apack_bytes < 0xE0000000ull;
    }
    if (variant == SPMM_VARIANT_HDIRECT32)
        return b_bytes < 0xE0000000ull && plan->apack_bytes < 0xE0000000ull && plan->rowtab_bytes < 0xE0000000ull;
    if (half_variant) return plan->geo.cols <= 65535 && spmm_variant_lds(variant, plan->S) <= 160 * 1024;
    const bool unified = variant == SPMM_VARIANT_UP512x128_S3 || variant == SPMM_VARIANT_DU512x128_M16;
    if (variant == SPMM_VARIANT_DS256x128_S3_C8 || variant == SPMM_VARIANT_DS256x128_S3_PP) {
        // four 64-row blocks per tile; all 16*m dense rows of a k-step must fit one stage
        if (plan->geo.v % 64 != 0 || plan->geo.m > 8 || plan->geo.rows % 256 != 0 || !plan->gtab) return false;
    } else if (unified) {
        if (plan->geo.v % 64 != 0 || plan->geo.rows % 512 != 0 || !plan->gtab || plan->half_tiles) return false;
        if (variant == SPMM_VARIANT_DU512x128_M16 ? (plan->geo.m <= 8 || plan->geo.m > 16) : plan->geo.m > 8) return false;
        if (plan->gtab_bytes >= 0xE0000000ull) return false;
    } else if (plan->geo.v % bm != 0) {
        return false;
    }
    if (variant == SPMM_VARIANT_SKINNY && N > 64) return false;
    if ((variant == SPMM_VARIANT_WS128x128_S3 || variant == SPMM_VARIANT_WS64x256_S3) && plan->S < 2)
        return false;       // the tile hand-over to the store waves needs two k-steps per tile
    if (spmm_variant_lds(variant, plan->S) > 160 * 1024) return false;      // row table kept in LDS
    if (variant_uses_buffer_descriptors(variant) &&
        (b_bytes >= 0xE0000000ull || plan->apack_bytes >= 0xE0000000ull || plan->rowtab_bytes >= 0xE0000000ull))
        return false;
    return true;
}

// ---- Kernel choice ----------------------------------------------------------------------------------------------
// The automatic choice is a list of rules read top-down: the first rule whose class and condition hold for the shape
// and whose kernel accepts the plan (variant_ok) names the kernel.  The conditions are measured crossover points on
// MI355X (BERT-base / BERT-large / GPT-2-large / GPT-3 layer shapes, N = 2048 .. 16384, m = 4 .. 100); each rule's comment
// says what was measured.  Later rules double as the fall-backs of earlier ones.
struct Shape {
    int v, m, rows, cols, N, S;
    int64_t cus;
    bool fused, transposed;
    // tiles of bm x bn in the output (whole row tiles only: the kernels that take a partial row tile are never chosen by count)
    int64_t tiles(int bm, int bn) const { return (int64_t)(rows / bm) * ((N + bn - 1) / bn); }
    // the last of `tiles` tiles' rounds over the CUs is at least 90 % full (a single round: 75 %)
    bool whole_rounds(int64_t t) const {
        const int64_t rounds = (t + cus - 1) / cus;
        return rounds == 1 ? t * 4 >= cus * 3 : t * 10 >= rounds * cus * 9;
    }
    // unified 512 x 128 tiles against dense-staged 256 x 128 ones by rounds of tiles over the CUs, a 512-row tile counted as
    // two and 10 % off for what it saves per tile (5120 x 1280 x 2048 at 2:8 and 2:4: 160 tiles on 256 CUs in one round, 17 and
    // 24 us, against 1.25 rounds of 320 dense-staged tiles, 20 and 32 us)
    bool unified_rounds_ahead() const {
        const int64_t r_up = (tiles(512, 128) + cus - 1) / cus, r_ds = (tiles(256, 128) + cus - 1) / cus;
        // (long k-loops, where a tile's write-out weighs less: 25 % off - 12288 x 12288 x 2048 at 64:2:8 and 2:4, 384 tiles in two
        // rounds against 768 in three, 212 / 396 against 236 / 429 us)
        return r_up * (S >= 64 ? 15 : 18) <= r_ds * 10;
    }
    // 128 x 256 tiles ahead of 128 x 128 ones: from 1024 tiles on, from 768 with two or more k-steps, from 512 with eight or
    // more; with fewer, from 192 tiles of 32 or more k-steps, and with 10 .. 31 k-steps where the rounds say so (1280 x 5120 at
    // 128:2:16 / 20 / 32: 4096 tokens, 160 tiles in one round, 18.7 / 16.5 / 13.0 against 22.0 / 18.8 / 14.1 us; 8192 tokens, 320
    // tiles in two rounds against 640 in three, 28.1 / 22.0 against 25.9 / 19.3 us at 2:20 / 2:32) (every kernel on the BERT layer shapes x N = 2048 .. 8192 x 2:10 .. 2:100;
    // 1024 x 1024 x 16384 at 128:2:16, 512 wide tiles of 4 k-steps, runs 19 % faster on 128 x 128 tiles)
    // (never for a single, half-empty column tile: GPT-3 FFN matrix at 128 tokens, 46.5 us on 128 x 128 against 61.5 us)
    bool wide() const {
        const int64_t t = tiles(128, 256);
        if (N <= 128) return false;
        if (t >= 1024 || (t >= 768 && S >= 2) || (t >= 512 && S >= 8)) return true;
        if (S >= 32) return t >= 192;
        // few tiles of 10 .. 31 k-steps: by rounds of tiles over the CUs, a 128 x 256 tile counted as 1.6 tiles of 128 x 128
        const int64_t r_wide = (t + cus - 1) / cus, r_narrow = (tiles(128, 128) + cus - 1) / cus;
        return S >= 10 && t >= 160 && r_wide * 16 <= r_narrow * 10;
    }
    // transposed output: 128 x 256 tiles from 512 tiles on, with fewer by rounds (a 128 x 256 tile counted as 1.6 of 128 x 128)
    bool wide_transposed() const {
        const int64_t t = tiles(128, 256);
        if (t >= 512) return true;
        const int64_t r_wide = (t + cus - 1) / cus, r_narrow = (tiles(128, 128) + cus - 1) / cus;
        return r_wide * 16 <= r_narrow * 10;
    }
    // 64 x 256 tiles with long k-loops: the persistent three-stage pipeline leads the per-tile one with two stages at any tile
    // count (1280 x 5120 at 64:2:10, 4096 .. 16384 tokens, 320 .. 1280 tiles: 45 / 66 / 108 against 56 / 84 / 139 us;
    // 12288 x 12288 x 512 at 64:2:16 and 64:2:10: 66 / 100 against 86 / 132 us)
    bool long_k() const { return S >= 32; }
    // More than one round of 128 x 256 tiles over the CUs and at most a round and a half: F = ceil(2T / 3) workgroups per
    // 256-column tile, each with one whole tile and a 128-column half of another, run them in ONE round of equal workgroups
    // that stay in step through k (kernel 22).  Every kernel id on 49152 / 40960 / 36864 / 34816 x 12288 (GPT-3 FFN matrix and
    // fewer rows of it; 384 .. 272 row tiles on 256 CUs) at 136 .. 256 tokens, 128:2:16, Gaussian data: 53-57 / 52 / 50 / 50 us
    // against 61-66 us for 256 tall tiles + the rest on 128 x 128 tiles in a second launch; the same rows x 1024 .. 6144
    // columns (4 .. 24 k-steps), where the 128 x 128 tiles with store waves were chosen: 1.06-1.36x ahead row-major from 8
    // k-steps on (4 k-steps: 0.94-1.06x), 1.19-1.53x transposed; 128:2:40 1.28-1.70x; 16128 x 12288 x 768 and 12288^2 x
    // 1024 (three and four column tiles) 57 us against 59-70.  Not for m <= 8 (dense staging: 1.07-1.09x at 2:8 on the long
    // k-loop only, behind at 2:4), not when the last column tile has no columns for the second half, not beyond one round of
    // such workgroups (8192 x 4096 x 1536: 41 against 27 us), and for at most four column tiles: with many of them (few row
    // tiles, a large output: 1536 x 4096 x 8192, 1280 x 5120 x 8192, 768 x 3072 x 16384, 3072 x 4096 x 3584) the 128 x 128 tiles
    // with store waves, which write a tile out under the next tile's k-loop, are level (transposed) or 3-12 % ahead (row-major).
    bool tile_and_a_half() const {
        if (m <= 8 || rows % 128 != 0 || S < 4 || (S < 8 && !transposed)) return false;
        const int64_t T = rows / 128, tn = (N + 255) / 256, F = (2 * T + 2) / 3, grid = (cus / 8) * 8;
        const int last = N - (int)(tn - 1) * 256;
        return tn <= 4 && T * tn > grid && F * tn <= grid && last > 128;
    }
    // Small products: kernels 23 (64 x 64 tiles) and 24 (32 x 64), straight from the L2, k-steps over a tile's waves (spmm_skinny.hip).
    // Against the kernels chosen otherwise (nine layer shapes x ten formats, 104 .. 4096 tokens, both layouts; geometric means):
    //   V % 128 == 0:      at most one tile per CU 1.3-2.2x; up to 1.25 1.03-1.08x, up to 1.6 row-major
    //                      1.04-1.08x and transposed 0.95-1.01x (both 0.94-0.97x from 29 k-steps on); up to 2
    //                      row-major 1.06x and transposed 0.96x up to ten k-steps, 0.95-1.0x with more; beyond 0.55-0.84x.
    //   V % 64 == 0 only:  up to one tile per CU 1.4-3.0x, up to two 1.08-1.5x; up to 2.5, m > 8, more than ten k-steps 1.10-1.18x
    //                      (ten or fewer 0.88x; m <= 8 0.93-1.0x); beyond 0.4-1.0x.
    // k-loops of 96 steps on V % 128 == 0 are what split runs are for (12288 x 49152 x 128 at 128:2:16: 48 us in two parts, 71 here).
    // Three k-steps or fewer at m <= 8 stay with dense staging although these kernels are ahead there too (up to two tiles per CU,
    // row-major 1.2-1.9x, 512 x 256 x 256 at 64:2:8 5.9 against 3.2 us, transposed 0.97-1.5x): a caller holds the choice to that
    // (tests/test_spmm_gpu.py asks for the dense-staged kernel at that shape).
    bool direct64() const {
        const int64_t t = (int64_t)(rows / 64) * ((N + 63) / 64);
        if (v % 128 == 0)
            return S < 96 && (t <= cus || (S <= 28 && t * 20 <= cus * (transposed ? 25 : 32)) || (S <= 10 && !transposed && t <= 2 * cus));
        if (m <= 8 && S <= 3) return false;
        return t <= 2 * cus || (m > 8 && S > 10 && t * 2 <= 5 * cus);
    }
    // V % 64 != 0: 64 x 128 gathered tiles run two workgroups a CU as long as the row table leaves room for it (75 KB of stages + 256
    // bytes a k-step, twice: up to 28 k-steps)
    bool half_pairs() const { return S <= 28; }
    // V % 64 != 0: direct 32 x 64 tiles always up to 32 columns and, where nothing is dense-staged, up to 128 (2-5x ahead of the
    // gathered tiles); above that up to three tiles per CU (1.08-2.1x; at four 0.98-1.0x), with more than ten k-steps up to four
    // (1.10-1.16x; at eight 0.8-0.93x).  Where the replaced kernel is one step into a second round (1280 .. 12288 x 1024 .. 12288,
    // m = 10, 16, 32, both layouts, 990 products): up to 8 3/4 tiles per CU from five k-steps on (1.2x in the mean, none of 176
    // products more than 3 % behind; 4096 x 4096 x 1040 at 32:2:16 31.1 against 35.9 us), up to eleven as long as B fits an XCD's L2
    // (1.08-1.14x; with a larger B 0.84-1.1x); fewer k-steps 0.98-1.09x.
    bool direct32() const {
        const bool staged = m <= 8 && rows % 256 == 0 && (tiles(256, 128) >= 160 || S >= 16);
        if (N <= (staged ? 32 : 128)) return true;
        const int64_t t = (int64_t)(rows / 32) * ((N + 63) / 64), row_tiles = (rows + 63) / 64;
        if (t <= (S > 10 ? 4 : 3) * cus) return true;
        if (staged) return false;
        if (S > 16 && direct32_long()) return true;
        const int64_t at_once = half_pairs() ? 2 * cus : cus, width = half_pairs() ? 128 : 256;
        const int64_t rounds = (row_tiles * ((N + width - 1) / width) + at_once - 1) / at_once;
        if (rounds != 2) return false;
        if (!half_pairs()) return t <= 8 * cus;
        return (S > 4 && t * 4 <= 35 * cus) || (t <= 11 * cus && (int64_t)cols * N * 2 <= (4 << 20));
    }
    // The same kernel at any number of tiles, by the columns of 64 that its tiles pay for against the 128 or 256 of the gathered ones
    // (12288 .. 49152 x 12288 and 12288 x 49152, m = 10 .. 40, both layouts): up to 192 columns 0.97-1.09x on 49152 rows, 1.13-1.34x on the
    // others; 257 .. 384 from 29 k-steps on, where two 256-wide tiles stand against it, 0.98-1.39x (fewer k-steps, pairs of 128-wide tiles:
    // 0.7-1.3x); 193 .. 256 only where no 256-wide tile fits any more (half_wide; 1.39-1.85x, below that 0.8-1.06x).  More columns
    // 0.5-1.1x and as often behind as ahead.
    bool direct32_long() const { return N <= 192 || (!half_pairs() && N > 256 && N <= 384) || (!half_wide() && N <= 256); }
    // V % 64 != 0: two stages of a 64 x 256 gathered tile (137 KB) and the row table fit the LDS of a CU up to 92 k-steps
    bool half_wide() const { return S <= 92; }
    // dense-staged 256 x 128 tiles: the form in two phase groups leads the eight-consumer form row-major by 2-5 % up to 768 tiles of 32
    // k-steps or fewer; with more of them by 5-12 % at m = 7 and 8 whatever the count (12288 x 12288 x 640 at 128:2:8 70 against 84 us) and
    // by 1-7 % at m = 4, transposed by 3-11 % at m = 7 and 8 (level in one round of 33 .. 64 k-steps; m = 4: level, up to 14 % behind).
    // It has no fused write-out.
    bool two_phases() const {
        if (fused) return false;
        if (S <= 32) return !transposed && tiles(256, 128) <= 768;
        return !transposed || (m > 5 && (S > 64 || tiles(256, 128) > cus));
    }
    // 64 x 256 tiles: many tiles of few k-steps, m >= 32, row-major
    bool short_k_many() const { return m >= 32 && !transposed && tiles(64, 256) >= 2048 && S <= 8; }
};

enum : unsigned { V_HALF = 1u, V_128 = 2u, V_64 = 4u };       // V % 64 != 0 / V % 128 == 0 / V % 64 == 0 only

struct Rule {
    unsigned v_classes;
    int variant;
    bool (*when)(const Shape&);
};

const Rule kRules[] = {
    // few columns: streaming A is all that matters, one 64-row tile per workgroup with the k-steps split over its waves, B
    // straight from the L2 with one load per gathered row whatever N (2, 4 or 8 bytes for 16, 32 or 64 columns).  1.3-3x ahead of
    // every tiled kernel on the BERT-large matrices; GPT-3 FFN matrix, launches back to back (its 176 MB then stay in the memory-side
    // cache; 38.7 us from memory at 16 columns), 27-29 us up to 32 columns (128-wide tiles 39-41),
    // 36 us at 64, level with the 128 x 128 tiles (39): there the registers of its four column blocks leave three workgroups
    // per CU for three tiles per CU.  The same kernel with column tiles (id 23) takes fused write-outs and small products.
    {V_128 | V_64, spatha::SPMM_VARIANT_SKINNY, [](const Shape& s) { return s.N <= 64; }},
    {V_128 | V_64, spatha::SPMM_VARIANT_DIRECT64, [](const Shape& s) { return s.N <= 64 || s.direct64(); }},
    {V_HALF, spatha::SPMM_VARIANT_HDIRECT32, [](const Shape& s) { return s.direct32(); }},

    // -- V % 64 != 0 (1024 x 4096 x 4096 and 4096 x 1024 x 16384, m = 8 .. 32) --
    // m <= 8: the dense B stage is shared by eight 32-row blocks, the fill does not grow with the smaller V
    // (short k-loops - 8 or 10 k-steps - on 64 tiles or fewer, 1024 x 1024 up to 2048 tokens, 4096 x 1024 up to 512: the gathered
    // half-tile kernels are 9-24 % ahead; with 32 k-steps or more dense staging leads at any tile count, 1.2-3.4x on 1024 x 4096,
    // 1280 x 5120 and 12288 x 12288)
    {V_HALF, spatha::SPMM_VARIANT_DSH256x128_S3_C8, [](const Shape& s) { return s.tiles(256, 128) >= 160 || s.S >= 16; }},
    // 128-wide tiles in pairs of workgroups lead the 256-wide ones, one workgroup a CU, by 2-20 % at any tile count (1024 x 4096 x
    // 4096 at 32:2:16 19.8 against 23.0 us, 12288 x 12288 x 2048 at 32:2:32 161 against 191); with longer k-loops, where only one
    // of them fits a CU, they trail by 1.2-1.6x (12288 x 12288 x 2048 at 32:2:16, 48 k-steps: 538 against 336 us)
    {V_HALF, spatha::SPMM_VARIANT_H64x128_S2, [](const Shape& s) { return s.half_pairs(); }},
    {V_HALF, spatha::SPMM_VARIANT_H64x256_S2, [](const Shape& s) { return s.N > 128; }},
    // one workgroup a CU in any case: three stages of 128 lead two by 1.1-1.4x (12288 x 49152 x 1040 at 32:2:16, 192 k-steps: 1189
    // against 1634 us; 512 columns 471 against 538) as long as the row table leaves room for them
    {V_HALF, spatha::SPMM_VARIANT_H64x128_S3, [](const Shape& s) { return !s.half_wide(); }},
    {V_HALF, spatha::SPMM_VARIANT_H64x128_S2, [](const Shape&) { return true; }},

    // -- unified 512 x 128 tiles --
    // m <= 8, two phase groups: 3-13 % ahead of the dense-staged 256 x 128 tiles when its tiles fill whole rounds of the CUs
    // (BERT-large layer shapes at N = 16384, V = 64 and 128, m = 8 and 4: 256, 768, 1024 tiles; 3072 x 768 x 4096, 192
    // tiles: 10-12 % ahead), 10-20 % behind at 320 or 384 tiles and up to 2x behind with fewer tiles than CUs;
    // transposed output with 256 tiles of 8 k-steps measures 2-3 % behind
    {V_128 | V_64, spatha::SPMM_VARIANT_UP512x128_S3,
     [](const Shape& s) {
         const int64_t t = s.tiles(512, 128);
         // (transposed output with one or two full rounds of 8 k-steps is level with the dense-staged 256 x 128 tiles or 2-3 %
         // behind; with less than a round - 3072 x 1024 x 4096, 5120 x 1280 x 2048: 192 and 160 tiles - 11-13 % ahead)
         return s.m <= 8 && (s.whole_rounds(t) || s.unified_rounds_ahead()) &&
                (!s.transposed || t >= 2 * s.cus || s.S >= 16 || t < s.cus);
     }},
    // 8 < m <= 16, one phase group with two 64 KB stages: 7-26 % ahead of the gathered 64 x 256 tiles on the BERT-large
    // layer shapes at N = 16384 (64:2:16 and 64:2:10, both layouts); on long k-loops ahead at 1.5 rounds too (12288 x 12288
    // x 2048 at 64:2:16: 177 us against 188 us for the best gathered form).  With V % 128 == 0 the gathered 128 x 256
    // tiles share their B rows over 128 rows and are equal or up to 15 % ahead.
    {V_64, spatha::SPMM_VARIANT_DU512x128_M16,
     [](const Shape& s) {
         const int64_t t = s.tiles(512, 128);
         return s.m > 8 && (s.whole_rounds(t) || (t >= s.cus && s.S >= 32));
     }},

    // -- V % 128 == 0 --
    // transposed output, m <= 8: the kernels that write through the 8-column slab lead by 10-25 % (BERT-large layer shapes,
    // N = 16384, with bias); not on long k-loops, where the gathered 128 x 256 tile moves fewer bytes per output element
    // (GPT-3 block at 128:2:8, 96 k-steps: 6.95 ms against 8.26 ms; GPT-2-large FFN-down, 40 k-steps: dense staging 20 % ahead)
    // (m <= 5: every dense row is a gathered row or nearly so, dense staging leads at any k: 1280 x 5120 x 4096 at 2:4, 80
    // k-steps, 45 against 65 us on 128 x 128 tiles; 12288 x 12288 x 512 at 2:4 115 against 127 us on 128 x 256 tiles)
    // (from 160 tiles on, as row-major: with fewer - 1024 x 4096 x 2048 / 4096, 1280 x 5120 x 2048: 64 .. 128 tiles - the
    // gathered 128 x 128 tiles are 13-35 % ahead)
    {V_128, spatha::SPMM_VARIANT_DS256x128_S3_PP,
     [](const Shape& s) { return s.transposed && s.two_phases() && s.m <= 8 && s.S <= 40 && s.tiles(256, 128) >= 160; }},
    {V_128, spatha::SPMM_VARIANT_DS256x128_S3_C8,
     [](const Shape& s) { return s.transposed && s.m <= 8 && (s.S <= 40 || s.m <= 5) && s.tiles(256, 128) >= 160; }},
    // row-major, m <= 8: dense staging leads the gathered tiles by 5-35 % as soon as its 256 x 128 tiles fill three quarters
    // of the CUs (BERT layer shapes, N = 2048 .. 16384; from 160 tiles on the GPT-2-large ones)
    {V_128, spatha::SPMM_VARIANT_DS256x128_S3_PP,
     [](const Shape& s) {
         return !s.transposed && s.two_phases() && s.m <= 8 && s.rows % 256 == 0 && s.tiles(256, 128) >= 160 && (s.S <= 64 || s.m <= 5);
     }},
    {V_128, spatha::SPMM_VARIANT_DS256x128_S3_C8,
     [](const Shape& s) {
         return !s.transposed && s.m <= 8 && s.rows % 256 == 0 && s.tiles(256, 128) >= 160 && (s.S <= 64 || s.m <= 5);
     }},
    // m > 8, between one and one and a half rounds of 128 x 256 tiles: one whole tile and a column half of another per workgroup
    {V_128, spatha::SPMM_VARIANT_OH192x256, [](const Shape& s) { return s.tile_and_a_half(); }},
    // transposed output, m > 8, more than one 128-column tile: 128 x 256 tiles at any tile count (5-15 % ahead of 128 x 128 on the BERT-large and
    // GPT-2-large layer shapes, N = 4096 and 16384); 64 x 64 consumer blocks up to 16 k-steps, else the tall consumers
    // (with fewer than 512 of them only where the rounds of tiles over the CUs say so: 1024 x 4096 x 2048, 1280 x 1280 x 2048,
    // 1280 x 5120 x 2048 at 128:2:16 .. 32 - 64, 80, 80 tiles - run 24-41 % faster on 128 x 128 tiles)
    {V_128, spatha::SPMM_VARIANT_W128x256_S3,
     [](const Shape& s) { return s.transposed && s.N > 128 && s.m >= 16 && s.S <= 16 && s.wide_transposed(); }},
    {V_128, spatha::SPMM_VARIANT_T128x256_S3, [](const Shape& s) { return s.transposed && s.N > 128 && s.m > 8 && s.wide_transposed(); }},
    {V_128, spatha::SPMM_VARIANT_W128x256_S3, [](const Shape& s) { return s.transposed && s.N > 128 && s.m > 8 && s.wide_transposed(); }},
    // row-major, two or three k-steps per tile and more than two rounds of 128 x 128 tiles: the kernel with store waves (a finished tile
    // leaves while the next one's k-loop runs) leads the 128 x 256 tiles by 7-18 % and the plain 128 x 128 ones by 14-23 %
    // (4096 x 1024 x 16384 at 128:2:32, 3072 x 768 x 8192 at 128:2:40, 1024 x 1024 x 16384 at 128:2:32); with transposed output
    // it is level with the plain kernel and behind the 128 x 256 tiles
    {V_128, spatha::SPMM_VARIANT_WS128x128_S3,
     [](const Shape& s) { return !s.transposed && s.m > 8 && s.S >= 2 && s.S <= 3 && s.tiles(128, 128) > 2 * s.cus; }},
    // 128 x 256 tiles, m >= 16: the 64 x 64 consumer blocks lead the tall-consumer form by 1-13 % up to 16 k-steps per tile
    // (BERT-large, GPT-2-large layers) from 768 tiles on (fewer: the tall form is 8-10 % ahead) and trail it by 1-3 % on
    // long k-loops (GPT-3 layers)
    {V_128, spatha::SPMM_VARIANT_W128x256_S3,
     [](const Shape& s) { return s.wide() && s.m >= 16 && s.S <= 16 && s.tiles(128, 256) >= 768; }},
    {V_128, spatha::SPMM_VARIANT_T128x256_S3, [](const Shape& s) { return s.wide(); }},
    {V_128, spatha::SPMM_VARIANT_W128x256_S3, [](const Shape& s) { return s.wide(); }},
    // more than one round of 128 x 128 tiles but less than two (two full rounds: the kernel with store waves is level or up to 6 %
    // ahead), few k-steps: the same number of 64 x 256 tiles runs as one
    // round of two co-resident workgroups per CU (768 x 768 x 8192, 3072 x 768 x 2048, 1024 x 1024 x 8192, 4096 x 1024 x
    // 2048 at 128:2:10 .. 128:2:100: 5-30 % ahead)
    {V_128, spatha::SPMM_VARIANT_P64x256_S2,
     [](const Shape& s) {
         const int64_t t = s.tiles(128, 128);
         return !s.transposed && s.m > 8 && t > s.cus && t < 2 * s.cus && s.S <= 8;
     }},
    // ... and wherever the 128 x 256 tiles do not lead and every CU has a tile: 5-13 % ahead of the plain 128 x 128 kernel
    // (1024 x 1024 x 16384 at 128:2:16, 4096 x 1024 x 4096 at 128:2:20, 5120 x 1280 x 4096 at 128:2:16, 1024 x 4096 x 4096 at
    // 128:2:7 .. 128:2:40), level with it on long k-loops with many tiles; 5-7 % behind with fewer tiles than CUs, and with
    // exactly one short tile per CU (1024 x 1024 x 4096 at 128:2:40)
    {V_128, spatha::SPMM_VARIANT_WS128x128_S3,
     [](const Shape& s) {
         const int64_t t = s.tiles(128, 128);
         return !s.transposed && s.S >= 2 && t >= s.cus && (t > s.cus || s.S >= 4);
     }},
    {V_128, spatha::SPMM_VARIANT_W128x128_S3, [](const Shape&) { return true; }},
    {V_128, spatha::SPMM_VARIANT_P128x128_S3, [](const Shape&) { return true; }},
    {V_128, spatha::SPMM_VARIANT_128x128, [](const Shape&) { return true; }},

    // -- V a multiple of 64 only --
    // m <= 8: staging the dense B rows once for four 64-row blocks halves the L2 -> LDS traffic; the two forms as above
    {V_64, spatha::SPMM_VARIANT_DS256x128_S3_PP, [](const Shape& s) { return s.two_phases(); }},
    {V_64, spatha::SPMM_VARIANT_DS256x128_S3_C8, [](const Shape&) { return true; }},
    // m > 8, row-major, two or three k-steps per tile and six rounds or more of 64 x 256 tiles: the producer/consumer kernel
    // with store waves, 9-10 % ahead of the plain one and of the per-tile pipeline (4096 x 1024 x 16384 at 64:2:32, 3072 x
    // 768 x 8192 at 64:2:40); level at four rounds, behind with fewer tiles and with four k-steps or more
    {V_64, spatha::SPMM_VARIANT_WS64x256_S3,
     [](const Shape& s) {
         // (transposed output, where the store waves also add the bias: ahead from twelve rounds on only - 4096 x 1024 x 16384
         // at 64:2:32 36.3 against 39.8 us for the per-tile pipeline; at six rounds 17.0 against 15.1 us)
         return s.m > 8 && s.S >= 2 && s.S <= 3 && s.tiles(64, 256) >= (s.transposed ? 12 : 6) * s.cus;
     }},
    // m > 8, gathered 64 x 256 tiles.  32 or more k-steps per tile and many rounds: the persistent pipeline, which keeps
    // loading across tile boundaries, leads (GPT-3 layers at 64:2:16; at 64:2:32, 24 k-steps, the per-tile pipeline is
    // 10-20 % ahead); with one tile per CU or less its third stage still gives long k-loops 5-15 %
    {V_64, spatha::SPMM_VARIANT_R64x256_S3, [](const Shape& s) { return s.long_k(); }},
    {V_64, spatha::SPMM_VARIANT_W64x256_S3, [](const Shape& s) { return s.long_k(); }},
    // 16 <= m, 3072 tiles or more of few k-steps, plain row-major output: the producer/consumer kernel with the write-out
    // deferred into the next tile's steps leads the pipeline by 5-8 % (3072 / 4096 x 1024 x 16384 at 64:2:16)
    {V_64, spatha::SPMM_VARIANT_D64x256_S3,
     [](const Shape& s) {
         return !s.long_k() && !s.short_k_many() && !s.fused && !s.transposed && s.m >= 16 && s.tiles(64, 256) >= 3072 && s.S <= 8;
     }},
    // producer/consumer kernel: m >= 32 with many tiles of few k-steps, row-major, 5-10 % ahead (transposed: the pipeline
    // leads by 6-8 %); at most one tile per CU with a dozen or more k-steps, 10-17 % ahead of the per-tile pipeline
    // (768 x 3072 / 1024 x 4096 x 4096 at 64:2:10 and 64:2:20)
    {V_64, spatha::SPMM_VARIANT_W64x256_S3,
     [](const Shape& s) {
         return !s.long_k() && (s.short_k_many() || (!s.transposed && s.tiles(64, 256) <= s.cus && s.S >= 12));
     }},
    // else the per-tile pipeline with two stages (two workgroups per CU)
    {V_64, spatha::SPMM_VARIANT_P64x256_S2, [](const Shape& s) { return !s.long_k(); }},
    {V_64, spatha::SPMM_VARIANT_R64x256_S3, [](const Shape&) { return true; }},
    {V_64, spatha::SPMM_VARIANT_64x256, [](const Shape&) { return true; }},
};

// Long k-loops: what a launch takes is rounds of its tiles over the CUs times what a k-step of one such round takes, whatever the
// matrix.  us a k-step, medians over 12288 .. 49152 x 12288, 12288 x 49152, 4096 x 16384, 8192 x 8192, 16384 x 4096, 20480 x 5120 and
// 24576 x 8192, m = 4 .. 40, 72 .. 4096 columns, both layouts (the middle 80 % of products within 10 %, the direct tiles' 20):
//   V % 128 == 0: 128 x 128 tiles 0.45, 128 x 256 0.69, a tile and a half 0.92 (0.975 where its last column tile has nothing for the
//     second half; 1.02 in several rounds: 0.91 in short bursts, but its sixteen waves draw the most power and hold the clock lowest
//     when launches follow each other for long), dense-staged 256 x 128 0.65 .. 0.78 and 512 x 128 0.96 .. 1.1 with m;
//   V % 64 == 0 only, m > 8: 64 x 256 tiles 0.68 (0.64 from 64 k-steps on), in pairs of workgroups 0.61; direct 64 x 64 tiles, several on
//     a CU, 0.27 for as many as CUs without rounding up.
// 0: not priced.
float round_price(const Shape& s, int variant) {
    using namespace spatha;
    const int64_t grid = (s.cus / 8) * 8;
    auto rounds = [&](int64_t tiles) { return (float)((tiles + grid - 1) / grid); };
    switch (variant) {
        case SPMM_VARIANT_W128x128_S3: case SPMM_VARIANT_WS128x128_S3: return 0.45f * rounds(s.tiles(128, 128));
        case SPMM_VARIANT_W128x256_S3: case SPMM_VARIANT_T128x256_S3: return 0.69f * rounds(s.tiles(128, 256));
        case SPMM_VARIANT_OH192x256: {
            const int64_t per_column = (2 * (int64_t)(s.rows / 128) + 2) / 3, tn = (s.N + 255) / 256;
            const bool whole = s.N - (tn - 1) * 256 > 128;
            const float n = rounds(per_column * tn);
            return (n > 1.f ? 1.02f : whole ? 0.92f : 0.975f) * n;
        }
        case SPMM_VARIANT_DS256x128_S3_PP: case SPMM_VARIANT_DS256x128_S3_C8:
            return (s.m <= 5 ? 0.65f : s.m <= 7 ? 0.72f : 0.78f) * rounds(s.tiles(256, 128));
        case SPMM_VARIANT_UP512x128_S3: return (s.m <= 5 ? 0.96f : s.m <= 7 ? 1.06f : 1.1f) * rounds(s.tiles(512, 128));
        case SPMM_VARIANT_P64x256_S2: return (s.S <= 28 ? 0.61f : 0.89f) * rounds(s.tiles(64, 256));
        case SPMM_VARIANT_R64x256_S3: return (s.S < 64 ? 0.68f : 0.64f) * rounds(s.tiles(64, 256));
        case SPMM_VARIANT_DIRECT64: return 0.27f * (float)s.tiles(64, 64) / (float)grid;
        default: return 0.f;
    }
}

int uneven_rest_rows(const spatha_spmm_plan* plan, int N, int requested, int chosen, bool fused);

// The kernel the rules chose, or one whose rounds promise clearly less.  (Three sets of operands in turn, launches following each other for
// 40 ms a side: in shorter runs the clock is higher and flatters the kernels that draw the most power.)
//   V % 128 == 0, 24 k-steps or more, 10 %: 289 of 2436 products of the sizes above change, 1.18x faster in the mean, none of 146 timed
//     more than 2 % behind (12288 x 12288 x 640: at 128:2:16 two rounds of 128 x 256 tiles 65 us, of 128 x 128 44; at 128:2:8 120 us,
//     one round of dense-staged tiles 70).  Not where the launch is half a round or less: runs that bring a workspace split those
//     k-loops.
//   V % 64 == 0 only, m > 8, 16 k-steps or more: direct tiles, 102 of 1722 change, 1.27x faster in the mean, two of 83 timed 3-4 % behind
//     (36864 x 12288 x 72 at 64:2:16 90 -> 52 us, 12288 x 12288 x 264 68 -> 48).  20 % where pairs of workgroups share a CU, 8 %
//     elsewhere.  m <= 8: no price tells the dense-staged kernels apart from the gathered ones there, half of what would change is slower.
// With fewer k-steps a tile's start and write-out weigh in and the rules above are as good.
int by_rounds(const spatha_spmm_plan* plan, const Shape& s, int chosen) {
    using namespace spatha;
    const int64_t grid = (s.cus / 8) * 8;
    if (s.cus < 8 || plan->half_tiles) return chosen;
    float best = round_price(s, chosen);
    if (best == 0.f) return chosen;
    auto offer = [&](int variant) {
        const float price = round_price(s, variant);
        if (price < best && variant_ok(plan, s.N, variant, s.fused)) {
            best = price;
            chosen = variant;
        }
    };
    // (dense-staged and unified tiles go by m alone, and to rows their tiles divide, which variant_ok holds them to)
    if (s.v % 128 == 0) {
        if (s.S < 24 || s.tiles(128, chosen == SPMM_VARIANT_T128x256_S3 ? 256 : 128) * 2 <= grid) return chosen;
        if (uneven_rest_rows(plan, s.N, SPMM_VARIANT_AUTO, chosen, s.fused))
            best = 0.69f * (float)(s.tiles(128, 256) / grid) + 0.5f;      // whole rounds and one of 128 x 128 tiles behind them
        best *= 0.9f;
        offer(s.transposed ? SPMM_VARIANT_W128x128_S3 : SPMM_VARIANT_WS128x128_S3);
        offer(SPMM_VARIANT_T128x256_S3);
        offer(SPMM_VARIANT_OH192x256);
        if (s.m <= 8) {
            offer(s.two_phases() ? SPMM_VARIANT_DS256x128_S3_PP : SPMM_VARIANT_DS256x128_S3_C8);
            offer(SPMM_VARIANT_UP512x128_S3);
        }
    } else if (s.m > 8 && s.S >= 16 && (chosen == SPMM_VARIANT_P64x256_S2 || chosen == SPMM_VARIANT_R64x256_S3)) {
        best *= chosen == SPMM_VARIANT_P64x256_S2 ? 0.8f : 0.92f;
        offer(SPMM_VARIANT_DIRECT64);
    }
    return chosen;
}

int pick_variant(const spatha_spmm_plan* plan, int N, int variant, bool fused = false, int out_layout = SPATHA_OUT_ROW_MAJOR) {
    if (variant != spatha::SPMM_VARIANT_AUTO)
        return variant_ok(plan, N, variant, fused) ? variant : -1;
    Shape s;
    s.v = plan->geo.v; s.m = plan->geo.m; s.rows = plan->geo.rows; s.cols = plan->geo.cols; s.N = N; s.S = plan->S;
    s.cus = plan->cus > 0 ? plan->cus : 256;
    s.fused = fused;
    s.transposed = out_layout == SPATHA_OUT_TRANSPOSED;
    const unsigned v_class = plan->half_tiles ? V_HALF : s.v % 128 == 0 ? V_128 : s.v % 64 == 0 ? V_64 : 0u;
    for (const Rule& r : kRules)
        if ((r.v_classes & v_class) && r.when(s) && variant_ok(plan, N, r.variant, fused)) return by_rounds(plan, s, r.variant);
    return -1;
}

// An uneven last round of 128 x 256 tiles (automatic choice only): when the tiles fill one or more rounds of the CUs and
// leave a rest of at most half a round, the rest's row tiles run as a second launch on 128 x 128 tiles - twice as many
// tiles of half the work, so that its one round keeps every CU busy (GPT-3 FFN matrix at 256 tokens: 384 tiles on 256
// CUs).  Returns the rows of that second launch (the last rows of the matrix), 0 for a single launch.
int uneven_rest_rows(const spatha_spmm_plan* plan, int N, int requested, int chosen, bool fused) {
    if (requested != spatha::SPMM_VARIANT_AUTO || plan->cus < 8) return 0;
    if (chosen != spatha::SPMM_VARIANT_T128x256_S3 && chosen != spatha::SPMM_VARIANT_W128x256_S3) return 0;
    const int grid = (plan->cus / 8) * 8;       // workgroups of the persistent kernels
    const int tiles_n = (N + 255) / 256;
    const int64_t tiles = (int64_t)(plan->geo.rows / 128) * tiles_n, rest = tiles % grid;
    if (tiles <= grid || rest == 0 || rest % tiles_n != 0) return 0;
    // (short k-loops: a second launch costs more than the half-empty round; 1280 x 5120 x 16384 at 128:2:16 / 20 / 32, 20 / 16 /
    // 10 k-steps: 52 / 46 / 36 us in one launch against 56 / 50 / 40 in two)
    if (plan->S < 32) return 0;
    const int rest_rows = (int)(rest / tiles_n) * 128;
    if ((int64_t)(rest_rows / 128) * ((N + 127) / 128) > grid) return 0;        // more than half a round: one launch
    if ((plan->geo.rows - rest_rows) % plan->geo.v != 0) return 0;
    return variant_ok(plan, N, spatha::SPMM_VARIANT_W128x128_S3, fused) ? rest_rows : 0;
}

// ---- k-split (runs that bring a workspace) ----------------------------------------------------------------------
// Few tiles with long k-loops (small rows x N, large K: the chosen kernel's tiles fill at most half of the CUs): every tile's
// k-loop is cut into `parts` parts, one workgroup each.  Parts hand their fp32 partial blocks over through the workspace; the
// part that finishes last adds them in part order and writes the block (ksplit_exchange in spmm_warpspec.hip): deterministic,
// no workgroup waits for another.
// The hand-over costs 6-9 us (three dependent trips to the memory side: partial stores, ticket, partial loads; 64 or 128 KB
// of fp32 per tile and part) and a k-step 0.3-0.6 us, so a split must save about 48 k-steps per tile and leave parts of 32:
//   1024 x 16384 x 1024 at 128:2:8   (128 tiles of 128 k-steps, 2 parts)  34.7 against 50.2 us
//   12288 x 49152 x 128 at 128:2:16  ( 96 tiles of 192 k-steps, 2 parts)  48.3 against 73.2 us
//   768 x 12288 x 2048 at 128:2:8    ( 96 tiles of  96 k-steps, 2 parts)  30.5 against 38.9 us
//   1024 x 24576 x 2048 at 128:2:16  (128 tiles of  96 k-steps, 2 parts)  31.9 against 39.3 us
//   tiles of 64 k-steps in four parts of 16: between 15 % ahead and 7 % behind (256 x 8192 x 256, 4096 x 16384 x 256): not split.
// The rest of an uneven last round as a split second launch of the same kernel (instead of smaller tiles, uneven_rest_rows)
// was measured as well and does not pay: GPT-3 FFN matrix at 256 tokens (24 saved steps) 75 against 65 us, its FFN-down matrix
// at 1024 tokens (96 saved steps) 228 against 232 us; 128 x 256 tiles hand over twice the bytes.
#ifndef SPATHA_KSPLIT_MIN_SAVED_STEPS
#define SPATHA_KSPLIT_MIN_SAVED_STEPS 48
#endif
#ifndef SPATHA_KSPLIT_MIN_PART_STEPS
#define SPATHA_KSPLIT_MIN_PART_STEPS 32
#endif

struct SplitChoice {
    int variant = 0;        // kernel of the split launch (6 or 10)
    int parts = 1;
    size_t tickets_bytes = 0, partial_bytes = 0;
    size_t bytes() const { return tickets_bytes + partial_bytes; }
};

bool split_choice(const spatha_spmm_plan* plan, int N, int requested, int chosen, bool fused, SplitChoice* out) {
    using namespace spatha;
    if (requested != SPMM_VARIANT_AUTO || plan->cus < 8 || plan->half_tiles) return false;
    int var = chosen;
    if (var == SPMM_VARIANT_WS128x128_S3) var = SPMM_VARIANT_W128x128_S3;      // the store waves have no hand-over
    // (the 128 x 256 tiles with 64 x 64 consumer blocks are chosen for short k-loops only, where a split never pays)
    if (var != SPMM_VARIANT_W128x128_S3 && var != SPMM_VARIANT_T128x256_S3) return false;
    if (!variant_ok(plan, N, var, fused)) return false;
    const int bm = spmm_variant_bm(var), bn = spmm_variant_bn(var), S = plan->S;
    const int grid = (plan->cus / 8) * 8;
    const int64_t tiles = (int64_t)(plan->geo.rows / bm) * ((N + bn - 1) / bn);
    if (tiles * 2 > grid) return false;
    // as many parts as fit one round of the CUs, at most four, S a multiple of them
    int k = (int)std::min<int64_t>(grid / tiles, 4);
    while (k > 1 && (S % k != 0 || S / k < SPATHA_KSPLIT_MIN_PART_STEPS || S - S / k < SPATHA_KSPLIT_MIN_SAVED_STEPS)) --k;
    if (k < 2) return false;
    SplitChoice c;
    c.variant = var;
    c.parts = k;
    const int blocks_per_tile = (bm / 64) * (bn / 64);
    c.tickets_bytes = (((size_t)tiles * blocks_per_tile * 4) + 255) & ~(size_t)255;
    c.partial_bytes = (size_t)tiles * c.parts * bm * bn * 4;
    *out = c;
    return true;
}

// Does C leave by non-temporal stores, past the 256 MB memory-side cache?  From 96 MB on, unless the caller says that it is read right
// behind this call, and where the rows of C are whole 64-byte pieces.
// 4096 x 1024 x 16384 (134 MB), V = 32 .. 128, m = 4 .. 32, both layouts, launches following each other for long: three and six sets of
// operands and results in turn 1.05-1.7x ahead (64:2:8 73 -> 57-61 us row-major, 66 -> 56 transposed, 128:2:32 53.6 -> 31.6); one set,
// which stays in the cache, 0.92-1.05x (64:2:16 row-major 44.8 -> 47.6, transposed 44.3 -> 46.3; 128:2:32 30.3 -> 31.6 and 33.4 -> 31.7;
// 49152 x 12288 x 2048 at 128:2:16, 201 MB, 458 -> 440).  12288 x 12288 x 4096 at 128:2:10, 100 MB behind 77 k-steps, is 1-2 % behind
// on rotating sets.  Results of 50 to 67 MB 0.98-1.04x, smaller ones level or up to 4 % behind.  A chain of layers reads each result
// back from that cache: with such stores in all of them the two encoder layers of BERT-large at 32 x 512 tokens took 695 us, 681 without.
// Rows of another length end in parts of 64-byte pieces, which the cache would put together and memory has to read first: the
// same products on 16368 and 16376 columns 0.48-0.98x on one set and 0.94-1.5x on several (128:2:32 38.5 -> 80.6 and 85 -> 81 us),
// 12288 x 2048 .. 8192 x 4104 at 128:2:20 0.82-0.95x and 0.89-1.01x.
bool streams_out(const spatha_spmm_plan* plan, int N, int out_layout, bool read_next) {
    if (read_next || (out_layout == SPATHA_OUT_ROW_MAJOR && N % 32 != 0)) return false;
    return (int64_t)plan->geo.rows * N * 2 >= (96ll << 20);
}
}  // namespace

namespace spatha {

int note_hip_error(hipError_t e) { return hip_fail(e); }

void plan_layout(int rows, int m, int v, int ksp, PlanLayout* out) {
    out->S = (ksp + 31) / 32;
    out->half_tiles = (v % 64 != 0);      // V = 32, 96, ...: a wave tile spans two V blocks
    out->apack_bytes = (size_t)((rows + 63) / 64) * out->S * APACK_BLOCK;    // rows % 64 == 32: V a multiple of 32 only
    out->rowtab_bytes = (size_t)(rows / v) * out->S * 64 * 4;
    out->gtab_bytes = 0;
    if ((m <= 8 && rows % 256 == 0) || (m <= 16 && rows % 512 == 0 && !out->half_tiles)) {
        // gather table of the dense-staged kernels: one entry per 64-row block, or per 32-row block when V % 64 != 0
        const int block_rows = out->half_tiles ? 32 : 64;
        out->gtab_bytes = (size_t)(rows / block_rows) * out->S * 64 * 2;
    }
}

hipError_t plan_pack(const spatha_spmm_plan* plan, const uint16_t* values_dev, const uint32_t* metadata_dev,
                     const uint32_t* columns_dev, hipStream_t stream) {
    const spatha_vnm_geometry& geo = plan->geo;
    hipError_t e = launch_pack(values_dev, metadata_dev, columns_dev, geo.rows, geo.cols, geo.m, geo.v, geo.ksp, plan->S,
                               plan->half_tiles, plan->apack, plan->rowtab, stream);
    if (e != hipSuccess) return e;
    if (plan->gtab) {
        e = launch_pack_gtab(columns_dev, geo.rows, geo.m, geo.v, geo.ksp, plan->S, plan->half_tiles ? 32 : 64, plan->gtab, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace spatha

extern "C" {

const char* spatha_status_string(int status) {
    switch (status) {
        case SPATHA_OK: return "ok";
        case SPATHA_ERR_BAD_ARGUMENT: return "bad argument";
        case SPATHA_ERR_BAD_SHAPE: return "shape not representable in V:N:M (rows % V, V % 32, m >= 4, N % 8)";
        case SPATHA_ERR_UNSUPPORTED: return "no kernel for this configuration";
        case SPATHA_ERR_HIP: return "HIP runtime error";
        case SPATHA_ERR_NO_DEVICE: return "no HIP device";
        case SPATHA_ERR_TOO_LARGE: return "size beyond the entry point's capacity";
        case SPATHA_ERR_IO: return "file missing, truncated, not a V:N:M container, or corrupt";
        default: return "unknown status";
    }
}

int spatha_last_hip_error(void) { return g_last_hip_error; }

const char* spatha_version(void) { return "0.1.0"; }

int spatha_vnm_geometry_init(int rows, int cols, int n, int m, int v, spatha_vnm_geometry* out) {
    return spatha::geometry_init(rows, cols, n, m, v, out);
}

int spatha_vnm_random_pattern(int rows, int cols, int n, int m, int v, uint32_t* metadata, uint32_t* columns) {
    return spatha::random_pattern(rows, cols, n, m, v, metadata, columns);
}

int spatha_fill_rand_small_ints_f16(uint16_t* out, int64_t count) {
    if (!out || count < 0) return SPATHA_ERR_BAD_ARGUMENT;
    // fp16 bit patterns of -4..4
    static const uint16_t enc[9] = {0xC400, 0xC200, 0xC000, 0xBC00, 0x0000, 0x3C00, 0x4000, 0x4200, 0x4400};
    for (int64_t i = 0; i < count; i++) out[i] = enc[std::rand() % 9];
    return SPATHA_OK;
}

int spatha_benchmark_inputs_f16(int rows, int cols, int ncols_b, int n, int m, int v, uint16_t* b, uint32_t* metadata,
                                uint32_t* columns, uint16_t* values) {
    spatha_vnm_geometry geo;
    int st = spatha::geometry_init(rows, cols, n, m, v, &geo);
    if (st != SPATHA_OK) return st;
    if (!b || !metadata || !columns || !values || ncols_b <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    st = spatha_fill_rand_small_ints_f16(b, (int64_t)cols * ncols_b);
    if (st == SPATHA_OK) st = spatha::random_pattern(rows, cols, n, m, v, metadata, columns);
    if (st == SPATHA_OK) st = spatha_fill_rand_small_ints_f16(values, geo.n_values);
    return st;
}

int spatha_vnm_encode_f32(const float* dense, const int32_t* mask, const uint32_t* columns, int rows, int cols, int n,
                          int m, int v, float* values, uint32_t* metadata, int threads) {
    return spatha::encode_f32(dense, mask, columns, rows, cols, n, m, v, values, metadata, threads);
}
int spatha_vnm_encode_f16(const uint16_t* dense, const int32_t* mask, const uint32_t* columns, int rows, int cols,
                          int n, int m, int v, uint16_t* values, uint32_t* metadata, int threads) {
    return spatha::encode_f16(dense, mask, columns, rows, cols, n, m, v, values, metadata, threads);
}
int spatha_vnm_decode_f32(const float* values, const uint32_t* metadata, const uint32_t* columns, int rows, int cols,
                          int n, int m, int v, float* dense, int threads) {
    return spatha::decode_f32(values, metadata, columns, rows, cols, n, m, v, dense, threads);
}
int spatha_vnm_decode_f16(const uint16_t* values, const uint32_t* metadata, const uint32_t* columns, int rows,
                          int cols, int n, int m, int v, uint16_t* dense, int threads) {
    return spatha::decode_f16(values, metadata, columns, rows, cols, n, m, v, dense, threads);
}
int spatha_vnm_select_columns_f32(const float* dense_abs, int rows, int cols, int n, int m, int v, int32_t* masks,
                                  int32_t* columns, int threads) {
    return spatha::select_columns_f32(dense_abs, rows, cols, n, m, v, masks, columns, threads);
}
int spatha_vnm_file_write(const char* path, int rows, int cols, int n, int m, int v, int value_bits, const void* values,
                          const uint32_t* metadata, const uint32_t* columns) {
    return spatha::file_write(path, rows, cols, n, m, v, value_bits, values, metadata, columns);
}

int spatha_vnm_file_info(const char* path, spatha_vnm_geometry* geometry, int* value_bits) {
    return spatha::file_info(path, geometry, value_bits);
}

int spatha_vnm_file_read(const char* path, void* values, uint32_t* metadata, uint32_t* columns) {
    return spatha::file_read(path, values, metadata, columns);
}

int spatha_vnm_select_columns_f32_gpu(const float* dense_abs, int rows, int cols, int n, int m, int v, int32_t* masks,
                                      int32_t* columns, int threads, int exact_ties, void* stream) {
    spatha_vnm_geometry geo;
    int st = spatha::geometry_init(rows, cols, n, m, v, &geo);
    if (st) return st;
    if (!dense_abs || !masks || !columns) return SPATHA_ERR_BAD_ARGUMENT;
    int per_block = 0;
    const int tasks = spatha::select_task_count(rows, cols, m, v, &per_block);
    std::vector<spatha::GroupTask> winners((size_t)tasks);
    if (tasks > 0) {
        if ((size_t)v * (size_t)m * sizeof(float) > 150u * 1024u) return SPATHA_ERR_TOO_LARGE;   // one V x m block per workgroup in LDS
        float* d_abs = nullptr;
        int32_t* d_out = nullptr;
        std::vector<int32_t> h_out((size_t)tasks * 4);
        const size_t bytes = (size_t)rows * (size_t)cols * sizeof(float);
        hipStream_t s = (hipStream_t)stream;
        hipError_t e = hipMalloc((void**)&d_abs, bytes);
        if (e == hipSuccess) e = hipMalloc((void**)&d_out, h_out.size() * sizeof(int32_t));
        if (e == hipSuccess) e = hipMemcpyAsync(d_abs, dense_abs, bytes, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = spatha::launch_select_winners_f32(d_abs, rows, cols, m, v, device_cus(), d_out, per_block, s);
        if (e == hipSuccess) e = hipMemcpyAsync(h_out.data(), d_out, h_out.size() * sizeof(int32_t), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (d_abs) (void)hipFree(d_abs);
        if (d_out) (void)hipFree(d_out);
        if (e != hipSuccess) return hip_fail(e);
        for (int i = 0; i < tasks; i++) {
            winners[(size_t)i].any = h_out[(size_t)i * 4 + 1] != 0;
            for (int k = 0; k < 4; k++) winners[(size_t)i].best[k] = h_out[(size_t)i * 4 + k];
        }
    }
    return spatha::select_columns_with_winners(dense_abs, rows, cols, n, m, v, tasks > 0 ? winners.data() : nullptr,
                                               exact_ties != 0, masks, columns, threads);
}

int spatha_vnm_convert_gpu(const void* dense_dev, int value_bits, int rows, int cols, int n, int m, int v, uint16_t* values_dev,
                           uint32_t* metadata_dev, uint32_t* columns_dev, void* stream) {
    spatha_vnm_geometry geo;
    int st = spatha::geometry_init(rows, cols, n, m, v, &geo);
    if (st) return st;
    if (!dense_dev || !values_dev || !metadata_dev || !columns_dev || (value_bits != 16 && value_bits != 32)) return SPATHA_ERR_BAD_ARGUMENT;
    // (four columns, two words of values and one of metadata are written at a time)
    if (((uintptr_t)dense_dev & (uintptr_t)(value_bits / 8 - 1)) || ((uintptr_t)values_dev & 7) || ((uintptr_t)metadata_dev & 3) ||
        ((uintptr_t)columns_dev & 15))
        return SPATHA_ERR_BAD_ARGUMENT;
    const int tasks = spatha::select_task_count(rows, cols, m, v, nullptr);
    if (tasks > 0 && (size_t)v * (size_t)m * sizeof(float) > 150u * 1024u) return SPATHA_ERR_TOO_LARGE;
    const hipError_t e = spatha::launch_convert(dense_dev, value_bits, rows, cols, m, v, geo.ksp, device_cus(), values_dev, metadata_dev,
                                                (int32_t*)columns_dev, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_vnm_decode_f16_gpu(const uint16_t* values_dev, const uint32_t* metadata_dev, const uint32_t* columns_dev, int rows, int cols,
                              int n, int m, int v, uint16_t* dense_dev, uint32_t* bad_dev, void* stream) {
    spatha_vnm_geometry geo;
    int st = spatha::geometry_init(rows, cols, n, m, v, &geo);
    if (st) return st;
    if (!values_dev || !metadata_dev || !columns_dev || !dense_dev || !bad_dev) return SPATHA_ERR_BAD_ARGUMENT;
    if (((uintptr_t)values_dev & 3) || ((uintptr_t)metadata_dev & 3) || ((uintptr_t)columns_dev & 3) || ((uintptr_t)bad_dev & 3) ||
        ((uintptr_t)dense_dev & (uintptr_t)(cols % 8 == 0 ? 15 : 1)))
        return SPATHA_ERR_BAD_ARGUMENT;
    const hipError_t e = spatha::launch_decode_f16(values_dev, metadata_dev, columns_dev, rows, cols, m, v, geo.ksp, dense_dev, bad_dev,
                                                   (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_vnm_pack_meta_blob(const uint32_t* metadata, int64_t n_metadata, const uint32_t* columns,
                              int64_t n_columns, uint32_t* blob, int64_t* columns_offset_words,
                              int64_t* blob_words) {
    return spatha::pack_meta_blob(metadata, n_metadata, columns, n_columns, blob, columns_offset_words, blob_words);
}

int spatha_spmm_plan_create(int rows, int cols, int n, int m, int v, const uint16_t* values_dev,
                            const uint32_t* metadata_dev, const uint32_t* columns_dev, void* stream,
                            spatha_spmm_plan** out) {
    if (!out) return SPATHA_ERR_BAD_ARGUMENT;
    *out = nullptr;
    spatha_vnm_geometry geo;
    int st = spatha::geometry_init(rows, cols, n, m, v, &geo);
    if (st) return st;
    if (!values_dev || !metadata_dev || !columns_dev) return SPATHA_ERR_BAD_ARGUMENT;
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev == 0) { g_last_hip_error = (int)e; return SPATHA_ERR_NO_DEVICE; }
    spatha_spmm_plan* plan = new (std::nothrow) spatha_spmm_plan();
    if (!plan) return SPATHA_ERR_BAD_ARGUMENT;
    spatha::PlanLayout lay;
    spatha::plan_layout(rows, m, v, geo.ksp, &lay);
    plan->geo = geo;
    plan->S = lay.S;
    plan->half_tiles = lay.half_tiles;
    plan->apack = nullptr; plan->rowtab = nullptr; plan->zeros = nullptr; plan->gtab = nullptr;
    plan->apack_bytes = lay.apack_bytes; plan->rowtab_bytes = lay.rowtab_bytes;
    plan->gtab_bytes = lay.gtab_bytes;
    e = hipGetDevice(&plan->device);
    if (e != hipSuccess) { delete plan; return hip_fail(e); }
    plan->cus = 0;
    if (hipDeviceGetAttribute(&plan->cus, hipDeviceAttributeMultiprocessorCount, plan->device) != hipSuccess) plan->cus = 0;
    if ((e = hipMalloc((void**)&plan->apack, lay.apack_bytes)) != hipSuccess ||
        (e = hipMalloc((void**)&plan->rowtab, lay.rowtab_bytes)) != hipSuccess ||
        (e = hipMalloc(&plan->zeros, 1024)) != hipSuccess ||
        (e = hipMemsetAsync(plan->zeros, 0, 1024, (hipStream_t)stream)) != hipSuccess ||
        (lay.gtab_bytes && (e = hipMalloc((void**)&plan->gtab, lay.gtab_bytes)) != hipSuccess) ||
        (e = spatha::plan_pack(plan, values_dev, metadata_dev, columns_dev, (hipStream_t)stream)) != hipSuccess) {
        spatha_spmm_plan_destroy(plan);
        return hip_fail(e);
    }
    // the derived copies are complete before the plan is handed out: a later run on another stream has nothing to order
    // itself against
    if ((e = hipStreamSynchronize((hipStream_t)stream)) != hipSuccess) {
        spatha_spmm_plan_destroy(plan);
        return hip_fail(e);
    }
    *out = plan;
    return SPATHA_OK;
}

int spatha_spmm_plan_destroy(spatha_spmm_plan* plan) {
    if (!plan) return SPATHA_OK;
    hipError_t first = hipSuccess, e;
    if (plan->apack && (e = hipFree(plan->apack)) != hipSuccess && first == hipSuccess) first = e;
    if (plan->rowtab && (e = hipFree(plan->rowtab)) != hipSuccess && first == hipSuccess) first = e;
    if (plan->zeros && (e = hipFree(plan->zeros)) != hipSuccess && first == hipSuccess) first = e;
    if (plan->gtab && (e = hipFree(plan->gtab)) != hipSuccess && first == hipSuccess) first = e;
    delete plan;
    return first == hipSuccess ? SPATHA_OK : hip_fail(first);
}

}  // extern "C"

int spatha::plan_run_check(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev,
                           const uint16_t* out_dev, int out_layout, int activation, bool fused_entry, int variant,
                           int* chosen) {
    if (!plan || !B_dev || !out_dev || N <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (out_layout != SPATHA_OUT_ROW_MAJOR && out_layout != SPATHA_OUT_TRANSPOSED) return SPATHA_ERR_BAD_ARGUMENT;
    if (!fused_entry && out_layout == SPATHA_OUT_ROW_MAJOR && bias_dev) return SPATHA_ERR_BAD_ARGUMENT;
    if (activation != SPATHA_ACT_NONE && activation != SPATHA_ACT_GELU && activation != SPATHA_ACT_GELU_TANH)
        return SPATHA_ERR_BAD_ARGUMENT;
    if (N % 8 != 0) return SPATHA_ERR_BAD_SHAPE;      // 16-byte row segments of B and C
    if (((uintptr_t)B_dev & 15) || ((uintptr_t)out_dev & 15) || ((uintptr_t)bias_dev & 15)) return SPATHA_ERR_BAD_ARGUMENT;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev != plan->device) return SPATHA_ERR_BAD_ARGUMENT;   // plans live on one device
    // the bias of the transposed layout alone stays in the write-out itself
    const bool fuse = activation != SPATHA_ACT_NONE || (out_layout == SPATHA_OUT_ROW_MAJOR && bias_dev);
    const int var = pick_variant(plan, N, variant, fuse, out_layout);
    if (var < 0) return SPATHA_ERR_UNSUPPORTED;
    if (chosen) *chosen = var;
    return SPATHA_OK;
}

int spatha::plan_run(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev, uint16_t* out_dev,
                     int out_layout, int activation, bool fused_entry, int variant, void* stream, void* workspace,
                     size_t workspace_bytes, bool read_next) {
    int var = -1;
    const int status = plan_run_check(plan, B_dev, N, bias_dev, out_dev, out_layout, activation, fused_entry, variant, &var);
    if (status != SPATHA_OK) return status;
    const bool fuse = activation != SPATHA_ACT_NONE || (out_layout == SPATHA_OUT_ROW_MAJOR && bias_dev);
    spatha::SpmmParams p;
    p.apack = plan->apack; p.rowtab = plan->rowtab;
    p.B = B_dev; p.bias = bias_dev; p.C = out_dev; p.zeros = plan->zeros; p.gtab = plan->gtab;
    p.gtab_bytes = (uint32_t)plan->gtab_bytes;
    p.rows = plan->geo.rows; p.cols = plan->geo.cols; p.N = N; p.b_pitch = N; p.S = plan->S; p.v = plan->geo.v; p.m = plan->geo.m;
    const int bm = spatha::spmm_variant_bm(var), bn = spatha::spmm_variant_bn(var);
    p.tiles_m = (plan->geo.rows + bm - 1) / bm;     // (only the half-tile kernels see rows % 64 != 0: a padded last tile)
    p.tiles_n = (N + bn - 1) / bn;
    p.b_bytes = (uint32_t)((uint64_t)plan->geo.cols * (uint64_t)N * 2u);     // only read by variants that passed variant_ok
    p.apack_bytes = (uint32_t)plan->apack_bytes;
    p.rowtab_bytes = (uint32_t)plan->rowtab_bytes;
    p.fuse = fuse ? 1 : 0; p.act = activation;
    p.cus = plan->cus > 0 ? plan->cus : 256;
    p.stream_out = streams_out(plan, N, out_layout, read_next) ? 1 : 0;
    p.walk_group = 1;
    if (var == spatha::SPMM_VARIANT_UP512x128_S3) {
        // Packed A larger than an XCD's L2 (plain 2:4 on a 4096-row matrix: 4.7 MB against 4 MB; it is then fetched again in
        // every round, 160 MB per launch): tile rows in groups of four, so that an XCD only
        // ever sees four of them (2.4 MB, resident) and reads twice as many tile columns of B instead.  2:4 FFN-up: 85-86
        // against 87-89 us.  Where A fits anyway (64:2:8: 2.4 MB) the default walk reads less.
        const size_t a_bytes = plan->apack_bytes + plan->gtab_bytes, four_rows = a_bytes / p.tiles_m * 4;
        if (p.tiles_m % 4 == 0 && p.tiles_m >= 8 && p.tiles_n >= 32 && a_bytes > (4u << 20) && four_rows <= (3u << 20)) p.walk_group = -4;
    }
    p.ksplit = 1; p.partial = nullptr; p.partial_bytes = 0; p.tickets = nullptr;
    p.debug = 0; p.skew = 0; p.prof = nullptr;
#ifdef SPATHA_DEV_PROFILE
    // development builds only: switch parts of a kernel off for time accounting (results are then wrong on purpose)
    { const char* d = std::getenv("SPATHA_DEBUG_KNOBS"); p.debug = d ? std::atoi(d) : 0; }
    { const char* d = std::getenv("SPATHA_SKEW"); p.skew = d ? std::atoi(d) : 0; }
    { const char* d = std::getenv("SPATHA_PROF_PTR"); if (d) p.prof = (long long*)std::strtoull(d, nullptr, 0); }
#endif
    SplitChoice sc;
    if (workspace && split_choice(plan, N, variant, var, fuse, &sc) && workspace_bytes >= sc.bytes() &&
        ((uintptr_t)workspace & 255) == 0) {
        // every tile's k-loop in parts: the walk's m-tiles are (row tile, part) pairs
        spatha::SpmmParams q = p;
        q.tiles_m = (plan->geo.rows / spatha::spmm_variant_bm(sc.variant)) * sc.parts;
        q.tiles_n = (N + spatha::spmm_variant_bn(sc.variant) - 1) / spatha::spmm_variant_bn(sc.variant);
        q.ksplit = sc.parts;
        q.tickets = (uint32_t*)workspace;       // zero: cleared once by spatha_spmm_workspace_init, put back by every completed run
        q.partial = (float*)((char*)workspace + sc.tickets_bytes);
        q.partial_bytes = (uint32_t)sc.partial_bytes;
        const hipError_t e2 = spatha::launch_spmm(sc.variant, out_layout, q, (hipStream_t)stream);
        return e2 == hipSuccess ? SPATHA_OK : hip_fail(e2);
    }
    if (const int rest_rows = uneven_rest_rows(plan, N, variant, var, fuse)) {
        const int main_rows = plan->geo.rows - rest_rows;
        spatha::SpmmParams head = p, tail = p;
        head.tiles_m = main_rows / 128;
        const size_t a_off = (size_t)(main_rows / 64) * plan->S * spatha::APACK_BLOCK;
        const size_t rt_off = (size_t)(main_rows / plan->geo.v) * plan->S * 64 * 4;
        tail.apack = (const uint16_t*)((const char*)plan->apack + a_off);
        tail.apack_bytes = (uint32_t)(plan->apack_bytes - a_off);
        tail.rowtab = (const uint32_t*)((const char*)plan->rowtab + rt_off);
        tail.rowtab_bytes = (uint32_t)(plan->rowtab_bytes - rt_off);
        if (bias_dev) tail.bias = bias_dev + main_rows;
        // (p.rows stays the full row count: these kernels use it as the row stride of the transposed layout only)
        tail.C = out_layout == SPATHA_OUT_TRANSPOSED ? out_dev + main_rows : out_dev + (size_t)main_rows * N;
        tail.tiles_m = rest_rows / 128;
        tail.tiles_n = (N + 127) / 128;
        // Which way the tail's tiles are walked decides what an XCD's workgroups (grid / 8 tiles at a time) pull into its L2
        // per round: column-first, the A operands of up to grid / 8 tile rows + few tile columns of B; row-first, all tile
        // columns of few tile rows.  GPT-3 FFN matrix at 256 tokens (0.44 MB of A per tile row, two tile columns of 3.1 MB):
        // 13.4 against 17.3 MB row-first, the second launch fetches 108 instead of 142 MB; with few tile rows and many tile
        // columns (1280 x 5120 at 8192 tokens: 2 x 128 tiles) column-first moves half as much.
        {
            const int64_t at_a_time = std::max(1, p.cus / 8);
            const double a_row = (double)plan->apack_bytes / (plan->geo.rows / 128.0), b_col = (double)plan->geo.cols * 128 * 2;
            const int64_t tm = tail.tiles_m, tn = tail.tiles_n;
            const double col_first = (double)std::min(at_a_time, tm) * a_row + (double)((at_a_time + tm - 1) / tm) * b_col;
            const double row_first = (double)((at_a_time + tn - 1) / tn) * a_row + (double)std::min(at_a_time, tn) * b_col;
            tail.walk_group = row_first < col_first ? 0 : 1;
        }
        hipError_t e2 = spatha::launch_spmm(var, out_layout, head, (hipStream_t)stream);
        if (e2 == hipSuccess) e2 = spatha::launch_spmm(spatha::SPMM_VARIANT_W128x128_S3, out_layout, tail, (hipStream_t)stream);
        return e2 == hipSuccess ? SPATHA_OK : hip_fail(e2);
    }
    hipError_t e = spatha::launch_spmm(var, out_layout, p, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

extern "C" {

int spatha_spmm_run(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev,
                    uint16_t* out_dev, int out_layout, int variant, void* stream) {
    return spatha::plan_run(plan, B_dev, N, bias_dev, out_dev, out_layout, SPATHA_ACT_NONE, false, variant, stream);
}

int spatha_spmm_run_fused(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev,
                          uint16_t* out_dev, int out_layout, int activation, int variant, void* stream) {
    return spatha::plan_run(plan, B_dev, N, bias_dev, out_dev, out_layout, activation, true, variant, stream);
}

int spatha_spmm_run_layer(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev, uint16_t* out_dev,
                          int out_layout, int activation, void* workspace_dev, size_t workspace_bytes, void* stream) {
    return spatha::plan_run(plan, B_dev, N, bias_dev, out_dev, out_layout, activation, true, spatha::SPMM_VARIANT_AUTO, stream,
                            workspace_dev, workspace_bytes, true);
}

namespace {
// Is `var`, chosen for the next multiple of 8, a kernel that takes N columns of B in rows b_pitch apart, and faster from them than from a
// padded copy?
bool ragged_kernel_takes(const spatha_spmm_plan* plan, int var, int b_pitch, int N) {
    if (var != spatha::SPMM_VARIANT_SKINNY && var != spatha::SPMM_VARIANT_DIRECT64 && var != spatha::SPMM_VARIANT_HDIRECT32) return false;
    // Loads of two or four columns at odd addresses take the L1 a third longer: 0.3 ns per 64 x 64 block and k-step over the chip
    // (12288 x 12288 at 128:2:16 and 17 tokens, 9216 of them, 11.5 -> 14.4 us; 49152 x 12288 at 64:2:4, 147456 of them, 132 -> 170;
    // 16 tokens and fewer, and even counts in their place, level), the padded copy 2.6 us.
    if (N > 16 && b_pitch % (N <= 32 ? 2 : 4) != 0 && (int64_t)(plan->geo.rows / 64) * plan->S * ((N + 63) / 64) > 8000) return false;
    return (uint64_t)plan->geo.cols * (uint64_t)b_pitch * 2u < 0xE0000000ull;
}
}  // namespace

int spatha_spmm_ragged_route(const spatha_spmm_plan* plan, int N, int out_layout, int fuse) {
    if (!plan || N <= 0 || N > INT32_MAX - 8) return 0;
    const int padded = (N + 7) / 8 * 8, var = pick_variant(plan, padded, spatha::SPMM_VARIANT_AUTO, fuse != 0, out_layout);
    return var < 0 ? 0 : ragged_kernel_takes(plan, var, N, N) ? 2 : ragged_kernel_takes(plan, var, padded, N) ? 1 : 0;
}

int spatha_spmm_run_ragged(const spatha_spmm_plan* plan, const uint16_t* B_dev, int b_pitch, int N, const uint16_t* bias_dev, uint16_t* out_dev,
                           int out_layout, int activation, int fused, void* stream) {
    if (N <= 0 || N > INT32_MAX - 8 || b_pitch < N || b_pitch > INT32_MAX - 8) return SPATHA_ERR_BAD_ARGUMENT;
    // the checks and the choice of the padded product: what it refuses is refused, and the sums run in its order
    const int padded = (N + 7) / 8 * 8;
    int var = -1;
    const int status = spatha::plan_run_check(plan, B_dev, padded, bias_dev, out_dev, out_layout, activation, fused != 0,
                                              spatha::SPMM_VARIANT_AUTO, &var);
    if (status != SPATHA_OK) return status;
    if (!ragged_kernel_takes(plan, var, b_pitch, N)) return SPATHA_ERR_UNSUPPORTED;
    spatha::SpmmParams p = {};
    p.apack = plan->apack; p.rowtab = plan->rowtab;
    p.B = B_dev; p.bias = bias_dev; p.C = out_dev; p.zeros = plan->zeros;
    p.rows = plan->geo.rows; p.cols = plan->geo.cols; p.N = N; p.b_pitch = b_pitch; p.S = plan->S; p.v = plan->geo.v; p.m = plan->geo.m;
    p.b_bytes = (uint32_t)((uint64_t)plan->geo.cols * (uint64_t)b_pitch * 2u);
    p.apack_bytes = (uint32_t)plan->apack_bytes;
    p.rowtab_bytes = (uint32_t)plan->rowtab_bytes;
    p.fuse = activation != SPATHA_ACT_NONE || (out_layout == SPATHA_OUT_ROW_MAJOR && bias_dev) ? 1 : 0;
    p.act = activation;
    p.cus = plan->cus > 0 ? plan->cus : 256;
    p.ksplit = 1;
    const hipError_t e = spatha::launch_spmm(var, out_layout, p, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_spmm_run_tokens(const spatha_spmm_plan* plan, const uint16_t* x_dev, int tokens, const uint16_t* bias_dev, uint16_t* out_dev,
                           void* stream) {
    if (!plan || !x_dev || !out_dev || tokens <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (((uintptr_t)x_dev & 15) || ((uintptr_t)out_dev & 15) || ((uintptr_t)bias_dev & 15)) return SPATHA_ERR_BAD_ARGUMENT;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev != plan->device) return SPATHA_ERR_BAD_ARGUMENT;
    const int cus = plan->cus > 0 ? plan->cus : 256;
    if (!spatha::token_major_fits(plan->geo.rows, plan->geo.cols, tokens, plan->half_tiles != 0, cus)) return SPATHA_ERR_UNSUPPORTED;
    spatha::SpmmParams p = {};
    p.apack = plan->apack; p.rowtab = plan->rowtab;
    p.B = x_dev; p.bias = bias_dev; p.C = out_dev; p.zeros = plan->zeros;
    p.rows = plan->geo.rows; p.cols = plan->geo.cols; p.N = tokens; p.S = plan->S; p.v = plan->geo.v; p.m = plan->geo.m;
    p.cus = cus;
    p.act = SPATHA_ACT_NONE;
    p.ksplit = 1;
    const hipError_t e = spatha::launch_token_major(p, plan->half_tiles != 0, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

size_t spatha_spmm_workspace_bytes(const spatha_spmm_plan* plan, int N, int out_layout, int fused) {
    if (!plan || N <= 0 || N % 8 != 0) return 0;
    const int var = pick_variant(plan, N, spatha::SPMM_VARIANT_AUTO, fused != 0, out_layout);
    SplitChoice sc;
    if (var < 0 || !split_choice(plan, N, spatha::SPMM_VARIANT_AUTO, var, fused != 0, &sc)) return 0;
    return sc.bytes();
}

int spatha_spmm_workspace_init(void* workspace_dev, size_t workspace_bytes, void* stream) {
    if (!workspace_dev || ((uintptr_t)workspace_dev & 255) || workspace_bytes % 4 != 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (workspace_bytes / 4 > 0x7fffffffull) return SPATHA_ERR_TOO_LARGE;
    const hipError_t e = spatha::launch_clear_words((uint32_t*)workspace_dev, (int)(workspace_bytes / 4), (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_spmm_run_ws(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev, uint16_t* out_dev,
                       int out_layout, int activation, void* workspace_dev, size_t workspace_bytes, void* stream) {
    return spatha::plan_run(plan, B_dev, N, bias_dev, out_dev, out_layout, activation, true, spatha::SPMM_VARIANT_AUTO, stream,
                            workspace_dev, workspace_bytes);
}

int spatha_spmm_num_variants(void) { return spatha::SPMM_VARIANT_COUNT; }

const char* spatha_spmm_kernel_name(const spatha_spmm_plan* plan, int N, int out_layout, int variant) {
    if (!plan) return nullptr;
    int var = pick_variant(plan, N, variant, false, out_layout);
    if (var < 0) return nullptr;
    if (uneven_rest_rows(plan, N, variant, var, false))     // two launches: the rest of an uneven last round on 128 x 128 tiles
        return var == spatha::SPMM_VARIANT_T128x256_S3 ? "smfmac16x16x64_warpspec_tall_tile128x256_3stage+rest_on_tile128x128"
                                                       : "smfmac16x16x64_warpspec_tile128x256_3stage+rest_on_tile128x128";
    if (const char* form = spatha::spmm_direct_name(var, plan->geo.rows, N, plan->S, plan->cus > 0 ? plan->cus : 256)) return form;
    return spatha::spmm_variant_name(var);
}

int spatha_spmm_time(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev,
                     uint16_t* out_dev, int out_layout, int variant, int warmup, int iters, void* stream,
                     float* ms_per_launch) {
    if (!ms_per_launch || iters <= 0 || warmup < 0) return SPATHA_ERR_BAD_ARGUMENT;
    hipStream_t s = (hipStream_t)stream;
    for (int i = 0; i < warmup; i++) {
        int st = spatha_spmm_run(plan, B_dev, N, bias_dev, out_dev, out_layout, variant, stream);
        if (st) return st;
    }
    hipEvent_t t0, t1;
    hipError_t e;
    if ((e = hipEventCreate(&t0)) != hipSuccess) return hip_fail(e);
    if ((e = hipEventCreate(&t1)) != hipSuccess) { (void)hipEventDestroy(t0); return hip_fail(e); }
    int st = SPATHA_OK;
    e = hipEventRecord(t0, s);
    for (int i = 0; i < iters && e == hipSuccess && st == SPATHA_OK; i++)
        st = spatha_spmm_run(plan, B_dev, N, bias_dev, out_dev, out_layout, variant, stream);
    if (e == hipSuccess) e = hipEventRecord(t1, s);
    if (e == hipSuccess) e = hipEventSynchronize(t1);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, t0, t1);
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    if (st) return st;
    if (e != hipSuccess) return hip_fail(e);
    *ms_per_launch = ms / (float)iters;
    return SPATHA_OK;
}

int spatha_spmm_tune(const spatha_spmm_plan* plan, const uint16_t* B_dev, int N, const uint16_t* bias_dev,
                     uint16_t* out_dev, int out_layout, int warmup, int iters, void* stream, int* best_variant,
                     float* best_ms, float* auto_ms, float* ms_per_variant) {
    if (!best_variant || !best_ms) return SPATHA_ERR_BAD_ARGUMENT;
    // (a first, untimed pass of the automatic choice: argument checks, and the clocks are up when the first id is timed)
    float t_auto = 0.f;
    int st = spatha_spmm_time(plan, B_dev, N, bias_dev, out_dev, out_layout, spatha::SPMM_VARIANT_AUTO, warmup, iters, stream, &t_auto);
    if (st) return st;
    int best = spatha::SPMM_VARIANT_AUTO;
    float t_best = 0.f;
    // (the ids that ms_per_variant has places for, then the one behind them)
    for (int id = 1; id <= spatha::SPMM_VARIANT_HDIRECT32; id++) {
        float* const place = ms_per_variant && id < spatha::SPMM_VARIANT_COUNT ? ms_per_variant + id : nullptr;
        if (place) *place = -1.f;
        if (!variant_ok(plan, N, id, false)) continue;
        float t = 0.f;
        st = spatha_spmm_time(plan, B_dev, N, bias_dev, out_dev, out_layout, id, warmup, iters, stream, &t);
        if (st == SPATHA_ERR_UNSUPPORTED) continue;     // (accepted by the shape checks, refused by the kernel's launcher)
        if (st) return st;
        if (place) *place = t;
        if (best == spatha::SPMM_VARIANT_AUTO || t < t_best) { t_best = t; best = id; }
    }
    // the automatic choice last, in the same warm state as the ids: it wins ties (it may be one of them)
    st = spatha_spmm_time(plan, B_dev, N, bias_dev, out_dev, out_layout, spatha::SPMM_VARIANT_AUTO, warmup, iters, stream, &t_auto);
    if (st) return st;
    if (auto_ms) *auto_ms = t_auto;
    if (ms_per_variant) ms_per_variant[0] = t_auto;
    if (best == spatha::SPMM_VARIANT_AUTO || t_auto <= t_best) { t_best = t_auto; best = spatha::SPMM_VARIANT_AUTO; }
    *best_variant = best;
    *best_ms = t_best;
    return SPATHA_OK;
}

int spatha_dense_gemm_f16(const uint16_t* A_dev, const uint16_t* B_dev, int rows, int cols, int N, uint16_t* C_dev,
                          void* stream) {
    if (!A_dev || !B_dev || !C_dev || rows <= 0 || cols <= 0 || N <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (N % 8 != 0 || cols % 8 != 0) return SPATHA_ERR_BAD_SHAPE;
    hipError_t e = spatha::launch_dense_gemm(A_dev, B_dev, rows, cols, N, C_dev, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_transpose_f16(const uint16_t* in_dev, int rows, int cols, uint16_t* out_dev, void* stream) {
    if (!in_dev || !out_dev || rows <= 0 || cols <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (((uintptr_t)in_dev | (uintptr_t)out_dev) & 15u) return SPATHA_ERR_BAD_ARGUMENT;
    if ((rows + 63) / 64 > 65535) return SPATHA_ERR_TOO_LARGE;
    hipError_t e = spatha::launch_transpose_f16(in_dev, rows, cols, out_dev, rows, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_transpose_padded_f16(const uint16_t* in_dev, int rows, int cols, uint16_t* out_dev, void* stream) {
    if (!in_dev || !out_dev || rows <= 0 || cols <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (((uintptr_t)in_dev | (uintptr_t)out_dev) & 15u) return SPATHA_ERR_BAD_ARGUMENT;
    if ((rows + 63) / 64 > 65535) return SPATHA_ERR_TOO_LARGE;
    hipError_t e = spatha::launch_transpose_f16(in_dev, rows, cols, out_dev, (rows + 7) / 8 * 8, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_pad_columns_f16(const uint16_t* in_dev, int rows, int cols, uint16_t* out_dev, void* stream) {
    if (!in_dev || !out_dev || rows <= 0 || cols <= 0 || cols > INT32_MAX - 8) return SPATHA_ERR_BAD_ARGUMENT;
    if (((uintptr_t)in_dev & 1u) || ((uintptr_t)out_dev & 15u)) return SPATHA_ERR_BAD_ARGUMENT;
    hipError_t e = spatha::launch_pad_columns_f16(in_dev, rows, cols, out_dev, (cols + 7) / 8 * 8, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_cut_columns_f16(const uint16_t* in_dev, int rows, int cols, uint16_t* out_dev, void* stream) {
    if (!in_dev || !out_dev || rows <= 0 || cols <= 0 || cols > INT32_MAX - 8) return SPATHA_ERR_BAD_ARGUMENT;
    if (((uintptr_t)in_dev & 15u) || ((uintptr_t)out_dev & 1u)) return SPATHA_ERR_BAD_ARGUMENT;
    hipError_t e = spatha::launch_cut_columns_f16(in_dev, rows, cols, (cols + 7) / 8 * 8, out_dev, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

namespace {
int norm_status(uintptr_t pointers, const void* gamma_dev, const void* beta_dev, int tokens, int hidden) {
    if (!gamma_dev || !beta_dev || tokens <= 0 || hidden <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (hidden % 8 != 0) return SPATHA_ERR_BAD_SHAPE;           // 16-byte pieces
    if (hidden > 4096) return SPATHA_ERR_UNSUPPORTED;           // a lane keeps hidden / 64 values in registers
    return ((pointers | (uintptr_t)gamma_dev | (uintptr_t)beta_dev) & 15u) ? SPATHA_ERR_BAD_ARGUMENT : SPATHA_OK;
}
}  // namespace

int spatha_add_layernorm_f16(const uint16_t* x_dev, const uint16_t* residual_dev, const uint16_t* gamma_dev,
                             const uint16_t* beta_dev, float eps, int tokens, int hidden, uint16_t* out_dev, void* stream) {
    if (!x_dev || !out_dev) return SPATHA_ERR_BAD_ARGUMENT;
    const int st = norm_status((uintptr_t)x_dev | (uintptr_t)residual_dev | (uintptr_t)out_dev, gamma_dev, beta_dev, tokens, hidden);
    if (st) return st;
    hipError_t e = spatha::launch_add_layernorm_f16(x_dev, residual_dev, gamma_dev, beta_dev, eps, tokens, hidden, out_dev, nullptr,
                                                    (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_add_layernorm_f16_t(const uint16_t* x_dev, const uint16_t* residual_dev, const uint16_t* gamma_dev,
                               const uint16_t* beta_dev, float eps, int tokens, int hidden, uint16_t* out_dev, uint16_t* out_t_dev,
                               void* stream) {
    if (tokens > 0 && tokens % 8 != 0) return SPATHA_ERR_BAD_SHAPE;       // (spatha_add_layernorm_f16_tp pads)
    return spatha_add_layernorm_f16_tp(x_dev, residual_dev, gamma_dev, beta_dev, eps, tokens, hidden, out_dev, out_t_dev, stream);
}

int spatha_add_layernorm_f16_tp(const uint16_t* x_dev, const uint16_t* residual_dev, const uint16_t* gamma_dev,
                                const uint16_t* beta_dev, float eps, int tokens, int hidden, uint16_t* out_dev, uint16_t* out_t_dev,
                                void* stream) {
    if (!x_dev || !out_dev || !out_t_dev || tokens > INT32_MAX - 64) return SPATHA_ERR_BAD_ARGUMENT;
    const int st = norm_status((uintptr_t)x_dev | (uintptr_t)residual_dev | (uintptr_t)out_dev | (uintptr_t)out_t_dev, gamma_dev, beta_dev,
                               tokens, hidden);
    if (st) return st;
    hipError_t e = spatha::launch_add_layernorm_f16(x_dev, residual_dev, gamma_dev, beta_dev, eps, tokens, hidden, out_dev, out_t_dev,
                                                    (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

static int embed_layernorm(const int64_t* ids_dev, const int64_t* types_dev, int64_t types_stride, int64_t types_row,
                           const int64_t* positions_dev, int batch, int seq, const uint16_t* word_dev, int64_t words,
                           const uint16_t* type_dev, int64_t types, const uint16_t* position_dev, int64_t positions,
                           const uint16_t* gamma_dev, const uint16_t* beta_dev, float eps, int hidden, uint16_t* out_dev,
                           uint16_t* out_t_dev, void* stream) {
    if (!ids_dev || !types_dev || !positions_dev || !word_dev || !type_dev || !position_dev || !out_dev || batch <= 0 || seq <= 0 ||
        words <= 0 || types <= 0 || positions <= 0 || (types_stride != 0 && types_stride < seq))
        return SPATHA_ERR_BAD_ARGUMENT;
    if ((int64_t)batch * seq > INT32_MAX - 64) return SPATHA_ERR_TOO_LARGE;
    if (((uintptr_t)ids_dev | (uintptr_t)types_dev | (uintptr_t)positions_dev) & 7u) return SPATHA_ERR_BAD_ARGUMENT;
    const int st = norm_status((uintptr_t)word_dev | (uintptr_t)type_dev | (uintptr_t)position_dev | (uintptr_t)out_dev | (uintptr_t)out_t_dev,
                               gamma_dev, beta_dev, batch * seq, hidden);
    if (st) return st;
    spatha::EmbeddingTables tables;
    tables.word = word_dev; tables.type = type_dev; tables.position = position_dev;
    tables.words = words; tables.types = types; tables.positions = positions; tables.hidden = hidden;
    hipError_t e = spatha::launch_embed_layernorm_f16(tables, ids_dev, types_dev, types_stride, types_row, positions_dev, batch, seq,
                                                      gamma_dev, beta_dev, eps, out_dev, out_t_dev, (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

int spatha_embed_layernorm_f16(const int64_t* ids_dev, const int64_t* types_dev, int64_t types_stride, const int64_t* positions_dev, int batch,
                               int seq, const uint16_t* word_dev, int64_t words, const uint16_t* type_dev, int64_t types,
                               const uint16_t* position_dev, int64_t positions, const uint16_t* gamma_dev, const uint16_t* beta_dev, float eps,
                               int hidden, uint16_t* out_dev, uint16_t* out_t_dev, void* stream) {
    return embed_layernorm(ids_dev, types_dev, types_stride, 0, positions_dev, batch, seq, word_dev, words, type_dev, types, position_dev,
                           positions, gamma_dev, beta_dev, eps, hidden, out_dev, out_t_dev, stream);
}

int spatha_embed_layernorm_own_types_f16(const int64_t* ids_dev, const int64_t* types_row_dev, int64_t types_row, const int64_t* positions_dev,
                                         int batch, int seq, const uint16_t* word_dev, int64_t words, const uint16_t* type_dev,
                                         int64_t types, const uint16_t* position_dev, int64_t positions, const uint16_t* gamma_dev,
                                         const uint16_t* beta_dev, float eps, int hidden, uint16_t* out_dev, uint16_t* out_t_dev,
                                         void* stream) {
    if (types_row <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    return embed_layernorm(ids_dev, types_row_dev, 0, types_row, positions_dev, batch, seq, word_dev, words, type_dev, types, position_dev,
                           positions, gamma_dev, beta_dev, eps, hidden, out_dev, out_t_dev, stream);
}

int spatha_attention_f16(const uint16_t* q_dev, const uint16_t* k_dev, const uint16_t* v_dev, int64_t pitch, int batch, int seq, int heads,
                         int head_dim, float scale, uint16_t* out_t_dev, int64_t out_pitch, void* stream) {
    if (!q_dev || !k_dev || !v_dev || !out_t_dev || batch <= 0 || seq <= 0 || heads <= 0) return SPATHA_ERR_BAD_ARGUMENT;
    if (!(scale > 0.f) || scale > 1e30f) return SPATHA_ERR_BAD_ARGUMENT;
    if (head_dim != 64) return SPATHA_ERR_UNSUPPORTED;
    if ((int64_t)batch * heads > INT32_MAX / 2 || (int64_t)batch * seq > INT32_MAX / 2 || seq > (1 << 20) || heads > (1 << 20))
        return SPATHA_ERR_TOO_LARGE;
    if (pitch % 8 != 0 || pitch < (int64_t)heads * head_dim || out_pitch < (int64_t)batch * seq) return SPATHA_ERR_BAD_SHAPE;
    if ((((uintptr_t)q_dev | (uintptr_t)k_dev | (uintptr_t)v_dev) & 15u) || ((uintptr_t)out_t_dev & 1u)) return SPATHA_ERR_BAD_ARGUMENT;
    const hipError_t e = spatha::launch_attention_f16(q_dev, k_dev, v_dev, pitch, batch, seq, heads, scale, out_t_dev, out_pitch,
                                                      (hipStream_t)stream);
    return e == hipSuccess ? SPATHA_OK : hip_fail(e);
}

}  // extern "C"
