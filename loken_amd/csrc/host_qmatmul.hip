// Host mirror of loken's QKernelMatMul for the card path: see include/loken_host.hpp.

#include "../../include/loken_host.hpp"
#include "lk_common.h"
#include "mmq_problem.h"
#include "rows16.h"
#include "stream_scratch.h"

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <type_traits>

namespace loken {
namespace {

constexpr int Q81_BLOCK = 36;
constexpr size_t MMQ_RECORD = 144;                      // bytes per 128 padded values per row

size_t pad_to(size_t v, size_t m) { return (v + m - 1) / m * m; }

// The 32-value nibble formats and the two-bit K-quants: served by the plain mat-vec (four of them by the
// tiled matmul as well, and Q2_K / Q3_K, from the row counts of nibble_tiles_pay below).
bool matvec_only(int dtype) {
    return dtype == LK_TYPE_Q4_0 || dtype == LK_TYPE_Q4_1 || dtype == LK_TYPE_Q5_0 || dtype == LK_TYPE_Q5_1 ||
           dtype == LK_TYPE_IQ4_NL || dtype == LK_TYPE_MXFP4 || dtype == LK_TYPE_Q2_K || dtype == LK_TYPE_Q3_K ||
           dtype == LK_TYPE_IQ4_XS;
}

bool nibble_tiles(int dtype) {
    return dtype == LK_TYPE_Q4_0 || dtype == LK_TYPE_Q4_1 || dtype == LK_TYPE_Q5_0 || dtype == LK_TYPE_Q5_1 || dtype == LK_TYPE_Q3_K ||
           dtype == LK_TYPE_Q2_K;
}

bool tiled_serves(int dtype, int k) {
    return (dtype == LK_TYPE_Q4_K || dtype == LK_TYPE_Q5_K || dtype == LK_TYPE_Q6_K || dtype == LK_TYPE_Q8_0 || nibble_tiles(dtype)) &&
           k % 256 == 0;
}

// One or two rows quantized in the mat-vec launch, against the quantizer's launch and the mat-vec's: every workgroup quantizes the
// rows, which a matrix that keeps the chip busy longer than the second launch costs pays for several times over. One launch / two
// (us; one figure on the right: all formats alike):
//   two rows         Q4_K          Q5_K          Q6_K          Q8_0
//   1024 x 4096      6.8 / 9.7
//   4096 x 4096      7.0 / 9.8                   8.3 / 9.8     7.9 / 9.8
//   8192 x 4096      7.9 / 10.0    10.2 / 10.0   11.2 / 10.0   11.1 / 10.0
//   14336 x 4096     9.6 / 10.4                                15.2 / 13.3
//   14336 x 2048                   10.6 / 9.9    11.9 / 10.5   9.5 / 9.7
//   1024 x 6144      7.8 / 9.8     8.3 / 9.8     9.6 / 9.8     7.7 / 9.8
//   2048 x 8192      8.2 / 9.7     8.8 / 9.7     10.2 / 9.7    10.6 / 9.7
//   4096 x 8192      11.5 / 10.0   12.6 / 10.0   13.8 / 10.0   13.3 / 10.0
//   12288 x 6144     17.4 / 12.8   19.4 / 14.9   22.0 / 17.4   20.2 / 16.1
//   one row          (up to 14336 x 4096 6.8 to 11.1 / 9.6 to 12.8)
//   4096 x 8192      8.4 / 9.9     8.8 / 9.9     10.0 / 10.0   10.0 / 10.0
//   12288 x 6144     12.5 / 11.7   14.3 / 13.3   16.2 / 14.3   14.4 / 15.3
//   28672 x 8192     25.8 / 26.3   30.9 / 31.5   38.5 / 37.6   45.9 / 46.0
bool pays_in_one_launch(int dtype, int n, int k, int rows) {
    const long long weights = (long long)n * k;
    if (rows == 1) return k <= 4096 || dtype == LK_TYPE_Q8_0 || weights <= (40ll << 20) || (dtype != LK_TYPE_Q6_K && weights >= (128ll << 20));
    if (k <= 4096) return dtype == LK_TYPE_Q4_K || weights <= (dtype == LK_TYPE_Q8_0 ? 28ll << 20 : 24ll << 20);
    return weights <= (dtype == LK_TYPE_Q4_K || dtype == LK_TYPE_Q5_K ? 16ll << 20 : 12ll << 20);
}

// Nine to sixteen rows of Q8_0 and Q4_0 on the f16 tiles, operands straight from the rows, against what served them else: the
// quantizer and two mat-vec launches, for Q4_0 from 16 rows or 48 M weights the int8 tiles. Those / f16 tiles (us):
//                         9 rows        12 rows       16 rows
//   Q8_0  14336 x 4096    32 / 30                     39 / 30
//         4096 x 14336    45 / 36                     65 / 36
//         64000 x 2048    72 / 55                     93 / 55
//         11003 x 3072    24 / 26       26 / 26       29 / 26
//         4096 x 4096     17.5 / 19     18.7 / 19     21 / 19
//         2048 x 2048     15.5 / 15.8   15.8 / 17.0   16.0 / 15.8
//   Q4_0  512 x 14336     30 / 24       38 / 25
//         11003 x 3072    26 / 22       30 / 22
//         4096 x 4096     17.5 / 17.7   18.6 / 17.0
//         1024 x 4096     17.4 / 16.4   16.5 / 16.5
bool few_rows_to_tiles(int dtype, int n, int k, int rows, const void* blob) {
    if (rows <= 8 || rows > 16 || n < 512 || k % 256 != 0 || ((uintptr_t)blob & 1) != 0) return false;
    const long long weights = (long long)n * k;
    if (dtype == LK_TYPE_Q8_0) return weights >= (48ll << 20) || (rows >= 12 && (weights >= (32ll << 20) || k >= 8192)) || (rows >= 14 && k >= 4096);
    return dtype == LK_TYPE_Q4_0;
}

// Q4_0 / Q4_1 / Q5_0 / Q5_1, Q3_K and Q2_K above eight rows: one tiled launch (with K cut into ranges
// where its tiles are few, mmq_problem.h) against mat-vec launches of eight rows each. Measured on MI355X,
// quantizer included, mat-vec against tiled (int8): Q4_0 4096 x 4096 at 9 / 16 / 32 rows 29 / 35 / 55 us against
// 31 / 27 / 29; 14336 x 4096 at 9 / 16 rows 42 / 58 against 37 / 38; 4096 x 14336 at 9 rows 57 against 41;
// 1024 x 4096 at 9 / 16 rows 27 / 31 against 33 / 26. Q5_1, Q3_K and Q2_K alike (Q3_K 4096 x 4096 at 9 / 16
// rows 31 / 40 against 29 / 27). So: from 16 rows, and from 9 on a matrix of 48 M weights or more.
bool nibble_tiles_pay(int dtype, int n, int k, int rows) {
    if (!nibble_tiles(dtype) || k % 256 != 0) return false;
    return rows >= 16 || (long long)n * k >= (48ll << 20);
}

// The buffer of a tiled call's partial products. A graph keeps its own and all graphs together are bounded, so a recorded call takes
// the larger size only where its plan uses it; a plan that fits the smaller one is the same in both.
struct Fixup {
    void* ptr;
    int64_t bytes;
};
Fixup fixup_of(LkScratch& scratch, int dtype, int n, int k, int rows) {
    if (!scratch.recording() || lk_mmq_tiles_parts(dtype, k, n, rows) > MMQ_FIXUP_BYTES)
        if (void* large = scratch.get(LK_SCRATCH_FIXUP, MMQ_HOST_FIXUP_BYTES)) return {large, MMQ_HOST_FIXUP_BYTES};
    return {scratch.get(LK_SCRATCH_FIXUP, MMQ_FIXUP_BYTES), MMQ_FIXUP_BYTES};
}

size_t elem_bytes(int type) { return type == LK_TYPE_F32 ? 4 : 2; }

}  // namespace

int matvec_rows(int dtype, int k) {
    if ((dtype == LK_TYPE_Q4_K || dtype == LK_TYPE_Q5_K || dtype == LK_TYPE_Q6_K) && k % 256 == 0) return 8;
    // Q8_0: mat-vec launches of eight rows up to 16 rows, but for few_rows_to_tiles
    return dtype == LK_TYPE_Q8_0 && tiled_serves(dtype, k) ? 16 : 8;
}

// Rows the matrix-unit rows kernels take before the tiled matmul does. A rows kernel reads the weights straight from HBM, once for
// every 16 or 32 activation rows; its time steps up once its workgroups (`items` above 32 rows, n / 16 up to 16) are more than the
// CUs. The f16 tiles cut K and read the weights once per 32 to 128 rows. Whole calls of forward on MI355X, rows kernel / f16 tiles
// (us; Q5_K like Q4_K; above sixteen rows with the 32-row tiles, before the sets below):
//                          9             16            24            32            64            128
//   Q4_K  512 x 4096       5.7 / 12.2    5.7 / 12.9    14.9 / 13.0   16.0 / 13.2   16.0 / 13.9   16.6 / 15.7
//         4096 x 4096      7.2 / 14.0    7.6 / 14.6    15.3 / 15.1   16.4 / 15.5   16.7 / 19.3   25.6 / 23.3
//         8192 x 4096      9.5 / 17.5    9.8 / 18.0    16.0 / 19.4   17.2 / 20.4   26.0 / 23.0   40.2 / 29.8
//         14336 x 4096     16.6 / 20.8   17.6 / 21.2   22.7 / 21.6   25.1 / 22.2   40.6 / 29.0   66.3 / 39.9
//         2048 x 5120      7.6 / 13.6    7.7 / 14.3    17.3 / 14.8   18.3 / 15.1   18.6 / 18.1   19.4 / 21.4
//         8192 x 8192      15.0 / 22.5   15.1 / 22.8   26.3 / 23.3   28.6 / 23.9   44.9 / 29.6   69.2 / 43.0
//         14336 x 8192     29.5 / 28.6   35.5 / 29.7   37.1 / 30.1   41.8 / 30.9   68.5 / 41.4   118 / 67.4
//         4096 x 14336     15.9 / 23.6   17.7 / 23.9   39.9 / 24.7   43.1 / 25.1   43.9 / 29.1   70.4 / 40.9
//   Q6_K  1024 x 2048      4.8 / 14.1    4.7 / 14.2    6.5 / 14.5    6.6 / 14.4    7.4 / 14.7    14.1 / 15.7
//         4096 x 4096      10.7 / 17.1   11.0 / 17.5   16.1 / 17.9   15.8 / 18.3   19.1 / 22.3   29.4 / 26.3
//         8192 x 4096      16.2 / 22.7   17.0 / 22.8   19.0 / 23.5   20.2 / 23.9   29.9 / 25.5   46.3 / 36.5
//         2048 x 5120      8.9 / 16.4    9.1 / 17.1    11.3 / 17.5   11.3 / 17.7   18.4 / 20.4   21.9 / 24.0
//         14336 x 5120     30.8 / 32.6   32.1 / 33.4   35.0 / 33.8   37.2 / 34.4   57.2 / 41.4   98.0 / 61.1
//         1024 x 8192      11.6 / 19.1   11.7 / 19.6   11.9 / 20.1   12.2 / 20.3   14.8 / 21.2   28.9 / 24.5
//         8192 x 8192      27.0 / 29.8   28.0 / 30.3   29.9 / 31.0   32.3 / 31.4   51.4 / 37.6   82.5 / 54.8
//         4096 x 14336     21.4 / 34.0   22.0 / 34.1   35.8 / 34.5   36.7 / 35.2   48.5 / 34.8   82.2 / 52.1
// Once the tiles were dealt evenly to the XCDs they took over (rows kernel / tiles):
//   Q6_K, 17 to 32 rows, more than 2048 matrix rows of more than 4352 values, or past 20 M weights where the 16-row tiles have no
//     granules: 4708 x 5376 at 26 26.7 / 21.0; 2165 x 7424 at 21 21.1 / 19.0; 6412 x 3584 at 29 23.3 / 19.8
//     (4145 x 4096 at 21 16.7 / 18.6; 2977 x 4352 at 31 16.5 / 18.1; 9054 x 1792 at 19 16.6 / 17.2; 1833 x 11264 at 24 18.3 / 22.8)
//     The 32-row tiles stay up to 40 M where a row is less than ten super-blocks, twelve or sixteen (14483 x 1792 at 18 16.9 / 20.4; 11261 x 3072 at 25 21.7 / 23.5;
//     ten from 9216 matrix rows on: 13147 x 2560 at 20 20.5 / 22.0, 8239 x 2560 at 27 20.4 / 21.2), and of rows of up to 24 where they are one round and the 16-row tiles
//     three or more to two CUs (6881 x 4608 at 30 19.7 / 22.6; 8073 x 4352 at 17 20.3 / 22.3; 5325 x 4608 at 24, 16-row tiles, 25.0 / 19.4)
//   Q6_K, 33 to 64 rows of fewer than 3072 values, past 320000 results: 9987 x 1536 at 36 23.9 / 18.5 (6621 x 1536 at 46 16.2 / 17.3); not where
//     they are two rounds at most of 2048 values or fewer (7315 x 1024 at 60 11.6 / 16.2; 6829 x 1536 at 52 16.0 / 17.4; 5062 x 2304 at 64 21.9 / 18.2)
//   Q4_K and Q5_K, rows of 3328 to 4096 values, 17 to 32 over fewer than 4096 matrix rows, and more where there are at most 128 items:
//     2077 x 3584 at 26 14.6 / 13.2; 962 x 3840 at 27 14.6 / 13.2; 627 x 4096 at 71 17.0 / 14.4; 1184 x 3584 at 58 14.8 / 13.4
//     (5246 x 3840 at 28 15.6 / 16.0; 1462 x 3584 at 124 15.6 / 17.6)
// Left where they were: Q6_K, 65 rows and more over fewer than 1024 matrix rows of 2560 to 5632 values (548 x 3584 at 154 23.0 / 17.4); 17 to 32 over
// 4097 to 6144 of 6144 (4642 x 6144 at 18 21.2 / 22.9).
//
// 17 to 128 rows as sets of sixteen in the short launches (rows16_short.hip, rows16_q6k_short.hip) moved lines the other way, quantizer and
// rows kernel / tiles:
//   Q4_K and Q5_K, where 1.1 times what the launch and its quantizer take (5.3 us and 0.81 of the launch in a graph, fitted to 1460 shapes) is under what the tiles
//     take (fitted too, 9 %), 1.2 times past 22 us and at 512 values, where both fits are at their ends (7930 x 11264 at 64 48.5 / 36.4, 6102 x 512 at 125 10.1 / 9.1): 2986 x 6144 at 26 11.3 / 18.3; 2665 x 6144 at 36 11.5 / 19.4; 805 x 3840 at 60 9.1 / 13.9; 1256 x 5120 at 70 10.7 /
//     17.3; 932 x 4096 at 127 10.2 / 16.2; 4060 x 14336 at 46 31.1 / 27.8; Q5_K 3456 x 5632 at 19 12.1 / 18.4, 1344 x 6144 at 44 11.2 / 17.8
//   Q6_K, where the launch takes the call: 3840 x 6656 at 26 15.2 / 21.7; 1664 x 7168 at 36 15.3 / 21.1, at 58 15.8 / 22.4; 1344 x 4096 at 95 12.9 /
//     20.2
// Left where they were, though rows would be faster there too (890 x 8192 at 55 rows 11.0 / 17.3): fewer than 1152 matrix rows of long rows, and at 17 to 32 rows
// of Q6_K past 12288 values those that are no multiple of 2048.
static bool sets_of_rows_pay(int dtype, int n, int k, int rows, const void* blob) {
    if (rows < 17 || rows > 128 || n < 512 || k % 256 != 0 || ((uintptr_t)blob & 15) != 0) return false;   // (off a 16-byte boundary: the 32-row tiles)
    if (dtype != LK_TYPE_Q4_K && dtype != LK_TYPE_Q5_K && dtype != LK_TYPE_Q6_K) return false;
    if (dtype == LK_TYPE_Q6_K) {
        if (!lk_rows16_q6k_short_pays(rows, n, k)) return false;
        const int tiles = (n + 15) / 16, cus = lk_device().cus;
        if (rows <= 32) return tiles <= cus && (k <= 12288 || k % 2048 == 0);
        if (rows <= 64) return 2 * tiles <= cus && (n >= 1152 || k <= 6144);
        return n >= 1152 || k <= 5632;
    }
    if (n < 1152 && k >= 4608) return false;
    const float launch = lk_rows16_short_us(rows, n, k / 256, dtype == LK_TYPE_Q5_K), weights = 1e-6f * (float)n * (float)k;
    const float rows_us = 5.3f + 0.81f * launch;
    return launch >= 0.f && (rows_us > 22.f || k <= 512 ? 1.2f : 1.1f) * rows_us < 10.2f + 0.00063f * (float)k + weights * (0.026f + 0.0041f * (float)rows);
}

static bool rows_kernel_serves(int dtype, int n, int k, int rows) {
    if (dtype != LK_TYPE_Q4_K && dtype != LK_TYPE_Q5_K && dtype != LK_TYPE_Q6_K) return false;
    if (rows <= 8) return true;
    const long long results = (long long)n * rows, weights = (long long)n * k;
    // few matrix rows yield few tiles whatever the cut, and under 512 they are the int8 ones
    if (n < 512) return rows <= 16 || results * (k > 4096 ? k : 4096) <= 450000ll * 4096 * (n > 0 ? 2048 / n : 2048);
    const long long items = (n + 31ll) / 32 * ((rows + 31) / 32);
    if (dtype == LK_TYPE_Q6_K) {
        if (rows <= 16) return k % 2048 == 0 || k < 4608 || n <= 12288;
        if (rows <= 32) {
            if (n <= 2048 || (k > 4096 && k <= 6144 && n > 6144 && items <= 256)) return true;
            return k <= 4352 && weights <= (k % 2048 == 0 || k < 2560 || k == 3072 || (k == 2560 && n >= 9216) ? 40ll << 20 : 20ll << 20);
        }
        if (rows <= 64) return n <= 1024 || (k < 3072 ? results <= 320000 || (k <= 2048 && items <= 512) : k <= 6144 && weights <= (17ll << 20));
        if (k < 5632 && n < 1024 && rows > 128 && items <= 256) return true;
        return (k < 3072 || (n < 1024 && k < 4608)) && results <= 450000;
    }
    if (rows <= 16) return k < 7168 || n <= 8192;
    if (k >= 3328 && rows > 32) return k < 5632 && items > 128 && items <= 256;
    if (k >= 4608) return false;
    if (rows <= 32) return (n < 12288 || k < 4096 || rows < 20) && (k < 3328 || k > 4096 || n >= 4096);
    return items <= 256 || (k <= 2048 && results <= 450000);
}

// The K-quants at 3 to 8 rows: the 16-row tiles of the matrix-unit kernels, whose time hardly moves with the row count, against
// mat-vec launches, whose dot work grows with every row. Up to 4096 values a row the rows kernel takes the rows themselves, one
// launch where the mat-vec kernels need the quantizer's too. Rows kernel / mat-vec (us):
//                          3 rows        5 rows        8 rows
//   Q4_K  256 x 256        3.6 / 7.4     3.7 / 9.3     3.7 / 12.2
//         2000 x 1024      3.6 / 7.4     3.6 / 9.3     3.6 / 12.2
//         256 x 2048       4.1 / 6.6     4.1 / 8.1     4.1 / 10.0
//         8192 x 4096      7.6 / 9.9     7.8 / 11.6    7.9 / 14.1
//   Q6_K  1024 x 1024      4.0 / 7.9     4.0 / 9.7     4.0 / 12.6
//         1024 x 4096      7.2 / 6.6     7.2 / 7.6     7.3 / 9.1
//         4096 x 4096      8.4 / 8.9     8.3 / 10.3    8.5 / 12.1
//         8192 x 4096      - / 11.7      13.7 / 13.6   13.9 / 16.9
// (fewer than 256 matrix rows have not been moved: 64 x 1024 3.6 / 7.0, 3.7 / 9.0, 3.6 / 12.0; Q6_K 200 x 4096 7.0 / 6.5, 7.0 / 7.4, 7.1 / 8.8).
// Longer rows, by way of the quantizer on both sides:
//   Q4_K and Q5_K  2048 x 8192 at 8 rows 9.8 / 10.8; 4096 x 8192 at 4 / 5 / 8 10.2 / 10.7, 10.5 / 11.7, 10.0 / 14.1; 8192 x 4096 at 4 / 5
//                  10.8 / 10.8, 10.1 / 11.6; 1024 x 14336 at 6 / 8 12.0 / 13.3, 12.2 / 15.5; 4096 x 14336 at 3 / 8 13.5 / 13.8, 14.1 / 24.0;
//                  of 2048 values more than 16384 matrix rows from 3 (151936 x 2048)
//   Q6_K           512 x 4096 at 8 9.8 / 10.0; 700 x 5120 at 8 10.0 / 12.2; 4096 x 8192 at 5 / 6 12.9 / 13.1, 12.9 / 13.8; 6144 x 2048 at 5 / 6
//                  10.0 / 10.6, 9.9 / 11.5; 1024 x 14336 at 5 / 8 14.6 / 13.8, 14.7 / 22.1; 4096 x 14336 at 3 / 4 16.8 / 16.6, 16.8 / 18.8
static bool small_rows_kernel_pays(int dtype, int n, int k, int rows) {
    if (rows < 3 || rows > 8 || k % 256 != 0 || (dtype != LK_TYPE_Q4_K && dtype != LK_TYPE_Q5_K && dtype != LK_TYPE_Q6_K)) return false;
    const long long weights = (long long)n * k;
    if (k <= 4096 && n >= 256 && n <= (dtype == LK_TYPE_Q6_K ? 6144 : 16384)) return true;
    if (dtype == LK_TYPE_Q6_K)
        return (rows >= 7 && n >= 512) || (rows >= 5 && weights * rows >= (76ll << 20)) || (k % 2048 == 0 && weights >= (48ll << 20));
    return k <= 2048 ? (long long)n * rows >= 8192 : weights * rows > (128ll << 20);
}

// Matrices whose 3 to 8 rows are refused as rows quantized beforehand, as they have been since the 16-row tiles took them over; the
// smaller ones of small_rows_kernel_pays are served from Q8_1 rows too.
static bool large_for_few_rows(int dtype, int n, int k, int rows) {
    if (dtype == LK_TYPE_Q6_K) return k % 2048 == 0 && ((long long)n * k >= (48ll << 20) || (rows >= 7 && n >= 1024));
    return (long long)n * rows >= (k <= 2048 ? 8192 : 57344);
}

// The K-quants' weights as the rows kernels take them.
static bool fits_rows_kernel(int dtype, int k, const void* blob) {
    return k % 256 == 0 && ((uintptr_t)blob & (dtype == LK_TYPE_Q6_K ? 1 : 15)) == 0;
}

// Three to eight rows go to the rows kernels by the lines of the 16-row tiles, which take weights from a 16-byte boundary on. Q6_K
// weights off it (a matrix that starts at some row of another one) would get the 32-row tiles. Those / mat-vec: 2048 x 3840 at 3 / 8
// rows 13.6 / 7.1, 14.0 / 10.2; 4096 x 8448 at 5 / 8 24.8 / 18.4, 25.3 / 23.6; 256 x 1280 at 3 / 8 7.9 / 7.4, 8.1 / 11.4.
static bool few_rows_to_kernel(int dtype, int n, int k, int rows, const void* blob) {
    return ((uintptr_t)blob & 15) == 0 && small_rows_kernel_pays(dtype, n, k, rows);
}

QKernelMatMul::QKernelMatMul(int dtype, int n, int k, const void* blob, int device)
    : dtype_(dtype), n_(n), k_(k), device_(device), blob_(blob) {}

int QKernelMatMul::forward(const void* x, int x_type, int rows, void* out, void* stream_ptr, bool decode_order) {
    last_path_ = Path::None;
    hipStream_t stream = (hipStream_t)stream_ptr;
    const bool plain = matvec_only(dtype_);
    if (!plain && dtype_ != LK_TYPE_Q4_K && dtype_ != LK_TYPE_Q5_K && dtype_ != LK_TYPE_Q6_K && dtype_ != LK_TYPE_Q8_0) return LK_ERR_TYPE;
    if (x_type != LK_TYPE_F32 && x_type != LK_TYPE_F16 && x_type != LK_TYPE_BF16) return LK_ERR_TYPE;
    if (rows == 0) return LK_OK;
    if (!x || !out || !blob_ || rows < 0 || n_ <= 0 || k_ <= 0) return LK_ERR_ARG;
    const int block_len = dtype_ == LK_TYPE_Q8_0 || (plain && dtype_ != LK_TYPE_Q2_K && dtype_ != LK_TYPE_Q3_K && dtype_ != LK_TYPE_IQ4_XS) ? 32 : 256;
    if (k_ % block_len != 0) return LK_ERR_ARG;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess || current != device_) {
        (void)hipGetLastError();
        return LK_ERR_ARG;   // "input on a different device" (kernel_matmul.rs:1499-1503)
    }
    const int mv_max = matvec_rows(dtype_, k_);
    // a quantize -> consume pair holds the stream's scratch, so that two host threads sharing the stream cannot
    // interleave their pairs (fast_mmvq.rs:15-32, kernel_matmul/mmq.rs:43-86)

    // --- mat-vec family: up to matvec_rows, or any count when every row must sum like a one-row call
    const bool rows_kernel_fits = fits_rows_kernel(dtype_, k_, blob_);
    const bool to_rows_kernel = few_rows_to_kernel(dtype_, n_, k_, rows, blob_);
    const bool few_to_tiles = few_rows_to_tiles(dtype_, n_, k_, rows, blob_);
    const bool to_nibble_tiles = !decode_order && (few_to_tiles || nibble_tiles_pay(dtype_, n_, k_, rows)) &&
                                 ((uintptr_t)blob_ & (dtype_ == LK_TYPE_Q2_K ? 3 : 1)) == 0;
    auto matvec = [&]() -> int {
        // One or two rows quantized in the mat-vec launch itself
        auto in_one_launch = [&]() -> int {
            last_path_ = Path::MatVecFused;
            if (x_type != LK_TYPE_F32) return lk_mmvq_half_rows(dtype_, blob_, x, x_type, out, rows, n_, k_, stream);
            const void* vx[1] = {blob_};
            void* dst[1] = {out};
            const int nn[1] = {n_};
            return lk_mmvq_fused(dtype_, 1, vx, (const float*)x, k_, dst, x_type, k_, nn, rows, n_, nullptr, stream);
        };
        const bool can_fuse = !plain && rows <= 2 && k_ <= 8192 && k_ % 4 == 0 && ((uintptr_t)x & (x_type == LK_TYPE_F32 ? 15 : 7)) == 0;
        if (can_fuse && pays_in_one_launch(dtype_, n_, k_, rows)) return in_one_launch();
        const int k_padded = (int)pad_to((size_t)k_, 512), blocks = k_padded / 32;
        LkScratch scratch(stream);
        uint8_t* act = (uint8_t*)scratch.get(LK_SCRATCH_LINEAR, (size_t)rows * blocks * Q81_BLOCK);
        if (!act) return can_fuse ? in_one_launch() : LK_ERR_NOMEM;   // (the same bits)
        if (int rc = lk_quantize_q8_1(x, x_type, act, k_, k_padded, rows, stream)) return rc;
        for (int r0 = 0; r0 < rows; r0 += 8) {
            const int b = rows - r0 < 8 ? rows - r0 : 8;
            const int rc = lk_mmvq(dtype_, blob_, act + (size_t)r0 * blocks * Q81_BLOCK,
                                   (uint8_t*)out + (size_t)r0 * n_ * elem_bytes(x_type), x_type, k_, n_, b, blocks, n_,
                                   nullptr, decode_order ? 1 : 0, stream);
            if (rc) return rc;
        }
        last_path_ = Path::MatVec;
        return LK_OK;
    };
    if ((rows <= mv_max && !to_rows_kernel && !few_to_tiles) || decode_order || (plain && !to_nibble_tiles)) return matvec();

    // --- a handful of rows (or a matrix too small to fill the chip with tiles): matrix unit, weights
    //     straight from HBM
    if ((rows_kernel_serves(dtype_, n_, k_, rows) || sets_of_rows_pay(dtype_, n_, k_, rows, blob_)) && rows_kernel_fits) {
        const int blocks = k_ / 32;
        int rc = lk_rows_linear_direct(dtype_, blob_, x, out, x_type, rows, n_, k_, stream);
        if (rc < 0) {
            LkScratch scratch(stream);
            void* act = scratch.get(LK_SCRATCH_LINEAR, (size_t)rows * blocks * Q81_BLOCK);
            // (rows too long for the kernels' scale tables in LDS launch nothing, and the call goes on to the
            // mat-vec or the tiled matmul below; so does one without memory for the quantized rows, a recorded one above all
            // of which only larger calls ran before, on the tiles, which work in other buffers)
            rc = LK_ERR_ARG;
            if (act) {
                if (int r = lk_quantize_q8_1(x, x_type, act, k_, k_, rows, stream)) return r;
                rc = lk_rows_linear(dtype_, blob_, act, blocks, out, x_type, rows, n_, k_, stream);
            }
        }
        if (rc == LK_OK) {
            last_path_ = Path::RowsOnMatrixUnit;
            return LK_OK;
        }
        if (rc != LK_ERR_ARG) return rc;
        if (rows <= mv_max) return matvec();   // a few rows the rows kernel declined: not worth a tile
    }

    // --- tiled matmul (mmq_forward, kernel_matmul/mmq.rs:21-159)
    if (!tiled_serves(dtype_, k_)) return LK_ERR_TYPE;
    const size_t k_padded = pad_to(pad_to((size_t)k_, 512), 128);
    const size_t ws_bytes = (size_t)rows * (k_padded / 128) * MMQ_RECORD + 128 * MMQ_RECORD;
    LkScratch scratch(stream);
    const Fixup fixup = fixup_of(scratch, dtype_, n_, k_, rows);
    if (!fixup.ptr) return LK_ERR_NOMEM;
    // The f16 tiles' operands straight from x where the product takes those tiles (Q6_K 4096 x 14336 at 2048 rows 527 ->
    // 502 us, Q4_K 14336 x 4096 at 512 rows 100 -> 96 against records in between); without memory for them, by way of the records.
    const int width = lk_mmq_tiles_linear(dtype_, fixup.ptr, fixup.bytes, blob_, x, x_type, out, k_, n_, rows, stream);
    if (width == 0) return LK_ERR_ARG;
    if (width > 0) {
        last_path_ = Path::Tiled;
        return LK_OK;
    }
    void* act = scratch.get(LK_SCRATCH_LINEAR, ws_bytes);
    if (!act) return LK_ERR_NOMEM;
    // the layouts of the reference's table (quantized/mmq.rs:274-285)
    auto quantizer = dtype_ == LK_TYPE_Q2_K ? launch_mmq_quantize_q8_1_D2S6
                     : dtype_ == LK_TYPE_Q6_K || dtype_ == LK_TYPE_Q8_0 || dtype_ == LK_TYPE_Q5_0 || dtype_ == LK_TYPE_Q3_K
                         ? launch_mmq_quantize_q8_1_D4
                         : launch_mmq_quantize_q8_1_DS4;
    quantizer(x, nullptr, act, x_type, k_, k_, 0, 0, (int64_t)k_padded, rows, 1, 1, stream);
    if (lk_mmq_linear(dtype_, fixup.ptr, blob_, act, out, x_type, k_, n_, rows, k_ / block_len, stream) == 0)
        return LK_ERR_ARG;   // "no tile fits, nothing ran": the reference falls back to dequantized
    last_path_ = Path::Tiled;
    return LK_OK;
}

// takes_matvec of the reference (kernel_matmul.rs:1069-1075), for rows quantized beforehand: mat-vec counts of rows, but for the
// K-quants' 3 to 8 rows over a large matrix (large_for_few_rows) and the formats with tiles from nibble_tiles_pay's row counts. Which
// launch serves the call is forward's choice all the same (forward_quantized). Three products over one activation, forward three
// times / quantized once (us): Q4_K 4096 x 4096 at 4 / 8 rows 18.9 / 17.1, 18.8 / 17.2; Q6_K 2048 x 3072 at 8 17.3 / 15.8; Q8_0 4096 x 8192
// at 16 81 / 83, 14336 x 4096 at 9 105 / 107.
bool QKernelMatMul::takes_quantized(int rows, bool decode_order) const {
    if (!blob_ || rows < 1) return false;
    if (decode_order && rows > 1) return true;
    if (matvec_only(dtype_)) return !nibble_tiles_pay(dtype_, n_, k_, rows) || rows <= matvec_rows(dtype_, k_);
    if (rows > matvec_rows(dtype_, k_)) return false;
    return !(fits_rows_kernel(dtype_, k_, blob_) && small_rows_kernel_pays(dtype_, n_, k_, rows) && large_for_few_rows(dtype_, n_, k_, rows));
}

size_t QKernelMatMul::quantized_bytes(int k, int rows) {
    return k > 0 && rows > 0 ? (size_t)rows * (pad_to((size_t)k, 512) / 32) * Q81_BLOCK : 0;
}

int QKernelMatMul::quantize_for_matvec(const void* x, int x_type, int rows, void* q81, void* stream, QuantizedActivation* a,
                                       bool decode_order) const {
    if (!x || !q81 || !a || rows <= 0) return LK_ERR_ARG;
    if (x_type != LK_TYPE_F32 && x_type != LK_TYPE_F16 && x_type != LK_TYPE_BF16) return LK_ERR_TYPE;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess || current != device_) {
        (void)hipGetLastError();
        return LK_ERR_ARG;
    }
    if (!takes_quantized(rows, decode_order)) return LK_NOT_TAKEN;
    const int k_padded = (int)pad_to((size_t)k_, 512);
    if (int rc = lk_quantize_q8_1(x, x_type, q81, k_, k_padded, rows, stream)) return rc;
    a->q81 = q81;
    a->k = k_;
    a->rows = rows;
    a->device = device_;
    a->x_type = x_type;
    return LK_OK;
}

int QKernelMatMul::forward_quantized(const QuantizedActivation& a, void* out, void* stream, bool decode_order) {
    last_path_ = Path::None;
    if (!a.q81 || !out) return LK_ERR_ARG;
    if (a.k != k_ || a.device != device_ || !takes_quantized(a.rows, decode_order)) return LK_NOT_TAKEN;
    if (a.x_type != LK_TYPE_F32 && a.x_type != LK_TYPE_F16 && a.x_type != LK_TYPE_BF16) return LK_ERR_TYPE;   // (as every mat-vec launch)
    if (((uintptr_t)a.q81 & 3) != 0) return LK_ERR_ARG;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess || current != device_) {
        (void)hipGetLastError();
        return LK_ERR_ARG;
    }
    const int blocks = (int)pad_to((size_t)k_, 512) / 32;
    // The launches forward takes at this row count, with its bits; where they decline, or the tiles have no scratch, the mat-vec launches
    const bool one_order = decode_order && a.rows > 1;
    if (!one_order && few_rows_to_kernel(dtype_, n_, k_, a.rows, blob_)) {
        const int rc = lk_rows_linear(dtype_, blob_, a.q81, blocks, out, a.x_type, a.rows, n_, k_, (hipStream_t)stream);
        if (rc == LK_OK) last_path_ = Path::RowsOnMatrixUnit;
        if (rc != LK_ERR_ARG) return rc;
    }
    if (!one_order && few_rows_to_tiles(dtype_, n_, k_, a.rows, blob_)) {
        LkScratch scratch((hipStream_t)stream);
        const Fixup fixup = fixup_of(scratch, dtype_, n_, k_, a.rows);
        const int width = fixup.ptr ? lk_mmq_tiles_linear_q8_1(dtype_, fixup.ptr, fixup.bytes, blob_, a.q81, blocks, a.x_type, out, k_, n_, a.rows, (hipStream_t)stream) : -1;
        if (width == 0) return LK_ERR_ARG;
        if (width > 0) {
            last_path_ = Path::Tiled;
            return LK_OK;
        }
    }
    for (int r0 = 0; r0 < a.rows; r0 += 8) {
        const int b = a.rows - r0 < 8 ? a.rows - r0 : 8;
        const int rc = lk_mmvq(dtype_, blob_, (const uint8_t*)a.q81 + (size_t)r0 * blocks * Q81_BLOCK,
                               (uint8_t*)out + (size_t)r0 * n_ * elem_bytes(a.x_type), a.x_type, k_, n_, b, blocks, n_,
                               nullptr, decode_order ? 1 : 0, stream);
        if (rc) return rc;
    }
    last_path_ = Path::MatVec;
    return LK_OK;
}

int QKernelMatMul::forward_quantized_pair(QKernelMatMul& other, const QuantizedActivation& a, void* out0, void* out1,
                                          void* stream) {
    last_path_ = other.last_path_ = Path::None;
    if (!a.q81 || !out0 || !out1) return LK_ERR_ARG;
    if (a.k != k_ || other.k_ != k_ || a.rows != 1 || a.x_type != LK_TYPE_F32 || dtype_ != other.dtype_ ||
        device_ != other.device_ || a.device != device_ || !takes_quantized(1, false) || !other.takes_quantized(1, false))
        return LK_NOT_TAKEN;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess || current != device_) {
        (void)hipGetLastError();
        return LK_ERR_ARG;
    }
    const void* vx[2] = {blob_, other.blob_};
    void* dst[2] = {out0, out1};
    const int nn[2] = {n_, other.n_};
    const int blocks = (int)pad_to((size_t)k_, 512) / 32;
    const int rc = lk_mmvq_multi(dtype_, 2, vx, a.q81, dst, LK_TYPE_F32, k_, nn, 1, blocks, n_ > other.n_ ? n_ : other.n_, nullptr,
                                 stream);
    if (rc == LK_ERR_TYPE) return LK_NOT_TAKEN;   // a format without the several-matrices launch
    if (rc) return rc;
    last_path_ = other.last_path_ = Path::MatVec;
    return LK_OK;
}

void release_workspaces() { lk_stream_scratch_release(-1, LK_SCRATCH_OF_LINEARS); }

}  // namespace loken

extern "C" void* lkh_qkernel_matmul_new(int dtype, int n, int k, const void* blob, int device) {
    return new loken::QKernelMatMul(dtype, n, k, blob, device);
}
extern "C" void lkh_qkernel_matmul_free(void* handle) { delete (loken::QKernelMatMul*)handle; }
extern "C" int lkh_qkernel_matmul_forward(void* handle, const void* x, int x_type, int rows, void* out, void* stream,
                                          int decode_order) {
    if (!handle) return LK_ERR_ARG;
    return ((loken::QKernelMatMul*)handle)->forward(x, x_type, rows, out, stream, decode_order != 0);
}
extern "C" int lkh_qkernel_matmul_last_path(void* handle) {
    return handle ? (int)((loken::QKernelMatMul*)handle)->last_path() : 0;
}
extern "C" size_t lkh_quantized_activation_bytes(int k, int rows) { return loken::QKernelMatMul::quantized_bytes(k, rows); }
extern "C" int lkh_qkernel_matmul_quantize_for_matvec(void* handle, const void* x, int x_type, int rows, void* q81, void* stream,
                                                      int decode_order) {
    if (!handle) return LK_ERR_ARG;
    loken::QKernelMatMul::QuantizedActivation a;
    return ((loken::QKernelMatMul*)handle)->quantize_for_matvec(x, x_type, rows, q81, stream, &a, decode_order != 0);
}
namespace {
loken::QKernelMatMul::QuantizedActivation activation_of(const loken::QKernelMatMul& m, const void* q81, int x_type, int rows) {
    loken::QKernelMatMul::QuantizedActivation a;
    a.q81 = q81;
    a.k = m.k();
    a.rows = rows;
    a.x_type = x_type;
    (void)hipGetDevice(&a.device);   // the rows were quantized on the current card
    return a;
}
}  // namespace
extern "C" int lkh_qkernel_matmul_forward_quantized(void* handle, const void* q81, int x_type, int rows, void* out, void* stream,
                                                    int decode_order) {
    if (!handle) return LK_ERR_ARG;
    if (x_type != LK_TYPE_F32 && x_type != LK_TYPE_F16 && x_type != LK_TYPE_BF16) return LK_ERR_TYPE;
    auto* m = (loken::QKernelMatMul*)handle;
    return m->forward_quantized(activation_of(*m, q81, x_type, rows), out, stream, decode_order != 0);
}
extern "C" int lkh_qkernel_matmul_forward_quantized_pair(void* handle, void* other, const void* q81, void* out0, void* out1,
                                                         void* stream) {
    if (!handle || !other) return LK_ERR_ARG;
    auto* m = (loken::QKernelMatMul*)handle;
    return m->forward_quantized_pair(*(loken::QKernelMatMul*)other, activation_of(*m, q81, LK_TYPE_F32, 1), out0, out1, stream);
}
extern "C" int lkh_matvec_rows(int dtype, int k) { return loken::matvec_rows(dtype, k); }
extern "C" void lkh_release_workspaces(void) { loken::release_workspaces(); }
