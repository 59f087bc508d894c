// Host mirror of loken's QKernelMatMul for the card path: see include/loken_host.hpp.

#include "../../include/loken_host.hpp"
#include "lk_common.h"
#include "mmq_problem.h"
#include "stream_scratch.h"

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <type_traits>

namespace loken {
namespace {

constexpr int Q81_BLOCK = 36;
constexpr size_t MMQ_RECORD = 144;                      // bytes per 128 padded values per row
constexpr size_t FIXUP_BYTES = 256u * 128u * 128u * 4u;  // kernel_matmul/mmq.rs:42

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

// One or two rows in one launch, against the quantizer's launch and the mat-vec's (us): every workgroup quantizes the rows, which a matrix that keeps
// the chip busy longer than the second launch costs pays for several times over. Two rows: 1024 x 4096 6.8 / 9.7, 4096 x 4096 Q4_K, Q6_K, Q8_0 7.0, 8.3, 7.9 / 9.8; 8192 x 4096 Q4_K,
// Q5_K, Q6_K, Q8_0 7.9, 10.2, 11.2, 11.1 / 10.0, 14336 x 4096 Q4_K, Q8_0 9.6, 15.2 / 10.4, 13.3, 14336 x 2048 Q5_K, Q6_K, Q8_0 10.6, 11.9, 9.5 / 9.9, 10.5, 9.7; 1024 x 6144 7.8, 8.3, 9.6, 7.7 / 9.8, 2048 x 8192 8.2, 8.8, 10.2, 10.6 / 9.7,
// 4096 x 8192 11.5, 12.6, 13.8, 13.3 / 10.0, 12288 x 6144 17.4, 19.4, 22.0, 20.2 / 12.8, 14.9, 17.4, 16.1. One row: up to 14336 x 4096 6.8 to
// 11.1 / 9.6 to 12.8, 4096 x 8192 8.4, 8.8, 10.0, 10.0 / 9.9, 9.9, 10.0, 10.0, 12288 x 6144 12.5, 14.3, 16.2, 14.4 / 11.7, 13.3, 14.3, 15.3,
// 28672 x 8192 25.8, 30.9, 38.5, 45.9 / 26.3, 31.5, 37.6, 46.0.
bool pays_in_one_launch(int dtype, int n, int k, int rows) {
    const long long weights = (long long)n * k;
    if (rows == 1) return k <= 4096 || dtype == LK_TYPE_Q8_0 || weights <= (40ll << 20) || (dtype != LK_TYPE_Q6_K && weights >= (128ll << 20));
    if (k <= 4096) return dtype == LK_TYPE_Q4_K || weights <= (dtype == LK_TYPE_Q8_0 ? 28ll << 20 : 24ll << 20);
    return weights <= (dtype == LK_TYPE_Q4_K || dtype == LK_TYPE_Q5_K ? 16ll << 20 : 12ll << 20);
}

// Nine to sixteen rows of Q8_0 and Q4_0 on the f16 tiles, operands straight from the rows, against the quantizer and two mat-vec
// launches (Q4_0 from 16 rows or 48 M weights: int8 tiles). us, before / tiles: Q8_0 14336 x 4096 at 9 / 16 rows 32 / 39 against 30 / 30,
// 4096 x 14336 45 / 65 against 36 / 36, 64000 x 2048 72 / 93 against 55 / 55, 11003 x 3072 at 9 / 12 / 16 24 / 26 / 29 against 26 / 26 / 26, 4096 x 4096 17.5 / 18.7 /
// 21 against 19 / 19 / 19, 2048 x 2048 15.5 / 15.8 / 16.0 against 15.8 / 17.0 / 15.8; Q4_0 512 x 14336 at 9 / 12 30 / 38 against 24 / 25, 11003 x 3072 26 / 30 against 22 / 22,
// 1024 x 4096 17.4 / 16.5 against 16.4 / 16.5, 4096 x 4096 17.5 / 18.6 against 17.7 / 17.0.
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

size_t elem_bytes(int type) { return type == LK_TYPE_F32 ? 4 : 2; }

}  // namespace

int matvec_rows(int dtype, int k) {
    if ((dtype == LK_TYPE_Q4_K || dtype == LK_TYPE_Q5_K || dtype == LK_TYPE_Q6_K) && k % 256 == 0) return 8;
    // Q8_0: mat-vec launches of eight rows up to 16 rows, but for few_rows_to_tiles
    return dtype == LK_TYPE_Q8_0 && tiled_serves(dtype, k) ? 16 : 8;
}

// Rows the matrix-unit rows kernels take before the tiled matmul does. A rows kernel reads the weights straight from HBM, once
// for every 16 or 32 activation rows; its time steps up once its workgroups are more than the CUs. The f16 tiles cut K and read the weights
// once per 32 to 128 rows. Measured on MI355X, quantizer included, rows kernel against f16 tiles (us), for matrices of 512 rows or more:
//   Q4_K, 9 to 16 rows: 512 x 8192 10..11 / 16, 2048 x 8192 9..10 / 17..18, 8192 x 8192 14 / 22, 4096 x 14336 15..16 / 23, 10000 x 5120 18 / 21, 12000 x 10240 35..42 / 29; Q5_K alike
//     17 to 32: 700 x 5120 18 / 15, 10000 x 5120 25 / 22, 2048 x 6144 21 / 16, 14336 x 4096 at 24 22 / 21; 4096 x 4096 16 / 16, 8192 x 4096 16 / 19
//     above: 1024 x 4608 at 33 18 / 14, 1100 x 8192 at 33 / 64 26 / 18, 26 / 19; 3000 x 5120 at 33 / 96 20 / 18, 27 / 24; 4096 x 4096 at 64 / 96 (256, 384 workgroups) 17 / 20, 25 / 25; 1024 x 4096 at 200 / 400
//     (224, 416) 19 / 21, 28 / 25; 2048 x 2048 at 200 17 / 19. Q5_K alike.
//   Q6_K, 9 to 16 rows: 2048 x 8192 13 / 20, 6144 x 6144 20 / 24, 4096 x 14336 20 / 30, 3000 x 5120 12 / 18, 10000 x 5120 26 / 26
//     17 to 32: 2048 x 14336 20 / 25, 8192 x 4096 17..19 / 23, 6144 x 6144 22..23 / 24..25, 700 x 11008 13 / 22; 10000 x 5120 30..33 / 27, 4096 x 14336 35 / 31,
//     4096 x 8192 25 / 22
//     33 to 64: 512 x 14336 17..18 / 26, 1024 x 14336 20..21 / 26, 2048 x 6144 19..20 / 20..22, 4096 x 4096 18..19 / 20..22; 2048 x 14336 34..36 / 27..29, 8192 x
//     4096 26..29 / 25, 6144 x 3072 22 / 20..22. Above: 4096 x 4096 at 96 28 / 26, 1024 x 6144 23 / 22
// `bench.py --workload rows-sweep` prints the table for a shape.
static bool rows_kernel_serves(int dtype, int n, int k, int rows) {
    if (dtype != LK_TYPE_Q4_K && dtype != LK_TYPE_Q5_K && dtype != LK_TYPE_Q6_K) return false;
    if (rows <= 8) return true;
    const long long results = (long long)n * rows, weights = (long long)n * k;
    // (few matrix rows yield few tiles whatever the cut: the int8 tiles' line)
    if (n < 512) return rows <= 16 || results * (k > 4096 ? k : 4096) <= 450000ll * 4096 * (n > 0 ? 2048 / n : 2048);
    const long long items = (n + 31ll) / 32 * ((rows + 31) / 32);
    if (dtype == LK_TYPE_Q6_K) {
        if (rows <= 16) return k % 2048 == 0 || k < 4608 || n <= 12288;
        if (rows <= 32) return weights <= (24ll << 20) || n <= 2048 || (k <= 6144 && weights <= (40ll << 20));
        if (rows <= 64) return n <= 1024 || (k < 3072 ? results <= 450000 : k <= 6144 && weights <= (17ll << 20));
        if (k < 5632 && n < 1024 && rows > 128 && items <= 256) return true;
        return (k < 3072 || (n < 1024 && k < 4608)) && results <= 450000;
    }
    if (rows <= 16) return k < 7168 || n <= 8192;
    if (k >= 4608) return k < 5632 && items > 128 && items <= 256 && rows > 32;
    if (rows <= 32) return n < 12288 || k < 4096 || rows < 20;
    return items <= 256 || (k <= 2048 && results <= 450000);
}

// The K-quants at 3 to 8 f32 rows: the 16-row tiles of the matrix-unit kernels (their time hardly moves
// with the row count) against mat-vec launches (whose dot work grows with every row). Up to 4096 values a row the rows kernel takes the rows
// themselves, one launch where the mat-vec kernels need the quantizer's too, rows kernel / mat-vec at 3, 5, 8 rows: Q4_K 256 x 256 3.6, 3.7, 3.7 / 7.4, 9.3, 12.2; 2000 x
// 1024 3.6 / 7.4, 9.3, 12.2; 256 x 2048 4.1 / 6.6, 8.1, 10.0; 8192 x 4096 7.6, 7.8, 7.9 / 9.9, 11.6, 14.1; Q6_K 1024 x 1024 4.0 / 7.9, 9.7, 12.6; 4096 x 4096 8.4, 8.3, 8.5 /
// 8.9, 10.3, 12.1 (fewer than 256 matrix rows have not been moved: 64 x 1024 3.6 / 7.0, 9.0, 12.0, Q6_K 200 x 4096 7.0 / 6.5, 7.4, 8.8). Longer rows: measured on MI355X, mat-vec against rows kernel, quantizer included (us): Q4_K / Q5_K 4096 x 8192 at 4 / 5 / 8 rows 10.7, 11.7, 14.1 / 10.2,
// 10.5, 10.0, 4096 x 14336 at 3 / 8 13.8, 24.0 / 13.5, 14.1, 8192 x 4096 at 4 / 5 10.8, 11.6 / 10.8, 10.1, 1024 x 14336 at 6 / 8 13.3, 15.5 / 12.0, 12.2; 2048 x 8192 at 8 10.8 / 9.8;
// k = 2048: 2048 rows from 4, 6144 and 151936 from 3. Q6_K 4096 x 8192 at 5 / 6 13.1, 13.8 / 12.9, 12.9, 6144 x 2048 at 5 / 6 10.6, 11.5 / 10.0, 9.9, 1024 x 14336 at
// 5 / 8 13.8, 22.1 / 14.6, 14.7, 700 x 5120 at 8 12.2 / 10.0, 512 x 4096 at 8 10.0 / 9.8, 4096 x 14336 at 3 / 4 16.6, 18.8 / 16.8, 16.8.
static bool small_rows_kernel_pays(int dtype, int n, int k, int rows) {
    if (rows < 3 || rows > 8 || k % 256 != 0 || (dtype != LK_TYPE_Q4_K && dtype != LK_TYPE_Q5_K && dtype != LK_TYPE_Q6_K)) return false;
    const long long weights = (long long)n * k;
    if (k <= 4096 && n >= 256 && n <= (dtype == LK_TYPE_Q6_K ? 6144 : 16384)) return true;
    if (dtype == LK_TYPE_Q6_K)
        return (rows >= 7 && n >= 512) || (rows >= 5 && weights * rows >= (76ll << 20)) || (k % 2048 == 0 && weights >= (48ll << 20));
    return k <= 2048 ? (long long)n * rows >= 8192 : weights * rows > (128ll << 20);
}

// Matrices whose 3 to 8 rows are refused as rows quantized beforehand, as they have been since the 16-row tiles took them over; the
// smaller ones small_rows_kernel_pays names are served from Q8_1 rows too.
static bool large_for_few_rows(int dtype, int n, int k, int rows) {
    if (dtype == LK_TYPE_Q6_K) return k % 2048 == 0 && ((long long)n * k >= (48ll << 20) || (rows >= 7 && n >= 1024));
    return (long long)n * rows >= (k <= 2048 ? 8192 : 57344);
}

// The K-quants' weights as the rows kernels take them.
static bool fits_rows_kernel(int dtype, int k, const void* blob) {
    return k % 256 == 0 && ((uintptr_t)blob & (dtype == LK_TYPE_Q6_K ? 1 : 15)) == 0;
}

// Three to eight rows go to the rows kernels by the lines of the 16-row tiles, which take weights from a 16-byte boundary on. Q6_K weights off it (a
// matrix that starts at some row of another one) would get the 32-row tiles: 3 / 8 rows, those / mat-vec: 2048 x 3840 13.6, 14.0 / 7.1, 10.2; 4096 x 8448
// at 5 / 8 24.8, 25.3 / 18.4, 23.6; 256 x 1280 at 3 / 8 7.9, 8.1 / 7.4, 11.4.
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
        const bool can_fuse = !plain && rows <= 2 && k_ <= 8192 && ((uintptr_t)x & (x_type == LK_TYPE_F32 ? 15 : 7)) == 0 && k_ % 4 == 0;
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
    if (rows_kernel_serves(dtype_, n_, k_, rows) && rows_kernel_fits) {
        const int blocks = k_ / 32;
        int rc = lk_rows_linear_direct(dtype_, blob_, x, out, x_type, rows, n_, k_, stream);
        if (rc < 0) {
            LkScratch scratch(stream);
            void* act = scratch.get(LK_SCRATCH_LINEAR, (size_t)rows * blocks * Q81_BLOCK);
            if (!act) return LK_ERR_NOMEM;
            if (int r = lk_quantize_q8_1(x, x_type, act, k_, k_, rows, stream)) return r;
            // (rows too long for the kernels' scale tables in LDS launch nothing, and the call goes on to the
            // mat-vec or the tiled matmul below)
            rc = lk_rows_linear(dtype_, blob_, act, blocks, out, x_type, rows, n_, k_, stream);
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
    void* fixup = scratch.get(LK_SCRATCH_FIXUP, FIXUP_BYTES);
    if (!fixup) return LK_ERR_NOMEM;
    // The f16 tiles' operands straight from x where the product takes those tiles (Q6_K 4096 x 14336 at 2048 rows 527 ->
    // 502 us, Q4_K 14336 x 4096 at 512 rows 100 -> 96 against records in between); without memory for them, by way of the records.
    const int width = lk_mmq_tiles_linear(dtype_, fixup, blob_, x, x_type, out, k_, n_, rows, stream);
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
    if (lk_mmq_linear(dtype_, fixup, blob_, act, out, x_type, k_, n_, rows, k_ / block_len, stream) == 0)
        return LK_ERR_ARG;   // "no tile fits, nothing ran": the reference falls back to dequantized
    last_path_ = Path::Tiled;
    return LK_OK;
}

// takes_matvec of the reference (kernel_matmul.rs:1069-1075), for rows quantized beforehand: mat-vec counts of rows, but for the K-quants'
// 3 to 8 rows over a large matrix (large_for_few_rows) and the formats with tiles from nibble_tiles_pay's row counts. Which launch serves the call
// is forward's choice all the same (forward_quantized). Three products over one activation, forward three times / quantized once (us): Q4_K 4096 x 4096
// at 4 / 8 rows 18.9, 18.8 / 17.1, 17.2; Q6_K 2048 x 3072 at 8 rows 17.3 / 15.8; Q8_0 4096 x 8192 at 16 81 / 83, 14336 x 4096 at 9 105 / 107.
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
        void* fixup = scratch.get(LK_SCRATCH_FIXUP, FIXUP_BYTES);
        const int width = fixup ? lk_mmq_tiles_linear_q8_1(dtype_, fixup, blob_, a.q81, blocks, a.x_type, out, k_, n_, a.rows, (hipStream_t)stream) : -1;
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
