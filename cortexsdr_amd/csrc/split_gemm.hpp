// split_gemm.hpp — fp32-accurate products on the fp16 matrix cores (split_gemm.hip), for the
// decoder's batched prefill.
#pragma once

#include "hsdb_impl.hpp"

namespace csdr {

// Rows of fp32 values as two fp16 planes: value = (hi + 2^-12 lo) * inv[row], ld values per row
// (zeros past the row's end). inv < 0 marks a row holding a NaN or an infinity.
struct SplitPlanes {
    _Float16* hi = nullptr;
    _Float16* lo = nullptr;
    float* inv = nullptr;
    int ld = 0;
};

constexpr int kSplitMats = 3;          // matrices of one grouped product
constexpr int kSplitMaxCols = 16384;   // a decoded row stays in registers, a token row in LDS
inline int split_ld(int cols) { return (cols + 63) / 64 * 64; }

// 1-row tiles of 64 and at most kSplitMaxCols columns.
bool split_eligible(const csdr_hsdb* s);

// Planes of the decoded matrices (csdr_hsdb_decompress's values), one launch.
int split_decode(int n, const csdr_hsdb* const* segs, const SplitPlanes* out, hipStream_t st);

// Planes of M token rows of n values: x itself, its RMSNorm (weight w), or silu(x) * x2. With
// `parts` (n_parts planes of M x n), x += their sum first (in order; x is updated).
enum class SplitOp { plain, rms_norm, silu_mul };
int split_rows(SplitOp op, float* x, const float* x2_or_w, const float* parts, int n_parts, int M,
               int n, float eps, const SplitPlanes& out, hipStream_t st);

// ys[i] (M x R[i]) = X . W_i^T (+ bias[i]). With splits > 1 the contraction is cut into that many
// parts and part z is written to ys[i] + z * M * R[i] (no bias).
int split_gemm(int n, const SplitPlanes* w, const int* R, const SplitPlanes& x, int M,
               float* const* ys, const float* const* bias, int splits, hipStream_t st);
int split_count(int R, int K, int M);  // parts that fill the chip

}  // namespace csdr
