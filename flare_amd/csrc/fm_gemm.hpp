// Arguments of the fused-epilogue contractions (fm_gemm.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

namespace fm {

enum { EP_KERNEL = 0, EP_STORE = 1, EP_SUMSQ = 2 };

struct EpArgs {
  // EP_KERNEL
  double sig2 = 1, power = 2;
  const double *row_norm = nullptr;  // |B_i| per row (atom) of the block
  const double *alpha = nullptr;     // alpha_j per column (sparse env)
  // Optional k matrix (rows x ldk), FP64.
  void *K = nullptr;
  long long ldk = 0;
  // EP_KERNEL writes w, EP_STORE writes C, into W (rows x ldw). In the int8
  // contraction EP_KERNEL instead writes w as the BF16 pair (hi, lo) of its
  // FP32 value into Wh / Wl (tiled split layout, ldw columns), zero in the
  // padding columns [N, ldw), the operand of the split-BF16 gradient contraction.
  void *W = nullptr;
  void *Wh = nullptr, *Wl = nullptr;
  long long ldw = 0;
  // EP_KERNEL: energy partials [column tile][row]; EP_SUMSQ: [row tile][col]
  // (16 columns, 32 rows of L in the FP64 contraction).
  double *part = nullptr;
  long long part_ld = 0;
  template <typename T>
  __device__ __forceinline__ T *W_as() const {
    return reinterpret_cast<T *>(W);
  }
  template <typename T>
  __device__ __forceinline__ T *K_as() const {
    return reinterpret_cast<T *>(K);
  }
};

// Number of column tiles a kernel contraction of the given form uses (one
// energy partial each), and of the FP64 contraction's variance partials, one per
// 32 rows, whose sum takes the two of each 64 rows together (always even).
int gemm_col_tiles(int form, int N);
int gemm_row_tiles(int M);

// One FP64 contraction C (M x N) = A B^T, rows of A (M x K) and B (N x K)
// contiguous with leading dimensions lda and ldb, any alignment of 8 bytes.
// lower_tri: A is lower triangular (zeros above the diagonal).
struct F64Gemm {
  const double *A = nullptr, *B = nullptr;
  long long lda = 0, ldb = 0;
  int M = 0, N = 0, K = 0, lower_tri = 0;
  EpArgs e;
};
// Several contractions with one epilogue (a model's species) in one launch:
// their workgroups share the chip, where one species at a time would leave it
// part empty on small structures. All triangular or none.
void gemm_f64_groups(hipStream_t st, int ep, const std::vector<F64Gemm> &groups);
void gemm_f64(hipStream_t st, int ep, int M, int N, int K, const double *A, long long lda,
              const double *B, long long ldb, int lower_tri, const EpArgs &e);
// Split-BF16 x3 contraction (EP_STORE: the gradient contraction G = W X_hat
// of the chosen form) on operands stored as two BF16 pieces of FP32
// values, x = x_0 + x_1 with x_0 = bf16(x), x_1 = bf16(x - x_0); it sums
// x_1 y_0 + x_0 y_1 + x_0 y_0 (3 MFMAs per product, about 16 significant
// bits; FP32 accumulation). Tiled split layout of a piece of n rows: blocks of
// kSplitRows rows x kSplitPad k (row, then k: 1 KB), the blocks of a row block
// one after the other along k; zeros in the padding of k, rows past n in the
// last block are never part of a kept result.
constexpr int kSplitPad = 32, kSplitRows = 16;
inline long long split_ld(long long k) { return (k + kSplitPad - 1) / kSplitPad * kSplitPad; }
inline size_t split_elems(long long n, long long k) {
  return (size_t)((n + kSplitRows - 1) / kSplitRows * kSplitRows * split_ld(k));
}
__host__ __device__ inline size_t split_offset(long long row, long long k, long long nk) {
  return (size_t)((row / kSplitRows * nk + k / kSplitPad) * (kSplitRows * kSplitPad) +
                  row % kSplitRows * kSplitPad + k % kSplitPad);
}
struct SplitGemm {
  const uint16_t *A[2] = {nullptr, nullptr}, *B[2] = {nullptr, nullptr};
  int M = 0, N = 0, nk = 0;  // nk steps of kSplitPad
  EpArgs e;                  // W, ldw
};
void gemm_split_groups(hipStream_t st, const std::vector<SplitGemm> &groups);
// The pieces of n FP64 rows of K values.
void split_rows(hipStream_t st, const double *X, long long ldx, int n, int K, uint16_t *hi,
                uint16_t *lo);
// Exact-integer kernel contraction (the chosen form's S = B X_hat^T with the
// EP_KERNEL epilogue, k in FP64 and w as BF16 pairs): both operands as
// kI8Slices int8 slices of their rows with a power-of-two scale per row, in
// the tiled slice layout below. The slices come from slice_rows (or the
// chosen form's descriptor pass).
constexpr int kI8Slices = 5;
constexpr int kI8Pad = 64;     // k step; the reduction length is padded to it with zeros
constexpr int kI8TileA = 128;  // row tile of the descriptor operand
constexpr int kI8TileN = 64;   // column tile (sparse set): the energy partials are per column tile
// Row tiles per group in the integer contraction's XCD tile order: 32
// resident workgroups per XCD then cover 4 row tiles x 8 column tiles
// (2 row tiles by 16 column tiles and 8 by 4 measured within 2 % of it).
constexpr int kI8Group = 4;
inline long long i8_ld(long long k) { return (k + kI8Pad - 1) / kI8Pad * kI8Pad; }
// Tiled slice layout of n rows with reduction length Kq = nk kI8Pad: rows in
// tiles of tr, and tile (row tile rt, k step ks) is kI8Slices consecutive
// blocks of tr x kI8Pad bytes (slice, then row, then k), so one k step of a
// row tile is a single contiguous run of kI8Slices tr kI8Pad bytes. Rows past
// n in the last tile are never read into a kept result.
__host__ __device__ inline long long i8_tile_offset(int tr, long long nk, long long row, int k,
                                                    int p) {
  return (((row / tr) * nk + (k >> 6)) * kI8Slices + p) * (long long)tr * kI8Pad +
         (row % tr) * kI8Pad + (k & (kI8Pad - 1));
}
inline size_t i8_tiled_bytes(long long n, int tr, long long Kq) {
  return (size_t)((n + tr - 1) / tr) * tr * Kq * kI8Slices;
}
// One contraction: rows of A (M, in tiles of kI8TileA) against rows of B (N, in
// tiles of kI8TileN), both starting a tile, over nk steps of kI8Pad.
struct I8Gemm {
  const int8_t *A = nullptr, *B = nullptr;
  const double *sa = nullptr, *sb = nullptr;  // scales per row
  int M = 0, N = 0, nk = 0;
  EpArgs e;
};
void slice_rows(hipStream_t st, const float *X, long long ldx, int n, int nd, int8_t *Q,
                long long Kq, int tr, double *scale);
void slice_rows(hipStream_t st, const double *X, long long ldx, int n, int nd, int8_t *Q,
                long long Kq, int tr, double *scale);
void gemm_i8_groups(hipStream_t st, const std::vector<I8Gemm> &groups);

}  // namespace fm
