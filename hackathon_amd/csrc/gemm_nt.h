// Internal interface of the large-tile NT GEMM (gemm_nt.hip), used by the C-ABI entry points
// of gemm.hip and by the fused layers. Not part of the public C-ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// True when the NT kernel takes this problem: K % 64 == 0, lda and ldb multiples of 8
// elements, A and B 16-B aligned.
bool ql_gemm_nt_fits(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, const void* B,
                     int64_t ldb);

// Split count that fills 256 CUs for this shape (1 = no split-K). `accumulate`: for beta != 0,
// which only the 256-row tile takes.
int ql_gemm_nt_auto_splits(int64_t M, int64_t N, int64_t K, bool accumulate = false);

// fp32 elements of workspace ql_gemm_nt needs with `splits` splits (0 when splits <= 1).
int64_t ql_gemm_nt_workspace_floats(int64_t M, int64_t N, int splits);

// C = alpha * A @ B^T (+ beta C) (+ bias); ws must hold ql_gemm_nt_workspace_floats floats
// (16-B aligned) when splits > 1.
int ql_gemm_nt(int in_dtype, int c_dtype, int64_t M, int64_t N, int64_t K, const void* A,
               int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc, const void* bias,
               float alpha, float beta, int splits, float* ws, hipStream_t s);

// C = alpha * (A @ B^T + A2 @ B2^T) (+ beta C) (+ bias): a second k-contiguous segment with
// K2 % 64 == 0 columns (A2 [M, K2], B2 [N, K2], same alignment rules; K2 = 0: none). With
// `residual` (16-bit C only, beta 0; [M, N] in C's type, 16-B aligned rows, ld % 8 == 0) the
// rounded result plus the residual, rounded again.
int ql_gemm_nt2(int in_dtype, int c_dtype, int64_t M, int64_t N, int64_t K, const void* A,
                int64_t lda, const void* B, int64_t ldb, const void* A2, int64_t lda2,
                const void* B2, int64_t ldb2, int64_t K2, void* C, int64_t ldc, const void* bias,
                float alpha, float beta, int splits, float* ws, hipStream_t s,
                const void* residual = nullptr, int64_t ld_residual = 0);

// The 4-bit linear for at most kSkinnyMaxRows rows of A (gemm_nf4_skinny.hip): qlora_gemm_nf4's
// arguments, checked by it (K % 64 == 0, blocksize a power of two >= 64 dividing K, K2 0 or 64,
// A 16-B aligned rows; log2 of the block sizes). No workspace.
constexpr int64_t kSkinnyMaxRows = 32;
int ql_gemm_nf4_skinny(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
                       const uint8_t* packed, const void* absmax, int nested, const float* code2,
                       const float* absmax2, float offset, int log2_bs, int log2_bs2,
                       const float* nf4_table, int64_t K2, const void* A2, int64_t lda2,
                       const void* B2, int64_t ldb2, int in_dtype, void* C, int64_t ldc,
                       const void* bias, float alpha, hipStream_t s);

// Output tiles of the NT GEMM's kernels: k256 is gemm_nt.hip's (256 x 256 or 256 x 224), the
// others gemm_mid.hip's.
enum class QlGemmTile { k256, k128x128, k64x128, k128x256 };

// One launch of the smaller tiles: ql_gemm_nt2's operands (beta 0; row strides below
// kMidMaxLd; K2 <= 128), K in `splits` ranges of k_per_split (a multiple of 64; every range
// non-empty); with splits > 1 the raw fp32 partials go to ws [splits][M][N].
constexpr int64_t kMidMaxLd = int64_t(1) << 22;
int ql_gemm_mid(QlGemmTile tile, int in_dtype, int c_dtype, int64_t M, int64_t N, int64_t K,
                const void* A, int64_t lda, const void* B, int64_t ldb, const void* A2,
                int64_t lda2, const void* B2, int64_t ldb2, int64_t K2, void* C, int64_t ldc,
                const void* bias, float alpha, int64_t k_per_split, int splits, float* ws,
                hipStream_t s, const void* residual, int64_t ld_residual);
