// Entry points of the library that only the host module (host.cpp) calls: products whose shapes
// the C ABI's functions refuse or whose workspace they have no argument for.  The conventions
// are the ABI's (fx_abi.h); return codes and messages too.
#pragma once

#include <stdint.h>

namespace fx {

// dX (M, N) = dY (M, K) W (K, N), times G (the GELU derivative, row stride N) when given, on the
// small tiles: any M, N and K multiples of 8, W and dX contiguous, 16-byte aligned buffers.
// Few tiles of a long K are cut into K slices whose fp32 partials go through `work`.
int64_t input_grad_workspace(int64_t M, int64_t N, int64_t K, bool gated);
int input_grad(const uint16_t* dY, int64_t ldy, const uint16_t* W, const uint16_t* G, uint16_t* dX, float* work, int64_t M,
               int64_t N, int64_t K, void* stream);

// out (cols) = bf16(column sums of g (rows, cols), row stride cols), fp32 sums in a fixed order;
// cols a multiple of 8, g, work and out 16-byte aligned
int64_t column_sums_workspace(int64_t rows, int64_t cols);
int column_sums(const uint16_t* g, int64_t rows, int64_t cols, float* work, uint16_t* out, void* stream);

// A decode step's small ends, one launch each.
// tok_out[0..n) = tok, *pos_out = pos, lens[0..n) = pos + 1
int decode_inputs(const int64_t* tok, int64_t n, int64_t pos, int64_t* tok_out, int64_t* pos_out, int32_t* lens, void* stream);
// x (n, D) = bf16(E[tok[i]] + P[*pos]), E (V, D) and P (T, D) contiguous, D a multiple of 8; a row of
// NaN for an id or a position outside its table
int decode_embed(const int64_t* tok, const int64_t* pos, const uint16_t* E, int64_t V, const uint16_t* P, int64_t T, uint16_t* x,
                 int64_t n, int64_t D, void* stream);
// out (M, N) fp32 = the bf16 values of norm(X) W^T (fx_linear_fwd_ex with the norm, M <= 64), X rows
// ldx apart
int few_rows_logits(const uint16_t* X, int64_t ldx, const uint16_t* W, const uint16_t* norm_w, float eps, float* out, int64_t M,
                    int64_t N, int64_t K, void* stream);

}  // namespace fx
