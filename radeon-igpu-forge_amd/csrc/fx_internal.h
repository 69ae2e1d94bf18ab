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

}  // namespace fx
