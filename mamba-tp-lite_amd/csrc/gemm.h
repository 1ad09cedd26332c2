// The fp32 GEMM on split f16 operands (gemm.hip), for the library's own callers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mtl {

struct SplitGemm {
    const float* x; const float* w;        // [M, ldx], [N, ldw]
    int64_t ldx, ldw;
    const float* bias;                     // [N] or null
    float* y0; float* y1;                  // columns [0, n_split) to y0, the others to y1 (null: all to y0)
    int64_t ldy0, ldy1, n_split;           // n_split a multiple of 32
    int64_t M, N, K;
    void* xbuf; void* wbuf;                // the split operands, split_bytes() each, 16-byte aligned
};

// bytes of a split [rows, K] matrix
int64_t split_bytes(int64_t rows, int64_t K);
// splits X [M, K] into xbuf and W [N, K] into wbuf (either may be null) in one launch
int split_rows(const float* x, int64_t ldx, int64_t M, const float* w, int64_t ldw, int64_t N, int64_t K, void* xbuf,
               void* wbuf, hipStream_t st);
// x_out = x + y (y, x_out null: none), normed = w rmsnorm(x_out) [M, K] and its
// split into xbuf, and the split of W [N, K] into wbuf, in one launch
int norm_split(const float* x, const float* y, float* x_out, const float* w, float eps, float* normed, int64_t M,
               int64_t K, const float* wmat, int64_t ldw, int64_t N, void* xbuf, void* wbuf, hipStream_t st);
// whether norm_split takes this width and these (possibly null) pointers
bool norm_split_ok(const float* x, const float* y, const float* w, const float* normed, int64_t K);
// where the split product is faster than the library's fp32 GEMM, the splits of x and W included
bool split_pays(int64_t M, int64_t N, int64_t K);
// the product of split operands; the sizes are the caller's to check (as mtl_linear_f32 does)
int gemm_split(const SplitGemm& g, hipStream_t st);

}  // namespace mtl
