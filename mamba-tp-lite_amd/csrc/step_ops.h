// The batched step's launches for either storage type (T = float, or uint16_t
// for bf16 activations, weights and conv history with fp32 partial sums, SSM
// state and residual): the fp32 C entry points and the one-call step
// (decode_step.cpp) share them.  Each checks its own sizes and alignments.
#pragma once

#include "common.h"

namespace mtl {

// in_proj + conv step + x_proj partials (linear.hip); sq null: x is already normed
template <typename T>
int in_proj_conv_xproj(const T* x, int64_t x_rs, const T* W_in, const T* b_in, T* conv_state, const T* conv_w,
                       const T* conv_b, int32_t d_conv, const T* W_xT, int32_t J, T* xc, T* z, int64_t z_rs,
                       float* xpart, int64_t batch, int64_t d_model, int64_t d_inner, int32_t channels_per_part,
                       const float* sq, int32_t sq_tiles, float eps, mtl_stream_t stream);

// ksplit partial products of y = x W^T (+ bias in part 0), fp32 (linear.hip)
template <typename T>
int linear_parts(const T* x, int64_t x_rs, const T* W, const T* bias, float* y, int64_t y_rs, int64_t y_ks, int64_t M,
                 int64_t N, int64_t K, int32_t ksplit, int32_t rows_per_block, mtl_stream_t stream);

// the same with the residual add and the next norm's inputs (linear.hip)
template <typename T>
int linear_residual(const T* x, int64_t x_rs, const T* W, const T* bias, float* parts, int64_t M, int64_t N, int64_t K,
                    int32_t ksplit, int32_t rows_per_block, float* h, const T* w_next, T* x_next, float* sq,
                    uint32_t* counters, mtl_stream_t stream);

// the SSM update from fp32 x_dbl, parameters in T (step.hip)
template <typename T>
int state_update(float* ssm_state, const T* x, int64_t x_sb, const T* z, int64_t z_sb, const float* x_dbl,
                 int64_t xdbl_sb, const T* W_dt, const T* b_dt, const T* A_log, const T* Dvec, T* y, int64_t y_sb,
                 int64_t batch, int64_t dim, int64_t dstate, int64_t dt_rank, mtl_stream_t stream);

// x_out = x + the parts (nparts 0: none), normed = w rmsnorm(x_out) in T (step.hip)
template <typename T>
int add_rmsnorm(const float* x, const float* parts, int32_t nparts, float* x_out, const T* w, T* normed, int64_t rows,
                int64_t cols, float eps, mtl_stream_t stream);

}  // namespace mtl
