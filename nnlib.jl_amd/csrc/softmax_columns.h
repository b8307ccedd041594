// The operations of the softmax family and the launcher of its kernels for contiguous columns (softmax.hip).
#pragma once
#include "common.h"

enum { OP_SOFTMAX = 0, OP_LOGSOFTMAX = 1, OP_LOGSUMEXP = 2, OP_GRAD_SOFTMAX = 3, OP_GRAD_LOGSOFTMAX = 4 };

// term / sum for results that are rounded to 16 bits, inv = 1 / sum: a product and its remainder's correction, which is the
// quotient's own rounding in all but the rarest cases at a third of a division's instructions.  (The product alone errs by up
// to 2^-23; where memory bounds the kernel, over strided dimensions, the correction costs nothing measurable.)
__device__ static inline float quotient(float term, float sum, float inv) {
    const float q = term * inv;
    return fmaf(fmaf(-sum, q, term), inv, q);
}

template <typename T> struct ColumnIO {
    typedef typename T::type t;
    __device__ static u32x4_t load(const t *p) {
        if constexpr (sizeof(t) == 4) return *(const mi_piece4_t *)p;
        else return *(const mi_piece2_t *)p;
    }
    __device__ static void store(t *p, const u32x4_t &v) {
        if constexpr (sizeof(t) == 4) *(mi_piece4_t *)p = v;
        else *(mi_piece2_t *)p = v;
    }
};

// y[:, c] from x[:, c] (gradients: x = dy, x2 = the forward result) for `cols` columns of `len` >= 1 contiguous elements
// of a Float32 or 16-bit type; logsumexp writes one value per column.  y may be x or x2.
void launch_softmax_columns(int32_t dtype, int op, const void *x, const void *x2, void *y, int64_t len, int64_t cols, hipStream_t st);
