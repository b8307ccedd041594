// The softmax family over the first (contiguous) dimension of a column-major (len, cols) matrix: softmax, logsoftmax,
// logsumexp and the two gradients.  Replaces, for dims = 1, NNlib's _softmax! (src/softmax.jl:69-79), _logsoftmax!
// (:137-147), logsumexp (:200-203), _∇softmax! (:107-110) and _∇logsoftmax! (:175-177).  Arithmetic in fp32.
//
// Bound by memory: every element has to be read and written once (the gradients read two arrays).  Columns therefore
// stay in registers between the reductions and the result, as 16-byte pieces, whatever their length and alignment:
// * A piece is VEC = 16 / sizeof(T) consecutive elements counted from the column's own start.  Columns of odd length
//   start at any element, so pieces are loads and stores of element alignment, which the memory pipeline takes at full
//   width.  The last piece is moved back to end with the column and its lane counts and stores only the elements that the piece
//   before it does not hold.
// * Short columns (up to 256 pieces): 4 to 64 lanes of a wavefront per column, up to four pieces a lane, reductions by
//   shuffles.  Longer ones (up to 8192 pieces): one workgroup of as many wavefronts as the column has work for, 4 or 8
//   pieces a lane, one barrier per reduction.  Beyond that the column is streamed twice (running maximum and sum, then
//   the result).
// Times before are those of the kernels this replaced (at most 4096 elements of a column in registers, one element a lane
// unless the columns were 16-byte aligned, three passes over longer ones); a large copy moves 4.8 TB/s on this card:
//   10000 x 4096 Float32          softmax 164 -> 80 us   logsoftmax 174 -> 75    its gradient 196 -> 91 (5.4 TB/s)
//   10007 x 8192 BFloat16                 269 -> 98                 282 -> 80                 328 -> 104
//   1001 x 65536 BFloat16                 161 -> 64                 200 -> 40                 357 -> 68
//   37 x 524288 Float32                    86 -> 30                1077 -> 27                1017 -> 35
//   131072 x 1024 Float32                 919 -> 293                876 -> 290                625 -> 368
#include "common.h"
#include "softmax_columns.h"

namespace {

template <typename T> struct Column : ColumnIO<T> {
    typedef typename T::type t;
    static constexpr int VEC = 16 / (int)sizeof(t);
    __device__ static float get(const u32x4_t &v, int e) {
        if constexpr (VEC == 4) return __builtin_bit_cast(floatx4_t, v)[e];
        else return T::to_f32(__builtin_bit_cast(typename T::vec8, v)[e]);
    }
    __device__ static void set(u32x4_t &v, int e, float x) {
        if constexpr (VEC == 4) {
            floatx4_t f = __builtin_bit_cast(floatx4_t, v);
            f[e] = x;
            v = __builtin_bit_cast(u32x4_t, f);
        } else {
            typename T::vec8 h = __builtin_bit_cast(typename T::vec8, v);
            h[e] = T::from_f32(x);
            v = __builtin_bit_cast(u32x4_t, h);
        }
    }
    // e^x: the library function for Float32, the hardware 2^x of x log2(e) for the 16-bit operations but softmax.  16-bit
    // softmax corrects that for what the product lost (4e-6 of the term at x = -80, a 24-bit x times 2^-24): 2^t e^r with
    // t = x log2(e) rounded and r = x - t ln 2, so small that e^r = 1 + r; at -Inf r is NaN and the minimum takes 1.  x <= 0.
    // (10007 x 8192 bf16: uncorrected 79 us, so 98, with the library function 109.)
    template <int OP> __device__ static float exp(float x) {
        if constexpr (VEC == 4) return expf(x);
        const float t = x * MI_LOG2E, e = mi_exp2(t);
        if constexpr (OP != OP_SOFTMAX) return e;
        constexpr float LN2 = 0x1.62e43p-1f, LN2_LOW = -0x1.05c610p-29f;   // ln 2 = LN2 + LN2_LOW
        return fmaf(e, fminf(fmaf(-t, LN2_LOW, fmaf(-t, LN2, x)), 1.0f), e);
    }
    // A BFloat16 result may be a subnormal number, which the hardware 2^x flushes to zero: pieces with one (elements 87 or
    // more below the maximum m) take the library function.
    static constexpr bool SUBNORMAL = __is_same(T, BF16);
    __device__ static bool subnormal(const u32x4_t &v, float m) {
        float low = get(v, 0);
#pragma unroll
        for (int e = 1; e < VEC; e++) low = fminf(low, get(v, e));
        return SUBNORMAL && low - m < -87.0f;
    }
    __device__ static float share(float term, float sum, float inv) { return VEC == 4 ? term / sum : quotient(term, sum, inv); }
};

// the reference's elementwise rules given the column maximum m
template <typename T> __device__ inline float softmax_term(float x, float m) {   // src/softmax.jl:72-75
    if (m == MI_POS_INF) return x == MI_POS_INF ? 1.0f : 0.0f;
    return Column<T>::template exp<OP_SOFTMAX>(x - m);
}
__device__ inline float logsoftmax_shift(float x, float m) {   // src/softmax.jl:140-144
    if (m == MI_POS_INF) return x == MI_POS_INF ? 0.0f : MI_NEG_INF;
    return x - m;
}
template <typename T, int OP> __device__ inline float term(float x, float m) {
    if (OP == OP_SOFTMAX) return softmax_term<T>(x, m);
    if (OP == OP_LOGSOFTMAX) return Column<T>::template exp<OP>(logsoftmax_shift(x, m));
    return Column<T>::template exp<OP>(x - m);   // logsumexp: no special cases (src/softmax.jl:202)
}
// the result of one element; forward: c0 = maximum, c1 = sum (softmax; c2 = 1 / sum) or log(sum); gradients: x = dy, c0 = the sum
template <typename T, int OP> __device__ inline float result(float x, float y, float c0, float c1, float c2, bool subnormal) {
    if (OP == OP_SOFTMAX) return Column<T>::share(subnormal && c0 < MI_POS_INF ? expf(x - c0) : softmax_term<T>(x, c0), c1, c2);
    if (OP == OP_LOGSOFTMAX) return logsoftmax_shift(x, c0) - c1;
    if (OP == OP_GRAD_SOFTMAX) return y * (x - c0);
    return x - c0 * Column<T>::template exp<OP>(y);
}

// The pieces stay in their packed form from pass to pass: without this the compiler keeps what the pass before computed
// of them (unpacked values, exponentials) as well, twice to three times the registers.
template <int N> __device__ inline void keep_packed(u32x4_t (&raw)[N]) {
#pragma unroll
    for (int u = 0; u < N; u++) asm volatile("" : "+v"(raw[u]));
}

// Reduction over the lanes of a column: G <= 64 lanes of a wavefront, or (G = 0) the whole workgroup.  `red` is the slot
// of this reduction; a slot is used again only after another reduction's barrier, so one barrier each is enough.
template <bool IS_MAX, int G> __device__ inline float reduce(float v, float *red) {
#pragma unroll
    for (int o = (G ? G : 64) / 2; o > 0; o >>= 1) {
        const float u = __shfl_xor(v, o, 64);
        v = IS_MAX ? fmaxf(v, u) : v + u;
    }
    if (G) return v;
    const int nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
    for (int w = 1; w < nw; w++) v = IS_MAX ? fmaxf(v, red[w]) : v + red[w];
    return v;
}

// One column held in registers.  G: lanes per column, 0 for a workgroup per column; NP: pieces per lane (the host picks
// both so that lanes * NP covers the column).
template <typename T, int OP, int NP, int G>
__global__ __launch_bounds__(G ? 256 : 1024) void softmax_column_kernel(const typename T::type *x, const typename T::type *x2,
                                                                         typename T::type *y, int len, int64_t cols) {
    typedef typename T::type t;
    typedef Column<T> C;
    constexpr int VEC = C::VEC;
    constexpr bool GRAD = OP >= OP_GRAD_SOFTMAX;
    constexpr bool KEEP_TERMS = OP == OP_SOFTMAX && VEC == 4;   // Float32 softmax: the terms take the place of the elements
    __shared__ float red[2][16];
    const int lanes = G ? G : blockDim.x, lane = G ? (int)threadIdx.x & (G - 1) : (int)threadIdx.x;
    const int per_block = G ? 256 / (G ? G : 1) : 1;
    const int last = (len - 1) / VEC;   // the column's last piece, which may be a partial one
    int parity = 0;
    for (int64_t c = (int64_t)blockIdx.x * per_block + (G ? threadIdx.x / (G ? G : 1) : 0); c < cols; c += (int64_t)gridDim.x * per_block) {
        const t *xc = x + c * len, *x2c = GRAD ? x2 + c * len : nullptr;
        t *yc = y + (OP == OP_LOGSUMEXP ? 0 : c * len);
        u32x4_t raw[NP], raw2[GRAD ? NP : 1];
        // lanes past the end read the last piece again: loads without branches, all of them in flight together
#pragma unroll
        for (int u = 0; u < NP; u++) {
            const int p = lane + u * lanes, at = p < last ? p * VEC : len - VEC;
            raw[u] = C::load(xc + at);
            if (GRAD) raw2[u] = C::load(x2c + at);
        }
        // elements of the last piece that another piece holds, and whole pieces past it, count for nothing
#pragma unroll
        for (int u = 0; u < NP; u++) {
            const int p = lane + u * lanes, skip = p * VEC - (len - VEC);
            if (p >= last && skip > 0) {
#pragma unroll
                for (int e = 0; e < VEC; e++)
                    if (e < skip) {
                        C::set(raw[u], e, GRAD ? 0.0f : MI_NEG_INF);
                        if (GRAD) C::set(raw2[u], e, 0.0f);
                    }
            }
        }
        float c0, c1 = 0.0f, c2 = 0.0f;
        if constexpr (GRAD) {
            float s = 0.0f;
#pragma unroll
            for (int u = 0; u < NP; u++)
#pragma unroll
                for (int e = 0; e < VEC; e++) s += OP == OP_GRAD_SOFTMAX ? C::get(raw[u], e) * C::get(raw2[u], e) : C::get(raw[u], e);
            c0 = reduce<false, G>(s, red[parity]);
            parity ^= 1;
            keep_packed(raw);
            keep_packed(raw2);
        } else {
            // fmaxf skips a NaN, but the NaN still reaches every element of its column through the sum
            float m = MI_NEG_INF, s = 0.0f;
#pragma unroll
            for (int u = 0; u < NP; u++)
#pragma unroll
                for (int e = 0; e < VEC; e++) m = fmaxf(m, C::get(raw[u], e));
            c0 = reduce<true, G>(m, red[0]);
            keep_packed(raw);
            // one test of the maximum for all elements of the column: a test per element becomes as many live values
            const auto add_terms = [&](auto rule) {
#pragma unroll
                for (int u = 0; u < NP; u++)
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        const float v = rule(C::get(raw[u], e));
                        if (KEEP_TERMS) C::set(raw[u], e, v);
                        s += v;
                    }
            };
            if (OP != OP_LOGSUMEXP && c0 == MI_POS_INF) add_terms([](float v) { return v == MI_POS_INF ? 1.0f : 0.0f; });
            else add_terms([&](float v) { return C::template exp<OP>(v - c0); });
            s = reduce<false, G>(s, red[1]);
            keep_packed(raw);
            c1 = OP != OP_SOFTMAX ? logf(s) : s;
            c2 = 1.0f / s;
        }
        if constexpr (OP == OP_LOGSUMEXP) {
            if (lane == 0) y[c] = T::from_f32(c0 + c1);
        } else {
            const auto write = [&](auto rule) {
#pragma unroll
                for (int u = 0; u < NP; u++) {
                    const int p = lane + u * lanes, at = p < last ? p * VEC : len - VEC, skip = p * VEC - at;
                    if (p > last) continue;
                    u32x4_t r = raw[u];
                    if (OP == OP_SOFTMAX && C::SUBNORMAL && C::subnormal(r, c0)) {
#pragma unroll
                        for (int e = 0; e < VEC; e++) C::set(r, e, result<T, OP>(C::get(raw[u], e), 0.0f, c0, c1, c2, true));
                    } else {
#pragma unroll
                        for (int e = 0; e < VEC; e++) C::set(r, e, rule(C::get(raw[u], e), GRAD ? C::get(raw2[GRAD ? u : 0], e) : 0.0f));
                    }
                    if (skip == 0) C::store(yc + at, r);
                    else
#pragma unroll
                        for (int e = 0; e < VEC; e++)
                            if (e >= skip) yc[at + e] = T::from_f32(C::get(r, e));
                }
            };
            if (!GRAD && !KEEP_TERMS && c0 == MI_POS_INF) write([&](float v, float) { return result<T, OP>(v, 0.0f, MI_POS_INF, c1, c2, false); });
            else write([&](float v, float v2) {
                if (KEEP_TERMS) return v / c1;
                if (OP == OP_SOFTMAX) return C::share(C::template exp<OP>(v - c0), c1, c2);
                if (OP == OP_LOGSOFTMAX) return v - c0 - c1;
                return result<T, OP>(v, v2, c0, c1, c2, false);
            });
        }
    }
}

// Columns longer than the registers of a workgroup: one pass for the running maximum and the sum against it, one for the
// result.  Four pieces in flight per lane; the tail piece is handled element by element.
template <typename T, int OP>
__global__ __launch_bounds__(1024) void softmax_column_stream_kernel(const typename T::type *x, const typename T::type *x2,
                                                                      typename T::type *y, int64_t len, int64_t cols) {
    typedef typename T::type t;
    typedef Column<T> C;
    constexpr int VEC = C::VEC, U = 4;
    constexpr bool GRAD = OP >= OP_GRAD_SOFTMAX;
    __shared__ float red[2][16];
    const int64_t whole = len / VEC, step = (int64_t)blockDim.x * U;
    for (int64_t c = blockIdx.x; c < cols; c += gridDim.x) {
        const t *xc = x + c * len, *x2c = GRAD ? x2 + c * len : nullptr;
        t *yc = y + (OP == OP_LOGSUMEXP ? 0 : c * len);
        float m = MI_NEG_INF, s = 0.0f;
        const auto add = [&](float v, float v2) {
            if (GRAD) s += OP == OP_GRAD_SOFTMAX ? v * v2 : v;
            else s += term<T, OP>(v, m);
        };
        // nothing but -Inf so far adds no terms; a column of nothing else is NaN in any case.  A NaN entry stays in the sum,
        // unless the maximum is +Inf: the sum then counts the +Inf entries (of logsumexp it is NaN), in any order.
        constexpr bool INDICATOR = OP == OP_SOFTMAX || OP == OP_LOGSOFTMAX;
        const auto raise = [&](float top) {
            if (top > m) {
                if (INDICATOR && top == MI_POS_INF) s = 0.0f;
                else s = m == MI_NEG_INF ? (s == s ? 0.0f : s) : s * C::template exp<OP>(m - top);
                m = top;
            }
        };
        for (int64_t p0 = threadIdx.x; p0 < whole; p0 += step) {
            u32x4_t raw[U], raw2[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int64_t p = p0 + (int64_t)u * blockDim.x, at = (p < whole ? p : p0) * VEC;
                raw[u] = C::load(xc + at);
                if (OP == OP_GRAD_SOFTMAX) raw2[u] = C::load(x2c + at);
            }
            if constexpr (!GRAD) {
                float top = MI_NEG_INF;
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int e = 0; e < VEC; e++) top = fmaxf(top, C::get(raw[u], e));
                raise(top);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (p0 + (int64_t)u * blockDim.x < whole)
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        const float v = C::get(raw[u], e);
                        if (GRAD || m != MI_NEG_INF || v != v) add(v, OP == OP_GRAD_SOFTMAX ? C::get(raw2[u], e) : 0.0f);
                    }
        }
        for (int64_t j = whole * VEC + threadIdx.x; j < len; j += blockDim.x) {
            const float v = T::to_f32(xc[j]);
            if (!GRAD) raise(v);
            if (GRAD || m != MI_NEG_INF || v != v) add(v, OP == OP_GRAD_SOFTMAX ? T::to_f32(x2c[j]) : 0.0f);
        }
        float c0, c1 = 0.0f, c2 = 0.0f;
        if constexpr (GRAD) {
            c0 = reduce<false, 0>(s, red[0]);
        } else {
            c0 = reduce<true, 0>(m, red[0]);
            // a lane that has seen nothing but -Inf holds no terms (or a NaN)
            if (INDICATOR && c0 == MI_POS_INF) s = m == c0 ? s : 0.0f;
            else s = m == c0 || s != s ? s : (m == MI_NEG_INF ? 0.0f : s * C::template exp<OP>(m - c0));
            s = reduce<false, 0>(s, red[1]);
            if (c0 == MI_NEG_INF) s = __builtin_nanf("");
            c1 = OP != OP_SOFTMAX ? logf(s) : s;
            c2 = 1.0f / s;
        }
        if constexpr (OP == OP_LOGSUMEXP) {   // the reference's x - max is Inf - Inf for an infinite maximum
            if (threadIdx.x == 0) y[c] = T::from_f32(c0 == MI_POS_INF ? __builtin_nanf("") : c0 + c1);
        } else {
            for (int64_t p0 = threadIdx.x; p0 < whole; p0 += step) {
                u32x4_t raw[U], raw2[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int64_t p = p0 + (int64_t)u * blockDim.x, at = (p < whole ? p : p0) * VEC;
                    raw[u] = C::load(xc + at);
                    if (GRAD) raw2[u] = C::load(x2c + at);
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int64_t p = p0 + (int64_t)u * blockDim.x;
                    if (p >= whole) break;
                    u32x4_t r = raw[u];
                    if (OP == OP_SOFTMAX && C::SUBNORMAL && C::subnormal(r, c0)) {
#pragma unroll
                        for (int e = 0; e < VEC; e++) C::set(r, e, result<T, OP>(C::get(raw[u], e), 0.0f, c0, c1, c2, true));
                    } else {
#pragma unroll
                        for (int e = 0; e < VEC; e++) C::set(r, e, result<T, OP>(C::get(raw[u], e), GRAD ? C::get(raw2[u], e) : 0.0f, c0, c1, c2, false));
                    }
                    C::store(yc + p * VEC, r);
                }
            }
            for (int64_t j = whole * VEC + threadIdx.x; j < len; j += blockDim.x)
                yc[j] = T::from_f32(result<T, OP>(T::to_f32(xc[j]), GRAD ? T::to_f32(x2c[j]) : 0.0f, c0, c1, c2, Column<T>::SUBNORMAL));
        }
        __syncthreads();   // red is written again by the next column
    }
}

// Columns shorter than one piece: a thread each.
template <typename T, int OP>
__global__ __launch_bounds__(256) void softmax_tiny_column_kernel(const typename T::type *x, const typename T::type *x2,
                                                                   typename T::type *y, int len, int64_t cols) {
    constexpr int MOST = Column<T>::VEC - 1;
    constexpr bool GRAD = OP >= OP_GRAD_SOFTMAX;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < cols; c += (int64_t)gridDim.x * 256) {
        float v[MOST], v2[MOST], m = MI_NEG_INF, s = 0.0f;
#pragma unroll
        for (int j = 0; j < MOST; j++)
            if (j < len) {
                v[j] = T::to_f32(x[c * len + j]);
                v2[j] = GRAD ? T::to_f32(x2[c * len + j]) : 0.0f;
                m = fmaxf(m, v[j]);
            }
#pragma unroll
        for (int j = 0; j < MOST; j++)
            if (j < len) s += GRAD ? (OP == OP_GRAD_SOFTMAX ? v[j] * v2[j] : v[j]) : term<T, OP>(v[j], m);
        if constexpr (OP == OP_LOGSUMEXP) {
            y[c] = T::from_f32(m + logf(s));
        } else {
            const float c0 = GRAD ? s : m, c1 = OP == OP_LOGSOFTMAX ? logf(s) : s, c2 = 1.0f / s;
#pragma unroll
            for (int j = 0; j < MOST; j++)
                if (j < len) y[c * len + j] = T::from_f32(result<T, OP>(v[j], v2[j], c0, c1, c2, Column<T>::SUBNORMAL));
        }
    }
}

template <typename T, int OP>
void launch(const void *x, const void *x2, void *y, int64_t len, int64_t cols, hipStream_t st) {
    typedef typename T::type t;
    constexpr int VEC = Column<T>::VEC;
    // A workgroup of 1024 threads (128 registers each) holds 8 pieces a lane.  Streamed instead, columns of 4096 to 8192
    // pieces are level (softmax, 32000 Float32: 131 / 132 us for 2048 columns) or slower (their gradient: 151 / 193 us);
    // 16 pieces a lane spill (50257 Float32, 1024 columns: 127 us, streamed 110).
    constexpr int64_t CACHED = 8192;
    const int64_t pieces = (len + VEC - 1) / VEC, most_blocks = 1 << 20;
    const auto blocks = [&](int64_t per_block) {
        const int64_t n = (cols + per_block - 1) / per_block;
        return dim3((unsigned)(n < most_blocks ? n : most_blocks));
    };
#define MI_COLUMN(NP, G, LANES)                                                                                                 \
    hipLaunchKernelGGL((softmax_column_kernel<T, OP, NP, G>), blocks(G ? 256 / (G ? G : 1) : 1), dim3(G ? 256 : LANES), 0, st,  \
                       (const t *)x, (const t *)x2, (t *)y, (int)len, cols)
    if (len < VEC) {
        hipLaunchKernelGGL((softmax_tiny_column_kernel<T, OP>), blocks(256), dim3(256), 0, st, (const t *)x, (const t *)x2, (t *)y,
                           (int)len, cols);
    } else if (pieces <= 4) MI_COLUMN(1, 4, 256);
    else if (pieces <= 8) MI_COLUMN(2, 4, 256);
    else if (pieces <= 16) MI_COLUMN(2, 8, 256);
    else if (pieces <= 32) MI_COLUMN(2, 16, 256);
    else if (pieces <= 64) MI_COLUMN(2, 32, 256);
    else if (pieces <= 128) MI_COLUMN(2, 64, 256);
    else if (pieces <= 256) MI_COLUMN(4, 64, 256);
    else if (pieces <= CACHED) {
        // whole wavefronts, as few as the pieces need
        const auto lanes = [&](int np) { return (unsigned)((pieces + 64 * np - 1) / (64 * np) * 64); };
        if (pieces <= 4096) MI_COLUMN(4, 0, lanes(4));
        else MI_COLUMN(8, 0, lanes(8));
    } else {
        hipLaunchKernelGGL((softmax_column_stream_kernel<T, OP>), blocks(1), dim3(1024), 0, st, (const t *)x, (const t *)x2, (t *)y, len, cols);
    }
#undef MI_COLUMN
}

template <typename T> void launch_op(int op, const void *x, const void *x2, void *y, int64_t len, int64_t cols, hipStream_t st) {
    if (op == OP_SOFTMAX) launch<T, OP_SOFTMAX>(x, x2, y, len, cols, st);
    else if (op == OP_LOGSOFTMAX) launch<T, OP_LOGSOFTMAX>(x, x2, y, len, cols, st);
    else if (op == OP_LOGSUMEXP) launch<T, OP_LOGSUMEXP>(x, x2, y, len, cols, st);
    else if (op == OP_GRAD_SOFTMAX) launch<T, OP_GRAD_SOFTMAX>(x, x2, y, len, cols, st);
    else launch<T, OP_GRAD_LOGSOFTMAX>(x, x2, y, len, cols, st);
}

}  // namespace

void launch_softmax_columns(int32_t dtype, int op, const void *x, const void *x2, void *y, int64_t len, int64_t cols, hipStream_t st) {
    if (dtype == MI_F32) launch_op<F32>(op, x, x2, y, len, cols, st);
    else if (dtype == MI_F16) launch_op<F16>(op, x, x2, y, len, cols, st);
    else launch_op<BF16>(op, x, x2, y, len, cols, st);
}

MI_API int32_t mi_softmax_dim1(int32_t dtype, const void *x, void *y, int64_t rows, int64_t cols, mi_stream s) {
    if (!mi_dtype_ok_f64(dtype)) return mi_set_error(MI_EDTYPE, "mi_softmax_dim1: unknown dtype %d", dtype);
    if (rows < 0 || cols < 0) return mi_set_error(MI_EINVAL, "mi_softmax_dim1: negative size");
    if (rows == 0 || cols == 0) return MI_OK;
    if (!x || !y) return mi_set_error(MI_EINVAL, "mi_softmax_dim1: null pointer");
    hipStream_t st = (hipStream_t)s;
    if (dtype == MI_F64) return launch_softmax_family_f64(OP_SOFTMAX, x, nullptr, y, 1, rows, cols, st);
    launch_softmax_columns(dtype, OP_SOFTMAX, x, nullptr, y, rows, cols, st);
    MI_LAUNCH_CHECK();
    return MI_OK;
}
