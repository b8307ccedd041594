// Float32 batched products whose tiles the kernels of batched_gemm32.hip leave half empty or too few: odd and narrow
// results, short or long k, small batches.  C[:,:,b] = alpha*op(A)*op(B) + beta*C, or the sum of such products over the
// batch (the gradient of an operand that every slice shares, src/batched/batchedmul.jl:96-110).
//
// A wavefront owns a result tile of BM x BN blocks of 32 x 32 by itself: its operands go from memory straight into the
// layout of the matrix instruction (lane l: row l % 32, eight consecutive k), are split into bf16 planes in registers (see
// common.h) and multiplied.  No LDS and no barrier stand between the loads of a step and its products, and the next step's
// loads are in flight meanwhile.  SPLIT wavefronts of a workgroup take every SPLIT-th step of 16 k of one tile and add up
// their sums through LDS, so that a small result still has many loads in flight; with SPLIT = 1 a wavefront is a workgroup.
//
// What bounds it: at k above about 100 the vector instructions (splitting, range checks, addresses: 14 a matrix instruction for
// 2 x 2 blocks, 56 cycles where the matrix pipe alone takes 32), which the two wavefronts of a SIMD overlap in part, and the
// last round of workgroups.  Counters of 333 x 77 x 517, 96 slices, 1152 workgroups where the chip holds 512: vector
// instructions 42 % of the SIMDs' cycles, matrix instructions 24 %, a CU has a wavefront 72 % of the time.  Below, a launch's
// 4 us, the first step's memory round trip and the store of the result.  Against the LDS-staged kernels (one stage of 16 k
// in flight, at least one 128 x 128 tile of four wavefronts): 320 x 16 x 816, 20 slices, 64.5 -> 8.0 us;
// 100 x 100 x 100, 50 slices, 13.0 -> 5.6; 464 x 16 x 416, 28 slices, 34.8 -> 7.5; 333 x 517 x 16, 96 slices, 22.6 -> 17
// (66 MB of results: 3.9 TB/s); 77 x 333 x 517, 96 slices, 59 to 69 -> 41 to 52 us by the operands' orientation.
#include "common.h"

namespace {

struct WaveArgs {
    const float *A, *B;
    float *C;
    int64_t m, n, k, lda, ldb, ldc, sA, sB, sC;
    float alpha, beta;
    int32_t slices;            // slices of A and B that are summed into one of C
    int32_t tiles_m, tiles_n;
};

typedef bf16x8_t plane8;

// Rows of op(X) in blocks of 32.  RM: element (row, kk) at X[row + kk*ld]; else at X[kk + row*ld].
template <bool RM, int NB>
struct WaveOperand {
    static constexpr int OOB = 0x7fffffff;
    const float *X;
    int64_t ld, stride;
    int bytes;
    int voff[NB];          // byte offset of this lane's row (RM: of its first k of a step too)
    __device__ void init(const float *X_, int64_t ld_, int64_t stride_, int64_t rows, int64_t k, int64_t row0) {
        const int lane = threadIdx.x & 63, r = lane & 31, hh = lane >> 5;
        X = X_;
        ld = ld_;
        stride = stride_;
        bytes = (int)((RM ? (k - 1) * ld + rows : (rows - 1) * ld + k) * 4);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            int64_t row = row0 + 32 * i + r;
            row = row < rows ? row : rows - 1;   // rows past the end repeat the last one; their results are not stored
            voff[i] = (int)((RM ? row + 8 * hh * ld : row * ld + 8 * hh) * 4);
        }
    }
    // the step of 16 k at k0 of slice `sl`: x[i][e] = element (row of block i, k0 + 8*hh + e), zero from `left` = k - k0 on
    __device__ void load(int64_t sl, int k0, int left, float (&x)[NB][8]) const {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)(X + sl * stride), 0, bytes, 0x00020000);
        if (left < 16) {   // the k term goes into the range-checked part of the address
            const int mine = left - 8 * (int)((threadIdx.x >> 5) & 1);
#pragma unroll
            for (int i = 0; i < NB; i++)
#pragma unroll
                for (int e = 0; e < 8; e++)
                    x[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, e < mine ? voff[i] + (int)((RM ? (k0 + e) * ld : k0 + e) * 4) : OOB, 0, 0));
        } else if (RM) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int at = (int)((k0 + e) * ld * 4);
#pragma unroll
                for (int i = 0; i < NB; i++) x[i][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, voff[i], at, 0));
            }
        } else {
#pragma unroll
            for (int i = 0; i < NB; i++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const floatx4_t v = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[i], (k0 + 4 * u) * 4, 0));
#pragma unroll
                    for (int e = 0; e < 4; e++) x[i][4 * u + e] = v[e];
                }
        }
    }
};

// Planes do not hold values beyond bf16's largest (an Inf among them: Inf times Inf would be NaN) and lose the low bits of
// values whose last plane leaves bf16's range (below 2^-100): 2 |x| - 1 in bits, a zero counting as the largest, must be at
// least `least` and, zeros aside, at most `most`.
template <int NB>
__device__ inline void extremes(const float (&x)[NB][8], uint32_t &lo, float &hi) {
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(hi) : "v"(x[i][e]), "v"(x[i][e + 1]));
            const uint32_t s0 = (__builtin_bit_cast(uint32_t, x[i][e]) << 1) - 1, s1 = (__builtin_bit_cast(uint32_t, x[i][e + 1]) << 1) - 1;
            lo = min(min(s0, s1), lo);
        }
}

template <int NB>
__device__ inline void split_step(const float (&x)[NB][8], plane8 (&pl)[NB][3]) {
#pragma unroll
    for (int i = 0; i < NB; i++) {
        u32x4_t w[3];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uint32_t a, b, c;
            split3_pair(x[i][2 * e], x[i][2 * e + 1], a, b, c);
            w[0][e] = a;
            w[1][e] = b;
            w[2][e] = c;
        }
#pragma unroll
        for (int q = 0; q < 3; q++) pl[i][q] = __builtin_bit_cast(plane8, w[q]);
    }
}

// SUM: one result, the sum over the slices.  Every slice's products have an accumulator of their own, which is added to the
// sum when the next slice starts, as a product per slice adds to C.  One accumulator over all of them errs with the root of
// its length (against 64 bits, 2-norm, one accumulator / this / a product per slice: 333 x 77 x 517 over 96 slices 1.5e-6 /
// 3.0e-7 / 3.0e-7, 32 x 32 x 77 over 96 5.1e-7 / 2.5e-7 / 2.7e-7), and is 3 to 9 % faster: the sums wait for a slice's last
// matrix instruction and take registers of their own (464 x 16 x 416 over 28 slices 69.4 / 71.6 us, 16 x 16 x 16 over 1000
// 122 / 132), for which the wavefronts a SIMD go from five to four, with 2 x 2 blocks from two to one.
template <bool A_RM, bool B_RM, int BM, int BN, int SPLIT, bool SUM>
__global__ __launch_bounds__(64 * SPLIT, BM * BN == 1 ? (SUM ? 4 : 5) : (SUM ? 1 : 2)) void gemm32_waves_kernel(WaveArgs g) {
    constexpr int LDW = 32 * BM + 4;   // floats per LDS row
    __shared__ __attribute__((aligned(16))) float part[SPLIT][32 * LDW];
    const int lane = threadIdx.x & 63, r = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // dies take contiguous runs of tiles, m fastest: the tiles of a slice share its operands, and the two halves of a cache
    // line that a tile's edge cuts, through one L2 (333 x 517 x 77, 96 slices: 49.8 -> 39.3 us)
    const int64_t item = mi_xcd_order(blockIdx.x, gridDim.x);
    const int in_slice = (int)(item % (g.tiles_m * g.tiles_n));
    const int64_t bz = item / (g.tiles_m * g.tiles_n);
    const int64_t m0 = (int64_t)(in_slice % g.tiles_m) * (32 * BM), n0 = (int64_t)(in_slice / g.tiles_m) * (32 * BN);

    WaveOperand<A_RM, BM> a;
    WaveOperand<B_RM, BN> b;
    const int64_t z = SUM ? 0 : bz;
    a.init(g.A + z * g.sA, g.lda, g.sA, g.m, g.k, m0);
    b.init(g.B + z * g.sB, g.ldb, g.sB, g.n, g.k, n0);

    floatx16_t acc[BN][BM];   // the transposed problem: rows = n, columns = m
#pragma unroll
    for (int i = 0; i < BN; i++)
#pragma unroll
        for (int j = 0; j < BM; j++) acc[i][j] = (floatx16_t){0};

    floatx16_t total[BN][BM];   // SUM: the slices before the present one
#pragma unroll
    for (int i = 0; i < BN; i++)
#pragma unroll
        for (int j = 0; j < BM; j++) total[i][j] = (floatx16_t){0};
    const auto next_slice = [&] {
#pragma unroll
        for (int i = 0; i < BN; i++)
#pragma unroll
            for (int j = 0; j < BM; j++) {
#pragma unroll
                for (int v = 0; v < 16; v++) total[i][j][v] += acc[i][j][v];
                acc[i][j] = (floatx16_t){0};
            }
    };

    // steps wave, wave + SPLIT, ... of the slices' steps, one after the other; two steps' loads are in flight
    const int per_slice = (int)((g.k + 15) / 16), k = (int)g.k;
    struct Step { int sl, st; };
    const auto next = [&](Step s) {
        s.st += SPLIT;
        while (s.st >= per_slice && s.sl < g.slices) {
            s.st -= per_slice;
            s.sl++;
        }
        return s;
    };
    float xa[2][BM][8], xb[2][BN][8];
    uint32_t lo = ~0u;
    float hi = 0.0f;
    const auto fetch = [&](Step s, int at) {
        if (s.sl >= g.slices) return;
        a.load(s.sl, 16 * s.st, k - 16 * s.st, xa[at]);
        b.load(s.sl, 16 * s.st, k - 16 * s.st, xb[at]);
    };
    const auto multiply = [&](Step ahead, int at, bool first_of_slice) {
        extremes<BM>(xa[at], lo, hi);
        extremes<BN>(xb[at], lo, hi);
        plane8 av[BM][3], bv[BN][3];
        split_step<BM>(xa[at], av);
        split_step<BN>(xb[at], bv);
        fetch(ahead, at);
        if (SUM && first_of_slice) next_slice();
        constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, ib[6] = {0, 2, 1, 0, 1, 0};   // small terms first
#pragma unroll
        for (int t = 0; t < 6; t++)
#pragma unroll
            for (int i = 0; i < BN; i++)
#pragma unroll
                for (int j = 0; j < BM; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bv[i][ib[t]], av[j][ia[t]], acc[i][j], 0, 0, 0);
    };
    const Step first = next({0, wave - SPLIT});
    // one or two terms a sum: the planes' own error, up to 2.6 * 2^-24 of a product, would show (2-norm against 64 bits, planes /
    // Float32 instruction: k = 1 3.5e-8 / 2.5e-8, 2 3.4e-8 / 3.1e-8, 3 3.3e-8 / 3.6e-8)
    const bool planes = k >= 3;
    if (planes) {
        Step s0 = first, s1 = next(first);
        int slice = first.sl;
        fetch(s0, 0);
        fetch(s1, 1);
        while (s0.sl < g.slices) {
            const Step s2 = next(s1), s3 = next(s2);
            multiply(s2, 0, s0.sl != slice);
            if (s1.sl < g.slices) multiply(s3, 1, s1.sl != s0.sl);
            slice = s1.sl;
            s0 = s2;
            s1 = s3;
        }
    }
    if (!planes || __builtin_amdgcn_ballot_w64(!(hi <= 0x1.fep127f && lo >= (27u << 24) - 1)) != 0) {
        // on the Float32 instruction, which takes one k of each half-wave: the registers as they are, in eight steps
#pragma unroll
        for (int i = 0; i < BN; i++)
#pragma unroll
            for (int j = 0; j < BM; j++) acc[i][j] = total[i][j] = (floatx16_t){0};
        int slice = first.sl;
        for (Step s = first; s.sl < g.slices; s = next(s)) {
            fetch(s, 0);
            if (SUM && s.sl != slice) next_slice();
            slice = s.sl;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (e >= 2 && !planes) break;
#pragma unroll
                for (int i = 0; i < BN; i++)
#pragma unroll
                    for (int j = 0; j < BM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xb[0][i][e], xa[0][j][e], acc[i][j], 0, 0, 0);
            }
        }
    }

    if (SUM) next_slice();

    // 32 columns of the tile at a time: every wavefront leaves its sums in LDS, the workgroup adds them and stores 16-byte
    // pieces along m.  Register v of lane (r, hh) of block (i, j): n = 32i + 8*(v/4) + 4*hh + v%4, m = 32j + r.
    float *C = g.C + bz * g.sC;
#pragma unroll
    for (int i = 0; i < BN; i++) {
        if (SPLIT > 1) __syncthreads();
        else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
#pragma unroll
        for (int j = 0; j < BM; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) part[wave][(8 * (v / 4) + 4 * hh + (v % 4)) * LDW + 32 * j + r] = SUM ? total[i][j][v] : acc[i][j][v];
        if (SPLIT > 1) __syncthreads();
        else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
#pragma unroll
        for (int u = 0; u < (32 * 8 * BM + 64 * SPLIT - 1) / (64 * SPLIT); u++) {
            const int c = (int)threadIdx.x + 64 * SPLIT * u;
            if ((32 * 8 * BM) % (64 * SPLIT) != 0 && c >= 32 * 8 * BM) break;
            const int nl = c / (8 * BM), ml = (c % (8 * BM)) * 4;
            floatx4_t val = *(const floatx4_t *)&part[0][nl * LDW + ml];
#pragma unroll
            for (int w = 1; w < SPLIT; w++) {
                const floatx4_t o = *(const floatx4_t *)&part[w][nl * LDW + ml];
#pragma unroll
                for (int e = 0; e < 4; e++) val[e] += o[e];
            }
            const int64_t nj = n0 + 32 * i + nl, mi = m0 + ml;
            if (nj >= g.n || mi >= g.m) continue;
            float *c4 = C + mi + nj * g.ldc;
#pragma unroll
            for (int e = 0; e < 4; e++) val[e] *= g.alpha;
            if (mi + 4 <= g.m) {
                if (g.beta != 0.0f) {
                    const floatx4_t old = __builtin_bit_cast(floatx4_t, *(const mi_piece4_t *)c4);
#pragma unroll
                    for (int e = 0; e < 4; e++) val[e] += g.beta * old[e];
                }
                *(mi_piece4_t *)c4 = __builtin_bit_cast(u32x4_t, val);
            } else {
#pragma unroll
                for (int e = 0; e < 3; e++)
                    if (mi + e < g.m) c4[e] = g.beta != 0.0f ? val[e] + g.beta * c4[e] : val[e];
            }
        }
    }
}

// work items of a launch are counted in 32 bits: larger batches go in slabs of slices
constexpr int64_t MOST_THREADS = ((int64_t)1 << 32) - 1;

template <int BM, int BN, int SPLIT, bool SUM>
int32_t launch_waves(WaveArgs g, bool a_rm, bool b_rm, int64_t nb, hipStream_t st) {
    g.tiles_m = (int32_t)((g.m + 32 * BM - 1) / (32 * BM));
    g.tiles_n = (int32_t)((g.n + 32 * BN - 1) / (32 * BN));
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n, most = MOST_THREADS / (64 * SPLIT) / tiles;   // slices per launch, at least one
    for (int64_t b0 = 0; b0 < nb; b0 += most) {
        const dim3 grid((unsigned)(tiles * (nb - b0 < most ? nb - b0 : most))), block(64 * SPLIT);
        if (a_rm && b_rm) hipLaunchKernelGGL((gemm32_waves_kernel<true, true, BM, BN, SPLIT, SUM>), grid, block, 0, st, g);
        else if (a_rm) hipLaunchKernelGGL((gemm32_waves_kernel<true, false, BM, BN, SPLIT, SUM>), grid, block, 0, st, g);
        else if (b_rm) hipLaunchKernelGGL((gemm32_waves_kernel<false, true, BM, BN, SPLIT, SUM>), grid, block, 0, st, g);
        else hipLaunchKernelGGL((gemm32_waves_kernel<false, false, BM, BN, SPLIT, SUM>), grid, block, 0, st, g);
        MI_LAUNCH_CHECK();
        g.A += most * g.sA;
        g.B += most * g.sB;
        g.C += most * g.sC;
    }
    return MI_OK;
}

// Time of a product in microseconds: a launch, then either one wavefront's chain of steps or, with more wavefronts than the
// chip's 1024 SIMDs work off in that time, their vector work.  {per step, per wavefront} of the chain and {per step, per
// wavefront} of a SIMD's share, fitted to 170 products of 16 to 1024 rows, columns and k and 1 to 256 slices in both
// orientations of both operands (mean deviation 5 to 7 %; the variant chosen by these is on average 3 % slower than the
// fastest one measured).
struct Variant { int bm, bn, split; double chain_step, chain, share_step, share; };
constexpr Variant variants[] = {
    {1, 1, 1, 0.45, 0.05, 0.42, 0.36}, {1, 1, 4, 0.31, 0.69, 0.37, 0.06}, {1, 1, 8, 0.50, 0.50, 0.355, 0.13},
    {2, 2, 1, 0.91, 0.49, 1.15, 2.26}, {2, 2, 4, 0.94, 0.36, 0.92, 0.86},
};

double estimate(const Variant &v, int64_t m, int64_t n, int64_t steps, int64_t batch) {
    const double mine = (double)((steps + v.split - 1) / v.split);
    const double per_simd = (double)((m + 32 * v.bm - 1) / (32 * v.bm)) * (double)((n + 32 * v.bn - 1) / (32 * v.bn)) * (double)batch * v.split / 1024.0;
    return 4.0 + fmax(v.chain_step * mine + v.chain, per_simd * (v.share_step * mine + v.share));
}

const Variant &fastest(int64_t m, int64_t n, int64_t steps, int64_t batch) {
    const Variant *best = variants;
    for (const Variant &v : variants)
        if (estimate(v, m, n, steps, batch) < estimate(*best, m, n, steps, batch)) best = &v;
    return *best;
}

template <bool SUM>
int32_t launch_variant(const WaveArgs &g, const Variant &v, bool a_rm, bool b_rm, int64_t batch, hipStream_t st) {
    if (v.bm == 2) return v.split == 1 ? launch_waves<2, 2, 1, SUM>(g, a_rm, b_rm, batch, st) : launch_waves<2, 2, 4, SUM>(g, a_rm, b_rm, batch, st);
    if (v.split == 1) return launch_waves<1, 1, 1, SUM>(g, a_rm, b_rm, batch, st);
    return v.split == 4 ? launch_waves<1, 1, 4, SUM>(g, a_rm, b_rm, batch, st) : launch_waves<1, 1, 8, SUM>(g, a_rm, b_rm, batch, st);
}

}  // namespace

// 32-bit byte offsets reach every element of a slice, and the end of its last step of 16 k; a slice fits one launch of eight
// wavefronts a tile
bool gemm32_waves_supports(int transA, int transB, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb) {
    const int64_t reachA = transA ? m * lda + k : (k + 16) * lda + m, reachB = transB ? (k + 16) * ldb + n : n * ldb + k;
    if (reachA >= (int64_t)1 << 29 || reachB >= (int64_t)1 << 29) return false;
    return ((m + 31) / 32) * ((n + 31) / 32) <= MOST_THREADS / 512;
}

double gemm32_waves_estimate(int64_t m, int64_t n, int64_t k, int64_t slices, int64_t batch) {
    const int64_t steps = slices * ((k + 15) / 16);
    return estimate(fastest(m, n, steps, batch), m, n, steps, batch);
}

// slices > 1: one result, the sum over that many slices of A and B (batch = 1)
int32_t launch_gemm32_waves(int transA, int transB, int64_t m, int64_t n, int64_t k, float alpha, const void *A, int64_t lda,
                            int64_t sA, const void *B, int64_t ldb, int64_t sB, float beta, void *C, int64_t ldc, int64_t sC,
                            int64_t slices, int64_t batch, hipStream_t st) {
    const WaveArgs g = {(const float *)A, (const float *)B, (float *)C, m, n, k, lda, ldb, ldc, sA, sB, sC, alpha, beta, (int32_t)slices, 0, 0};
    const Variant &v = fastest(m, n, slices * ((k + 15) / 16), batch);
    return slices > 1 ? launch_variant<true>(g, v, !transA, transB != 0, batch, st) : launch_variant<false>(g, v, !transA, transB != 0, batch, st);
}
