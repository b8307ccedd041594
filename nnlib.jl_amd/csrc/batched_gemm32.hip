// Strided batched GEMM for Float32 on the matrix cores: the fast path of mi_batched_gemm, operands
// moved in 16-byte pieces (of any alignment in the kernels on bf16 planes).  Products that would leave these tiles empty or
// too few run in batched_gemm32_waves.hip.  Stands where the
// reference calls sgemm per slice (src/gemm.jl:141-149, reached through _batched_gemm!,
// src/batched/batchedmul.jl:298).  Sums are Float32; products run on three bf16 planes per operand (gemm32s_kernel
// below), or, where MI355ATTN_F32_MFMA asks for it, on the Float32 matrix instruction (gemm32_kernel, aligned operands).
//
// gemm32_kernel: workgroup = 4 wavefronts (2 x 2), output tile 128 (m) x 128 (n), 64 x 64 per wavefront as 2 x 2 MFMA
// blocks; k advances 16 per stage through double-buffered LDS tiles kept as [k][row] (row contiguous),
// so an MFMA operand (one float per lane: row = lane % 32, k = 2*step + lane / 32) is a conflict-free
// 4-byte read whatever the memory layout of the matrix.  As in the other GEMM kernels the MFMA runs on
// the transposed problem so that a half-wave stores 32 consecutive elements of a C column.
#include "common.h"
#include <cstdlib>
#include <type_traits>

// a wavefront per tile, no LDS between operands and products (batched_gemm32_waves.hip)
bool gemm32_waves_supports(int transA, int transB, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb);
double gemm32_waves_estimate(int64_t m, int64_t n, int64_t k, int64_t slices, int64_t batch);
int32_t launch_gemm32_waves(int transA, int transB, int64_t m, int64_t n, int64_t k, float alpha, const void *A, int64_t lda,
                            int64_t sA, const void *B, int64_t ldb, int64_t sB, float beta, void *C, int64_t ldc, int64_t sC,
                            int64_t slices, int64_t batch, hipStream_t st);

namespace {

constexpr int TM = 128, TN = 128, KC = 16;
constexpr int LDT = 128 + 4;   // floats per k-row of a tile (+4: the strided stores of k-contiguous operands spread over banks)

struct Gemm32Args {
    const float *A, *B;
    float *C;
    int64_t m, n, k, lda, ldb, ldc, sA, sB, sC;
    float alpha, beta;
};

// RM: element (row, kk) at X[row + kk*ld] (contiguous along row); else at X[kk + row*ld]
template <bool RM>
struct Operand32 {
    const float *X;
    int64_t ld, rows, k, row0;
    floatx4_t reg[2];   // 512 pieces of 16 bytes per tile, 2 per thread

    __device__ void load(int64_t k0) {
        const int tid = threadIdx.x;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int c = tid + 256 * u;
            const floatx4_t z = {0.f, 0.f, 0.f, 0.f};
            if (RM) {
                const int kk = c >> 5, r4 = (c & 31) * 4;     // 32 pieces per k-row
                reg[u] = (k0 + kk < k && row0 + r4 < rows) ? *(const floatx4_t *)(X + (row0 + r4) + (k0 + kk) * ld) : z;
            } else {
                const int r = c >> 2, k4 = (c & 3) * 4;       // 4 pieces per row
                reg[u] = (row0 + r < rows && k0 + k4 < k) ? *(const floatx4_t *)(X + (k0 + k4) + (row0 + r) * ld) : z;
            }
        }
    }
    __device__ void store(float *tile) const {
        const int tid = threadIdx.x;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int c = tid + 256 * u;
            if (RM) {
                const int kk = c >> 5, r4 = (c & 31) * 4;
                *(floatx4_t *)(tile + kk * LDT + r4) = reg[u];
            } else {
                const int r = c >> 2, k4 = (c & 3) * 4;
#pragma unroll
                for (int e = 0; e < 4; e++) tile[(k4 + e) * LDT + r] = reg[u][e];
            }
        }
    }
};

template <bool A_RM, bool B_RM>
__global__ __launch_bounds__(256, 2) void gemm32_kernel(Gemm32Args g) {
    __shared__ __attribute__((aligned(16))) float As[2][KC * LDT];
    __shared__ __attribute__((aligned(16))) float Bs[2][KC * LDT];
    const int64_t bz = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave & 1, wn = wave >> 1;
    const int r = lane & 31, hh = lane >> 5;

    Operand32<A_RM> a;
    Operand32<B_RM> b;
    a.X = g.A + bz * g.sA;
    a.ld = g.lda;
    a.rows = g.m;
    a.k = g.k;
    a.row0 = (int64_t)blockIdx.x * TM;
    b.X = g.B + bz * g.sB;
    b.ld = g.ldb;
    b.rows = g.n;
    b.k = g.k;
    b.row0 = (int64_t)blockIdx.y * TN;

    floatx16_t acc[2][2];   // [n block][m block]
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = (floatx16_t){0};

    const int nk = (int)((g.k + KC - 1) / KC);
    a.load(0);
    b.load(0);
    a.store(As[0]);
    b.store(Bs[0]);
    __syncthreads();
    for (int it = 0; it < nk; it++) {
        const int buf = it & 1;
        if (it + 1 < nk) {
            a.load((int64_t)(it + 1) * KC);
            b.load((int64_t)(it + 1) * KC);
        }
        const float *at = As[buf] + 64 * wm + r, *bt = Bs[buf] + 64 * wn + r;
#pragma unroll
        for (int ks = 0; ks < KC / 2; ks++) {
            float av[2], bv[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                av[j] = at[(2 * ks + hh) * LDT + 32 * j];
                bv[j] = bt[(2 * ks + hh) * LDT + 32 * j];
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[i], av[j], acc[i][j], 0, 0, 0);
        }
        if (it + 1 < nk) {
            a.store(As[buf ^ 1]);
            b.store(Bs[buf ^ 1]);
        }
        __syncthreads();
    }

    // accumulator register v of lane (r, hh) of block (i, j): n = 32i + 8*(v/4) + 4*hh + v%4, m = 32j + r
    float *C = g.C + bz * g.sC;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int64_t mi = a.row0 + 64 * wm + 32 * j + r;
        if (mi >= g.m) continue;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int64_t nj = b.row0 + 64 * wn + 32 * i + 8 * (v / 4) + 4 * hh + (v % 4);
                if (nj < g.n) {
                    float *c = C + mi + nj * g.ldc;
                    float val = g.alpha * acc[i][j][v];
                    if (g.beta != 0.0f) val += g.beta * *c;
                    *c = val;
                }
            }
    }
}

// ---------------------------------------------------------------------------------------------------
// The same product on the 16-bit matrix cores: both operands as three bf16 planes (see common.h), six
// v_mfma_f32_32x32x16_bf16 per 32x32x16 block.  Same workgroup shape and double-buffered 16-k stages; a tile
// is split when it is stored to LDS and keeps the orientation its memory has, as in the 16-bit kernel:
//   RMAJ (contiguous along its row index): [16 k][rows] per plane, k-rows of 2 bytes per row with swizzled
//        16-byte chunks, MFMA operand through the transposing LDS read;
//   KMAJ (contiguous along k): [rows][16 k] per plane, 32-byte rows whose two 16-byte chunks hold
//        k {0-3, 8-11} and {4-7, 12-15}, the order in which the transposing read delivers a step to the two
//        half-waves; the operand is one 16-byte read.
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef bf16x8_t plane8;
typedef bf16x4_t plane4;
// Two shapes, as in the 16-bit kernel: 128 x 128 output tiles on 4 wavefronts (64 x 64 each, two or three
// workgroups per CU), and 256 x 256 on 8 wavefronts (128 (m) x 64 (n) each, one workgroup per CU), which splits every
// operand element for twice as many products and reads 3/4 of the LDS operands per matrix instruction.
template <bool LARGE>
struct ShapeS {
    static constexpr int TILE = LARGE ? 256 : 128;       // rows of an operand tile (m of A, n of B)
    static constexpr int THREADS = LARGE ? 512 : 256;
    static constexpr int BM = LARGE ? 4 : 2, BNB = 2;     // 32 x 32 blocks per wavefront along m and n
    static constexpr int RMAJ_ROWB = TILE * 2;            // bytes per k-row of an RMAJ plane
    static constexpr int PLANEB = TILE * KC * 2;          // bytes of one plane of one operand tile
    static constexpr int TILE3B = 3 * PLANEB;
};

__device__ inline int rmaj_swz(int kk) { return ((kk & 3) << 2) | ((kk >> 2) & 3); }

// ANY: bases, leading dimensions and extents are any number of elements (at least 4) and the slice is below 2 GiB: pieces
// are loads of element alignment through a buffer resource.  Past the end of a row (RM) a piece holds the next k's
// elements, which only enter rows of C that are not stored; past k (not RM) the next row's, which `trim` zeroes.  A piece
// that would end past the slice is moved back to end with it and shifted into place by `trim`.  Both happen in the last
// stage only.
// Planes do not hold values beyond bf16's largest (an Inf among them: Inf times Inf would be NaN) and lose the low bits of
// values whose last plane leaves bf16's range (below 2^-110).  ANY products keep what the Float32 instruction gives there:
// `store` notes the extremes of the tile's operands, and the kernel computes a tile that has such values again on that
// instruction.  (A NaN is a NaN in the first plane already.)
template <bool RM, bool LARGE, bool ANY>
struct OperandS {
    typedef ShapeS<LARGE> S;
    static constexpr int ROWB = S::RMAJ_ROWB, PLANEB = S::PLANEB, CPR = S::TILE / 4;   // float4 pieces per k-row
    static constexpr int OOB = 0x7fffffff;
    const float *X;
    int64_t ld, rows, k, row0;
    __amdgpu_buffer_rsrc_t rsrc;   // ANY
    int bytes;                     // ANY: of the slice
    float most = 0.0f;             // ANY: largest |x| so far (NaNs do not count)
    uint32_t least = ~0u;          // ANY: smallest 2 |x| - 1 so far, in bits (a zero counts as the largest)
    __device__ bool fit() const { return most <= 0x1.fep127f && least >= (27u << 24) - 1; }   // bf16's largest; 2^-100
    static constexpr int LDR = S::TILE + 4;             // floats per k-row of a tile kept as it is
    floatx4_t reg[2];   // TILE * KC / 4 pieces per tile: 2 per thread in either shape

    __device__ void init(const float *X_, int64_t ld_, int64_t rows_, int64_t k_, int64_t row0_) {
        X = X_;
        ld = ld_;
        rows = rows_;
        k = k_;
        row0 = row0_;
        bytes = ANY ? (int)((RM ? (k - 1) * ld + rows : (rows - 1) * ld + k) * 4) : 0;
        if (ANY) rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)X, 0, bytes, 0x00020000);
    }
    // ANY: byte offset of this thread's piece u of the stage at k0; OOB: outside the matrix
    __device__ int offset(int u, int64_t k0) const {
        const int c = threadIdx.x + S::THREADS * u;
        const int row = RM ? (c % CPR) * 4 : c >> 2, kk = RM ? c / CPR : (c & 3) * 4;
        if (row0 + row >= rows || k0 + kk >= k) return OOB;
        return (int)((RM ? (row0 + row) + (k0 + kk) * ld : (k0 + kk) + (row0 + row) * ld) * 4);
    }
    __device__ int overhang(int o) const { return o < bytes && o > bytes - 16 ? o - (bytes - 16) : 0; }
    __device__ void load(int64_t k0) {
        const int tid = threadIdx.x;
        const bool last = ANY && k0 + KC >= k;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int c = tid + S::THREADS * u;
            const floatx4_t z = {0.f, 0.f, 0.f, 0.f};
            if (ANY) {
                int o = offset(u, k0);
                if (last) o -= overhang(o);
                reg[u] = __builtin_bit_cast(floatx4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, o, 0, 0));
            } else if (RM) {
                const int kk = c / CPR, r4 = (c % CPR) * 4;
                reg[u] = (k0 + kk < k && row0 + r4 < rows) ? *(const floatx4_t *)(X + (row0 + r4) + (k0 + kk) * ld) : z;
            } else {
                const int r = c >> 2, k4 = (c & 3) * 4;       // 4 pieces per row
                reg[u] = (row0 + r < rows && k0 + k4 < k) ? *(const floatx4_t *)(X + (k0 + k4) + (row0 + r) * ld) : z;
            }
        }
    }
    __device__ void trim(int64_t k0) {
        if (!ANY || k0 + KC < k) return;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            u32x4_t v = mi_drop_bytes(__builtin_bit_cast(u32x4_t, reg[u]), overhang(offset(u, k0)));
            if (!RM) {
                const int64_t left = k - k0 - ((threadIdx.x + S::THREADS * u) & 3) * 4;
                v = mi_keep_bytes(v, left < 4 ? (left > 0 ? (int)left * 4 : 0) : 16);
            }
            reg[u] = __builtin_bit_cast(floatx4_t, v);
        }
    }
    // split into planes; `tile` is the LDS byte address of the hi plane
    __device__ void store(unsigned tile) {
        typedef __attribute__((address_space(3))) u32x2_t *lds8_t;
        const int tid = threadIdx.x;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int c = tid + S::THREADS * u;
            const floatx4_t x = reg[u];
            uint32_t pl[3][2];
            split3_pair(x[0], x[1], pl[0][0], pl[1][0], pl[2][0]);
            split3_pair(x[2], x[3], pl[0][1], pl[1][1], pl[2][1]);
            if constexpr (ANY) {
                const u32x4_t bits = __builtin_bit_cast(u32x4_t, x);
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most) : "v"(x[e]), "v"(x[e + 1]));
                    const uint32_t s0 = (bits[e] << 1) - 1, s1 = (bits[e + 1] << 1) - 1;
                    least = min(min(s0, s1), least);
                }
            } else if (mi_plane_word_special(pl[0][0]) || mi_plane_word_special(pl[0][1])) {   // an Inf, a NaN or a value beyond the bf16 range among the four (rare)
                split3_pair_wide(x[0], x[1], pl[0][0], pl[1][0], pl[2][0]);
                split3_pair_wide(x[2], x[3], pl[0][1], pl[1][1], pl[2][1]);
            }
            unsigned at;
            if (RM) {
                const int kk = c / CPR, r4 = (c % CPR) * 4;   // rows r4 .. r4+3 of k-row kk
                at = (unsigned)(kk * ROWB + ((((r4 >> 3) ^ rmaj_swz(kk)) << 4) + (r4 & 7) * 2));
            } else {
                const int r = c >> 2, k4 = (c & 3) * 4;       // k k4 .. k4+3 of row r: chunk (k4/4)%2, 8-byte slot k4/8
                at = (unsigned)(r * 32 + (((((k4 >> 2) & 1) ^ ((r >> 3) & 1)) << 4) + 8 * (k4 >> 3)));
            }
#pragma unroll
            for (int q = 0; q < 3; q++) *(lds8_t)(uintptr_t)(tile + at + q * PLANEB) = (u32x2_t){pl[q][0], pl[q][1]};
        }
    }
    // ANY: the stage as it is, [16 k][TILE rows + 4], for the Float32 instruction
    __device__ void store_whole(unsigned tile) const {
        typedef __attribute__((address_space(3))) float *ldsf_t;
        typedef __attribute__((address_space(3))) floatx4_t *ldsf4_t;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int c = threadIdx.x + S::THREADS * u;
            if (RM) {
                *(ldsf4_t)(uintptr_t)(tile + (unsigned)(((c / CPR) * LDR + (c % CPR) * 4) * 4)) = reg[u];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) *(ldsf_t)(uintptr_t)(tile + (unsigned)((((c & 3) * 4 + e) * LDR + (c >> 2)) * 4)) = reg[u][e];
            }
        }
    }
    // the three planes of the MFMA operand of the 32-row block `blk`
    __device__ static void fetch(unsigned tile, int blk, int lane, plane8 (&out)[3]) {
        const int hh = lane >> 5;
        if (RM) {
            const int vrow = 4 * hh + ((lane & 15) >> 2);
            const int vchunk = 4 * blk + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), vsub = 8 * (lane & 1);
            const unsigned lo_at = tile + (unsigned)(vrow * ROWB + vsub + ((vchunk ^ rmaj_swz(vrow)) << 4));
            const unsigned hi_at = tile + (unsigned)((vrow + 8) * ROWB + vsub + ((vchunk ^ rmaj_swz(vrow + 8)) << 4));
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t *)(uintptr_t)(lo_at + q * PLANEB));
                const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t *)(uintptr_t)(hi_at + q * PLANEB));
                out[q] = __builtin_shufflevector(__builtin_bit_cast(plane4, lo), __builtin_bit_cast(plane4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        } else {
            const int row = 32 * blk + (lane & 31);
            const unsigned at = tile + (unsigned)(row * 32 + ((hh ^ ((row >> 3) & 1)) << 4));
#pragma unroll
            for (int q = 0; q < 3; q++) out[q] = *(__attribute__((address_space(3))) const plane8 *)(uintptr_t)(at + q * PLANEB);
        }
    }
};

template <bool A_RM, bool B_RM, bool LARGE, bool ANY>
__global__ __launch_bounds__(ShapeS<LARGE>::THREADS, LARGE ? 1 : 2) void gemm32s_kernel(Gemm32Args g) {
    typedef ShapeS<LARGE> S;
    constexpr int TILE3B = S::TILE3B, BM = S::BM, BNB = S::BNB;
    extern __shared__ __attribute__((aligned(16))) unsigned char gemm_smem[];   // A and B tiles, two buffers each
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)gemm_smem;
    // tiles in an order in which those in flight on one die share operands and cut cache lines of C: a few per cent on
    // k >= 1024 with the large tiles; 333 x 517 x 77, 96 slices, with the small ones 45.3 -> 40.8 us, 384 x 512 x 80 36.4 -> 33.0
    const int64_t id = blockIdx.x + (int64_t)gridDim.x * (blockIdx.y + (int64_t)gridDim.y * blockIdx.z);
    const MiTile tile = mi_gemm_tile_order(id, gridDim.x, gridDim.y, gridDim.z);
    const int64_t bz = tile.batch;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave & 1, wn = wave >> 1;
    const int r = lane & 31, hh = lane >> 5;

    OperandS<A_RM, LARGE, ANY> a;
    OperandS<B_RM, LARGE, ANY> b;
    a.init(g.A + bz * g.sA, g.lda, g.m, g.k, tile.m * S::TILE);
    b.init(g.B + bz * g.sB, g.ldb, g.n, g.k, tile.n * S::TILE);

    typedef __attribute__((address_space(3))) uint32_t *lds_word_t;
    const lds_word_t unfit = (lds_word_t)(uintptr_t)(lds0 + 4 * TILE3B);   // ANY: the planes do not hold the tile's operands
    if (ANY && threadIdx.x == 0) *unfit = 0;
    floatx16_t acc[BNB][BM];   // [n block][m block]
#pragma unroll
    for (int i = 0; i < BNB; i++)
#pragma unroll
        for (int j = 0; j < BM; j++) acc[i][j] = (floatx16_t){0};

    // One stage of loads in flight.  Three (two more register sets) measured 0.25 against 0.19 ms on the
    // 1024 x 64 x 1024 x 128 product with the small shape: the registers cost the third workgroup per CU.
    const int nk = (int)((g.k + KC - 1) / KC);
    a.load(0);
    b.load(0);
    a.trim(0);
    b.trim(0);
    a.store(lds0);
    b.store(lds0 + 2 * TILE3B);
    __syncthreads();
    for (int it = 0; it < nk; it++) {
        const int buf = it & 1;
        if (it + 1 < nk) {
            a.load((int64_t)(it + 1) * KC);
            b.load((int64_t)(it + 1) * KC);
        }
        const unsigned at = lds0 + buf * TILE3B, bt = lds0 + (2 + buf) * TILE3B;
        plane8 av[BM][3], bv[BNB][3];
#pragma unroll
        for (int j = 0; j < BM; j++) OperandS<A_RM, LARGE, ANY>::fetch(at, BM * wm + j, lane, av[j]);
#pragma unroll
        for (int i = 0; i < BNB; i++) OperandS<B_RM, LARGE, ANY>::fetch(bt, BNB * wn + i, lane, bv[i]);
        // the transposed problem (rows = n, columns = m), small terms first
        constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, ib[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int t = 0; t < 6; t++)
#pragma unroll
            for (int i = 0; i < BNB; i++)
#pragma unroll
                for (int j = 0; j < BM; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bv[i][ib[t]], av[j][ia[t]], acc[i][j], 0, 0, 0);
        if (it + 1 < nk) {
            a.trim((int64_t)(it + 1) * KC);
            b.trim((int64_t)(it + 1) * KC);
            a.store(lds0 + (buf ^ 1) * TILE3B);
            b.store(lds0 + (2 + (buf ^ 1)) * TILE3B);
        } else if (ANY && !(a.fit() && b.fit())) {
            *unfit = 1;
        }
        __syncthreads();
    }
    if (ANY && *unfit) {   // the same word for the whole workgroup
#pragma unroll
        for (int i = 0; i < BNB; i++)
#pragma unroll
            for (int j = 0; j < BM; j++) acc[i][j] = (floatx16_t){0};
        typedef __attribute__((address_space(3))) const float *ldsf_t;
        for (int it = 0; it < nk; it++) {
            a.load((int64_t)it * KC);
            b.load((int64_t)it * KC);
            a.trim((int64_t)it * KC);
            b.trim((int64_t)it * KC);
            a.store_whole(lds0);
            b.store_whole(lds0 + 2 * TILE3B);
            __syncthreads();
#pragma unroll
            for (int ks = 0; ks < KC / 2; ks++) {
                float av[BM], bv[BNB];
                const unsigned row = (unsigned)((2 * ks + hh) * a.LDR + r);
#pragma unroll
                for (int j = 0; j < BM; j++) av[j] = *(ldsf_t)(uintptr_t)(lds0 + (row + 32 * (BM * wm + j)) * 4);
#pragma unroll
                for (int i = 0; i < BNB; i++) bv[i] = *(ldsf_t)(uintptr_t)(lds0 + 2 * TILE3B + (row + 32 * (BNB * wn + i)) * 4);
#pragma unroll
                for (int i = 0; i < BNB; i++)
#pragma unroll
                    for (int j = 0; j < BM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[i], av[j], acc[i][j], 0, 0, 0);
            }
            __syncthreads();
        }
    }

    // accumulator register v of lane (r, hh) of block (i, j): n = 32i + 8*(v/4) + 4*hh + v%4, m = 32j + r
    // A lane holds single elements of 16 columns of C: stored directly, every instruction moves 4 bytes per lane.
    // Instead each wavefront passes [32 n][64 m] blocks through a private LDS region (the operand buffers are
    // free now) and reads them back as rows of m, so that a store instruction writes four columns of 256
    // contiguous bytes, 16 bytes per lane (C is 512 MiB of the 1024 x 64 x 1024 x 128 product: 0.195 -> 0.178 ms).
    float *C = g.C + bz * g.sC;
    typedef __attribute__((address_space(3))) float *ldsf_t;
    typedef __attribute__((address_space(3))) const floatx4_t *ldsf4_t;
    constexpr int LDW = 64 + 4;   // floats per LDS row
    const unsigned region = lds0 + (unsigned)wave * (32 * LDW * 4);
    const int64_t mw = a.row0 + 32 * BM * wm, nw = b.row0 + 32 * BNB * wn;
    const auto write = [&](auto whole_c) {
        constexpr bool whole = decltype(whole_c)::value;   // columns of C are whole pieces
#pragma unroll
        for (int i = 0; i < BNB; i++)
#pragma unroll
            for (int jp = 0; jp < BM / 2; jp++) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int jj = 0; jj < 2; jj++)
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        *(ldsf_t)(uintptr_t)(region + (unsigned)(((8 * (v / 4) + 4 * hh + (v % 4)) * LDW + 32 * jj + r) * 4)) =
                            g.alpha * acc[i][2 * jp + jj][v];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int nl = 4 * q + (lane >> 4), ml = (lane & 15) * 4;
                    floatx4_t val = *(ldsf4_t)(uintptr_t)(region + (unsigned)((nl * LDW + ml) * 4));
                    const int64_t nj = nw + 32 * i + nl, mi = mw + 64 * jp + ml;
                    if (nj >= g.n || mi >= g.m) continue;
                    float *c = C + mi + nj * g.ldc;
                    if (whole || mi + 4 <= g.m) {
                        if (g.beta != 0.0f) {
                            const floatx4_t old = __builtin_bit_cast(floatx4_t, *(const mi_piece4_t *)c);
#pragma unroll
                            for (int e = 0; e < 4; e++) val[e] += g.beta * old[e];
                        }
                        *(mi_piece4_t *)c = __builtin_bit_cast(u32x4_t, val);
                    } else {
#pragma unroll
                        for (int e = 0; e < 3; e++)
                            if (mi + e < g.m) c[e] = g.beta != 0.0f ? val[e] + g.beta * c[e] : val[e];
                    }
                }
            }
    };
    // two variants: the code for the last piece of columns of odd length costs the others 1.5 %
    if ((g.m & 3) == 0) write(std::integral_constant<bool, true>());
    else write(std::integral_constant<bool, false>());
}

template <bool A_RM, bool B_RM, bool LARGE, bool ANY>
int32_t launch_planes(const Gemm32Args &g, int64_t nb, hipStream_t st) {
    typedef ShapeS<LARGE> S;
    auto kern = gemm32s_kernel<A_RM, B_RM, LARGE, ANY>;
    constexpr size_t smem = 4 * S::TILE3B + (ANY ? 16 : 0);
    static bool attr_set = false;  // per instantiation; the attribute is idempotent, so a race is harmless
    if (!attr_set) {
        MI_HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_set = true;
    }
    dim3 grid((unsigned)((g.m + S::TILE - 1) / S::TILE), (unsigned)((g.n + S::TILE - 1) / S::TILE), (unsigned)nb);
    hipLaunchKernelGGL(kern, grid, dim3(S::THREADS), smem, st, g);
    MI_LAUNCH_CHECK();
    return MI_OK;
}

template <bool LARGE, bool ANY>
int32_t launch_planes_l(const Gemm32Args &g, bool a_rm, bool b_rm, int64_t nb, hipStream_t st) {
    if (a_rm) return b_rm ? launch_planes<true, true, LARGE, ANY>(g, nb, st) : launch_planes<true, false, LARGE, ANY>(g, nb, st);
    return b_rm ? launch_planes<false, true, LARGE, ANY>(g, nb, st) : launch_planes<false, false, LARGE, ANY>(g, nb, st);
}

// the Float32 matrix instruction instead of the bf16 planes (MI355ATTN_F32_MFMA=1 in the environment, read once)
bool exact_instruction_wanted() {
    static const bool wanted = [] {
        const char *e = getenv("MI355ATTN_F32_MFMA");
        return e && e[0] == '1';
    }();
    return wanted;
}

}  // namespace

// every 16-byte piece of the operands is aligned and wholly inside or outside its matrix
static bool aligned_pieces(int transA, int transB, int64_t m, int64_t n, int64_t k, const void *A, int64_t lda, int64_t sA, const void *B,
                           int64_t ldb, int64_t sB) {
    return ((((uintptr_t)A) | ((uintptr_t)B)) & 15) == 0 && ((lda | ldb | sA | sB | (transA ? k : m) | (transB ? n : k)) & 3) == 0;
}

// true when the tiles of this file take the product.  Operands that do not come in aligned pieces need slices that 32-bit
// byte offsets address and that hold a piece, and the bf16 planes.
static bool tiles_support(int transA, int transB, int64_t m, int64_t n, int64_t k, const void *A, int64_t lda, int64_t sA, const void *B,
                          int64_t ldb, int64_t sB) {
    if (k < 1 || m * n < 64 * 64) return false;   // tiny products: the small-tile kernel wastes less
    if ((n + TN - 1) / TN > 65535) return false;
    if (aligned_pieces(transA, transB, m, n, k, A, lda, sA, B, ldb, sB)) return true;
    if (exact_instruction_wanted()) return false;
    const int64_t extA = transA ? (m - 1) * lda + k : (k - 1) * lda + m, extB = transB ? (k - 1) * ldb + n : (n - 1) * ldb + k;
    // leading dimensions of at least a piece: only the last k or row of a slice can hold a piece that ends past it
    return lda >= 4 && ldb >= 4 && extA >= 4 && extB >= 4 && extA * 4 < 2147483647LL && extB * 4 < 2147483647LL;
}
static bool waves_support(int transA, int transB, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb) {
    return k >= 1 && !exact_instruction_wanted() && gemm32_waves_supports(transA, transB, m, n, k, lda, ldb);
}

bool batched_gemm32_supports(int32_t dtype, int transA, int transB, int64_t m, int64_t n, int64_t k, const void *A, int64_t lda,
                             int64_t sA, const void *B, int64_t ldb, int64_t sB) {
    if (dtype != MI_F32) return false;
    return waves_support(transA, transB, m, n, k, lda, ldb) || tiles_support(transA, transB, m, n, k, A, lda, sA, B, ldb, sB);
}

// The large tile where the share of its slots that does useful work, counting padded rows and columns and the last round of
// workgroups (one per CU; three of the small ones), times its higher rate once k is long enough to pay for its prologue
// (2047^3 x 8: 188 against 163 TFLOP/s; 1000 x 1000 x 130: level) is the larger.
static bool large_tiles(int64_t m, int64_t n, int64_t k, int64_t nb) {
    const auto useful = [&](int64_t tile, int64_t slots) {
        const int64_t tiles = ((m + tile - 1) / tile) * ((n + tile - 1) / tile) * nb;
        return (double)(m * n * nb) / ((double)((tiles + slots - 1) / slots * slots) * (double)(tile * tile));
    };
    return m >= 256 && n >= 256 && k >= 128 && (k >= 512 ? 1.15 : 1.0) * useful(256, 256) > useful(128, 768);
}
// Microseconds on the tiles of this file, fitted like those of batched_gemm32_waves.hip (mean deviation 10 %): the chain of
// a workgroup's steps, or the steps of the fullest CU.
static double tiles_estimate(int64_t m, int64_t n, int64_t k, int64_t nb) {
    const double steps = (double)((k + KC - 1) / KC);
    const double per_cu = ceil((double)((m + TM - 1) / TM) * (double)((n + TN - 1) / TN) * (double)nb / 256.0);
    return 4.0 + fmax(1.18 * steps + 1.6, per_cu * (0.72 * steps + 2.4)) * (large_tiles(m, n, k, nb) ? 0.87 : 1.0);
}

int32_t launch_batched_gemm32(int transA, int transB, int64_t m, int64_t n, int64_t k, float alpha, const void *A, int64_t lda,
                              int64_t sA, const void *B, int64_t ldb, int64_t sB, float beta, void *C, int64_t ldc, int64_t sC,
                              int64_t batch, hipStream_t st) {
    const bool a_rm = !transA, b_rm = transB != 0;
    if (waves_support(transA, transB, m, n, k, lda, ldb) &&
        (!tiles_support(transA, transB, m, n, k, A, lda, sA, B, ldb, sB) || gemm32_waves_estimate(m, n, k, 1, batch) < tiles_estimate(m, n, k, batch)))
        return launch_gemm32_waves(transA, transB, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, 1, batch, st);
    for (int64_t b0 = 0; b0 < batch; b0 += 65535) {   // gridDim.z is limited to 65535: issue the batch in slabs
        const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
        Gemm32Args g = {(const float *)A + b0 * sA, (const float *)B + b0 * sB, (float *)C + b0 * sC,
                        m, n, k, lda, ldb, ldc, sA, sB, sC, alpha, beta};
        dim3 grid((unsigned)((m + TM - 1) / TM), (unsigned)((n + TN - 1) / TN), (unsigned)nb);
        if (exact_instruction_wanted()) {
            if (a_rm && b_rm) hipLaunchKernelGGL((gemm32_kernel<true, true>), grid, dim3(256), 0, st, g);
            else if (a_rm) hipLaunchKernelGGL((gemm32_kernel<true, false>), grid, dim3(256), 0, st, g);
            else if (b_rm) hipLaunchKernelGGL((gemm32_kernel<false, true>), grid, dim3(256), 0, st, g);
            else hipLaunchKernelGGL((gemm32_kernel<false, false>), grid, dim3(256), 0, st, g);
        } else {
            const bool large = large_tiles(m, n, k, nb);
            const bool aligned = aligned_pieces(transA, transB, m, n, k, g.A, lda, sA, g.B, ldb, sB);
            const int32_t rc = aligned ? (large ? launch_planes_l<true, false>(g, a_rm, b_rm, nb, st) : launch_planes_l<false, false>(g, a_rm, b_rm, nb, st))
                                       : (large ? launch_planes_l<true, true>(g, a_rm, b_rm, nb, st) : launch_planes_l<false, true>(g, a_rm, b_rm, nb, st));
            if (rc != MI_OK) return rc;
        }
        MI_LAUNCH_CHECK();
    }
    return MI_OK;
}

// C = alpha * sum over the batch of op(A) op(B) + beta*C: one launch that walks the slices, or a product per slice where
// these fill the chip by themselves
int32_t launch_batched_gemm32_sum(int transA, int transB, int64_t m, int64_t n, int64_t k, float alpha, const void *A, int64_t lda,
                                  int64_t sA, const void *B, int64_t ldb, int64_t sB, float beta, void *C, int64_t ldc, int64_t batch,
                                  hipStream_t st) {
    const bool tiles = tiles_support(transA, transB, m, n, k, A, lda, sA, B, ldb, sB);
    const double apart = (double)batch * fmin(gemm32_waves_estimate(m, n, k, 1, 1), tiles ? tiles_estimate(m, n, k, 1) : 1e30);
    if (batch <= 2147483647LL / ((k + 15) / 16) && waves_support(transA, transB, m, n, k, lda, ldb) && gemm32_waves_estimate(m, n, k, batch, 1) < apart)
        return launch_gemm32_waves(transA, transB, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, 0, batch, 1, st);
    for (int64_t b = 0; b < batch; b++) {
        const int32_t rc = launch_batched_gemm32(transA, transB, m, n, k, alpha, (const float *)A + b * sA, lda, sA, (const float *)B + b * sB, ldb, sB,
                                                 b == 0 ? beta : 1.0f, C, ldc, 0, 1, st);
        if (rc != MI_OK) return rc;
    }
    return MI_OK;
}
