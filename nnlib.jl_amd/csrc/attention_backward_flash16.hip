// MFMA attention backward for bf16/f16 inputs: eligibility, workspace size and dispatch to the
// per-(dtype, head dim) instantiations of attention_backward_flash16.inc.
#include "common.h"
#include "attention_params.h"
#include "flash_common.h"
#include "attention_pair_rule.h"

int32_t launch_bwd_flash16_bf16_d32(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_bf16_d64(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_bf16_d96(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_bf16_d128(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_f16_d32(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_f16_d64(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_f16_d96(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_f16_d128(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_bf16_d256(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_flash16_f16_d256(const AttnBwdParams &, hipStream_t);

// dQ, dK and dV of a (head, batch) pair in one workgroup (attention_backward_pair16.inc)
int32_t launch_bwd_pair16_bf16(const AttnBwdParams &, hipStream_t);
int32_t launch_bwd_pair16_f16(const AttnBwdParams &, hipStream_t);

static inline bool aligned16(const void *p) { return (((uintptr_t)p) & 15) == 0; }

bool attention_bwd_flash16_supports(const AttnBwdParams &bp) {
    const AttnParams &p = bp.p;
    if (p.dtype != MI_F16 && p.dtype != MI_BF16) return false;
    // one head dim for q, k and v: a multiple of 8 (16-byte chunks) up to the 256-wide tiles
    if (p.D != p.Dv || p.D < 8 || p.D > 256 || (p.D & 7)) return false;
    // the kernels need the forward result (for delta) and take no weight cotangent
    if (!p.out || bp.dweights) return false;
    if (!aligned16(p.q) || !aligned16(p.k) || !aligned16(p.v) || !aligned16(p.out) || !aligned16(bp.dout)) return false;
    if ((bp.dq && !aligned16(bp.dq)) || (bp.dk && !aligned16(bp.dk)) || (bp.dv && !aligned16(bp.dv))) return false;
    // tiles are fetched with 32-bit byte offsets from the (batch, head) slice
    if (p.Lq * p.E * 2 >= 2147483647LL || p.Lkv * p.E * 2 >= 2147483647LL) return false;
    const int64_t tiles = (p.Lq + 127) / 128 > (p.Lkv + 127) / 128 ? (p.Lq + 127) / 128 : (p.Lkv + 127) / 128;
    return tiles * p.H * p.B <= 2147483647LL;
}

// ---- dense masks packed into bits for the key-stationary kernels ----------------------------------------------
// A dense mask without bias keeps the lean gradient kernels (raw scores, two wavefronts per SIMD).  The dQ kernel
// stages the mask tiles through LDS as the forward kernel does; in the dK / dV kernels a lane owns one key and walks
// the queries, so it wants the mask of (its key, the 64 queries of a tile) as one 64-bit word: a small kernel packs
// those words once per call, [slice][query tile][key], slices being the distinct (head, batch) planes of the mask.
static bool takes_mask_bits(const AttnParams &p) {
    if (!p.mask || p.bias || p.D > 128 || flash_is_query_independent_mask(p) || (p.Lkv & 3) != 0) return false;
    FlashArgs a;
    a.p = p;
    a.p.weights = nullptr;
    flash_fill_vec_flags(a);
    return a.mask_lds != 0;   // the dQ kernel's staged mask tiles: unit key stride, 16-byte aligned rows
}
static int64_t mask_bits_slices(const AttnParams &p) { return (p.mask_strides[2] ? p.H : 1) * (p.mask_strides[3] ? p.B : 1); }
static int64_t mask_bits_lkv_pad(const AttnParams &p) { return (p.Lkv + 255) / 256 * 256; }

static size_t mask_bits_bytes(const AttnParams &p) {
    if (!takes_mask_bits(p)) return 0;
    return sizeof(uint64_t) * (size_t)(mask_bits_slices(p) * ((p.Lq + 63) / 64) * mask_bits_lkv_pad(p));
}

__global__ __launch_bounds__(256) void mask_bits_kernel(const uint8_t *mask, int64_t s0, int64_t s1, int64_t s2, int64_t s3, int64_t Lq,
                                                        int64_t Lkv, int64_t lkv_pad, int64_t heads, uint64_t *out) {
    const int64_t kv = (int64_t)blockIdx.x * 256 + threadIdx.x, qt = blockIdx.y, slice = blockIdx.z;
    const int64_t h = slice % heads, b = slice / heads;   // heads == 1: the mask is shared by the heads (stride 0)
    uint64_t word = 0;
    if (kv < Lkv) {
        const uint8_t *col = mask + kv * s0 + h * s2 + b * s3;
#pragma unroll 8
        for (int i = 0; i < 64; i++) {
            const int64_t q = qt * 64 + i;
            if (q < Lq && col[q * s1]) word |= (uint64_t)1 << i;
        }
    }
    out[(slice * gridDim.y + qt) * lkv_pad + kv] = word;
}

// Key-padding masks: the (head, batch) pairs are classified on the device and the pairs whose mask is a context
// length run the unmasked kernels on that many keys (workgroups past it only write zeros).
static size_t lengths_bytes(const AttnParams &p) {
    if (!flash_is_query_independent_mask(p) || p.H * p.B > 2147483647LL / 4) return 0;
    if (flash_is_key_mask(p) && p.Lkv <= 128) return 0;   // short sequences: less is saved than the classification costs
    return ((size_t)(p.H * p.B) * sizeof(int32_t) + 15) & ~(size_t)15;
}

// ---- short sequences: one workgroup per (head, batch) pair --------------------------------------------------------------
// Head dims up to 64, all three gradients wanted, saved statistics, no mask that depends on the query.  Dropout at rows that do
// not start on a hash group takes the decisions from words.
static bool pair_kernel_fits(const AttnBwdParams &bp) {
    const AttnParams &p = bp.p;
    return bp.have_stats && bp.dq && bp.dk && bp.dv && p.D <= 64 && (!p.mask || flash_is_key_mask(p)) && !(p.bias && p.drop_thresh) &&
           pair_kernel_sizes(p.Lq, p.Lkv, p.H * p.B, p.drop_thresh && (p.Lkv & 3) != 0);
}

// ---- fused dropout: the keep decisions drawn once ---------------------------------------------------------------
// A keep decision costs a 64-bit hash per four weights (about 175 issue cycles a wavefront instruction: 64-bit products at a
// quarter of the rate), and each of the
// three gradient kernels needs every decision.  This kernel draws them once, any L_kv: a wavefront takes a block of 64
// queries x 64 keys, a lane hashes the 16 or (rows that do not start on a group of four) 17 groups of its query's row,
// and the 64 x 64 bits are transposed between the lanes for the kernels whose lanes hold a key.  Bound by the hashes; the
// decisions are taken from a hash two at a time, and blocks past a context length are not drawn (24 x 12 pairs of 333 x 333
// 17.3 -> 15.8 us, with a key-padding mask 19.6 -> 15.1; 32 pairs of 2000 x 2000 44.6 -> 38.7).  (Gradient of 24 x 12
// pairs of 333 x 333, head dim 64,
// p = 0.1: 296 -> 114 us, with a key-padding mask 436 -> 114; 332 x 332: 123 -> 112; 64 pairs of 2048 x 2048, head dim
// 128: 705 -> 659.)
// Redrawn (DROP_REDRAW) where that is faster, rows on hash groups given: causal calls, whose kernels visit half the blocks
// (16 x 4 pairs of 4096 x 4096, head dim 128: 1518 us with words, 1458 redrawn; 64 pairs of 2048 x 2048: 436 / 413), and
// calls of less than 2^24 weights, bound by their launches (8 x 4 pairs of 512 x 512, head dim 64: 48 / 42; 128 x 128: 40 / 34).
// Two bits a weight are O(L^2) bytes where the rest of the call is O(L): the words of as many (head, batch) pairs as
// DROP_WORDS_MOST bytes hold are drawn at a time, and the gradient kernels run on those pairs before the next are drawn.  A
// pair whose own words are more than that (65536 x 65536 is 1 GiB) has them redrawn by the kernels.
static bool takes_drop_words(const AttnBwdParams &bp, bool lengths) {
    const AttnParams &p = bp.p;
    if (p.drop_thresh == 0 || p.bias) return false;
    if (pair_kernel_fits(bp)) return (p.Lkv & 3) != 0;   // meets every decision once
    if ((p.Lkv & 3) == 0 && (p.causal || p.H * p.B * p.Lq * p.Lkv < (1 << 24))) return false;
    return !p.mask || flash_is_key_mask(p) || lengths || takes_mask_bits(p);   // what the lean kernels take
}
static int64_t pad128(int64_t n) { return (n + 127) / 128 * 128; }
constexpr size_t DROP_WORDS_MOST = (size_t)1 << 30;
// per pair
static size_t drop_rows_words(const AttnParams &p) { return (size_t)((p.Lkv + 63) / 64 * pad128(p.Lq)); }
static size_t drop_keys_words(const AttnParams &p) { return (size_t)((p.Lq + 63) / 64 * pad128(p.Lkv)); }

__global__ __launch_bounds__(256) void drop_words_kernel(AttnParams p, int64_t pair0, int64_t nkt, int64_t nqt, int64_t lq_pad, int64_t lkv_pad,
                                                         int64_t blocks, uint64_t *rows, uint64_t *keys, const int32_t *lens) {
    const uint32_t id = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), per = (uint32_t)(nkt * nqt);   // `blocks` is at most 2^20
    if (id >= blocks) return;
    const int lane = threadIdx.x & 63;
    const int64_t kt = id % (uint32_t)nkt, qt = id / (uint32_t)nkt % (uint32_t)nqt, pair = id / per;   // of this piece: b * H + h - pair0
    if (p.causal && 64 * kt > 64 * qt + 63) return;   // no kernel visits a tile above the diagonal
    if (lens && lens[pair0 + pair] != 0 && 64 * kt >= lens[pair0 + pair]) return;   // nor one past a context length
    const int64_t qi = 64 * qt + lane;
    const uint64_t first = (uint64_t)(p.Lkv * (qi + p.Lq * (pair0 + pair)) + 64 * kt);   // linear index of the row's first weight
    const int off = (int)(first & 3);
    // four decisions of a group as bits 0 to 3: in 16-bit lanes, u -sat (thresh - 1) is not zero iff u >= thresh (thresh >= 1);
    // in assembly, since the compiler turns the builtins into compares, whose lane masks cost wait states and selects
    const uint32_t below = (p.drop_thresh - 1) * 0x10001u, ones = 0x10001u;
    uint64_t z = p.drop_key + (first >> 2) * 0x9E3779B97F4A7C15ull;
    const auto group = [&]() -> uint32_t {
        const uint64_t bits = mi_mix64(z);
        z += 0x9E3779B97F4A7C15ull;
        const auto kept = [&](uint32_t w) {
            uint32_t d;
            asm("v_pk_sub_u16 %0, %1, %2 clamp\n\tv_pk_min_u16 %0, %0, %3" : "=&v"(d) : "v"(w), "v"(below), "v"(ones));
            return d;
        };
        const uint32_t t = kept((uint32_t)bits) | kept((uint32_t)(bits >> 32)) << 2;   // bits 0, 16, 2, 18
        return (t | t >> 15) & 15u;
    };
    uint32_t half[2] = {0, 0};
#pragma unroll
    for (int g = 0; g < 16; g++) half[g >> 3] |= group() << (4 * (g & 7));
    uint64_t word = (uint64_t)half[1] << 32 | half[0];
    if (p.Lkv & 3) word = word >> off | ((uint64_t)group() << 1) << (63 - off);   // the row starts `off` decisions into its first group
    if (rows) rows[(pair * nkt + kt) * lq_pad + qi] = word;
    // transpose: bit k of lane i becomes bit i of lane k; first the halves, then within 32 x 32
    uint32_t lo = (uint32_t)word, hi = (uint32_t)(word >> 32);
    mi_pair_halves(lo, hi);   // lo of lanes 32-63 <-> hi of lanes 0-31
#pragma unroll
    for (int d = 16; d > 0; d >>= 1) {
        const uint32_t m = d == 16 ? 0x0000ffffu : d == 8 ? 0x00ff00ffu : d == 4 ? 0x0f0f0f0fu : d == 2 ? 0x33333333u : 0x55555555u;
        const uint32_t plo = __shfl_xor(lo, d, 64), phi = __shfl_xor(hi, d, 64);
        const bool upper = lane & d;
        lo = upper ? (lo & ~m) | ((plo & ~m) >> d) : (lo & m) | ((plo & m) << d);
        hi = upper ? (hi & ~m) | ((phi & ~m) >> d) : (hi & m) | ((phi & m) << d);
    }
    keys[(pair * nqt + qt) * lkv_pad + 64 * kt + lane] = (uint64_t)hi << 32 | lo;
}

// ---- a bias shared by the batch elements, laid out once for the kernels ------------------------------------------
// Each batch element's workgroups read the same bias.  One small kernel writes two copies in the order the accumulators hold
// the scores, so that a lane of the dQ (dK, dV) kernel reads its 16 entries of a block as 32 contiguous bytes, whatever the
// alignment of the bias rows, and the kernels stay lean (two wavefronts per SIMD).
// Calls of few scores: the dQ kernel's atomics cost less than the two launches more that the copies and the kernel of the
// bias gradient are, as long as its chain of tiles with atomics is short (training steps, bf16, us, dQ kernel / apart; bias rows
// staged through LDS: 8 x 4 pairs of 128 x 128 43 / 49, 32 x 8 48 / 57, 16 x 8 of 96 x 160 48 / 49; 2 x 4 of 200 x 200 58 / 51,
// 4 x 4 of 512 x 128 63 / 52, of 128 x 512 70 / 58, 2 x 2 of 512 x 512 95 / 70; unaligned rows: 12 x 4 of 61 x 61 44 / 48,
// 4 x 8 of 77 x 77 49 / 49, 8 x 4 of 99 x 99 53 / 49, 8 x 2 of 81 x 81 at head dim 128 59 / 52).  Whole tiles of up to 256 once
// there are enough pairs that the bias gradient's two products count (8 x 8 of 256 x 256 61 / 65, 4 x 8 58 / 56, 2 x 4 58 / 51;
// head dim 128 78 / 87 and 74 / 66).
static bool bias_gradient_in_dq(const AttnParams &p) {
    FlashArgs a;
    a.p = p;
    a.p.weights = nullptr;
    flash_fill_vec_flags(a);
    const bool whole = p.Lq % 128 == 0 && p.Lkv % 64 == 0;
    const int64_t scores = p.H * p.B * p.Lq * p.Lkv, longest = p.Lq > p.Lkv ? p.Lq : p.Lkv;
    if (!a.bias_lds || p.D > 128) return scores <= 3 << 17 && (longest <= 80 || p.D > 128);
    return scores <= (whole ? 1 << 22 : 1 << 21) && (longest <= 160 || (whole && longest <= 256 && scores > 1 << 21));
}
static bool takes_bias_blocks(const AttnBwdParams &bp) {
    const AttnParams &p = bp.p;
    if (p.bias && bias_gradient_in_dq(p)) return false;
    // entries of their own per key, query and head: what the kernel of the bias gradient takes too
    return p.bias && !p.mask && p.drop_thresh == 0 && bp.have_stats && p.D <= 128 && p.B > 1 && p.bias_strides[3] == 0 &&
           p.bias_strides[0] == 1 && (p.bias_strides[1] != 0 || p.Lq == 1) && (p.bias_strides[2] != 0 || p.H == 1) &&
           pad128(p.Lq) / 128 * (pad128(p.Lkv) / 64) * p.H <= 2147483647LL / 16;
}
static size_t bias_copy_entries(const AttnParams &p) { return (size_t)(p.H * pad128(p.Lq) * pad128(p.Lkv)); }

// A wavefront copies 64 of the (query, key) rows of one form: grid.y 0 rows (a block of 32 keys per query, read four keys at
// a time), 1 keys (a block of 32 queries per key, neighbouring lanes reading neighbouring keys).
typedef uint32_t u32x2_any2_t __attribute__((ext_vector_type(2), aligned(2)));
__global__ __launch_bounds__(256) void bias_blocks_kernel(AttnParams p, int64_t lq_pad, int64_t lkv_pad, uint16_t *rows, uint16_t *keys) {
    const bool by_key = blockIdx.y != 0;
    const int64_t own_len = by_key ? lkv_pad : lq_pad, blocks = (by_key ? lq_pad : lkv_pad) / 32;
    const int lane = threadIdx.x & 63;
    for (int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); item < p.H * blocks * (own_len / 32); item += 4 * (int64_t)gridDim.x) {
        // 64 lanes: rows form 32 queries x 2 halves of a block, so that a query's 64 bytes are read and written together; keys
        // form 64 keys of one half
        const int64_t per = own_len / 32, part = item % per, blk = item / per % blocks, h = item / (per * blocks);
        const int hh = by_key ? (int)(part & 1) : lane & 1;
        const int64_t own = by_key ? 64 * (part >> 1) + lane : 32 * part + (lane >> 1);
        const uint16_t *src = (const uint16_t *)p.bias + h * p.bias_strides[2];
        uint32_t out[8];
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int64_t first = 32 * blk + 8 * g + 4 * hh;
            uint32_t x[4] = {0, 0, 0, 0};
            if (!by_key && own < p.Lq && first + 4 <= p.Lkv) {   // four keys at any alignment
                const u32x2_any2_t v = *(const u32x2_any2_t *)(src + own * p.bias_strides[1] + first);
                out[2 * g] = v[0];
                out[2 * g + 1] = v[1];
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int64_t q = by_key ? first + e : own, kv = by_key ? own : first + e;
                if (q < p.Lq && kv < p.Lkv) x[e] = src[q * p.bias_strides[1] + kv];
            }
            out[2 * g] = x[0] | x[1] << 16;
            out[2 * g + 1] = x[2] | x[3] << 16;
        }
        u32x4_t *dst = (u32x4_t *)((by_key ? keys : rows) + ((h * blocks + blk) * own_len + own) * 32 + 16 * hh);
        dst[0] = (u32x4_t){out[0], out[1], out[2], out[3]};
        dst[1] = (u32x4_t){out[4], out[5], out[6], out[7]};
    }
}

// ---- dQ kernel split over the keys ---------------------------------------------------------------------------
// The dQ kernel has one workgroup per (query tile, head, batch): cross-attention with few queries and many keys
// leaves most of the chip idle (32 workgroups for 128 queries, 16 heads, 2 batch elements).  With saved statistics
// every key piece is independent, so the key range is cut like the forward kernel's and the Float32 partial sums are
// added up by dq_merge_kernel.
int attention_bwd_flash16_dq_nsplit(const AttnBwdParams &bp) {
    const AttnParams &p = bp.p;
    if (!bp.have_stats || !bp.dq || p.causal) return 1;
    const int64_t wgs = ((p.Lq + 127) / 128) * p.H * p.B;
    if (wgs >= 256 || p.Lkv < 2048) return 1;
    int64_t n = (512 + wgs - 1) / wgs;
    if (n > p.Lkv / 512) n = p.Lkv / 512;
    if (n > 32) n = 32;
    return n < 2 ? 1 : (int)n;
}
size_t attention_bwd_flash16_dq_partial_bytes(const AttnBwdParams &bp) {
    const int n = attention_bwd_flash16_dq_nsplit(bp);
    return n > 1 ? sizeof(float) * (size_t)n * (size_t)(bp.p.B * bp.p.Lq * bp.p.E) : 0;
}

template <typename T>
__global__ __launch_bounds__(256) void dq_merge_kernel(const float *ws, typename T::type *dq, int nsplit, int64_t n) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;   // E is a multiple of 8: whole groups of 4
    if (i >= n) return;
    floatx4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = 0; s < nsplit; s++) {
        const floatx4_t v = *(const floatx4_t *)(ws + (int64_t)s * n + i);
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] += v[e];
    }
    typename T::vec4 r;
#pragma unroll
    for (int e = 0; e < 4; e++) r[e] = T::from_f32(acc[e]);
    *(typename T::vec4 *)(dq + i) = r;
}

// ---- the workspace -------------------------------------------------------------------------------------------------
// [statistics][packed mask bits | context lengths][partial sums of dQ][keep words | bias copies].  The last part only saves
// time, as the context lengths do for a mask that also runs without them: a call whose workspace has no room for it (a
// gradient with saved statistics and dropout or a shared bias may be given none at all) runs without, see
// DROP_REDRAW and launch_extras in attention_backward_flash16.inc.
struct BwdScratch {
    size_t stats = 0, bits = 0, lengths = 0, partial = 0, words = 0, bias = 0;   // bytes of each part, 0: not taken
    int64_t word_pairs = 0;                                                      // pairs that `words` holds
    size_t total() const { return stats + bits + lengths + partial + words + bias; }
};
static BwdScratch plan_scratch(const AttnBwdParams &bp, size_t room) {
    const AttnParams &p = bp.p;
    BwdScratch s;
    s.stats = bp.have_stats ? 0 : attention_stats_bytes(p);
    s.bits = mask_bits_bytes(p);
    s.partial = attention_bwd_flash16_dq_partial_bytes(bp);
    s.lengths = lengths_bytes(p);
    const auto left = [&] { return s.total() < room ? room - s.total() : (size_t)0; };
    if (takes_drop_words(bp, s.lengths != 0)) {
        const size_t pair = sizeof(uint64_t) * (drop_rows_words(p) + drop_keys_words(p));
        const size_t pairs = (left() < DROP_WORDS_MOST ? left() : DROP_WORDS_MOST) / pair;
        s.word_pairs = pairs < (size_t)(p.H * p.B) ? (int64_t)pairs : p.H * p.B;
        s.words = pair * (size_t)s.word_pairs;
    }
    // the one kind of call that has lengths only along with words: its kernels without mask code cannot redraw
    if (p.drop_thresh && (p.Lkv & 3) != 0 && !s.words) s.lengths = 0;
    if (takes_bias_blocks(bp)) {
        const size_t n = 2 * sizeof(uint16_t) * bias_copy_entries(p);
        if (n <= left()) s.bias = n;
    }
    return s;
}
size_t attention_bwd_flash16_workspace_needed(const AttnBwdParams &bp) { return plan_scratch(bp, 0).total(); }
size_t attention_bwd_flash16_workspace_wanted(const AttnBwdParams &bp) { return plan_scratch(bp, SIZE_MAX).total(); }

int32_t launch_attention_bwd_flash16(const AttnBwdParams &bp_in, hipStream_t st) {
    AttnBwdParams bp = bp_in;
    const AttnParams &p = bp.p;
    const BwdScratch scratch = plan_scratch(bp, bp.workspace_bytes);
    char *at = (char *)bp.workspace + scratch.stats;   // statistics that are not the caller's come first (validate_bwd)
    bp.dq_nsplit = attention_bwd_flash16_dq_nsplit(bp);
    bp.dbias_in_dq = p.bias && bias_gradient_in_dq(p);
    if (scratch.bits) {
        const int64_t nqt = (p.Lq + 63) / 64, pad = mask_bits_lkv_pad(p), slices = mask_bits_slices(p);
        if (nqt > 65535 || slices > 65535) return mi_set_error(MI_ESHAPE, "attention gradient: mask packing supports at most 65535 query tiles and mask planes");
        uint64_t *bits = (uint64_t *)at;
        const int64_t heads = p.mask_strides[2] ? p.H : 1;
        hipLaunchKernelGGL(mask_bits_kernel, dim3((unsigned)(pad / 256), (unsigned)nqt, (unsigned)slices), dim3(256), 0, st, p.mask,
                           p.mask_strides[0], p.mask_strides[1], p.mask_strides[2], p.mask_strides[3], p.Lq, p.Lkv, pad, heads, bits);
        MI_LAUNCH_CHECK();
        bp.mask_bits = bits;
        bp.mb_h = p.mask_strides[2] ? 1 : 0;
        bp.mb_b = p.mask_strides[3] ? heads : 0;
        bp.mb_lkv_pad = pad;
        bp.mb_nqt = nqt;
        at += scratch.bits;
    }
    if (scratch.lengths) {
        const int32_t rc = launch_key_mask_lengths(p, (int32_t *)at, st);
        if (rc != MI_OK) return rc;
        bp.kv_len = (int32_t *)at;
        at += scratch.lengths;
    }
    if (scratch.partial) {
        bp.dq_partial = (float *)at;
        at += scratch.partial;
    }
    if (scratch.bias) {
        const int64_t lq_pad = pad128(p.Lq), lkv_pad = pad128(p.Lkv), groups = (int64_t)bias_copy_entries(p) / 4096;   // four wavefronts each
        uint16_t *rows = (uint16_t *)at, *keys = rows + bias_copy_entries(p);
        hipLaunchKernelGGL(bias_blocks_kernel, dim3((unsigned)(groups < 8192 ? groups : 8192), 2), dim3(256), 0, st, p, lq_pad, lkv_pad, rows, keys);
        MI_LAUNCH_CHECK();
        bp.bias_rows = rows;
        bp.bias_keys = keys;
    }
    const int64_t pairs = p.H * p.B, step = scratch.words ? scratch.word_pairs : pairs;
    for (int64_t pair0 = 0; pair0 < pairs; pair0 += step) {   // one piece, unless the keep words of all pairs do not fit
        bp.pair0 = (int32_t)pair0;
        bp.npairs = (int32_t)(pairs - pair0 < step ? pairs - pair0 : step);
        if (scratch.words) {
            uint64_t *rows = (uint64_t *)at, *keys = rows + drop_rows_words(p) * (size_t)step;
            const int64_t nkt = (p.Lkv + 63) / 64, nqt = (p.Lq + 63) / 64, blocks = nkt * nqt * bp.npairs;   // at most 2^20 (DROP_WORDS_MOST)
            hipLaunchKernelGGL(drop_words_kernel, dim3((unsigned)((blocks + 3) / 4)), dim3(256), 0, st, p, pair0, nkt, nqt, pad128(p.Lq),
                               pad128(p.Lkv), blocks, pair_kernel_fits(bp) ? nullptr : rows, keys, bp.kv_len);   // the pair kernel's lanes hold keys
            MI_LAUNCH_CHECK();
            bp.drop_rows = rows;
            bp.drop_keys = keys;
        }
        int32_t rc;
        // a bias only from its copies, whose calls have a kernel of their own for its gradient; dropout at rows that do not
        // start on a hash group only from words
        const bool pair = pair_kernel_fits(bp) && (p.bias ? bp.bias_keys != nullptr : !p.drop_thresh || bp.drop_keys || (p.Lkv & 3) == 0);
        if (pair) {
            rc = p.dtype == MI_BF16 ? launch_bwd_pair16_bf16(bp, st) : launch_bwd_pair16_f16(bp, st);
            if (rc != MI_OK) return rc;
            if (!bp.dbias) continue;
            bp.dbias_only = 1;
        }
        if (p.dtype == MI_BF16)
            rc = p.D <= 32 ? launch_bwd_flash16_bf16_d32(bp, st)
                 : p.D <= 64 ? launch_bwd_flash16_bf16_d64(bp, st) : p.D <= 96 ? launch_bwd_flash16_bf16_d96(bp, st) : p.D <= 128 ? launch_bwd_flash16_bf16_d128(bp, st) : launch_bwd_flash16_bf16_d256(bp, st);
        else
            rc = p.D <= 32 ? launch_bwd_flash16_f16_d32(bp, st)
                 : p.D <= 64 ? launch_bwd_flash16_f16_d64(bp, st) : p.D <= 96 ? launch_bwd_flash16_f16_d96(bp, st) : p.D <= 128 ? launch_bwd_flash16_f16_d128(bp, st) : launch_bwd_flash16_f16_d256(bp, st);
        if (rc != MI_OK) return rc;
    }
    if (bp.dq_nsplit <= 1) return MI_OK;
    return launch_dq_merge(p.dtype, bp.dq_partial, bp.dq, bp.dq_nsplit, p.B * p.Lq * p.E, st);
}

int32_t launch_dq_merge(int32_t dtype, const float *partial, void *dq, int nsplit, int64_t n, hipStream_t st) {
    const dim3 grid((unsigned)((n / 4 + 255) / 256));
    if (dtype == MI_BF16) hipLaunchKernelGGL(dq_merge_kernel<BF16>, grid, dim3(256), 0, st, partial, (__bf16 *)dq, nsplit, n);
    else if (dtype == MI_F16) hipLaunchKernelGGL(dq_merge_kernel<F16>, grid, dim3(256), 0, st, partial, (_Float16 *)dq, nsplit, n);
    else hipLaunchKernelGGL(dq_merge_kernel<F32>, grid, dim3(256), 0, st, partial, (float *)dq, nsplit, n);
    MI_LAUNCH_CHECK();
    return MI_OK;
}
