// Split-kv attention for a single query per (head, batch) ("decode" shape, Lq = 1), bf16 / f16 / Float32; calls with
// two to four queries (no weights, a mask only if it does not depend on the query) run through the same kernels
// with that many softmax states per wavefront (template parameter NQ).
//
// The work is a stream over K and V: every byte is read once and used once, so the kernel is
// organised around HBM, not around the matrix cores.  A kv row (all heads) is E contiguous elements;
// a wavefront owns a 1 KiB segment of the row (512 16-bit features: 4 heads at D = 128, 8 heads at D = 64; half as
// many in Float32), each lane one 16-byte load (8 or 4 consecutive features), and walks kv rows eight at a time.  The
// dot product over a head is finished with a butterfly over the lanes that share the head.  A wavefront keeps an
// online-softmax state (m, l, o[8]); the eight of a workgroup, which share a segment, merge theirs through LDS and write
// one partial result to a workspace; a second small kernel merges those.
//
// What bounds it: large calls the K / V stream (8 segments x 16 x 32768 keys, 8.6 GB: 1380 us, 6.2 TB/s; 1434 with a
// partial result per wavefront and four segments of a row in a workgroup), small ones the chain of one block's loads, the two
// launches and the merge, since a call fills the chip with wavefronts of a single 8-row block where its keys allow it
// (head dim 64, 8 heads, 2 x 5000 keys: 74 -> 13 us; 12 x 18 x 528: 45 -> 14; one sequence of 4096 keys, 32 heads of 128, with
// the weights: 80 -> 22).
//
// Same arithmetic as the reference chain (src/attention.jl:112-127, fdrop = identity, no bias):
//   s_j = sum_d k[d,j] * q[d] / sqrt(D),  a = softmax_j(s),  x[d] = sum_j a_j v[d,j].
// An optional mask (src/attention.jl:133-138; with a single query every mask is a key mask, e.g. the context
// lengths of a padded batch) costs one byte per key row and head: dropped keys get the score -Inf, a (head,
// batch) pair with no key kept gives NaN like the reference.
// When the caller wants the attention weights too (the reference always returns them), the first kernel also writes
// the raw scores (Float32, 4 bytes per key and head: a few per mille of the K / V stream), the merge kernel leaves the
// final maximum and 1 / sum per (head, batch), and a third, elementwise kernel turns the scores into weights.
#include "common.h"
#include "attention_params.h"

namespace {

constexpr int ROWS = 8;        // kv rows in flight per lane and tensor
constexpr int WAVES = 8;       // wavefronts per workgroup
constexpr int MAX_SPLITS = 1024;
// features per lane (one 16-byte load) and per wavefront
template <typename T> constexpr int epl() { return 16 / (int)sizeof(typename T::type); }
template <typename T> constexpr int seg_width() { return 64 * epl<T>(); }

struct DecodeArgs {
    AttnParams p;
    float c;           // log2(e) / sqrt(D)
    int32_t nsplit;
    int32_t rows_per_wave;   // weights requested: contiguous keys of a wavefront, a multiple of ROWS
    float *scores;     // weights requested: [B][H][Lkv] raw dot products (-Inf where masked), else null
    float *final_ml;   // weights requested: [B][H][2] final maximum (raw units) and 1 / sum
};

__device__ inline void unpack8(const u32x4_t &v, float *out, BF16) {
    const bf16x8_t h = __builtin_bit_cast(bf16x8_t, v);
#pragma unroll
    for (int e = 0; e < 8; e++) out[e] = (float)h[e];
}
__device__ inline void unpack8(const u32x4_t &v, float *out, F16) {
    const f16x8_t h = __builtin_bit_cast(f16x8_t, v);
#pragma unroll
    for (int e = 0; e < 8; e++) out[e] = (float)h[e];
}
__device__ inline void unpack8(const u32x4_t &v, float *out, F32) {   // four features
    const floatx4_t h = __builtin_bit_cast(floatx4_t, v);
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = h[e];
}

// workspace layout: [B][nsplit][E] floats of o, then [B][nsplit][H] of m, then [B][nsplit][H] of l
// NQ: queries of one batch element that a wavefront carries through the stream (1, 2 or 4).  A handful of queries
// against a long context (a few speculated tokens, a short chunk) is the same stream over K and V with NQ states: every
// K / V row is read once for all of them, where the tiled kernel reads head-dim-wide pieces of it per head.
//
// The WAVES wavefronts of a workgroup share a segment and take different key rows, and their states are merged through
// LDS before they leave, so a split costs one partial result per workgroup.
template <typename T, int D, bool MASKED, bool SCORES, int NQ = 1>
__global__ __launch_bounds__(WAVES * 64, NQ <= 2 ? 4 : 2) void decode_split_kernel(DecodeArgs a) {
    const AttnParams &p = a.p;
    typedef typename T::type t;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int EPL = epl<T>(), SEG = seg_width<T>(), LPH = D / EPL;   // features per lane and wavefront, lanes per head
    constexpr int NH = SEG / D;                        // heads per wavefront
    __shared__ float sc_lds[SCORES ? WAVES * NH * 64 : 1]; // scores on their way out: [wavefront][head][64 keys]
    __shared__ float o_lds[NQ * WAVES * SEG], ml_lds[NQ * WAVES * NH * 2];   // states of the wavefronts
    const int seg = blockIdx.x;
    const int split = blockIdx.y;
    const int64_t ngroups = (p.Lq + NQ - 1) / NQ;      // groups of NQ queries per batch element
    const int64_t b = blockIdx.z / ngroups, q0 = (blockIdx.z % ngroups) * NQ;
    const int64_t f = (int64_t)seg * SEG + lane * EPL; // first feature of this lane
    const bool lane_ok = f < p.E;                      // E is a multiple of EPL (D is 64 or 128)

    const t *kb = (const t *)p.k + p.E * p.Lkv * b + (lane_ok ? f : 0);
    const t *vb = (const t *)p.v + p.E * p.Lkv * b + (lane_ok ? f : 0);
    float qf[NQ][EPL] = {};
#pragma unroll
    for (int n = 0; n < NQ; n++) {   // queries past Lq: copies of the last one, computed and not stored
        const int64_t qi = q0 + n < p.Lq ? q0 + n : p.Lq - 1;
        if (lane_ok) unpack8(*(const u32x4_t *)((const t *)p.q + p.E * (qi + p.Lq * b) + f), qf[n], T());
    }

    // Without the score output the wavefronts take the 8-row blocks of the key range in turn (block t belongs to
    // wavefront t mod nwaves of the pair) instead of one contiguous range each: the splits of a batch element run side by side, so at any
    // moment the chip reads one moving window of consecutive rows rather than nwaves separate streams (a plain read
    // of 8 GiB on this GPU: 6.97 TB/s with interleaved workgroups against 6.2-6.35 with a contiguous chunk per workgroup).
    // The online softmax does not depend on the order.  With scores the ranges stay contiguous: they leave in runs of
    // 64 consecutive keys.
    const bool interleave = !SCORES;
    const int64_t part = (int64_t)split * WAVES + wave, nwaves = (int64_t)a.nsplit * WAVES;
    const int64_t j_begin = interleave ? part * ROWS : part * a.rows_per_wave;
    int64_t j_end = interleave ? p.Lkv : j_begin + a.rows_per_wave;
    if (j_end > p.Lkv) j_end = p.Lkv;
    const int64_t j_step = interleave ? nwaves * ROWS : ROWS;

    float m[NQ], l[NQ], o[NQ][EPL] = {};
#pragma unroll
    for (int n = 0; n < NQ; n++) {
        m[n] = MI_NEG_INF;
        l[n] = 0.0f;
    }
    const u32x4_t zero = {0, 0, 0, 0};
    const float scale = p.drop_thresh != 0 ? p.drop_scale : 1.0f;
    // mask bytes of this lane's head: element (kv, 0, h, b)
    const uint8_t *mrow = MASKED ? p.mask + (lane_ok ? f / D : 0) * p.mask_strides[2] + b * p.mask_strides[3] : nullptr;

    for (int64_t j = j_begin; j < j_end; j += j_step) {
        u32x4_t kr[ROWS], vr[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const bool ok = lane_ok && j + r < j_end;
            kr[r] = ok ? *(const u32x4_t *)(kb + p.E * (j + r)) : zero;
        }
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const bool ok = lane_ok && j + r < j_end;
            vr[r] = ok ? *(const u32x4_t *)(vb + p.E * (j + r)) : zero;
        }
        bool keep[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) keep[r] = j + r < j_end && (!MASKED || mrow[(j + r) * p.mask_strides[0]] != 0);
        float s[NQ][ROWS];
        float mx[NQ];
#pragma unroll
        for (int n = 0; n < NQ; n++) mx[n] = MI_NEG_INF;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            float kf[EPL];
            unpack8(kr[r], kf, T());
#pragma unroll
            for (int n = 0; n < NQ; n++) {
                float d = 0.0f;
#pragma unroll
                for (int e = 0; e < EPL; e++) d = fmaf(kf[e], qf[n][e], d);
#pragma unroll
                for (int off = 1; off < LPH; off <<= 1) d += __shfl_xor(d, off, 64);
                s[n][r] = keep[r] ? d : MI_NEG_INF;
                mx[n] = fmaxf(mx[n], s[n][r]);
            }
        }
        float mref[NQ];
#pragma unroll
        for (int n = 0; n < NQ; n++) {
            const float mnew = fmaxf(m[n], mx[n]);
            mref[n] = mnew == MI_NEG_INF ? 0.0f : mnew;   // no score above -Inf so far (dropped keys, infinite features of k): every term below is 0
            const float resc = mi_exp2((m[n] - mref[n]) * a.c);
            m[n] = mnew;
            l[n] *= resc;
#pragma unroll
            for (int e = 0; e < EPL; e++) o[n][e] *= resc;
        }
        // fused dropout (src/attention.jl:126 with fdrop = dropout; calls without returned weights, Lkv a multiple of 4):
        // the row sum takes the weight as the softmax gives it, the value product takes it times the keep factor of
        // weight (key, query, head, batch) in the shared counter stream.  A chunk starts at a multiple of 8 keys, so it
        // is two hash groups of four; the hashes hide under the K / V stream.
        // The decisions stay a bit each until the products: as factors they would take a register each.
        uint32_t kept[NQ];
#pragma unroll
        for (int n = 0; n < NQ; n++) kept[n] = ~0u;
        if (p.drop_thresh != 0) {
            const int64_t hd = lane_ok ? f / D : 0;
#pragma unroll
            for (int n = 0; n < NQ; n++) {
                const int64_t qi = q0 + n < p.Lq ? q0 + n : p.Lq - 1;
                const uint64_t i0 = (uint64_t)(j + p.Lkv * (qi + p.Lq * (hd + p.H * b)));
                kept[n] = 0;
#pragma unroll
                for (int g = 0; g < ROWS / 4; g++) {
                    const uint64_t bits = mi_dropout_group_bits(p.drop_key, (i0 + 4 * g) >> 2);
#pragma unroll
                    for (int e = 0; e < 4; e++) kept[n] |= mi_dropout_keep_in(bits, e, p.drop_thresh) ? 1u << (4 * g + e) : 0u;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            float vf[EPL];
            unpack8(vr[r], vf, T());
#pragma unroll
            for (int n = 0; n < NQ; n++) {
                const float pr = mi_exp2((s[n][r] - mref[n]) * a.c);
                l[n] += pr;
                const float pd = pr * ((kept[n] >> r) & 1 ? scale : 0.0f);
#pragma unroll
                for (int e = 0; e < EPL; e++) o[n][e] = fmaf(pd, vf[e], o[n][e]);
            }
        }
        if (SCORES) {
            // Scores leave in runs of 64 keys per head (256 contiguous bytes): written 32 bytes at a time, one piece per
            // head and iteration, the scattered small writes cost the K / V stream a fifth of its rate.  The first lane
            // of each head parks the 8 scores of this iteration in the wavefront's LDS rows; every 8th iteration the
            // 64 lanes write one row per head.
            const int slot8 = (int)(((j - j_begin) / ROWS) & 7);
            if ((lane & (LPH - 1)) == 0) {
                float *row = sc_lds + (wave * NH + lane / LPH) * 64 + 8 * slot8;
                *(floatx4_t *)row = (floatx4_t){s[0][0], s[0][1], s[0][2], s[0][3]};
                *(floatx4_t *)(row + 4) = (floatx4_t){s[0][4], s[0][5], s[0][6], s[0][7]};
            }
            if (slot8 == 7 || j + ROWS >= j_end) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const int64_t jrun = j - 8 * slot8;     // first key of the run
#pragma unroll
                for (int hl = 0; hl < NH; hl++) {
                    const int64_t h = (int64_t)seg * NH + hl;
                    const float val = sc_lds[(wave * NH + hl) * 64 + lane];
                    if (h < p.H && jrun + lane < j_end) a.scores[((int64_t)b * p.H + h) * p.Lkv + jrun + lane] = val;
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
    }
    // merge of the wavefronts' states; one that kept no key has m = -Inf and weight 0
#pragma unroll
    for (int n = 0; n < NQ; n++) {
        float *wo = o_lds + (n * WAVES + wave) * SEG + lane * EPL;
        *(floatx4_t *)wo = (floatx4_t){o[n][0], o[n][1], o[n][2], o[n][3]};
        if constexpr (EPL == 8) *(floatx4_t *)(wo + 4) = (floatx4_t){o[n][4], o[n][5], o[n][6], o[n][7]};
        if ((lane & (LPH - 1)) == 0) {
            float *wml = ml_lds + ((n * WAVES + wave) * NH + lane / LPH) * 2;
            wml[0] = m[n];
            wml[1] = l[n];
        }
    }
    __syncthreads();
    // partial results: one slot per (batch element, query, split); the merge kernel sees B * Lq batch elements
    float *ws = (float *)p.workspace;
    const int64_t nbq = p.B * p.Lq;
    for (int i = threadIdx.x; i < NQ * SEG; i += WAVES * 64) {
        const int n = i / SEG, fl = i % SEG, hl = fl / D;
        const int64_t fo = (int64_t)seg * SEG + fl;
        if (fo >= p.E || q0 + n >= p.Lq) continue;
        float mw[WAVES], mm = MI_NEG_INF;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            mw[w] = ml_lds[((n * WAVES + w) * NH + hl) * 2];
            mm = fmaxf(mm, mw[w]);
        }
        const float mr = mm == MI_NEG_INF ? 0.0f : mm;
        float oo = 0.0f, ll = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const float wt = mi_exp2((mw[w] - mr) * a.c);
            oo = fmaf(o_lds[(n * WAVES + w) * SEG + fl], wt, oo);
            ll = fmaf(ml_lds[((n * WAVES + w) * NH + hl) * 2 + 1], wt, ll);
        }
        const int64_t slot = (b * p.Lq + q0 + n) * a.nsplit + split;
        ws[slot * p.E + fo] = oo;
        if (fl % D == 0) {
            const int64_t h = fo / D;
            float *wm = ws + nbq * a.nsplit * p.E;
            float *wl = wm + nbq * a.nsplit * p.H;
            wm[slot * p.H + h] = mm;
            wl[slot * p.H + h] = ll;
        }
    }
}

// Merge of the splits with the usual log-sum-exp rule.  One workgroup per (64 features, batch), 64 features being (half of)
// a head: the weights 2^(m_s - m) of the splits are computed once into LDS, then 16 groups of 16 threads each add up a
// sixteenth of the splits, four features a thread and eight independent loads at a time.
template <typename T>
__global__ __launch_bounds__(256) void decode_merge_kernel(DecodeArgs a) {
    const AttnParams &p = a.p;
    __shared__ float wgt[MAX_SPLITS];
    __shared__ float red[2][4];
    __shared__ floatx4_t part[4][16];
    const int64_t b = blockIdx.y;
    const int64_t f0 = (int64_t)blockIdx.x * 64, h = f0 / p.D;
    const float *ws = (const float *)p.workspace;
    const float *wm = ws + (int64_t)p.B * a.nsplit * p.E + b * a.nsplit * p.H + h;
    const float *wl = wm + (int64_t)p.B * a.nsplit * p.H;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float ms[MAX_SPLITS / 256], ls[MAX_SPLITS / 256], m = MI_NEG_INF;
#pragma unroll
    for (int u = 0; u < MAX_SPLITS / 256; u++) {
        const int s = u * 256 + threadIdx.x;
        ms[u] = s < a.nsplit ? wm[(int64_t)s * p.H] : MI_NEG_INF;
        ls[u] = s < a.nsplit ? wl[(int64_t)s * p.H] : 0.0f;
        m = fmaxf(m, ms[u]);
    }
    m = mi_wave_max(m);
    if (lane == 0) red[0][wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    float l = 0.0f;
#pragma unroll
    for (int u = 0; u < MAX_SPLITS / 256; u++) {
        const int s = u * 256 + threadIdx.x;
        if (s >= a.nsplit) break;
        const float w = mi_exp2((ms[u] - m) * a.c);   // every key of the pair dropped: NaN, as the reference's softmax gives
        wgt[s] = w;
        l = fmaf(ls[u], w, l);
    }
    l = mi_wave_sum(l);
    if (lane == 0) red[1][wave] = l;
    __syncthreads();
    const float inv = 1.0f / (red[1][0] + red[1][1] + red[1][2] + red[1][3]);
    if (a.final_ml && threadIdx.x == 0 && f0 % p.D == 0) {
        a.final_ml[(b * p.H + h) * 2] = m;
        a.final_ml[(b * p.H + h) * 2 + 1] = inv;
    }
    const int fl = threadIdx.x & 15, g = threadIdx.x >> 4;
    const float *src = ws + b * a.nsplit * p.E + f0 + fl * 4;
    floatx4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = g; s < a.nsplit; s += 16 * 8) {
        floatx4_t x[8];
        float w[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const bool ok = s + 16 * u < a.nsplit;
            x[u] = ok ? *(const floatx4_t *)(src + (int64_t)(s + 16 * u) * p.E) : (floatx4_t){0.0f, 0.0f, 0.0f, 0.0f};
            w[u] = ok ? wgt[s + 16 * u] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = fmaf(x[u][e], w[u], o[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        o[e] += __shfl_xor(o[e], 16, 64);
        o[e] += __shfl_xor(o[e], 32, 64);
    }
    if (lane < 16) part[wave][lane] = o;
    __syncthreads();
    // one element a thread: the output may start at any element
    if (threadIdx.x < 64) {
        const int pf = threadIdx.x >> 2, e = threadIdx.x & 3;
        const float sum = (part[0][pf][e] + part[1][pf][e]) + (part[2][pf][e] + part[3][pf][e]);
        ((typename T::type *)p.out)[p.E * b + f0 + threadIdx.x] = T::from_f32(sum * inv);
    }
}

// weights[kv, 0, h, b] = 2^((s - m) c) / l from the saved scores; a (head, batch) pair with every key masked has
// s = m = -Inf and gets NaN, as the reference's softmax gives
template <typename TW>
__global__ __launch_bounds__(256) void decode_weights_kernel(DecodeArgs a, TW *weights) {
    const AttnParams &p = a.p;
    const int64_t hb = blockIdx.y, j = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    const float m = a.final_ml[hb * 2], inv = a.final_ml[hb * 2 + 1];
    const float *src = a.scores + hb * p.Lkv;
    TW *dst = weights + hb * p.Lkv;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (j + e < p.Lkv) dst[j + e] = (TW)(mi_exp2((src[j + e] - m) * a.c) * inv);
}

// queries per wavefront: 1, 2, or 4 (three queries run as four)
int decode_nq(const AttnParams &p) { return p.Lq <= 1 ? 1 : p.Lq == 2 ? 2 : 4; }

// Bytes of the partial results of ns splits, then (weights requested) the raw scores and the final statistics
size_t workspace_of(const AttnParams &p, size_t ns) {
    return sizeof(float) * (ns * (size_t)(p.B * p.Lq) * (size_t)(p.E + 2 * p.H) + (p.weights ? (size_t)(p.Lkv * p.H * p.B + 2 * p.H * p.B) : 0));
}

// Share of the chip at work when every (segment, batch element, query group) has n workgroups: compute units in the last of the
// rounds of 256 workgroups, wavefronts in the last 8-row blocks.
double share_at_work(int64_t pairs, int64_t blocks, int64_t n) {
    const int64_t rounds = (pairs * n + 255) / 256, per_wave = (blocks + WAVES * n - 1) / (WAVES * n);
    return (double)(pairs * n) / (double)(256 * rounds) * (double)blocks / (double)(WAVES * n * per_wave);
}

// Workgroups along the keys of one (segment, batch element, query group).  A CU holds two workgroups of eight wavefronts with one
// or two queries and one with four (171-207 registers).  Measured, us of GPU time, one segment unless said:
//   - up to 512, down to one 8-row block per wavefront: another round with little left in it costs more than it gives
//     (head dim 128, 4 segments x 3 x 3300 keys: 26.6 with 512 workgroups, 30 with 624), more blocks per wavefront leave CUs idle
//     (2 x 5000 keys: 13.1 with one block per wavefront, 14.5 with two, 19.8 with four; one wavefront per 250 keys, as it was: 74);
//   - two to four queries: two blocks, since a workgroup's partial results are that many times larger (31041 keys, two queries:
//     23.9 with one, 20.7 with two), and from 16 blocks on one workgroup per CU (two queries, 8 segments x 8 x 8192 keys
//     192 with 256 workgroups, 211 with 512; Float32, 8 x 16 x 16384 704, 817; four queries, 16-bit 199, 205; 718, 718);
//   - a single query, 12 blocks and more for each wavefront of 256 workgroups: four blocks per wavefront, at most 8192 workgroups.  Where
//     the batch elements are powers of two apart, few long wavefronts run in step on the same channels (head dim 64, 16-bit, 4 segments x
//     8 x 16384 keys 219 with 512 workgroups, 197 with 2048, 188 with one result per wavefront as it was; 4 x 16 x 8192 220, 185, 185; Float32, head
//     dim 128, 8 x 16 x 16384 765, 708 with 8192, 722); elsewhere it costs up to 2 % (15 x 5 x 20000 109, 111).  With the weights requested
//     four rounds of 512 (8 segments x 16 x 32768 keys 1524, as it was 1597), which cost two to four queries, with more to merge, up to a
//     sixth (four queries, 8 segments x 8 x 8192 keys: 211, 222, 247);
//   - more pairs than CUs, or two to four queries and a number of them that fills no round: the fewest that keep 0.88 (0.8) of the
//     chip at work, or the best of 16.  With one
//     workgroup per pair a few CUs have two of them and the others wait (2 segments x 140 pairs, a single query, keys: 600 80.7 with one / 66.7
//     with ten, two queries 1000 147 / 114; 2 x 130 x 4096 539 / 413 with eight; 2 x 270 x 600, a single query 136 / 124 with five), or some
//     have none (three queries, Float32, 2 x 88 x 8192 645 with one / 520 with four).  At most 8192 partial rows of a segment: 16 MiB of workspace.
// With the weights requested the 256 keys per workgroup keep the partial results to what a call needed with one per split.
int pick_nsplit(const AttnParams &p) {
    const int64_t SEG = p.dtype == MI_F32 ? seg_width<F32>() : seg_width<BF16>();
    const int64_t nseg = (p.E + SEG - 1) / SEG;
    const int64_t pairs = nseg * p.B * ((p.Lq + decode_nq(p) - 1) / decode_nq(p));   // (segment, batch element, query group)
    const int64_t blocks = p.weights ? 4 : p.Lq == 1 ? 1 : 2;   // 8-row blocks per wavefront, at least
    const int64_t maxs = (p.Lkv + ROWS * WAVES * blocks - 1) / (ROWS * WAVES * blocks);
    const int64_t all = (p.Lkv + ROWS - 1) / ROWS;
    int64_t want = pairs < 512 ? 512 / pairs : 1;
    const bool long_range = p.Lkv >= (p.Lq == 1 ? 32 : 16) * ROWS * WAVES * want;
    if (p.Lq == 1 && p.weights && long_range) {
        want = pairs < 2048 ? 2048 / pairs : 1;
    } else if (p.Lq == 1 && !p.weights && p.Lkv >= 1024 && pairs * all >= 12 * WAVES * 256) {
        want = (all + WAVES * 4 - 1) / (WAVES * 4);
        if (want * pairs > 8192) want = pairs < 8192 ? 8192 / pairs : 1;
    } else if (pairs > 256 || (p.Lq > 1 && long_range)) {
        const int64_t first = pairs > 256 ? 1 : 256 / pairs;
        const double enough = pairs > 256 ? 0.88 : 0.8;
        double best = 0.0;
        for (int64_t n = first; n <= maxs && (n == first || (n <= 16 && n * pairs * decode_nq(p) <= 8192)) && best < enough; n++) {
            // scores that the built-in workspace holds beside one workgroup's results stay in it
            if (n > first && p.weights && workspace_of(p, (size_t)n) > MI_ATTN_STATIC_WORKSPACE_BYTES && workspace_of(p, (size_t)first) <= MI_ATTN_STATIC_WORKSPACE_BYTES) break;
            const double share = share_at_work(pairs, all, n);
            if (share > best) {
                best = share;
                want = n;
            }
        }
    }
    if (want > maxs) want = maxs;
    if (want > MAX_SPLITS) want = MAX_SPLITS;
    return (int)want;
}

}  // namespace

bool attention_decode_supports(const AttnParams &p) {
    if (p.Lq < 1 || p.Lq > 4 || p.bias || p.causal || !p.out || p.stats) return false;   // saved statistics: the tiled kernels write them
    if (p.drop_thresh && (p.weights || (p.Lkv & 3) != 0)) return false;   // fused dropout: in the streaming kernel only, whole hash groups
    // two to four queries: without the weights, and with a mask only when it does not depend on the query
    if (p.Lq > 1 && (p.weights || (p.mask && p.mask_strides[1] != 0) || p.B * p.Lq > 65535)) return false;
    if (p.weights && p.H * p.B > 65535) return false;
    if (p.D != p.Dv || (p.D != 64 && p.D != 128)) return false;
    if (p.Lkv < 512) return false;   // short contexts: the tiled kernel is fine
    if (p.B > 65535) return false;
    auto al = [](const void *x) { return (((uintptr_t)x) & 15) == 0; };
    return al(p.q) && al(p.k) && al(p.v);
}

size_t attention_decode_workspace(const AttnParams &p) {
    return workspace_of(p, (size_t)pick_nsplit(p));
}

int32_t launch_attention_decode(const AttnParams &p, hipStream_t st) {
    DecodeArgs a;
    a.p = p;
    a.c = MI_LOG2E / sqrtf((float)p.D);
    a.nsplit = pick_nsplit(p);
    const int64_t per_wave = (p.Lkv + (int64_t)a.nsplit * WAVES - 1) / ((int64_t)a.nsplit * WAVES);
    a.rows_per_wave = (int32_t)((per_wave + ROWS - 1) / ROWS * ROWS);
    const int64_t SEG = p.dtype == MI_F32 ? seg_width<F32>() : seg_width<BF16>();
    if ((((uintptr_t)p.workspace) & 15) != 0)
        return mi_set_error(MI_EWORKSPACE, "decode workspace must be 16-byte aligned");
    a.scores = a.final_ml = nullptr;
    if (p.weights) {
        a.scores = (float *)p.workspace + (size_t)a.nsplit * (size_t)p.B * (size_t)(p.E + 2 * p.H);
        a.final_ml = a.scores + p.Lkv * p.H * p.B;
    }
    const int nq = decode_nq(p);
    dim3 grid((unsigned)((p.E + SEG - 1) / SEG), (unsigned)a.nsplit, (unsigned)(p.B * ((p.Lq + nq - 1) / nq)));
    dim3 mgrid((unsigned)(p.E / 64), (unsigned)(p.B * p.Lq));
    DecodeArgs am = a;      // the merge kernel takes every (batch element, query) pair for a batch element of its own:
    am.p.B = p.B * p.Lq;    // q and the output are (E, Lq, B) arrays, the partial results [B * Lq][split][...]
    am.p.Lq = 1;
#define DECODE_LAUNCH(TT, DD)                                                                                        \
    {                                                                                                                \
        if (p.weights) {                                                                                             \
            if (p.mask) hipLaunchKernelGGL((decode_split_kernel<TT, DD, true, true>), grid, dim3(WAVES * 64), 0, st, a);     \
            else hipLaunchKernelGGL((decode_split_kernel<TT, DD, false, true>), grid, dim3(WAVES * 64), 0, st, a);           \
        } else if (nq == 1) {                                                                                        \
            if (p.mask) hipLaunchKernelGGL((decode_split_kernel<TT, DD, true, false>), grid, dim3(WAVES * 64), 0, st, a);    \
            else hipLaunchKernelGGL((decode_split_kernel<TT, DD, false, false>), grid, dim3(WAVES * 64), 0, st, a);          \
        } else if (nq == 2) {                                                                                        \
            if (p.mask) hipLaunchKernelGGL((decode_split_kernel<TT, DD, true, false, 2>), grid, dim3(WAVES * 64), 0, st, a); \
            else hipLaunchKernelGGL((decode_split_kernel<TT, DD, false, false, 2>), grid, dim3(WAVES * 64), 0, st, a);       \
        } else {                                                                                                     \
            if (p.mask) hipLaunchKernelGGL((decode_split_kernel<TT, DD, true, false, 4>), grid, dim3(WAVES * 64), 0, st, a); \
            else hipLaunchKernelGGL((decode_split_kernel<TT, DD, false, false, 4>), grid, dim3(WAVES * 64), 0, st, a);       \
        }                                                                                                            \
    }
    if (p.dtype == MI_BF16) {
        if (p.D == 128) DECODE_LAUNCH(BF16, 128) else DECODE_LAUNCH(BF16, 64)
        MI_LAUNCH_CHECK();
        hipLaunchKernelGGL(decode_merge_kernel<BF16>, mgrid, dim3(256), 0, st, am);
    } else if (p.dtype == MI_F32) {
        if (p.D == 128) DECODE_LAUNCH(F32, 128) else DECODE_LAUNCH(F32, 64)
        MI_LAUNCH_CHECK();
        hipLaunchKernelGGL(decode_merge_kernel<F32>, mgrid, dim3(256), 0, st, am);
    } else {
        if (p.D == 128) DECODE_LAUNCH(F16, 128) else DECODE_LAUNCH(F16, 64)
        MI_LAUNCH_CHECK();
        hipLaunchKernelGGL(decode_merge_kernel<F16>, mgrid, dim3(256), 0, st, am);
    }
#undef DECODE_LAUNCH
    MI_LAUNCH_CHECK();
    if (p.weights) {
        dim3 wgrid((unsigned)((p.Lkv + 1023) / 1024), (unsigned)(p.H * p.B));
        if (p.weights_dtype == MI_F32) hipLaunchKernelGGL(decode_weights_kernel<float>, wgrid, dim3(256), 0, st, a, (float *)p.weights);
        else if (p.dtype == MI_BF16) hipLaunchKernelGGL(decode_weights_kernel<__bf16>, wgrid, dim3(256), 0, st, a, (__bf16 *)p.weights);
        else hipLaunchKernelGGL(decode_weights_kernel<_Float16>, wgrid, dim3(256), 0, st, a, (_Float16 *)p.weights);
        MI_LAUNCH_CHECK();
    }
    return MI_OK;
}
