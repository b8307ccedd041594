// Sizes that the gradient kernel of short sequences takes (attention_backward_pair16.inc): plain arithmetic, shared by the
// rule that sends calls there (attention_backward_flash16.hip) and by the launch.
#pragma once
#include <cstddef>
#include <cstdint>

constexpr int PAIR_SMALL = 128;                        // keys up to which its tiles are 32 queries, not 64
constexpr size_t PAIR_LDS_MOST = 160 * 1024;           // a compute unit's LDS
constexpr int PAIR_ROWS = 32 * 128;                    // bytes of 32 rows of Q, dO or K (64 features of 16 bits)
constexpr int PAIR_DS = 32 * 64;                       // bytes of a dS block: 32 keys x 32 queries

// LDS: K rows, two Q and dO tiles, two sets of dS blocks, three floats per query; words: a keep bit per weight
inline size_t pair_kernel_lds(int64_t Lq, int64_t Lkv, bool words) {
    const size_t waves = (size_t)((Lkv + 31) / 32), QT = Lkv <= PAIR_SMALL ? 1 : 2, tiles = (size_t)((Lq + 32 * (int64_t)QT - 1) / (32 * (int64_t)QT));
    return waves * (PAIR_ROWS + 2 * QT * PAIR_DS) + 4 * QT * PAIR_ROWS + 12 * tiles * 32 * QT + (words ? waves * 32 * 8 * ((tiles * QT + 1) / 2) : 0);
}

// Up to 256 keys (eight wavefronts).  The tiles of queries are one chain on a wavefront per 32 keys: not many more queries than
// keys (16 x 16 pairs of 1000 x 77: 77 us against 68), and more than 256 only where the pairs fill the chip (500 x 200: 41
// against 60).  With keep words the largest of these need more LDS than there is (720 x 255: 161 KiB).
inline bool pair_kernel_sizes(int64_t Lq, int64_t Lkv, int64_t pairs, bool words) {
    return Lkv <= 256 && (Lq <= 3 * Lkv || Lq <= 64) && (Lq <= 256 || pairs >= 256) && pair_kernel_lds(Lq, Lkv, words) <= PAIR_LDS_MOST;
}
