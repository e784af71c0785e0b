// gemm_shape.h -- which tile a product takes and how k is cut, as plain C++
// (gemm.hip; compiled for the host alone by the tests).  Extents go up to
// 2^31 - 1, so every sum of one and a tile or chunk is formed in 64 bits.
#pragma once

#include <cmath>
#include <cstdint>
#include <initializer_list>

namespace ember {

constexpr int64_t ceil_div(int64_t a, int64_t b) { return a / b + (a % b != 0); }

// The three tiles, and what a launch with each costs: the 16-k steps of the
// busiest CU, at the time one takes with the chip nearly empty (light_us: the
// chain of waits of one tile) and full (full_us: throughput, and the clock
// the power limit leaves), plus a launch's fixed cost.  Fitted to measured
// times of 17 shapes with every tile and 1 to 8 splits (4096^3 down to
// 17 x 33 x 5): the choice by this cost is the fastest of the measured ones
// for 16 of them, 6 % off for one.  full_us as throughput: 256 x 256 tiles
// 228 TFLOP/s at 4096^3 (128 x 128: 188), 128 x 128 181 TFLOP/s at
// 8192 x 1024 x 1024 (64 x 64: 133, 256 x 256: 154); light_us: 12 products of
// 197 x 333 x 250 11 us with 64 x 64, 17 with 128 x 128, 45 with 256 x 256.
struct GemmShape {
    int tm, tn, per_cu;
    double full_us, light_us, fixed_us;
};
constexpr GemmShape kGemmShapes[3] = {
    {256, 256, 1, 2.3, 1.75, 6.5}, {128, 128, 1, 0.73, 0.55, 4.5}, {64, 64, 3, 0.285, 0.36, 3.5}};
constexpr int64_t kSplitBytes = int64_t(1) << 29;  // most scratch that splitting k may take

// A grid holds fewer than 2^32 threads in x, which thin outputs of more than
// 2^30 rows or columns pass: the rest goes in further launches.
constexpr int64_t kTilesPerLaunch = int64_t(1) << 22;

// k per split for `want` splits, a multiple of every tile's slab.
inline int64_t split_chunk(int64_t k, int want) { return ceil_div(ceil_div(k, want), 32) * 32; }

// The cheapest tile and number of k splits (1: k whole; else splits of
// split_chunk(k, want) each, the last one shorter).
struct GemmChoice {
    int shape, ksplit;
    int64_t kchunk;
};

inline GemmChoice choose_gemm(int64_t n, int64_t m, int64_t k, int64_t batch, int ncu)
{
    const double cus = ncu, total = (double)batch * n * m;
    GemmChoice choice = {2, 1, k};
    double best = INFINITY;
    for (int s = 0; s < 3; ++s) {
        const GemmShape &p = kGemmShapes[s];
        const double tiles = (double)ceil_div(n, p.tm) * ceil_div(m, p.tn) * batch;
        for (int want : {1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32, 48, 64}) {
            if (want > 1 && (k / want < 64 || 4 * want * total > kSplitBytes)) break;
            // The 256 x 256 tile sums all six part products together, the
            // others keep the small ones apart and err a third as much: it
            // splits k only as often as fills the chip, with short sums.
            if (s == 0 && want > 1 && (want + 1) * tiles <= cus) continue;
            const int64_t chunk = want > 1 ? split_chunk(k, want) : k;
            const int splits = want > 1 ? (int)ceil_div(k, chunk) : 1;
            const double work = tiles * splits, rounds = std::ceil(work / cus), steps = (double)ceil_div(chunk, 16);
            const double step_us = p.per_cu > 1
                                       ? std::fmax(p.light_us, p.full_us * rounds)
                                       : rounds * (p.light_us + (p.full_us - p.light_us) * std::fmin(1.0, work / cus));
            double us = p.fixed_us + steps * step_us;
            if (splits > 1) us += 3.0 + (2 * splits + 1) * 4 * total / 5e6;  // the reduction's launch and bytes
            if (us < best) {
                best = us;
                choice = {s, splits, chunk};
            }
        }
    }
    return choice;
}

// The part of k that split z walks, and its slabs of `slab` k: the first takes
// what the others, which are whole, leave over.
struct KRange {
    int beg, end, slabs, first;
};
constexpr KRange k_range(int k, int kchunk, int z, int slab)
{
    const int64_t beg = (int64_t)z * kchunk;
    const int len = (int)(k - beg < kchunk ? k - beg : kchunk);
    const int slabs = (int)ceil_div(len, slab);
    return {(int)beg, (int)(beg + len), slabs, len - (slabs - 1) * slab};
}

}  // namespace ember
