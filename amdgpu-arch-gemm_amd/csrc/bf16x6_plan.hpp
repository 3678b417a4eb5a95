// When, and in which tile and K split, sgemm_launch runs the split-BF16
// kernels of sgemm_bf16x6.hip instead of the handle's FP32 ones: a time model of
// both, fitted to back-to-back launches of 216 shapes on an MI355X (the package's
// workloads, cubes from 512 to 6144, thin, tall, deep, shallow and ragged shapes in
// all four layouts, C read or not).  Over 220 other shapes drawn from the same
// ranges its times are within 5-8% rms of the measured ones (K splits the most;
// FP32 kernels 12%), and the 155 that it gives to the split kernels run at
// 1.25 times the FP32 kernels' speed (geometric mean).  Launches with pauses
// between them start on a faster clock and take up to a fifth less time than it
// says.  Host only; no HIP.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace bf16x6 {

constexpr int kStep = 16;                       // k values of one MFMA
constexpr uint64_t kMaxPartialBytes = 32u << 20;  // of a K split: the static scratch of sgemm_launch_noalloc,
constexpr uint64_t kMaxTickets = 16384;           // so that both entry points run the same plan
constexpr uint32_t kMaxSplits = 16;
constexpr uint32_t kMinRange = 128;             // k values of one range, at least
// Leading dimensions below this keep one tile's span of every operand below
// 2^31 bytes (256 rows or columns of 4 bytes).
constexpr uint32_t kMaxLd = 1u << 21;
// k values per accumulator chain, at most: as far as the errors of every sign
// pattern are measured (0.36 of the FP32 kernels' at 24500)
constexpr uint64_t kMaxChain = 24576;

// One kernel: its tile, the K waves of a work-group (chains per range) and its
// times in microseconds: a launch, a step of 16 in a sparse and in a full round
// of work-groups (there the power limit sets the clock), the same where A is
// read along k (a factor), a work-group's prologue and epilogue, and per MB of
// a full round's tiles their stores, their C and a split's partials.
struct Tile {
    int m, n, k_waves;
    double launch, step_few, step_full, trans_a, fixed, store, read_c, partial;
};
constexpr Tile kTiles[] = {
    {128, 128, 2, 2.68, 0.484, 0.678, 1.0, 5.18, 4.0, 34.0, 9.01},
    {128, 64, 4, 2.07, 0.307, 0.399, 1.0, 4.34, 0.0, 31.6, 12.9},
    {256, 128, 1, 3.81, 0.898, 1.25, 1.015, 4.78, 9.9, 34.5, 8.79},
};
constexpr int kTileCount = (int)(sizeof(kTiles) / sizeof(kTiles[0]));
constexpr double kBytesPerUs = 4.5e6;           // operands and D through HBM
// the split-BF16 kernels must be predicted this much faster
constexpr double kMargin = 0.93;
// Below this depth a launch is mostly its prologue and stores: ragged shapes
// of K = 64 .. 128 ran at 0.7 to 1.1 of the FP32 kernels' speed.
constexpr uint32_t kMinDepth = 144;
// below this many FLOPs no measured shape gained
constexpr double kMinFlops = 2.0e9;

inline uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// Microseconds of an m x n x k launch on `t` with `splits` K ranges over `cus` compute units.
inline double time_us(const Tile& t, uint32_t splits, uint64_t m, uint64_t n, uint64_t k, bool trans_a, bool reads_c,
                      int cus) {
    const uint64_t groups = ceil_div(m, (uint64_t)t.m) * ceil_div(n, (uint64_t)t.n) * splits;
    const double steps = (double)ceil_div(ceil_div(k, kStep), splits) * (trans_a ? t.trans_a : 1.0);
    const uint64_t full = groups / (uint64_t)cus;
    const double part = (double)(groups % (uint64_t)cus) / cus;
    const double mb = t.m * t.n * 4e-6;
    auto round = [&](double fill) {
        return steps * std::max(t.step_few, t.step_full * fill) + t.fixed +
               mb * fill / splits * (t.store + (reads_c ? t.read_c : 0.0));
    };
    double us = t.launch + (double)full * round(1.0) + (part > 0.0 ? round(part) : 0.0);
    if (splits > 1) us += t.partial * (2 + splits) * mb;
    // near ties go to the launch without a workspace, which a handle's first
    // split launch allocates, and to few ranges, where the model is closer
    if (splits > 1) us *= splits > 4 ? 1.04 : 1.02;
    const double bytes = 4.0 * ((double)m * k + (double)k * n + (double)m * n * (reads_c ? 2 : 1));
    return std::max(us, bytes / kBytesPerUs + t.launch);
}

struct Choice {
    int tile = -1;   // index into kTiles, -1: none
    uint32_t splits = 1;
    double us = 0.0;
    size_t partial_bytes = 0, ticket_count = 0;
};

// The fastest predicted tile and split count whose partials fit the static
// scratch and whose sums run in at least `chains` chains per output (as many
// as the FP32 launch's K ranges: a shorter chain rounds less).
inline Choice choose(uint64_t m, uint64_t n, uint64_t k, bool trans_a, bool reads_c, int cus, uint32_t chains) {
    Choice best;
    for (int i = 0; i < kTileCount; ++i) {
        const Tile& t = kTiles[i];
        const uint64_t tiles = ceil_div(m, (uint64_t)t.m) * ceil_div(n, (uint64_t)t.n);
        for (uint32_t s = 1; s <= kMaxSplits; ++s) {
            const uint64_t bytes = s > 1 ? tiles * s * (uint64_t)t.m * (uint64_t)t.n * 4u : 0u;
            if (s > 1 && (bytes > kMaxPartialBytes || tiles > kMaxTickets || k / s < kMinRange ||
                          tiles * s > 4u * (uint64_t)cus))
                break;
            if (s * (uint32_t)t.k_waves < chains || k > kMaxChain * s * (uint64_t)t.k_waves) continue;
            const double us = time_us(t, s, m, n, k, trans_a, reads_c, cus);
            if (best.tile < 0 || us < best.us) {
                best.tile = i;
                best.splits = s;
                best.us = us;
                best.partial_bytes = (size_t)bytes;
                best.ticket_count = s > 1 ? (size_t)tiles : 0;
            }
        }
    }
    return best;
}

// Microseconds of an FP32 launch: `groups` work-groups (tiles x K ranges) of a
// tile_m x tile_n tile and `range` k values over `cus` compute units; a
// stream-K launch has no partial round.
inline double fp32_time_us(uint64_t tile_m, uint64_t tile_n, uint64_t groups, uint64_t range, uint32_t splits,
                           bool stream_k, uint64_t m, uint64_t n, uint64_t k, bool reads_c, int cus) {
    const double area = (double)tile_m * tile_n;
    const double rounds = stream_k ? (double)groups / cus : (double)ceil_div(groups, (uint64_t)cus);
    double us = 3.48 + rounds * (2.0 * area * range / 614e3 / 0.883 + (reads_c ? 2.38 : 1.57) * area / 8192);
    if (splits > 1) us += 0.519 * splits;
    const double bytes = 4.0 * ((double)m * k + (double)k * n + (double)m * n * (reads_c ? 2 : 1));
    return std::max(us, bytes / kBytesPerUs + 3.48);
}

// a launch of the FP32 edge kernel over a thin strip
inline double strip_time_us(uint64_t m, uint64_t n, uint64_t k) {
    return 8.0 + 4.0 * ((double)m * k + (double)k * n + (double)m * n) / kBytesPerUs;
}

}  // namespace bf16x6
