// When sgemm_launch runs the thin kernel (sgemm_thin.hip), and in which shape.
// Host only; no HIP.
#pragma once

#include <algorithm>
#include <cstdint>

namespace thin {

struct Shape {
    bool on = false;
    bool x_is_a = false;   // the large operand is op(A) (n thin), else op(B) (m thin)
    int x_atoms = 0, waves = 0;   // 16 * x_atoms of its rows to a work-group
};

// one 16-wide atom; with a second one 1280 x 30 x 832 took 5.4 us against 4.7,
// 10176 x 26 x 1344 24.0 against 19.7
constexpr uint32_t kMaxCols = 16;
constexpr uint32_t kMaxLd = 1u << 21;     // 64 rows or 64 k of it are a 32-bit byte offset
constexpr uint32_t kMinRows = 1024;       // 64 work-groups
constexpr uint32_t kMaxRows = 1u << 27;   // 2^23 work-groups of 256: a grid holds fewer than 2^32 work-items
constexpr uint32_t kMinDepth = 256;       // a chunk for each of four waves
constexpr uint32_t kMaxDepth = 16384;     // a wave's FP32 chain is at most 2048 long, as far as errors are measured

// Microseconds of a launch with n thin and one or two atoms to a work-group: one
// work-group streams at the same rate whether its CU has one or two, so a
// launch takes as long as its rounds of one work-group per CU (4096 x 16 x 4608
// TN 18.8 us, 5000 rows 35.2, 6100 rows 35.3).  Fitted to 430 launches; 8% rms.
inline double time_us(uint32_t rows, uint32_t cols, uint32_t k, bool xkc, bool ykc, int x_atoms, int cus) {
    const uint32_t groups = (rows + 16u * (uint32_t)x_atoms - 1) / (16u * (uint32_t)x_atoms);
    const uint32_t rounds = (groups + (uint32_t)cus - 1) / (uint32_t)cus;
    double per_k = xkc ? (!ykc ? 2.45e-3 : x_atoms == 2 ? 5.2e-3 : 3.0e-3) : (ykc ? 3.0e-3 : x_atoms == 2 ? 4.5e-3 : 2.75e-3);
    if (cols <= 8) per_k *= 0.82;
    if (xkc && ykc && x_atoms == 1 && k % 512u == 0) per_k *= 1.22;   // rows a multiple of 2 KB apart meet in few channels
    if ((double)rows * k * 4e-6 > 256.0) per_k *= rounds < 3 ? 1.25 : 1.18;   // past the last-level cache
    return 2.5 + rounds * per_k * k;
}
// the same call on the tile kernels (6% rms)
inline double tile_time_us(uint32_t rows, uint32_t k) {
    return std::max(7.2 + (double)rows * k * 4e-6 / 4.0, 10.0 + 1.3e-3 * k);
}

// Times below: this kernel -> the FP32 tile kernels it replaces.  `cus`: compute units.
inline Shape choose(uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldb, bool trans_a, bool trans_b, int cus = 256) {
    Shape t;
    if (std::max(lda, ldb) >= kMaxLd || k < kMinDepth || k > kMaxDepth) return t;
    t.x_is_a = n <= m;
    const uint32_t rows = t.x_is_a ? m : n, cols = t.x_is_a ? n : m;
    if (cols > kMaxCols || rows < kMinRows || rows > kMaxRows) return t;
    const bool xkc = t.x_is_a ? trans_a : !trans_b, ykc = t.x_is_a ? !trans_b : trans_a;
    // Wider tiles read Y less often, narrower ones make more work-groups.  X
    // contiguous in k: two atoms gain with many rows and a Y that is read in
    // float4s along k (7296 x 12 x 5184 29.5 us against 36.0 with one, 2816 x
    // 15 x 5760 33.0 against 22.3; Y along the rows: 11456 x 2 x 4992 47.5
    // against 38.6).  X contiguous in its rows: 4 atoms from 128 work-groups of
    // them on (10176 x 10 x 7616 61.6 against 86.6 with one, 80.0 with two; 8200 x
    // 12 x 4000 29.0 against 35.6; 7000 x 12 x 4000 28.5 against 25.9); 2 before
    // that where Y is read along its rows (4864 x 1 x 2432 13.9 against 14.7).
    if (xkc) t.x_atoms = ykc && rows >= 6144 ? 2 : 1;
    else t.x_atoms = rows > 8192 ? 4 : (!ykc && rows >= 4800 ? 2 : 1);
    if (t.x_is_a && t.x_atoms < 4) {
        // Within the model's error the thin kernel is kept: over the 430 launches
        // the choice is within 0.5% of always knowing the faster (a last round
        // mostly empty: 5000 x 16 x 4096 TN 30.9 us against 26.3; few rows, which
        // leave CUs idle that the tile kernels fill by cutting K: 1152 x 16 x 8192
        // 30.3 against 20.3; but 10000 x 10 x 8192 TT 77.8 against 95.2).
        if (time_us(rows, cols, k, xkc, ykc, t.x_atoms, cus) >= 1.06 * tile_time_us(rows, k)) return t;
    } else if (!t.x_is_a) {
        // m thin: the tile kernels are slower (12 x 16385 x 6000 TN 181 us -> 111), so
        // only few rows with a long K (12 x 1500 x 10000 TT 28.8 against 24.0) and a
        // second round mostly empty (12 x 10000 x 10000 TN 124 against 110) stay there.
        const uint32_t groups = (rows + 16u * (uint32_t)t.x_atoms - 1) / (16u * (uint32_t)t.x_atoms);
        if (rows < 2048 && k >= 5632) return t;
        if (xkc && ykc && k > 8192 && groups > (uint32_t)cus && groups < 7u * (uint32_t)cus / 5u) return t;
    }
    // Short K: fewer waves, so that each has a chunk or two and more groups
    // share a CU (16384 x 16 x 512 TN 8.2 us with 4, 10.3 with 8); long K and
    // wide tiles: 16, a whole CU, if that leaves one round (10176 x 10 x 7616
    // 61.6 against 64.7 with 8; 11211 x 9 x 7659 TN, 351 groups, 112 with 16).
    const uint32_t groups = (rows + 16u * (uint32_t)t.x_atoms - 1) / (16u * (uint32_t)t.x_atoms);
    t.waves = k < 1024 && (xkc || t.x_atoms == 1) ? 4 : (k >= 2048 && t.x_atoms > 1 && groups <= (uint32_t)cus ? 16 : 8);
    t.on = true;
    return t;
}

}  // namespace thin
