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
constexpr uint32_t kMinDepth = 256;       // a chunk for each of four waves
constexpr uint32_t kMaxDepth = 16384;     // a wave's FP32 chain is at most 2048 long, as far as errors are measured

// Times below: this kernel -> the FP32 tile kernels it replaces.
inline Shape choose(uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldb, bool trans_a, bool trans_b) {
    Shape t;
    if (std::max(lda, ldb) >= kMaxLd || k < kMinDepth || k > kMaxDepth) return t;
    t.x_is_a = n <= m;
    const uint32_t rows = t.x_is_a ? m : n, cols = t.x_is_a ? n : m;
    if (cols > kMaxCols || rows < kMinRows) return t;
    // One work-group streams at most about 25 GB/s, and few rows are few
    // work-groups, where the tile kernels can cut K; more columns cost both
    // operands' loads: 1163 x 15 x 6199 21.5 us against 18.9, 2304 x 16 x 5824
    // 22.5 against 21.3, 5706 x 16 x 5501 39.3 against 38.5, 4927 x 14 x
    // 4911 25.4 against 24.8; but 1152 x 2 x 5248 13.3 against 16.9, 4096 x 16 x 4096 14.4 against 15.7.
    if (k >= 5632 && rows < 2048) return t;
    if (cols > 8 && ((k >= 4096 && rows < 2048) || (k >= 4608 && rows < 6144))) return t;
    const bool xkc = t.x_is_a ? trans_a : !trans_b, ykc = t.x_is_a ? !trans_b : trans_a;
    // a long K, X read along it, and a round and a half of the chip
    // (12769 x 14 x 5989 92.4 us against 83.3, 9001 x 16 x 8001 94.4 against
    // 86.0; but 16384 x 16 x 8192 115.3 against 145.4, 9000 x 7 x 7001 66.8
    // against 68.6)
    if (xkc && cols > 8 && k >= 5120 && rows > 8192 && rows < 16384) return t;
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
    // Short K: fewer waves, so that each has a chunk or two and more groups
    // share a CU (16384 x 16 x 512 TN 8.2 us with 4, 10.3 with 8); long K and
    // wide tiles: 16, a whole CU, if that leaves one round (10176 x 10 x 7616
    // 61.6 against 64.7 with 8; 11211 x 9 x 7659 TN, 351 groups, 112 with 16).
    const uint32_t groups = (rows + 16u * (uint32_t)t.x_atoms - 1) / (16u * (uint32_t)t.x_atoms);
    t.waves = k < 1024 && (xkc || t.x_atoms == 1) ? 4 : (k >= 2048 && t.x_atoms > 1 && groups <= 256u ? 16 : 8);
    t.on = true;
    return t;
}

}  // namespace thin
