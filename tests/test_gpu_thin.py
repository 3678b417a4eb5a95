"""The thin kernel (csrc/sgemm_thin.hip: m or n at most 16) through the public
launch path, against float64 and against the same handle's tile kernels."""
import os
import subprocess

import numpy as np
import pytest

from test_gpu_split_bf16 import _device, _handles, _matrix, _rel
from shim import sgemm_shim as S

# (m, n, k, layout, pad, shift, alpha, beta): every layout with n and with m thin,
# 1, 2 and 4 atoms of rows, 4, 8 and 16 waves, whole and ragged rows, columns
# and chunks of k, chunks for some of the waves only, odd leading dimensions
# and pointers `shift` floats past a 16-byte boundary
CASES = [
    (1024, 16, 256, "nn", 0, 0, 1.0, 0.0),
    (1025, 1, 257, "tn", 0, 1, 1.0, 0.0),
    (1, 1039, 319, "nt", 1, 0, 0.5, 1.0),
    (15, 2047, 1023, "tn", 0, 3, 1.0, -1.5),
    (2000, 7, 1024, "tt", 3, 2, -2.0, 0.75),
    (4801, 3, 2049, "nt", 1, 1, 1.0, 0.0),
    (6145, 16, 2111, "tn", 0, 0, 1.0, 1.0),
    (16, 6151, 2048, "tn", 2, 1, 0.75, 0.0),
    (9, 4900, 700, "tt", 1, 0, 1.0, 1.0),
    (2, 4805, 2050, "nt", 0, 0, 1.0, 0.0),
    (8193, 5, 1500, "nt", 1, 3, 1.0, -1.0),
    (12289, 13, 2100, "nn", 0, 0, 1.0, 0.0),
    (4, 12291, 999, "tt", 1, 1, 1.0, 0.5),
    (7, 2050, 16384, "nn", 0, 0, 1.0, 0.0),
    (2048, 8, 16384, "nn", 0, 0, 1.0, 0.0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,layout,pad,shift,alpha,beta", CASES)
def test_thin_launch(kernels, m, n, k, layout, pad, shift, alpha, beta):
    print(f"thin {m}x{n}x{k} {layout} pad {pad} shift {shift}", flush=True)
    ta, tb = layout[0] == "t", layout[1] == "t"
    ra, ca = (k, m) if ta else (m, k)
    rb, cb = (n, k) if tb else (k, n)
    Af, A = _matrix(ra, ca, ra + pad, 61, 0, S.SGEMM_DIST_NORMAL)
    Bf, B = _matrix(rb, cb, rb + 2 * pad, 61, 1, S.SGEMM_DIST_UNIFORM)
    Cf, C = _matrix(m, n, m + pad, 61, 2, S.SGEMM_DIST_UNIFORM)
    opA, opB = (A.T if ta else A), (B.T if tb else B)
    # a row of the large operand with a NaN and one with an Inf spoil their own results only
    large = opA if n <= m else opB.T
    large[17, k // 2], large[large.shape[0] - 1, k - 1] = np.nan, np.inf
    (_a, dA), (_b, dB), (_c, dC) = (_device(x, shift) for x in (Af, Bf, Cf))
    ldd = m + 3 * pad
    ref = alpha * (opA.astype(np.float64) @ opB.astype(np.float64))
    mag = abs(alpha) * (abs(opA).astype(np.float64) @ abs(opB).astype(np.float64))
    if beta:
        ref += beta * C.astype(np.float64)
        mag += abs(beta * C.astype(np.float64))
    kern, edges = _handles(m, n, k, layout)
    ld = dict(lda=ra + pad, ldb=rb + 2 * pad, ldc=m + pad, ldd=ldd)
    outs = {}
    try:
        for what, mode, entry in (("thin", 1, "launch"), ("again", 1, "launch"), ("noalloc", 1, "launch_noalloc"),
                                  ("tile", 0, "launch")):
            kern.set_split_bf16(mode)
            _d, dD = _device(np.full((ldd, n), 9.5, dtype=np.float32), shift)
            getattr(kern, entry)(dA, dB, dC, dD, m, n, k, alpha=alpha, beta=beta, **ld)
            kern.synchronize()
            full = dD.download().reshape(n, ldd).T
            assert np.all(full[m:, :] == 9.5), "rows past m of D were written"
            outs[what] = full[:m, :].copy()
    finally:
        kern.close()
        for e in edges:
            e.close()
    assert np.array_equal(outs["thin"], outs["again"], equal_nan=True), "repeated launches differ"
    assert np.array_equal(outs["thin"], outs["noalloc"], equal_nan=True), "launch_noalloc differs"
    assert not np.array_equal(outs["thin"], outs["tile"], equal_nan=True), "the thin kernel did not run"
    finite = np.isfinite(ref)
    assert np.array_equal(finite, np.isfinite(outs["thin"]))
    # any order of k FP32 products and sums, alpha's and C's roundings after it
    bound = (k + 3) * 2.0 ** -24 * mag + 2.0 ** -149
    with np.errstate(invalid="ignore"):
        assert np.all((abs(outs["thin"] - ref) <= bound)[finite])
    err, tile = (_rel(np.where(finite, outs[w], 0), np.where(finite, ref, 0)) for w in ("thin", "tile"))
    print(f"  relative error {err:.3e}, tile kernels {tile:.3e}", flush=True)
    # shorter chains than the tile kernels'; 2-norms of m * n >= 1025 random
    # errors are within 1 / sqrt(2 m n) = 2.2%, five of those for their ratio
    assert err <= 1.11 * tile


PLAN = r"""
#include "thin_plan.hpp"
#include <cmath>
#include <random>
int main() {
    std::mt19937 rng(5);
    auto size = [&](double lo, double hi) { return (uint32_t)std::lround(std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi))(rng))); };
    int seen[5] = {0}, off = 0;
    for (int i = 0; i < 200000; ++i) {
        const uint32_t rows = size(500, 3e6), cols = size(1, 40), k = size(100, 40000);
        const bool ta = i & 1, tb = i & 2, a = i & 4;
        const uint32_t m = a ? rows : cols, n = a ? cols : rows, lda = ta ? k : m, ldb = tb ? n : k;
        const thin::Shape t = thin::choose(m, n, k, lda, ldb, ta, tb);
        if (!t.on) { ++off; continue; }
        const bool xkc = a ? ta : !tb, ykc = a ? !tb : ta;
        // the compiled kernels, their LDS, and 32-bit offsets
        if (t.x_is_a != a || cols > 16 || rows < 1024 || k < 256 || k > 16384 || std::max(lda, ldb) >= 1u << 21) return 1;
        if (t.x_atoms != 1 && !(t.x_atoms == 2 && xkc == ykc) && !(t.x_atoms == 4 && !xkc)) return 2;
        if (t.waves != 4 && t.waves != 8 && t.waves != 16) return 3;
        if (t.waves * t.x_atoms > 64 || (k + t.waves - 1) / t.waves > 2048) return 4;
        ++seen[t.x_atoms];
    }
    return seen[1] && seen[2] && seen[4] && off ? 0 : 5;
}
"""


def test_every_thin_shape_has_a_kernel(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PLAN)
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amdgpu-arch-gemm_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", csrc, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


ROUNDS = r"""
#include "thin_plan.hpp"
#include <cstdio>
#include <random>
static bool on(uint32_t m, uint32_t n, uint32_t k, bool ta, bool tb, int cus) {
    return thin::choose(m, n, k, ta ? k : m, tb ? n : k, ta, tb, cus).on;
}
int main() {
    // one grid, one time: every row count of a whole round's last work-groups takes the same route
    for (uint32_t rows = 16353; rows <= 16384; ++rows)
        if (!on(rows, 16, 8192, true, false, 256)) { std::printf("%u rows\n", rows); return 1; }
    // a second round of a few work-groups takes as long as a full one, and on another chip begins elsewhere
    if (!on(4096, 16, 4096, true, false, 256) || on(4400, 16, 4096, true, false, 256) || !on(4400, 16, 4096, true, false, 304)) return 2;
    // a grid of 2^32 work-items cannot be launched (2^28 rows by 256 of k, A^T: 275 GB): the tile kernels take the call
    for (uint64_t rows = 1u << 20; rows < 1u << 29; rows += 1u << 20)
        for (uint32_t k : {256u, 512u, 1023u, 1024u, 4096u})
            for (int layout = 0; layout < 2; ++layout) {
                if (rows * k * 4 > 288000000000ull) continue;   // more than the device holds
                const thin::Shape t = thin::choose((uint32_t)rows, 16, k, k, layout ? 16 : k, true, layout);
                if (t.on && (rows + 16 * t.x_atoms - 1) / (16 * t.x_atoms) * 64u * t.waves >= 1ull << 32) {
                    std::printf("%llu rows, k = %u: %d atoms, %d waves\n", (unsigned long long)rows, k, t.x_atoms, t.waves);
                    return 5;
                }
            }
    // within one grid more rows cost the thin kernel nothing: a route taken is kept
    std::mt19937 rng(11);
    int taken = 0;
    for (int i = 0; i < 200000; ++i) {
        const uint32_t step = 64, base = 1024 + step * (rng() % 300), cols = 1 + rng() % 16, k = 256 + rng() % 9000;
        const bool ta = i & 1, tb = i & 2;
        const uint32_t lo = base + 1 + rng() % (step - 1), hi = base + step;
        if (base == 4736 || base == 6080 || base == 8128) continue;   // the tile's width changes
        if ((lo * 4e-6 * k > 256.0) != (hi * 4e-6 * k > 256.0)) continue;   // the last-level cache ends
        const thin::Shape a = thin::choose(lo, cols, k, ta ? k : lo, tb ? cols : k, ta, tb), b = thin::choose(hi, cols, k, ta ? k : hi, tb ? cols : k, ta, tb);
        const uint32_t w = 16u * (uint32_t)(a.x_atoms > 0 ? a.x_atoms : 1);
        if ((lo + w - 1) / w != (hi + w - 1) / w) continue;
        taken += a.on;
        if (a.on && !b.on) { std::printf("%u on, %u off: %u x %u\n", lo, hi, cols, k); return 3; }
    }
    return taken > 10000 ? 0 : 4;
}
"""


def test_the_route_follows_the_rounds_of_work_groups(tmp_path):
    src, exe = tmp_path / "rounds.cpp", tmp_path / "rounds"
    src.write_text(ROUNDS)
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amdgpu-arch-gemm_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", csrc, str(src), "-o", str(exe)], check=True)
    ret = subprocess.run([str(exe)], stdout=subprocess.PIPE)
    assert ret.returncode == 0, (ret.returncode, ret.stdout.decode())
