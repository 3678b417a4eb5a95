"""The split-BF16 kernels (csrc/bf16x6_kernel.hpp) through the public launch
path, against float64 and against the same handle's FP32 kernels."""
import ctypes

import numpy as np
import pytest

from generator import catalog
from shim import sgemm_shim as S

pytestmark = pytest.mark.gpu

# (m, n, k, layout, pad, shift, alpha, beta, tile, K split): each tile whole and
# ragged, a K remainder and none, every layout, odd leading dimensions and
# pointers `shift` floats past a 16-byte boundary, the K split on and off
CASES = [
    (4096, 4096, 520, "nn", 0, 0, 1.0, 0.0, (256, 128), False),
    (3585, 3501, 149, "tt", 3, 2, 1.0, 1.0, (256, 128), False),
    (5397, 3401, 331, "tn", 0, 3, 0.75, -1.5, (256, 128), False),
    (2304, 2304, 1024, "nn", 0, 0, 1.0, 0.0, (256, 128), False),
    (4095, 2047, 1001, "nt", 1, 1, -0.5, 0.75, (256, 128), False),
    (1536, 1536, 1531, "tn", 1, 0, 1.0, 0.0, (256, 128), True),
    (2048, 2048, 1023, "nt", 0, 0, 1.0, 0.0, (128, 128), False),
    (1000, 999, 4097, "tn", 3, 1, 1.0, 1.0, (128, 128), True),
    (128, 9001, 2049, "nt", 1, 2, 1.0, -1.0, (128, 128), True),
    (16383, 127, 1001, "nn", 0, 0, 1.0, 0.0, (128, 64), False),
    (1281, 1155, 2113, "tt", 1, 3, 2.0, 0.5, (128, 64), False),
    (511, 513, 16400, "nn", 0, 1, 0.5, 0.0, (128, 64), True),
    (250, 700, 18881, "nt", 1, 0, 1.0, 0.75, (128, 64), True),
    (4097, 4097, 520, "nn", 0, 0, 1.0, 0.5, (256, 128), False),      # thin strips on the edge kernels
]


def _matrix(rows, cols, ld, seed, mid, dist):
    full = S.fill(ld * cols, seed, mid, dist).reshape(cols, ld).T
    return np.asfortranarray(full), full[:rows, :]


def _device(full, shift):
    flat = full.ravel(order="F")
    buf = S.DeviceBuffer(flat.nbytes + 16)
    view = buf.view(4 * shift, flat.nbytes)
    view.upload(flat)
    return buf, view


def _handles(m, n, k, layout):
    name = catalog.select(m, n, k, layout[0] == "t", layout[1] == "t")
    kern = S.Kernel(*catalog.paths(name))
    edges = [S.Kernel(*catalog.paths(e)) for e in catalog.EDGE_KERNEL.get(name, ())]
    if edges:
        kern.set_edge_kernels(*edges)
    return kern, edges


def _rel(d, ref):
    return float(np.linalg.norm(d.astype(np.float64) - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("m,n,k,layout,pad,shift,alpha,beta,tile,split", CASES)
def test_split_bf16_is_no_further_from_float64_than_fp32(kernels, m, n, k, layout, pad, shift, alpha, beta, tile, split):
    print(f"split-BF16 {m}x{n}x{k} {layout} pad {pad} shift {shift}", flush=True)
    ta, tb = layout[0] == "t", layout[1] == "t"
    ra, ca = (k, m) if ta else (m, k)
    rb, cb = (n, k) if tb else (k, n)
    Af, A = _matrix(ra, ca, ra + pad, 51, 0, S.SGEMM_DIST_NORMAL)
    Bf, B = _matrix(rb, cb, rb + 2 * pad, 51, 1, S.SGEMM_DIST_UNIFORM)
    Cf, C = _matrix(m, n, m + pad, 51, 2, S.SGEMM_DIST_UNIFORM)
    (_a, dA), (_b, dB), (_c, dC) = (_device(x, shift) for x in (Af, Bf, Cf))
    ldd = m + 3 * pad
    ref = alpha * ((A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64))
    if beta:
        ref += beta * C.astype(np.float64)
    kern, edges = _handles(m, n, k, layout)
    ld = dict(lda=ra + pad, ldb=rb + 2 * pad, ldc=m + pad, ldd=ldd)
    plan = kern.split_bf16_plan(m, n, k, alpha, beta, **ld)
    print(f"  plan {plan}", flush=True)
    assert plan is not None and (tile is None or plan["tile"] == tile) and (split is None or (plan["splits"] > 1) == split)
    outs = {}
    try:
        for what, mode, entry in (("split", 1, "launch"), ("again", 1, "launch"), ("noalloc", 1, "launch_noalloc"),
                                  ("fp32", 0, "launch")):
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
    assert np.array_equal(outs["split"], outs["again"]), "repeated launches differ"
    assert np.array_equal(outs["split"], outs["noalloc"]), "launch_noalloc differs"
    split_err, fp32_err = _rel(outs["split"], ref), _rel(outs["fp32"], ref)
    print(f"  relative error {split_err:.3e}, FP32 kernels {fp32_err:.3e}", flush=True)
    # a million random errors or more: their 2-norm ratio is certain to well under a percent
    assert split_err <= fp32_err


@pytest.mark.parametrize("m,n,k,layout", [(3585, 3501, 149, "nn"), (1000, 999, 4097, "tt"), (511, 513, 16400, "nt"),
                                          (2304, 2304, 1024, "tn")])
def test_special_values_take_the_fp32_way(kernels, m, n, k, layout):
    """NaN, Inf and values whose scaled product overflows give the pattern and
    the finite values of the FP32 kernels; subnormal operands keep their bits."""
    ta, tb = layout[0] == "t", layout[1] == "t"
    A = S.fill(m * k, 52, 0).reshape((m, k) if ta else (k, m)).copy()    # the stored matrix, transposed
    B = S.fill(k * n, 52, 1).reshape((k, n) if tb else (n, k)).copy()
    opA, opB = (A if ta else A.T), (B if tb else B.T)                    # views: op(A) is m x k, op(B) k x n
    opA[3, 5], opA[m - 1, k - 1], opA[m // 2, 7] = np.nan, np.inf, -np.inf
    opB[5, 3], opB[k - 1, n - 1] = np.inf, -np.inf
    opA[10, 11], opB[11, 12] = 3.0e38, 1.0e-3
    opA[20, :] *= np.float32(1e-38)     # a row of subnormal and barely normal values
    opB[:, 21] *= np.float32(1e-38)
    dA, dB = (S.DeviceBuffer.from_array(x.ravel()) for x in (A, B))
    kern, edges = _handles(m, n, k, layout)
    outs = []
    try:
        assert kern.split_bf16_plan(m, n, k) is not None
        for mode in (1, 0):
            kern.set_split_bf16(mode)
            dD = S.DeviceBuffer(4 * m * n)
            kern.launch(dA, dB, None, dD, m, n, k)
            kern.synchronize()
            outs.append(dD.download().reshape(n, m).T.astype(np.float64))
    finally:
        kern.close()
        for e in edges:
            e.close()
    got, want = outs
    with np.errstate(invalid="ignore", over="ignore"):
        ref = opA.astype(np.float64) @ opB.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any()
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf]) and np.array_equal(np.isinf(got), inf)
    fin = np.isfinite(want)
    # row 20 and column 21 (away from planted values and from one another's product) have a scale of their own
    for rows, cols in ((slice(20, 21), slice(30, n - 1)), (slice(30, m // 2), slice(21, 22)), (slice(30, 90), slice(30, 90))):
        f = fin[rows, cols]
        e = [np.linalg.norm((o[rows, cols] - ref[rows, cols])[f]) / np.linalg.norm(ref[rows, cols][f]) for o in outs]
        print(f"  {layout} block error {e[0]:.3e}, FP32 kernels {e[1]:.3e}", flush=True)
        # Where the launch has one K range, these blocks lie in tiles that met a
        # planted value and ran again with FP32 MFMAs in one chain of k: 1.8e-8 * sqrt(k),
        # which the handle's own kernels undercut where they cut K (stream-K); with
        # several, ranges without one keep their split sums.  The error of a block of
        # n outputs is random to about 1 / sqrt(n)
        assert e[0] <= max(e[1], 1.8e-8 * np.sqrt(k)) * (1.0 + 6.0 / np.sqrt(f.sum()))


def test_split_bf16_is_off_where_the_handle_is_fixed(kernels):
    m = n = k = 2048
    kern, edges = _handles(m, n, k, "nn")
    try:
        assert kern.split_bf16_plan(m, n, k) is not None
        assert kern.split_bf16_plan(512, 512, 512) is None                   # too small to gain
        assert kern.split_bf16_plan(m, n, k, alpha=1e-30) is None            # alpha * 2^-32 would be subnormal
        assert kern.split_bf16_plan(m, n, k, lda=1 << 21) is None
        for off, on in ((lambda: kern.set_split_k(2), lambda: kern.set_split_k(0)),
                        (lambda: kern.set_stream_k(0), lambda: kern.set_stream_k(1)),
                        (lambda: kern.set_split_bf16(0), lambda: kern.set_split_bf16(1))):
            try:
                off()
            except S.SgemmError:
                continue        # this code object has no such kernel
            assert kern.split_bf16_plan(m, n, k) is None
            on()
            assert kern.split_bf16_plan(m, n, k) is not None
        with pytest.raises(S.SgemmError, match="outside 0..1"):
            kern.set_split_bf16(2)
    finally:
        kern.close()
        for e in edges:
            e.close()
    with S.Kernel(*catalog.paths("mt256x256_a32_wg2x2_dk16")) as other:      # no split_bf16 key
        assert other.split_bf16_plan(m, n, k) is None


@pytest.mark.parametrize("m,n,k,entry", [(2048, 2048, 512, "launch"), (1000, 999, 4097, "launch_noalloc"),
                                         (2048, 8, 1024, "launch"), (333, 129, 517, "launch_noalloc")])
def test_an_earlier_error_is_not_the_launchs(kernels, m, n, k, entry):
    """The split, thin and ticket-clearing kernels report their own launch: an
    error that the program left behind before (here a device that does not
    exist) must not fail them."""
    print(f"stale error {m}x{n}x{k} {entry}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    a, b = (S.DeviceBuffer.from_array(S.fill_matrix(*s, 56, i)) for i, s in enumerate(((m, k), (k, n))))
    d = S.DeviceBuffer(4 * m * n)
    kern, edges = _handles(m, n, k, "nn")
    try:
        kern.launch(a, b, None, d, m, n, k)
        kern.synchronize()
        want = d.download()
        d.upload(np.full(m * n, np.nan, dtype=np.float32))
        assert hip.hipSetDevice(9999) != 0
        getattr(kern, entry)(a, b, None, d, m, n, k)
        hip.hipGetLastError()
        kern.synchronize()
        assert np.array_equal(d.download(), want)
    finally:
        kern.close()
        for e in edges:
            e.close()
