"""Split-BF16 launches under HIP graph capture, and what they must not touch:
in-place updates, a C that is not read, the memory beside D."""
import ctypes

import numpy as np
import pytest

from test_gpu_noalloc_streams import _Hip, _ok
from test_gpu_split_bf16 import _handles, _rel
from shim import sgemm_shim as S

pytestmark = pytest.mark.gpu


def _bits(m, n, k, entry, kern, a, b, d):
    getattr(kern, entry)(a, b, None, d, m, n, k)
    kern.synchronize()
    return d.download()


@pytest.mark.parametrize("entry,m,n,k,warm", [
    ("launch", 16384, 128, 4096, False),         # needs no workspace on the FP32 kernel, K ranges on the split one
    ("launch", 16384, 128, 4096, True),          # the handle holds the workspace already, until a larger launch replaces it
    ("launch_noalloc", 16384, 128, 4096, False),
    ("launch_noalloc", 1000, 999, 4097, False),
    ("launch", 2048, 2048, 1024, False),         # no K split
])
def test_captured_split_launches_replay(kernels, entry, m, n, k, warm):
    print(f"captured {entry} {m}x{n}x{k}", flush=True)
    hip = _Hip()
    stream = hip.stream()
    a, b = (S.DeviceBuffer.from_array(S.fill_matrix(*s, 55, i)) for i, s in enumerate(((m, k), (k, n))))
    d = S.DeviceBuffer(4 * m * n)
    other, others = _handles(m, n, k, "nn")
    kern, edges = _handles(m, n, k, "nn")
    try:
        plan = kern.split_bf16_plan(m, n, k)
        assert plan and (plan["splits"] > 1) == (k >= 4096)
        split = _bits(m, n, k, "launch", other, a, b, d)
        other.set_split_bf16(0)
        own = _bits(m, n, k, "launch", other, a, b, d)
        kern.set_stream(stream.value)
        if warm:
            _bits(m, n, k, entry, kern, a, b, d)
        hip.begin(stream, 0)
        try:
            getattr(kern, entry)(a, b, None, d, m, n, k)
        finally:
            exe = hip.end(stream)
        # a graph of sgemm_launch uses no workspace: the handle cannot allocate it under capture, and may replace it later
        want = own if entry == "launch" and plan["splits"] > 1 else split
        if warm:
            assert kern.workspace_size(1536, 1536, 1531) > kern.workspace_size(m, n, k)
            large = [S.DeviceBuffer(4 * 1536 * 1536) for _ in range(3)]
            kern.launch(*large[:2], None, large[2], 1536, 1536, 1531)
        for q in range(3):
            d.upload(np.full(m * n, np.nan, dtype=np.float32))
            _ok(hip.lib.hipGraphLaunch(exe, stream))
            kern.synchronize()
            assert np.array_equal(d.download(), want), q
            assert np.array_equal(_bits(m, n, k, entry, kern, a, b, d), split), q   # eager, between the replays
        _ok(hip.lib.hipGraphExecDestroy(exe))
    finally:
        for x in (kern, other, *edges, *others):
            x.set_stream(None)
            x.close()
        hip.lib.hipStreamDestroy(stream)


# each split tile and the thin kernel, ragged in m and n, with and without K ranges
RAGGED = [(4001, 3997, 333, "nn"), (2047, 2001, 1023, "nt"), (1000, 999, 4097, "tn"), (16383, 127, 1001, "tt"),
          (511, 513, 16400, "nn"), (3001, 13, 700, "nt"), (11, 9001, 513, "tn")]


@pytest.mark.parametrize("m,n,k,layout", RAGGED)
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_nothing_beside_d_is_written(kernels, m, n, k, layout, beta):
    """D's columns past n belong to the caller: a tile's worth of them, and the
    rows past m of every column, keep their values; so does D's own pass in place
    (dC == dD), and a C that beta = 0 leaves unread may hold NaN."""
    print(f"beside D {m}x{n}x{k} {layout} beta {beta}", flush=True)
    ta, tb = layout[0] == "t", layout[1] == "t"
    guard, ldd = 256, m + 5
    a = S.DeviceBuffer.from_array(S.fill_matrix(*((k, m) if ta else (m, k)), 58, 0))
    b = S.DeviceBuffer.from_array(S.fill_matrix(*((n, k) if tb else (k, n)), 58, 1))
    C = S.fill_matrix(ldd, n, 58, 2) if beta else np.full((ldd, n), np.nan, dtype=np.float32)
    c = S.DeviceBuffer.from_array(C)
    d = S.DeviceBuffer(4 * ldd * (n + guard))
    kern, edges = _handles(m, n, k, layout)
    try:
        assert min(m, n) <= 16 or kern.split_bf16_plan(m, n, k, 1.0, beta, ldc=ldd, ldd=ldd) is not None
        outs = []
        for in_place in (False, True):
            full = np.full((n + guard, ldd), 9.5, dtype=np.float32)   # the columns of D
            if in_place and beta:
                full[:n] = C.T
            d.upload(full.ravel())
            kern.launch(a, b, d if in_place else c, d, m, n, k, alpha=1.5, beta=beta, ldc=ldd, ldd=ldd)
            kern.synchronize()
            got = d.download().reshape(n + guard, ldd)
            assert np.array_equal(got[n:], full[n:]), "columns past n of D were written"
            assert np.array_equal(got[:n, m:], full[:n, m:]), "rows past m of D were written"
            outs.append(got[:n, :m])
        assert np.all(np.isfinite(outs[0]))
        assert np.array_equal(outs[0], outs[1]), "in place differs"
    finally:
        kern.close()
        for e in edges:
            e.close()


@pytest.mark.parametrize("m,n,k", [(2304, 2304, 1024), (2048, 2048, 1024), (16384, 128, 1024), (1000, 999, 4097)])
def test_subnormal_operands_keep_their_bits(kernels, m, n, k):
    """Rows of A and columns of B of subnormal and barely normal values, nothing
    that makes a tile run again: the scaled BF16 terms hold all their bits."""
    print(f"subnormals {m}x{n}x{k}", flush=True)
    A, B = S.fill_matrix(m, k, 59, 0), S.fill_matrix(k, n, 59, 1)
    A[32:64] *= np.float32(1e-38)
    B[:, 64:96] *= np.float32(1e-38)
    a, b, d = S.DeviceBuffer.from_array(A), S.DeviceBuffer.from_array(B), S.DeviceBuffer(4 * m * n)
    kern, edges = _handles(m, n, k, "nn")
    outs = []
    try:
        assert kern.split_bf16_plan(m, n, k) is not None
        for mode in (1, 0):
            kern.set_split_bf16(mode)
            kern.launch(a, b, None, d, m, n, k)
            kern.synchronize()
            outs.append(d.download().reshape(n, m).T)
    finally:
        kern.close()
        for e in edges:
            e.close()
    for rows, cols in ((slice(32, 64), slice(0, 64)), (slice(128, 256), slice(64, 96)), (slice(128, 256), slice(0, 64))):
        ref = A[rows].astype(np.float64) @ B[:, cols].astype(np.float64)
        split, fp32 = (_rel(o[rows, cols], ref) for o in outs)
        print(f"  relative error {split:.3e}, FP32 kernels {fp32:.3e}", flush=True)
        # 2048 outputs or more: 2-norms to 1.6%, and results near 1e-37 are rounded as FP32 normals
        assert split <= fp32
