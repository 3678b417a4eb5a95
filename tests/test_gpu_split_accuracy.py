"""Errors of the split-BF16 kernels against float64, beside the same handle's FP32
kernels, on data that is hard on them: long chains of one sign, operands with
zeros (a rectified A, a B with few nonzeros), in every tile."""
import numpy as np
import pytest

from test_gpu_split_bf16 import _handles
from shim import sgemm_shim as S

pytestmark = pytest.mark.gpu

ROWS = 96   # of D that are compared: m * n / rows independent outputs, or 12288 at least


def _operands(m, n, k, data):
    A = S.fill_matrix(m, k, 57, 0, S.SGEMM_DIST_NORMAL)
    B = S.fill_matrix(k, n, 57, 1, S.SGEMM_DIST_NORMAL)
    if data in ("positive", "negative"):
        A, B = abs(A), (abs(B) if data == "positive" else -abs(B))
    elif data == "rectified":
        A = np.maximum(A, 0)
    elif data.startswith("nonzeros"):
        # `count` nonzeros to a column of B, in places spread over K
        count, keep = int(data.split("-")[1]), B
        B = np.zeros((k, n), dtype=np.float32, order="F")
        cols = np.arange(n)
        for i in range(count):
            at = (cols * 7919 + i * (k // count) + 13) % k
            B[at, cols] = keep[at, cols]
    return np.asfortranarray(A, dtype=np.float32), np.asfortranarray(B, dtype=np.float32)


SHAPES = [(2304, 2304, 1024, (256, 128)), (2048, 2048, 1024, (128, 128)), (16384, 128, 1024, (128, 64)),
          (1000, 999, 4097, (128, 128))]
LONG = [(2304, 2304, 8192, (256, 128)), (2304, 2304, 24500, (256, 128))]   # in one chain
DATA = ["normal", "positive", "negative", "rectified", "nonzeros-256", "nonzeros-16", "nonzeros-1"]


@pytest.mark.parametrize("m,n,k,tile,data", [(*s, d) for s in SHAPES for d in DATA] + [(*s, d) for s in LONG for d in DATA[:3]])
def test_error_against_float64(kernels, m, n, k, tile, data):
    print(f"accuracy {m}x{n}x{k} {data}", flush=True)
    A, B = _operands(m, n, k, data)
    a, b, d = S.DeviceBuffer.from_array(A), S.DeviceBuffer.from_array(B), S.DeviceBuffer(4 * m * n)
    kern, edges = _handles(m, n, k, "nn")
    outs = []
    try:
        plan = kern.split_bf16_plan(m, n, k)
        assert plan and plan["tile"] == tile and (plan["splits"] == 1 or m == 1000), plan
        for mode in (1, 0):
            kern.set_split_bf16(mode)
            kern.launch(a, b, None, d, m, n, k)
            kern.synchronize()
            outs.append(d.download().reshape(n, m).T)
    finally:
        kern.close()
        for e in edges:
            e.close()
    rows = np.arange(ROWS) * (m // ROWS) + 3
    A64, B64 = A[rows].astype(np.float64), B.astype(np.float64)
    ref = A64 @ B64
    split, fp32 = (o[rows].astype(np.float64) - ref for o in outs)
    norm = np.linalg.norm(ref)
    print(f"  relative error {np.linalg.norm(split) / norm:.3e}, FP32 kernels {np.linalg.norm(fp32) / norm:.3e}", flush=True)
    if data == "nonzeros-1":
        # One product ab: the terms left out are at most (2^-8 2^-17 2 + 2^-34) |ab|
        # (a bf16 is within 2^-8 of its value, two of them within 2^-17), the sum of the small
        # products, at most 2^-7 |ab|, is rounded five times to 24 bits, and the result once.
        assert np.all(abs(split) <= (1 + 2.0 ** -10 + 5 * 2.0 ** -6 + 1) * 2.0 ** -24 * abs(ref))
    else:
        # over 12000 outputs: a ratio of the 2-norms is certain to about a percent, and the
        # measured ones are 0.13 to 0.65
        assert np.linalg.norm(split) <= np.linalg.norm(fp32)
