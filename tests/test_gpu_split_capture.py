"""Split-BF16 launches under HIP graph capture, and what they must not touch:
in-place updates, a C that is not read, the memory beside D."""
import ctypes

import numpy as np
import pytest

from test_gpu_noalloc_streams import _Hip, _ok
from test_gpu_split_bf16 import _handles
from shim import sgemm_shim as S

pytestmark = pytest.mark.gpu


def _bits(m, n, k, entry, kern, a, b, d):
    getattr(kern, entry)(a, b, None, d, m, n, k)
    kern.synchronize()
    return d.download()


@pytest.mark.parametrize("entry,m,n,k,warm", [
    ("launch", 16384, 128, 4096, False),         # needs no workspace on the FP32 kernel, K ranges on the split one
    ("launch", 16384, 128, 4096, True),          # the handle holds the workspace already
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
        # a cold handle has no workspace for the K ranges and cannot allocate it under capture
        want = own if entry == "launch" and plan["splits"] > 1 and not warm else split
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
