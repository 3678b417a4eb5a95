"""sgemm_launch_noalloc on several streams: the calls share one static scratch
in slots of their own, or wait for one another, waited for by the host or not."""
import numpy as np
import pytest

from generator import catalog
from shim import sgemm_shim as S

pytestmark = pytest.mark.gpu

NAME = "mt64x64_a16_wg1x4_dk32_s3"


def test_noalloc_on_streams_that_take_turns(kernels):
    # partials of 0.6, 4 and 0.1 MB in slots of 4 MB, and 8 MB, which take all of them
    shapes = [(333, 129, 517), (256, 256, 4096), (70, 45, 1001), (640, 640, 8192)]
    bufs, want = [], []
    with S.Kernel(*catalog.paths(NAME)) as ref:
        for i, (m, n, k) in enumerate(shapes):
            ref.set_split_bf16(0)
            assert ref.launch_splits(m, n, k) > 1
            # a slot is an eighth of the scratch; the workspace's size counts its tickets too
            assert (ref.workspace_size(m, n, k) > S.SGEMM_NOALLOC_PARTIAL_BYTES // 8 + 4096) == (i == 3)
            bufs.append([S.DeviceBuffer.from_array(S.fill_matrix(*s, 60 + i, j))
                         for j, s in enumerate(((m, k), (k, n)))] + [S.DeviceBuffer(4 * m * n)])
            ref.launch(bufs[i][0], bufs[i][1], None, bufs[i][2], m, n, k)
            ref.synchronize()
            want.append(bufs[i][2].download())

    def overlap(kerns, order):
        """Calls of several handles, each on its own stream, with no wait between them."""
        outs = [S.DeviceBuffer(4 * shapes[i][0] * shapes[i][1]) for _, i in order]
        for (q, i), d in zip(order, outs):
            kerns[q].set_split_bf16(0)
            kerns[q].launch_noalloc(bufs[i][0], bufs[i][1], None, d, *shapes[i])
        for kern in kerns:
            kern.synchronize()
        for (_, i), d in zip(order, outs):
            assert np.array_equal(d.download(), want[i])

    def check(kern, i):
        m, n, k = shapes[i]
        bufs[i][2].upload(np.full(m * n, np.nan, dtype=np.float32))
        kern.set_split_bf16(0)
        kern.launch_noalloc(bufs[i][0], bufs[i][1], None, bufs[i][2], m, n, k)
        kern.synchronize()
        assert np.array_equal(bufs[i][2].download(), want[i])

    one, two = S.Kernel(*catalog.paths(NAME)), S.Kernel(*catalog.paths(NAME))
    try:
        for kern, i in ((one, 0), (one, 1), (one, 2), (two, 1), (two, 1), (one, 0), (two, 2), (one, 1), (one, 1)):
            check(kern, i)
        for _ in range(20):
            overlap((one, two), ((0, 1), (1, 0), (0, 0), (1, 1), (1, 2), (0, 3), (1, 0), (0, 1), (1, 3), (0, 2)))
        many = [S.Kernel(*catalog.paths(NAME)) for _ in range(11)]   # more streams than slots
        try:
            for _ in range(5):
                overlap(many, [(q, (q + r) % 3) for r in range(3) for q in range(len(many))])
        finally:
            for kern in many:
                kern.close()
        one.close()                             # its stream goes; a new handle may get the same address
        one = S.Kernel(*catalog.paths(NAME))
        for kern, i in ((one, 1), (one, 0), (two, 0)):
            check(kern, i)
    finally:
        one.close()
        two.close()
