"""sgemm_launch_noalloc between streams that capture, fork, are shared or stand
for one stream per thread: no call spoils another's partial sums.  The rules
themselves run against a model in test_noalloc_slots.py."""
import ctypes
import threading

import numpy as np
import pytest

from generator import catalog
from shim import sgemm_shim as S

pytestmark = pytest.mark.gpu

NAME = "mt64x64_a16_wg1x4_dk32_s3"
BIG = (640, 640, 8192)       # 100 tiles in 5 K ranges, 8 MB of partials: every slot
SMALL = (256, 256, 4096)     # 4 MB: one slot
GLOBAL, THREAD_LOCAL = 0, 1
PER_THREAD = 2               # hipStreamPerThread
_vp = ctypes.c_void_p


def _ok(rc):
    assert rc == 0, rc


class _Hip:
    def __init__(self):
        self.lib = ctypes.CDLL("libamdhip64.so")
        for name in ("hipStreamDestroy", "hipStreamSynchronize", "hipGraphExecDestroy", "hipGraphDestroy",
                     "hipEventDestroy"):
            getattr(self.lib, name).argtypes = [_vp]

    def stream(self):
        s = _vp()
        _ok(self.lib.hipStreamCreate(ctypes.byref(s)))
        return s

    def event(self):
        e = _vp()
        _ok(self.lib.hipEventCreateWithFlags(ctypes.byref(e), 2))
        return e

    def begin(self, s, mode=THREAD_LOCAL):
        _ok(self.lib.hipStreamBeginCapture(s, mode))

    def end(self, s):
        graph, exe = _vp(), _vp()
        _ok(self.lib.hipStreamEndCapture(s, ctypes.byref(graph)))
        _ok(self.lib.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0))
        _ok(self.lib.hipGraphDestroy(graph))
        return exe


class _Call:
    """One problem's operands, its D and the D that sgemm_launch gives."""

    def __init__(self, shape, seed):
        m, n, k = self.shape = shape
        self.a = S.DeviceBuffer.from_array(S.fill_matrix(m, k, seed, 0))
        self.b = S.DeviceBuffer.from_array(S.fill_matrix(k, n, seed, 1))
        self.d = S.DeviceBuffer(4 * m * n)
        with _kernel() as kern:
            # a slot holds an eighth of the scratch
            assert (kern.workspace_size(m, n, k) > S.SGEMM_NOALLOC_PARTIAL_BYTES // 8 + 4096) == (shape == BIG)
            assert kern.launch_splits(m, n, k) > 1
            kern.launch(self.a, self.b, None, self.d, m, n, k)
            kern.synchronize()
        self.want = self.d.download()
        self.spoil()

    def spoil(self):
        self.d.upload(np.full(self.want.size, np.nan, dtype=np.float32))

    def run(self, kern):
        kern.launch_noalloc(self.a, self.b, None, self.d, *self.shape)

    def check(self, what):
        assert np.array_equal(self.d.download(), self.want), what


def _kernel():
    kern = S.Kernel(*catalog.paths(NAME))
    kern.set_split_bf16(0)
    return kern


def test_a_captured_call_takes_nothing_over(kernels):
    hip = _Hip()
    eager, captured, after = _Call(BIG, 71), _Call(BIG, 72), _Call(BIG, 73)
    one, two = _kernel(), _kernel()
    s, t = hip.stream(), hip.stream()
    exe = _vp()
    try:
        one.set_stream(s.value)
        two.set_stream(t.value)
        print("capture beside eager calls", flush=True)
        for r in range(10):
            eager.run(two)                 # in flight on t ...
            hip.begin(s)
            captured.run(one)              # ... while a call that needs every slot is captured on s
            exe = hip.end(s)
            after.run(one)                 # and s takes the slots over from t
            one.synchronize()
            two.synchronize()
            eager.check(f"eager {r}")
            after.check(f"after {r}")
            for q in range(3):             # the replay, with nothing beside it
                captured.spoil()
                _ok(hip.lib.hipGraphLaunch(exe, s))
                one.synchronize()
                captured.check(f"replay {r} {q}")
                after.run(one)
                one.synchronize()
                after.check(f"between {r} {q}")
            _ok(hip.lib.hipGraphExecDestroy(exe))
            for c in (eager, captured, after):
                c.spoil()
    finally:
        one.close()
        two.close()
        hip.lib.hipStreamDestroy(s)
        hip.lib.hipStreamDestroy(t)


def test_branches_of_one_capture_are_a_chain(kernels):
    hip = _Hip()
    calls = [_Call(BIG, 74), _Call(BIG, 75), _Call(SMALL, 76), _Call(SMALL, 77)]
    one, two = _kernel(), _kernel()
    s, t = hip.stream(), hip.stream()
    fork, join = hip.event(), hip.event()
    exe = _vp()
    try:
        one.set_stream(s.value)
        two.set_stream(t.value)
        print("two branches in one capture", flush=True)
        hip.begin(s)
        _ok(hip.lib.hipEventRecord(fork, s))
        _ok(hip.lib.hipStreamWaitEvent(t, fork, 0))
        for i, c in enumerate(calls):      # the branches take turns, no edge between them from here
            c.run((one, two)[i % 2])
        _ok(hip.lib.hipEventRecord(join, t))
        _ok(hip.lib.hipStreamWaitEvent(s, join, 0))
        exe = hip.end(s)
        for q in range(5):
            for c in calls:
                c.spoil()
            _ok(hip.lib.hipGraphLaunch(exe, s))
            one.synchronize()
            for i, c in enumerate(calls):
                c.check(f"replay {q} call {i}")
            calls[2].run(two)              # eager work between the replays
            two.synchronize()
        _ok(hip.lib.hipGraphExecDestroy(exe))
    finally:
        one.close()
        two.close()
        for e in (fork, join):
            hip.lib.hipEventDestroy(e)
        hip.lib.hipStreamDestroy(s)
        hip.lib.hipStreamDestroy(t)


def test_a_capturing_owner_keeps_its_slots(kernels):
    """The owner's eager call may still run while it captures: a call that needs
    its slots runs without scratch, each tile's K in one work-group."""
    hip = _Hip()
    first, captured, other, small = _Call(BIG, 78), _Call(BIG, 79), _Call(BIG, 80), _Call(SMALL, 81)
    one, two = _kernel(), _kernel()
    s = hip.stream()
    try:
        two.set_stream(s.value)
        whole = []
        one.set_split_k(1)
        for c in (other, small):
            one.launch(c.a, c.b, None, c.d, *c.shape)
            one.synchronize()
            whole.append(c.d.download())
            assert not np.array_equal(whole[-1], c.want)
        one.set_split_k(0)
        print("an owner that captures", flush=True)
        for r in range(5):
            first.run(two)
            hip.begin(s)
            captured.run(two)
            other.run(one)                 # every slot is the capturing stream's
            small.run(one)
            exe = hip.end(s)
            one.synchronize()
            two.synchronize()
            first.check(f"first {r}")
            for c, w in zip((other, small), whole):
                assert np.array_equal(c.d.download(), w), r
            for q in range(3):
                captured.spoil()
                _ok(hip.lib.hipGraphLaunch(exe, s))
                two.synchronize()
                captured.check(f"replay {r} {q}")
            _ok(hip.lib.hipGraphExecDestroy(exe))
            other.run(one)                 # the capture has ended: with scratch again
            one.synchronize()
            other.check(f"other {r}")
            first.run(two)                 # and the slots are the first stream's again
            two.synchronize()
    finally:
        one.close()
        two.close()
        hip.lib.hipStreamDestroy(s)


def test_a_handle_leaves_a_stream_that_others_use(kernels):
    hip = _Hip()
    a, b, c = _Call(BIG, 82), _Call(SMALL, 83), _Call(BIG, 84)
    s = hip.stream()
    two, three = _kernel(), _kernel()
    try:
        two.set_stream(s.value)
        print("a shared stream", flush=True)
        for r in range(10):
            one = _kernel()
            one.set_stream(s.value)
            b.run(one)
            leaver = threading.Thread(target=one.close)   # while `two` keeps launching on the stream
            leaver.start()
            a.run(two)
            c.run(three)                   # from a third stream, over a's slots
            leaver.join()
            c.run(three)
            two.synchronize()
            three.synchronize()
            for i, x in enumerate((a, b, c)):
                x.check(f"{r} {i}")
                x.spoil()
    finally:
        two.close()
        three.close()
        hip.lib.hipStreamDestroy(s)


def test_one_name_for_a_stream_of_every_thread(kernels):
    calls = [[_Call(SMALL, 85), _Call(BIG, 86)], [_Call(SMALL, 87), _Call(BIG, 88)]]
    handles = [_kernel(), _kernel()]
    failed = []

    def work(q):
        try:
            handles[q].set_stream(PER_THREAD)
            for _ in range(20):
                for c in calls[q]:
                    c.run(handles[q])
            handles[q].synchronize()
            for i, c in enumerate(calls[q]):
                c.check(f"thread {q} call {i}")
            handles[q].set_stream(None)
        except BaseException as e:   # reported by the test's own thread
            failed.append(e)

    print("two threads on their own per-thread streams", flush=True)
    threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not failed, failed
    finally:
        for h in handles:
            h.close()


def test_split_bf16_calls_share_the_slots(kernels):
    """K splits of the split-BF16 kernels, small and large, from more streams than slots."""
    shapes = [(511, 513, 16400), (1536, 1536, 1531), (1000, 999, 4097)]
    calls = []
    for i, (m, n, k) in enumerate(shapes):
        name = catalog.select(m, n, k)
        a = S.DeviceBuffer.from_array(S.fill_matrix(m, k, 90 + i, 0))
        b = S.DeviceBuffer.from_array(S.fill_matrix(k, n, 90 + i, 1))
        d = S.DeviceBuffer(4 * m * n)
        with S.Kernel(*catalog.paths(name)) as kern:
            plan = kern.split_bf16_plan(m, n, k)
            assert plan and plan["splits"] > 1
            kern.launch(a, b, None, d, m, n, k)
            kern.synchronize()
        calls.append((name, a, b, d.download()))
    handles = [S.Kernel(*catalog.paths(calls[q % 3][0])) for q in range(10)]
    try:
        print("split-BF16 K splits on ten streams", flush=True)
        for r in range(5):
            outs = []
            for q, kern in enumerate(handles):
                name, a, b, want = calls[q % 3]
                d = S.DeviceBuffer(want.nbytes)
                d.upload(np.full(want.size, np.nan, dtype=np.float32))
                outs.append(d)
            for q, kern in enumerate(handles):
                _, a, b, _ = calls[q % 3]
                kern.launch_noalloc(a, b, None, outs[q], *shapes[q % 3])
            for kern in handles:
                kern.synchronize()
            for q in range(len(handles)):
                assert np.array_equal(outs[q].download(), calls[q % 3][3]), (r, q)
    finally:
        for kern in handles:
            kern.close()
