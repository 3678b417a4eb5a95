"""The work this framework is measured on: single-precision GEMM calls through its public path.

A user's program asks ``catalog.select`` for the instance of a problem, opens
it (with the edge kernels the catalog names for it), and launches it on
matrices that live in GPU memory: D = alpha * op(A) * op(B) + beta * C,
column-major, FP32.  One pass is one launch.  The sizes are those of the
package's benchmark workloads, shape sweep and tests, and of the small, thin
and ragged problems beside them.

A column-major r x c matrix with leading dimension ld is the row-major
(c, ld) torch tensor whose rows are its columns.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "amdgpu-arch-gemm_amd"))

from generator import catalog  # noqa: E402
from shim import sgemm_shim as S  # noqa: E402


def _case(name, m, n, k, layout="nn", alpha=1.0, beta=0.0, dist="uniform", pad=0, noalloc=False):
    return {"name": name, "m": m, "n": n, "k": k, "layout": layout, "alpha": alpha, "beta": beta, "dist": dist,
            "pad": pad, "noalloc": noalloc}


def listed():
    return [
        # the smallest calls: a block update inside a factorisation or a small
        # dense layer, where the launch itself is most of the time
        _case("small_256", 256, 256, 256),
        # a small odd problem in a serving loop that may not allocate
        _case("small_333x129x517_tt", 333, 129, 517, "tt", alpha=0.5, beta=-1.5, noalloc=True),
        # one tile per compute unit: the benchmark's 1024^3
        _case("cube_1024", 1024, 1024, 1024),
        # a ragged weight gradient accumulated into a buffer with padded rows
        _case("ragged_1000x999x4097_tn", 1000, 999, 4097, "tn", beta=1.0, pad=3),
        # few right-hand sides: a wide layer applied to a small batch
        _case("thin_4096x16x4096_tn", 4096, 16, 4096, "tn"),
        # the benchmark's tall matrix with 128 columns
        _case("tall_16384x128x4096", 16384, 128, 4096),
        # the benchmark's deep K: an inner product of two long thin panels
        _case("deepk_512x512x16384", 512, 512, 16384),
        # a size no tile divides, as in the shape sweep, updating C
        _case("cube_3000_nt", 3000, 3000, 3000, "nt", alpha=0.75, beta=-1.5),
        # the benchmark's headline
        _case("cube_4096", 4096, 4096, 4096),
        # one past the headline in every dimension
        _case("ragged_4097", 4097, 4097, 4097),
        # the benchmark's shallow K on normal data: D's stores dominate
        _case("rank256_8192", 8192, 8192, 256, dist="normal"),
        # the largest square of the shape sweep
        _case("cube_8192_tt", 8192, 8192, 8192, "tt", dist="normal"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["small", "cube", "ragged", "thin", "tall", "deep", "shallow"])
    if kind == "small":
        m, n, k = log(64, 700), log(64, 700), log(64, 1000)
    elif kind == "cube":
        m = n = k = log(700, 7000)
    elif kind == "ragged":
        m, n, k = log(500, 7000), log(500, 7000), log(300, 7000)
    elif kind == "thin":
        m, n, k = log(1000, 16384), log(1, 64), log(500, 8192)
        if rng.random() < 0.5:
            m, n = n, m
    elif kind == "tall":
        m, n, k = log(6000, 24000), log(96, 400), log(1000, 5000)
        if rng.random() < 0.5:
            m, n = n, m
    elif kind == "deep":
        m, n, k = log(128, 800), log(128, 800), log(6000, 40000)
    else:
        m, n, k = log(3000, 9000), log(3000, 9000), log(64, 400)
    if rng.random() < 0.4:  # half-way to the sizes people round to
        m, n, k = (max(1, 64 * round(x / 64)) if x >= 64 else x for x in (m, n, k))
    case = _case("", m, n, k, rng.choice(["nn", "tn", "nt", "tt"]), rng.choice([1.0, 1.0, -0.5]),
                 rng.choice([0.0, 0.0, 1.0, 0.75]), rng.choice(["uniform", "normal"]), rng.choice([0, 0, 1, 4]),
                 kind == "small" and rng.random() < 0.5)
    del case["name"]
    return case


class _Buffer:
    """A torch tensor's memory as the launch entry points take it."""

    def __init__(self, t):
        self.tensor = t
        self.ptr = t.data_ptr()


def _stored(case):
    """(rows, columns) of the stored A, B and of C and D."""
    m, n, k = case["m"], case["n"], case["k"]
    ta, tb = case["layout"][0] == "t", case["layout"][1] == "t"
    return ((k, m) if ta else (m, k)), ((n, k) if tb else (k, n)), (m, n)


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def matrix(shape):
        rows, cols = shape
        size = (cols, rows + case["pad"])
        if case["dist"] == "normal":
            return torch.randn(size, generator=g, device="cuda", dtype=torch.float32)
        return torch.rand(size, generator=g, device="cuda", dtype=torch.float32).mul_(2).sub_(1)

    a, b, c = _stored(case)
    return matrix(a), matrix(b), (matrix(c) if case["beta"] else None)


def prepare(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    ta, tb = case["layout"][0] == "t", case["layout"][1] == "t"
    a, b, c = _inputs(case, seed)
    d = torch.zeros((n, m + case["pad"]), device="cuda", dtype=torch.float32)
    name = catalog.select(m, n, k, ta, tb)
    kernel = S.Kernel(*catalog.paths(name))
    edges = [S.Kernel(*catalog.paths(e)) for e in catalog.EDGE_KERNEL.get(name, ())]
    if edges:
        kernel.set_edge_kernels(*edges)
    return {"case": case, "kernel": kernel, "edges": edges, "a": _Buffer(a), "b": _Buffer(b),
            "c": None if c is None else _Buffer(c), "d": _Buffer(d), "out": d[:, :m],
            "launch": kernel.launch_noalloc if case["noalloc"] else kernel.launch,
            "ld": dict(lda=a.shape[1], ldb=b.shape[1], ldc=m if c is None else c.shape[1], ldd=d.shape[1])}


def run(state):
    case = state["case"]
    state["launch"](state["a"], state["b"], state["c"], state["d"], case["m"], case["n"], case["k"], case["alpha"],
                    case["beta"], **state["ld"])
    return state["out"]


def work(case):
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": 4 * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2 * m * n * k}


def tolerance(case):
    # FP32 sums of k random terms: against 64 bits the calls measure up to
    # 1.8e-8 * sqrt(k) relative (1.15e-6 at k = 4096, 2.9e-7 at k = 256); four
    # times that, and a last rounding
    return {"rel": 4 * (5e-8 + 1.8e-8 * math.sqrt(case["k"]))}


def exact(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    ta, tb = case["layout"][0] == "t", case["layout"][1] == "t"
    a, b, c = _inputs(case, seed)
    (ra, _), (rb, _), _ = _stored(case)
    a, b = a[:, :ra].double(), b[:, :rb].double()      # A and B, transposed
    a, b = (a.t() if ta else a), (b.t() if tb else b)  # op(A)^T and op(B)^T
    d = case["alpha"] * (b.contiguous() @ a.contiguous())
    if c is not None:
        d += case["beta"] * c[:, :m].double()
    return d
