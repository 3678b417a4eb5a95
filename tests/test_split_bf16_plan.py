"""The host's choice of split-BF16 launches (csrc/bf16x6_plan.hpp), without a GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include "bf16x6_plan.hpp"
#include <cmath>
#include <cstdio>
#include <random>
using namespace bf16x6;
int main() {
    std::mt19937_64 rng(7);
    auto size = [&](double lo, double hi) {
        return (uint64_t)std::lround(std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi))(rng)));
    };
    int chosen[kTileCount] = {0}, split = 0;
    for (int i = 0; i < 20000; ++i) {
        const uint64_t m = size(1, 200000), n = size(1, 200000), k = size(1, 300000);
        const uint32_t chains = 1 + (uint32_t)(rng() % 16);
        const Choice c = choose(m, n, k, i & 2, i & 1, 256, chains);
        if (c.tile < 0) continue;
        const Tile& t = kTiles[c.tile];
        const uint64_t tiles = ceil_div(m, t.m) * ceil_div(n, t.n);
        bool ok = c.tile < kTileCount && c.splits >= 1 && c.splits <= kMaxSplits && c.us > 0.0;
        // no fewer accumulator chains than asked for, none longer than the limit
        ok = ok && c.splits * t.k_waves >= chains && ceil_div(k, c.splits * (uint64_t)t.k_waves) <= kMaxChain;
        // a split's workspace fits the static scratch; an unsplit launch has none
        if (c.splits > 1)
            ok = ok && c.partial_bytes == tiles * c.splits * t.m * t.n * 4 && c.partial_bytes <= kMaxPartialBytes &&
                 c.ticket_count == tiles && tiles <= kMaxTickets && k / c.splits >= kMinRange;
        else
            ok = ok && c.partial_bytes == 0 && c.ticket_count == 0;
        if (!ok) {
            std::printf("%llu x %llu x %llu chains %u: tile %d splits %u\n", (unsigned long long)m, (unsigned long long)n,
                        (unsigned long long)k, chains, c.tile, c.splits);
            return 1;
        }
        ++chosen[c.tile];
        split += c.splits > 1;
    }
    for (int i = 0; i < kTileCount; ++i)
        if (!chosen[i]) return 2;
    return split ? 0 : 3;
}
"""


def test_every_choice_fits_the_scratch_and_the_chain_rules(tmp_path):
    src = tmp_path / "check.cpp"
    src.write_text(CHECK)
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "amdgpu-arch-gemm_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    ret = subprocess.run([str(exe)], stdout=subprocess.PIPE)
    assert ret.returncode == 0, ret.stdout.decode()


HOST = r"""
#include "sgemm_shim.cpp"
#include <cmath>
#include <random>
static int split_launches = 0;
int sgemm_internal::noalloc_prepare(int) { return SGEMM_OK; }
int sgemm_internal::bf16x6_launch(int, uint32_t, bool, bool, const float*, const float*, const float*, float*, uint32_t,
                                  uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, float, float, float*,
                                  uint32_t*, hipStream_t) { ++split_launches; return SGEMM_OK; }
int sgemm_internal::bf16x6_prepare() { return SGEMM_OK; }
int sgemm_internal::thin_prepare() { return SGEMM_OK; }
int sgemm_internal::thin_launch(const thin::Shape&, bool, bool, const float*, const float*, const float*, float*, uint32_t,
                                uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, float, float, hipStream_t) { return SGEMM_OK; }
void sgemm_internal::noalloc_forget(int, hipStream_t) {}
static sgemm_handle* handle(int tm, int tn, int dk) {
    sgemm_handle* h = new sgemm_handle();
    h->info.tile_m = tm; h->info.tile_n = tn; h->info.depth_k = dk; h->info.workitems = 256;
    h->info.split_k = 0; h->info.split_k_max = SGEMM_MAX_SPLIT_K;
    h->compute_units = 256; h->resident = 256; h->split_bf16 = true;
    return h;
}
"""

STRIPS = HOST + r"""
int main() {
    // the catalog's 256 x 256 instance and its edge pair
    sgemm_handle *h = handle(256, 256, 24), *rows = handle(16, 128, 64), *cols = handle(64, 16, 64);
    if (sgemm_set_edge_kernels(h, rows, cols)) return 2;
    std::mt19937 rng(3);
    auto size = [&](double lo, double hi) { return (uint32_t)std::lround(std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi))(rng))); };
    int strips = 0, wide = 0;
    for (int i = 0; i < 400000; ++i) {
        const uint32_t m = size(129, 3000) / 128 * 128 + 128 + rng() % 17, n = size(1000, 1.6e7), k = size(144, 2000);
        const uint32_t ld = m > k ? m : k;
        if (sgemm_check_shape(h, m, n, k, m, k, m, m)) continue;
        const sgemm_internal::SplitPlan p = sgemm_internal::split_plan(h, m, n, k, m, k, m, m, 1.0f, 0.0f);
        if (p.tile < 0) continue;
        sgemm_internal::Part parts[2];
        const int count = sgemm_internal::split_strips(h, p, m, n, m, k, m, m, parts);
        wide += n > 65535u * 128u;
        strips += count;
        for (int q = 0; q < count; ++q)
            if (sgemm_check_shape(parts[q].kh, parts[q].m, parts[q].n, k, m, k, m, m)) {
                std::printf("%u x %u x %u (ld %u): strip %u x %u: %s\n", m, n, k, ld, parts[q].m, parts[q].n, sgemm_last_error());
                return 1;
            }
    }
    return strips && wide ? 0 : 3;
}
"""


def _build_and_run(tmp_path, name, text):
    src, exe = tmp_path / (name + ".cpp"), tmp_path / name
    src.write_text(text)
    csrc = os.path.join(ROOT, "amdgpu-arch-gemm_amd", "csrc")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", csrc, "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(rocm, "include"), str(src), "-o", str(exe), "-L", os.path.join(rocm, "lib"), "-lamdhip64",
                    "-Wl,-rpath," + os.path.join(rocm, "lib"), "-pthread"], check=True)
    ret = subprocess.run([str(exe)], stdout=subprocess.PIPE)
    assert ret.returncode == 0, (ret.returncode, ret.stdout.decode())


def test_no_strip_goes_to_an_edge_kernel_that_refuses_it(tmp_path):
    """A launch that the handle's own kernel accepts is not refused for a strip
    that the split plan alone would cut (the edge kernel's grid ends at 65535
    of its narrower tiles)."""
    _build_and_run(tmp_path, "strips", STRIPS)


# HIP calls that sgemm_launch makes, answered here
WORKSPACE = HOST + r"""
static bool capturing = false, memory = true;
static int own_launches = 0, allocations = 0;
static char block[64];
extern "C" {
hipError_t hipMalloc(void** p, size_t) { if (!memory) return hipErrorOutOfMemory; ++allocations; *p = block; return hipSuccess; }
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 hipStream_t, void**, void**) { ++own_launches; return hipSuccess; }
}
int main() {
    // 16384 x 128 x 4096: 256 tiles of 128 x 64, no K ranges on the handle's own kernel
    sgemm_handle* h = handle(128, 64, 64);
    const uint32_t m = 16384, n = 128, k = 4096;
    float *a = (float*)(1ull << 40), *b = a + (1u << 28), *d = b + (1u << 28);
    const sgemm_internal::SplitPlan p = sgemm_internal::split_plan(h, m, n, k, m, k, m, m, 1.0f, 0.0f);
    if (p.tile < 0 || p.splits < 2 || sgemm_internal::plan(h, m, n, k).partial_bytes) return 2;
    auto launch = [&](int split, int own) {
        split_launches = own_launches = 0;
        const int r = sgemm_launch(h, a, b, nullptr, d, m, n, k, m, k, m, m, 1.0f, 0.0f);
        if (r == SGEMM_OK && split_launches == split && own_launches == own) return true;
        std::printf("returned %d (%s), %d split, %d own launches, expected %d, %d\n", r, sgemm_last_error(), split_launches,
                    own_launches, split, own);
        return false;
    };
    capturing = true;
    if (!launch(0, 1) || allocations) return 3;    // the first launch, captured
    capturing = false, memory = false;
    if (!launch(0, 1)) return 4;                   // no memory for the workspace
    memory = true;
    if (!launch(1, 0) || allocations != 2) return 5;
    if (!launch(1, 0) || allocations != 2) return 6;
    capturing = true;
    if (!launch(0, 1)) return 7;                   // a graph holds no workspace
    return 0;
}
"""


def test_a_split_launch_without_a_workspace_runs_the_handles_own_kernel(tmp_path):
    _build_and_run(tmp_path, "workspace", WORKSPACE)
