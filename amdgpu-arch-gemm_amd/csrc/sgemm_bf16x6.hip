// The library's split-BF16 kernels: the instances of bf16x6_kernel.hpp, in the
// tile order of bf16x6_plan.hpp, for the four operand layouts.
//
//   256 x 128  eight waves of 64 x 64, K tiles of 16 in three LDS buffers: the
//              fewest split operations per MFMA, and the fastest wherever its
//              tiles fill the GPU (4096^3: 213 TFLOP/s)
//   128 x 128  two groups of four 64 x 64 waves, each multiplying every other
//              step of 16 (2048^3: 91 us, against 132 in 256 x 128 tiles)
//   128 x 64   four groups of two 64 x 64 waves: few output tiles
//              (511 x 513 x 16400 in 6 K ranges)
//
// The first two stagger their waves: half of them splits the next tile's
// operands while the other half multiplies (2048^3: 91 us against 92, 8192^3 TT
// 5226 against 5441).

#include "bf16x6_kernel.hpp"
#include "bf16x6_plan.hpp"
#include "sgemm_internal.hpp"

#include <hip/hip_runtime.h>

#include <cstdio>
#include <mutex>

namespace {

using bf16x6::Args;
using bf16x6::Config;

//                                          waves      tiles  K
//                                          m  n  k    m  n   steps, buffers, register sets; group; waves per SIMD; staggered
template <bool TA, bool TB> using T128x128 = Config<2, 2, 2, 2, 2, 2, 3, 1, 4, 2, 1, TA, TB>;
template <bool TA, bool TB> using T128x64 = Config<2, 1, 4, 2, 2, 4, 2, 1, 8, 2, 0, TA, TB>;
template <bool TA, bool TB> using T256x128 = Config<4, 2, 1, 2, 2, 1, 3, 1, 4, 2, 1, TA, TB>;

template <template <bool, bool> class T, int INDEX> constexpr bool matches() {
    typedef T<false, false> G;
    return G::MT0 == bf16x6::kTiles[INDEX].m && G::MT1 == bf16x6::kTiles[INDEX].n &&
           G::KW == bf16x6::kTiles[INDEX].k_waves;
}
static_assert(matches<T128x128, 0>() && matches<T128x64, 1>() && matches<T256x128, 2>(),
              "the instances follow the plan's tile order");

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
bool g_loaded[kMaxDevices];  // devices that hold the kernels

template <template <bool, bool> class T>
hipError_t launch_tile(bool ta, bool tb, const Args& p, hipStream_t stream) {
    // The launch's own result, not hipGetLastError: that may still hold an error
    // of an earlier call of the program.
    const dim3 grid((unsigned)p.nwgx * (unsigned)p.nwgy, p.splits), block(T<false, false>::NT);
    void (*const f)(Args) = ta ? (tb ? bf16x6::kernel<T<true, true>> : bf16x6::kernel<T<true, false>>)
                               : (tb ? bf16x6::kernel<T<false, true>> : bf16x6::kernel<T<false, false>>);
    void* args[] = {const_cast<Args*>(&p)};
    return hipLaunchKernel(reinterpret_cast<const void*>(f), grid, block, args, 0, stream);
}

}  // namespace

int sgemm_internal::bf16x6_launch(int tile, uint32_t splits, bool trans_a, bool trans_b, const float* dA, const float* dB,
                                  const float* dC, float* dD, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                                  uint32_t ldb, uint32_t ldc, uint32_t ldd, float alpha, float beta, float* partials,
                                  uint32_t* tickets, hipStream_t stream) {
    Args p;
    p.a = dA; p.b = dB; p.c = dC; p.d = dD;
    p.m = m; p.n = n; p.k = k; p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.ldd = ldd;
    p.alpha = alpha; p.beta = beta;
    p.nwgx = (int32_t)bf16x6::ceil_div(m, (uint64_t)bf16x6::kTiles[tile].m);
    p.nwgy = (int32_t)bf16x6::ceil_div(n, (uint64_t)bf16x6::kTiles[tile].n);
    p.ws = partials;
    p.tickets = tickets;
    p.splits = splits;
    hipError_t e = hipErrorInvalidValue;
    if (tile == 0) e = launch_tile<T128x128>(trans_a, trans_b, p, stream);
    else if (tile == 1) e = launch_tile<T128x64>(trans_a, trans_b, p, stream);
    else if (tile == 2) e = launch_tile<T256x128>(trans_a, trans_b, p, stream);
    if (e == hipSuccess) return SGEMM_OK;
    char msg[160];
    snprintf(msg, sizeof(msg), "launch of the split-BF16 kernel failed: %s (%d)", hipGetErrorString(e), (int)e);
    return set_error((int)e, msg);
}

int sgemm_internal::bf16x6_prepare() {
    // once per device: the query that loads the code object takes 0.15 ms each time
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = -1;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (dev >= 0 && g_loaded[dev]) return SGEMM_OK;
    hipFuncAttributes a;
    const hipError_t e = hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&bf16x6::kernel<T256x128<false, false>>));
    if (e == hipSuccess) {
        if (dev >= 0) g_loaded[dev] = true;
        return SGEMM_OK;
    }
    char msg[160];
    snprintf(msg, sizeof(msg), "loading the split-BF16 kernels failed: %s (%d)", hipGetErrorString(e), (int)e);
    return set_error((int)e, msg);
}
