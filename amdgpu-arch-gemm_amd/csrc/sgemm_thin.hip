// FP32 GEMM with a thin D (gfx950): m or n at most 16, so that the call is one
// pass over the large operand and bounded by memory.
//
// X is the large operand (op(A) when n is thin, op(B)^T when m is), Y the thin
// one.  A work-group owns 16 * XA rows of X and all of Y; its waves take the
// chunks of 64 k in turn, each multiplying its chunks from registers
// (v_mfma_f32_16x16x4_f32, no LDS, no barrier) with the next chunk's loads in
// flight, and the waves' sums meet in LDS once, in wave order.  No K split over
// work-groups: D needs no workspace and no second pass.
//
// What bounds it is the X stream: 4096 x 16 x 4096 TN, 67 MB, 15.7 -> 14.4 us;
// 10176 x 10 x 7616 NT, 310 MB, 89.7 -> 61.6 us (5.0 TB/s; a large copy
// reaches 4.9).  The tile kernels' 16 or 32 wide
// work-groups wait for a K tile's loads before the next one's are issued, and
// K splits add a pass over partial sums: 2.4-3.6 TB/s.
//
// Loads.  Along k (X or Y contiguous in k): lane (r, g) of a wave, r < 16, g < 4,
// reads the float4s k = 16 s + 4 g .. + 3 (s < 4) of row r: 64 contiguous bytes of a
// row per instruction, 256 per chunk.  Along the rows: XA consecutive rows r *
// XA .. of k = 16 s + 4 g + e, XA * 64 contiguous bytes per k.  Step (s, e) of
// the MFMA sequence multiplies k = 16 s + 4 g + e of every lane group g, the same
// permutation for X and Y.
#include "sgemm_internal.hpp"
#include "thin_plan.hpp"

#include <hip/hip_runtime.h>

#include <cstdio>
#include <mutex>

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxDevices = 16;
std::mutex g_mutex;
bool g_loaded[kMaxDevices];

constexpr int CHUNK = 64;
constexpr int BUFFER_RSRC_WORD3 = 0x00020000;

struct Args {
    const float* x;
    const float* y;
    const float* c;
    float* d;
    uint32_t rows, cols, k, ldx, ldy, ldc, ldd;
    float alpha, beta;
};

// Values of W atoms of 16 rows of one operand for a chunk of 64 k.
template <int W, bool KC> struct Operand {
    const float* base;
    uint32_t ld, last, row[W];
    uint64_t extent;   // floats from base to past the operand's last element

    __device__ __forceinline__ void init(const float* p, uint32_t ld_, uint32_t row0, uint32_t rows, uint32_t k, int lane) {
        ld = ld_;
        base = KC ? p + (size_t)row0 * ld : p + row0;
        extent = KC ? (uint64_t)(rows - 1 - row0) * ld + k : (uint64_t)(k - 1) * ld + (rows - row0);
        last = rows - 1 - row0;
#pragma unroll
        for (int i = 0; i < W; ++i) {
            // rows past the last one repeat it (k contiguous), or start the
            // last W-row piece again (rows contiguous; its own tail past the
            // operand's end reads 0): their results are not stored
            const uint32_t r = KC ? (uint32_t)(i * 16 + (lane & 15)) : (uint32_t)((lane & 15) * W);
            row[i] = KC ? (r < last ? r : last) : (r < last ? r : last / W * W);
        }
    }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(uint32_t k0, bool on) const {
        const float* p = KC ? base + k0 : base + (size_t)k0 * ld;
        const uint64_t left = (extent - (KC ? (uint64_t)k0 : (uint64_t)k0 * ld)) * 4u;
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0,
                                                 on ? (int)(left < 0x7fffffffu ? left : 0x7fffffffu) : 0, BUFFER_RSRC_WORD3);
    }
    // v[s][e][i]: k = k0 + 16 s + 4 g + e of atom i's row; on == false: zeros, nothing is read
    __device__ __forceinline__ void load(uint32_t k0, bool on, int lane, float (&v)[4][4][W]) const {
        const __amdgpu_buffer_rsrc_t rs = rsrc(on ? k0 : 0u, on);
        const uint32_t g = (uint32_t)lane >> 4;
        if constexpr (KC) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < W; ++i) {
                    const f32x4 t = __builtin_bit_cast(
                        f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)((row[i] * ld + g * 4u) * 4u + s * 64u), 0, 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[s][e][i] = t[e];
                }
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int off = (int)((row[0] + g * 4u * ld) * 4u);
                    const int so = __builtin_amdgcn_readfirstlane((int)((uint32_t)(16 * s + e) * ld * 4u));
                    if constexpr (W == 1) {
                        v[s][e][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, so, 0));
                    } else if constexpr (W == 2) {
                        const f32x2 t = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, so, 0));
                        v[s][e][0] = t[0]; v[s][e][1] = t[1];
                    } else {
                        const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, so, 0));
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[s][e][i] = t[i];
                    }
                }
        }
    }
    // the last, partial chunk: `rem` values of k, element by element, then zeros
    __device__ __forceinline__ void load_part(uint32_t k0, uint32_t rem, int lane, float (&v)[4][4][W]) const {
        const __amdgpu_buffer_rsrc_t rs = rsrc(k0, true);
        const uint32_t g = (uint32_t)lane >> 4;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t kk = (uint32_t)(16 * s + e) + 4u * g, kc = kk < rem ? kk : rem - 1;
#pragma unroll
                for (int i = 0; i < W; ++i) {
                    const uint32_t r = KC ? row[i] : (row[0] + i < last ? row[0] + i : last);
                    const uint32_t off = KC ? r * ld + kc : r + kc * ld;
                    const float t = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)(off * 4u), 0, 0));
                    v[s][e][i] = kk < rem ? t : 0.0f;
                }
            }
    }
    // row of atom i that lane position r stands for
    __device__ __forceinline__ static constexpr uint32_t place(int i, int r) {
        return KC ? (uint32_t)(i * 16 + r) : (uint32_t)(r * W + i);
    }
};

// X_IS_A: D(x, y) at d[x + y * ldd], else at d[y + x * ldd].
template <int XA, bool XKC, bool YKC, bool X_IS_A>
__global__ void __launch_bounds__(1024) thin_kernel(const Args p) {
    extern __shared__ float red[];   // [wave][i * 4 + q][lane]
    constexpr int PER = XA * 256;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = (int)blockDim.x >> 6;
    // An XCD (work-group b runs on XCD b % 8) owns consecutive tiles: the
    // neighbours that share the 128-byte lines at a tile's edge share an L2
    // (rows contiguous, 16 of them 64 bytes: 4096 x 1 x 4096 NN 21.7 -> 13.9
    // us, 7111 x 2 x 2535 31.4 -> 15.9).
    const uint32_t per = gridDim.x / 8u, more = gridDim.x % 8u, xcd = blockIdx.x % 8u;
    const uint32_t tile = xcd * per + (xcd < more ? xcd : more) + blockIdx.x / 8u;
    const uint32_t x0 = tile * (16u * XA);

    Operand<XA, XKC> ox;
    Operand<1, YKC> oy;
    ox.init(p.x, p.ldx, x0, p.rows, p.k, lane);
    oy.init(p.y, p.ldy, 0u, p.cols, p.k, lane);

    const uint32_t full = p.k / CHUNK, rem = p.k % CHUNK;
    // several sums to an atom where registers allow: shorter chains, smaller
    // errors (15 x 2047 x 1023 TN 2.9e-7 -> 1.6e-7, the tile kernels' 2.1e-7)
    constexpr int SUMS = 4 / XA;
    f32x4 acc[SUMS][XA];
#pragma unroll
    for (int u = 0; u < SUMS; ++u)
#pragma unroll
        for (int i = 0; i < XA; ++i) acc[u][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    float vx[2][4][4][XA], vy[2][4][4][1];
    auto mul = [&](const float (&a)[4][4][XA], const float (&b)[4][4][1]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < XA; ++i)
                    // lane % 16 counts the dimension that D holds contiguously
                    acc[e % SUMS][i] =
                        X_IS_A ? __builtin_amdgcn_mfma_f32_16x16x4f32(b[s][e][0], a[s][e][i], acc[e % SUMS][i], 0, 0, 0)
                               : __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][e][i], b[s][e][0], acc[e % SUMS][i], 0, 0, 0);
    };
    // this wave's chunks: wave, wave + waves, ... of the whole ones
    const uint32_t step = (uint32_t)waves;
    uint32_t c = (uint32_t)wave;
    ox.load(c * CHUNK, c < full, lane, vx[0]);
    oy.load(c * CHUNK, c < full, lane, vy[0]);
    for (; c < full; c += 2 * step) {
        ox.load((c + step) * CHUNK, c + step < full, lane, vx[1]);
        oy.load((c + step) * CHUNK, c + step < full, lane, vy[1]);
        mul(vx[0], vy[0]);
        ox.load((c + 2 * step) * CHUNK, c + 2 * step < full, lane, vx[0]);
        oy.load((c + 2 * step) * CHUNK, c + 2 * step < full, lane, vy[0]);
        mul(vx[1], vy[1]);
    }
    // the partial chunk goes to the wave whose turn it is
    if (rem != 0u && (uint32_t)wave == full % step) {
        ox.load_part(full * CHUNK, rem, lane, vx[0]);
        oy.load_part(full * CHUNK, rem, lane, vy[0]);
        mul(vx[0], vy[0]);
    }
#pragma unroll
    for (int i = 0; i < XA; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float sum = acc[0][i][q];
            if constexpr (SUMS == 2) sum += acc[1][i][q];
            if constexpr (SUMS == 4) sum = (sum + acc[1][i][q]) + (acc[2][i][q] + acc[3][i][q]);
            red[wave * PER + (i * 4 + q) * 64 + lane] = sum;
        }
    __syncthreads();
    for (int t = tid; t < PER; t += (int)blockDim.x) {
        float sum = red[t];
        for (int w = 1; w < waves; ++w) sum += red[w * PER + t];
        const int l = t & 63, q = t >> 6 & 3, i = t >> 8;
        const int line = q + 4 * (l >> 4), along = l & 15;   // MFMA row and column
        const uint32_t x = x0 + Operand<XA, XKC>::place(i, X_IS_A ? along : line);
        const uint32_t y = Operand<1, YKC>::place(0, X_IS_A ? line : along);
        if (x < p.rows && y < p.cols) {
            float v = p.alpha * sum;
            const size_t at = X_IS_A ? (size_t)y * p.ldd + x : (size_t)x * p.ldd + y;
            if (p.beta != 0.0f) v = __builtin_fmaf(p.beta, p.c[X_IS_A ? (size_t)y * p.ldc + x : (size_t)x * p.ldc + y], v);
            p.d[at] = v;
        }
    }
}

template <int XA, bool XKC, bool YKC, bool X_IS_A> hipError_t go(const Args& p, int waves, hipStream_t s) {
    const size_t lds = (size_t)waves * XA * 1024;
    // its own result: hipGetLastError may still hold an earlier call's error
    void* args[] = {const_cast<Args*>(&p)};
    return hipLaunchKernel(reinterpret_cast<const void*>(&thin_kernel<XA, XKC, YKC, X_IS_A>),
                           dim3((p.rows + 16 * XA - 1) / (16 * XA)), dim3(64 * waves), args, lds, s);
}

template <bool XKC, bool YKC, bool X_IS_A> hipError_t pick(const Args& p, const thin::Shape& t, hipStream_t s) {
    // the shapes that thin::choose can give
    if (t.x_atoms == 1) return go<1, XKC, YKC, X_IS_A>(p, t.waves, s);
    if constexpr (XKC == YKC) if (t.x_atoms == 2) return go<2, XKC, YKC, X_IS_A>(p, t.waves, s);
    if constexpr (!XKC) if (t.x_atoms == 4) return go<4, XKC, YKC, X_IS_A>(p, t.waves, s);
    return hipErrorInvalidValue;
}

}  // namespace

int sgemm_internal::thin_launch(const thin::Shape& t, bool trans_a, bool trans_b, const float* dA, const float* dB,
                                const float* dC, float* dD, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                                uint32_t ldb, uint32_t ldc, uint32_t ldd, float alpha, float beta, hipStream_t s) {
    Args p;
    p.x = t.x_is_a ? dA : dB; p.y = t.x_is_a ? dB : dA; p.c = dC; p.d = dD;
    p.rows = t.x_is_a ? m : n; p.cols = t.x_is_a ? n : m; p.k = k;
    p.ldx = t.x_is_a ? lda : ldb; p.ldy = t.x_is_a ? ldb : lda; p.ldc = ldc; p.ldd = ldd;
    p.alpha = alpha; p.beta = beta;
    // op(A) is contiguous along k when A is transposed, op(B) when B is not
    const bool xkc = t.x_is_a ? trans_a : !trans_b, ykc = t.x_is_a ? !trans_b : trans_a;
    hipError_t e;
    if (t.x_is_a) {
        if (xkc) e = ykc ? pick<true, true, true>(p, t, s) : pick<true, false, true>(p, t, s);
        else e = ykc ? pick<false, true, true>(p, t, s) : pick<false, false, true>(p, t, s);
    } else {
        if (xkc) e = ykc ? pick<true, true, false>(p, t, s) : pick<true, false, false>(p, t, s);
        else e = ykc ? pick<false, true, false>(p, t, s) : pick<false, false, false>(p, t, s);
    }
    if (e == hipSuccess) return SGEMM_OK;
    char msg[160];
    snprintf(msg, sizeof(msg), "launch of the thin kernel failed: %s (%d)", hipGetErrorString(e), (int)e);
    return set_error((int)e, msg);
}

int sgemm_internal::thin_prepare() {
    // once per device: the query that loads the code object takes 0.15 ms each time
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) dev = -1;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (dev >= 0 && g_loaded[dev]) return SGEMM_OK;
    hipFuncAttributes a;
    const hipError_t e = hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&thin_kernel<1, true, true, true>));
    if (e == hipSuccess) {
        if (dev >= 0) g_loaded[dev] = true;
        return SGEMM_OK;
    }
    char msg[160];
    snprintf(msg, sizeof(msg), "loading the thin kernels failed: %s (%d)", hipGetErrorString(e), (int)e);
    return set_error((int)e, msg);
}
