// FP32 column-major GEMM on the BF16 matrix cores (gfx950): D = alpha * op(A) *
// op(B) + beta * C with every FP32 operand value split into three BF16 terms
// and six of their nine products summed in FP32.
//
// The split.  x = x1 + x2 + x3, x1 = bf16(x), x2 = bf16(x - x1), x3 = x - x1 -
// x2: both differences are exact in FP32 and the last one has at most 8
// significant bits, so the three terms hold all 24 bits of x.  The products
// a3 b1, a2 b2, a1 b3, a2 b1, a1 b2 go, smallest first, into one FP32 accumulator,
// a1 b1 into another (v_mfma_f32_32x32x16_bf16), and the two are added after the
// K loop; a2 b3, a3 b2 and a3 b3, together at most 2^-24 |a b| and of random
// sign, are left out.
//
// Accuracy.  a1 b1 has 16 bits, so few of its sums round, and the small
// products' sums round 2^-8 lower.  (In one accumulator, as these kernels had
// it first, each of the six products is rounded at the full sum's size, some bits
// below it are cut off downwards, and operands with zeros were up to 2.07 times
// further from 64 bits than on the FP32 MFMAs, v_mfma_f32_32x32x2_f32, which
// round once per two products.)  Relative error (2-norm) against 64 bits, this
// kernel / the FP32 kernel, M = N = 4096:
//   N(0,1), K = 256 / 1024 / 4096 / 24576   8.9e-8 / 1.9e-7 / 4.0e-7 / 1.0e-6
//                                           2.9e-7 / 5.7e-7 / 1.1e-6 / 2.8e-6
//   |N|, any sign, the same                 8.4e-8 / 1.6e-7 / 3.0e-7 / 8.4e-7
//                                           2.2e-7 / 4.3e-7 / 8.4e-7 / 2.4e-6
//   K = 4096, A rectified / 256 / 16 / 2 nonzeros to a column of B
//                                           3.2e-7 / 1.1e-7 / 3.4e-8 / 2.6e-8
//                                           8.1e-7 / 2.9e-7 / 7.4e-8 / 3.1e-8
// What stays behind is the product left out: an output of a single nonzero product
// is 2.6e-8 off (at most 1.8 * 2^-24 of it), a correctly rounded one 2.5e-8; so are
// outputs of a few nonzeros that fall into different K waves or ranges (1.04
// times the FP32 kernel's at four).
//
// Range.  BF16 has FP32's exponents, so no value loses range, but the low
// terms of a value below 2^-110 would fall under BF16's smallest subnormal:
// operands are scaled by 2^16 each before the split (exact), which puts the
// lowest bit of every FP32 number, subnormals included, on a BF16 one; the
// sums are unscaled by 2^-32 in the epilogue.  Where that scaling overflows,
// or where an operand is infinite or NaN, some accumulator of the tile is not
// finite (Inf - Inf = NaN in the split); the work-group then finds one and
// runs its K range again with FP32 MFMAs on the unsplit values, so the result
// is the one the FP32 kernels give.
//
// Rate.  Six BF16 products replace an FP32 MFMA step that takes 16 times as
// long per product: 2.5 PFLOP/s / 6 = 419 TFLOP/s against 157.  What bounds
// these kernels is power, and between the matrix instructions the splitting and the
// LDS: 4096^3 635-645 us back to back (213 TFLOP/s; the FP32 kernel 902), the matrix
// cores 68% busy at 1.82 GHz of 2.4.
//
// Registers.  Two accumulators are what a 256 x 256 tile has no registers for (512
// KB a CU); with one it took 580 us at 4096^3, 10 to 20% less than 256 x 128 tiles.
//
// Data path per K tile of KS steps of 16:
//   HBM --buffer_load--> VGPR (FP32) --split--> LDS, three BF16 planes --> MFMA
// Each element is split once per work-group, by the thread that loads it: a
// unit is one row of op(A) or column of op(B) by 8 values of k, 6.5 VALU
// operations each, that run beside the other wave's MFMAs.  LDS holds plane
// by plane [k group of 8][row][8 values]: 16-byte writes and reads of
// consecutive rows, no bank conflicts (the k groups are padded apart so that
// threads that load k first write to distinct banks).
//
// K permutation: k group kg of a tile of depth DK holds k = 4 kg .. 4 kg + 3
// and DK / 2 + 4 kg .. + 3, the same for A and B, so that the two float4 loads
// of a unit along k each cover whole 64- or 128-byte pieces with their
// neighbours.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bf16x6 {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int BUFFER_RSRC_WORD3 = 0x00020000;
constexpr int CPOL_NT = 0x2;
constexpr int CPOL_SC1 = 0x10;
constexpr int XCDS = 8;

constexpr float SCALE = 65536.0f;                      // 2^16
constexpr float UNSCALE = 1.0f / (65536.0f * 65536.0f);  // 2^-32

template <int WG0_, int WG1_, int KW_, int WT0_, int WT1_, int KS_, int NBUF_, int PD_, int WGM_, int OCC_, int PP_, bool TA_, bool TB_>
struct Config {
    static constexpr int WG0 = WG0_, WG1 = WG1_, KW = KW_, WT0 = WT0_, WT1 = WT1_, KS = KS_, NBUF = NBUF_, PD = PD_;
    static constexpr int WGM = WGM_, OCC = OCC_;
    static constexpr bool TA = TA_, TB = TB_, PINGPONG = PP_ != 0;
    static constexpr int NT = WG0 * WG1 * KW * 64;
    static constexpr int MT0 = 32 * WG0 * WT0, MT1 = 32 * WG1 * WT1;
    static constexpr int DK = 16 * KS, KG = 2 * KS;
    static constexpr int PAD = 128 / KG;                 // bytes
    static constexpr int A_KG = MT0 * 16 + PAD, B_KG = MT1 * 16 + PAD;  // bytes per k group
    static constexpr int A_PLANE = KG * A_KG, B_PLANE = KG * B_KG;
    static constexpr int A_BYTES = 3 * A_PLANE, B_BYTES = 3 * B_PLANE;
    static constexpr int STAGE = A_BYTES + B_BYTES;
    static constexpr int RING = NBUF * STAGE;
    static constexpr int CHUNKS = WT0 * WT1 * 4;         // float4s of a wave's accumulators per lane
    static constexpr int OWN = CHUNKS / KW;              // of them, those the wave stores
    static constexpr int REDUCE = KW > 1 ? KW * MT0 * MT1 * 4 : 0;
    static constexpr int LDS = RING > REDUCE ? RING : REDUCE;
    static constexpr int UA = (MT0 * KG + NT - 1) / NT, UB = (MT1 * KG + NT - 1) / NT;
    static_assert(KS % KW == 0 && CHUNKS % KW == 0, "whole shares per K wave");
    static_assert(LDS + 16 <= 163840, "LDS of a gfx950 CU");
};

__device__ __forceinline__ int xcd_order(int lin, int total) {
    const int x = lin % XCDS, q = total / XCDS, r = total % XCDS;
    return x * q + (x < r ? x : r) + lin / XCDS;
}

template <int WGM> __device__ __forceinline__ void tile_coords(int z, int nwgx, int nwgy, int& tx, int& ty) {
    const int span = WGM * nwgy;
    const int group = z / span;
    const int first_x = group * WGM;
    const int rem = nwgx - first_x;
    const int width = rem < WGM ? rem : WGM;
    const int in_group = z - group * span;
    tx = first_x + in_group % width;
    ty = in_group / width;
}

// x0, x1 -> packed bf16 pair, and the remainders
__device__ __forceinline__ uint32_t split_pair(float& x0, float& x1) {
    const f32x2 v = {x0, x1};
    const bf16x2 h = __builtin_convertvector(v, bf16x2);
    const uint32_t u = __builtin_bit_cast(uint32_t, h);
    x0 -= __builtin_bit_cast(float, u << 16);
    x1 -= __builtin_bit_cast(float, u & 0xffff0000u);
    return u;
}

struct Args {
    const float* a;
    const float* b;
    const float* c;
    float* d;
    uint32_t m, n, k, lda, ldb, ldc, ldd;
    float alpha, beta;
    int32_t nwgx, nwgy;
    float* ws;
    uint32_t* tickets;
    uint32_t splits;
};

// One operand's share of a K tile: R rows of op() by DK values of k.
template <int R, bool KC, int KS, int NT, int U> struct Loader {
    static constexpr int DK = 16 * KS, KG = 2 * KS;
    static constexpr int KGB = R * 16 + 128 / KG;
    const float* base;   // first row of the tile, k = 0
    uint32_t ld;
    uint32_t voff[U];
    uint32_t soff[U];    // MC: byte offset of the unit's first k
    int lds[U];
    int kg[U];
    uint32_t foot;

    __device__ __forceinline__ void init(const float* p, uint32_t ld_, uint32_t row0, uint32_t rows, int tid) {
        ld = ld_;
        base = KC ? p + (size_t)row0 * ld : p + row0;
        const uint32_t last = rows - 1 - row0;   // row0 < rows
        foot = KC ? ((uint32_t)(R - 1) * ld + DK) * 4u : ((uint32_t)(DK - 1) * ld + R) * 4u;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int u = tid + i * NT;
            int r;
            if constexpr (KC) {
                r = u / KG; kg[i] = u % KG;
            } else {
                // R is a multiple of the wave: one k group per wave
                r = u % R; kg[i] = __builtin_amdgcn_readfirstlane(tid >> 6) * 64 / R + i * (NT / R);
            }
            const uint32_t rc = (uint32_t)r < last ? (uint32_t)r : last;
            voff[i] = KC ? (rc * ld + (uint32_t)kg[i] * 4u) * 4u : rc * 4u;
            soff[i] = KC ? 0u : (uint32_t)kg[i] * 4u * ld * 4u;
            lds[i] = kg[i] * KGB + r * 16;
        }
    }
    __device__ __forceinline__ static constexpr bool live(int i, int tid) {
        return (R * KG) % NT == 0 || tid + i * NT < R * KG;
    }
    // the whole K tile from k0; on == false: nothing is read, values are 0
    __device__ __forceinline__ void load(int i, uint32_t k0, bool on, float (&raw)[U][8], int tid) const {
        const float* p = KC ? base + k0 : base + (size_t)k0 * ld;
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, on ? (int)foot : 0, BUFFER_RSRC_WORD3);
        if (!live(i, tid)) return;
        if constexpr (KC) {
            const f32x4 v0 = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)voff[i], 0, 0));
            const f32x4 v1 = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(voff[i] + DK * 2), 0, 0));
#pragma unroll
            for (int j = 0; j < 4; ++j) { raw[i][j] = v0[j]; raw[i][4 + j] = v1[j]; }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane(
                    (int)(soff[i] + (uint32_t)(j < 4 ? j : DK / 2 + j - 4) * (ld * 4u)));
                raw[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)voff[i], (int)so, 0));
            }
        }
    }
    // a partial K tile of `rem` values of k from k0: the others are 0
    __device__ __forceinline__ void load_part(uint32_t k0, uint32_t rem, float (&raw)[U][8], int tid) const {
        const float* p = KC ? base + k0 : base + (size_t)k0 * ld;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)foot, BUFFER_RSRC_WORD3);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if (!live(i, tid)) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t kk = (uint32_t)(kg[i] * 4 + (j < 4 ? j : DK / 2 + j - 4));
                const uint32_t kc = kk < rem ? kk : rem - 1;
                const uint32_t row = KC ? voff[i] - (uint32_t)kg[i] * 16u : voff[i];
                const uint32_t off = row + (KC ? kc * 4u : kc * ld * 4u);
                const float x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0));
                raw[i][j] = kk < rem ? x : 0.0f;
            }
        }
    }
};

// Orders up to `n` vector ALU instructions next (the builtin's count is a constant).
__device__ __forceinline__ void order_valu(int n) {
    if (n >= 9) __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
    else if (n >= 5) __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
    else if (n == 4) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    else if (n == 3) __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
    else if (n == 2) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    else if (n == 1) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
}

template <int V> struct Int { static constexpr int value = V; };
template <bool V> struct Flag { static constexpr bool value = V; };

// After the K loop: the K waves' sums meet, a split launch's ranges meet, D is written.
template <class G>
__device__ __forceinline__ void finish(const Args& p, unsigned char* lds, f32x16 (&acc)[G::WT0][G::WT1], int tid, int lane,
                                       int wm, int wn, int wk, int tx, int ty, uint32_t row0, uint32_t col0, float unscale) {
    constexpr int NT = G::NT, MT0 = G::MT0, MT1 = G::MT1, KW = G::KW, WT0 = G::WT0, WT1 = G::WT1;
    const int r = lane & 31, g = lane >> 5;
    // The wave's share of the tile: chunks of four columns of D at one row of
    // each atom along m.  Atoms are counted fastest, so that neighbouring rows
    // of a column are stored one after the other.
    const int c0 = KW > 1 ? wk * G::OWN : 0;
    f32x4 own[G::OWN];
    if constexpr (KW > 1) {
        // the K waves' sums meet in LDS and are added in wave order
        constexpr int CHUNKS = G::CHUNKS;
        f32x4* red = reinterpret_cast<f32x4*>(lds) + (size_t)(wn * G::WG0 + wm) * KW * CHUNKS * 64 + lane;
#pragma unroll
        for (int i = 0; i < WT0; ++i)
#pragma unroll
            for (int j = 0; j < WT1; ++j)
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    red[(wk * CHUNKS + (j * 4 + h) * WT0 + i) * 64] =
                        f32x4{acc[i][j][4 * h], acc[i][j][4 * h + 1], acc[i][j][4 * h + 2], acc[i][j][4 * h + 3]};
        __syncthreads();
#pragma unroll
        for (int c = 0; c < G::OWN; ++c) {
            own[c] = red[(c0 + c) * 64];
#pragma unroll
            for (int w = 1; w < KW; ++w) own[c] += red[(w * CHUNKS + c0 + c) * 64];
        }
    } else {
#pragma unroll
        for (int c = 0; c < G::OWN; ++c) {
            const int i = c % WT0, j = c / WT0 / 4, h = c / WT0 % 4;
            own[c] = f32x4{acc[i][j][4 * h], acc[i][j][4 * h + 1], acc[i][j][4 * h + 2], acc[i][j][4 * h + 3]};
        }
    }

    if (p.splits > 1) {
        constexpr uint32_t PART = (uint32_t)MT0 * MT1 * 4;   // bytes of one partial
        const uint32_t tile = (uint32_t)tx + (uint32_t)ty * (uint32_t)p.nwgx;
        float* ws = p.ws + (size_t)tile * p.splits * (MT0 * MT1);
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(ws, (short)0, (int)(p.splits * PART), BUFFER_RSRC_WORD3);
#pragma unroll
        for (int c = 0; c < G::OWN; ++c) own[c] *= unscale;
        // every product is computed before the first store: a 16-byte store
        // with a scalar offset may still be reading its last register when the
        // next instruction writes it (seen as a wrong fourth float)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < G::OWN; ++c) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, own[c]), rs, tid * 16,
                                                   (int)(blockIdx.y * PART) + c * NT * 16, CPOL_SC1);
        }
        unscale = 1.0f;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __shared__ uint32_t arrived;
        __syncthreads();
        if (tid == 0) arrived = __hip_atomic_fetch_add(p.tickets + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (arrived + 1 != p.splits) return;
        auto read_part = [&](uint32_t sp, int c) __attribute__((always_inline)) {
            return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 rs, tid * 16, (int)(sp * PART) + c * NT * 16, CPOL_SC1));
        };
#pragma unroll
        for (int c = 0; c < G::OWN; ++c) own[c] = read_part(0, c);
        for (uint32_t sp = 1; sp < p.splits; ++sp) {
#pragma unroll
            for (int c = 0; c < G::OWN; ++c) own[c] += read_part(sp, c);
        }
        if (tid == 0) __hip_atomic_store(p.tickets + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    const float factor = p.alpha * unscale;
    const uint32_t wrow = row0 + (uint32_t)(wm * 32 * WT0), wcol = col0 + (uint32_t)(wn * 32 * WT1);
    auto sub_rsrc = [&](const float* base, uint32_t ld) __attribute__((always_inline)) {
        const uintptr_t at = reinterpret_cast<uintptr_t>(base) + ((uint64_t)wcol * ld + wrow) * 4u;
        const uintptr_t end = reinterpret_cast<uintptr_t>(base) + ((uint64_t)(p.n - 1) * ld + p.m) * 4u;
        const uint64_t foot = ((uint64_t)(32 * WT1 - 1) * ld + 32 * WT0) * 4u;
        const uint64_t left = end > at ? (uint64_t)(end - at) : 0u;
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at), (short)0,
                                                 (int)(left < foot ? left : foot), BUFFER_RSRC_WORD3);
    };
    const __amdgpu_buffer_rsrc_t rsd = sub_rsrc(p.d, p.ldd);
    const __amdgpu_buffer_rsrc_t rsc = sub_rsrc(p.beta != 0.0f ? p.c : p.d, p.beta != 0.0f ? p.ldc : p.ldd);
    // Element e of chunk (j * 4 + h) * WT0 + i: row i * 32 + r, column j * 32 + 8 h + 4 g + e,
    // one dword per lane: 32 consecutive rows, whole 128-byte lines.  Columns
    // past n lie past the descriptor's end, rows past m get an offset that
    // does: the range check, which counts the scalar offset too, drops both, so edge
    // tiles run the same code.
    constexpr uint32_t NOWHERE = 0x80000000u;
    const uint32_t voc = ((uint32_t)(4 * g) * p.ldc + (uint32_t)r) * 4u, vod = ((uint32_t)(4 * g) * p.ldd + (uint32_t)r) * 4u;
    static_assert(G::OWN % WT0 == 0, "a share holds every atom along m");
    // With one wave's stores down whole columns the L2 joins the pieces of a
    // line that columns off a 128-byte boundary leave (5399 x 4428 x 267 in
    // tiles of 256 x 256, which are gone: 92 us, against 105 with streaming stores and
    // 130 with the atoms' rows stored far apart); shares of K waves are spread thinner and gain
    // 2-3% from streaming.
    constexpr int STORE_POLICY = KW > 1 ? CPOL_NT : 0;
    auto chunk_row = [&](int c) __attribute__((always_inline)) { return (uint32_t)(c % WT0) * 32u; };
    auto chunk_col = [&](int c) __attribute__((always_inline)) { return (uint32_t)((c0 + c) / WT0) * 8u; };
    // C in batches of CB chunks, each batch's loads ahead of its use: a load
    // at a time would wait for memory 4 * OWN times
    constexpr int CB = G::OWN < 8 ? G::OWN : 8;
    static_assert(G::OWN % CB == 0 && CB % WT0 == 0, "whole batches of whole columns");
    auto store_batch = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int q = b; q < b + CB; q += WT0)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = q; c < q + WT0; ++c) {
                    const float x = own[c][e];
                    __builtin_amdgcn_raw_buffer_store_b32(
                        __builtin_bit_cast(uint32_t, x), rsd, (int)(wrow + chunk_row(c) + (uint32_t)r < p.m ? vod : NOWHERE),
                        (int)((chunk_col(c) + (uint32_t)e) * p.ldd * 4u + chunk_row(c) * 4u), STORE_POLICY);
                }
    };
    if (p.beta == 0.0f) {
#pragma unroll
        for (int c = 0; c < G::OWN; ++c) own[c] *= factor;
#pragma unroll
        for (int b = 0; b < G::OWN; b += CB) store_batch(b);
        return;
    }
    float cv[2][CB][4];
    auto load_batch = [&](int b, float (&v)[CB][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[c][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                              rsc, (int)voc, (int)((chunk_col(b + c) + (uint32_t)e) * p.ldc * 4u + chunk_row(b + c) * 4u), 0));
    };
    load_batch(0, cv[0]);
#pragma unroll
    for (int b = 0; b < G::OWN; b += CB) {
        if (b + CB < G::OWN) load_batch(b + CB, cv[b / CB + 1 & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) own[b + c][e] = __builtin_fmaf(p.beta, cv[b / CB & 1][c][e], factor * own[b + c][e]);
        store_batch(b);
    }
}

template <class G>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(G::OCC, G::OCC))) kernel(const Args p) {
    constexpr int NT = G::NT, MT0 = G::MT0, MT1 = G::MT1, KS = G::KS, NBUF = G::NBUF, DK = G::DK, KW = G::KW;
    constexpr int WT0 = G::WT0, WT1 = G::WT1;
    __shared__ __attribute__((aligned(16))) unsigned char lds[G::LDS];

    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % G::WG0, wn = wave / G::WG0 % G::WG1, wk = wave / (G::WG0 * G::WG1);
    int tx, ty;
    tile_coords<G::WGM>(xcd_order((int)blockIdx.x, p.nwgx * p.nwgy), p.nwgx, p.nwgy, tx, ty);
    const uint32_t row0 = (uint32_t)tx * MT0, col0 = (uint32_t)ty * MT1;

    Loader<MT0, G::TA, KS, NT, G::UA> la;
    Loader<MT1, !G::TB, KS, NT, G::UB> lb;
    la.init(p.a, p.lda, row0, p.m, tid);
    lb.init(p.b, p.ldb, col0, p.n, tid);

    // K tiles [first, first + full) and, in the last range, the partial one
    // after them, which is run first
    const uint32_t all = p.k / DK;
    const uint32_t per = (all + p.splits - 1) / p.splits;
    const uint32_t first = blockIdx.y * per < all ? blockIdx.y * per : all;
    const uint32_t full = first + per < all ? per : all - first;
    const uint32_t rem = blockIdx.y + 1 == p.splits ? p.k % DK : 0u;
    const int has = rem != 0u;
    const int tiles = (int)full + has;

    f32x16 acc[WT0][WT1];

    const int r = lane & 31, g = lane >> 5;
    const int a_rd = (wk * 2 + g) * G::A_KG + (wm * 32 * WT0 + r) * 16;
    const int b_rd = G::A_BYTES + (wk * 2 + g) * G::B_KG + (wn * 32 * WT1 + r) * 16;

    auto kloop = [&](auto f32_tag) __attribute__((always_inline)) {
        constexpr bool F32 = decltype(f32_tag)::value;
        constexpr int PL = F32 ? 2 : 3;   // 16-byte pieces of 8 values of k
        constexpr int PD = G::PD;
        float ra[PD][G::UA][8], rb[PD][G::UB][8];

        auto k_of = [&](int s) __attribute__((always_inline)) { return (first + (uint32_t)(s - has)) * DK; };
        struct Pieces { u32x4 v[3]; };
        // half of a unit's values (two pairs) into its pieces
        auto split_half = [&](int half, const float (&x)[8], Pieces& o) __attribute__((always_inline)) {
            if constexpr (F32) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o.v[half][e] = __builtin_bit_cast(uint32_t, x[4 * half + e]);
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int q = 2 * half + h;
                    float y0 = x[2 * q] * SCALE, y1 = x[2 * q + 1] * SCALE;
#pragma unroll
                    for (int pl = 0; pl < 3; ++pl) o.v[pl][q] = split_pair(y0, y1);
                }
            }
        };
        auto put = [&](unsigned char* dst, int plane_bytes, const Pieces& o) __attribute__((always_inline)) {
#pragma unroll
            for (int pl = 0; pl < PL; ++pl) *reinterpret_cast<u32x4*>(dst + pl * plane_bytes) = o.v[pl];
        };
        // half `half` of unit u (A's units, then B's) to the LDS buffer at buf_off
        auto stage = [&](int u, int half, int buf_off, float (&xa)[G::UA][8], float (&xb)[G::UB][8], Pieces& o)
            __attribute__((always_inline)) {
            if (u < G::UA) {
                if (la.live(u, tid)) {
                    split_half(half, xa[u], o);
                    if (half == 1) put(lds + buf_off + la.lds[u], G::A_PLANE, o);
                }
            } else {
                if (lb.live(u - G::UA, tid)) {
                    split_half(half, xb[u - G::UA], o);
                    if (half == 1) put(lds + buf_off + G::A_BYTES + lb.lds[u - G::UA], G::B_PLANE, o);
                }
            }
        };
        auto load = [&](int u, int s, float (&xa)[G::UA][8], float (&xb)[G::UB][8]) __attribute__((always_inline)) {
            if (u < G::UA) la.load(u, k_of(s), s < tiles, xa, tid);
            else lb.load(u - G::UA, k_of(s), s < tiles, xb, tid);
        };
        constexpr int UNITS = G::UA + G::UB;

        // prologue: NBUF - 1 tiles to LDS, the next PD to registers
        {
            float xa[NBUF - 1][G::UA][8], xb[NBUF - 1][G::UB][8];
#pragma unroll
            for (int s = 0; s < NBUF - 1; ++s) {
                if (s == 0 && has) {
                    la.load_part(k_of(tiles), rem, xa[0], tid);
                    lb.load_part(k_of(tiles), rem, xb[0], tid);
                } else {
#pragma unroll
                    for (int u = 0; u < UNITS; ++u) load(u, s, xa[s], xb[s]);
                }
            }
#pragma unroll
            for (int s = 0; s < PD; ++s)
#pragma unroll
                for (int u = 0; u < UNITS; ++u) load(u, NBUF - 1 + s, ra[s], rb[s]);
#pragma unroll
            for (int s = 0; s < NBUF - 1; ++s)
#pragma unroll
                for (int u = 0; u < UNITS; ++u) {
                    Pieces o;
                    stage(u, 0, s * G::STAGE, xa[s], xb[s], o);
                    stage(u, 1, s * G::STAGE, xa[s], xb[s], o);
                }
        }
        __syncthreads();

        f32x16 low[WT0][WT1];   // sums of the products below a1 b1
#pragma unroll
        for (int i = 0; i < WT0; ++i)
#pragma unroll
            for (int j = 0; j < WT1; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[i][j][q] = low[i][j][q] = 0.0f;

        struct FragA { u32x4 v[PL]; };
        struct FragB { u32x4 v[WT1][PL]; };
        auto read_a = [&](int buf_off, int sub, int i, FragA& f) __attribute__((always_inline)) {
#pragma unroll
            for (int pl = 0; pl < PL; ++pl)
                f.v[pl] = *reinterpret_cast<const u32x4*>(lds + buf_off + a_rd + pl * G::A_PLANE + sub * KW * 2 * G::A_KG + i * 512);
        };
        auto read_b = [&](int buf_off, int sub, FragB& f) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < WT1; ++j)
#pragma unroll
                for (int pl = 0; pl < PL; ++pl)
                    f.v[j][pl] = *reinterpret_cast<const u32x4*>(lds + buf_off + b_rd + pl * G::B_PLANE + sub * KW * 2 * G::B_KG + j * 512);
        };
        // D^T: the B values take the MFMA's row operand, so that a lane's
        // accumulators are columns of D at one row and stores run down columns
        auto mul = [&](int i, const FragA& fa, const FragB& fb) __attribute__((always_inline)) {
            if constexpr (F32) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int j = 0; j < WT1; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                            __builtin_bit_cast(f32x4, fb.v[j][e / 4])[e % 4],
                            __builtin_bit_cast(f32x4, fa.v[e / 4])[e % 4], acc[i][j], 0, 0, 0);
            } else {
                constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
                for (int e = 0; e < 6; ++e)
#pragma unroll
                    for (int j = 0; j < WT1; ++j) {
                        f32x16& sum = e < 5 ? low[i][j] : acc[i][j];
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fb.v[j][PB[e]]),
                                                                      __builtin_bit_cast(bf16x8, fa.v[PA[e]]), sum, 0, 0, 0);
                    }
            }
        };

        constexpr int SUBS = KS / KW, STEPS = SUBS * WT0;
        // the unrolled tiles of one trip: register sets and operand buffers are compile-time
        constexpr int U = 2;
        static_assert(PD <= 2, "one or two register sets");
        // Staggered waves stage either before or after they multiply: their
        // operands are read ahead of the staging, and one set is enough.
        constexpr bool STAGGERED = G::PINGPONG && !F32;
        static_assert(!STAGGERED || (SUBS == 1 && STEPS % 2 == 0 && NBUF >= 3), "operands of a tile in two sets of A, one of B");
        FragA fa[2];
        FragB fb[STAGGERED ? 1 : 2];
        auto read_first = [&](int buf_off, FragA& a, FragB& b) __attribute__((always_inline)) {
            read_b(buf_off, 0, b);
            read_a(buf_off, 0, 0, a);
        };
        if (!STAGGERED) read_first(0, fa[0], fb[0]);
        int cur = 0;                               // LDS offset of tile t's buffer
        int fill = (NBUF - 1) * G::STAGE;          // of the buffer tile t + NBUF - 1 goes to
        auto body = [&](int t, auto uu_tag, auto order_tag) __attribute__((always_inline)) {
            constexpr int UU = decltype(uu_tag)::value;
            constexpr int ORDER = decltype(order_tag)::value;   // 0: interleaved, 1: stage first, 2: multiply first
            constexpr int set = UU % PD;
            const int nxt = cur + G::STAGE == G::RING ? 0 : cur + G::STAGE;
            Pieces o;
            auto stage_all = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < UNITS; ++u) {
                    stage(u, 0, fill, ra[set], rb[set], o);
                    stage(u, 1, fill, ra[set], rb[set], o);
                    load(u, t + NBUF - 1 + PD, ra[set], rb[set]);
                }
            };
            if constexpr (ORDER == 1) {
                read_first(cur, fa[0], fb[0]);
                stage_all();
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (ORDER != 0) __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int sub = 0; sub < SUBS; ++sub) {
#pragma unroll
                for (int i = 0; i < WT0; ++i) {
                    const int step = sub * WT0 + i;
                    const int as = (step + UU * STEPS) & 1;     // operand sets of this step
                    const int bs = STAGGERED ? 0 : (sub + UU * SUBS) & 1;
                    const bool last = step + 1 == STEPS;
                    int reads = 0, items = 0, vmem = 0;
                    if (!last) {
                        reads = PL;
                        if (i + 1 < WT0) {
                            read_a(cur, sub, i + 1, fa[as ^ 1]);
                        } else {
                            read_b(cur, sub + 1, fb[STAGGERED ? 0 : bs ^ 1]);
                            read_a(cur, sub + 1, 0, fa[as ^ 1]);
                            reads += PL * WT1;
                        }
                    } else if (NBUF >= 3 && !STAGGERED) {
                        read_first(nxt, fa[as ^ 1], fb[STAGGERED ? 0 : bs ^ 1]);
                        reads = PL + PL * WT1;
                    }
#pragma unroll
                    for (int q = 0; q < 2 * UNITS; ++q) {
                        if (ORDER != 0 || q * STEPS / (2 * UNITS) != step) continue;
                        stage(q / 2, q % 2, fill, ra[set], rb[set], o);
                        ++items;
                        if (q % 2) {
                            load(q / 2, t + NBUF - 1 + PD, ra[set], rb[set]);
                            vmem += (q / 2 < G::UA ? G::TA : !G::TB) ? 2 : 8;
                        }
                    }
                    mul(i, fa[as], fb[bs]);
                    if constexpr (!F32 && ORDER == 0) {
                        constexpr int NM = 6 * WT1;
                        const int valu = (items * 28 + NM - 1) / NM;
                        const int rper = (reads + NM - 1) / NM, vper = (vmem + NM - 1) / NM;
#pragma unroll
                        for (int q = 0; q < NM; ++q) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            if (q * rper < reads) { if (rper == 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0); else __builtin_amdgcn_sched_group_barrier(0x100, 2, 0); }
                            order_valu(valu);
                            if (q >= NM / 2 && (items > 1 || step % 2)) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                            if (q * vper < vmem) { if (vper == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0); else __builtin_amdgcn_sched_group_barrier(0x020, 2, 0); }
                        }
                    }
                    if (ORDER == 0) __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (ORDER != 0) __builtin_amdgcn_s_setprio(0);
            if constexpr (ORDER == 2) {
                __builtin_amdgcn_sched_barrier(0);
                read_first(nxt, fa[0], fb[0]);
                stage_all();
            }
            fill = cur;
            cur = nxt;
            __syncthreads();
            if constexpr (NBUF == 2) {
                constexpr int as = (STEPS + UU * STEPS) & 1, bs = (SUBS + UU * SUBS) & 1;
                read_first(cur, fa[as], fb[bs]);
            }
        };
        auto run = [&](auto order_tag) __attribute__((always_inline)) {
            if constexpr (decltype(order_tag)::value == 2) read_first(cur, fa[0], fb[0]);
            for (int t = 0; t < tiles; t += U) {
                body(t, Int<0>{}, order_tag);
                if (t + 1 < tiles) body(t + 1, Int<1>{}, order_tag);
            }
        };
        if constexpr (G::PINGPONG && !F32) {
            if (wave < NT / 128) run(Int<1>{});
            else run(Int<2>{});
        } else {
            run(Int<0>{});
        }
        if constexpr (!F32) {
#pragma unroll
            for (int i = 0; i < WT0; ++i)
#pragma unroll
                for (int j = 0; j < WT1; ++j)
#pragma unroll
                    for (int q = 0; q < 16; ++q) acc[i][j][q] += low[i][j][q];
        }
    };

    kloop(Flag<false>{});
    float unscale = UNSCALE;

    // a value that is not finite: see the header
    float z = 0.0f;
#pragma unroll
    for (int i = 0; i < WT0; ++i)
#pragma unroll
        for (int j = 0; j < WT1; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) z = __builtin_fmaf(acc[i][j][q], 0.0f, z);
    if (__syncthreads_or(z != 0.0f)) {
        kloop(Flag<true>{});
        unscale = 1.0f;
    }

    finish<G>(p, lds, acc, tid, lane, wm, wn, wk, tx, ty, row0, col0, unscale);
}

}  // namespace bf16x6
