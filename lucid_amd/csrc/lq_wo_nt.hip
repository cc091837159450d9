// lq_wo_nt.hip -- y[m, k] = sum_n x[m, n] w_hat[n, k] for group-wise packed w_hat[N, K] (groups
// along k): quantized_matmul with transpose=false and the input gradient of the transpose=true
// product, dX = dY dequant(W) (QuantizedMatmulBackward::apply,
// lucid/_C/ops/quantized/QuantizedMatmul.cpp:73-90), on the matrix cores.
//
// The group scale and bias change along the summed axis, so they cannot be taken out of the sums:
// w_hat is formed per element as lq_group_dequantize_f32 writes it, fl32(fl32(c s) + b).  Both operands
// enter v_mfma_f32_16x16x32_bf16 as sums of bfloat16 terms, which have float32's exponents: a float32
// value is exactly three of them (8 bits each), a half value two.  x w is the six products of terms
// that may reach 2^-16 of it (half x: five); what is left out is at most 2^-23 |x| |w|.
// So each product keeps float32's precision whatever lies beside it in its row, column or tile.  Nothing is
// prepared in memory (the call has no workspace): a workgroup splits its own BM x 32 piece of x and 32 x BN
// piece of w_hat per step into LDS, in MFMA fragment order, while it multiplies the pieces of the step
// before; the pieces after come from memory meanwhile.
//
// The terms of a value must be finite and, since these instructions read subnormal terms as 0, not
// far below it.  A tile that meets an infinity, a scale that may make one, or eight values or a scale
// below 2^-100 (but not 0) is computed again with v_mfma_f32_16x16x4_f32 on the float32 values
// themselves, through the same stages: infinities, NaN and subnormals as a float32 sum has them
// (M = 2048, N = K = 4096 with an infinity in every tile: 1025 us in all).  Beside larger ones of its
// eight, a smaller value is exact to 2^-126.
//
// What bounds it: the issue of instructions and the waits around a step's barrier (matrix cores busy
// 38%, VALU 29% of the time; 1.13 PFLOP/s of bf16 products).  Per wave and step of the largest tiles 96
// MFMA (half x: 80) and 290 VALU: conversion to terms 11 per pair of values, one addition per sum, three
// per weight code.  Tiles are as large as the shape allows: 256 x 128 in eight waves of 64 x 64,
// 128 x 128 in waves of 64 x 32, 32 x 64 with the steps split between four groups of four waves.
// N = K = 4096, 4 bits, groups of 64, back to back, against the float32 VALU kernel before (128 x 128
// tiles, 75 of at most 79 TFLOP/s without packed fp32): M = 2048 922 -> 392 us (364 with pauses between
// calls), M = 512 881 -> 229, M = 26 880 -> 64; half x M = 2048 1323 -> 317.  The float32 matrix
// instructions alone took 595, 335 and 73 us.  Two fp16 terms per value (three products, 312, 211 and
// 71 us) need a scale per row and tile, and lost values far below it.  The error against 64 bits at
// M = 2048 fell from 1.1e-6 to 2.3e-7: shorter chains of additions.  Ordering the instructions by hand
// (3 VALU after each MFMA), conversions before the products in half of the waves and after them in the
// others, or a higher priority for the products measured the same or slower.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "lq_dma.h"
#include "lq_internal.h"
#include "lq_wo.h"

namespace lq {
namespace {

struct NtArgs {
    const void* x;
    int64_t ldx;
    const uint8_t* w;      // packed rows
    const float* scales;   // [N][G]
    const float* biases;   // [N][G] or null
    const float* bias;     // [K] or null
    void* y;
    int64_t ldy;
    int M, N, K, G, gs;
    int relu, hmode;
    int64_t tiles_m, tiles_k;
};

constexpr float NT_TINY = 0x1p-100f;

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

// 16-byte slot of (quarter q, row r) in a fragment's 1 KB: the rotation by 4 q spreads the four
// quarters of one row (written by neighbouring lanes) over the banks.
__device__ __forceinline__ int nt_slot(int q, int r) { return q * 16 + ((r + 4 * q) & 15); }

// Eight values as T bfloat16 terms, each the nearest to what those before it leave: their sum is the
// value itself, for float32 with T = 3 and for half with T = 2.
template <int T>
__device__ __forceinline__ void split_terms(const float (&v)[8], vu4 (&term)[T]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        f2 r = {v[2 * p], v[2 * p + 1]};
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, b2));
            term[j][p] = u;
            r[0] -= __uint_as_float(u << 16);
            r[1] -= __uint_as_float(u & 0xFFFF0000u);
        }
    }
}

__device__ __forceinline__ f4 mfma_bf16(vu4 a, vu4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

// VEC: rows of x are 16-byte aligned and N a multiple of 8 (an octet past N re-reads the row's last
// one: its weights are 0).
// GR: wave groups of a workgroup, each with its own steps of the sum (few tiles: shorter chains).
template <int BITS, bool XF32, bool VEC, int WM, int WN, int FM, int FN, int GR>
__global__ __launch_bounds__(64 * WM * WN * GR) void group_matmul_nt_kernel(NtArgs a) {
    constexpr int W = WM * WN, NT = 64 * W, BM = 16 * WM * FM, BN = 16 * WN * FN;
    constexpr int TX = XF32 ? 3 : 2, TW = 3;  // terms of a value of x, of w_hat
    constexpr float L = (float)((1 << BITS) - 1);
    constexpr int XO = (BM * 4 + NT - 1) / NT, WO = BN * 4 / NT;  // octets per thread and step
    static_assert(BN * 4 % NT == 0 && NT % BN == 0 && WO >= 1, "one k per thread");
    constexpr int X_BYTES = BM * 64 * TX, W_BYTES = BN * 64 * TW, STAGE = X_BYTES + W_BYTES;
    constexpr int SBN = BN / 32 * 32;  // pairs per step: up to BN / 32 groups x 32 rows
    __shared__ __attribute__((aligned(1024))) char lds_[GR][2 * STAGE];
    __shared__ __attribute__((aligned(16))) float2 sbuf_[GR][2][SBN];
    static_assert(GR == 1 || (GR - 1) * FM * FN * NT * 16 <= GR * 2 * STAGE, "the groups' sums fit the stages");
    const int grp = GR == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const int tid = threadIdx.x - grp * NT, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    char* const lds = lds_[grp];
    float2 (*const sbuf)[SBN] = sbuf_[grp];
    const int wm = wave / WN, wn = wave % WN;
    const int steps = ((a.N + 31) / 32 + GR - 1) / GR, s0 = grp * steps;  // steps past N add zeros
    const int64_t row_bytes = (int64_t)a.K * BITS / 8;
    const int ngt = max(1, BN / a.gs);  // groups of a tile
    const int64_t tiles = a.tiles_m * a.tiles_k;

    for (int64_t tile0 = blockIdx.x; tile0 < tiles; tile0 += gridDim.x) {
        // consecutive tiles (eight tile rows, column by column) on one XCD: their x and weight
        // pieces meet in its L2
        int64_t tile = tile0;
        if (tiles == (int64_t)gridDim.x) {
            const int64_t per = tiles / 8, rest = tiles % 8, xcd = tile0 % 8;
            tile = xcd * per + min(xcd, rest) + tile0 / 8;
        }
        const int64_t band = tile / (8 * a.tiles_k), h = min((int64_t)8, a.tiles_m - band * 8), in = tile - band * 8 * a.tiles_k;
        const int m0 = (int)(band * 8 + in % h) * BM, k0 = (int)(in / h) * BN;
        __syncthreads();

        // ---- this thread's pieces
        bool bad = false;  // a value whose terms are not finite, or are subnormal
        int xr[XO];
        const int xq = tid & 3;
        const void* xrow[XO];
#pragma unroll
        for (int u = 0; u < XO; ++u) {
            xr[u] = (tid + u * NT) >> 2;
            xrow[u] = static_cast<const uint8_t*>(a.x) + (int64_t)min(m0 + xr[u], a.M - 1) * a.ldx * (XF32 ? 4 : 2);
        }
        // the weight octets' rows are the same for a wave (BN a multiple of 64): scalar addresses
        const int wk = tid % BN, wk_c = BITS == 8 ? min(k0 + wk, a.K - 1) : min(k0 + wk, a.K - 1) >> 1;
        const int oq0 = __builtin_amdgcn_readfirstlane(tid / BN);
        float xv[XF32 ? XO : 1][8];
        h8 xh[XF32 ? 1 : XO];
        uint32_t wv[WO][8];
        float2 sb = make_float2(0.0f, 0.0f);
        auto load = [&](int t) __attribute__((always_inline)) {  // x and codes of step t
#pragma unroll
            for (int u = 0; u < XO; ++u) {
                const int n = VEC ? min((s0 + t) * 32 + xq * 8, a.N - 8) : (s0 + t) * 32 + xq * 8;
                if constexpr (XF32) {
                    const float* p = static_cast<const float*>(xrow[u]) + n;
                    if constexpr (VEC) {
                        const vf4 v0 = reinterpret_cast<const vf4*>(p)[0], v1 = reinterpret_cast<const vf4*>(p)[1];
#pragma unroll
                        for (int i = 0; i < 4; ++i) xv[u][i] = v0[i], xv[u][4 + i] = v1[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i) xv[u][i] = n + i < a.N ? p[i] : 0.0f;
                    }
                } else {
                    const _Float16* p = static_cast<const _Float16*>(xrow[u]) + n;
                    if constexpr (VEC) {
                        xh[u] = *reinterpret_cast<const h8*>(p);
                    } else {
#pragma unroll
                        for (int i = 0; i < 8; ++i) xh[u][i] = n + i < a.N ? p[i] : (_Float16)0.0f;
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < WO; ++u) {
                const int n = (s0 + t) * 32 + (oq0 + u * (NT / BN)) * 8;
#pragma unroll
                for (int i = 0; i < 8; ++i) wv[u][i] = (a.w + (int64_t)min(n + i, a.N - 1) * row_bytes)[wk_c];
            }
        };
        const bool sb_wave = wave * 64 < ngt * 32;
        auto load_sb = [&](int t) __attribute__((always_inline)) {  // a pair of step t, past the end 0
            if (!sb_wave) return;
            const int j = tid >> 5, n = (s0 + t) * 32 + (tid & 31), g = k0 / a.gs + j;
            sb = make_float2(0.0f, 0.0f);
            if (j < ngt && n < a.N && g < a.G) {
                sb.x = a.scales[(int64_t)n * a.G + g];
                sb.y = a.biases ? a.biases[(int64_t)n * a.G + g] : 0.0f;
            }
        };
        auto store_sb = [&](int t) __attribute__((always_inline)) {
            if (sb_wave && (tid >> 5) < ngt) {
                const float s = round_to(sb.x, a.hmode), b = round_to(sb.y, a.hmode);
                bad |= !(fabsf(s) * L + fabsf(b) <= 3.0e38f) || (s != 0.0f && fabsf(s) < NT_TINY);
                sbuf[t & 1][tid] = make_float2(s, b);
            }
        };
        // Step t into LDS: bfloat16 terms, or (EXACT) the float32 values as two pieces of four.
        auto convert = [&](int t, auto exact) __attribute__((always_inline)) {
            constexpr bool EXACT = decltype(exact)::value;
            char* base = lds + (t & 1) * STAGE;
            auto put = [&](vu4* dst, const float (&v)[8], auto terms) __attribute__((always_inline)) {
                constexpr int T = decltype(terms)::value;
                if constexpr (EXACT) {
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        dst[64 * j] = __builtin_bit_cast(vu4, vf4{v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]});
                } else {
                    vu4 term[T];
                    split_terms(v, term);
#pragma unroll
                    for (int j = 0; j < T; ++j) dst[64 * j] = term[j];
                }
            };
#pragma unroll
            for (int u = 0; u < WO; ++u) {
                const int oq = oq0 + u * (NT / BN);
                const float4* p = reinterpret_cast<const float4*>(&sbuf[t & 1][wk / a.gs * 32 + oq * 8]);
                float v[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 s = p[i];  // {s, b} of rows 2 i and 2 i + 1
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const uint32_t c = BITS == 8 ? wv[u][2 * i + j] : (wv[u][2 * i + j] >> (4 * (wk & 1))) & 15u;
                        v[2 * i + j] = (float)(uint8_t)c * (j ? s.z : s.x) + (j ? s.w : s.y);
                    }
                }
                put(reinterpret_cast<vu4*>(base + X_BYTES) + (wk >> 4) * TW * 64 + nt_slot(oq, wk & 15), v,
                    std::integral_constant<int, TW>{});
            }
#pragma unroll
            for (int u = 0; u < XO; ++u) {
                float v[8], am = 0.0f;
                // (a value past N would meet a zero weight: an infinity there must not)
                const bool in = !EXACT || (s0 + t) * 32 + xq * 8 < a.N;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if constexpr (XF32) v[i] = in ? xv[u][i] : 0.0f;
                    else v[i] = in ? (float)xh[u][i] : 0.0f;
                    am = fmaxf(am, fabsf(v[i]));
                }
                bad |= am > (XF32 ? 3.0e38f : 65504.0f) || (XF32 && am != 0.0f && am < NT_TINY);
                if (XO * NT == BM * 4 || xr[u] < BM)
                    put(reinterpret_cast<vu4*>(base) + (xr[u] >> 4) * TX * 64 + nt_slot(xq, xr[u] & 15), v,
                        std::integral_constant<int, TX>{});
            }
        };

        f4 acc[FM][FN];
        const int slot = nt_slot(q, l16);
        auto multiply = [&](int t, auto exact, auto between) __attribute__((always_inline)) {
            constexpr bool EXACT = decltype(exact)::value;
            constexpr int NX = EXACT ? 2 : TX, NW = EXACT ? 2 : TW;
            const vu4* X = reinterpret_cast<const vu4*>(lds + (t & 1) * STAGE) + slot;
            const vu4* Wf = reinterpret_cast<const vu4*>(lds + (t & 1) * STAGE + X_BYTES) + slot;
            vu4 xf[FM][NX];
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int j = 0; j < NX; ++j) xf[m][j] = X[((wm * FM + m) * TX + j) * 64];
            between();
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                vu4 wf[NW];
#pragma unroll
                for (int j = 0; j < NW; ++j) wf[j] = Wf[((wn * FN + n) * TW + j) * 64];
                if constexpr (EXACT) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
#pragma unroll
                        for (int m = 0; m < FM; ++m)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wf[e / 4][e % 4]),
                                                                             __uint_as_float(xf[m][e / 4][e % 4]), acc[m][n], 0, 0, 0);
                } else {
                    // the small products first; one addition to the long sum per step
                    f4 blk[FM];
#pragma unroll
                    for (int m = 0; m < FM; ++m) blk[m] = f4{0.f, 0.f, 0.f, 0.f};
                    auto add = [&](auto ix, auto iw) __attribute__((always_inline)) {
#pragma unroll
                        for (int m = 0; m < FM; ++m) blk[m] = mfma_bf16(wf[decltype(iw)::value], xf[m][decltype(ix)::value], blk[m]);
                    };
                    using I0 = std::integral_constant<int, 0>;
                    using I1 = std::integral_constant<int, 1>;
                    using I2 = std::integral_constant<int, 2>;
                    if constexpr (XF32) add(I2{}, I0{});
                    add(I0{}, I2{});
                    add(I1{}, I1{});
                    add(I1{}, I0{});
                    add(I0{}, I1{});
                    add(I0{}, I0{});
#pragma unroll
                    for (int m = 0; m < FM; ++m) acc[m][n] += blk[m];
                }
            }
        };
        auto walk = [&](auto exact) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int n = 0; n < FN; ++n) acc[m][n] = f4{0.f, 0.f, 0.f, 0.f};
            if (steps <= 0) return;
            load_sb(0);
            load(0);
            store_sb(0);
            load_sb(1);
            __syncthreads();
            convert(0, exact);
            load(min(1, steps - 1));
            store_sb(1);
            load_sb(2);
            for (int t = 0; t < steps; ++t) {
                block_barrier();  // step t's pieces and step t + 1's scales are in LDS
                store_sb(t + 2);
                load_sb(t + 3);
                // the last step converts a step past the end once more: no branch around the products
                multiply(t, exact, [&]() __attribute__((always_inline)) {
                    convert(t + 1, exact);
                    load(min(t + 2, steps - 1));
                });
            }
        };
        walk(std::false_type{});
        if (__syncthreads_or(bad)) {
            walk(std::true_type{});
            __syncthreads();
        }

        // ---- the outputs: the groups' sums meet, added in order
        if constexpr (GR > 1) {
            f4* sums = reinterpret_cast<f4*>(lds_[0]) + tid;
            if (grp > 0) {
#pragma unroll
                for (int i = 0; i < FM * FN; ++i) sums[((grp - 1) * FM * FN + i) * NT] = acc[i / FN][i % FN];
            }
            __syncthreads();
            if (grp > 0) continue;
#pragma unroll
            for (int g = 0; g < GR - 1; ++g)
#pragma unroll
                for (int i = 0; i < FM * FN; ++i) acc[i / FN][i % FN] += sums[(g * FM * FN + i) * NT];
        }
#pragma unroll
        for (int m = 0; m < FM; ++m) {
            const int ml = (wm * FM + m) * 16 + l16, row = m0 + ml;
            if (row >= a.M) continue;
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                const int col = k0 + (wn * FN + n) * 16 + 4 * q;
                if (col >= a.K) continue;  // K is a multiple of 32: whole groups of four
                f4 v = acc[m][n];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[i] = wo_finish(v[i], a.bias != nullptr, a.bias ? a.bias[col + i] : 0.0f, a.relu, a.hmode);
                }
                const int64_t at = (int64_t)row * a.ldy + col;
                if constexpr (XF32) {
                    float* y = static_cast<float*>(a.y) + at;
                    if ((reinterpret_cast<uintptr_t>(y) & 15) == 0) {
                        *reinterpret_cast<f4*>(y) = v;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) y[i] = v[i];
                    }
                } else {
                    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                    _Float16* y = static_cast<_Float16*>(a.y) + at;
                    const h4 o = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                    if ((reinterpret_cast<uintptr_t>(y) & 7) == 0) {
                        *reinterpret_cast<h4*>(y) = o;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) y[i] = o[i];
                    }
                }
            }
        }
    }
}

}  // namespace

void group_matmul_nt_launch(const WoNtCall& c, hipStream_t st) {
    NtArgs a{c.x, c.ldx, c.w, c.scales, c.biases, c.bias, c.y, c.ldy, c.M, c.N, c.K, c.K / c.gs, c.gs, c.relu, c.hmode, 0, 0};
    const bool vec = aligned16(c.x) && c.ldx % (c.xf32 ? 4 : 8) == 0 && c.N % 8 == 0 && c.N >= 8;
    auto go = [&](auto bits, auto xf, auto wm, auto wn, auto fm, auto fn, auto gr, const char* path) {
        constexpr int BM = 16 * decltype(wm)::value * decltype(fm)::value, BN = 16 * decltype(wn)::value * decltype(fn)::value;
        a.tiles_m = ((int64_t)a.M + BM - 1) / BM;
        a.tiles_k = ((int64_t)a.K + BN - 1) / BN;
        const dim3 grid((unsigned)std::min<int64_t>(a.tiles_m * a.tiles_k, 1 << 20));
        const dim3 block(64 * decltype(wm)::value * decltype(wn)::value * decltype(gr)::value);
        if (vec)
            hipLaunchKernelGGL((group_matmul_nt_kernel<decltype(bits)::value, decltype(xf)::value, true, decltype(wm)::value,
                                                       decltype(wn)::value, decltype(fm)::value, decltype(fn)::value, decltype(gr)::value>),
                               grid, block, 0, st, a);
        else
            hipLaunchKernelGGL((group_matmul_nt_kernel<decltype(bits)::value, decltype(xf)::value, false, decltype(wm)::value,
                                                       decltype(wn)::value, decltype(fm)::value, decltype(fn)::value, decltype(gr)::value>),
                               grid, block, 0, st, a);
        note_path(path);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    auto tiles = [&](int bm, int bn) { return (((int64_t)a.M + bm - 1) / bm) * (((int64_t)a.K + bn - 1) / bn); };
    auto pick = [&](auto bits, auto xf) {
        // Rounds of 256 workgroups times a round's time per step, measured at N = 4096 in float32 (us
        // per step; in half all three take about 0.85 of it): 256 x 128 tiles 3.06, 128 x 128 1.94,
        // 32 x 64 with the steps split between four wave groups 0.56.
        auto cost = [&](int bm, int bn, double step) { return (double)((tiles(bm, bn) + 255) / 256) * step; };
        const double c256 = cost(256, 128, 3.06), c128 = cost(128, 128, 1.94), c32 = cost(32, 64, 0.56);
        if (c256 < c128 && c256 < c32) go(bits, xf, I4{}, I2{}, I4{}, I4{}, I1{}, "wo nt 256x128");
        else if (c128 < c32) go(bits, xf, I2{}, I4{}, I4{}, I2{}, I1{}, "wo nt 128x128");
        else go(bits, xf, I2{}, I2{}, I1{}, I2{}, I4{}, "wo nt 32x64");
    };
    using B8 = std::integral_constant<int, 8>;
    using B4 = std::integral_constant<int, 4>;
    if (c.bits == 8) c.xf32 ? pick(B8{}, std::true_type{}) : pick(B8{}, std::false_type{});
    else c.xf32 ? pick(B4{}, std::true_type{}) : pick(B4{}, std::false_type{});
}

}  // namespace lq
