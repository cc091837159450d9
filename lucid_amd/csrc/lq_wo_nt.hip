// lq_wo_nt.hip -- y[m, k] = sum_n x[m, n] w_hat[n, k] for group-wise packed w_hat[N, K] (groups
// along k): quantized_matmul with transpose=false and the input gradient of the transpose=true
// product, dX = dY dequant(W) (QuantizedMatmulBackward::apply,
// lucid/_C/ops/quantized/QuantizedMatmul.cpp:73-90), on v_mfma_f32_16x16x32_f16.
//
// The group scale and bias change along the summed axis, so they cannot be taken out of the sums:
// w_hat is formed per element, w = fma(c, s, b) in fp32, and both operands enter the MFMA as two
// fp16 terms hi + lo (~22 significant bits): x w = hi hi + lo hi + hi lo, fp32 accumulation (half x
// is its own hi term: two products).  Nothing is prepared in memory (the call has no workspace):
// a workgroup splits its own BM x 32 piece of x and 32 x BN piece of w_hat per step into LDS, in
// MFMA fragment order, while it multiplies the pieces of the step before; the pieces after come from
// memory meanwhile.
//
// Exponents.  fp16 terms need values below 2^16 with room for 22 bits under them.  w_hat of a tile
// is scaled by one power of two from the tile's largest |b| and |s L + b| (first pass over the
// scales).  A row of x carries a running power of two: set by its first nonzero step (largest value
// into [2^11, 2^12)), changed only by a step whose largest value leaves [2^-3, 2^15); the sums are
// then multiplied by the change, exactly.  Infinite inputs would turn into NaN by the split: a tile
// that meets one is computed again element by element in fp32.
//
// What bounds it: instruction issue.  Per thread and step 8 values of w_hat (byte load, convert, fma,
// two roundings) and 8 or 16 of x (two fused multiply-round each) beside 24 or 48 MFMA of a wave, so
// tiles are as large as the shape allows: 256 x 128 in eight waves of 64 x 64, 128 x 128 in waves of
// 64 x 32, 32 x 64 with the steps split between four groups of four waves.  Against the float32 VALU
// kernel this replaced (128 x 128 tiles, 75 of at most 79 TFLOP/s without packed fp32), N = K = 4096,
// 4 bits, groups of 64: M = 2048 922 -> 300 us, M = 512 881 -> 209, M = 26 880 -> 69; half x, 8 bits,
// groups of 128: M = 2048 1323 -> 194, M = 26 940 -> 54.  The error against 64 bits fell too
// (M = 2048: 1.1e-6 -> 7.1e-7): shorter chains of additions.
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

constexpr int NT_E_UNSET = 1 << 20;

// 16-byte slot of (quarter q, row r) in a fragment's 1 KB: the rotation by 4 q spreads the four
// quarters of one row (written by neighbouring lanes) over the banks.
__device__ __forceinline__ int nt_slot(int q, int r) { return q * 16 + ((r + 4 * q) & 15); }

__device__ __forceinline__ float pow2(int e) { return __int_as_float((e + 127) << 23); }  // -126 <= e <= 127

// VEC: rows of x are 16-byte aligned and N a multiple of 8 (an octet past N re-reads the row's last
// one: its weights are 0).
// GR: wave groups of a workgroup, each with its own steps of the sum (few tiles: shorter chains).
template <int BITS, bool XF32, bool VEC, int WM, int WN, int FM, int FN, int GR>
__global__ __launch_bounds__(64 * WM * WN * GR) void group_matmul_nt_kernel(NtArgs a) {
    constexpr int W = WM * WN, NT = 64 * W, BM = 16 * WM * FM, BN = 16 * WN * FN;
    constexpr int T = XF32 ? 2 : 1;
    constexpr float L = (float)((1 << BITS) - 1);
    constexpr int XO = (BM * 4 + NT - 1) / NT, WO = BN * 4 / NT;  // octets per thread and step
    static_assert(BN * 4 % NT == 0 && NT % BN == 0 && WO >= 1, "one k per thread");
    constexpr int X_BYTES = BM * 64 * T, W_BYTES = BN * 64 * 2, STAGE = X_BYTES + W_BYTES;
    constexpr int SBN = BN / 32 * 32;  // pairs per step: up to BN / 32 groups x 32 rows
    __shared__ __attribute__((aligned(1024))) char lds_[GR][2 * STAGE];
    __shared__ __attribute__((aligned(16))) float2 sbuf_[GR][2][SBN];
    __shared__ float row_scale_[GR][3][BM];
    __shared__ int row_e_[GR][BM];
    __shared__ int changed_[GR][3];
    __shared__ float wmax[W * GR];
    static_assert(GR == 1 || (GR - 1) * FM * FN * NT * 16 <= GR * 2 * STAGE, "the groups' sums fit the stages");
    const int grp = GR == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const int tid = threadIdx.x - grp * NT, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    char* const lds = lds_[grp];
    float2 (*const sbuf)[SBN] = sbuf_[grp];
    float (*const row_scale)[BM] = row_scale_[grp];
    int* const row_e = row_e_[grp];
    int* const changed = changed_[grp];
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

        // ---- the tile's weight exponent
        float wm_ = 0.0f;
        for (int i = threadIdx.x; i < a.N * ngt; i += NT * GR) {
            const int n = i / ngt, g = k0 / a.gs + i % ngt;
            if (g < a.G) {
                const float s = round_to(a.scales[(int64_t)n * a.G + g], a.hmode);
                const float b = a.biases ? round_to(a.biases[(int64_t)n * a.G + g], a.hmode) : 0.0f;
                wm_ = fmaxf(wm_, fmaxf(fabsf(b), fabsf(__builtin_fmaf(s, L, b))));
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) wm_ = fmaxf(wm_, __shfl_xor(wm_, off, 64));
        if (lane == 0) wmax[grp * W + wave] = wm_;
        if (tid < 3) changed[tid] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < W * GR; ++i) wm_ = fmaxf(wm_, wmax[i]);
        bool bad = !(wm_ <= 3.0e38f);  // an infinity: the fp32 pass below
        const int ew = wm_ > 0.0f && !bad ? min(max(14 - ilogbf(wm_), -120), 120) : 0;

        // ---- this thread's pieces
        int xr[XO], e[XO];
        float mx[XO], up[XO];  // the row's largest |x| so far, its 2^e
        const int xq = tid & 3;
        const void* xrow[XO];
#pragma unroll
        for (int u = 0; u < XO; ++u) {
            xr[u] = (tid + u * NT) >> 2;
            e[u] = NT_E_UNSET;
            mx[u] = 0.0f;
            up[u] = 1.0f;
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
        const float uw = pow2(ew);
        auto store_sb = [&](int t) __attribute__((always_inline)) {
            if (sb_wave && (tid >> 5) < ngt)
                sbuf[t & 1][tid] = make_float2(round_to(sb.x, a.hmode) * uw, round_to(sb.y, a.hmode) * uw);
        };
        // Step t's rows keep their power of two unless a largest value leaves its range: one branch
        // for the wave, rarely taken.
        auto decide = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < XO; ++u) {
                if constexpr (XF32) {
                    float am = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(xv[u][i]));
                    am = fmaxf(am, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(am), 0xB1, 0xF, 0xF, true)));
                    am = fmaxf(am, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(am), 0x4E, 0xF, 0xF, true)));
                    bad |= am > 3.0e38f;
                    const float at = am * up[u];
                    mx[u] = fmaxf(mx[u], am);
                    const bool need = am > 0.0f && (e[u] == NT_E_UNSET || at >= 32768.0f || at < 0.125f);
                    if (__ballot(need)) {
                        float by = 1.0f;
                        if (need) {
                            // the sums of the steps before stay finite: they are at most 2^75 2^15 N
                            const int to = min(min(max(11 - ilogbf(am), -120), 120), 75 - ilogbf(mx[u]));
                            if (e[u] != NT_E_UNSET && to != e[u]) {
                                by = ldexpf(1.0f, to - e[u]);
                                changed[t % 3] = 1;
                            }
                            e[u] = to;
                            up[u] = pow2(to);
                        }
                        if (xr[u] < BM && xq == 0) row_scale[t % 3][xr[u]] = by;
                    } else if (xr[u] < BM && xq == 0) {
                        row_scale[t % 3][xr[u]] = 1.0f;
                    }
                } else {
                    float am = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf((float)xh[u][i]));
                    bad |= am > 65504.0f;
                }
            }
        };
        auto convert = [&](int t) __attribute__((always_inline)) {  // step t into LDS
            char* base = lds + (t & 1) * STAGE;
#pragma unroll
            for (int u = 0; u < WO; ++u) {
                const int oq = oq0 + u * (NT / BN);
                const float4* p = reinterpret_cast<const float4*>(&sbuf[t & 1][wk / a.gs * 32 + oq * 8]);
                h8 hi, lo;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 v = p[i];  // {s, b} of rows 2 i and 2 i + 1
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const uint32_t c = BITS == 8 ? wv[u][2 * i + j] : (wv[u][2 * i + j] >> (4 * (wk & 1))) & 15u;
                        const float w = __builtin_fmaf((float)(uint8_t)c, j ? v.z : v.x, j ? v.w : v.y);
                        const _Float16 hh = (_Float16)w;
                        hi[2 * i + j] = hh;
                        lo[2 * i + j] = (_Float16)(w - (float)hh);
                    }
                }
                h8* dst = reinterpret_cast<h8*>(base + X_BYTES) + (wk >> 4) * 128 + nt_slot(oq, wk & 15);
                dst[0] = hi;
                dst[64] = lo;
            }
#pragma unroll
            for (int u = 0; u < XO; ++u) {
                h8* dst = reinterpret_cast<h8*>(base) + (xr[u] >> 4) * T * 64 + nt_slot(xq, xr[u] & 15);
                if constexpr (XF32) {
                    h8 hi, lo;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        hi[i] = (_Float16)(xv[u][i] * up[u]);
                        lo[i] = (_Float16)__builtin_fmaf(xv[u][i], up[u], -(float)hi[i]);
                    }
                    if (XO * NT == BM * 4 || xr[u] < BM) {
                        dst[0] = hi;
                        dst[64] = lo;
                    }
                } else {
                    if (XO * NT == BM * 4 || xr[u] < BM) dst[0] = xh[u];
                }
            }
        };

        f4 acc[FM][FN];
#pragma unroll
        for (int m = 0; m < FM; ++m)
#pragma unroll
            for (int n = 0; n < FN; ++n) acc[m][n] = f4{0.f, 0.f, 0.f, 0.f};
        const int slot = nt_slot(q, l16);
        auto multiply = [&](int t, auto between) __attribute__((always_inline)) {
            const vu4* X = reinterpret_cast<const vu4*>(lds + (t & 1) * STAGE) + slot;
            const vu4* Wf = reinterpret_cast<const vu4*>(lds + (t & 1) * STAGE + X_BYTES) + slot;
            h8 xf[FM][T];
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int j = 0; j < T; ++j) xf[m][j] = __builtin_bit_cast(h8, X[((wm * FM + m) * T + j) * 64]);
            between();
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                h8 wf[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) wf[j] = __builtin_bit_cast(h8, Wf[((wn * FN + n) * 2 + j) * 64]);
                // the small terms first
                if constexpr (XF32) {
#pragma unroll
                    for (int m = 0; m < FM; ++m) acc[m][n] = mfma16(wf[0], xf[m][T - 1], acc[m][n]);
                }
#pragma unroll
                for (int m = 0; m < FM; ++m) acc[m][n] = mfma16(wf[1], xf[m][0], acc[m][n]);
#pragma unroll
                for (int m = 0; m < FM; ++m) acc[m][n] = mfma16(wf[0], xf[m][0], acc[m][n]);
            }
        };

        if (steps > 0) {
            load_sb(0);
            load(0);
            store_sb(0);
            load_sb(1);
            __syncthreads();
            decide(0);
            convert(0);
            load(min(1, steps - 1));
            store_sb(1);
            load_sb(2);
            for (int t = 0; t < steps; ++t) {
                block_barrier();  // step t's pieces and step t + 1's scales are in LDS
                store_sb(t + 2);
                load_sb(t + 3);
                if constexpr (XF32) {
                    if (__builtin_amdgcn_readfirstlane(changed[t % 3])) {
#pragma unroll
                        for (int m = 0; m < FM; ++m) {
                            const float by = row_scale[t % 3][(wm * FM + m) * 16 + l16];
#pragma unroll
                            for (int n = 0; n < FN; ++n) acc[m][n] *= by;
                        }
                    }
                    if (tid == 0) changed[(t + 2) % 3] = 0;  // read by every wave before this barrier
                }
                if (t + 1 < steps) decide(t + 1);
                // the last step converts a step past the end once more: no branch around the products
                multiply(t, [&]() __attribute__((always_inline)) {
                    convert(t + 1);
                    load(min(t + 2, steps - 1));
                });
            }
        }

        // ---- the outputs
        if constexpr (XF32) {
#pragma unroll
            for (int u = 0; u < XO; ++u)
                if (xr[u] < BM && xq == 0) row_e[xr[u]] = e[u] == NT_E_UNSET ? 0 : e[u];
        }
        if (__syncthreads_or(bad)) {  // element by element in fp32
            for (int i = threadIdx.x; i < BM * BN; i += NT * GR) {
                const int row = m0 + i / BN, k = k0 + i % BN;
                if (row >= a.M || k >= a.K) continue;
                float v = 0.0f;
                for (int r = 0; r < a.N; ++r) {
                    const float xx = XF32 ? static_cast<const float*>(a.x)[(int64_t)row * a.ldx + r]
                                          : (float)static_cast<const _Float16*>(a.x)[(int64_t)row * a.ldx + r];
                    const uint32_t byte = a.w[(int64_t)r * row_bytes + (BITS == 8 ? k : k >> 1)];
                    const float c = (float)(BITS == 8 ? byte : (byte >> (4 * (k & 1))) & 15u);
                    const int64_t gi = (int64_t)r * a.G + k / a.gs;
                    const float cs = c * round_to(a.scales[gi], a.hmode);
                    v = __builtin_fmaf(xx, a.biases ? cs + round_to(a.biases[gi], a.hmode) : cs, v);
                }
                v = wo_finish(v, a.bias != nullptr, a.bias ? a.bias[k] : 0.0f, a.relu, a.hmode);
                if constexpr (XF32) static_cast<float*>(a.y)[(int64_t)row * a.ldy + k] = v;
                else static_cast<_Float16*>(a.y)[(int64_t)row * a.ldy + k] = (_Float16)v;
            }
            continue;
        }
        // the rows' powers of two leave the sums, then the groups' sums meet, added in order
#pragma unroll
        for (int m = 0; m < FM; ++m) {
            const int down = -(XF32 ? row_e[(wm * FM + m) * 16 + l16] : 0) - ew;  // -240 .. 240, in two exact steps
            const float d0 = ldexpf(1.0f, down / 2), d1 = ldexpf(1.0f, down - down / 2);
#pragma unroll
            for (int n = 0; n < FN; ++n) acc[m][n] = acc[m][n] * d0 * d1;
        }
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
        // per step; in half all three take about 0.65 of it): 256 x 128 tiles 2.36, 128 x 128 1.64,
        // 32 x 64 with the steps split between four wave groups 0.58.
        auto cost = [&](int bm, int bn, double step) { return (double)((tiles(bm, bn) + 255) / 256) * step; };
        const double c256 = cost(256, 128, 2.36), c128 = cost(128, 128, 1.64), c32 = cost(32, 64, 0.58);
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
