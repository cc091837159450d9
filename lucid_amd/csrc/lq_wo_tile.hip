// lq_wo_tile.hip -- weight-only product y = x . w^T for many activation rows (prompts, batches):
// a tiled GEMM on v_mfma_f32_16x16x32_f16 over the operands of lq_wo.hip.
//
// The GEMV kernels give a workgroup 16 weight rows and 16 activation rows and stream the weight
// again for every 16 rows; the product ran at 60-70 TFLOP/s whatever its size.  Here a workgroup of
// eight waves owns BM x 128 outputs (BM 128 in waves of 64 x 32, or 64 / 32 for few rows) and walks
// K in stages of 64 through two LDS slots:
//  * the activations are prepared once per call (wo_tile_prep_kernel): float32 values split into
//    fp16 hi + lo terms after an exact power-of-two pre-scale, half values as they are, both in
//    the order in which a stage's 16-byte pieces are read; with each block's sum.
//  * the weight codes go to LDS as stored; each wave unpacks its fragments to fp16.
//  * the group scales and biases, transposed by the same prepare launch, and the block sums ride
//    along.  LDS holds everything in MFMA fragment order: reads and writes without bank conflicts.
// Measured (float32 x, 8 bits, groups of 64, N = K = 4096; the GEMV kernels before): M = 64 34.5 ->
// 24 us, M = 1024 504 -> 114 us = 301 TFLOP/s (two fp16 products each), M = 2048 992 -> 240;
// half x, 4 bits, M = 1024 456 -> 92.  What bounds it now is the issue of instructions and the waits around a
// stage's barrier: per wave and stage 32 MFMA (16 cycles each), 96 multiplications and FMA of scales, 32 VALU for
// unpacking, 26 LDS reads; the matrix cores are busy 23% of the time (half x 16%), the VALU 29%.
// Arithmetic per 64-wide block (32 for groups of 32), that of the GEMV kernels: the block's values of a
// row are scaled by 2^e (its largest into [2^14, 2^15)) before the split, blk = sum c (hi + lo) in fp32,
// then acc += s (blk 2^-e) + b bsum.  2^-e goes to the scale, ahead of the products (after them, 137 us
// instead of 126 in calls back to back at M = 1024, 8 bits, groups of 64): exact, unless 2^-e is so small
// that s 2^-e may not be a normal number, so below 2^-90 the rest of it goes to blk.  One scale for the
// whole row instead took 117 us, and lost bits of values far below the row's largest.
// Few tiles: K is split into ranges over workgroups, their sums added in range order by
// wo_tile_reduce_kernel.  Without a workspace wo_tile_direct_kernel makes the same sums: the same bits.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lq_dma.h"
#include "lq_internal.h"
#include "lq_wo.h"

namespace lq {
namespace {

struct WtArgs {
    WoTileCall c;
    int G;             // groups per weight row
    int KB;            // stages of 64 k
    int Mp;            // rows padded to 16
    int tiles_m, tiles_n;
    int rs;            // stages per K range
    int ranges;        // K ranges
    const char* xp;    // split activations: [Mp][KB][2 steps][T][4 quarters] of 8 halves
    const float2* xm;  // [KB][NG][Mp]: block sum, 2^-e
    const float2* xr;  // [Mp]: row sum (per-channel weights), 1 if a block's 2^-e lies below WT_TINY
    const float2* sb;  // [G][Np]: group scale, group bias
    int Np;            // columns padded to 128
    float* part;       // range sums [ranges][tile][frag][thread] f4, or null
};

constexpr int WT_FLUSH = 8;  // stages per first-level sum
constexpr float WT_TINY = 0x1p-90f;

// 2^-e as the factor of a group scale and what is left of it for the block's sum (1 above WT_TINY).
__device__ __forceinline__ float down_scale(float down) { return fmaxf(down, WT_TINY); }
__device__ __forceinline__ float down_rest(float down) { return fminf(down * (1.0f / WT_TINY), 1.0f); }

// Blocks per stage: groups of 32 make two blocks of 32 k, everything else one of 64.
template <int S>
constexpr int wt_blocks() { return S == 2 ? 1 : 2; }

// MFMA fragment position of the stage's octet o (8 consecutive k) of a row: step and lane quarter.
template <int S>
__device__ __forceinline__ void octet_pos(int o, int& step, int& q) {
    if (S == 2) { step = o & 1; q = o >> 1; }   // a lane quarter holds 16 consecutive k
    else { step = o >> 2; q = o & 3; }          // one block of 32 per step
}

// The 8 values of octet o of one row (0 past K or for rows past M).
template <bool XF32>
__device__ __forceinline__ void load_octet(const WoTileCall& c, int m, int k, bool vec, float (&v)[8]) {
    const bool in = m < c.M;
    if (vec && in && k + 8 <= c.K) {
        if constexpr (XF32) {
            const vf4* p = reinterpret_cast<const vf4*>(static_cast<const float*>(c.x) + (int64_t)m * c.ldx + k);
            const vf4 a = p[0], b = p[1];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = a[i], v[4 + i] = b[i];
        } else {
            const h8 a = *reinterpret_cast<const h8*>(static_cast<const _Float16*>(c.x) + (int64_t)m * c.ldx + k);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = (float)a[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = 0.0f;
            if (in && k + i < c.K) {
                if constexpr (XF32) v[i] = static_cast<const float*>(c.x)[(int64_t)m * c.ldx + k + i];
                else v[i] = (float)static_cast<const _Float16*>(c.x)[(int64_t)m * c.ldx + k + i];
            }
        }
    }
}

template <bool XF32>
__device__ __forceinline__ bool x_vec(const WoTileCall& c) {
    return (reinterpret_cast<uintptr_t>(c.x) & 15) == 0 && c.ldx % (XF32 ? 4 : 8) == 0;
}

__device__ __forceinline__ float octet_sum(const float (&v)[8]) {
    float s = v[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) s += v[i];
    return s;
}

__device__ __forceinline__ float octet_amax(const float (&v)[8]) {
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) a = fmaxf(a, fabsf(v[i]));
    return a;
}

// 2^e and 2^-e of a block from its largest |value|: 14 - exponent, clamped (a subnormal's exponent
// field is 0: the upper clamp).
template <int T>
__device__ __forceinline__ void block_scale(float am, float& up, float& down) {
    const int e = T == 2 && am > 0.0f && am <= 3.0e38f ? min(max(14 + 127 - (int)(__float_as_uint(am) >> 23), -120), 120) : 0;
    up = __uint_as_float((uint32_t)(127 + e) << 23);
    down = __uint_as_float((uint32_t)(127 - e) << 23);
}

template <int BITS, int T>
__device__ __forceinline__ void octet_terms(const float (&v)[8], float up, h8 (&x)[T]) {
#pragma unroll
    for (int h = 0; h < 8; ++h) {
        const float f = T == 2 ? v[korder<BITS>(h)] * up : v[korder<BITS>(h)];
        x[0][h] = (_Float16)f;
        if constexpr (T == 2) x[1][h] = (_Float16)(f - (float)x[0][h]);
    }
}

// Terms, block sum and 2^-e of one octet; the 4 S lanes of a block's octets are consecutive lanes
// of one wave.
template <int BITS, int S, int T>
__device__ __forceinline__ void split_octet(const float (&v)[8], h8 (&x)[T], float& bsum, float& down) {
    bsum = octet_sum(v);
    float am = octet_amax(v), up;
#pragma unroll
    for (int off = 1; off < 4 * S; off <<= 1) {
        bsum += __shfl_xor(bsum, off, 64);
        am = fmaxf(am, __shfl_xor(am, off, 64));
    }
    block_scale<T>(am, up, down);
    octet_terms<BITS, T>(v, up, x);
}

// The sum over a wave of its lanes' values.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// One row's sum, by one wave, as the prepare launch adds it: thread t of 256 owns octets t, t + 256, ...,
// each quarter of the threads is summed over a wave and the four quarters in order.
template <bool XF32>
__device__ __forceinline__ float row_sum(const WoTileCall& c, int m, int lane, bool vec) {
    float sum = 0.0f;
    for (int w = 0; w < 4; ++w) {
        float s = 0.0f;
        for (int o = 64 * w + lane; o < (c.K + 7) / 8; o += 256) {
            float v[8];
            load_octet<XF32>(c, m, o * 8, vec, v);
            s += octet_sum(v);
        }
        s = wave_sum(s);
        sum = w ? sum + s : s;
    }
    return sum;
}

// The operands the tiled kernel wants contiguous.  The first Mp workgroups: one activation row
// each, as [stage][step][term][lane quarter] 16-byte pieces, with its blocks' sums and scales and (for
// per-channel zero points) its sum.  The others (group-wise): 32 x 32 pieces of the group scales and biases transposed to
// [group][column] pairs, rounded to the activation's type (a missing bias is 0).
template <int BITS, int S, int T, bool GROUPED, int HM>
__global__ __launch_bounds__(256) void wo_tile_prep_kernel(WtArgs a, char* xp, float2* xm, float2* xr, float2* sb) {
    constexpr int NG = wt_blocks<S>();
    constexpr bool XF32 = T == 2;
    __shared__ float2 sh[32][33];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (GROUPED && (int)blockIdx.x >= a.Mp) {
        const int id = blockIdx.x - a.Mp, gt = (a.G + 31) / 32;
        const int g0 = id % gt * 32, n0 = id / gt * 32, x = tid & 31, y = tid >> 5;
#pragma unroll
        for (int r = y; r < 32; r += 8) {
            const int n = n0 + r, g = g0 + x;
            const bool in = n < a.c.N && g < a.G;
            const int64_t at = (int64_t)n * a.G + g;
            sh[r][x] = make_float2(in ? round_to(a.c.w_scale[at], HM) : 0.0f,
                                   in && a.c.g_bias ? round_to(a.c.g_bias[at], HM) : 0.0f);
        }
        __syncthreads();
#pragma unroll
        for (int r = y; r < 32; r += 8)
            if (g0 + r < a.G) sb[(int64_t)(g0 + r) * a.Np + n0 + x] = sh[x][r];
        return;
    }
    const int m = blockIdx.x;
    const bool vec = x_vec<XF32>(a.c);
    float sum = 0.0f;
    bool tiny = false;
    for (int og = tid; og < a.KB * 8; og += 256) {
        const int kb = og >> 3, o = og & 7;
        float v[8];
        load_octet<XF32>(a.c, m, og * 8, vec, v);
        if (!GROUPED) sum += octet_sum(v);
        h8 x[T];
        float bsum, down;
        split_octet<BITS, S, T>(v, x, bsum, down);
        tiny |= down < WT_TINY;
        int step, q;
        octet_pos<S>(o, step, q);
        h8* dst = reinterpret_cast<h8*>(xp) + ((int64_t)m * a.KB + kb) * 8 * T + step * T * 4 + q;
#pragma unroll
        for (int t = 0; t < T; ++t) dst[4 * t] = x[t];
        if ((o & (4 * S - 1)) == 0) xm[((int64_t)kb * NG + o / (4 * S)) * a.Mp + m] = make_float2(bsum, down);
    }
    if (!GROUPED) {
        sum = wave_sum(sum);
        if (lane == 0) sh[0][wave].x = sum;
    }
    tiny = __syncthreads_or(tiny);
    if (tid == 0)
        xr[m] = make_float2(GROUPED ? 0.0f : ((sh[0][0].x + sh[0][1].x) + sh[0][2].x) + sh[0][3].x, tiny ? 1.0f : 0.0f);
}

// Tile of a workgroup: consecutive tiles (groups of eight tile rows, column by column) on one
// XCD, so the 32 workgroups of an XCD share activation and weight panels in its L2.
__device__ __forceinline__ void wt_tile_of(int id, int tm, int tn, int& m, int& n) {
    const int total = tm * tn, q = total / 8, r = total % 8, x = id % 8;
    const int p = x * q + min(x, r) + id / 8;
    const int band = p / (8 * tn), m0 = band * 8, h = min(8, tm - m0), in = p - m0 * tn;
    m = m0 + in % h;
    n = in / h;
}

// A block's part of an output: acc + s blk + b bsum (group-wise, s with 2^-e in it), acc + blk 2^-e.
__device__ __forceinline__ float wt_add(float acc, float blk, float s, float b, float bsum) {
    return __builtin_fmaf(b, bsum, __builtin_fmaf(s, blk, acc));
}
template <int T>
__device__ __forceinline__ float wt_add(float acc, float blk, float down) {
    return T == 2 ? __builtin_fmaf(blk, down, acc) : acc + blk;
}

// The finished value of four consecutive columns of one row.
template <bool GROUPED, bool XF32>
__device__ __forceinline__ void wt_store(const WoTileCall& c, int m, int n, f4 v, float sum) {
    if (m >= c.M || n >= c.N) return;
    const bool xf = XF32;
    f4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int nn = min(n + i, c.N - 1);
        float t = v[i];
        if constexpr (!GROUPED) {
            if (c.w_zp) t = t - c.w_zp[nn] * sum;
            t = c.w_scale[nn] * t;
        }
        out[i] = wo_finish(t, c.bias != nullptr, c.bias ? c.bias[nn] : 0.0f, c.relu, c.hmode);
    }
    const int64_t at = (int64_t)m * c.ldy + n;
    const bool whole = n + 4 <= c.N && (c.ldy & 3) == 0;
    if (xf) {
        float* y = static_cast<float*>(c.y) + at;
        if (whole && (reinterpret_cast<uintptr_t>(c.y) & 15) == 0) {
            *reinterpret_cast<f4*>(y) = out;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < c.N) y[i] = out[i];
        }
    } else {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        _Float16* y = static_cast<_Float16*>(c.y) + at;
        const h4 o = {(_Float16)out[0], (_Float16)out[1], (_Float16)out[2], (_Float16)out[3]};
        if (whole && (reinterpret_cast<uintptr_t>(c.y) & 7) == 0) {
            *reinterpret_cast<h4*>(y) = o;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < c.N) y[i] = o[i];
        }
    }
}

template <int BITS, int S, int T, bool GROUPED, int WM, int WN, int FM, int FN>
__global__ __launch_bounds__(64 * WM * WN) void wo_tile_kernel(WtArgs a) {
    constexpr int W = WM * WN, BM = 16 * WM * FM, BN = 16 * WN * FN, NG = wt_blocks<S>();
    constexpr int A_BYTES = BM * 128 * T, B_BYTES = BN * 8 * BITS;
    constexpr int SB_BYTES = GROUPED ? NG * 2 * BN * 4 : 0, XF_BYTES = NG * 2 * BM * 4;
    constexpr int STAGE = A_BYTES + B_BYTES + SB_BYTES + XF_BYTES;
    constexpr int NST = 2, NT = 64 * W;
    // 16-byte pieces per thread and stage, then pairs (scale, bias; block sum, factor)
    constexpr int A_I = (A_BYTES + 16 * NT - 1) / (16 * NT), B_I = (B_BYTES + 16 * NT - 1) / (16 * NT);
    constexpr int F_N = (SB_BYTES + XF_BYTES) / 8, F_I = (F_N + NT - 1) / NT;
    constexpr int TOT_BYTES = BM * BN * 4;
    static_assert(NST * STAGE + TOT_BYTES <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) char lds[NST * STAGE + TOT_BYTES];
    const WoTileCall& c = a.c;
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tm, tn;
    wt_tile_of(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- one stage: global memory -> registers -> LDS (LDS-DMA copies, with the scales gathered
    // from their rows, took 178 us where this form took 157, at M = 1024, four waves)
    struct Stage {
        vu4 x[A_I];
        vu4 w[B_I];
        float2 f[F_I];
    };
    const int row_bytes = c.K * BITS / 8;
    const uint8_t* b_row[B_I];
    int b_chunk[B_I];
#pragma unroll
    for (int u = 0; u < B_I; ++u) {
        // 8 bits: 1 KB is one 16-row tile of four 16-byte chunks; 4 bits: two tiles of two chunks
        const int i = (tid + u * NT) % (B_BYTES / 16), l = i & 63;
        const int r = BITS == 8 ? (i >> 6) * 16 + (l & 15) : (i >> 5) * 16 + (l & 15);
        b_row[u] = c.w + (int64_t)min(n0 + r, c.N - 1) * c.ldw_bytes;
        b_chunk[u] = (BITS == 8 ? l >> 4 : (l >> 4) & 1) * 16;
    }
    const char* a_ptr[A_I];
#pragma unroll
    for (int u = 0; u < A_I; ++u) {
        // the piece's place in LDS (fragment order) -> its place in its row
        const int i = (tid + u * NT) % (A_BYTES / 16), fr = i >> 6, l = i & 63;
        const int m = min(m0 + fr / (2 * T) * 16 + (l & 15), a.Mp - 1);
        a_ptr[u] = a.xp + (int64_t)m * a.KB * 128 * T + (fr % (2 * T) * 4 + (l >> 4)) * 16;
    }
    const float2* f_ptr[F_I];  // the first stage's pair and the stages' distance
    int64_t f_step[F_I];
    auto pair = [&](int u) __attribute__((always_inline)) { return min(tid + u * NT, F_N - 1); };
#pragma unroll
    for (int u = 0; u < F_I; ++u) {
        const int i = pair(u);
        if (i < SB_BYTES / 8) {  // [block][BN]
            f_ptr[u] = a.sb + (int64_t)(i / BN) * a.Np + n0 + i % BN;
            f_step[u] = 0;
        } else {                 // [block][BM]
            const int j = i - SB_BYTES / 8;
            f_ptr[u] = a.xm + (int64_t)(j / BM) * a.Mp + min(m0 + j % BM, a.Mp - 1);
            f_step[u] = (int64_t)NG * a.Mp;
        }
    }
    auto load = [&](Stage& s, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < A_I; ++u) s.x[u] = *reinterpret_cast<const vu4*>(a_ptr[u] + (int64_t)kb * 128 * T);
#pragma unroll
        for (int u = 0; u < B_I; ++u)
            s.w[u] = *reinterpret_cast<const vu4*>(b_row[u] + min(kb * 8 * BITS + b_chunk[u], row_bytes - 16));
#pragma unroll
        for (int u = 0; u < F_I; ++u) {
            const int i = pair(u);
            if (GROUPED && i < SB_BYTES / 8) {
                const int blk = i / BN, g = min((kb * 64 + blk * 32) / c.gs, a.G - 1);
                s.f[u] = f_ptr[u][(int64_t)(g - blk) * a.Np];
            } else {
                s.f[u] = f_ptr[u][kb * f_step[u]];
            }
        }
    };
    auto store = [&](const Stage& s, int slot) __attribute__((always_inline)) {
        char* base = lds + slot * STAGE;
#pragma unroll
        for (int u = 0; u < A_I; ++u) *reinterpret_cast<vu4*>(base + (tid + u * NT) % (A_BYTES / 16) * 16) = s.x[u];
#pragma unroll
        for (int u = 0; u < B_I; ++u) *reinterpret_cast<vu4*>(base + A_BYTES + (tid + u * NT) % (B_BYTES / 16) * 16) = s.w[u];
#pragma unroll
        for (int u = 0; u < F_I; ++u) {
            reinterpret_cast<float2*>(base + A_BYTES + B_BYTES)[pair(u)] = s.f[u];
        }
    };

    constexpr bool XF32 = T == 2;
    // ---- one stage's products
    // two levels of sums: acc over WT_FLUSH stages, tot over those, in LDS (a chain of all K / 64
    // additions would lose about a bit against the GEMV kernels' sums per wave)
    f4 acc[FM][FN];
    f4* const tot = reinterpret_cast<f4*>(lds + NST * STAGE) + tid;  // [fragment][thread]
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < FM; ++m)
#pragma unroll
            for (int n = 0; n < FN; ++n) acc[m][n] = f4{0.f, 0.f, 0.f, 0.f};
    };
    // acc (stages t0 .. t) joins the range's sum; each thread touches its own slots only
    auto flush = [&](bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < FM; ++m)
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                f4* p = tot + (m * FN + n) * NT;
                *p = first ? acc[m][n] : *p + acc[m][n];
            }
        clear();
    };
    // a wave's operands of one block, as they lie in LDS
    struct Frags {
        vu4 x[FM][S][T];
        uint32_t w[FN][S * BITS / 4];
        f4 sb[GROUPED ? FN : 1][2];  // scale, bias of four columns, interleaved
        float2 xf[FM];               // block sum, 2^-e
    };
    auto read = [&](Frags& r, const char* base, int b) __attribute__((always_inline)) {
        const vu4* A = reinterpret_cast<const vu4*>(base) + lane;
        const char* B = base + A_BYTES;
        const float2* sb = reinterpret_cast<const float2*>(base + A_BYTES + B_BYTES) + b * BN + 4 * q;
        const float2* xf = reinterpret_cast<const float2*>(base + A_BYTES + B_BYTES + SB_BYTES) + b * BM + wm * FM * 16 + l16;
#pragma unroll
        for (int m = 0; m < FM; ++m) r.xf[m] = xf[m * 16];
#pragma unroll
        for (int n = 0; n < FN; ++n) {
            const int nt = wn * FN + n;
            uint32_t* w = r.w[n];
            if constexpr (BITS == 8 && S == 2) {
                const vu4 v = *reinterpret_cast<const vu4*>(B + nt * 1024 + lane * 16);
                w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
            } else if constexpr (BITS == 8) {
                const u2v v = *reinterpret_cast<const u2v*>(B + nt * 1024 + ((b * 2 + (q >> 1)) * 16 + l16) * 16 + (q & 1) * 8);
                w[0] = v.x; w[1] = v.y;
            } else if constexpr (S == 2) {
                const u2v v = *reinterpret_cast<const u2v*>(B + nt * 512 + ((q >> 1) * 16 + l16) * 16 + (q & 1) * 8);
                w[0] = v.x; w[1] = v.y;
            } else {
                w[0] = *reinterpret_cast<const uint32_t*>(B + nt * 512 + (b * 16 + l16) * 16 + q * 4);
            }
        }
#pragma unroll
        for (int j = 0; j < S; ++j)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int m = 0; m < FM; ++m) r.x[m][j][t] = A[(((wm * FM + m) * 2 + (S == 2 ? j : b)) * T + t) * 64];
        if constexpr (GROUPED) {
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                const f4* p = reinterpret_cast<const f4*>(sb + (wn * FN + n) * 16);
                r.sb[n][0] = p[0];
                r.sb[n][1] = p[1];
            }
        }
    };
    auto products = [&](const Frags& r, auto tiny) __attribute__((always_inline)) {
        constexpr bool TINY = decltype(tiny)::value;  // some block's 2^-e lies below WT_TINY
#pragma unroll
        for (int n = 0; n < FN; ++n) {
            h8 wa[S];
#pragma unroll
            for (int j = 0; j < S; ++j) wa[j] = unpack_step<BITS, !GROUPED>(&r.w[n][j * BITS / 4]);
            f4 blk[FM];
#pragma unroll
            for (int m = 0; m < FM; ++m) blk[m] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < S; ++j)
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int m = 0; m < FM; ++m) blk[m] = mfma16(wa[j], __builtin_bit_cast(h8, r.x[m][j][t]), blk[m]);
#pragma unroll
            for (int m = 0; m < FM; ++m) {
                const float down = TINY ? down_scale(r.xf[m].y) : r.xf[m].y;
                if constexpr (TINY && GROUPED) blk[m] *= down_rest(r.xf[m].y);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (GROUPED) {
                        const float sc = r.sb[n][i / 2][i % 2 * 2];
                        acc[m][n][i] = wt_add(acc[m][n][i], blk[m][i], T == 2 ? sc * down : sc,
                                              r.sb[n][i / 2][i % 2 * 2 + 1], r.xf[m].x);
                    } else {
                        acc[m][n][i] = wt_add<T>(acc[m][n][i], blk[m][i], r.xf[m].y);
                    }
                }
            }
        }
    };
    auto finish = [&](int m, int n, f4 v) __attribute__((always_inline)) {
        const int row = m0 + (wm * FM + m) * 16 + l16, col = n0 + (wn * FN + n) * 16 + 4 * q;
        const float sum = !GROUPED && c.w_zp ? a.xr[min(row, a.Mp - 1)].x : 0.0f;
        wt_store<GROUPED, XF32>(c, row, col, v, sum);
    };

    {
        const int k0 = blockIdx.y * a.rs, n = min(a.rs, a.KB - k0);
        clear();
        // stage t + 1 goes from registers to LDS and stage t + 2 from memory to registers while
        // stage t is computed (the last stages repeat the range's last one: no branch in the loop)
        Stage st;
        load(st, k0);
        store(st, 0);
        load(st, k0 + min(1, n - 1));
        auto walk = [&](auto tiny) __attribute__((always_inline)) {
            for (int t = 0; t < n; ++t) {
                block_barrier();  // stage t is in LDS; the other slot has been read
                store(st, (t + 1) & 1);
                load(st, k0 + min(t + 2, n - 1));
#pragma unroll
                for (int b = 0; b < NG; ++b) {
                    Frags r;
                    read(r, lds + (t & 1) * STAGE, b);
                    products(r, tiny);
                }
                if (t % WT_FLUSH == WT_FLUSH - 1 || t == n - 1) flush(t < WT_FLUSH);
            }
        };
        // one test per workgroup: a test per block would wait for the factors before every product
        if (GROUPED && T == 2 && __syncthreads_or(tid < BM && a.xr[min(m0 + tid, a.Mp - 1)].y != 0.0f))
            walk(std::integral_constant<bool, GROUPED && T == 2>{});
        else
            walk(std::false_type{});
        if (a.part) {
            f4* dst = reinterpret_cast<f4*>(a.part) + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * FM * FN * 64 * W + tid;
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int nn = 0; nn < FN; ++nn) dst[(m * FN + nn) * NT] = tot[(m * FN + nn) * NT];
        } else {
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int nn = 0; nn < FN; ++nn) finish(m, nn, tot[(m * FN + nn) * NT]);
        }
    }
}

// ---- the same sums without a workspace
//
// The tiled kernel adds K / 512 or more groups of up to WT_FLUSH stages, first within a range, then the
// ranges.  Here each wave makes whole groups of 32 rows x 16 FN columns, of activations that it splits
// itself, straight from memory; GW waves share a row tile's groups, and the sums meet in LDS in that
// order.  Within a group nothing waits for another wave.  FN = 4 splits x once for 64 columns, FN = 2 and 1
// fill the chip where tiles are few; GW = 2 keeps the waves of a workgroup on the same weights, and busy
// where a row tile has few groups.
// N = K = 4096, 8 bits, groups of 64, float32 x (the kernel for few rows, and the tiled kernel in a form
// that split x in every workgroup): M = 33 40 and 126 -> 27 us, M = 128 106 and 131 -> 34, M = 1024 822 and
// 285 -> 233; half x M = 33 25 and 117 -> 19; M = 2048, N = K = 1024 98 and 52 -> 35.  That form was ahead
// only for groups of 32 and per-channel weights at M = 1024 (235 against 332 us, 187 against 212).
constexpr int WD_WAVES = 8, WD_FM = 2;

template <int BITS, int S, int T, bool GROUPED, int HM, int FN, int GW>
__global__ __launch_bounds__(64 * WD_WAVES) void wo_tile_direct_kernel(WtArgs a) {
    constexpr int NG = wt_blocks<S>(), FM = WD_FM, BM = 16 * FM, BN = 16 * FN, SLOTS = FM * FN * 64;
    constexpr int WB = S * BITS;  // weight bytes of a lane's part of a block
    constexpr bool XF32 = T == 2;
    constexpr int RT = WD_WAVES / GW;                       // row tiles of a workgroup
    constexpr int ST = (SLOTS + 64 * GW - 1) / (64 * GW);  // fours of outputs that a thread finishes
    constexpr int GG = WT_FLUSH * (S == 2 ? 1 : 2);  // most group scales of a column in WT_FLUSH stages
    __shared__ f4 red[WD_WAVES][SLOTS];
    __shared__ float rows[RT * BM];
    __shared__ __attribute__((aligned(16))) float2 scales[GROUPED ? WD_WAVES : 1][GROUPED ? GG * BN : 1];  // [group][column]
    const WoTileCall& c = a.c;
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rt = wave / GW, gw = wave % GW;  // this wave's row tile, and which of its waves it is
    const int cols = (c.N + BN - 1) / BN, row0 = blockIdx.x / cols * RT * BM;  // consecutive workgroups share rows of x
    const int m0 = row0 + rt * BM, n0 = blockIdx.x % cols * BN;
    const bool vec = x_vec<XF32>(c);
    const int row_bytes = c.K * BITS / 8;
    if (!GROUPED && c.w_zp) {
        for (int r = wave; r < RT * BM; r += WD_WAVES) {
            const float sum = row_sum<XF32>(c, row0 + r, lane, vec);
            if (lane == 0) rows[r] = sum;
        }
    }
    // the group scales and biases of stages k0 .. k0 + n of this wave's columns
    const int sg = GROUPED ? c.gs : 64;
    auto load_scales = [&](int k0, int n) __attribute__((always_inline)) {
        const int g0 = k0 * 64 / sg, ng = min((k0 + n) * 64 - 1, c.K - 1) / sg - g0 + 1;
        for (int i = lane; i < GG * BN; i += 64) {
            const int g = i % GG, col = i / GG;
            if (g < ng) {
                const int64_t at = (int64_t)min(n0 + col, c.N - 1) * a.G + g0 + g;
                scales[wave][g * BN + col] =
                    make_float2(round_to(c.w_scale[at], HM), c.g_bias ? round_to(c.g_bias[at], HM) : 0.0f);
            }
        }
    };
    struct Raw {
        vu4 x[FM][2][T];  // the stage's two octets of a lane's rows
        uint32_t w[FN][NG][WB / 4];
    };
    // octet j of a lane in a stage: of one block of 64 the lane quarter holds 16 consecutive k, of each
    // block of 32 eight
    auto octet = [&](int j) __attribute__((always_inline)) { return S == 2 ? 2 * q + j : 4 * j + q; };
    auto load = [&](Raw& r, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < FM; ++m) {
            const int row = min(m0 + 16 * m + l16, c.M - 1);
#pragma unroll
            for (int j = 0; j < 2; ++j) {  // K is a multiple of 8: whole octets, zeroed past K where they are used
                const int64_t at = (int64_t)row * c.ldx + min(kb * 64 + octet(j) * 8, c.K - 8);
                if (vec) {
                    const vu4* p = reinterpret_cast<const vu4*>(static_cast<const uint8_t*>(c.x) + at * (XF32 ? 4 : 2));
#pragma unroll
                    for (int t = 0; t < T; ++t) r.x[m][j][t] = p[t];
                } else {
#pragma unroll
                    for (int i = 0; i < 4 * T; ++i) {
                        if constexpr (XF32) {
                            r.x[m][j][i / 4][i % 4] = static_cast<const uint32_t*>(c.x)[at + i];
                        } else {
                            const uint16_t* p = static_cast<const uint16_t*>(c.x) + at + 2 * i;
                            r.x[m][j][0][i] = p[0] | (uint32_t)p[1] << 16;
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int n = 0; n < FN; ++n) {
            const uint8_t* p = c.w + (int64_t)min(n0 + 16 * n + l16, c.N - 1) * c.ldw_bytes;
#pragma unroll
            for (int b = 0; b < NG; ++b) {  // past the row's end: its last bytes, which meet zeros
                const uint8_t* s = p + min((kb * NG + b) * 4 * WB + q * WB, row_bytes - WB);
                if constexpr (WB == 16) {
                    const vu4 v = *reinterpret_cast<const vu4*>(s);
#pragma unroll
                    for (int i = 0; i < 4; ++i) r.w[n][b][i] = v[i];
                } else if constexpr (WB == 8) {
                    const u2v v = *reinterpret_cast<const u2v*>(s);
                    r.w[n][b][0] = v.x;
                    r.w[n][b][1] = v.y;
                } else {
                    r.w[n][b][0] = *reinterpret_cast<const uint32_t*>(s);
                }
            }
        }
    };
    f4 acc[FM][FN];
    auto add = [&](const Raw& r, int kb, int kg) __attribute__((always_inline)) {  // kg: the group's first stage
#pragma unroll
        for (int b = 0; b < NG; ++b) {
            h8 x[FM][S][T];
            float bsum[FM], down[FM];
#pragma unroll
            for (int m = 0; m < FM; ++m) {
                const bool row = m0 + 16 * m + l16 < c.M;
                float v[S][8], am = 0.0f, up;
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    const int o = S == 2 ? j : b;
                    const bool in = row && kb * 64 + octet(o) * 8 < c.K;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        float f;
                        if constexpr (XF32) f = __uint_as_float(r.x[m][o][i / 4][i % 4]);
                        else f = (float)bits_h2(r.x[m][o][0][i / 2])[i % 2];
                        v[j][i] = in ? f : 0.0f;
                    }
                    bsum[m] = j ? bsum[m] + octet_sum(v[j]) : octet_sum(v[j]);
                    am = fmaxf(am, octet_amax(v[j]));
                }
                // the additions of split_octet: octet pairs, then lane quarters 1 and 2 apart
#pragma unroll
                for (int off = 16; off < 64; off <<= 1) {
                    bsum[m] += __shfl_xor(bsum[m], off, 64);
                    am = fmaxf(am, __shfl_xor(am, off, 64));
                }
                block_scale<T>(am, up, down[m]);
#pragma unroll
                for (int j = 0; j < S; ++j) octet_terms<BITS, T>(v[j], up, x[m][j]);
            }
            const int g = GROUPED ? min(kb * 64 + b * 32, c.K - 1) / sg - kg * 64 / sg : 0;
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                f4 sb[2];  // {scale, bias} of columns 4 q .. 4 q + 3
                if constexpr (GROUPED) {
                    const f4* p = reinterpret_cast<const f4*>(&scales[wave][g * BN + 16 * n + 4 * q]);
                    sb[0] = p[0];
                    sb[1] = p[1];
                }
                h8 wa[S];
#pragma unroll
                for (int j = 0; j < S; ++j) wa[j] = unpack_step<BITS, !GROUPED>(&r.w[n][b][j * BITS / 4]);
                f4 blk[FM];
#pragma unroll
                for (int m = 0; m < FM; ++m) blk[m] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < S; ++j)
#pragma unroll
                    for (int t = 0; t < T; ++t)
#pragma unroll
                        for (int m = 0; m < FM; ++m) blk[m] = mfma16(wa[j], x[m][j][t], blk[m]);
#pragma unroll
                for (int m = 0; m < FM; ++m) {
                    if constexpr (T == 2 && GROUPED) blk[m] *= down_rest(down[m]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (GROUPED) {
                            const float sc = sb[i / 2][i % 2 * 2];
                            acc[m][n][i] = wt_add(acc[m][n][i], blk[m][i], T == 2 ? sc * down_scale(down[m]) : sc,
                                                  sb[i / 2][i % 2 * 2 + 1], bsum[m]);
                        } else {
                            acc[m][n][i] = wt_add<T>(acc[m][n][i], blk[m][i], down[m]);
                        }
                    }
                }
            }
        }
    };
    const int per = (a.rs + WT_FLUSH - 1) / WT_FLUSH;  // groups of a range
    auto first = [&](int g) { return g / per * a.rs + g % per * WT_FLUSH; };
    auto count = [&](int g) { return min(WT_FLUSH, min((g / per + 1) * a.rs, a.KB) - first(g)); };  // none: <= 0
    f4 tot[ST], sum[ST];  // of a range, of the ranges before
    const int groups = a.ranges * per, slot0 = gw * 64 + lane;
    for (int g0 = 0; g0 < groups; g0 += GW) {
        const int g = g0 + gw, k0 = first(g), n = g < groups && m0 < c.M ? count(g) : 0;
        if (n > 0) {
            if constexpr (GROUPED) load_scales(k0, n);
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[m][j] = f4{0.f, 0.f, 0.f, 0.f};
            Raw r[2];
            load(r[0], k0);
            for (int t = 0; t < n; t += 2) {
                load(r[1], k0 + min(t + 1, n - 1));
                add(r[0], k0 + t, k0);
                if (t + 1 < n) {
                    load(r[0], k0 + min(t + 2, n - 1));
                    add(r[1], k0 + t + 1, k0);
                }
            }
#pragma unroll
            for (int m = 0; m < FM; ++m)
#pragma unroll
                for (int j = 0; j < FN; ++j) red[wave][(m * FN + j) * 64 + lane] = acc[m][j];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < ST; ++u) {
            const int slot = slot0 + u * 64 * GW;
            if (slot < SLOTS)
                for (int w = 0; w < GW && g0 + w < groups; ++w) {
                    if (count(g0 + w) <= 0) continue;
                    const f4 v = red[rt * GW + w][slot];
                    if ((g0 + w) % per == 0) {
                        if (g0 + w > 0) sum[u] = g0 + w > per ? sum[u] + tot[u] : tot[u];
                        tot[u] = v;
                    } else {
                        tot[u] += v;
                    }
                }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < ST; ++u) {
        const int slot = slot0 + u * 64 * GW, f = slot >> 6, ml = f / FN * 16 + l16;
        if (slot < SLOTS)
            wt_store<GROUPED, XF32>(c, m0 + ml, n0 + f % FN * 16 + 4 * q, groups > per ? sum[u] + tot[u] : tot[u],
                                    !GROUPED && c.w_zp ? rows[rt * BM + ml] : 0.0f);
    }
}

// Adds the K ranges' sums in range order and finishes the outputs: blockIdx.x the tile,
// blockIdx.y the fragment, a thread the four outputs of its lane.
template <bool GROUPED, bool XF32, int WM, int WN, int FM, int FN>
__global__ __launch_bounds__(64 * WM * WN) void wo_tile_reduce_kernel(WtArgs a) {
    constexpr int W = WM * WN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, l16 = lane & 15;
    const int m = blockIdx.y / FN, n = blockIdx.y % FN;
    int tm, tn;
    wt_tile_of(blockIdx.x, a.tiles_m, a.tiles_n, tm, tn);
    const int row = tm * 16 * WM * FM + (wave / WN * FM + m) * 16 + l16;
    const int col = tn * 16 * WN * FN + (wave % WN * FN + n) * 16 + 4 * q;
    const f4* src = reinterpret_cast<const f4*>(a.part) + ((int64_t)blockIdx.x * FM * FN + blockIdx.y) * 64 * W + tid;
    const int64_t stride = (int64_t)gridDim.x * FM * FN * 64 * W;
    const float sum = !GROUPED && a.c.w_zp ? a.xr[min(row, a.Mp - 1)].x : 0.0f;
    f4 v = src[0];
    int r = 1;
    for (; r + 3 < a.ranges; r += 4) {
        const f4 p0 = src[r * stride], p1 = src[(r + 1) * stride], p2 = src[(r + 2) * stride], p3 = src[(r + 3) * stride];
        v += p0; v += p1; v += p2; v += p3;
    }
    for (; r < a.ranges; ++r) v += src[r * stride];
    wt_store<GROUPED, XF32>(a.c, row, col, v, sum);
}

// ------------------------------------------------------------------ host side

enum { WT_128 = 0, WT_64 = 1, WT_32 = 2 };

struct WtPlan {
    int cfg, BM, BN;
    int64_t tiles_m, tiles_n;
    int KB, rs, ranges;
    size_t xp, xm, xr, sb, part;  // byte sizes
};

WtPlan wt_plan(int64_t M, int64_t N, int64_t K, bool xf32, int gs) {
    WtPlan p{};
    p.cfg = M <= 32 ? WT_32 : M <= 64 ? WT_64 : WT_128;
    p.BM = p.cfg == WT_128 ? 128 : p.cfg == WT_64 ? 64 : 32;
    p.BN = 128;
    p.tiles_m = (M + p.BM - 1) / p.BM;
    p.tiles_n = (N + p.BN - 1) / p.BN;
    p.KB = (int)((K + 63) / 64);
    const int64_t t = p.tiles_m * p.tiles_n;
    // fewer tiles than CUs: K ranges of at least four stages, about one workgroup per CU
    const int64_t want = t > 128 ? 1 : std::min<int64_t>({16, 256 / t, std::max(1, p.KB / 4)});
    p.rs = (int)((p.KB + want - 1) / want);
    p.ranges = (p.KB + p.rs - 1) / p.rs;
    const int NG = gs == 32 ? 2 : 1, T = xf32 ? 2 : 1;
    const int64_t Mp = (M + 15) / 16 * 16;
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    p.xp = up((size_t)Mp * p.KB * 128 * T);
    p.xm = up((size_t)p.KB * NG * 2 * Mp * 4);
    p.xr = up((size_t)Mp * 8);
    p.sb = gs ? up((size_t)(K / gs) * 8 * (size_t)(p.tiles_n * p.BN)) : 0;
    p.part = p.ranges > 1 ? up((size_t)p.ranges * t * p.BM * p.BN * 4) : 0;
    return p;
}

template <int BITS, int S, int T, bool GROUPED, int HM, int WM, int WN, int FM, int FN>
void wt_go(const WtPlan& p, WtArgs& a, hipStream_t st) {
    const unsigned t = (unsigned)(p.tiles_m * p.tiles_n);
    const unsigned scale_blocks = GROUPED ? (unsigned)((a.G + 31) / 32) * (unsigned)(a.Np / 32) : 0;
    hipLaunchKernelGGL((wo_tile_prep_kernel<BITS, S, T, GROUPED, HM>), dim3((unsigned)a.Mp + scale_blocks), dim3(256), 0, st, a,
                       const_cast<char*>(a.xp), const_cast<float2*>(a.xm), const_cast<float2*>(a.xr),
                       const_cast<float2*>(a.sb));
    hipLaunchKernelGGL((wo_tile_kernel<BITS, S, T, GROUPED, WM, WN, FM, FN>), dim3(t, (unsigned)p.ranges),
                       dim3(64 * WM * WN), 0, st, a);
    if (p.ranges > 1)
        hipLaunchKernelGGL((wo_tile_reduce_kernel<GROUPED, T == 2, WM, WN, FM, FN>), dim3(t, FM * FN), dim3(64 * WM * WN), 0, st, a);
}

template <int BITS, int S, bool GROUPED>
void wt_config(const WtPlan& p, WtArgs& a, bool inl, hipStream_t st) {
    auto go = [&](auto t, auto h) {
        constexpr int T = decltype(t)::value, HM = decltype(h)::value;
        if (inl) {
            // 64 columns a workgroup where that leaves none of the chip idle, then two waves a row tile where it
            // has up to four groups
            auto direct = [&](auto fn, auto gw) {
                constexpr int FN = decltype(fn)::value, GW = decltype(gw)::value;
                constexpr int BM = 16 * WD_FM * (WD_WAVES / GW), BN = 16 * FN;
                const unsigned grid = (unsigned)((a.c.N + BN - 1) / BN) * (unsigned)((a.c.M + BM - 1) / BM);
                hipLaunchKernelGGL((wo_tile_direct_kernel<BITS, S, T, GROUPED, HM, FN, GW>), dim3(grid),
                                   dim3(64 * WD_WAVES), 0, st, a);
            };
            using I1 = std::integral_constant<int, 1>;
            using I2 = std::integral_constant<int, 2>;
            using I4 = std::integral_constant<int, 4>;
            using I8 = std::integral_constant<int, 8>;
            auto groups = [&](int cols) { return (int64_t)((a.c.N + cols - 1) / cols) * ((a.c.M + 31) / 32); };
            if (groups(32) < 256) direct(I1{}, I8{});
            else if (groups(64) < 256) direct(I2{}, I8{});
            else if (groups(64) < 1024) direct(I4{}, I8{});
            else direct(I4{}, I2{});
        } else if (p.cfg == WT_128) wt_go<BITS, S, T, GROUPED, HM, 2, 4, 4, 2>(p, a, st);
        else if (p.cfg == WT_64) wt_go<BITS, S, T, GROUPED, HM, 2, 4, 2, 2>(p, a, st);
        else wt_go<BITS, S, T, GROUPED, HM, 2, 4, 1, 2>(p, a, st);
    };
    using T1 = std::integral_constant<int, 1>;
    using T2 = std::integral_constant<int, 2>;
    using None = std::integral_constant<int, LQ_ROUND_NONE>;
    if constexpr (!GROUPED) {
        a.c.xf32 ? go(T2{}, None{}) : go(T1{}, None{});
    } else {  // scales rounded to the activation's type: half always, bfloat16 on request
        if (!a.c.xf32) go(T1{}, std::integral_constant<int, LQ_ROUND_F16>{});
        else if (a.c.hmode == LQ_ROUND_BF16) go(T2{}, std::integral_constant<int, LQ_ROUND_BF16>{});
        else go(T2{}, None{});
    }
}

}  // namespace

bool wo_tile_takes(const WoTileCall& c) {
    // Three launches and their latencies (17 us at M = 32, N = K = 4096) against a GEMV kernel whose
    // time grows with the 16-row blocks times the weight: measured equal near 2^25 (M = 32: 19.4
    // against 16.9 us in float32, 16.7 against 17.3 in half; M = 33: 27.2 against 20.7; M = 600,
    // N = 512, K = 1024, 2^24.2: 15.2 against 21.2 us).
    if (c.M <= 16 || c.K < 64 || (int64_t)((c.M + 15) / 16) * c.N * c.K <= ((int64_t)1 << 25)) return false;
    const int64_t row_bytes = (int64_t)c.K * c.bits / 8;
    if (!aligned16(c.w) || c.ldw_bytes % 16 || row_bytes % 16) return false;
    // 32-bit offsets inside a workgroup's weight rows and scales; grid and tile counts
    if (128 * c.ldw_bytes >= ((int64_t)1 << 31)) return false;
    const WtPlan p = wt_plan(c.M, c.N, c.K, c.xf32, c.gs);
    return p.tiles_m * p.tiles_n < ((int64_t)1 << 24) && (c.gs == 0 || (int64_t)128 * (c.K / c.gs) < ((int64_t)1 << 28)) &&
           (int64_t)4 * c.M < ((int64_t)1 << 28);
}

size_t wo_tile_ws_bytes(int64_t M, int64_t N, int64_t K, int gs) {
    size_t need = 0;
    for (int xf32 = 0; xf32 < 2; ++xf32) {
        const WtPlan p = wt_plan(M, std::max<int64_t>(N, 1), K, xf32 != 0, gs);
        need = std::max(need, p.xp + p.xm + p.xr + p.sb + p.part);
    }
    return need;
}

int wo_tile_launch(const WoTileCall& c, void* ws, size_t ws_bytes, hipStream_t st) {
    const WtPlan p = wt_plan(c.M, c.N, c.K, c.xf32, c.gs);
    WtArgs a{};
    a.c = c;
    a.G = c.gs ? c.K / c.gs : 1;
    a.KB = p.KB;
    a.Mp = (c.M + 15) / 16 * 16;
    a.Np = (int)(p.tiles_n * p.BN);
    a.tiles_m = (int)p.tiles_m;
    a.tiles_n = (int)p.tiles_n;
    a.rs = p.rs;
    a.ranges = p.ranges;
    const bool inl = !ws || !aligned16(ws) || ws_bytes < p.xp + p.xm + p.xr + p.sb + p.part;
    if (!inl) {
        char* b = static_cast<char*>(ws);
        a.xp = b;
        a.xm = reinterpret_cast<const float2*>(b + p.xp);
        a.xr = reinterpret_cast<const float2*>(b + p.xp + p.xm);
        a.sb = reinterpret_cast<const float2*>(b + p.xp + p.xm + p.xr);
        a.part = p.part ? reinterpret_cast<float*>(b + p.xp + p.xm + p.xr + p.sb) : nullptr;
    }
    if (c.gs == 0) wt_config<8, 2, false>(p, a, inl, st);
    else if (c.bits == 8) c.gs == 32 ? wt_config<8, 1, true>(p, a, inl, st) : wt_config<8, 2, true>(p, a, inl, st);
    else c.gs == 32 ? wt_config<4, 1, true>(p, a, inl, st) : wt_config<4, 2, true>(p, a, inl, st);
    note_path(inl ? "wo tiles inline" : p.ranges > 1 ? "wo tiles split" : "wo tiles");
    return LQ_OK;
}

}  // namespace lq
