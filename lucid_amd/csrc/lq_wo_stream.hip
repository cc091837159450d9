// lq_wo_stream.hip -- weight-only int8 products of 1 to 16 activation rows over the MFMA-packed
// weight (lq_gemv_w8_packed), in one pass over the weight.
//
// A decode step reads each weight once; what counts is keeping loads of it in flight and the chain
// of latencies around them short.  A workgroup of eight waves (one per CU) stays for all its column
// tiles: its waves split the K range (512 k a wave, or half or a quarter of that where K is short)
// and hold their slices of x, as fp16 hi + lo terms, in registers for the whole launch.  Per tile of
// 16 columns a wave needs only its weight bytes -- 1 KB per block of 64 k, contiguous; the next
// tile's are loaded while this tile's are multiplied -- and the waves' 16 x 16 sums meet in LDS once.
// K up to 4096 is one range: no partial sums in memory, no second launch.  Longer K is cut into
// ranges whose sums wo_stream_reduce_kernel adds in range order.
//
// The products, block sums and their scaling are wo_gemv_sk_kernel's (per row and block of 64 k a
// power of two, two fp16 terms, fp32 sums) and, up to K = 4096, so is the order of the additions:
// blocks s and s + 4 of 512 k, those four sums in order, then the 512-k sums: the same bits.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lq_dma.h"
#include "lq_internal.h"
#include "lq_wo.h"

namespace lq {
namespace {

constexpr int WS_WAVES = 8;

struct WsArgs {
    WoTileCall c;
    int KB;         // 64-k blocks of a weight row
    int tiles;      // column tiles of 16
    int ranges;     // K ranges of 64 blocks
    int wgs;        // workgroups per range
    float* part;    // [range][tile][256] sums, or null
    float* part_x;  // [range][16] row sums
};

// Largest / sum of a lane's value over the four lanes 16 apart (every lane gets it).
__device__ __forceinline__ float quarters_max(float v) {
    const uint32_t u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const uint32_t m = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane32_swap(m, m, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float quarters_sum(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// The end of one output.
template <bool XF32>
__device__ __forceinline__ void ws_finish(const WoTileCall& c, int m, int n, float v, float xtot, float ws, float wz, float wb) {
    if (c.w_zp) v = v - wz * xtot;
    v = wo_finish(ws * v, c.bias != nullptr, wb, c.relu, c.hmode);
    if constexpr (XF32) static_cast<float*>(c.y)[(int64_t)m * c.ldy + n] = v;
    else static_cast<_Float16*>(c.y)[(int64_t)m * c.ldy + n] = (_Float16)v;
}

// NB: 64-k blocks per wave; 8 / NB waves share 512 k, each with NB / 2 of its four sums.
template <bool XF32, int NB>
__global__ __launch_bounds__(64 * WS_WAVES) void wo_stream_kernel(WsArgs a) {
    constexpr int T = XF32 ? 2 : 1;
    constexpr int PW = 8 / NB, SUBS = NB / 2, R = WS_WAVES / PW;  // waves per 512 k, sums per wave, 512s
    constexpr int PUT = PW == 1 ? 1 : SUBS;                         // sums a wave leaves in LDS
    __shared__ f4 red[2][WS_WAVES * PUT][64];
    __shared__ __attribute__((aligned(16))) float down[WS_WAVES][NB][16];  // 2^-e of row and block
    __shared__ float xsum[R][4][16];
    const WoTileCall& c = a.c;
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int range = blockIdx.x % a.ranges, first = blockIdx.x / a.ranges;
    const int r5 = wave / PW, part = wave % PW;
    auto block = [&](int b) { return range * 64 + r5 * 8 + b / SUBS * 4 + part * SUBS + b % SUBS; };  // the wave's block b

    auto load = [&](vu4 (&w)[NB], int tile) __attribute__((always_inline)) {
        const uint8_t* p = c.w + (int64_t)tile * a.KB * 1024 + lane * 16;
#pragma unroll
        for (int b = 0; b < NB; ++b)  // blocks past the last re-read it: their x is 0
            w[b] = __builtin_nontemporal_load(reinterpret_cast<const vu4*>(p + (int64_t)min(block(b), a.KB - 1) * 1024));
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- this wave's slice of x.  Its loads go out before the first tile's: vmcnt counts in issue
    // order, so the split waits for x (L2) alone and runs while the weights come from memory.
    vu4 cur[NB];
    h8 x[NB][2][T];  // values q 16 + 8 h .. + 7 of the block
    {
        const bool row = l16 < c.M;
        const uint8_t* xr = static_cast<const uint8_t*>(c.x) + (int64_t)min(l16, c.M - 1) * c.ldx * (XF32 ? 4 : 2);
        vu4 raw[NB][2 * T];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 2 * T; ++i) {
                const int k = block(b) * 64 + q * 16 + i * (XF32 ? 4 : 8);
                raw[b][i] = *reinterpret_cast<const vu4*>(xr + (int64_t)min(k, c.K - (XF32 ? 4 : 8)) * (XF32 ? 4 : 2));
            }
        __builtin_amdgcn_sched_barrier(0);
        load(cur, first);
        float tot[SUBS] = {};
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            // K is a multiple of 16: this lane's 16 values are inside or outside as a whole
            const bool in = row && block(b) * 64 + q * 16 < c.K;
            if constexpr (XF32) {
                auto v = [&](int i) __attribute__((always_inline)) { return __uint_as_float(raw[b][i / 4][i % 4]); };
                float am = 0.0f;
#pragma unroll
                for (int i = 0; i < 16; ++i) am = fmaxf(am, fabsf(v(i)));
                am = quarters_max(am);
                // 14 - exponent; values that are not there are multiplied by 0
                const int e = am > 0.0f && am <= 3.0e38f ? min(max(14 + 127 - (int)(__float_as_uint(am) >> 23), -120), 120) : 0;
                const float up = in ? __uint_as_float((uint32_t)(e + 127) << 23) : 0.0f;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const _Float16 hi = (_Float16)(v(i) * up);
                    x[b][i / 8][0][i % 8] = hi;
                    x[b][i / 8][T - 1][i % 8] = (_Float16)__builtin_fmaf(v(i), up, -(float)hi);
                }
                if (q == 0) down[wave][b][l16] = __uint_as_float((uint32_t)(127 - e) << 23);
                if (c.w_zp) {
                    float bs = 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; ++i) bs += v(i);
                    tot[b % SUBS] += quarters_sum(in ? bs : 0.0f);
                }
            } else {
                float bs = 0.0f;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    x[b][h][0] = __builtin_bit_cast(h8, in ? raw[b][h] : vu4{0, 0, 0, 0});
                    if (c.w_zp) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) bs += (float)x[b][h][0][i];
                    }
                }
                if (c.w_zp) tot[b % SUBS] += quarters_sum(bs);
            }
        }
        if (q == 0) {
#pragma unroll
            for (int u = 0; u < SUBS; ++u) xsum[r5][part * SUBS + u][l16] = tot[u];
        }
    }

    // ---- the tiles
    const int om = (tid & 255) >> 4, on = tid & 15;  // the output of a thread of the finishing half
    int buf = 0;
    for (int tile = first; tile < a.tiles; tile += a.wgs) {
        vu4 nxt[NB];
        load(nxt, min(tile + a.wgs, a.tiles - 1));
        const bool ends = (tid >> 8) == buf;  // the halves of the workgroup take turns
        const int n = min(tile * 16 + on, c.N - 1);
        float ws = 1.0f, wz = 0.0f, wb = 0.0f;
        if (ends && !a.part) {
            ws = c.w_scale[n];
            if (c.w_zp) wz = c.w_zp[n];
            if (c.bias) wb = c.bias[n];
        }
        f4 acc[SUBS];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            f4 blk = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t wd[2] = {cur[b][2 * h], cur[b][2 * h + 1]};
                const h8 w = unpack_step<8, true>(wd);
#pragma unroll
                for (int t = 0; t < T; ++t) blk = mfma16(x[b][h][t], w, blk);
            }
            if constexpr (XF32) blk *= *reinterpret_cast<const f4*>(&down[wave][b][4 * q]);  // rows 4 q .. 4 q + 3
            if (b < SUBS) acc[b] = blk;
            else acc[b - SUBS] += blk;
        }
        if constexpr (PW == 1) {
#pragma unroll
            for (int u = 1; u < SUBS; ++u) acc[0] += acc[u];
        }
#pragma unroll
        for (int u = 0; u < PUT; ++u) red[buf][wave * PUT + u][lane] = acc[u];
        block_barrier();  // the other buffer's readers are a whole tile behind
        if (ends) {
            const float* r = reinterpret_cast<const float*>(red[buf][0]) + (om >> 2) * 64 + on * 4 + (om & 3);
            float v = 0.0f, t = 0.0f;
#pragma unroll
            for (int g = 0; g < R; ++g) {
                float u = r[g * (PW == 1 ? 1 : 4) * 256];
#pragma unroll
                for (int w = 1; w < (PW == 1 ? 1 : 4); ++w) u += r[(g * 4 + w) * 256];
                v += u;
            }
            if (c.w_zp) {
                for (int g = 0; g < R; ++g) t += ((xsum[g][0][om] + xsum[g][1][om]) + xsum[g][2][om]) + xsum[g][3][om];
            }
            if (a.part) {
                a.part[((int64_t)range * a.tiles + tile) * 256 + (tid & 255)] = v;
                if (tile == 0 && on == 0) a.part_x[range * 16 + om] = t;
            } else if (om < c.M && tile * 16 + on < c.N) {
                ws_finish<XF32>(c, om, n, v, t, ws, wz, wb);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) cur[b] = nxt[b];
        buf ^= 1;
    }
}

template <bool XF32>
__global__ __launch_bounds__(256) void wo_stream_reduce_kernel(WsArgs a) {
    const WoTileCall& c = a.c;
    const int m = threadIdx.x >> 4, n = blockIdx.x * 16 + (threadIdx.x & 15);
    if (m >= c.M || n >= c.N) return;
    const float ws = c.w_scale[n], wz = c.w_zp ? c.w_zp[n] : 0.0f, wb = c.bias ? c.bias[n] : 0.0f;
    float v = 0.0f, t = 0.0f;
    for (int r = 0; r < a.ranges; ++r) {
        v += a.part[((int64_t)r * a.tiles + blockIdx.x) * 256 + threadIdx.x];
        if (c.w_zp) t += a.part_x[r * 16 + m];
    }
    ws_finish<XF32>(c, m, n, v, t, ws, wz, wb);
}

struct WsPlan {
    int ranges;
    int64_t KB, tiles;
    size_t part, bytes;
};

WsPlan ws_plan(int64_t N, int64_t K) {
    WsPlan p{};
    p.KB = (K + 63) / 64;
    p.ranges = (int)((p.KB + 63) / 64);
    p.tiles = (N + 15) / 16;
    p.part = p.ranges > 1 ? (size_t)p.ranges * p.tiles * 256 * 4 : 0;
    p.bytes = p.ranges > 1 ? p.part + (size_t)p.ranges * 16 * 4 : 0;
    return p;
}

template <bool XF32>
void ws_go(const WsArgs& a, hipStream_t st) {
    const dim3 grid((unsigned)(a.wgs * a.ranges)), block(64 * WS_WAVES);
    if (a.KB <= 16) hipLaunchKernelGGL((wo_stream_kernel<XF32, 2>), grid, block, 0, st, a);
    else if (a.KB <= 32) hipLaunchKernelGGL((wo_stream_kernel<XF32, 4>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((wo_stream_kernel<XF32, 8>), grid, block, 0, st, a);
    if (a.ranges > 1) hipLaunchKernelGGL(wo_stream_reduce_kernel<XF32>, dim3((unsigned)a.tiles), dim3(256), 0, st, a);
}

}  // namespace

// Against wo_gemv_sk_kernel's pair of launches over the same weight (M = 1 to 16, N = 256 to 16384, K = 256 to
// 14336, 1288 sizes, weights from memory; the rule's choice is within 5% of the faster one at all but 15, within 12%
// at all):
//  * K up to 512 is one launch there too: this one's second round of tiles costs more than a second round of
//    its small workgroups (M = 1, K = 512: N = 4096 4.4 us here, 4.9 there; N = 8192 5.8 and 5.0; N = 16384 7.7 and 5.4).
//  * Up to 2048 the second launch is what counts (M = 16, N = 4096: K = 1024 5.4 and 8.3; K = 2048 8.5 and 9.1).
//  * Beyond, every wave reads and splits 512 k of x before its first product, 9 us with one row and 13 with 16,
//    half x 5 to 8, and the weight has to be worth it (K = 4096: M = 1, N = 2048 8.8 and 8.6, N = 8192 12.4 and 15.6;
//    M = 16, N = 2048 13.7 and 9.1, N = 6144 15.9 and 15.0, N = 8192 16.8 and 17.7; half x 16 x 512 8.1 and 7.2).
//  * Ranges of 4096 that are not full leave their workgroups idle, most of all a second one that is all but
//    empty (N = 8192, K = 4112: M = 1 18.2 and 16.6, M = 16 21.4 and 18.1, half x 15.1 and 15.8, 16.5 and 15.4;
//    K = 8192, M = 1 23 and 29).
bool wo_stream_preferred(int64_t M, int64_t N, int64_t K, bool xf32) {
    const WsPlan p = ws_plan(N, K);
    const int64_t cus = device_cu_count();
    if (K <= 512) return p.tiles <= (xf32 && M <= 8 ? cus : cus * 3 / 2);
    if (K <= 2048) return true;
    if (K > 4096 && (xf32 ? K < 5120 : M > 8 && K < 4608)) return false;
    const double fill = p.ranges > 1 ? (double)K / (p.ranges * 4096.0) : 1.0;  // of the ranges
    return 5.0 * N * K * fill > (double)((xf32 ? 68 + 4 * M : 4 * (M - 4)) * (1 << 20));
}

size_t wo_stream_ws_bytes(int64_t N, int64_t K) { return ws_plan(N, K).bytes; }

void wo_stream_launch(const WoTileCall& c, void* ws, hipStream_t st) {
    const WsPlan p = ws_plan(c.N, c.K);
    WsArgs a{};
    a.c = c;
    a.KB = (int)p.KB;
    a.tiles = (int)p.tiles;
    a.ranges = p.ranges;
    // one workgroup per CU; with ranges, their workgroups share the CUs
    a.wgs = (int)std::min<int64_t>(p.tiles, std::max(1, device_cu_count() / p.ranges));
    if (p.ranges > 1) {
        a.part = static_cast<float*>(ws);
        a.part_x = reinterpret_cast<float*>(static_cast<char*>(ws) + p.part);
    }
    c.xf32 ? ws_go<true>(a, st) : ws_go<false>(a, st);
    note_path(p.ranges > 1 ? "wo stream ranges" : "wo stream");
}

}  // namespace lq
