// lq_wo.h -- pieces shared by the weight-only kernels (lq_wo.hip, lq_wo_tile.hip): fp16 code
// unpacking, the MFMA step, the epilogue of one output.
#pragma once

#include <hip/hip_runtime.h>

#include "lq_internal.h"

namespace lq {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2 bits_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }

// k offset of half h within a lane's 8-element step for a code width.
template <int BITS>
__device__ __forceinline__ int korder(int h) {
    return BITS == 4 ? ((h & 1) * 4 + (h >> 1)) : h;
}

// Four bytes -> four halves (byte - off) in byte order.
__device__ __forceinline__ void bytes_to_h2(uint32_t w, _Float16 off, h2& a, h2& b) {
    const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u);
    const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u);
    const h2 o = {off, off};
    a = bits_h2(p0) - o;
    b = bits_h2(p1) - o;
}

// One MFMA step's 8 codes as fp16: 8-bit from two words (signed codes are xor'ed with
// 0x80 so the byte is c + 128), 4-bit from one word.
template <int BITS, bool SIGNED>
__device__ __forceinline__ h8 unpack_step(const uint32_t* w) {
    if constexpr (BITS == 8) {
        const uint32_t x0 = SIGNED ? (w[0] ^ 0x80808080u) : w[0];
        const uint32_t x1 = SIGNED ? (w[1] ^ 0x80808080u) : w[1];
        const _Float16 off = SIGNED ? (_Float16)1152.0f : (_Float16)1024.0f;
        h2 a, b, c, d;
        bytes_to_h2(x0, off, a, b);
        bytes_to_h2(x1, off, c, d);
        return h8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
    } else {
        const h2 o = {(_Float16)1024.0f, (_Float16)1024.0f};
        h2 r[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) r[s] = bits_h2(((w[0] >> (4 * s)) & 0x000F000Fu) | 0x64006400u) - o;
        return h8{r[0].x, r[0].y, r[1].x, r[1].y, r[2].x, r[2].y, r[3].x, r[3].y};
    }
}

__device__ __forceinline__ f4 mfma16(h8 a, h8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Epilogue of one output: the float32 product rounded to the activation's type (hmode, a
// LQ_ROUND_* value), the layer bias rounded to that type and added there, then ReLU --
// Lucid's quantized_matmul returning x's dtype and QuantizedLinearMLX's y + bias.to(y.dtype),
// relu (lucid/nn/quantized/mlx_linear.py:215-222).  A half or bfloat16 sum of two such values
// is exact in float32 before its rounding (24 >= 2 p + 2 bits), so the float32 add then round
// equals the narrow add.  hmode 0 leaves the float32 result as it is.
__device__ __forceinline__ float wo_finish(float v, bool has_bias, float b, int relu, int hmode) {
    if (hmode == LQ_ROUND_NONE) {
        if (has_bias) v = v + b;
    } else {
        v = round_result_to(v, hmode);
        if (has_bias) v = round_result_to(v + round_to(b, hmode), hmode);
    }
    if (relu && v <= 0.0f) v = 0.0f;
    return v;
}

// ---------------------------------------------- tiled kernel for many rows (lq_wo_tile.hip)

// One weight-only product of more rows than the GEMV kernels are made for: y = x . w^T with the
// operands of wo_gemv_kernel (int8 rows, or group-wise packed rows of 4 / 8-bit codes).
struct WoTileCall {
    const void* x;
    int64_t ldx;
    bool xf32;
    const uint8_t* w;
    int64_t ldw_bytes;
    const float* w_scale;  // per-channel [N] or group [N][G]
    const float* w_zp;     // per-channel zero points [N] or null
    const float* g_bias;   // group biases [N][G] or null
    const float* bias;     // layer bias [N] or null
    void* y;
    int64_t ldy;
    int relu, hmode;
    int M, N, K;
    int bits;              // 4 or 8
    int gs;                // group size, 0 for per-channel int8
};

// Whether the tiled kernel takes the call (from the shape and the weight's alignment alone).
bool wo_tile_takes(const WoTileCall& c);
// Workspace of an M x N x K call: the split activations and, for few tiles, the K ranges' sums.
size_t wo_tile_ws_bytes(int64_t M, int64_t N, int64_t K, int gs);
// Launches it; a smaller (or NULL) workspace selects the form that splits the activations in
// every workgroup, with the same results.
int wo_tile_launch(const WoTileCall& c, void* ws, size_t ws_bytes, hipStream_t st);

// ---------------------------------------------- x . w_hat (lq_wo_nt.hip)

// y[M, K] = x[M, N] w_hat[N, K] (+ bias, ReLU) of group-wise packed rows.
struct WoNtCall {
    const void* x;
    int64_t ldx;
    bool xf32;
    const uint8_t* w;
    const float* scales;   // [N][K / gs]
    const float* biases;   // [N][K / gs] or null
    const float* bias;     // layer bias [K] or null
    void* y;
    int64_t ldy;
    int relu, hmode;
    int M, N, K, bits, gs;
};

void group_matmul_nt_launch(const WoNtCall& c, hipStream_t st);

// ---------------------------------------------- 1 to 16 rows over the packed weight (lq_wo_stream.hip)

// Workspace of the K ranges' sums (0 up to K = 4096).
size_t wo_stream_ws_bytes(int64_t N, int64_t K);
// Whether it is the faster form for the shape.
bool wo_stream_preferred(int64_t M, int64_t N, int64_t K, bool xf32);
// c.w is lq_pack_weights_i8's form; M <= 16, K a multiple of 16, 16-byte aligned x rows and weight.
void wo_stream_launch(const WoTileCall& c, void* ws, hipStream_t st);

}  // namespace lq
