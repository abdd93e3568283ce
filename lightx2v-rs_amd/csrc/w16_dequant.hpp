// w16_dequant.hpp -- the Q8 / Q4 / FP8 weight decode of the bf16 MFMA kernels
// (k_gemm_w16.hip, k_gemm_rows.hip).
#pragma once

#include "device_common.hpp"

namespace lx2v {

namespace {

// Q4 with every zero 8 (lx2v_hip_weight::zero8): the same codes and scales,
// no zeros loaded (a format id of these kernels only)
constexpr int kWfmtQ4Sym = 100;

// 16 consecutive K elements of one weight row, as 8 packed bf16 pairs
// (element 2i low), each rounded from the reference's f32 dequantization
// (quant.rs:183-191, 279-289, 432-440): c = 16 code bytes (Q8, FP8) or 8
// (Q4, in c.x, c.y), s / z = the group's scale / zero.
template <int WF>
__device__ __forceinline__ void unit_dequant(u32x4 c, float s, float z, uint32_t (&o)[8]) {
    const uint32_t w[4] = {c.x, c.y, c.z, c.w};
    if constexpr (WF == LX2V_WFMT_Q8) {
        // byte ^ 0x80 reads as q + 128 unsigned, and fma(q + 128, s, -128 s)
        // rounds the exact q * s once (128 s is exact): the reference's q * s.
        const float nb = -128.0f * s;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t b = w[q] ^ 0x80808080u;
            const float f0 = __builtin_fmaf((float)(b & 0xFFu), s, nb);
            const float f1 = __builtin_fmaf((float)((b >> 8) & 0xFFu), s, nb);
            const float f2 = __builtin_fmaf((float)((b >> 16) & 0xFFu), s, nb);
            const float f3 = __builtin_fmaf((float)(b >> 24), s, nb);
            o[2 * q] = pack_bf16x2(f0, f1);
            o[2 * q + 1] = pack_bf16x2(f2, f3);
        }
    } else if constexpr (WF == kWfmtQ4Sym) {
        // zero 8: (c - 8) s is exact before its one rounding, and so is
        // fma(c, s, -8 s) (8 s is exact): the same f32 value
        const float nb = -8.0f * s;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t lo = w[q] & 0x0F0F0F0Fu, hi = (w[q] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const float e0 = __builtin_fmaf((float)((lo >> (8 * b)) & 0xFFu), s, nb);
                const float e1 = __builtin_fmaf((float)((hi >> (8 * b)) & 0xFFu), s, nb);
                o[4 * q + b] = pack_bf16x2(e0, e1);
            }
        }
        (void)z;
    } else if constexpr (WF == LX2V_WFMT_Q4) {
        // element 2i in the low nibble of byte i (quant.rs:305-311)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t lo = w[q] & 0x0F0F0F0Fu, hi = (w[q] >> 4) & 0x0F0F0F0Fu;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const float e0 = ((float)((lo >> (8 * b)) & 0xFFu) - z) * s;
                const float e1 = ((float)((hi >> (8 * b)) & 0xFFu) - z) * s;
                o[4 * q + b] = pack_bf16x2(e0, e1);
            }
        }
    } else {
        // e4m3 through the hardware OCP decode; the reference decodes
        // exponent field 0 as m * 2^-12, an eighth of OCP's m * 2^-9.
#pragma unroll
        for (int q = 0; q < 4; q++) {
            typedef float f32x2_t __attribute__((ext_vector_type(2)));
            const f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[q], false);
            const f32x2_t b = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[q], true);
            float f[4] = {a.x, a.y, b.x, b.y};
            const uint32_t e = w[q] & 0x78787878u;
            if ((e - 0x01010101u) & ~e & 0x80808080u) {  // some byte has exponent field 0
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (((e >> (8 * k)) & 0xFFu) == 0) f[k] *= 0.125f;
            }
            o[2 * q] = pack_bf16x2(f[0] * s, f[1] * s);
            o[2 * q + 1] = pack_bf16x2(f[2] * s, f[3] * s);
        }
    }
}

}  // namespace

}  // namespace lx2v
