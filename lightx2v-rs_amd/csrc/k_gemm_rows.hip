// k_gemm_rows.hip -- Backend::linear over few activation rows
// (crates/lightx2v-core/src/backend.rs:198-212): every weight format on the
// MFMA that the tiled kernels use for it (k_gemm_fp8.hip, k_gemm_w16.hip),
// laid out for few rows beside the weight's bytes.
//
//   Y[m, n] = act( sum_k X[m, k] W[n, k] + bias[n] )
//
// A workgroup takes 32 MB rows (MB = 1 or 2) and 32 channels: the weight is
// read once for every 64 rows (up to 64 with FP8 weights on the fp8 MFMA, 256
// with the others).
//
// What bounds it: latency and the weight's bytes.  A tile of the other
// kernels walks all of K in one workgroup, 128 channels wide: at 17 rows,
// 1536 -> 1536 occupies 12 CUs for 12 serial stages (8.2 us), and 1536 <-
// 14336 for 112 (33 us).  Here a workgroup splits K over its eight waves in
// steps of 128 elements (64 where the operands of one take more registers;
// wave w: steps w, w + 8, ...).  Each wave loads its operands from global
// memory straight into MFMA fragments, one or two steps ahead of the one it
// contracts, with no LDS and no barrier; the eight partial sums meet once in
// LDS, in wave order, and the epilogue stores (6.0 and 22 us).
//
// Fragments: the activations are the MFMA's A operand and the weight its B
// operand, so a lane holds one channel (l % 32) and 16 rows, and a group's
// scale is one value per lane.  K within a step is taken in whatever order
// gives each lane contiguous bytes, the same for both operands:
//   fp8   slice kk (64 bytes): 16-byte chunks h and h + 2 (h = l / 32), which
//         for MX activations makes each lane half one 32-element scale block;
//   bf16  unit i (32 elements): elements 16 h .. 16 h + 15, the first eight in
//         one MFMA and the last eight in the next.
#include <algorithm>

#include "gemm_common.hpp"
#include "w16_dequant.hpp"

namespace lx2v {

namespace {

constexpr int RN = 32;    // channels per workgroup
constexpr int RW = 8;     // waves per workgroup
constexpr int RK = 128;   // K elements per step

struct RowsArgs {
    const void *x;
    const float *xs;                      // fp8: row scales (null: MX or none)
    const uint8_t *mxa;                   // fp8 MX: scale bytes (mx_sidx), of row 0
    uint32_t mxa_len, mxa_rows;
    const void *w;
    const float *cs;                      // channel scales [N] (null: none)
    const float *ws;                      // groups: the stage-major scales
    const float *wz;                      // Q4 zeros, stage-major
    int spr;
    const float *bias;
    const float *gate;                    // residual mode: Y += y * gate
    void *y;
    uint8_t *ymx;
    int ymx_rows;
    int M, N, K, act;
};

// h + y g, the product and the sum rounded apart, as linear followed by
// gate_residual rounds them.
__device__ __forceinline__ float gated(float h, float y, float g) {
#pragma clang fp contract(off)
    return h + y * g;
}

// One output value's epilogue and store.  Columns n0 .. n0 + 31 are 32
// consecutive lanes (an MX block).
template <int YDT>
__device__ __forceinline__ void rows_store(const RowsArgs &a, int m, int n, bool in, float v) {
    if (a.act == LX2V_ACT_GELU_TANH) v = gelu_tanh_fast(v);
    const size_t off = (size_t)m * a.N + n;
    if constexpr (YDT == LX2V_DTYPE_MXE4M3) {
        float amax = in ? fabsf(v) : 0.0f;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
        const int k = mx_exponent(amax);
        const float q[4] = {v, 0.0f, 0.0f, 0.0f};
        if (!in) return;
        ((uint8_t *)a.y)[off] = (uint8_t)quant4_sc(q, mx_scale(k));
        if (n % 32 == 0) a.ymx[mx_sidx(m, n / 32, a.ymx_rows)] = (uint8_t)(k + 127);
    } else if (!in) {
        return;
    } else if constexpr (YDT == LX2V_DTYPE_BF16) {
        uint16_t *p = (uint16_t *)a.y + off;
        const uint16_t r = f32_to_bf16_bits(v);
        *p = a.gate ? f32_to_bf16_bits(gated(bf16_bits_to_f32(*p), bf16_bits_to_f32(r), a.gate[n])) : r;
    } else {
        float *p = (float *)a.y + off;
        *p = a.gate ? gated(*p, v, a.gate[n]) : v;
    }
}

// The waves' partial sums acc (register e of lane l: row 32 b + 8 (e / 4) +
// 4 (l / 32) + e % 4, channel l % 32), added in wave order, and the epilogue.
template <int MB, int YDT>
__device__ __forceinline__ void rows_reduce(const RowsArgs &a, const f32x16 (&acc)[MB], float *red, int m0, int n0) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
        for (int e = 0; e < 16; e++) red[((wv * MB + b) * 16 + e) * 64 + lane] = acc[b][e];
    __syncthreads();
    const int n = n0 + (lane & 31);
    const float cs = a.cs && n < a.N ? a.cs[n] : 1.0f;
    const float bias = a.bias && n < a.N ? a.bias[n] : 0.0f;
#pragma unroll
    for (int q = 0; q < 2 * MB; q++) {
        const int b = q / 2, e = (q % 2) * 8 + wv;
        float v = red[(b * 16 + e) * 64 + lane];
#pragma unroll
        for (int p = 1; p < RW; p++) v += red[((p * MB + b) * 16 + e) * 64 + lane];
        const int m = m0 + 32 * b + 8 * (e / 4) + 4 * (lane >> 5) + e % 4;
        const bool in = m < a.M && n < a.N;
        const float s = a.xs ? a.xs[m < a.M ? m : 0] : 1.0f;
        rows_store<YDT>(a, m, n, in, v * s * cs + bias);
    }
}

// FP8 weight x e4m3 activations.  GS: weight scales per 128 columns (one per
// step, from the stage-major copy), applied to the step's sums; MXA: MX
// activations.
template <int MB, bool GS, bool MXA, int YDT>
__global__ __launch_bounds__(64 * RW) void k_gemm_rows_fp8(RowsArgs a) {
    __shared__ float red[RW * MB * 16 * 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, l32 = lane & 31, hf = lane >> 5;
    const int n0 = blockIdx.x * RN, m0 = blockIdx.y * (32 * MB);
    const uint32_t K = (uint32_t)a.K;
    const int steps = (a.K + RK - 1) / RK;
    // rows and channels past the matrices read zero
    const auto rx = make_rsrc((const uint8_t *)a.x + (size_t)m0 * K, (uint32_t)(a.M - m0) * K);
    const auto rw = make_rsrc((const uint8_t *)a.w + (size_t)n0 * K, (uint32_t)(a.N - n0) * K);
    const auto rs = make_rsrc(GS ? a.ws + n0 : a.cs, GS ? ((uint32_t)(a.K / 64) * (uint32_t)a.N - (uint32_t)n0) * 4u : 0u);
    const auto rm = make_rsrc(MXA ? a.mxa : (const uint8_t *)a.w, MXA ? a.mxa_len : 0u);
    const uint32_t wo = (uint32_t)l32 * K + 16u * hf;
    struct Step {
        u32x4 w[2][2], x[MB][2][2];
        uint32_t s, mx[MB];
    };
    auto load = [&](Step &f, int s) __attribute__((always_inline)) {
        const uint32_t k0 = (uint32_t)s * RK;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            const uint32_t k = k0 + 64u * kk, dead = s < steps && k < K ? 0u : kOob;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                f.w[kk][c] = buffer_load_x4(rw, (wo + k + 32u * c) | dead);
#pragma unroll
                for (int b = 0; b < MB; b++) f.x[b][kk][c] = buffer_load_x4(rx, (wo + 32u * b * K + k + 32u * c) | dead);
            }
        }
        if constexpr (GS) f.s = buffer_load_x1(rs, ((uint32_t)(2 * s) * (uint32_t)a.N + (uint32_t)l32) * 4u | (s < steps ? 0u : kOob));
        if constexpr (MXA)
#pragma unroll
            for (int b = 0; b < MB; b++)
                f.mx[b] = buffer_load_x1(rm, ((uint32_t)s * a.mxa_rows + (uint32_t)(m0 + 32 * b + l32)) * 4u | (s < steps ? 0u : kOob));
    };
    f32x16 acc[MB];
#pragma unroll
    for (int b = 0; b < MB; b++) acc[b] = (f32x16){};
    auto as8 = [](const u32x4 (&p)[2]) {
        return (i32x8){(int)p[0].x, (int)p[0].y, (int)p[0].z, (int)p[0].w, (int)p[1].x, (int)p[1].y, (int)p[1].z, (int)p[1].w};
    };
    auto contract = [&](const Step &f) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < MB; b++) {
            f32x16 t = GS ? (f32x16){} : acc[b];
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                if constexpr (MXA)
                    t = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(as8(f.x[b][kk]), as8(f.w[kk]), t, 0, 0, 0,
                                                                        (int)(f.mx[b] >> (8 * (2 * kk + hf))), 0, 0x7F);
                else
                    t = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(as8(f.x[b][kk]), as8(f.w[kk]), t, 0, 0, 0, 0, 0, 0);
            }
            if constexpr (GS) {
#pragma unroll
                for (int e = 0; e < 16; e++) acc[b][e] = __builtin_fmaf(t[e], __uint_as_float(f.s), acc[b][e]);
            } else {
                acc[b] = t;
            }
        }
    };
    Step f[3];
    load(f[0], wv);
    load(f[1], wv + RW);
    for (int s = wv; s < steps; s += 3 * RW) {
        static_for<3>([&](auto i) {
            constexpr int I = decltype(i)::value;
            load(f[(I + 2) % 3], s + (I + 2) * RW);
            contract(f[I]);
        });
    }
    rows_reduce<MB, YDT>(a, acc, red, m0, n0);
}

// Weights dequantized to bf16 (Q8, Q4, FP8 groups; native: the bf16 copy) x
// bf16 activations (f32 ones rounded as they are loaded).
constexpr int kWfmtBf16 = 101;  // the native weight's bf16 copy (a format id of this file only)

template <int WF, int MB, int XT, int YDT>
__global__ __launch_bounds__(64 * RW) void k_gemm_rows_w16(RowsArgs a) {
    constexpr bool Q4 = WF == LX2V_WFMT_Q4 || WF == kWfmtQ4Sym, ZL = WF == LX2V_WFMT_Q4, NATIVE = WF == kWfmtBf16;
    constexpr int WR = NATIVE ? 2 : 1;                         // 16-byte loads of 16 weights (Q4: 8 bytes)
    constexpr int XE = XT == LX2V_DTYPE_BF16 ? 2 : 4, XR = XE;  // bytes per activation; 16-byte loads of 16
    // units per step and steps held, by the registers a step takes
    constexpr int UR = WR * 4 + (NATIVE ? 0 : 1 + ZL) + MB * XR * 4, U = 4 * UR > 90 ? 2 : 4, ND = U * UR > 56 ? 2 : 3;
    constexpr int RKU = 32 * U;
    __shared__ float red[RW * MB * 16 * 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, l32 = lane & 31, hf = lane >> 5;
    const int n0 = blockIdx.x * RN, m0 = blockIdx.y * (32 * MB);
    const uint32_t K = (uint32_t)a.K, wrow = Q4 ? K / 2 : (NATIVE ? K * 2 : K);  // bytes per weight row
    const int steps = (a.K + RKU - 1) / RKU;
    const auto rx = make_rsrc((const uint8_t *)a.x + (size_t)m0 * K * XE, (uint32_t)(a.M - m0) * K * XE);
    const auto rw = make_rsrc((const uint8_t *)a.w + (size_t)n0 * wrow, (uint32_t)(a.N - n0) * wrow);
    const uint32_t slen = NATIVE ? 0u : ((uint32_t)(a.K / 64) * (uint32_t)a.N) * (uint32_t)a.spr * 4u;
    const auto rs = make_rsrc(a.ws, slen), rz = make_rsrc(ZL ? a.wz : a.ws, ZL ? slen : 0u);
    struct Step {
        u32x4 w[U][WR], x[MB][U][XR];
        uint32_t s[U], z[U];
    };
    auto load = [&](Step &f, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < U; i++) {
            const uint32_t k = (uint32_t)s * RKU + 32u * i, ku = k + 16u * hf, dead = s < steps && k < K ? 0u : kOob;
            const uint32_t wo = (uint32_t)l32 * wrow + (Q4 ? ku / 2 : (NATIVE ? ku * 2 : ku));
            if constexpr (Q4) {
                const u32x2 h = buffer_load_x2(rw, wo | dead);
                f.w[i][0] = (u32x4){h.x, h.y, 0u, 0u};
            } else {
#pragma unroll
                for (int r = 0; r < WR; r++) f.w[i][r] = buffer_load_x4(rw, (wo + 16u * r) | dead);
            }
            if constexpr (!NATIVE) {
                const uint32_t u64 = (ku % 64) / 16, so =
                    (((k / 64) * (uint32_t)a.N + (uint32_t)(n0 + l32)) * (uint32_t)a.spr + ((u64 * (uint32_t)a.spr) >> 2)) * 4u | dead;
                f.s[i] = buffer_load_x1(rs, so);
                if constexpr (ZL) f.z[i] = buffer_load_x1(rz, so);
            }
#pragma unroll
            for (int b = 0; b < MB; b++)
#pragma unroll
                for (int r = 0; r < XR; r++)
                    f.x[b][i][r] = buffer_load_x4(rx, (((uint32_t)(32 * b + l32) * K + ku) * XE + 16u * r) | dead);
        }
    };
    f32x16 acc[MB];
#pragma unroll
    for (int b = 0; b < MB; b++) acc[b] = (f32x16){};
    // (a call of it would put every Step in scratch memory: left to itself the
    // compiler made one for FP8 weights with f32 rows, 62 us for 11 at 17 x 1536
    // -> 1536)
    auto contract = [&](const Step &f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < U; i++) {
            u32x4 w[2];
            if constexpr (NATIVE) {
                w[0] = f.w[i][0];
                w[1] = f.w[i][WR - 1];
            } else {
                uint32_t o[8];
                unit_dequant<WF>(f.w[i][0], __uint_as_float(f.s[i]), ZL ? __uint_as_float(f.z[i]) : 0.0f, o);
                w[0] = (u32x4){o[0], o[1], o[2], o[3]};
                w[1] = (u32x4){o[4], o[5], o[6], o[7]};
            }
#pragma unroll
            for (int b = 0; b < MB; b++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    u32x4 x;
                    if constexpr (XT == LX2V_DTYPE_BF16) {
                        x = f.x[b][i][h];
                    } else {
                        const f32x4 p = __builtin_bit_cast(f32x4, f.x[b][i][2 * h]), q = __builtin_bit_cast(f32x4, f.x[b][i][2 * h + 1]);
                        x = (u32x4){pack_bf16x2(p.x, p.y), pack_bf16x2(p.z, p.w), pack_bf16x2(q.x, q.y), pack_bf16x2(q.z, q.w)};
                    }
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, w[h]),
                                                                   acc[b], 0, 0, 0);
                }
        }
    };
    Step f[ND];
    static_for<ND - 1>([&](auto i) { load(f[decltype(i)::value], wv + decltype(i)::value * RW); });
    for (int s = wv; s < steps; s += ND * RW) {
        static_for<ND>([&](auto i) {
            constexpr int I = decltype(i)::value;
            load(f[(I + ND - 1) % ND], s + (I + ND - 1) * RW);
            contract(f[I]);
        });
    }
    rows_reduce<MB, YDT>(a, acc, red, m0, n0);
}

template <int MB, bool GS, bool MXA>
void launch_rows_fp8_y(hipStream_t s, dim3 grid, const RowsArgs &a, int y_dtype) {
    if (y_dtype == LX2V_DTYPE_BF16)
        hipLaunchKernelGGL((k_gemm_rows_fp8<MB, GS, MXA, LX2V_DTYPE_BF16>), grid, dim3(64 * RW), 0, s, a);
    else if (y_dtype == LX2V_DTYPE_MXE4M3)
        hipLaunchKernelGGL((k_gemm_rows_fp8<MB, GS, MXA, LX2V_DTYPE_MXE4M3>), grid, dim3(64 * RW), 0, s, a);
    else
        hipLaunchKernelGGL((k_gemm_rows_fp8<MB, GS, MXA, LX2V_DTYPE_F32>), grid, dim3(64 * RW), 0, s, a);
}
template <int MB>
void launch_rows_fp8_mb(hipStream_t s, dim3 grid, const RowsArgs &a, int y_dtype, bool gs) {
    if (gs)
        a.mxa ? launch_rows_fp8_y<MB, true, true>(s, grid, a, y_dtype) : launch_rows_fp8_y<MB, true, false>(s, grid, a, y_dtype);
    else
        a.mxa ? launch_rows_fp8_y<MB, false, true>(s, grid, a, y_dtype) : launch_rows_fp8_y<MB, false, false>(s, grid, a, y_dtype);
}
template <int WF, int MB, int XT>
void launch_rows_w16_y(hipStream_t s, dim3 grid, const RowsArgs &a, int y_dtype) {
    if (y_dtype == LX2V_DTYPE_BF16)
        hipLaunchKernelGGL((k_gemm_rows_w16<WF, MB, XT, LX2V_DTYPE_BF16>), grid, dim3(64 * RW), 0, s, a);
    else
        hipLaunchKernelGGL((k_gemm_rows_w16<WF, MB, XT, LX2V_DTYPE_F32>), grid, dim3(64 * RW), 0, s, a);
}
template <int WF>
void launch_rows_w16_x(hipStream_t s, dim3 grid, const RowsArgs &a, int x_dtype, int y_dtype, bool two) {
    if (x_dtype == LX2V_DTYPE_BF16)
        two ? launch_rows_w16_y<WF, 2, LX2V_DTYPE_BF16>(s, grid, a, y_dtype) : launch_rows_w16_y<WF, 1, LX2V_DTYPE_BF16>(s, grid, a, y_dtype);
    else
        two ? launch_rows_w16_y<WF, 2, LX2V_DTYPE_F32>(s, grid, a, y_dtype) : launch_rows_w16_y<WF, 1, LX2V_DTYPE_F32>(s, grid, a, y_dtype);
}

dim3 rows_grid(size_t M, size_t N, int mb) {
    return dim3((unsigned)((N + RN - 1) / RN), (unsigned)((M + 32 * mb - 1) / (32 * mb)));
}

}  // namespace

size_t gemm_rows_limit(RowsKind kind) {
    const char *e = getenv("LIGHTX2V_HIP_ROWS");
    return e && *e ? (size_t)std::max(0, atoi(e)) : kind <= RowsKind::Fp8Scaled ? 64 : 256;
}

namespace {

// The modelled time of a call among others, by the most rows a workgroup takes
// (32 or 64): `us` a step of a wave's share of K (K / 1024 rounded up), plus, per
// 1024 of K, `row` for each row loaded and `busy` where every CU reads its part
// of the weight; a CU runs one workgroup at a time, so all of it once more for
// every 256 workgroups.  Fitted over 512 .. 14336 x 64 .. 14336 (M 1 .. 256, weights
// hot and cold): rms 4 to 12%.
struct RowsCost {
    double base, us, row, busy;
};
constexpr RowsCost kRowsCost[][2] = {
    {{4.8, 0.83, 0.024, 0.44}, {4.9, 0.93, 0.027, 1.17}},  // Fp8
    {{4.7, 0.93, 0.024, 0.55}, {4.6, 1.15, 0.028, 1.10}},  // Fp8Scaled
    {{5.3, 1.63, 0.042, 1.15}, {4.1, 2.55, 0.032, 1.56}},  // W16
    {{4.2, 1.06, 0.134, 1.30}, {3.6, 3.21, 0.081, 0.85}},  // W16F32
    {{4.1, 1.93, 0.048, 0.65}, {5.2, 2.18, 0.047, 1.18}},  // Native
    {{4.5, 2.25, 0.087, 0.91}, {4.5, 3.00, 0.090, 0.91}},  // NativeF32
};

double rows_cost_us(RowsKind kind, int num_cu, size_t M, size_t N, size_t K) {
    const RowsCost &c = kRowsCost[(int)kind][M > 32];
    const size_t cols = (N + RN - 1) / RN, blocks = (M + 63) / 64, wg = cols * blocks, rounds = (wg + num_cu - 1) / num_cu;
    const double own = (double)((K + 1023) / 1024), kf = (double)K / 1024;
    const double per = own * c.us + kf * (c.row * (double)std::min<size_t>(M, 64) + c.busy * std::min(1.0, (double)wg / num_cu));
    double n = (double)rounds;
    if (rounds > 1 && blocks > 1 && wg - (rounds - 1) * num_cu <= cols)  // the last round: the last block's rows only
        n += (double)std::max<size_t>(M - 64 * (blocks - 1), 16) / 64 - 1.0;
    return c.base + n * per;
}

}  // namespace

// Where the tiles leave CUs idle over a long K and there are few rows to load
// beside the weight's.  Rows / the other kernels (us, other_us): FP8, e4m3
// input, 17 x 14336 -> 3072 22 / 29, 33 x 14336 -> 3072 36 / 29; group 128, 64 x
// 1536 -> 8960 19 / 11; Q8, 17 x 1536 -> 1536 9 / 13, 200 x 14336 -> 3072 147 /
// 77, f32 rows 64 x 14336 -> 1536 130 / 71.  Over 2100 shapes the kernel taken
// is on average 0.6% slower than the fastest.
// LIGHTX2V_HIP_ROWS=<n> takes it for every call of up to n rows instead.
bool gemm_rows_chosen(RowsKind kind, int num_cu, size_t M, size_t N, size_t K, double other_us) {
    if (K % 64 || N == 0 || M == 0) return false;
    // 32-bit offsets into the rows as they are (the tiles read f32 ones as bf16)
    if ((kind == RowsKind::W16F32 || kind == RowsKind::NativeF32) && M * K * 4 >= (1ull << 31)) return false;
    if (M > gemm_rows_limit(kind)) return false;
    // a pinned tile configuration stays the tile kernels'
    const char *pin = getenv(kind <= RowsKind::Fp8Scaled ? "LIGHTX2V_HIP_FP8_CFG"
                             : kind <= RowsKind::W16F32  ? "LIGHTX2V_HIP_W16_CFG"
                                                         : "LIGHTX2V_HIP_BF16_CFG");
    if (pin && *pin && atoi(pin) >= 0) return false;
    const char *e = getenv("LIGHTX2V_HIP_ROWS");
    if (e && *e) return true;
    // (a native call's choices lie within a microsecond where K is short: there the
    // tiles, which sum every row the same way whatever the row count, keep it)
    return rows_cost_us(kind, num_cu, M, N, K) < (kind == RowsKind::NativeF32 ? 0.9 : 1.0) * other_us;
}

void launch_gemm_rows_fp8(hipStream_t s, const uint8_t *x, const float *x_scale, const lx2v_hip_weight *w, bool grouped,
                          const float *bias, int act, void *y, int y_dtype, size_t M, const Fp8Mx &mx) {
    RowsArgs a{};
    a.x = x;
    a.xs = x_scale;
    a.mxa = mx.a;
    a.mxa_len = (uint32_t)mx.a_len;
    a.mxa_rows = (uint32_t)mx.a_rows;
    a.w = w->codes;
    (grouped ? a.ws : a.cs) = grouped ? w->sscale : w->scales;
    a.bias = bias;
    a.gate = mx.gate;
    a.y = y;
    a.ymx = mx.y;
    a.ymx_rows = (int)mx.y_rows;
    a.M = (int)M;
    a.N = (int)w->rows;
    a.K = (int)w->cols;
    a.act = act;
    if (M > 32)
        launch_rows_fp8_mb<2>(s, rows_grid(M, w->rows, 2), a, y_dtype, grouped);
    else
        launch_rows_fp8_mb<1>(s, rows_grid(M, w->rows, 1), a, y_dtype, grouped);
}

void launch_gemm_rows_w16(hipStream_t s, const void *x, int x_dtype, const lx2v_hip_weight *w, const float *bias, int act,
                          void *y, int y_dtype, size_t M) {
    RowsArgs a{};
    a.x = x;
    a.ws = w->sscale;
    a.wz = w->szero;
    a.spr = w->spr;
    a.bias = bias;
    a.y = y;
    a.M = (int)M;
    a.N = (int)w->rows;
    a.K = (int)w->cols;
    a.act = act;
    const bool two = M > 32;
    const dim3 grid = rows_grid(M, w->rows, two ? 2 : 1);
    a.w = w->fmt == LX2V_WFMT_F32 ? (const void *)w->wbf16 : w->codes;
    switch (w->fmt) {
        case LX2V_WFMT_F32: launch_rows_w16_x<kWfmtBf16>(s, grid, a, x_dtype, y_dtype, two); break;
        case LX2V_WFMT_Q8: launch_rows_w16_x<LX2V_WFMT_Q8>(s, grid, a, x_dtype, y_dtype, two); break;
        case LX2V_WFMT_Q4:
            if (w->zero8)
                launch_rows_w16_x<kWfmtQ4Sym>(s, grid, a, x_dtype, y_dtype, two);
            else
                launch_rows_w16_x<LX2V_WFMT_Q4>(s, grid, a, x_dtype, y_dtype, two);
            break;
        default: launch_rows_w16_x<LX2V_WFMT_FP8>(s, grid, a, x_dtype, y_dtype, two); break;
    }
}

}  // namespace lx2v
