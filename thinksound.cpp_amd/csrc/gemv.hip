// gemv.hip — ggml_mul_mat over a few activation rows (src/mmdit.cpp:12-16 on
// the conditioning vectors: the t_embed, adaLN and global-conditioning
// layers run on one row per batch item):
//
//   Y[n, m] = sum_k X[n, k] * W[m, k] + bias[m],  n < N <= 8
//
// The weights are read once and nothing else counts, so every weight load of
// the launch should be in flight at once: one wave per R weight rows, 8
// consecutive k per lane, no LDS, and the activations converted to the
// weight's vec_dot type (bf16, Q8_0 blocks) by every wave for itself instead
// of in a launch of their own. A tile kernel walks K alone in M / 64
// workgroups: 2 rows, 1024 -> 6144 BF16 9.8 -> 4.2 us with its conversion
// launch (3.3 us is an empty launch's rate), Q8_0 10.9 -> 5.6, F32 24.5 -> 4.4.
#include "tsk_common.h"
#include "tsk_internal.h"
#include "tsk_runtime.h"

namespace tsk {

namespace {

enum class GW { BF16, F32, Q8 };

__device__ __forceinline__ int quad_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);
    return v + __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);
}

// 8 activations of row n from k on as f32
template <bool XBF16>
__device__ __forceinline__ void load_x8(const GemvRows &p, int n, int k, float (&v)[8]) {
    if constexpr (XBF16) {
        const u32x4 raw = *(const u32x4 *) ((const uint16_t *) p.x + (int64_t) n * p.ld_x + k);
        const uint16_t *h = (const uint16_t *) &raw;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = bf16_bits_to_f32(h[e]);
    } else {
        const float *xr = (const float *) p.x + (int64_t) n * p.ld_x + k;
        const f32x4 a = *(const f32x4 *) xr, b = *(const f32x4 *) (xr + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    }
}

template <GW W, bool XBF16, int R, int NMAX>
__global__ __launch_bounds__(256) void gemv_rows_kernel(const GemvRows p) {
    const int lane = threadIdx.x & 63;
    const int m0 = ((int) blockIdx.x * 4 + (int) (threadIdx.x >> 6)) * R;
    if (m0 >= p.M) return;                                    // whole waves
    float acc[R][NMAX];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < NMAX; ++n) acc[r][n] = 0.0f;
    // No branch in a step, so that the loads of two are issued together (the lane
    // exchanges of a Q8_0 step keep two from being merged): lanes
    // past K load their first chunk and drop it, rows past N repeat the last
#pragma unroll W == GW::Q8 ? 1 : 2
    for (int k0 = 0; k0 < p.K; k0 += 512) {
        const int kl = k0 + 8 * lane;
        const bool in = kl < p.K;                             // Q8_0: the same for a block's four lanes (K % 32 == 0)
        const int k = in ? kl : 0;
        float wv[R][8], xv[NMAX][8];
        u32x2 wq[R];
        float wd[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t m = min(m0 + r, p.M - 1);
            if constexpr (W == GW::BF16) {
                const u32x4 raw = *(const u32x4 *) ((const uint16_t *) p.w + m * p.ld_w + k);
                const uint16_t *h = (const uint16_t *) &raw;
#pragma unroll
                for (int e = 0; e < 8; ++e) wv[r][e] = bf16_bits_to_f32(h[e]);
            } else if constexpr (W == GW::F32) {
                const float *wr = (const float *) p.w + m * p.ld_w + k;
                const f32x4 a = *(const f32x4 *) wr, b = *(const f32x4 *) (wr + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    wv[r][e] = a[e];
                    wv[r][4 + e] = b[e];
                }
            } else {
                wq[r] = *(const u32x2 *) (p.qw + m * p.K + k);
                wd[r] = f16_bits_to_f32(p.dw[m * (p.K / 32) + k / 32]);
            }
        }
#pragma unroll
        for (int n = 0; n < NMAX; ++n) load_x8<XBF16>(p, min(n, p.N - 1), k, xv[n]);
        if constexpr (W != GW::Q8) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int e = 0; e < 8; ++e) wv[r][e] = in ? wv[r][e] : 0.0f;
        }
#pragma unroll
        for (int n = 0; n < NMAX; ++n) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = in ? xv[n][e] : 0.0f;
            if constexpr (W == GW::Q8) {
                // ggml-cpu's x86 Q8_0 conversion of the block (quantize_rows_q8_kernel's arithmetic)
                float am = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(v[e]));
                am = fmaxf(am, dpp_f(am, 0));
                am = fmaxf(am, dpp_f(am, 1));
                const float id = am != 0.0f ? 127.0f / am : 0.0f;
                const float dx = f16_bits_to_f32(f32_to_f16_bits(am / 127.0f));
                int8_t q[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) q[e] = (int8_t) __builtin_rintf(v[e] * id);
                u32x2 xq;
                __builtin_memcpy(&xq, q, 8);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int s = __builtin_amdgcn_sdot4((int) wq[r][1], (int) xq[1],
                                                         __builtin_amdgcn_sdot4((int) wq[r][0], (int) xq[0], 0, false), false);
                    const float t = (float) quad_sum(s) * (wd[r] * dx);
                    acc[r][n] += in && (lane & 3) == 0 ? t : 0.0f;
                }
            } else {
                if constexpr (W == GW::BF16 && !XBF16) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = bf16_bits_to_f32(f32_to_bf16_bits(v[e]));
                }
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[r][n] = fmaf(wv[r][e], v[e], acc[r][n]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int m = m0 + r;
#pragma unroll
        for (int n = 0; n < NMAX; ++n) {
            const float s = wave_sum(acc[r][n]);
            if (lane == 0 && m < p.M && n < p.N) {
                const float o = s + (p.bias ? p.bias[m] : 0.0f);
                if (p.y_bf16) ((uint16_t *) p.y)[(int64_t) n * p.ld_y + m] = f32_to_bf16_bits(o);
                else ((float *) p.y)[(int64_t) n * p.ld_y + m] = o;
            }
        }
    }
}

template <GW W, bool XBF16, int NMAX>
void launch_rows(const GemvRows &p, hipStream_t s) {
    // rows per wave: two share a wave's conversion of the activations where
    // that still leaves two waves per SIMD (2 rows, BF16, us with 1 / 2 / 4:
    // M = 6144 4.7 / 4.2 / 4.9, M = 1024 3.8 / 3.7 / 4.6; 8 rows 11.7 / 9.8 /
    // 11.7, 5.5 / 6.9 / 10.1)
    if (p.M >= 4096) launch_kernel((gemv_rows_kernel<W, XBF16, 2, NMAX>), dim3((p.M + 7) / 8), dim3(256), 0, s, p);
    else launch_kernel((gemv_rows_kernel<W, XBF16, 1, NMAX>), dim3((p.M + 3) / 4), dim3(256), 0, s, p);
}
template <GW W, bool XBF16>
void launch_n(const GemvRows &p, hipStream_t s) {
    if (p.N == 1) launch_rows<W, XBF16, 1>(p, s);
    else if (p.N == 2) launch_rows<W, XBF16, 2>(p, s);
    else if (p.N <= 4) launch_rows<W, XBF16, 4>(p, s);
    else launch_rows<W, XBF16, 8>(p, s);
}

}  // namespace

hipError_t launch_gemv_rows(const GemvRows &p, hipStream_t s) {
    const bool q8 = p.qw != nullptr;
    if (p.N < 1 || p.N > GEMV_MAX_ROWS || p.M < 1 || p.K < 8 || p.K % (q8 ? 32 : 8) || !p.x || !p.y || (q8 ? !p.dw : !p.w) ||
        p.M > (1 << 30))
        return hipErrorInvalidValue;
    if (q8) p.x_bf16 ? launch_n<GW::Q8, true>(p, s) : launch_n<GW::Q8, false>(p, s);
    else if (p.w_f32) launch_n<GW::F32, false>(p, s);
    else p.x_bf16 ? launch_n<GW::BF16, true>(p, s) : launch_n<GW::BF16, false>(p, s);
    return hipGetLastError();
}

}  // namespace tsk
