// gemm_split.hip — products of F32 operands on the 16-bit matrix cores of
// gfx950 (the VAE's convolutions, src/vae_decoder.cpp:26-58, and the F32
// weights of ggml_mul_mat / conv_cl, src/mmdit.cpp:13-34):
//
//   Y[n, m] = sum_k X[n, k] * W[m, k] + bias[m]
//
// Every operand value v is held as two halves of its scaled value: with e the
// exponent of a bound on |v| over its row or tensor, s = v * 2^(15 - e) (exact;
// |s| < 2^15), hi = fp16(s), lo = fp16(s - hi). s - hi is exact, so hi + lo is s
// to 2^-23 of s (or 2^-25 absolute where lo is subnormal: 2^-40 of the bound).
// Three fp16 MFMAs sum x_hi w_hi + x_hi w_lo + x_lo w_hi in fp32; what is left
// out, x_lo w_lo, is at most 2^-22 of |x w| with a random sign per term, below
// what summing K terms in fp32 rounds away, and one MFMA adds 32 products with
// one rounding of the sum where the fp32 MFMA adds 4. Against 64-bit results
// the products are as close as the fp32 MFMA's or closer (measured: 30 s VAE
// decode 1.2e-4 with fp32 MFMAs, see the drivers' tests), at 2.5 PFLOP/s / 3
// against 157 TFLOP/s.
//
// Layout: a row of C values (C % 32 == 0) is C 4-byte words in groups of 32 values, one
// 128-byte line each: [32 hi][32 lo]. So rows, strides and bytes are those of
// the f32 rows, and a 32-wide K step of a row is one line.
#include <algorithm>

#include "tsk_common.h"
#include "tsk_internal.h"
#include "tsk_runtime.h"

namespace tsk {

namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((__vector_size__(4 * sizeof(_Float16)))) _Float16 f16x4;

constexpr int NT = 256;
constexpr int BK = 32;

__device__ __forceinline__ bool finite_f(float v) { return fabsf(v) <= 3.4028234664e38f; }

// the smallest e with b < 2^e (b >= 0), from -112 on: 2^(15 - e) stays finite
__device__ __forceinline__ int bound_exp(float b) {
    const int e = (int) (__float_as_uint(b) >> 23) - 126;
    return e < -112 ? -112 : e;
}
__device__ __forceinline__ float exp2_int(int e) { return __uint_as_float((uint32_t) (e + 127) << 23); }

__device__ __forceinline__ void split4(const float (&v)[4], float scale, f16x4 &hi, f16x4 &lo) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float s = v[r] * scale;
        hi[r] = (_Float16) s;
        lo[r] = (_Float16) (s - (float) hi[r]);
    }
}
// word offset of channel c's group and the halfword of its hi inside a split row
__device__ __forceinline__ void store_split4(uint32_t *row, int c, const f16x4 hi, const f16x4 lo) {
    uint16_t *g = (uint16_t *) (row + (c & ~31)) + (c & 31);
    *(f16x4 *) g = hi;
    *(f16x4 *) (g + 32) = lo;
}

// sin(a)^2 of four values. The argument modulo pi: a - n pi with n = rint(a / pi)
// and pi in two parts (Cody and Waite; the fused products are exact), then an
// odd polynomial of degree 9 for sin on [-pi/2, pi/2] (least squares weighted
// to a minimax fit, 6e-9 relative): 14 instructions where sinf takes about 40.
// Measured against 64 bits: rms 3.7e-8, max 3e-7 up to |a| = 1e6 (sinf: 2.9e-8,
// 1.2e-7; the fp32 a itself is off by 2^-25 |a|). Larger and non-finite
// arguments go through sinf.
__device__ __forceinline__ void sin2_x4(const float (&a)[4], float (&s2)[4]) {
    bool small = true;
#pragma unroll
    for (int r = 0; r < 4; ++r) small = small && fabsf(a[r]) < 524288.0f;
    if (small) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float n = __builtin_rintf(a[r] * 0.31830988618f);
            const float x = fmaf(n, 8.7422777e-8f, fmaf(n, -3.14159274f, a[r]));
            const float z = x * x;
            const float q = fmaf(fmaf(fmaf(2.6056309093e-6f, z, -1.9809538876e-4f), z, 8.3330654288e-3f), z, -1.6666659521e-1f);
            const float sn = fmaf(x * z, q, x);
            s2[r] = sn * sn;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float sn = sinf(a[r]);
            s2[r] = sn * sn;
        }
    }
}

// raise a slot to m (>= 0, finite): the slot only grows, so a stale read can
// only cause an atomic that changes nothing
__device__ __forceinline__ void raise_slot(float *slot, float m) {
    if (m > __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax((int *) slot, __float_as_int(m));
}

// fp32 product of one output, for results that are not finite in the split
// products: an infinity or NaN in its operands (finite ones cannot overflow:
// |s| < 2^15). The f32 operands give what fp32 products give.
__device__ __forceinline__ float f32_dot(const SplitGemm &p, int m, int n, int k0, int k1) {
    float s = 0.0f;
    const float *w = m < p.wf_rows ? p.wf + (int64_t) m * p.ld_wf : p.wf2 + (int64_t) (m - p.wf_rows) * p.ld_wf;
    if (p.conv_ic) {
        const int b = n / p.conv_ow, o = n - b * p.conv_ow;
        for (int k = k0; k < k1; ++k) {
            const int kw = k / p.conv_ic, ic = k - kw * p.conv_ic;
            const int iw = o * p.conv_s + kw * p.conv_d - p.conv_p;
            if (iw >= 0 && iw < p.conv_iw) s = fmaf(p.xf[(int64_t) b * p.xf_batch + (int64_t) iw * p.ld_xf + ic], w[k], s);
        }
    } else {
        for (int k = k0; k < k1; ++k) s = fmaf(p.xf[(int64_t) n * p.ld_xf + k], w[k], s);
    }
    return s;
}

// UNIT: a residual unit of the VAE in one launch where its channels fit one
// tile (M <= 128, M % 32 == 0): the tile's convolution, bias and SnakeBeta stay in
// the workgroup (split at the tile's own exponent into the ring's LDS, in the
// layout of M / 32 activation steps) and are the operand of the k1 convolution
// (w2, its fragments straight from L2 into registers). As two launches the
// k1's was bound by its four passes over the activations (30 s, 128 channels,
// 1.3 M frames: 980 + 790 us); one launch reads the snake once and writes the
// residual and the next snake.
//
// Workgroup = 2 x 2 waves of TM x TN 16x16 tiles; operand lines by direct
// global -> LDS loads into a two-stage ring of 32-wide K steps (line chunk c of
// a row at slot c ^ ((row / 2) % 8): the 16 rows of a fragment read hit
// distinct banks). Per step and 64 x 64 wave tile: 16 16-byte LDS reads for 48
// MFMAs of 16 cycles; two workgroups per CU.
template <int TM, int TN, int WPC, bool SNAKE, bool UNIT>
__global__ __launch_bounds__(NT, WPC) void gemm_split_kernel(const SplitGemm p) {
    constexpr int BM = 2 * TM * 16, BN = 2 * TN * 16;
    constexpr int ROWS = BM + BN, STAGE = ROWS * BK;          // words per stage
    constexpr int NWL = ROWS / 8, WLW = NWL / 4;             // wave-loads (8 rows) per stage, per wave
    static_assert(NWL % 4 == 0, "whole wave-loads per wave");
    constexpr int LDT = BM + 4;
    constexpr int RING = 2 * STAGE, EPI_F = BN * LDT;
    __shared__ __attribute__((aligned(16))) float smem[RING > EPI_F ? RING : EPI_F];

    // workgroup -> tile. L % 8 is the XCD: each takes a consecutive eighth of
    // the tiles in (slice, larger operand, smaller operand) order, so that the
    // tiles it runs at one time share one K slice and a block of both operands
    // in its L2
    int tm, tn, z;
    {
        const int L = (int) blockIdx.x, T = p.tiles_m * p.tiles_n;
        const int u = (L & 7) * p.per_xcd + (L >> 3);
        if (u >= T * p.splits) return;
        z = u / T;
        const int t = u - z * T;
        tm = p.m_inner ? t % p.tiles_m : t / p.tiles_n;
        tn = p.m_inner ? t / p.tiles_m : t % p.tiles_n;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    const int bm0 = tm * BM, bn0 = tn * BN;

    // activation rows relative to the tile's first row, so that 32-bit byte
    // offsets reach every row of the tile whatever the tensor's size
    int64_t r0 = bn0;
    if (p.conv_ic) {
        const int b = bn0 / p.conv_ow, o = bn0 - b * p.conv_ow;
        r0 = (int64_t) b * p.conv_iw + min(max(o * p.conv_s - p.conv_p, 0), p.conv_iw - 1);
    }
    const int64_t x_left = (p.x_rows - r0) * p.ld_x * 4;
    const int x_range = (int) min(x_left, (int64_t) 0x7fffffff);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        (void *) p.w, (short) 0, (int) ((int64_t) p.M * p.ld_w * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        (void *) (p.x + r0 * p.ld_x), (short) 0, x_range, 0x00020000);
    constexpr uint32_t PAST = 0x80000000u;                   // beyond every range: reads zero
    uint32_t voff[WLW];                                      // byte offsets of this lane's chunks
    bool isw[WLW];                                           // wave-uniform
    int xb[WLW], xi[WLW];                                    // activation rows: item's first row - r0, first position
#pragma unroll
    for (int q = 0; q < WLW; ++q) {
        const int j = wave * WLW + q, R = 8 * j + (lane >> 3);
        const uint32_t c16 = (uint32_t) ((lane & 7) ^ ((R >> 1) & 7)) * 16;
        xb[q] = xi[q] = 0;
        isw[q] = j < BM / 8;
        if (isw[q]) {
            voff[q] = bm0 + R < p.M ? (uint32_t) ((int64_t) (bm0 + R) * p.ld_w * 4) + c16 : PAST;
        } else {
            const int n = bn0 + R - BM;
            if (p.conv_ic) {
                const int b = n / p.conv_ow, o = n - b * p.conv_ow;
                xb[q] = (int) ((int64_t) b * p.conv_iw - r0);
                xi[q] = n < p.N ? o * p.conv_s - p.conv_p : INT32_MIN / 2;
            } else {
                voff[q] = n < p.N ? (uint32_t) (((int64_t) n - r0) * p.ld_x * 4) + c16 : PAST;
            }
        }
    }
    const int nk_all = p.K / BK, kt0 = (int) ((int64_t) z * nk_all / p.splits);
    const int nk = (int) ((int64_t) (z + 1) * nk_all / p.splits) - kt0;
    // the tap and channel step of the next load
    int ic_left = 0, kw = 0;
    uint32_t sw = (uint32_t) kt0 * 128, sx = sw;
    auto set_tap = [&]() {
#pragma unroll
        for (int q = 0; q < WLW; ++q) {
            if (isw[q]) continue;
            const int R = 8 * (wave * WLW + q) + (lane >> 3);
            const int iw = xi[q] + kw * p.conv_d;
            const uint32_t c16 = (uint32_t) ((lane & 7) ^ ((R >> 1) & 7)) * 16;
            voff[q] = iw >= 0 && iw < p.conv_iw ? (uint32_t) ((xb[q] + iw) * (int) p.ld_x * 4) + c16 : PAST;
        }
    };
    if (p.conv_ic) {
        const int steps = p.conv_ic / BK;
        kw = kt0 / steps;
        sx = (uint32_t) (kt0 - kw * steps) * 128;
        ic_left = steps - (kt0 - kw * steps);
        set_tap();
    }
    auto issue = [&](int slot) {
        float *st = smem + slot * STAGE;
#pragma unroll
        for (int q = 0; q < WLW; ++q) {
            // (arguments of template-dependent type, voff[q] itself, would leave
            // the kernel uninstantiated on the host side)
            const int j = wave * WLW + q;
            const uint32_t off = voff[q];
            if (isw[q])
                __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (lds_void *) (st + j * 8 * BK), 16, off, sw, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (lds_void *) (st + j * 8 * BK), 16, off, sx, 0, 0);
        }
        sw += 128;
        sx += 128;
        if (p.conv_ic && --ic_left == 0) {
            ++kw;
            sx = 0;
            ic_left = p.conv_ic / BK;
            set_tap();
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0, 0, 0, 0};
    auto at = [](int row, int c) { return row * BK + ((c ^ ((row >> 1) & 7)) << 2); };
    // Row exponents (xe_per_row): the accumulators are in units of the row that
    // the current tap reads; a tap whose row has another exponent rescales them
    // by a power of two (at most 2^60 either way, see split_rows_kernel). Rows
    // in the padding change nothing.
    constexpr int UNSET = -100000;
    int ecur[TN], xrow[TN], xpos[TN], etap = 0, eleft = 0;
    auto tap_exps = [&]() {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int iw = xpos[j] + etap * p.conv_d;
            const bool in = !p.conv_ic || (iw >= 0 && iw < p.conv_iw);
            const int e = in ? p.xe[p.conv_ic ? xrow[j] + iw : xrow[j]] : UNSET;
            if (e == UNSET || e == ecur[j]) continue;
            const float f = ecur[j] == UNSET ? 1.0f : exp2_int(ecur[j] - e);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] *= f;
            ecur[j] = e;
        }
    };
    if constexpr (!SNAKE) {
        if (p.xe_per_row) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = min(bn0 + (wn * TN + j) * 16 + lr, p.N - 1);
                const int b = p.conv_ic ? n / p.conv_ow : 0;
                ecur[j] = UNSET;
                xrow[j] = p.conv_ic ? b * p.conv_iw : n;
                xpos[j] = p.conv_ic ? (n - b * p.conv_ow) * p.conv_s - p.conv_p : 0;
            }
            etap = p.conv_ic ? kw : 0;
            eleft = p.conv_ic ? ic_left : nk;
            tap_exps();
        }
    }
    if (nk > 0) issue(0);
    for (int it = 0; it < nk; ++it) {
        if constexpr (!SNAKE) {
            if (p.xe_per_row && eleft-- == 0) {
                ++etap;
                eleft = p.conv_ic / BK - 1;
                tap_exps();
            }
        }
        // this wave's loads of the step have landed, then every wave's; the
        // barrier also ends every wave's reads of the other slot
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        if (it + 1 < nk) issue((it + 1) & 1);
        const float *st = smem + (it & 1) * STAGE;
        f16x8 ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            ah[i] = *(const f16x8 *) &st[at((wm * TM + i) * 16 + lr, lg)];
            al[i] = *(const f16x8 *) &st[at((wm * TM + i) * 16 + lr, 4 + lg)];
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            bh[j] = *(const f16x8 *) &st[at(BM + (wn * TN + j) * 16 + lr, lg)];
            bl[j] = *(const f16x8 *) &st[at(BM + (wn * TN + j) * 16 + lr, 4 + lg)];
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bh[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bl[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bh[j], acc[i][j], 0, 0, 0);
    }

    int mid_e = 0;
    if constexpr (UNIT) {
        __shared__ float red[4];
        const int ns = p.M / BK;
        // second weights, row m's step s: hi at chunk lg, lo at chunk 4 + lg (rows past M: the last one)
        f16x8 ah[2][TM], al[2][TM];
        const uint32_t *wr[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            wr[i] = p.w2 + (int64_t) min((wm * TM + i) * 16 + lr, p.M - 1) * p.M + 4 * lg;
            ah[0][i] = *(const f16x8 *) wr[i];
            al[0][i] = *(const f16x8 *) (wr[i] + 16);
        }
        // this lane's four channels of a token: bias, SnakeBeta
        float tm_ = 0.0f;
        const int xe = *p.xe - 30;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int mc = min((wm * TM + i) * 16 + 4 * lg, p.M - 4);
            const i32x4 we = *(const i32x4 *) (p.we + mc);
            const f32x4 mb = *(const f32x4 *) (p.mid_bias + mc), me = *(const f32x4 *) (p.mid_ea + mc),
                        mf = *(const f32x4 *) (p.mid_eb + mc);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                float v[4], ar[4], s2[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] = __builtin_ldexpf(acc[i][j][r], xe + we[r]) + mb[r];
                    ar[r] = v[r] * me[r];
                }
                sin2_x4(ar, s2);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[i][j][r] = v[r] + s2[r] * mf[r];
                    if (finite_f(acc[i][j][r])) tm_ = fmaxf(tm_, fabsf(acc[i][j][r]));
                }
            }
        }
        tm_ = wave_max(tm_);
        if (lane == 0) red[wave] = tm_;
        __syncthreads();                                      // also: the ring's last reads are done
        mid_e = bound_exp(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
        const float scale = exp2_int(15 - mid_e);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int mc = (wm * TM + i) * 16 + 4 * lg, c = (mc & 31) >> 3;
            float *st = smem + (mc >> 5) * (BN * BK) + ((mc & 7) >> 1);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int row = (wn * TN + j) * 16 + lr;
                const float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                f16x4 hi, lo;
                split4(v, scale, hi, lo);
                if (mc < p.M) {
                    *(f16x4 *) &st[at(row, c)] = hi;
                    *(f16x4 *) &st[at(row, 4 + c)] = lo;
                }
                acc[i][j] = f32x4{0, 0, 0, 0};
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < BM / BK; ++t) {
            if (t >= ns) break;
            if (t + 1 < ns) {
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    ah[(t + 1) & 1][i] = *(const f16x8 *) (wr[i] + 32 * (t + 1));
                    al[(t + 1) & 1][i] = *(const f16x8 *) (wr[i] + 32 * (t + 1) + 16);
                }
            }
            const float *st = smem + t * (BN * BK);
            f16x8 bh[TN], bl[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                bh[j] = *(const f16x8 *) &st[at((wn * TN + j) * 16 + lr, lg)];
                bl[j] = *(const f16x8 *) &st[at((wn * TN + j) * 16 + lr, 4 + lg)];
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[t & 1][i], bh[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[t & 1][i], bl[j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[t & 1][i], bh[j], acc[i][j], 0, 0, 0);
        }
    }

    // ---- epilogue: the accumulators as the workgroup's [BN][BM] tile in LDS,
    // then four consecutive outputs of one token per thread
    constexpr int G = BM / 4;
    static_assert(NT % G == 0, "fixed channel group per thread");
    const int ml = (tid % G) * 4, m0 = bm0 + ml;
    const bool mok = m0 < p.M;                                // M % 4 == 0: all four or none
    // the old rows of a residual update, eight at a time and the first ones
    // before the tile is staged: read one by one, each waits for memory
    constexpr int STEP = NT / G, ITER = BN / STEP, NB = 8;
    static_assert(ITER % NB == 0, "whole batches of rows");
    f32x4 old[NB];
    auto load_old = [&](int b) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int n = bn0 + tid / G + (b * NB + u) * STEP;
            old[u] = f32x4{0, 0, 0, 0};
            if (n < p.N && mok) old[u] = *(const f32x4 *) ((const float *) p.y + (int64_t) n * p.ld_y + m0);
        }
    };
    if constexpr (SNAKE)
        if (p.accumulate) load_old(0);
    __shared__ int row_e[SNAKE ? 1 : BN];
    if constexpr (!SNAKE) {
        if (p.xe_per_row && wm == 0 && lg == 0) {
#pragma unroll
            for (int j = 0; j < TN; ++j) row_e[(wn * TN + j) * 16 + lr] = ecur[j] == UNSET ? 0 : ecur[j];
        }
    }
    __syncthreads();                                          // the ring's last reads are done
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            *(f32x4 *) &smem[((wn * TN + j) * 16 + lr) * LDT + (wm * TM + i) * 16 + 4 * lg] = acc[i][j];
    __syncthreads();
    float bv[4] = {0, 0, 0, 0}, ea[4], eb[4];
    int we[4] = {0, 0, 0, 0};
    float oscale = 0.0f, ym = 0.0f, sm = 0.0f;
    if (mok) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (p.bias) bv[r] = p.bias[m0 + r];
            we[r] = (UNIT ? p.we2 : p.we)[m0 + r] - 30;
        }
        if constexpr (SNAKE) {
            const int c0 = m0 % p.period;                     // period % 4 == 0: c0 + 3 < period
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ea[r] = p.ea[c0 + r];
                eb[r] = p.eb[c0 + r];
            }
        }
    }
    if constexpr (SNAKE) {
        if (p.yp) {
            // |y| <= sum |w| max |x| + max |bias| (+ max |old y|), |snake(y)| <= |y| + max eb
            // (l1 and badd hold these maxima and 1 % for the roundings)
            float bound = *p.amax_x;
            if constexpr (UNIT) bound = p.mid_l1 * bound + p.mid_badd;
            bound = p.l1 * bound + p.badd;
            if (p.amax_old) bound += 1.01f * *p.amax_old;
            const int eo = bound_exp(bound);
            oscale = exp2_int(15 - eo);
            if (blockIdx.x == 0 && tid == 0) *p.e_out = eo;
        }
    }
    const int k_lo = kt0 * BK, k_hi = (kt0 + nk) * BK;
#pragma unroll 1
    for (int b = 0; b < ITER / NB; ++b) {
    if constexpr (SNAKE)
        if (p.accumulate && b) load_old(b);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const int nl = tid / G + (b * NB + u) * STEP, n = bn0 + nl;
        if (n >= p.N || !mok) continue;
        const f32x4 a4 = *(const f32x4 *) &smem[nl * LDT + ml];
        const int xe = UNIT ? mid_e : !SNAKE && p.xe_per_row ? row_e[SNAKE ? 0 : nl] : p.xe[0];
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float a = __builtin_ldexpf(a4[r], xe + we[r]);
            if (!SNAKE && !finite_f(a4[r])) a = f32_dot(p, m0 + r, n, k_lo, k_hi);
            o[r] = a + bv[r];
        }
        if constexpr (!SNAKE) {
            if (p.y_bf16) {
                uint16_t *yr = (uint16_t *) p.y + (int64_t) n * p.ld_y + m0;
#pragma unroll
                for (int r = 0; r < 4; ++r) yr[r] = f32_to_bf16_bits(o[r]);
            } else {
                *(f32x4 *) ((float *) p.y + (int64_t) z * p.part_stride + (int64_t) n * p.ld_y + m0) =
                    f32x4{o[0], o[1], o[2], o[3]};
            }
        } else {
            if (p.y) {
                float *yr = (float *) p.y + (int64_t) n * p.ld_y + m0;
                if (p.accumulate) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = old[u][r] + o[r];
                }
                *(f32x4 *) yr = f32x4{o[0], o[1], o[2], o[3]};
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (finite_f(o[r])) ym = fmaxf(ym, fabsf(o[r]));
            }
            float ar[4], s2[4], sv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) ar[r] = o[r] * ea[r];
            sin2_x4(ar, s2);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sv[r] = o[r] + s2[r] * eb[r];
                if (finite_f(sv[r])) sm = fmaxf(sm, fabsf(sv[r]));
            }
            if (p.yp) {
                f16x4 hi, lo;
                split4(sv, oscale, hi, lo);
                store_split4(p.yp + (int64_t) n * p.ld_y, m0, hi, lo);
            } else {
                *(f32x4 *) (p.y2 + (int64_t) n * p.ld_y + m0) = f32x4{sv[0], sv[1], sv[2], sv[3]};
            }
        }
    }
    }
    if constexpr (SNAKE) {
        ym = wave_max(ym);
        sm = wave_max(sm);
        if (lane == 0) {
            if (p.amax_y) raise_slot(p.amax_y, ym);
            if (p.amax_s) raise_slot(p.amax_s, sm);
        }
    }
}

template <int TM, int TN, int WPC>
void launch_split_tiles(SplitGemm &p, hipStream_t s) {
    p.tiles_m = (p.M + 32 * TM - 1) / (32 * TM);
    p.tiles_n = (p.N + 32 * TN - 1) / (32 * TN);
    p.per_xcd = (int) (((int64_t) p.tiles_m * p.tiles_n * p.splits + 7) / 8);
    const int grid = 8 * p.per_xcd;
    if (p.w2) launch_kernel((gemm_split_kernel<TM, TN, WPC, true, true>), dim3(grid), dim3(NT), 0, s, p);
    else if (p.ea) launch_kernel((gemm_split_kernel<TM, TN, WPC, true, false>), dim3(grid), dim3(NT), 0, s, p);
    else launch_kernel((gemm_split_kernel<TM, TN, WPC, false, false>), dim3(grid), dim3(NT), 0, s, p);
}

// one workgroup: max |x| over n values into slot[0] and its exponent into
// e[0]; slots 1 .. nslot - 1 cleared
__global__ __launch_bounds__(1024) void split_begin_kernel(const float *x, int64_t n, float *slot, int nslot, int *e) {
    __shared__ float red[16];
    float m = 0.0f;
    for (int64_t i = threadIdx.x; i < n; i += 1024) {
        const float a = fabsf(x[i]);
        if (finite_f(a)) m = fmaxf(m, a);
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    for (int i = threadIdx.x; i < nslot; i += 1024)
        if (i) slot[i] = 0.0f;
    if (threadIdx.x == 0) {
        for (int i = 1; i < 16; ++i) m = fmaxf(m, red[i]);
        slot[0] = m;
        e[0] = bound_exp(m);
    }
}

// x [C][T] -> split rows [T][C] at exponent e[0]; one thread per (4 channels, t)
__global__ __launch_bounds__(256) void split_transpose_kernel(const float *x, int C, int T, const int *e, uint32_t *y) {
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    const int t = (int) (i % T), c = (int) (i / T) * 4;
    if (c >= C) return;
    const float scale = exp2_int(15 - *e);
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = x[(int64_t) (c + r) * T + t];
    f16x4 hi, lo;
    split4(v, scale, hi, lo);
    store_split4(y + (int64_t) t * C, c, hi, lo);
}

// f32 rows -> split rows at their own exponents: the row's maximum, then its
// groups (8 lanes each). In place works: a wave has loaded all of a group
// before it writes it, and no other wave reads or writes the group.
template <int T>
__device__ __forceinline__ float row_max(const float *x, int cols, int t) {
    float m = 0.0f;
#pragma unroll 4
    for (int c = 4 * t; c < cols; c += 4 * T) {
        const f32x4 v = *(const f32x4 *) (x + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, finite_f(v[r]) ? fabsf(v[r]) : 0.0f);
    }
    return wave_max(m);
}
template <int T>
__device__ __forceinline__ void split_row(const float *x, int cols, int t, int e, uint32_t *y) {
    const float scale = exp2_int(15 - e);
#pragma unroll 4
    for (int c = 4 * t; c < cols; c += 4 * T) {
        const f32x4 v = *(const f32x4 *) (x + c);
        const float a[4] = {v[0], v[1], v[2], v[3]};
        f16x4 hi, lo;
        split4(a, scale, hi, lo);
        store_split4(y + (c & ~31), c & 31, hi, lo);
    }
}

// Up to four sets of rows in one launch (a product's weights and activations:
// two memory-bound passes of a few microseconds that overlap). A workgroup of
// eight waves takes rows_wg rows: a wave walks a row's maximum alone, then the
// whole workgroup splits the rows. One row where there are few (388 rows of
// 2816 values: 15 us with eight rows and four waves), since then the chip is
// idle and every step waits for memory; four from 2048 rows on, where the
// maxima of the rows beside them would be read once more for each row.
// Rows a convolution reads (halo = (KW - 1) * dilation > 0): one output sums
// rows of different exponents, so a row's exponent is raised to 60 below the
// largest among the rows up to `halo` away in its batch item; what that drops
// is 2^-100 of such a neighbour.
constexpr int ST = 512;
__global__ __launch_bounds__(ST) void split_rows_kernel(const SplitRowsGroup g) {
    __shared__ int es[SPLIT_RB + 2 * SPLIT_HALO];
    __shared__ float red[ST / 64];
    int k = 0;
    while (k + 1 < g.n && (int) blockIdx.x >= g.j[k + 1].begin) ++k;
    const SplitRows &p = g.j[k];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto row_at = [&](int64_t r) { return p.x + (p.rows_b ? (r / p.rows_b) * p.ld_b + (r % p.rows_b) * p.ld_x : r * p.ld_x); };
    const int64_t r0 = (int64_t) ((int) blockIdx.x - p.begin) * p.rows_wg;
    if (p.rows_wg == 1 && p.halo == 0) {
        // one row for all waves
        const float *x = row_at(r0);
        const float m = row_max<ST>(x, p.cols, threadIdx.x);
        if (lane == 0) red[wave] = m;
        __syncthreads();
        float t = red[0];
        for (int i = 1; i < ST / 64; ++i) t = fmaxf(t, red[i]);
        const int e = bound_exp(t);
        if (threadIdx.x == 0) p.e[r0] = e;
        split_row<ST>(x, p.cols, threadIdx.x, e, p.y + r0 * p.cols);
        return;
    }
    for (int i = wave; i < p.rows_wg + 2 * p.halo; i += ST / 64) {
        const int64_t r = r0 - p.halo + i;
        const bool in = r >= 0 && r < p.rows;
        const float m = in ? row_max<64>(row_at(r), p.cols, lane) : 0.0f;
        if (lane == 0) es[i] = bound_exp(m);
    }
    __syncthreads();
    for (int i = 0; i < p.rows_wg && r0 + i < p.rows; ++i) {
        const int64_t r = r0 + i;
        int e = es[p.halo + i];
        if (p.halo) {
            const int pos = (int) (p.rows_b ? r % p.rows_b : r), last = (int) (p.rows_b ? p.rows_b : p.rows) - 1;
            for (int d = 1; d <= p.halo; ++d) {
                if (pos - d >= 0) e = max(e, es[p.halo + i - d] - 60);
                if (pos + d <= last) e = max(e, es[p.halo + i + d] - 60);
            }
        }
        if (threadIdx.x == 0) p.e[r] = e;
        split_row<ST>(row_at(r), p.cols, threadIdx.x, e, p.y + r * p.cols);
    }
}

}  // namespace

hipError_t launch_split_rows(SplitRowsGroup &g, hipStream_t s) {
    if (g.n < 1 || g.n > 4) return hipErrorInvalidValue;
    int64_t blocks = 0;
    for (int k = 0; k < g.n; ++k) {
        SplitRows &p = g.j[k];
        if (p.cols % BK || p.ld_x % 4 || p.ld_b % 4 || ((uintptr_t) p.x & 15) || p.rows < 1 || p.rows > INT32_MAX ||
            p.halo < 0 || p.halo > SPLIT_HALO)
            return hipErrorInvalidValue;
        p.rows_wg = p.halo == 0 ? (p.cols >= 2048 ? 1 : SPLIT_RB) : p.rows < 2048 ? 1 : SPLIT_RB / 2;
        p.begin = (int) blocks;
        blocks += (p.rows + p.rows_wg - 1) / p.rows_wg;
        if (blocks > INT32_MAX) return hipErrorInvalidValue;
    }
    launch_kernel(split_rows_kernel, dim3((unsigned) blocks), dim3(ST), 0, s, g);
    return hipGetLastError();
}

bool split_gemm_fits(int64_t M, int64_t K, int64_t x_rows, int64_t ld_x, int items) {
    const int64_t lim = (int64_t) 1 << 31;
    return M % 4 == 0 && K % BK == 0 && M * K * 4 < lim && (x_rows * ld_x * 4 < lim || items == 1);
}

namespace {
// estimated microseconds of a launch on 128 x 128 tiles (wide; two workgroups
// per CU) or 128 x 64 (three): a K step of all of a CU's workgroups takes
// 1.2, 1.65 or 0.6, 0.9, 1.35 us with one, two or three of them (measured on
// 1292 rows of K = 1024 and 3072), and K slices cost the pass that sums them
double split_cost(int64_t M, int64_t N, int64_t K, int S, bool wide) {
    static const double step[2][4] = {{0, 0.6, 0.9, 1.35}, {0, 1.2, 1.65, 0}};
    const int per_cu = wide ? 2 : 3, cus = device_info().cus;
    const int64_t units = ((M + 127) / 128) * (wide ? (N + 127) / 128 : (N + 63) / 64) * S;
    const int64_t full = units / (per_cu * cus), rest = units % (per_cu * cus);
    const double round = full * step[wide][per_cu] + step[wide][(rest + cus - 1) / cus];
    return (double) ((K / BK + S - 1) / S) * round + (S > 1 ? 3.5 + 1.3e-6 * S * N * M : 0.0);
}
}  // namespace

int split_gemm_slices(int64_t M, int64_t N, int64_t K, int most) {
    int sp = 1;
    double best = 1e30;
    for (int c = 1; c <= most && (c == 1 || K / BK / c >= 8); ++c) {
        const double t = std::min(split_cost(M, N, K, c, false), split_cost(M, N, K, c, true));
        if (t < best) {
            best = t;
            sp = c;
        }
    }
    return sp;
}

hipError_t launch_gemm_split(SplitGemm &p, hipStream_t s) {
    if (p.M < 4 || p.M % 4 || p.N < 1 || p.K < BK || p.K % BK || p.splits < 1 || p.splits > p.K / BK || !p.x || !p.w ||
        !p.we || !p.xe || p.ld_y % 4 || (int64_t) p.M * p.ld_w * 4 >= ((int64_t) 1 << 31))
        return hipErrorInvalidValue;
    if (p.ea && (p.period < 4 || p.period % 4 || p.M % p.period || p.splits != 1 || p.y_bf16 || (!p.yp && !p.y2) ||
                 (p.yp && (p.ld_y % 32 || p.period % 32 || !p.amax_x || !p.e_out))))
        return hipErrorInvalidValue;
    if (p.w2 && (!p.ea || !p.y || p.M % 32 || p.M > 128 || !p.we2 || !p.mid_bias || !p.mid_ea || !p.mid_eb || p.xe_per_row))
        return hipErrorInvalidValue;
    if (!p.ea && (!p.y || !p.xf || !p.wf || (p.M > p.wf_rows && !p.wf2) || p.accumulate || (p.splits > 1 && (p.bias || p.y_bf16))))
        return hipErrorInvalidValue;
    if (p.conv_ic && (p.conv_ic % BK || p.K % p.conv_ic || p.conv_ow < 1 || p.conv_iw < 1 || p.conv_s < 1 ||
                      p.conv_d < 1 || p.conv_p < 0 || p.N % p.conv_ow))
        return hipErrorInvalidValue;
    p.x_rows = p.conv_ic ? (int64_t) (p.N / p.conv_ow) * p.conv_iw : p.N;
    p.m_inner = p.x_rows * p.ld_x > (int64_t) p.M * p.K;
    const int64_t tiles42 = (int64_t) ((p.M + 127) / 128) * ((p.N + 63) / 64) * p.splits;
    if (tiles42 > INT32_MAX / 16) return hipErrorInvalidValue;
    if (split_cost(p.M, p.N, p.K, p.splits, true) <= split_cost(p.M, p.N, p.K, p.splits, false)) launch_split_tiles<4, 4, 2>(p, s);
    else launch_split_tiles<4, 2, 3>(p, s);
    return hipGetLastError();
}

hipError_t launch_split_begin(const float *x, int64_t n, float *slot, int nslot, int *e, hipStream_t s) {
    launch_kernel(split_begin_kernel, dim3(1), dim3(1024), 0, s, x, n, slot, nslot, e);
    return hipGetLastError();
}

hipError_t launch_split_transpose(const float *x, int C, int T, const int *e, uint32_t *y, hipStream_t s) {
    if (C % 32) return hipErrorInvalidValue;
    const int64_t n = (int64_t) (C / 4) * T;
    launch_kernel(split_transpose_kernel, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, x, C, T, e, y);
    return hipGetLastError();
}

}  // namespace tsk
