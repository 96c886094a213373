// gemm_f32x6.hip — products of F32 operands on the bf16 matrix cores of gfx950
// (ggml_mul_mat / conv_cl with F32 weights, src/mmdit.cpp:13-34, and the VAE's
// convolutions, src/vae_decoder.cpp:26-58):
//
//   Y[n, m] = sum_k X[n, k] * W[m, k] + bias[m]
//
// Every operand value is held in three bf16 parts, v = hi + mid + lo: hi =
// bf16(v), mid = bf16(v - hi), lo = v - hi - mid, all exact (8 bits each with a
// sign), so the three hold all 24 bits of v, whatever the other values of its
// row are. (Parts below 2^-126 are flushed: a value below 2^-102 loses bits of
// at most 2^-126, fp32's smallest normal number.) Six of the nine products are
// summed: hi hi in one accumulator, hi mid, mid hi, hi lo, lo hi and mid mid in
// a second; mid lo, lo mid and lo lo are at most 2^-25 of |x w| together, less
// than one rounding of an fp32 sum. The first accumulator rounds once per 32
// products where the fp32 MFMA rounds once per 4, the second's roundings are
// 2^-8 of that, so the results are closer to 64-bit ones than fp32 MFMAs' on
// every input measured (K = 1024: 1.3e-7 against 5.7e-7, K = 3072: 2.3e-7
// against 9.9e-7; a column 2^40 above the rest against zero weights 1.3e-7).
// At 2.5 PFLOP/s / 6 against 157 TFLOP/s: 2 x 646 rows of a k3 convolution of
// 1024 -> 1024 channels 151 -> 65 us, 388 rows of 1024 -> 1024 47 -> 18 us, a
// 30 s VAE decode 35.5 -> 21.6 ms.
//
// The operands are read as f32 and split once per workgroup on the way into
// LDS. (Measured and not kept: a split by every wave from f32 in LDS, 90 us for
// the convolution above; the subtractions as v_dot2c_f32_bf16, which does not
// overlap with MFMAs, 96 us; MFMAs and conversions interleaved by hand, no gain.)
#include <algorithm>
#include <cstring>

#include "tsk_common.h"
#include "tsk_internal.h"
#include "tsk_runtime.h"

namespace tsk {

namespace {

constexpr int BK = 32;

__device__ __forceinline__ bool finite_f(float v) { return fabsf(v) <= 3.4028234664e38f; }

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;

struct Parts {
    bf16x8 p[3];
};
// (the empty asm keeps the pair one value: the compiler would convert the low one again instead of shifting it out)
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    uint32_t u = __builtin_bit_cast(uint32_t, bf16x2{(__bf16) a, (__bf16) b});
    asm("" : "+v"(u));
    return u;
}
// the parts of eight values
__device__ __forceinline__ Parts split8(const f32x4 a, const f32x4 b) {
    u32x4 h, m, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float v0 = e < 2 ? a[2 * e] : b[2 * e - 4], v1 = e < 2 ? a[2 * e + 1] : b[2 * e - 3];
        h[e] = pack2(v0, v1);
        const float r0 = v0 - __uint_as_float(h[e] << 16), r1 = v1 - __uint_as_float(h[e] & 0xffff0000u);
        m[e] = pack2(r0, r1);
        l[e] = pack2(r0 - __uint_as_float(m[e] << 16), r1 - __uint_as_float(m[e] & 0xffff0000u));
    }
    return Parts{{__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)}};
}

// In LDS a row's 32 values of a step are 192 bytes, [32 hi][32 mid][32 lo] of
// four 16-byte chunks each; chunk g of a part holds the values 4 g .. 4 g + 3 and
// 16 more (the group a thread stages from two 16-byte loads; the same order
// for both operands, so the sum's order alone depends on it). A row covers 48 of
// the 64 banks; chunk c of it is at c with bit 1 turned by row / 8: the 16 rows of
// a fragment read hit distinct banks in the groups that the reads are served
// in (turned by row / 4 they do not: 33 % of the LDS cycles were conflicts, the
// convolution above 72 -> 70 us without them)
__device__ __forceinline__ int chunk_at(int row, int c) { return c ^ ((row >> 2) & 2); }

struct X6 {
    GemmProblem p;
    F32Snake sk;
    F32Unit un;
    int64_t x_end, w_end;  // floats of x and of a weight that may be read
    int y_bf16;
    int tiles_m, tiles_n, m_inner, per_xcd, one_item;
};

// sin(a)^2 of four values, modulo pi / 2: x = a - n pi/2 with n = rint(2 a / pi)
// and pi/2 in three parts (Cody and Waite; the first fused product is exact),
// sin(x)^2 = z + z^2 q(z) on z = x^2 <= (pi/4)^2 with q a cubic (least squares
// weighted to a minimax fit, 2e-10), and 1 - sin(x)^2 for an odd n: 17
// instructions where sinf takes about 40. Against 64 bits, up to |a| = 2^19:
// max 1.0e-7, rms 1.9e-8 (sinf squared: 1.2e-7, 2.9e-8). Larger and non-finite
// arguments go through sinf.
__device__ __forceinline__ void sin2_x4(const float (&a)[4], float (&s2)[4]) {
    bool small = true;
#pragma unroll
    for (int r = 0; r < 4; ++r) small = small && fabsf(a[r]) < 524288.0f;
    if (small) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float n = __builtin_rintf(a[r] * 0.636619772f);
            const float x = fmaf(n, 1.7151245e-15f, fmaf(n, 4.37113883e-8f, fmaf(n, -1.57079637f, a[r])));
            const float z = x * x;
            const float q = fmaf(fmaf(fmaf(1.34098664e-4f, z, -3.17045464e-3f), z, 4.44434136e-2f), z, -3.33333254e-1f);
            const float s = fmaf(z * z, q, z);
            s2[r] = (int) n & 1 ? 1.0f - s : s;
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float sn = sinf(a[r]);
            s2[r] = sn * sn;
        }
    }
}

// fp32 product of one output whose parts' products are not finite (an infinity
// or NaN among its operands, or a value within 2^-9 of fp32's largest) or tiny
__device__ __forceinline__ float f32_dot(const GemmProblem &p, const float *w, int n, int k0, int k1) {
    float s = 0.0f;
    const float *x = (const float *) p.x;
    if (p.conv_ic) {
        const int b = n / p.conv_ow, o = n - b * p.conv_ow;
        for (int k = k0; k < k1; ++k) {
            const int kw = k / p.conv_ic, ic = k - kw * p.conv_ic;
            const int iw = o * p.conv_s + kw * p.conv_d - p.conv_p;
            if (iw >= 0 && iw < p.conv_iw) s = fmaf(x[(int64_t) b * p.x_group_stride + (int64_t) iw * p.ld_x + ic], w[k], s);
        }
    } else {
        const int64_t r = p.x_group_rows ? (int64_t) (n / p.x_group_rows) * p.x_group_stride + (int64_t) (n % p.x_group_rows) * p.ld_x
                                         : (int64_t) n * p.ld_x;
        for (int k = k0; k < k1; ++k) s = fmaf(x[r + k], w[k], s);
    }
    return s;
}

// UNIT: a residual unit of the VAE in one launch where its channels fit one
// tile (M <= 128, M % 32 == 0): the tile's convolution, bias and SnakeBeta stay
// in the workgroup (split into the ring's LDS, in the layout of M / 32
// activation steps) and are the operand of the k1 convolution (un.w2, its
// fragments from L2). Two launches read and write the activations twice more.
enum : int { PLAIN = 0, SNAKE = 1, UNIT = 2 };

// Workgroup = KG halves of K, each of 2 x WN waves of TM x TN 16x16 tiles with
// a ring of two 32-wide steps: while a step's MFMAs run, the threads split the
// next one into the other slot and load the one after it into registers.
// KG = 2 where tiles are few: eight waves per CU hide a step's latency, and the
// halves' sum in LDS costs no pass over memory (388 rows of 1024 -> 1024: 25 ->
// 20 us, the convolution above 94 -> 79, before the waves' order below).
template <int TM, int TN, int WN, int KG, int WPC, int EPI>
__global__ __launch_bounds__(128 * WN * KG, WPC) void gemm_f32x6_kernel(const X6 a) {
    constexpr int BM = 2 * TM * 16, BN = WN * TN * 16, NG = 128 * WN, NT = NG * KG;
    constexpr int ROWS = BM + BN, STAGE = ROWS * 48;          // floats
    constexpr int PR = NG / 4, PA = BM / PR, PB = BN / PR, NP = PA + PB;   // groups that a thread stages: weights, activations
    constexpr int LDT = BM + 4;
    constexpr int RING = 2 * STAGE, EPI_F = BN * LDT;
    static_assert(BM % PR == 0 && BN % PR == 0 && EPI_F <= KG * RING, "whole groups per thread; the output tile fits the ring");
    __shared__ __attribute__((aligned(16))) float smem[KG * RING];
    const GemmProblem &p = a.p;

    // workgroup -> tile. L % 8 is the XCD: each takes a consecutive eighth of
    // the tiles in (slice, larger operand, smaller operand) order, so that the
    // tiles it runs at one time share one K slice and a block of both operands
    // in its L2
    const int S = p.splits > 1 ? p.splits : 1;
    int tm, tn, z;
    {
        const int L = (int) blockIdx.x, T = a.tiles_m * a.tiles_n;
        const int u = (L & 7) * a.per_xcd + (L >> 3);
        if (u >= T * S) return;
        z = u / T;
        const int t = u - z * T;
        tm = a.m_inner ? t % a.tiles_m : t / a.tiles_n;
        tn = a.m_inner ? t / a.tiles_m : t % a.tiles_n;
    }
    // the weight this tile's outputs belong to: a second one's follow the first's
    const int half = p.wf3 ? a.tiles_m / 2 : a.tiles_m;
    const bool second = tm >= half;
    const float *w = second ? p.wf3 : p.wf;
    const int y0 = second ? p.M : 0;
    if (second) tm -= half;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) % (2 * WN);
    const int kg = __builtin_amdgcn_readfirstlane(tid >> 6) / (2 * WN);   // the waves' half of K
    const int lr = lane & 15, lg = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    const bool late = EPI != PLAIN || __builtin_amdgcn_readfirstlane(tid >> 6) >= NT / 128;   // (see the loop)
    const int bm0 = tm * BM, bn0 = tn * BN;

    // activation rows relative to a base of the tile, so that 32-bit byte
    // offsets reach every row of the tile whatever the tensor's size: its first
    // row (one item), else its first item
    const int grp = p.conv_ic ? p.conv_ow : p.x_group_rows ? p.x_group_rows : p.N;
    const int b0 = bn0 / grp;
    int64_t r0 = (int64_t) b0 * p.x_group_stride;
    if (a.one_item) {
        const int o = bn0 - b0 * grp;
        r0 += (int64_t) (p.conv_ic ? min(max(o * p.conv_s - p.conv_p, 0), p.conv_iw - 1) : o) * p.ld_x;
    }
    const int64_t x_left = (a.x_end - r0) * 4;
    const int x_range = (int) min(x_left, (int64_t) 0x7fffffff);
    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc((void *) w, (short) 0, (int) (a.w_end * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc((void *) ((const float *) p.x + r0), (short) 0, x_range, 0x00020000);
    constexpr uint32_t PAST = 0x80000000u;                   // beyond every range: reads zero
    // this thread's groups: values 4 gi .. 4 gi + 3 and 16 more of row t4 + PR q of either operand's tile
    const int gi = tid & 3, t4 = (tid % NG) >> 2;
    uint32_t woff[PA], voff[PB];                             // their byte offsets
    uint32_t xb[PB];                                         // convolution rows: their item's first row
    int xi[PB];                                              // and first position
#pragma unroll
    for (int q = 0; q < PA; ++q) {
        const int m = bm0 + t4 + PR * q;
        woff[q] = m < p.M ? (uint32_t) ((int64_t) m * p.ld_w * 4) + gi * 16 : PAST;
    }
    const int64_t rel = (int64_t) b0 * p.x_group_stride - r0;
#pragma unroll
    for (int q = 0; q < PB; ++q) {
        const int n = bn0 + t4 + PR * q, nn = min(n, p.N - 1), b = nn / grp, o = nn - b * grp;
        const int64_t first = rel + (int64_t) (b - b0) * p.x_group_stride;
        xb[q] = (uint32_t) (int32_t) (first * 4) + gi * 16;
        xi[q] = n < p.N ? o * p.conv_s - p.conv_p : INT32_MIN / 2;
        voff[q] = n < p.N ? (uint32_t) (int32_t) ((first + (int64_t) o * p.ld_x) * 4) + gi * 16 : PAST;
    }
    const int nk_all = p.K / BK, ks0 = (int) ((int64_t) z * nk_all / S);
    const int nks = (int) ((int64_t) (z + 1) * nk_all / S) - ks0;
    const int steps = (nks + KG - 1) / KG;                   // of the longer half
    const int kt0 = ks0 + kg * steps, nk = kg ? nks - steps : steps;
    // the tap and channel step of the next load
    int ic_left = 0, kw = 0;
    uint32_t sw = (uint32_t) kt0 * 128, sx = sw;
    auto set_tap = [&]() {
#pragma unroll
        for (int q = 0; q < PB; ++q) {
            const int iw = xi[q] + kw * p.conv_d;
            voff[q] = iw >= 0 && iw < p.conv_iw ? xb[q] + (uint32_t) ((int64_t) iw * p.ld_x * 4) : PAST;
        }
    };
    if (p.conv_ic) {
        const int per_tap = p.conv_ic / BK;
        kw = kt0 / per_tap;
        sx = (uint32_t) (kt0 - kw * per_tap) * 128;
        ic_left = per_tap - (kt0 - kw * per_tap);
        set_tap();
    }
    f32x4 raw[NP][2];                                        // the step under way
    auto load = [&](int q) {
        const uint32_t off = q < PA ? woff[q < PA ? q : 0] : voff[q < PA ? 0 : q - PA];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 v;
            if (q < PA) v = __builtin_amdgcn_raw_buffer_load_b128(wrs, off + 64 * h, sw, 0);
            else v = __builtin_amdgcn_raw_buffer_load_b128(xrs, off + 64 * h, sx, 0);
            raw[q][h] = __builtin_bit_cast(f32x4, v);
        }
    };
    int left = nk - 1;
    auto next_step = [&]() {                                  // (past the last step: that one again)
        if (left <= 0) return;
        --left;
        sw += 128;
        sx += 128;
        if (p.conv_ic && --ic_left == 0) {
            ++kw;
            sx = 0;
            ic_left = p.conv_ic / BK;
            set_tap();
        }
    };
    auto store = [&](int q, float *st) {
        const Parts v = split8(raw[q][0], raw[q][1]);
        const int row = t4 + PR * q;                          // (BM is a multiple of PR)
#pragma unroll
        for (int u = 0; u < 3; ++u) *(bf16x8 *) &st[row * 48 + chunk_at(row, 4 * u + gi) * 4] = v.p[u];
    };

    // acc: hi hi; cor: the five smaller products
    f32x4 acc[TM][TN], cor[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = cor[i][j] = f32x4{0, 0, 0, 0};
    };
    auto parts_at = [&](const float *st, int row) {
        Parts x;
#pragma unroll
        for (int u = 0; u < 3; ++u) x.p[u] = *(const bf16x8 *) &st[row * 48 + chunk_at(row, 4 * u + lg) * 4];
        return x;
    };
    auto mfmas = [&](int i, const Parts &x, const Parts (&y)[TN]) {
        constexpr int U[6] = {1, 0, 0, 2, 0, 1}, V[6] = {1, 0, 2, 0, 1, 0};
#pragma unroll
        for (int o = 0; o < 6; ++o)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 &c = o == 1 ? acc[i][j] : cor[i][j];
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.p[U[o]], y[j].p[V[o]], c, 0, 0, 0);
            }
    };
    clear();
    float *ring = smem + kg * RING;
    if (nk > 0) {
#pragma unroll
        for (int q = 0; q < NP; ++q) load(q);
        next_step();
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            store(q, ring);
            load(q);
        }
        next_step();
    }
    for (int it = 0; it < steps; ++it) {
        // this wave's writes of the step and its reads of the other slot are done, then every wave's
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (it >= nk) break;                                  // (the last step of the shorter half)
        const float *st = ring + (it & 1) * STAGE;
        float *nx = ring + (~it & 1) * STAGE;
        // of the two waves on a SIMD one splits first and one multiplies first,
        // so that each uses one pipe (in one order MFMAs and vector instructions
        // took turns: 78 -> 73 us for the convolution above, 76 -> 70 at 2 x 194
        // rows; the VAE's eight waves, at the chip's power limit, lose 4 %)
        auto multiply = [&]() {
            Parts y[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) y[j] = parts_at(st, BM + (wn * TN + j) * 16 + lr);
#pragma unroll
            for (int i = 0; i < TM; ++i) mfmas(i, parts_at(st, (wm * TM + i) * 16 + lr), y);
        };
        if (late) multiply();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            store(q, nx);                                     // (past the last step: values that nothing reads)
            load(q);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!late) multiply();
        next_step();
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += cor[i][j];

    if constexpr (EPI == UNIT) {
        const int ns = p.M / BK;
        __syncthreads();                                      // the ring's last reads are done
        // this lane's four channels of a token: bias, SnakeBeta, then the tile as M / 32 activation steps; then
        // the second product, its weights from L2 (rows past M: the last one)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int mi = (wm * TM + i) * 16 + 4 * lg, mc = min(mi, p.M - 4);
            const f32x4 mb = *(const f32x4 *) (a.un.bias + mc), me = *(const f32x4 *) (a.un.ea + mc),
                        mf = *(const f32x4 *) (a.un.eb + mc);
            const int c = (mi & 31) >> 2;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 v;
                float ar[4], s2[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] = acc[i][j][r] + mb[r];
                    ar[r] = v[r] * me[r];
                }
                sin2_x4(ar, s2);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] += s2[r] * mf[r];
                const Parts q = split8(v, v);                     // (the second half is the first again)
                const int row = (wn * TN + j) * 16 + lr;
                uint16_t *st = (uint16_t *) &smem[((mi >> 5) * BN + row) * 48];
                if (mi < p.M) {
#pragma unroll
                    for (int u = 0; u < 3; ++u)
                        __builtin_memcpy(st + chunk_at(row, 4 * u + (c & 3)) * 8 + (c >> 2) * 4, &q.p[u], 8);
                }
            }
        }
        clear();
        __syncthreads();
#pragma unroll
        for (int t = 0; t < BM / BK; ++t) {
            if (t >= ns) break;
            const float *st = smem + t * (BN * 48);
            Parts y[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) y[j] = parts_at(st, (wn * TN + j) * 16 + lr);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const float *wr = a.un.w2 + (int64_t) min((wm * TM + i) * 16 + lr, p.M - 1) * p.M + BK * t + 4 * lg;
                mfmas(i, split8(*(const f32x4 *) wr, *(const f32x4 *) (wr + 16)), y);
            }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += cor[i][j];
    }

    // ---- epilogue: the accumulators as the workgroup's [BN][BM] tile in LDS,
    // then four consecutive outputs of one token per thread
    constexpr int G = BM / 4;
    static_assert(NT % G == 0, "fixed channel group per thread");
    const int ml = (tid % G) * 4, m0 = bm0 + ml;
    const bool mok = m0 < p.M;                                // M % 4 == 0: all four or none
    // the old rows of a residual update, eight at a time and the first ones
    // before the tile is staged: read one by one, each waits for memory
    constexpr int STEP = NT / G, ITER = BN / STEP, NB = ITER < 8 ? ITER : 8;
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
    if constexpr (EPI != PLAIN)
        if (p.accumulate) load_old(0);
#pragma unroll
    for (int h = KG - 1; h >= 0; --h) {
        __syncthreads();                                      // the ring's last reads are done; the upper half of K is in place
        if (KG > 1 && kg != h) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 *t = (f32x4 *) &smem[((wn * TN + j) * 16 + lr) * LDT + (wm * TM + i) * 16 + 4 * lg];
                *t = h == KG - 1 ? acc[i][j] : acc[i][j] + *t;
            }
    }
    __syncthreads();
    float bv[4] = {0, 0, 0, 0}, ea[4], eb[4];
    if (mok) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (p.bias) bv[r] = p.bias[m0 + r];
        if constexpr (EPI != PLAIN) {
            const int c0 = m0 % a.sk.period;                  // period % 4 == 0: c0 + 3 < period
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ea[r] = a.sk.ea[c0 + r];
                eb[r] = a.sk.eb[c0 + r];
            }
        }
    }
#pragma unroll 1
    for (int b = 0; b < ITER / NB; ++b) {
        if constexpr (EPI != PLAIN)
            if (p.accumulate && b) load_old(b);
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int nl = tid / G + (b * NB + u) * STEP, n = bn0 + nl;
            if (n >= p.N || !mok) continue;
            const f32x4 a4 = *(const f32x4 *) &smem[nl * LDT + ml];
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v = a4[r];
                if constexpr (EPI == PLAIN) {
                    if (!finite_f(v) || (v != 0.0f && fabsf(v) < 8.2718061e-25f)) v = f32_dot(p, w + (int64_t) (m0 + r) * p.ld_w, n, ks0 * BK, (ks0 + nks) * BK);
                }
                o[r] = v + bv[r];
            }
            if constexpr (EPI == PLAIN) {
                const int64_t at_y = (int64_t) n * p.ld_y + y0 + m0;
                if (a.y_bf16) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) ((uint16_t *) p.y)[at_y + r] = f32_to_bf16_bits(o[r]);
                } else {
                    *(f32x4 *) ((float *) p.y + (int64_t) z * p.N * p.ld_y + at_y) = f32x4{o[0], o[1], o[2], o[3]};
                }
            } else {
                float *yr = (float *) p.y + (int64_t) n * p.ld_y + m0;
                if (p.accumulate) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = old[u][r] + o[r];
                }
                float ar[4], s2[4], sv[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) ar[r] = o[r] * ea[r];
                sin2_x4(ar, s2);
#pragma unroll
                for (int r = 0; r < 4; ++r) sv[r] = o[r] + s2[r] * eb[r];
                if (a.sk.y2) {
                    *(f32x4 *) yr = f32x4{o[0], o[1], o[2], o[3]};
                    *(f32x4 *) (a.sk.y2 + (int64_t) n * p.ld_y + m0) = f32x4{sv[0], sv[1], sv[2], sv[3]};
                } else {
                    *(f32x4 *) yr = f32x4{sv[0], sv[1], sv[2], sv[3]};
                }
            }
        }
    }
}

template <int TM, int TN, int WN, int KG, int WPC, int EPI>
void launch_tiles(X6 &a, hipStream_t s) {
    a.tiles_m = (a.p.M + 32 * TM - 1) / (32 * TM) * (a.p.wf3 ? 2 : 1);
    a.tiles_n = (a.p.N + 16 * WN * TN - 1) / (16 * WN * TN);
    const int S = a.p.splits > 1 ? a.p.splits : 1;
    a.per_xcd = (int) (((int64_t) a.tiles_m * a.tiles_n * S + 7) / 8);
    launch_kernel((gemm_f32x6_kernel<TM, TN, WN, KG, WPC, EPI>), dim3(8 * a.per_xcd), dim3(128 * WN * KG), 0, s, a);
}

// the operands' extents, or false where the kernel does not take them
bool extents(X6 &a) {
    GemmProblem &p = a.p;
    constexpr int64_t LIM = (int64_t) 1 << 29;               // floats: 31-bit byte offsets
    if (p.M % 4 || p.K % BK || p.ld_w % 4 || (((uintptr_t) p.x | (uintptr_t) p.wf | (uintptr_t) p.wf3) & 15)) return false;
    if (p.conv_ic && p.conv_ic % BK) return false;
    // rows of one item, their row stride and the items' (both say nothing for a single one)
    const int64_t grp = p.conv_ic ? p.conv_ow : p.x_group_rows ? p.x_group_rows : p.N;
    const int64_t items = (p.N + grp - 1) / grp, rows = p.conv_ic ? p.conv_iw : std::min<int64_t>(grp, p.N);
    if (rows == 1) p.ld_x = 0;
    if (items == 1) p.x_group_stride = 0;
    if (p.ld_x % 4 || p.ld_x < 0 || p.x_group_stride % 4 || p.x_group_stride < 0) return false;
    const int64_t row = p.conv_ic ? p.conv_ic : p.K;
    a.one_item = items == 1;
    a.w_end = (int64_t) (p.M - 1) * p.ld_w + p.K;
    a.x_end = (items - 1) * p.x_group_stride + (rows - 1) * p.ld_x + row;
    // what a tile of up to 128 rows reaches beyond its base
    const int64_t near = p.conv_ic ? (int64_t) 127 * p.conv_s + (int64_t) (p.K / p.conv_ic) * p.conv_d : 127;
    const int64_t span = a.one_item ? std::min(near, rows - 1) * p.ld_x
                                    : std::min<int64_t>(items - 1, 127 / grp + 1) * p.x_group_stride + (rows - 1) * p.ld_x;
    return a.w_end < LIM && span + row < LIM;
}

X6 problem(const GemmProblem &p, int y_bf16, const F32Snake *snake, const F32Unit *unit) {
    X6 a;
    memset(&a, 0, sizeof(a));
    a.p = p;
    a.y_bf16 = y_bf16;
    if (snake) a.sk = *snake;
    if (unit) a.un = *unit;
    return a;
}

}  // namespace

namespace {
// estimated microseconds of a launch on 128 x 64 tiles (wide) or 64 x 64, one
// workgroup per CU: 1.35 or 0.85 us per 64 k (measured on 388 rows of K = 1024,
// 100 of K = 4096, 1292 of K = 3072); K slices cost the pass that sums them
double tiles_cost(int64_t M, int64_t N, int64_t K, int S, bool wide) {
    const int64_t units = (M + (wide ? 127 : 63)) / (wide ? 128 : 64) * ((N + 63) / 64) * S, cus = device_info().cus;
    return (double) ((units + cus - 1) / cus * ((K / BK + 2 * S - 1) / (2 * S))) * (wide ? 1.35 : 0.85) +
           (S > 1 ? 3.5 + 1.3e-6 * S * N * M : 0.0);
}
}  // namespace

int gemm_f32x6_slices(int64_t M, int64_t N, int64_t K, int most) {
    int sp = 1;
    double best = 1e30;
    for (int c = 1; c <= most && (c == 1 || K / BK / c >= 8); ++c) {
        const double t = std::min(tiles_cost(M, N, K, c, false), tiles_cost(M, N, K, c, true));
        if (t < best) {
            best = t;
            sp = c;
        }
    }
    return sp;
}

bool gemm_f32x6_fits(const GemmProblem &p) {
    X6 a = problem(p, 0, nullptr, nullptr);
    return tuning().f32_split && extents(a);
}

hipError_t launch_gemm_f32x6(const GemmProblem &p0, int y_bf16, hipStream_t s, const F32Snake *snake, const F32Unit *unit) {
    X6 a = problem(p0, y_bf16, snake, unit);
    const GemmProblem &p = a.p;
    const int S = p.splits > 1 ? p.splits : 1;
    if (p.M < 4 || p.N < 1 || p.K < BK || !p.wf || !p.x || !p.y || !extents(a)) return hipErrorInvalidValue;
    if (S > p.K / BK || (S > 1 && (p.bias || snake || y_bf16)) || (p.accumulate && !snake)) return hipErrorInvalidValue;
    if (snake && (y_bf16 || p.wf3 || !snake->ea || !snake->eb || snake->period < 4 || snake->period % 4 || p.M % snake->period))
        return hipErrorInvalidValue;
    if (unit && (!snake || p.M % 32 || p.M > 128 || !unit->w2 || !unit->bias || !unit->ea || !unit->eb))
        return hipErrorInvalidValue;
    if (p.conv_ic && (p.K % p.conv_ic || p.x_group_rows || p.conv_ow < 1 || p.conv_iw < 1 || p.conv_s < 1 || p.conv_d < 1 ||
                      p.conv_p < 0 || p.N % p.conv_ow))
        return hipErrorInvalidValue;
    const int Mt = p.wf3 ? 2 : 1;
    if ((int64_t) ((p.M + 63) / 64) * Mt * ((p.N + 63) / 64) * S > INT32_MAX / 16) return hipErrorInvalidValue;
    a.m_inner = a.x_end > (int64_t) p.M * Mt * p.K;
    // the SnakeBeta forms (the VAE) on 128 x 128 tiles of whole K, the others on
    // 128 x 64 or 64 x 64 tiles of two K halves: both sum every output in the
    // same order, whatever N is
    const int tile = tuning().f32_tile;
    if (unit) launch_tiles<4, 2, 4, 1, 2, UNIT>(a, s);
    else if (snake) launch_tiles<4, 2, 4, 1, 2, SNAKE>(a, s);
    else if (tile ? tile != 22 : tiles_cost((int64_t) p.M * Mt, p.N, p.K, S, true) <= tiles_cost((int64_t) p.M * Mt, p.N, p.K, S, false))
        launch_tiles<4, 2, 2, 2, 2, PLAIN>(a, s);
    else launch_tiles<2, 2, 2, 2, 2, PLAIN>(a, s);
    return hipGetLastError();
}

}  // namespace tsk
