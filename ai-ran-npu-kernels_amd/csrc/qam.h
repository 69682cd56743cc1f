// qam.h -- QAM max-log soft demapping in the reference's integer units,
// shared by the per-operator demapper and the fused detector of the chain.
#pragma once

#include "common.h"

namespace airan {

// fp16 bit patterns of D*32 and D^2*32, D = constellation normalisation
// (qam256_demod.h:50-56 for 256QAM; the same definition for Qm = 2, 4, 6).
__host__ __device__ inline void QamConsts(uint32_t qm, uint16_t *dq, uint16_t *d2q)
{
    switch (qm) {
    case 2: *dq = 0x4da8; *d2q = 0x4c00; break;   // 22.627, 16.0
    case 4: *dq = 0x490f; *d2q = 0x4266; break;   // 10.117, 3.199
    case 6: *dq = 0x44f0; *d2q = 0x3a18; break;   // 4.9375, 0.7617
    default: *dq = 0x40e9; *d2q = 0x3206; break;  // 2.455, 0.1882
    }
}

// Quantisation of gen_data.py:20-27: every fp16 operation rounds once.
__device__ inline void QamUT(uint32_t qm, __half y, __half n, int *u, int *t)
{
    uint16_t dq, d2q;
    QamConsts(qm, &dq, &d2q);
    float nf = __half2float(n);
    if (!(nf >= 6.103515625e-05f) || !isfinite(nf)) nf = 6.103515625e-05f;
    const float dqf = __half2float(__ushort_as_half(dq));
    const float d2qf = __half2float(__ushort_as_half(d2q));
    const __half scale = __float2half_rn(dqf / nf);
    const __half thr = __float2half_rn(d2qf / nf);
    float prod = __half2float(__float2half_rn(__half2float(y) * __half2float(scale)));
    if (!isfinite(prod)) prod = prod > 0.0f ? 65504.0f : -65504.0f;
    int uu = static_cast<int>(rintf(prod));
    float tf = __half2float(thr);
    if (!isfinite(tf)) tf = 65504.0f;
    *t = static_cast<int>(rintf(tf));
    *u = uu > 1000 ? 1000 : (uu < -1000 ? -1000 : uu);
}

__host__ __device__ inline int Clip2560(int v) { return v > 2560 ? 2560 : (v < -2560 ? -2560 : v); }

// 256QAM closed form (gen_data.py:28-40), returned already negated (positive
// => bit 0).
__device__ inline void Axis256(int u, int t, int *out)
{
    const int a = u < 0 ? -u : u;
    int cl[8];
    int sa = 0;
#pragma unroll
    for (int i = 1; i <= 7; ++i) {
        const int kt = 2 * i * t;
        cl[i] = a < kt ? a : kt;
        sa += cl[i];
    }
    // cl[i] = min(a, 2i t) for k = 2i, and clamp(u, -2i t, 2i t) =
    // sign(u) min(|u|, 2i t) (t >= 0), so the sum of the clamps is +-sa.
    const int ss = u < 0 ? -sa : sa;
    const int v0 = 32 * u - 4 * ss;
    const int v1 = 80 * t - 16 * a - 4 * (cl[1] + cl[2] + cl[3]) + 4 * (cl[5] + cl[6] + cl[7]);
    const int v2 = -24 * t - 8 * a + 4 * cl[1] - 4 * cl[3] + 16 * cl[4] - 4 * cl[5] + 4 * cl[7];
    const int v3 = -8 * t - 4 * a + 8 * cl[2] - 8 * cl[4] + 8 * cl[6];
    out[0] = -Clip2560(v0);
    out[1] = -Clip2560(v1);
    out[2] = -Clip2560(v2);
    out[3] = -Clip2560(v3);
}

// PAM level under the reference mapper polarity (bit i of code = c_i, c_0 the
// sign bit): level = d0 e1, e_m = 1, e_i = 2^(m-i) - d_i e_{i+1}, d = 2c - 1.
__host__ __device__ inline int PamLevel(int m, int code)
{
    int e = 1;
    for (int i = m - 1; i >= 1; --i) e = (1 << (m - i)) - (2 * ((code >> i) & 1) - 1) * e;
    return (2 * (code & 1) - 1) * e;
}

// Max-log by exhaustion over the 2^m levels: LLR_i = min_{c_i=1} cost -
// min_{c_i=0} cost with cost = t s^2 - 2 u s; equal to the 256QAM closed form
// for every integer (u, t).
__host__ __device__ inline void AxisExhaustive(int m, int u, int t, int *out)
{
    int b0[4], b1[4];
    for (int i = 0; i < m; ++i) b0[i] = b1[i] = 0x7fffffff;
    for (int code = 0; code < (1 << m); ++code) {
        const int s = PamLevel(m, code);
        const int cost = t * s * s - 2 * u * s;
        for (int i = 0; i < m; ++i) {
            if ((code >> i) & 1)
                b1[i] = cost < b1[i] ? cost : b1[i];
            else
                b0[i] = cost < b0[i] ? cost : b0[i];
        }
    }
    for (int i = 0; i < m; ++i) out[i] = Clip2560(b1[i] - b0[i]);
}

// All 2m axis LLRs of one symbol: streams 0..m-1 from the I axis (NR bits
// b0, b2, ...), m..2m-1 from the Q axis (b1, b3, ...).
__device__ inline void QamSymbolLlrs(uint32_t qm, __half xr, __half xi, __half n, int *out)
{
    int ui, ti, uq, tq;
    QamUT(qm, xr, n, &ui, &ti);
    QamUT(qm, xi, n, &uq, &tq);
    const int m = static_cast<int>(qm / 2);
    if (qm == 8) {
        Axis256(ui, ti, out);
        Axis256(uq, tq, out + 4);
    } else {
        AxisExhaustive(m, ui, ti, out);
        AxisExhaustive(m, uq, tq, out + m);
    }
}

// ------------------------------------------------- packed (I, Q) demapper
typedef short s16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h16x2_t __attribute__((ext_vector_type(2)));

// The LLRs of one symbol in the units above divided by 4, the I axis in the
// low and the Q axis in the high half: w[k] holds streams k and Qm/2 + k.
// Closed forms of the max-log over the 2^(Qm/2) levels for every modulation
// (equal to AxisExhaustive for every integer u in +-1000 and t >= 0), with
// cl_i = min(|u|, 2 i t); every coefficient is a multiple of 4, so the clip
// to +-2560 is one to +-640 here.  From t = 1024 on each LLR is clipped or
// constant in t (2 i t >= |u|, and the t terms exceed the clip), so t is
// limited there and all sums fit 16 bits.
template <int QM>
__host__ __device__ inline void AxisPair(s16x2_t u, s16x2_t t, s16x2_t (&w)[QM / 2])
{
    constexpr int M = QM / 2;
    const s16x2_t a = __builtin_elementwise_max(u, -u), t2 = t + t;
    s16x2_t cl[8], kt = t2, sum = {0, 0};
#pragma unroll
    for (int i = 1; i < (1 << (M - 1)); ++i) {
        cl[i] = __builtin_elementwise_min(a, kt);
        sum += cl[i];
        kt += t2;
    }
    const s16x2_t neg = u >> 15;  // -1 where u < 0
    w[0] = ((sum ^ neg) - neg) - u * static_cast<short>(1 << (M - 1));
    if constexpr (M == 2) w[1] = a - t2;
    if constexpr (M == 3) {
        w[1] = (a + a + cl[1]) - (t2 * static_cast<short>(3) + cl[3]);
        w[2] = (t2 + a) - (cl[2] + cl[2]);
    }
    if constexpr (M == 4) {
        w[1] = (a * static_cast<short>(4) + (cl[1] + cl[2] + cl[3])) -
               (t2 * static_cast<short>(10) + (cl[5] + cl[6] + cl[7]));
        w[2] = (t2 * static_cast<short>(3) + (a + a) + cl[3] + cl[5]) - (cl[4] * static_cast<short>(4) + cl[1] + cl[7]);
        w[3] = (t2 + a) + (cl[4] - cl[2] - cl[6]) * static_cast<short>(2);
    }
    const s16x2_t hi = {640, 640}, lo = {-640, -640};
#pragma unroll
    for (int k = 0; k < M; ++k) w[k] = __builtin_elementwise_max(__builtin_elementwise_min(w[k], hi), lo);
}

// QamUT and AxisPair of one symbol (x = (I, Q) in fp16).  The fp16 quotients
// D / n by the hardware reciprocal: rounded to fp16 they equal the division's
// for every fp16 n and each of the eight constants: none lies as close to a
// boundary of fp16 rounding as 1 ulp of the reciprocal and the product's
// rounding reach, but for thresholds below 1/4, where t is 0 either way.
// The limits of u apply before its rounding (integers, so the same), the
// order of max and min giving a NaN u = -1000 as QamUT does.
template <int QM>
__device__ inline void QamSymbolPair(h16x2_t x, __half n, s16x2_t (&w)[QM / 2])
{
    uint16_t dq, d2q;
    QamConsts(QM, &dq, &d2q);
    float nf = __half2float(n);
    if (!(nf >= 6.103515625e-05f) || !isfinite(nf)) nf = 6.103515625e-05f;
    const float rn = __builtin_amdgcn_rcpf(nf);
    const _Float16 scale = static_cast<_Float16>(__half2float(__ushort_as_half(dq)) * rn);
    const float thr = static_cast<float>(static_cast<_Float16>(__half2float(__ushort_as_half(d2q)) * rn));
    const h16x2_t s2 = {scale, scale}, lim = {static_cast<_Float16>(1000.0f), static_cast<_Float16>(1000.0f)};
    const h16x2_t p = __builtin_elementwise_min(__builtin_elementwise_max(x * s2, -lim), lim);
    const s16x2_t u = __builtin_convertvector(__builtin_elementwise_rint(p), s16x2_t);
    const short t = static_cast<short>(rintf(fminf(thr, 1024.0f)));
    const s16x2_t tt = {t, t};
    AxisPair<QM>(u, tt, w);
}

}  // namespace airan
