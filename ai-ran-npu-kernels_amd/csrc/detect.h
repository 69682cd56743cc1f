// detect.h -- exact per-RE LMMSE solve (L <= 4) shared by the detector
// operator and the fused detectors of the chain and the ragged batch.  Every
// multiply-add is an explicit fma, so every kernel that inlines these
// functions rounds identically.
#pragma once

#include <type_traits>

#include "common.h"

namespace airan {

// ------------------------------------------------------------ small solver
struct Cf {
    float r, i;
};
// Address of byte `off` of a uniform plane.  The plane's address is made opaque
// in scalar registers: the compiler would otherwise add the planes' distances
// to each lane's 64-bit address, in vector instructions.
template <typename T>
__device__ inline __attribute__((address_space(1))) T *PlaneAt(T *plane, uint32_t off)
{
    uint64_t p = reinterpret_cast<uint64_t>(plane);
    asm("" : "+s"(p));
    return reinterpret_cast<__attribute__((address_space(1))) T *>(
        reinterpret_cast<__attribute__((address_space(1))) char *>(p) + off);
}

// The fp16 there, widened.
__device__ inline float LoadAt(const __half *plane, uint32_t off)
{
    return static_cast<float>(*PlaneAt(reinterpret_cast<const _Float16 *>(plane), off));
}

// s + conj(a) b and s - a b: four fmas each.
__device__ inline Cf AddConjMul(Cf s, Cf a, Cf b)
{
    return {fmaf(a.i, b.i, fmaf(a.r, b.r, s.r)), fmaf(-a.i, b.r, fmaf(a.r, b.i, s.i))};
}
__device__ inline Cf SubMul(Cf s, Cf a, Cf b)
{
    return {fmaf(a.i, b.i, fmaf(-a.r, b.r, s.r)), fmaf(-a.i, b.r, fmaf(-a.r, b.i, s.i))};
}
__device__ inline Cf Conj(Cf a) { return {a.r, -a.i}; }
__device__ inline float Norm2(Cf a) { return fmaf(a.i, a.i, a.r * a.r); }

// 1 / d by one Newton step on the hardware's reciprocal and the division's own
// last instruction for zero, infinite and NaN d: four instructions against ten
// of the IEEE division, and equal to it for every significand at fourteen
// exponents from 2^-100 to 2^100 and both signs (pivots are sums of products
// of fp16 values, 2^-48 to 2^39).
__device__ inline float Recip(float d)
{
    const float r = __builtin_amdgcn_rcpf(d);
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, r, 1.0f), r, r), d, 1.0f);
}

// Solve A x = m and return diag(A^-1) for Hermitian PD A (lower triangle
// used, real diagonal), order NL known at compile time.  A = L D L^H without
// pivoting; W = L D below the diagonal.
template <int NL>
__device__ inline void HermSolve(const Cf (&A)[4][4], const Cf (&m)[4], Cf (&x)[4], float (&dinv)[4])
{
    Cf W[4][4], Lm[4][4];
    float Dinv[4];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        float dj = A[j][j].r;
#pragma unroll
        for (int k = 0; k < j; ++k)  // D_k |L_jk|^2 = Re(W_jk conj(L_jk))
            dj = fmaf(-W[j][k].i, Lm[j][k].i, fmaf(-W[j][k].r, Lm[j][k].r, dj));
        Dinv[j] = Recip(dj);
#pragma unroll
        for (int i = j + 1; i < NL; ++i) {
            Cf s = A[i][j];
#pragma unroll
            for (int k = 0; k < j; ++k) s = SubMul(s, W[i][k], Conj(Lm[j][k]));
            W[i][j] = s;
            Lm[i][j] = {s.r * Dinv[j], s.i * Dinv[j]};
        }
    }
    // forward: L z = m
    Cf z[4];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        Cf s = m[i];
#pragma unroll
        for (int k = 0; k < i; ++k) s = SubMul(s, Lm[i][k], z[k]);
        z[i] = s;
    }
    // diagonal: w = D^-1 z, backward L^H x = w
#pragma unroll
    for (int i = NL - 1; i >= 0; --i) {
        Cf s = {z[i].r * Dinv[i], z[i].i * Dinv[i]};
#pragma unroll
        for (int k = i + 1; k < NL; ++k) s = SubMul(s, Conj(Lm[k][i]), x[k]);
        x[i] = s;
    }
    // diag(A^-1)_c = sum_i |(L^-1)_ic|^2 / D_i, with L^-1 (unit diagonal) by
    // forward substitution.
#pragma unroll
    for (int c = 0; c < NL; ++c) {
        Cf col[4];
        float acc = Dinv[c];
#pragma unroll
        for (int i = c + 1; i < NL; ++i) {
            Cf s = {-Lm[i][c].r, -Lm[i][c].i};
#pragma unroll
            for (int k = c + 1; k < i; ++k) s = SubMul(s, Lm[i][k], col[k]);
            col[i] = s;
            acc = fmaf(Norm2(s), Dinv[i], acc);
        }
        dinv[c] = acc;
    }
}

// Unbiased LMMSE from the Gram matrix A = H^H H (lower triangle, real
// diagonal) and the matched filter m = H^H y: x = (A + no I)^-1 m scaled by
// 1 / d per layer, d = max(1 - no diag((A + no I)^-1), 1e-3), no_eff =
// (1 - d) / d.
template <int NL>
__device__ inline void DetectFromGram(float no, Cf (&A)[4][4], const Cf (&m)[4], Cf (&xh)[4], float (&ne)[4])
{
#pragma unroll
    for (int i = 0; i < NL; ++i) A[i][i].r += no;
    Cf x[4];
    float dinv[4];
    HermSolve<NL>(A, m, x, dinv);
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const float d = fmaxf(fmaf(-no, dinv[l], 1.0f), 1e-3f);
        const float inv = Recip(d);
        xh[l] = {x[l].r * inv, x[l].i * inv};
        ne[l] = (1.0f - d) * inv;
        // Rounded to fp32 before the callers round to fp16: the empty asm keeps
        // the compiler from fusing the two roundings in some of them.
        asm("" : "+v"(xh[l].r), "+v"(xh[l].i), "+v"(ne[l]));
    }
}

// One thread per RE.  H(r, l) and y(r) are fetched by the caller-specific
// loader, four receive antennas at a time with their loads in flight
// together; the solve is shared.
template <int NL, typename LoadH, typename LoadY>
__device__ inline void Detect(int nr, float no, LoadH loadh, LoadY loady, Cf (&xh)[4], float (&ne)[4])
{
    Cf A[4][4], m[4];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        m[i] = {0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j <= i; ++j) A[i][j] = {0.0f, 0.0f};
    }
    auto antennas = [&](int r0, auto count) {
        constexpr int N = decltype(count)::value;
        Cf h[N][NL], y[N];
#pragma unroll
        for (int r = 0; r < N; ++r) {
#pragma unroll
            for (int l = 0; l < NL; ++l) h[r][l] = loadh(r0 + r, l);
            y[r] = loady(r0 + r);
        }
#pragma unroll
        for (int r = 0; r < N; ++r) {
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                m[i] = AddConjMul(m[i], h[r][i], y[r]);
                A[i][i].r = fmaf(h[r][i].i, h[r][i].i, fmaf(h[r][i].r, h[r][i].r, A[i][i].r));
#pragma unroll
                for (int j = 0; j < i; ++j) A[i][j] = AddConjMul(A[i][j], h[r][i], h[r][j]);  // (H^H H)_ij
            }
        }
    };
    int r = 0;
    for (; r + 4 <= nr; r += 4) antennas(r, std::integral_constant<int, 4>{});
    for (; r < nr; ++r) antennas(r, std::integral_constant<int, 1>{});
    DetectFromGram<NL>(no, A, m, xh, ne);
}

// Single-tap zero forcing (equalization/equalize_zf_siso/equalize_kernel.cpp:
// Process; operator.yaml:72-84) on fp16 inputs in fp32: g = max(hr^2 + hi^2,
// floor), x = conj(h) y / g, no_eff = n0 / g, IEEE divisions.  Products of
// fp16 values are exact in fp32, so every sum rounds once whether or not it
// is contracted (the reference's MulAddDst gives the same value).
__device__ inline void ZfSolve(float hr, float hi, float yr, float yi, float n0, float *xr, float *xi, float *ne)
{
#pragma clang fp contract(off)
    const float g = fmaxf(hr * hr + hi * hi, AIRAN_ZF_G_FLOOR);
    *xr = (hr * yr + hi * yi) / g;
    *xi = (hr * yi - hi * yr) / g;
    *ne = n0 / g;
}

}  // namespace airan
