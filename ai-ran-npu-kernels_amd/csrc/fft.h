// fft.h -- Stockham FFT passes in LDS, shared by the OFDM demodulator and the
// synthetic channel's modulator.  No multiply-add contraction: instantiations
// in different kernels round identically, element for element.
#pragma once

#include <hip/hip_runtime.h>

namespace airan {

// W_4096^k = exp(-2 pi i k / 4096); smaller sizes index it with stride 4096/N.
// Filled once per device by InitOfdmTables.
extern __device__ float2 kTwiddle4096[4096];
int InitOfdmTables();

namespace fft {

constexpr int kMaxN = 4096;

__device__ inline float2 CMul(float2 a, float2 b)
{
#pragma clang fp contract(off)
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline float2 CAdd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ inline float2 CSub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ inline float2 MulMinusI(float2 a) { return make_float2(a.y, -a.x); }

// Forward 4-point DFT in place.
__device__ inline void Dft4(float2 &x0, float2 &x1, float2 &x2, float2 &x3)
{
    const float2 s0 = CAdd(x0, x2), d0 = CSub(x0, x2);
    const float2 s1 = CAdd(x1, x3), d1 = MulMinusI(CSub(x1, x3));
    x0 = CAdd(s0, s1);
    x2 = CSub(s0, s1);
    x1 = CAdd(d0, d1);
    x3 = CSub(d0, d1);
}

// exp(-2 pi i m / 16), m = 0..9.
__device__ inline float2 W16(int m)
{
    constexpr float c1 = 0.92387953251128674f, s1 = 0.38268343236508978f, h = 0.70710678118654752f;
    switch (m) {
    case 0: return make_float2(1.0f, 0.0f);
    case 1: return make_float2(c1, -s1);
    case 2: return make_float2(h, -h);
    case 3: return make_float2(s1, -c1);
    case 4: return make_float2(0.0f, -1.0f);
    case 6: return make_float2(-h, -h);
    default: return make_float2(-c1, s1);  // m = 9
    }
}

// Forward R-point DFT of v[0..R-1], natural order out.
template <int R>
__device__ inline void Dft(float2 *v)
{
    if constexpr (R == 2) {
        const float2 t = v[0];
        v[0] = CAdd(t, v[1]);
        v[1] = CSub(t, v[1]);
    } else if constexpr (R == 4) {
        Dft4(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        // r = b + 2a: DFT4 over a, twiddle W8^(b c), DFT2 over b -> k = c + 4 d.
        float2 u[2][4];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            u[b][0] = v[b];
            u[b][1] = v[b + 2];
            u[b][2] = v[b + 4];
            u[b][3] = v[b + 6];
            Dft4(u[b][0], u[b][1], u[b][2], u[b][3]);
        }
#pragma unroll
        for (int c = 1; c < 4; ++c) u[1][c] = CMul(u[1][c], W16(2 * c));
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            v[c] = CAdd(u[0][c], u[1][c]);
            v[c + 4] = CSub(u[0][c], u[1][c]);
        }
    } else {
        static_assert(R == 16, "radix");
        // r = b + 4a: DFT4 over a, twiddle W16^(b c), DFT4 over b -> k = c + 4 d.
        float2 u[4][4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            u[b][0] = v[b];
            u[b][1] = v[b + 4];
            u[b][2] = v[b + 8];
            u[b][3] = v[b + 12];
            Dft4(u[b][0], u[b][1], u[b][2], u[b][3]);
        }
#pragma unroll
        for (int b = 1; b < 4; ++b)
#pragma unroll
            for (int c = 1; c < 4; ++c) u[b][c] = CMul(u[b][c], W16(b * c));
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            Dft4(u[0][c], u[1][c], u[2][c], u[3][c]);
            v[c] = u[0][c];
            v[c + 4] = u[1][c];
            v[c + 8] = u[2][c];
            v[c + 12] = u[3][c];
        }
    }
}

__device__ inline uint32_t Pad(uint32_t i) { return i + (i >> 4); }

// One Stockham pass of radix R over N points held in LDS (natural-order
// in, natural-order out after the last pass).  Each thread of a symbol owns
// 16 / R butterflies.  The last pass applies the output scale before its
// LDS store, so the write-out is a pure fp32 -> fp16 conversion (no multiply
// the compiler could fold into a single-rounding v_fma_mix).
template <int LOGN, int R, bool LAST>
__device__ inline void LdsPass(float *lre, float *lim, uint32_t j, uint32_t ns, bool active, float scale)
{
    constexpr uint32_t N = 1u << LOGN;
    constexpr uint32_t TPS = N / 16;
    constexpr int B = 16 / R;
    float2 v[B][R], tw[B][R];
    if (active) {
        // Twiddle loads first: their latency overlaps the LDS reads and the
        // barrier instead of following them.
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const uint32_t k = (j + t * TPS) & (ns - 1);  // ns is a power of two
            const uint32_t step = (kMaxN / R) / ns;
#pragma unroll
            for (int r = 1; r < R; ++r) tw[t][r] = kTwiddle4096[k * r * step];
        }
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const uint32_t jj = j + t * TPS;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t i = Pad(jj + r * (N / R));
                v[t][r] = make_float2(lre[i], lim[i]);
            }
        }
    }
    __syncthreads();
    if (active) {
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const uint32_t jj = j + t * TPS;
            const uint32_t k = jj & (ns - 1);
#pragma unroll
            for (int r = 1; r < R; ++r) v[t][r] = CMul(v[t][r], tw[t][r]);
            Dft<R>(v[t]);
            const uint32_t base = (jj - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t i = Pad(base + r * ns);
                lre[i] = LAST ? v[t][r].x * scale : v[t][r].x;
                lim[i] = LAST ? v[t][r].y * scale : v[t][r].y;
            }
        }
    }
    __syncthreads();
}

}  // namespace fft
}  // namespace airan
