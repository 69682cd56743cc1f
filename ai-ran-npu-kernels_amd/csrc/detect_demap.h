// detect_demap.h -- the tail of the fused detector shared by the batched
// chain and the ragged multi-grant batch: per layer, the equalised symbol
// and no_eff rounded to fp16, no_eff floored, the QAM max-log LLRs
// (qam256_demod arithmetic), then layer demap and Gold descrambling into the
// codeword LLRs, one NL-element store per bit plane.
#pragma once

#include "detect.h"
#include "qam.h"

namespace airan {

// xh / ne: the RE's LMMSE outputs; gw: the scrambling bits from this RE's
// first codeword bit on (bit l * QM + b for layer l, bit plane b); out: bit
// plane 0 (uniform; planes cw_stride apart), pos: the RE's first codeword
// position.  The LLRs (at most 2560 in magnitude) stay packed by axis, plane 2 k in the low
// and 2 k + 1 in the high half, and leave as one NL-element store per plane.
template <int NL, int QM>
__device__ inline void DemapStore(const Cf (&xh)[4], const float (&ne)[4], __half floor16, uint64_t gw, int16_t *out,
                                  uint32_t pos, uint32_t cw_stride)
{
    constexpr int M = QM / 2;
    // l QM + b < NL QM <= 32: the RE's bits are the low word's.
    const uint32_t g32 = static_cast<uint32_t>(gw);
    s16x2_t v[M][NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const h16x2_t x = {static_cast<_Float16>(xh[l].r), static_cast<_Float16>(xh[l].i)};
        __half ne16 = __float2half_rn(ne[l]);
        if (__half2float(ne16) < __half2float(floor16)) ne16 = floor16;
        s16x2_t w[M];
        QamSymbolPair<QM>(x, ne16, w);
#pragma unroll
        for (int k = 0; k < M; ++k) {
            // Times 4, or -4 where the scrambling bit is set.
            const uint32_t b = g32 >> (l * QM + 2 * k);
            const s16x2_t bit = __builtin_bit_cast(s16x2_t, (b & 1u) | (b & 2u) << 15);
            const s16x2_t four = {4, 4};
            v[k][l] = w[k] * (bit * static_cast<short>(-8) + four);
        }
    }
    auto half = [](s16x2_t x, int q) { return static_cast<uint32_t>(static_cast<uint16_t>(q ? x.y : x.x)); };
#pragma unroll
    for (int b = 0; b < QM; ++b) {
        int16_t *plane = out + static_cast<size_t>(b) * cw_stride;
        const s16x2_t *p = v[b / 2];
        const uint32_t at = 2u * pos;
        if constexpr (NL == 4) {
            typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
            *PlaneAt(reinterpret_cast<u32x2_t *>(plane), at) =
                u32x2_t{half(p[0], b & 1) | half(p[1], b & 1) << 16, half(p[2], b & 1) | half(p[3], b & 1) << 16};
        } else if constexpr (NL == 2) {
            *PlaneAt(reinterpret_cast<uint32_t *>(plane), at) = half(p[0], b & 1) | half(p[1], b & 1) << 16;
        } else {
#pragma unroll
            for (int l = 0; l < NL; ++l) *PlaneAt(plane, at + 2u * l) = static_cast<int16_t>(half(p[l], b & 1));
        }
    }
}

}  // namespace airan
