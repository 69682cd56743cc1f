// txgen_gpu.hip -- the synthetic transmitter and fading channel on the
// device (include/airan_pusch_tx.h, airan_pusch_txgpu_*): the bit-level
// stages of txgen.cpp for a batch of transport blocks, bit for bit, then a
// tapped-delay-line channel, OFDM modulation and AWGN straight to IQ.
//
//   TbCrcKernel    TB CRC attach.  A remainder is linear in the message
//       bits: the 64-bit chunk k of the message (counted from its end: bits
//       n - 64 (k + 1) .. n - 64 k - 1) contributes rho_k x^L x^(64 k) mod g
//       (a host table of x^(64 k)); a workgroup writes the XOR over its
//       chunks.
//   EncodeKernel   one workgroup per code block, from payload bits to grid
//       symbols: the info bits packed 32 to a word, the CB CRC from them, the
//       BG1 parities a word at a time, then rate matching from k0 skipping
//       filler, the bit interleaver, Gold scrambling, QAM mapping with the
//       reference mapper's polarity and the layer mapping onto the data REs.
//   DmrsGridKernel  the DMRS symbols of every layer: the slot's DMRS on the
//       layer's comb (FD-OCC sign on ports 1001/1003), zero on the other.
//   ChannelOfdmKernel  one workgroup per (slot, Rx, symbol): y = sum_l H x_l
//       with H = sum_taps g e^(-j 2 pi f tau) on the used subcarriers, a
//       4096-point (or smaller) radix-2 IFFT in LDS, the cyclic prefix and
//       AWGN from a counter-based generator, written as IQ.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "airan_ldpc_bg1.h"
#include "airan_pusch_tx.h"
#include "common.h"
#include "crc.h"
#include "gold.h"

using airan::DevGeom;
using airan::Geom;

namespace {

constexpr uint32_t kPolyA = 0x864CFBu;   // CRC24A
constexpr uint32_t kPolyB = 0x800063u;   // CRC24B
constexpr uint32_t kPoly16 = 0x1021u;    // CRC16
constexpr uint32_t kTbChunkBits = 64, kCbChunkBits = 160;
constexpr uint32_t kMaxZ = 384;
constexpr uint32_t kMaxFft = 4096;

struct TxPlan {
    uint32_t Z, C, K, kprime, per_cb, crc_cb, crc_tb, tbs, filler, ncb, q0, G, e_low, e_high, n_low;
    uint32_t s22;                 // shift of column 22 left after summing the four core rows
    uint32_t nsteps;              // core solve steps
    uint32_t step_row[4], step_col[4];
    uint32_t tb_poly, tb_len;     // TB CRC polynomial
};

// Host: x^e mod g (len-bit residues, poly without the x^len term).
uint32_t HostMulMod(uint32_t a, uint32_t b, uint32_t poly, uint32_t len)
{
    const uint32_t mask = (1u << len) - 1u;
    uint32_t r = 0;
    for (int i = static_cast<int>(len) - 1; i >= 0; --i) {
        const uint32_t top = (r >> (len - 1)) & 1u;
        r = (r << 1) & mask;
        if (top) r ^= poly;
        if ((b >> i) & 1u) r ^= a;
    }
    return r;
}

uint32_t HostXpow(uint64_t e, uint32_t poly, uint32_t len)
{
    uint32_t r = 1u, base = 2u;
    while (e != 0) {
        if (e & 1u) r = HostMulMod(r, base, poly, len);
        base = HostMulMod(base, base, poly, len);
        e >>= 1;
    }
    return r;
}

// Table x^(bits k) mod g for k < chunks.
std::vector<uint32_t> ChunkPowers(uint32_t chunks, uint32_t bits, uint32_t poly, uint32_t len)
{
    std::vector<uint32_t> t(chunks);
    uint32_t p = 1u;
    const uint32_t step = HostXpow(bits, poly, len);
    for (uint32_t k = 0; k < chunks; ++k) {
        t[k] = p;
        p = HostMulMod(p, step, poly, len);
    }
    return t;
}

// Gold bits c(0 .. 32 n - 1) of sequence cinit, 32 to a word.  The recurrences
// squared five times step whole words (x1(n + 31 * 32) = x1(n + 3 * 32) + x1(n)).
std::vector<uint32_t> GoldWords(uint32_t cinit, uint32_t n)
{
    std::vector<uint32_t> x1(n), x2(n);
    uint32_t s1 = 1u, s2 = cinit & 0x7fffffffu;
    for (uint32_t k = 0; k < 1600u / 32u; ++k) (void)airan::GoldNext32(&s1, &s2);
    for (uint32_t i = 0, none = 0; i < n && i < 31u; ++i) {
        x1[i] = airan::GoldNext32(&s1, &none);
        x2[i] = airan::GoldNext32(&none, &s2);
    }
    for (uint32_t i = 31; i < n; ++i) {
        x1[i] = x1[i - 28] ^ x1[i - 31];
        x2[i] = x2[i - 28] ^ x2[i - 29] ^ x2[i - 30] ^ x2[i - 31];
    }
    for (uint32_t i = 0; i < n; ++i) x1[i] ^= x2[i];
    return x1;
}

// Derives the core-parity schedule of the BG1 encoder (the same order
// txgen.cpp's encoder solves in).
bool CoreSchedule(uint32_t z, TxPlan *tp)
{
    std::vector<uint32_t> s22;
    for (int r = 0; r < 4; ++r)
        for (int e = AIRAN_BG1_ROW_START[r]; e < AIRAN_BG1_ROW_START[r + 1]; ++e)
            if (AIRAN_BG1_COL[e] == 22) {
                const uint32_t s = AIRAN_BG1_SHIFT[e] % z;
                bool found = false;
                for (size_t k = 0; k < s22.size(); ++k)
                    if (s22[k] == s) {
                        s22.erase(s22.begin() + static_cast<long>(k));
                        found = true;
                        break;
                    }
                if (!found) s22.push_back(s);
            }
    if (s22.size() != 1) return false;
    tp->s22 = s22[0];
    bool known[26] = {};
    for (int c = 0; c <= 22; ++c) known[c] = true;
    tp->nsteps = 0;
    for (int pass = 0; pass < 4; ++pass)
        for (int r = 0; r < 4; ++r) {
            int unknown = -1, count = 0;
            for (int e = AIRAN_BG1_ROW_START[r]; e < AIRAN_BG1_ROW_START[r + 1]; ++e) {
                const int c = AIRAN_BG1_COL[e];
                if (c >= 22 && c < 26 && !known[c]) {
                    unknown = e;
                    ++count;
                }
            }
            if (count != 1) continue;
            if (AIRAN_BG1_SHIFT[unknown] % z != 0 || tp->nsteps >= 4) return false;
            tp->step_row[tp->nsteps] = static_cast<uint32_t>(r);
            tp->step_col[tp->nsteps] = AIRAN_BG1_COL[unknown];
            ++tp->nsteps;
            known[AIRAN_BG1_COL[unknown]] = true;
        }
    return known[23] && known[24] && known[25];
}

// ------------------------------------------------------------------ CRC
// Residues in this file are left-aligned: an L-bit residue r is r << (32 - L),
// its polynomial likewise, so that a step needs no mask.
__device__ inline uint32_t CrcTimesX(uint32_t r, uint32_t poly)
{
    return (r << 1) ^ (poly & static_cast<uint32_t>(static_cast<int32_t>(r) >> 31));
}

// Table of i x^L mod g for the 256 values i of a byte: a message byte m then
// takes residue r (times x^L) to table[r's top byte ^ m] ^ r << 8.
__device__ inline uint32_t CrcByte(uint32_t i, uint32_t poly)
{
    uint32_t r = i << 24;
#pragma nounroll
    for (int k = 0; k < 8; ++k) r = CrcTimesX(r, poly);
    return r;
}

// Residue r extended by 32 message bits, bit 0 of v the highest power.
__device__ inline uint32_t CrcWord(uint32_t r, uint32_t v, const uint32_t *table)
{
    const uint32_t m = __brev(v);
#pragma unroll
    for (int k = 3; k >= 0; --k) r = table[(r >> 24) ^ ((m >> (8 * k)) & 0xffu)] ^ r << 8;
    return r;
}

// a * b mod g, a left-aligned, b the plain residue of at most 24 bits.  A
// short loop: a kernel's code is cold when it starts.
__device__ inline uint32_t CrcTimes(uint32_t a, uint32_t b, uint32_t poly)
{
    uint32_t r = 0;
    b <<= 8;
#pragma unroll 4
    for (int i = 0; i < 24; ++i, b <<= 1)
        r = CrcTimesX(r, poly) ^ (a & static_cast<uint32_t>(static_cast<int32_t>(b) >> 31));
    return r;
}

// Bit 0 of 16 consecutive bytes (any alignment), byte 0 in bit 0.
__device__ inline uint32_t Pack16(const uint8_t *m)
{
    uint32_t x[4];
    __builtin_memcpy(x, m, 16);
    uint32_t v = 0;
#pragma unroll
    for (int k = 3; k >= 0; --k) v = v << 4 | ((x[k] & 0x01010101u) * 0x01020408u) >> 24;
    return v;
}

__device__ inline uint32_t WaveXor(uint32_t v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v ^= __shfl_xor(v, o, 64);
    return v;
}

// TB CRC: part[tb][block] is the XOR over the workgroup's 64-bit chunks of
// (chunk x^L mod g) x^(64 k): a thread packs the 64 bytes of its chunk,
// reduces them by table lookups in LDS and multiplies once.  16 TBs of
// 1.07 Mbit (17 MB of bytes): 80 -> 6.8 us against one thread reading a chunk
// byte after byte with a shift register.
constexpr uint32_t kTbBlockChunks = 256;

__global__ void __launch_bounds__(256) TbCrcKernel(const uint8_t *__restrict__ payload, TxPlan p,
                                                   const uint32_t *__restrict__ pw, uint32_t chunks,
                                                   uint32_t *__restrict__ part)
{
    __shared__ uint32_t table[256], red[4];
    const uint32_t tb = blockIdx.y, k = blockIdx.x * kTbBlockChunks + threadIdx.x;
    const uint32_t up = 32u - p.tb_len, poly = p.tb_poly << up;
    const uint8_t *m = payload + static_cast<size_t>(tb) * p.tbs;
    const uint32_t pk = k < chunks ? pw[k] : 0u;
    const int64_t beg = static_cast<int64_t>(p.tbs) - kTbChunkBits * (static_cast<int64_t>(k) + 1);
    uint64_t v = 0;
    if (beg > -64) {
        // The first chunk starts before the message: its bits read from the
        // start and shifted (zeros before a message change no residue).
        if (p.tbs >= kTbChunkBits) {
            const uint8_t *c = m + (beg < 0 ? 0 : beg);
#pragma unroll
            for (int j = 3; j >= 0; --j) v = v << 16 | Pack16(c + 16 * j);
            if (beg < 0) v <<= -beg;
        } else {
            for (int64_t i = 0; i < beg + 64; ++i) v |= static_cast<uint64_t>(m[i] & 1u) << (i - beg);
        }
    }
    table[threadIdx.x] = CrcByte(threadIdx.x, poly);
    __syncthreads();
    uint32_t r = CrcWord(0, static_cast<uint32_t>(v), table);
    r = CrcWord(r, static_cast<uint32_t>(v >> 32), table);
    const uint32_t contrib = WaveXor(CrcTimes(r, pk, poly) >> up);
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = contrib;
    __syncthreads();
    if (threadIdx.x == 0) part[tb * gridDim.x + blockIdx.x] = red[0] ^ red[1] ^ red[2] ^ red[3];
}

// -------------------------------------------------------------- encode
// A column of the codeword is kept as its periodic extension: bit i of the
// row is bit i mod z of the column, kColWords words, so that the 32 bits from
// any shift on are one unaligned read.
constexpr uint32_t kColWords = kMaxZ / 32 + 2;
constexpr uint32_t kEncodeThreads = 256;
constexpr int kBg1Edges = 316;

// Bits q .. q + 31 (mod z) of the z bits at bit `base` of `w`.
__device__ inline uint32_t CyclicBits(const uint32_t *w, uint32_t base, uint32_t q, uint32_t z)
{
    uint32_t v = 0, n = 0;
    do {
        const uint32_t left = z - q, x = airan::BitsAt(w, base + q);
        v |= (left < 32u ? x & ((1u << left) - 1u) : x) << n;
        n += left;
        q = 0;
    } while (n < 32u);
    return v;
}

// 32 bits of an extended column from bit `s` + `q` on, both below z.
__device__ inline uint32_t RotWord(const uint32_t *col, uint32_t s, uint32_t q, uint32_t z)
{
    const uint32_t x = s + q;
    return airan::BitsAt(col, x >= z ? x - z : x);
}

// Axis level d0 (2^(m-1) - d1 (2^(m-2) - ... d_{m-1})), d_i = 2 c_i - 1, of
// bits 0, 2, 4, ..: m of them.
__device__ inline float AxisLevel(uint32_t bits, uint32_t m)
{
    float e = 1.0f;
#pragma nounroll
    for (uint32_t i = m - 1; i >= 1; --i)
        e = static_cast<float>(1u << (m - i)) - (2.0f * static_cast<float>((bits >> (2u * i)) & 1u) - 1.0f) * e;
    return (2.0f * static_cast<float>(bits & 1u) - 1.0f) * e;
}

struct EncodeArgs {
    DevGeom g;
    uint32_t tb_parts, slots_per_tb;
    uint32_t start[2][8];  // first stream position of each bit of a symbol, E = e_low, e_high
    float norm;
    const uint32_t *tb_part, *pow_cb, *gold;
};

// Workgroup: one code block, info bits to grid symbols (and the scrambled
// bits, if wanted).  Everything between the payload bytes and the symbols
// stays in LDS, 32 bits to a word: an edge of a parity row is one unaligned
// read of a rotated column per 32 checks, all the extension rows (which
// depend on the information and the core parities only) are one step without
// a barrier, and rows past the last transmitted bit are left out.  A symbol's
// Qm bits come from Qm places of the rate-matched stream, lanes take
// consecutive symbols (an LDS word serves 32 lanes, a layer's row is written
// in runs of 64 / L symbols) and look the point up.  Bound by vector
// instructions, three quarters of them in the symbol loop.  2048 blocks of
// 8448 bits (16 full-carrier 256QAM TBs): 34 us, against 271 + 108 + 48 us for
// bytes in LDS with a barrier per row, a coded-bit array and CRC and
// modulation passes of their own.
template <uint32_t QM>
__global__ void __launch_bounds__(kEncodeThreads) EncodeKernel(const uint8_t *__restrict__ payload, TxPlan p,
                                                               EncodeArgs a, float2 *__restrict__ grid,
                                                               uint8_t *__restrict__ coded_out)
{
    __shared__ uint32_t lin[68 * kMaxZ / 32 + 2];  // packed bits: the information, then the rate-matching stream
    __shared__ uint32_t col[68][kColWords];
    __shared__ uint32_t lam[4][kColWords];
    __shared__ uint32_t edge[kBg1Edges];  // column | shift mod z << 8, in row order
    __shared__ uint32_t row_start[AIRAN_BG1_ROWS + 1];
    __shared__ uint32_t table[256];  // CRC24B of a byte
    __shared__ float2 point[1u << QM];
    __shared__ uint32_t data_sym[airan::kSymbols];
    const uint32_t cb = blockIdx.x, tb = cb / p.C, r = cb % p.C;
    const uint32_t z = p.Z, t = threadIdx.x, lane = t & 63u;
    const uint32_t high = r < p.n_low ? 0u : 1u;
    const uint32_t E = high ? p.e_high : p.e_low, eq = E / QM;
    const uint32_t nf = p.ncb - p.filler, fstart = p.kprime - 2u * z;
    if (E == 0) return;
    static_assert(sizeof(AIRAN_BG1_COL) / sizeof(AIRAN_BG1_COL[0]) == kBg1Edges, "edges");
    static_assert((1u << QM) <= kEncodeThreads && AIRAN_BG1_ROWS < kEncodeThreads, "one thread each");
    static_assert(64 * kCbChunkBits >= 22 * kMaxZ, "one wave reduces a code block");

    // Information bits, 32 to a word: payload || TB CRC, zeros after.
    const uint32_t first = r * p.per_cb;
    uint32_t tb_crc = 0;
    if (p.crc_tb != 0 && first + p.per_cb > p.tbs) {
        for (uint32_t k = lane; k < a.tb_parts; k += 64u) tb_crc ^= a.tb_part[tb * a.tb_parts + k];
        tb_crc = WaveXor(tb_crc);
    }
    // n payload bits from `first` on belong to the block; the last word is
    // read from 32 bytes before their end and shifted (no loop of single
    // loads: each costs a memory latency).
    const uint8_t *m = payload + static_cast<size_t>(tb) * p.tbs;
    const uint32_t n = first >= p.tbs ? 0u : min(p.per_cb, p.tbs - first);
#pragma unroll 2
    for (uint32_t w = t; w < 22 * kMaxZ / 32 + 2; w += kEncodeThreads) {
        const uint32_t k = 32u * w;
        uint32_t v = 0;
        if (k < n) {
            const uint32_t end = min(first + k + 32u, first + n), back = first + k + 32u - end;
            if (end >= 32u)
                v = (Pack16(m + end - 16u) << 16 | Pack16(m + end - 32u)) >> back;
            else
                for (uint32_t i = first + k; i < end; ++i) v |= (m[i] & 1u) << (i - first - k);
        }
        if (k + 32u > n && k < p.per_cb && p.crc_tb != 0) {
            // TB CRC bits, the first the highest power, from bit tbs on.
            const uint32_t crc = __brev(tb_crc << (32u - p.crc_tb));
            const int64_t d = static_cast<int64_t>(p.tbs) - first - k;
            if (d >= 0 && d < 32) v |= crc << d;
            if (d < 0 && d > -32) v |= crc >> -d;
            if (k + 32u > p.per_cb) v &= (1u << (p.per_cb - k)) - 1u;
        }
        lin[w] = v;
    }
#pragma nounroll
    for (uint32_t e = t; e < static_cast<uint32_t>(kBg1Edges); e += kEncodeThreads)
        edge[e] = AIRAN_BG1_COL[e] | (AIRAN_BG1_SHIFT[e] % z) << 8;
    if (t <= AIRAN_BG1_ROWS) row_start[t] = AIRAN_BG1_ROW_START[t];
    if (t < (1u << QM)) point[t] = make_float2(AxisLevel(t, QM / 2) * a.norm, AxisLevel(t >> 1, QM / 2) * a.norm);
    if (t == 0)  // not by lane: a lane-dependent index reads the argument segment
#pragma unroll
        for (uint32_t k = 0; k < airan::kSymbols; ++k) data_sym[k] = a.g.data_sym[k];
    table[t] = CrcByte(t, kPolyB << 8);
    static_assert(kEncodeThreads == 256, "one table entry each");
    __syncthreads();
    if (p.crc_cb != 0) {
        // CRC24B: lane l of the first wave reduces the 160 bits from bit
        // n - 160 (l + 1) on.
        if (t < 64u) {
            uint32_t res = 0;
#pragma nounroll
            for (uint32_t j = 0; j < kCbChunkBits; j += 32u) {
                const int32_t b = static_cast<int32_t>(p.per_cb + j) - static_cast<int32_t>(kCbChunkBits * (t + 1u));
                uint32_t v = 0;
                if (b > -32)
                    v = b < 0 ? lin[0] << static_cast<uint32_t>(-b) : airan::BitsAt(lin, static_cast<uint32_t>(b));
                res = CrcWord(res, v, table);
            }
            const uint32_t pk = kCbChunkBits * t < p.per_cb ? a.pow_cb[t] : 0u;
            const uint32_t crc = WaveXor(CrcTimes(res, pk, kPolyB << 8));
            if (t == 0) {
                // The first bit is the highest power.
                const uint64_t v = static_cast<uint64_t>(__brev(crc)) << (p.per_cb & 31u);
                lin[p.per_cb >> 5] |= static_cast<uint32_t>(v);
                lin[(p.per_cb >> 5) + 1] |= static_cast<uint32_t>(v >> 32);
            }
        }
        __syncthreads();
    }

    const uint32_t words = (z + 31u) / 32u, ext = words + 2u;  // of a column, of its extension
    auto word_start = [&](uint32_t w) { return 32u * w % z; };
#pragma nounroll
    for (uint32_t k = t; k < 22u * ext; k += kEncodeThreads) {
        const uint32_t c = k / ext, w = k - c * ext;
        col[c][w] = CyclicBits(lin, c * z, word_start(w), z);
    }
    __syncthreads();
    // XOR over the edges of row `row` with columns below `limit`, from bit q
    // of the check on.
    auto row_xor = [&](uint32_t row, uint32_t q, uint32_t limit) {
        uint32_t v = 0;
        const uint32_t end = row_start[row + 1];
#pragma unroll 2
        for (uint32_t e = row_start[row]; e < end; ++e) {
            const uint32_t x = edge[e], c = x & 0xffu;
            if (c < limit) v ^= RotWord(col[c], x >> 8, q, z);
        }
        return v;
    };
    // Core parities: lambda sums, column 22 through its unmatched shift, then
    // the rows with one unknown.
    if (t < 4u * ext) {
        const uint32_t row = t / ext, w = t - row * ext;
        lam[row][w] = row_xor(row, word_start(w), 22u);
    }
    __syncthreads();
    const uint32_t q_t = word_start(t);
    if (t < ext) {
        const uint32_t back = p.s22 == 0 ? 0u : z - p.s22;
        uint32_t v = 0;
        for (uint32_t row = 0; row < 4u; ++row) v ^= RotWord(lam[row], back, q_t, z);
        col[22][t] = v;
    }
    __syncthreads();
#pragma nounroll
    for (uint32_t s = 0; s < p.nsteps; ++s) {
        const uint32_t row = p.step_row[s], u = p.step_col[s];
        if (t < ext) {
            // A core row ends with its two or three parity edges.
            uint32_t v = lam[row][t];
#pragma nounroll
            for (uint32_t e = row_start[row + 1] - 3u; e < row_start[row + 1]; ++e) {
                const uint32_t x = edge[e], c = x & 0xffu;
                if (c >= 22u && c != u) v ^= RotWord(col[c], x >> 8, q_t, z);
            }
            col[u][t] = v;
        }
        __syncthreads();
    }
    // Columns that hold a transmitted bit: all once the stream wraps.
    const uint64_t last_q = static_cast<uint64_t>(p.q0) + E;
    const uint32_t last = last_q >= nf ? nf - 1u : static_cast<uint32_t>(last_q) - 1u;
    const uint32_t cols = min(68u, (2u * z + (last < fstart ? last : last + p.filler)) / z + 1u);
    const uint32_t nrows = cols > 26u ? cols - 26u : 0u;
#pragma nounroll
    for (uint32_t k = t; k < nrows * words; k += kEncodeThreads) {
        const uint32_t row = k / words, w = k - row * words, own = 26u + row;
        col[own][w] = row_xor(row + 4u, word_start(w), own);
    }
    __syncthreads();
    // The stream: bit q is codeword bit 2 z + q, past the filler from fstart on.
#pragma nounroll
    for (uint32_t i = t; 32u * i <= last; i += kEncodeThreads) {
        uint32_t q = 32u * i, v = 0, got = 0;
        do {
            const uint32_t b = 2u * z + (q < fstart ? q : q + p.filler), c = b / z, x = b - c * z;
            const uint32_t left = min(z - x, q < fstart ? fstart - q : 32u);
            const uint32_t y = airan::BitsAt(col[c], x);
            v |= (left < 32u ? y & ((1u << left) - 1u) : y) << got;
            got += left;
            q += left;
        } while (got < 32u && q <= last);
        lin[i] = v;
    }
    __syncthreads();

    // Symbol j of the block: bit i is bit i eq + j of the stream, modulo nf.
    const DevGeom &g = a.g;
    const uint32_t sym0 = (high ? p.n_low * p.e_low + (r - p.n_low) * p.e_high : r * p.e_low) / QM;
    const uint32_t slot0 = sym0 / g.cw_symbols, i0 = sym0 - slot0 * g.cw_symbols;
    const size_t slot_plane = static_cast<size_t>(g.nl) * airan::kSymbols * g.used;
#pragma nounroll
    for (uint32_t j = t; j < eq; j += kEncodeThreads) {
        const size_t bit0 = static_cast<size_t>(sym0 + j) * QM;
        const uint32_t jq = eq > nf ? j % nf : j;
        uint32_t bits = 0;
#pragma unroll
        for (uint32_t i = 0; i < QM; ++i) {
            uint32_t q = a.start[high][i] + jq;
            q = min(q, q - nf);  // q < 2 nf; q - nf wraps below nf
            bits |= ((lin[q >> 5] >> (q & 31u)) & 1u) << i;
        }
        const uint64_t w = static_cast<uint64_t>(a.gold[(bit0 >> 5) + 1]) << 32 | a.gold[bit0 >> 5];
        bits ^= static_cast<uint32_t>(w >> (bit0 & 31u)) & ((1u << QM) - 1u);
        if (coded_out != nullptr) {
            uint8_t *dst = coded_out + static_cast<size_t>(tb) * p.G + bit0;
#pragma unroll
            for (uint32_t i = 0; i < QM; ++i) dst[i] = static_cast<uint8_t>((bits >> i) & 1u);
        }
        uint32_t slot = slot0, i = i0 + j;
        while (i >= g.cw_symbols) {
            i -= g.cw_symbols;
            ++slot;
        }
        const uint32_t re = g.nl == 3u ? i / 3u : i >> (g.nl >> 1);  // 1, 2, 4 layers: a shift by 0, 1, 2
        const uint32_t l = i - re * g.nl, ds = re / g.used, sc = re - ds * g.used;
        const size_t o = (static_cast<size_t>(tb) * a.slots_per_tb + slot) * slot_plane +
                         (static_cast<size_t>(l) * airan::kSymbols + data_sym[ds]) * g.used + sc;
        grid[o] = point[bits];
    }
}

struct DmrsArgs {
    DevGeom g;
    uint32_t slots, rb_start, n_id, n_scid, default_slot;
    uint32_t wf_odd[4];
};

// Workgroup (slot, layer, DMRS symbol): its pilots' Gold bits in LDS, then
// the row in order, pilots on the layer's comb and zeros on the other.
__global__ void __launch_bounds__(256) DmrsGridKernel(DmrsArgs a, const uint16_t *__restrict__ slot_numbers,
                                                      float2 *__restrict__ grid)
{
    __shared__ uint32_t x1[airan::kGoldSpanWords + 2], x2[airan::kGoldSpanWords + 2];
    const DevGeom &g = a.g;
    const uint32_t d = blockIdx.x % g.ndmrs, rest = blockIdx.x / g.ndmrs;
    const uint32_t l = rest % g.nl, s = rest / g.nl;
    const uint64_t slot_number = slot_numbers != nullptr ? slot_numbers[s] : a.default_slot;
    const uint64_t term = (1ull << 17) * (14ull * slot_number + g.dmrs_sym[d] + 1ull) * (2ull * a.n_id + 1ull);
    const uint32_t cdmrs = static_cast<uint32_t>((term + 2ull * a.n_id + a.n_scid) & 0x7fffffffull);
    const uint32_t off = airan::GoldSpan(x1, x2, cdmrs, 12ull * a.rb_start, 2u * g.n_dmrs_re);
    const float h = 0.70710678118654752f;
    float2 *row = grid + (static_cast<size_t>(s) * g.nl + l) * airan::kSymbols * g.used +
                  static_cast<size_t>(g.dmrs_sym[d]) * g.used;
    for (uint32_t sc = threadIdx.x; sc < g.used && sc < 2u * g.n_dmrs_re; sc += blockDim.x) {
        const uint32_t mm = sc >> 1;
        float2 v = make_float2(0.0f, 0.0f);
        if ((sc & 1u) == g.comb[l]) {
            const uint32_t b = airan::BitsAt(x1, off + 2u * mm);
            const float f = a.wf_odd[l] && (mm & 1u) ? -h : h;
            v = make_float2((b & 1u) ? -f : f, (b & 2u) ? -f : f);
        }
        row[sc] = v;
    }
}

// ------------------------------------------------- channel + OFDM + noise
struct ChanArgs {
    uint32_t nr, nl, used, fft, log2n, taps, samples, iq_float;
    uint32_t cp[14], start[14];
    float scs, sigma, inv_sqrt_n;
    uint64_t seed;
};

__device__ inline uint64_t Mix64(uint64_t z)
{
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

// Two independent N(0, 1) values (Box-Muller) from a counter.
__device__ inline float2 Gauss2(uint64_t key)
{
    const uint64_t r = Mix64(key);
    const float u1 = (static_cast<float>(r >> 40) + 0.5f) * (1.0f / 16777216.0f);
    const float u2 = static_cast<float>((r >> 16) & 0xffffffull) * (1.0f / 16777216.0f);
    const float rad = sqrtf(-2.0f * logf(u1));
    float sn, cs;
    sincospif(2.0f * u2, &sn, &cs);
    return make_float2(rad * cs, rad * sn);
}

// Workgroup (slot, rx, symbol).  grid: complex64 [slots][L][14][used];
// gains complex64 [slots][NR][L][taps][14]; delays [slots][taps].
__global__ void __launch_bounds__(256) ChannelOfdmKernel(const float2 *__restrict__ grid,
                                                         const float2 *__restrict__ gains,
                                                         const float *__restrict__ delays,
                                                         const float2 *__restrict__ twiddle, ChanArgs a,
                                                         void *__restrict__ iq)
{
    __shared__ float2 buf[kMaxFft];
    __shared__ float2 gs[4][32];  // this symbol's tap gains per layer
    __shared__ double tau[32];
    const uint32_t sym = blockIdx.x % 14u, rest = blockIdx.x / 14u;
    const uint32_t rx = rest % a.nr, slot = rest / a.nr;
    const uint32_t t = threadIdx.x, n = a.fft;
    for (uint32_t k = t; k < a.nl * a.taps; k += blockDim.x) {
        const uint32_t l = k / a.taps, tp = k % a.taps;
        gs[l][tp] = gains[((((static_cast<size_t>(slot) * a.nr + rx) * a.nl + l) * a.taps + tp) * 14u) + sym];
    }
    for (uint32_t k = t; k < a.taps; k += blockDim.x) tau[k] = delays[static_cast<size_t>(slot) * a.taps + k];
    __syncthreads();
    const uint32_t half = a.used / 2u;
    const size_t gplane = static_cast<size_t>(14) * a.used;
    const float2 *gx = grid + static_cast<size_t>(slot) * a.nl * gplane + static_cast<size_t>(sym) * a.used;
    for (uint32_t k = t; k < n; k += blockDim.x) {
        // Bin k carries subcarrier u = (k + used/2) mod N when u < used.
        const uint32_t u = (k + half) & (n - 1u);
        float2 y = make_float2(0.0f, 0.0f);
        if (u < a.used) {
            const double f = (static_cast<double>(u) - static_cast<double>(half)) * static_cast<double>(a.scs);
            float hr[4] = {0.0f, 0.0f, 0.0f, 0.0f}, hi[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            for (uint32_t tp = 0; tp < a.taps; ++tp) {
                // e^(-j 2 pi f tau), the phase reduced to (-1/2, 1/2] cycles in fp64.
                const double cyc = f * tau[tp];
                const float frac = static_cast<float>(cyc - rint(cyc));
                float sn, cs;
                sincospif(2.0f * frac, &sn, &cs);
#pragma unroll
                for (uint32_t l = 0; l < 4; ++l) {
                    if (l < a.nl) {
                        const float2 gv = gs[l][tp];
                        hr[l] += gv.x * cs + gv.y * sn;
                        hi[l] += gv.y * cs - gv.x * sn;
                    }
                }
            }
#pragma unroll
            for (uint32_t l = 0; l < 4; ++l) {
                if (l < a.nl) {
                    const float2 x = gx[static_cast<size_t>(l) * gplane + u];
                    y.x += hr[l] * x.x - hi[l] * x.y;
                    y.y += hr[l] * x.y + hi[l] * x.x;
                }
            }
        }
        buf[__brev(k) >> (32u - a.log2n)] = y;
    }
    __syncthreads();
    // Radix-2 decimation-in-time inverse DFT: e^(+j 2 pi k n / N).
    for (uint32_t h = 1; h < n; h <<= 1) {
        const uint32_t stride = n / (2u * h);
        for (uint32_t b = t; b < n / 2u; b += blockDim.x) {
            const uint32_t grp = b / h, pos = b - grp * h;
            const uint32_t i0 = grp * 2u * h + pos, i1 = i0 + h;
            const float2 w = twiddle[pos * stride];
            const float2 v = buf[i1], uu = buf[i0];
            const float2 vw = make_float2(v.x * w.x - v.y * w.y, v.x * w.y + v.y * w.x);
            buf[i0] = make_float2(uu.x + vw.x, uu.y + vw.y);
            buf[i1] = make_float2(uu.x - vw.x, uu.y - vw.y);
        }
        __syncthreads();
    }
    const uint32_t cp = a.cp[sym], first = a.start[sym] - cp;
    const size_t row = (static_cast<size_t>(slot) * a.nr + rx) * a.samples;
    for (uint32_t p = t; p < cp + n; p += blockDim.x) {
        const float2 v = buf[p < cp ? n - cp + p : p - cp];
        const uint64_t pos = row + first + p;
        const float2 z = Gauss2(a.seed ^ (pos * 0x632be59bd9b4e019ull));
        const float re = v.x * a.inv_sqrt_n + a.sigma * z.x, im = v.y * a.inv_sqrt_n + a.sigma * z.y;
        if (a.iq_float) {
            static_cast<float2 *>(iq)[pos] = make_float2(re, im);
        } else {
            const float qr = fminf(fmaxf(rintf(re * 256.0f), -32768.0f), 32767.0f);
            const float qi = fminf(fmaxf(rintf(im * 256.0f), -32768.0f), 32767.0f);
            static_cast<short2 *>(iq)[pos] = make_short2(static_cast<short>(qr), static_cast<short>(qi));
        }
    }
}

void FreeDev(void *p)
{
    if (p != nullptr) (void)hipFree(p);
}

}  // namespace

struct AiranPuschTxGpu {
    PuschMimoConfig cfg{};
    Geom g{};
    TxPlan tp{};
    uint32_t max_tbs = 0, T = 1;
    uint32_t tb_chunks = 0, cb_chunks = 0, tb_parts = 0;
    uint32_t *tb_part = nullptr, *pow_tb = nullptr, *pow_cb = nullptr, *gold = nullptr;
    float2 *twiddle = nullptr;
};

extern "C" {

int32_t airan_pusch_txgpu_Create(const PuschMimoConfig *config, const AiranTbPlanV1 *plan, uint32_t max_tbs,
                                 uint32_t slots_per_tb, AiranPuschTxGpu **tx)
{
    if (config == nullptr || plan == nullptr || tx == nullptr || max_tbs == 0 || slots_per_tb == 0)
        return AIRAN_INVALID_ARGUMENT;
    *tx = nullptr;
    Geom g;
    int32_t st = airan::DeriveGeom(*config, &g);
    if (st != AIRAN_OK) return st;
    const AiranTbPlanV1 &p = *plan;
    if (p.C == 0 || p.Z == 0 || p.Z > kMaxZ || p.K != 22u * p.Z || p.Kprime > p.K || p.filler != p.K - p.Kprime ||
        p.Kprime < 2u * p.Z || p.Ncb == 0 || p.Ncb > 66u * p.Z || p.Ncb <= p.filler || p.k0 >= p.Ncb ||
        p.E_low % g.qm != 0 || p.E_high % g.qm != 0 || p.n_low > p.C ||
        static_cast<uint64_t>(p.G) != static_cast<uint64_t>(slots_per_tb) * g.cw_symbols * g.qm ||
        static_cast<uint64_t>(p.n_low) * p.E_low + static_cast<uint64_t>(p.C - p.n_low) * p.E_high != p.G ||
        p.tbs + p.crc_tb + static_cast<uint64_t>(p.C) * p.crc_cb != static_cast<uint64_t>(p.C) * p.Kprime ||
        (p.crc_tb != 0 && p.crc_tb != 16 && p.crc_tb != 24) || (p.crc_cb != 0 && p.crc_cb != 24))
        return AIRAN_UNSUPPORTED_PROFILE;
    auto *t = new AiranPuschTxGpu{};
    t->cfg = *config;
    t->g = g;
    t->max_tbs = max_tbs;
    t->T = slots_per_tb;
    TxPlan &tp = t->tp;
    tp.Z = p.Z;
    tp.C = p.C;
    tp.K = p.K;
    tp.kprime = p.Kprime;
    tp.crc_cb = p.crc_cb;
    tp.crc_tb = p.crc_tb;
    tp.per_cb = p.Kprime - p.crc_cb;
    tp.tbs = p.tbs;
    tp.filler = p.filler;
    tp.ncb = p.Ncb;
    const uint32_t fstart = p.Kprime - 2u * p.Z;
    tp.q0 = p.k0 < fstart ? p.k0 : (p.k0 >= fstart + p.filler ? p.k0 - p.filler : fstart);
    tp.G = p.G;
    tp.e_low = p.E_low;
    tp.e_high = p.E_high;
    tp.n_low = p.n_low;
    tp.tb_poly = p.crc_tb == 16 ? kPoly16 : kPolyA;
    tp.tb_len = p.crc_tb == 16 ? 16u : 24u;
    auto fail = [&](int32_t code) {
        airan_pusch_txgpu_Destroy(t);
        return code;
    };
    if (!CoreSchedule(p.Z, &tp)) return fail(AIRAN_UNSUPPORTED_PROFILE);
    t->tb_chunks = (p.tbs + kTbChunkBits - 1) / kTbChunkBits;
    t->cb_chunks = (tp.per_cb + kCbChunkBits - 1) / kCbChunkBits;
    t->tb_parts = airan::CeilDiv(t->tb_chunks, kTbBlockChunks);
    const std::vector<uint32_t> gold = GoldWords(
        (static_cast<uint32_t>(config->rnti) << 15) | ((static_cast<uint32_t>(config->codeword_index) & 1u) << 14) |
            config->data_scrambling_id,
        p.G / 32u + 2u);
    const std::vector<uint32_t> ptb = ChunkPowers(t->tb_chunks, kTbChunkBits, tp.tb_poly, tp.tb_len);
    const std::vector<uint32_t> pcb = ChunkPowers(t->cb_chunks, kCbChunkBits, kPolyB, 24);
    std::vector<float2> tw(g.fft / 2);
    for (uint32_t k = 0; k < g.fft / 2; ++k) {
        const double ph = 2.0 * M_PI * static_cast<double>(k) / static_cast<double>(g.fft);
        tw[k] = make_float2(static_cast<float>(std::cos(ph)), static_cast<float>(std::sin(ph)));
    }
    auto alloc = [](auto **ptr, size_t bytes) { return hipMalloc(reinterpret_cast<void **>(ptr), bytes) == hipSuccess; };
    if (!alloc(&t->tb_part, sizeof(uint32_t) * max_tbs * t->tb_parts) ||
        !alloc(&t->pow_tb, sizeof(uint32_t) * t->tb_chunks) || !alloc(&t->pow_cb, sizeof(uint32_t) * t->cb_chunks) ||
        !alloc(&t->gold, sizeof(uint32_t) * gold.size()) || !alloc(&t->twiddle, sizeof(float2) * tw.size()))
        return fail(AIRAN_RESOURCE_TOO_SMALL);
    if (hipMemcpy(t->pow_tb, ptb.data(), sizeof(uint32_t) * ptb.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(t->pow_cb, pcb.data(), sizeof(uint32_t) * pcb.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(t->gold, gold.data(), sizeof(uint32_t) * gold.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(t->twiddle, tw.data(), sizeof(float2) * tw.size(), hipMemcpyHostToDevice) != hipSuccess)
        return fail(AIRAN_LAUNCH_FAILED);
    if ((st = airan::InitGoldTables()) != AIRAN_OK) return fail(st);
    *tx = t;
    return AIRAN_OK;
}

void airan_pusch_txgpu_Destroy(AiranPuschTxGpu *t)
{
    if (t == nullptr) return;
    FreeDev(t->tb_part);
    FreeDev(t->pow_tb);
    FreeDev(t->pow_cb);
    FreeDev(t->gold);
    FreeDev(t->twiddle);
    delete t;
}

int32_t airan_pusch_txgpu_EncodeTbs(AiranPuschTxGpu *t, const uint8_t *payload, uint32_t num_tbs,
                                    const uint16_t *slot_numbers, float *grid, uint8_t *coded_bits, void *stream)
{
    if (t == nullptr || payload == nullptr || grid == nullptr || stream == nullptr || num_tbs == 0 ||
        num_tbs > t->max_tbs)
        return AIRAN_INVALID_ARGUMENT;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Geom &g = t->g;
    const TxPlan &tp = t->tp;
    if (tp.tbs == 0) return AIRAN_LAUNCH_FAILED;  // a CRC over nothing: no chunk to launch for
    const uint32_t ncb = num_tbs * tp.C;
    if (tp.crc_tb)
        hipLaunchKernelGGL(TbCrcKernel, dim3(t->tb_parts, num_tbs), dim3(256), 0, s, payload, tp, t->pow_tb,
                           t->tb_chunks, t->tb_part);
    EncodeArgs ea{};
    ea.g = airan::ToDev(g);
    ea.tb_parts = t->tb_parts;
    const uint32_t nf = tp.ncb - tp.filler;
    for (uint32_t i = 0; i < g.qm; ++i) {
        ea.start[0][i] = static_cast<uint32_t>((tp.q0 + static_cast<uint64_t>(i) * (tp.e_low / g.qm)) % nf);
        ea.start[1][i] = static_cast<uint32_t>((tp.q0 + static_cast<uint64_t>(i) * (tp.e_high / g.qm)) % nf);
    }
    ea.slots_per_tb = t->T;
    ea.norm = g.qm == 2 ? 1.0f / std::sqrt(2.0f)
                        : (g.qm == 4 ? 1.0f / std::sqrt(10.0f) : (g.qm == 6 ? 1.0f / std::sqrt(42.0f) : 1.0f / std::sqrt(170.0f)));
    ea.tb_part = t->tb_part;
    ea.pow_cb = t->pow_cb;
    ea.gold = t->gold;
    const auto encode = g.qm == 2   ? EncodeKernel<2>
                        : g.qm == 4 ? EncodeKernel<4>
                        : g.qm == 6 ? EncodeKernel<6>
                                    : EncodeKernel<8>;
    hipLaunchKernelGGL(encode, dim3(ncb), dim3(kEncodeThreads), 0, s, payload, tp, ea, reinterpret_cast<float2 *>(grid),
                       coded_bits);
    DmrsArgs da{};
    da.g = ea.g;
    da.slots = num_tbs * t->T;
    da.rb_start = t->cfg.rb_start;
    da.n_id = t->cfg.dmrs_scrambling_id;
    da.n_scid = t->cfg.n_scid;
    da.default_slot = t->cfg.slot_number;
    for (uint32_t l = 0; l < g.nl; ++l) da.wf_odd[l] = t->cfg.dmrs_ports[l] == 1001 || t->cfg.dmrs_ports[l] == 1003;
    hipLaunchKernelGGL(DmrsGridKernel, dim3(da.slots * g.nl * g.ndmrs), dim3(256), 0, s, da, slot_numbers,
                       reinterpret_cast<float2 *>(grid));
    return airan::LaunchStatus();
}

int32_t airan_pusch_txgpu_Channel(AiranPuschTxGpu *t, const float *grid, uint32_t slots, const float *gains,
                                  const float *delays, uint32_t taps, float scs_hz, float noise_var, uint64_t seed,
                                  uint32_t iq_format, void *iq, void *stream)
{
    if (t == nullptr || grid == nullptr || gains == nullptr || delays == nullptr || iq == nullptr ||
        stream == nullptr || slots == 0 || taps == 0 || taps > 32 || !(scs_hz > 0.0f) || !(noise_var >= 0.0f) ||
        (iq_format != AIRAN_IQ_INT16_Q8_8 && iq_format != AIRAN_IQ_COMPLEX64))
        return AIRAN_INVALID_ARGUMENT;
    const Geom &g = t->g;
    if (g.fft > kMaxFft) return AIRAN_UNSUPPORTED_PROFILE;
    ChanArgs a{};
    a.nr = g.nr;
    a.nl = g.nl;
    a.used = g.used;
    a.fft = g.fft;
    a.log2n = 0;
    while ((1u << a.log2n) < g.fft) ++a.log2n;
    a.taps = taps;
    a.samples = g.samples;
    a.iq_float = iq_format == AIRAN_IQ_COMPLEX64;
    for (uint32_t k = 0; k < 14; ++k) {
        a.cp[k] = k == 0 ? g.cp_long : g.cp_short;
        a.start[k] = g.sym_start[k];
    }
    a.scs = scs_hz;
    a.sigma = std::sqrt(noise_var * 0.5f);
    a.inv_sqrt_n = 1.0f / std::sqrt(static_cast<float>(g.fft));
    a.seed = seed;
    hipLaunchKernelGGL(ChannelOfdmKernel, dim3(slots * g.nr * 14u), dim3(256), 0, static_cast<hipStream_t>(stream),
                       reinterpret_cast<const float2 *>(grid), reinterpret_cast<const float2 *>(gains), delays,
                       t->twiddle, a, iq);
    return airan::LaunchStatus();
}

}  // extern "C"
