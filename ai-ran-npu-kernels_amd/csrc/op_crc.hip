// op_crc.hip -- code-block CRC24B and transport-block CRC24A/CRC16 checks
// (TS 38.212 5.1) on decoded bits, plus payload packing.
//
// The CRC remainder is linear in the message bits: for an n-bit message
// (data followed by its parity) it is the XOR over set bits j of
// x^(L + n - 1 - j) mod g, a GF(2) matrix times the bit vector.  Two kernels:
// CbCrcKernel, a workgroup per code block, whose threads multiply the 32 bits of
// a chunk, as a polynomial, by the tabulated power of the chunk's end; and from
// kCrcMfmaMin blocks on CrcMfmaKernel, the product on the matrix cores, 32 blocks
// to a workgroup.  Each block's share of its TB's remainder is its local one times
// x^(bits after it) mod g, written per block and XORed by a wave per TB.
#include <algorithm>
#include <mutex>
#include <vector>

#include "common.h"
#include "crc.h"
#include "launch.h"
#include "ragged.h"

namespace {

constexpr uint32_t kPolyA = 0x864CFBu;   // CRC24A
constexpr uint32_t kPolyB = 0x800063u;   // CRC24B
constexpr uint32_t kPoly16 = 0x1021u;    // CRC16
constexpr uint32_t kMaxPow = 8448 + 64;  // exponents 0..kMaxPow-1 above the CRC length

struct CrcTables {
    uint32_t *pow_a = nullptr;    // x^(24 + e) mod g_A
    uint32_t *pow_b = nullptr;    // x^(24 + e) mod g_B
    uint32_t *pow_16 = nullptr;   // x^(16 + e) mod g_16
};

std::mutex g_crc_mutex;
CrcTables g_tables[64];

uint32_t HostPow(uint32_t poly, uint32_t len, uint32_t e)
{
    // x^(len + e) mod g by repeated shift.
    uint32_t mask = (1u << len) - 1u;
    uint32_t r = 1;  // x^0
    for (uint32_t i = 0; i < len + e; ++i) {
        uint32_t top = (r >> (len - 1)) & 1u;
        r = (r << 1) & mask;
        if (top) r ^= poly;
    }
    return r;
}

int32_t EnsureTables(CrcTables **out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return AIRAN_LAUNCH_FAILED;
    std::lock_guard<std::mutex> lock(g_crc_mutex);
    CrcTables &t = g_tables[dev];
    if (t.pow_a == nullptr) {
        std::vector<uint32_t> a(kMaxPow), b(kMaxPow), c(kMaxPow);
        // iterative: x^(len+e) = x * x^(len+e-1)
        auto fill = [](std::vector<uint32_t> &v, uint32_t poly, uint32_t len) {
            uint32_t mask = (1u << len) - 1u;
            uint32_t r = HostPow(poly, len, 0);
            for (uint32_t e = 0; e < kMaxPow; ++e) {
                v[e] = r;
                uint32_t top = (r >> (len - 1)) & 1u;
                r = (r << 1) & mask;
                if (top) r ^= poly;
            }
        };
        fill(a, kPolyA, 24);
        fill(b, kPolyB, 24);
        fill(c, kPoly16, 16);
        if (hipMalloc(&t.pow_a, kMaxPow * 4) != hipSuccess || hipMalloc(&t.pow_b, kMaxPow * 4) != hipSuccess ||
            hipMalloc(&t.pow_16, kMaxPow * 4) != hipSuccess)
            return AIRAN_LAUNCH_FAILED;
        if (hipMemcpy(t.pow_a, a.data(), kMaxPow * 4, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(t.pow_b, b.data(), kMaxPow * 4, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(t.pow_16, c.data(), kMaxPow * 4, hipMemcpyHostToDevice) != hipSuccess)
            return AIRAN_LAUNCH_FAILED;
    }
    *out = &t;
    return AIRAN_OK;
}

struct CrcDev {
    uint32_t C, K, kprime, crc_cb, crc_tb, tbs;
    uint32_t poly_tb, len_tb;
};

// ------------------------------------------------------- one block per group
constexpr uint32_t kChunkThreads = 320;  // 32 positions each: 10240 >= 8448, the largest K

// The four 0/1 bytes of w as 4 bits, the first byte highest.
__device__ inline uint32_t Pack4(uint32_t w)
{
    return (((w & 0x01010101u) * 0x08040201u) >> 24) & 0xfu;
}

// v(x) p(x) mod g for the 32-bit polynomial v and a residue p, by Horner's
// rule with the residues left-aligned (the top bit is the sign bit).
__device__ inline uint32_t CrcMul32(uint32_t v, uint32_t p, uint32_t poly, uint32_t len)
{
    const uint32_t sh = 32u - len, pl = p << sh, gl = poly << sh;
    int32_t r = 0;
#pragma unroll
    for (int i = 31; i >= 0; --i) {
        const uint32_t top = static_cast<uint32_t>(r >> 31) & gl;
        const uint32_t bit = static_cast<uint32_t>(static_cast<int32_t>(v << (31 - i)) >> 31) & pl;
        r = static_cast<int32_t>((static_cast<uint32_t>(r) << 1) ^ top ^ bit);
    }
    return static_cast<uint32_t>(r) >> sh;
}

// Remainders of one block by a workgroup of kChunkThreads: rb of its first nb
// bits (CRC24B), ra of its first na (the TB CRC).  Thread t takes positions
// [32 t, 32 t + 32): their bits as a polynomial times x^(len + bits after
// them), tabulated in pow_*.  The result is valid in thread 0.
__device__ inline void CrcBlockRemainders(const int8_t *__restrict__ b, uint32_t K, uint32_t nb, uint32_t na,
                                          const uint32_t *__restrict__ pow_b, const uint32_t *__restrict__ pow_tb,
                                          uint32_t poly_tb, uint32_t len_tb, uint32_t *rb_out, uint32_t *ra_out)
{
    __shared__ uint32_t red[2][kChunkThreads / 64];
    const uint32_t t = threadIdx.x, p0 = 32u * t, n = max(nb, na);
    uint32_t v = 0;
    if (p0 < n) {
        if (K % 16u == 0 && (reinterpret_cast<uintptr_t>(b) & 15u) == 0) {
            const uint4 lo = *reinterpret_cast<const uint4 *>(b + p0);
            const uint4 hi = p0 + 16u < K ? *reinterpret_cast<const uint4 *>(b + p0 + 16) : make_uint4(0, 0, 0, 0);
            v = Pack4(lo.x) << 28 | Pack4(lo.y) << 24 | Pack4(lo.z) << 20 | Pack4(lo.w) << 16 | Pack4(hi.x) << 12 |
                Pack4(hi.y) << 8 | Pack4(hi.z) << 4 | Pack4(hi.w);
        } else {
            for (uint32_t j = 0; j < 32u && p0 + j < n; ++j) v |= static_cast<uint32_t>(b[p0 + j] & 1) << (31u - j);
        }
    }
    auto part = [&](uint32_t len_msg, const uint32_t *pw, uint32_t poly, uint32_t len) {
        if (p0 >= len_msg) return 0u;
        const uint32_t m = min(32u, len_msg - p0);
        return CrcMul32(v >> (32u - m), pw[len_msg - p0 - m], poly, len);
    };
    uint32_t rb = part(nb, pow_b, airan::kCrcPolyB, 24u), ra = part(na, pow_tb, poly_tb, len_tb);
    for (int off = 32; off > 0; off >>= 1) {
        rb ^= __shfl_xor(rb, off);
        ra ^= __shfl_xor(ra, off);
    }
    if ((t & 63u) == 0) {
        red[0][t >> 6] = rb;
        red[1][t >> 6] = ra;
    }
    __syncthreads();
    rb = ra = 0;
#pragma unroll
    for (uint32_t w = 0; w < kChunkThreads / 64u; ++w) {
        rb ^= red[0][w];
        ra ^= red[1][w];
    }
    *rb_out = rb;
    *ra_out = ra;
}

// bits: int8 0/1 per bit, [cb][K], any K and alignment; a workgroup per block.
// About 500 VALU instructions a wave, no table but the powers: 129 blocks take
// 5.2 us (latency), where the matrix product's few workgroups of 32 blocks
// take 16 (see kCrcMfmaMin).
__global__ void __launch_bounds__(kChunkThreads) CbCrcKernel(const int8_t *__restrict__ bits, airan::CrcJob c,
                                                            uint32_t K)
{
    const uint32_t cb = blockIdx.x;
    uint32_t rb, ra;
    CrcBlockRemainders(bits + static_cast<size_t>(cb) * K, K, c.crc_cb ? c.kprime : 0u, c.L, c.pow_b, c.pow_tb,
                       c.poly_tb, c.len_tb, &rb, &ra);
    if (threadIdx.x == 0) airan::CrcFinishBlock(c, cb, rb, ra);
}

// The same products on the matrix cores when K is a multiple of 32: the
// remainders of all blocks are R = M B over the integers, then mod 2, with
// M [64][K] the 0/1 term bits (rows 0..23 CRC24B, rows 32.. the TB CRC) and
// B [K][blocks] the 0/1 decoded bytes as they lie in memory (block-major).
// One v_mfma_i32_32x32x16_i8 step takes 16 positions; positions are taken
// in pairs of steps, lane l (half h = l / 32) supplying bytes
// [32 p + 16 h, 32 p + 16 h + 16) of its row (A) or block (B): the first 8
// for step 2p, the next 8 for step 2p+1 (any order of the positions serves,
// A and B agreeing).  The fragment table holds M in that order,
// frag[(tile P + p) 64 + l], so a wave loads 1 KB contiguous per tile and
// pair.
typedef int i32x16_t __attribute__((ext_vector_type(16)));
constexpr uint32_t kCrcCols = 32;   // blocks per workgroup (MFMA columns)
constexpr uint32_t kCrcWaves = 4;   // waves splitting the positions
constexpr uint32_t kCrcUnroll = 6;  // position pairs of a wave in flight together

__global__ void __launch_bounds__(256) CrcFragKernel(airan::CrcJob c, uint32_t P, uint4 *__restrict__ frag)
{
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= 2 * P * 64) return;
    const uint32_t l = e % 64, p = (e / 64) % P, tile = e / (64 * P);
    const uint32_t row = l % 32, pos0 = 32 * p + 16 * (l / 32);
    const uint32_t *pw = tile ? c.pow_tb : c.pow_b;
    const uint32_t n = tile ? c.L : (c.crc_cb ? c.kprime : 0u);
    const uint32_t len = tile ? c.len_tb : 24u;
    uint32_t w[4] = {0, 0, 0, 0};
    if (row < len) {
        for (uint32_t j = 0; j < 16; ++j) {
            const uint32_t pos = pos0 + j;
            if (pos < n) w[j / 4] |= ((pw[n - 1 - pos] >> row) & 1u) << (8 * (j % 4));
        }
    }
    frag[e] = make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ inline long Lo8(uint4 v) { return static_cast<long>(static_cast<uint64_t>(v.y) << 32 | v.x); }
__device__ inline long Hi8(uint4 v) { return static_cast<long>(static_cast<uint64_t>(v.w) << 32 | v.z); }

// bits: int8 0/1, [cb][K], K a multiple of 32 and bits 16-byte aligned.
// Workgroup b checks blocks 32 b .. 32 b + 31; wave w takes a contiguous
// quarter of the position pairs (consecutive loads of a lane share cache
// lines); the parities of the waves' partial sums are XOR-combined.
__global__ void __launch_bounds__(kCrcWaves * 64) CrcMfmaKernel(const int8_t *__restrict__ bits, airan::CrcJob c,
                                                               uint32_t K, uint32_t num_cb,
                                                               const uint4 *__restrict__ frag)
{
    const uint32_t l = threadIdx.x & 63u, w = threadIdx.x >> 6, h = l >> 5, col = l & 31u;
    const uint32_t P = K / 32;
    const uint32_t cb = blockIdx.x * kCrcCols + col;
    const bool live = cb < num_cb;
    const uint4 *src = reinterpret_cast<const uint4 *>(bits + static_cast<size_t>(live ? cb : 0u) * K) + h;
    i32x16_t acc_b = {}, acc_a = {};
    const uint32_t span = (P + kCrcWaves - 1) / kCrcWaves, pe = min(P, (w + 1) * span);
    for (uint32_t p0 = w * span; p0 < pe; p0 += kCrcUnroll) {
        // Every load is unconditional (clamped to a valid pair, masked at
        // use): a guarded load would make the compiler wait for it before
        // the next one.
        uint4 b[kCrcUnroll], a0[kCrcUnroll], a1[kCrcUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kCrcUnroll; ++u) {
            const uint32_t p = min(p0 + u, pe - 1);
            b[u] = src[2 * p];
            a0[u] = frag[p * 64 + l];
            a1[u] = frag[(P + p) * 64 + l];
        }
#pragma unroll
        for (uint32_t u = 0; u < kCrcUnroll; ++u) {
            if (!live || p0 + u >= pe) b[u] = make_uint4(0, 0, 0, 0);
            acc_b = __builtin_amdgcn_mfma_i32_32x32x16_i8(Lo8(a0[u]), Lo8(b[u]), acc_b, 0, 0, 0);
            acc_b = __builtin_amdgcn_mfma_i32_32x32x16_i8(Hi8(a0[u]), Hi8(b[u]), acc_b, 0, 0, 0);
            acc_a = __builtin_amdgcn_mfma_i32_32x32x16_i8(Lo8(a1[u]), Lo8(b[u]), acc_a, 0, 0, 0);
            acc_a = __builtin_amdgcn_mfma_i32_32x32x16_i8(Hi8(a1[u]), Hi8(b[u]), acc_a, 0, 0, 0);
        }
    }
    // Accumulator r of lane l is row 8 (r / 4) + 4 h + r % 4 of column col.
    uint32_t pb = 0, pa = 0;
#pragma unroll
    for (uint32_t r = 0; r < 16; ++r) {
        const uint32_t row = 8 * (r / 4) + 4 * h + r % 4;
        pb |= (static_cast<uint32_t>(acc_b[r]) & 1u) << row;
        pa |= (static_cast<uint32_t>(acc_a[r]) & 1u) << row;
    }
    pb |= __shfl_xor(pb, 32);
    pa |= __shfl_xor(pa, 32);
    __shared__ uint32_t red[kCrcWaves][2][kCrcCols];
    if (h == 0) {
        red[w][0][col] = pb;
        red[w][1][col] = pa;
    }
    __syncthreads();
    if (threadIdx.x < kCrcCols && live) {
        uint32_t xb = 0, xa = 0;
        for (uint32_t v = 0; v < kCrcWaves; ++v) {
            xb ^= red[v][0][col];
            xa ^= red[v][1][col];
        }
        airan::CrcFinishBlock(c, cb, xb, xa);
    }
}

// tb_ok of TB blockIdx.x (one wave): the XOR of its C blocks' shifted
// remainder parts is zero.
__global__ void __launch_bounds__(64) TbFinishKernel(const uint32_t *__restrict__ tb_part,
                                                     uint8_t *__restrict__ tb_ok, uint32_t C)
{
    const uint32_t tb = blockIdx.x, l = threadIdx.x;
    const uint32_t *p = tb_part + static_cast<size_t>(tb) * C;
    uint32_t x = 0;
    for (uint32_t r = l; r < C; r += 64) x ^= p[r];
    for (int off = 32; off > 0; off >>= 1) x ^= __shfl_xor(x, off);
    if (l == 0) tb_ok[tb] = x == 0;
}
// Payload byte b of TB tb: bits 8b..8b+7 (MSB first) of the TB bit stream.
__global__ void __launch_bounds__(256) PackKernel(const int8_t *__restrict__ bits,
                                                  uint8_t *__restrict__ out, CrcDev d)
{
    const uint32_t nbytes = (d.tbs + 7) / 8;
    const uint32_t byte = blockIdx.x * blockDim.x + threadIdx.x;
    if (byte >= nbytes) return;
    const uint32_t tb = blockIdx.y;
    const uint32_t L = d.kprime - d.crc_cb;
    uint32_t v = 0;
    for (uint32_t k = 0; k < 8; ++k) {
        const uint32_t t = byte * 8 + k;
        uint32_t bit = 0;
        if (t < d.tbs) {
            const uint32_t r = t / L, j = t - r * L;
            bit = bits[(static_cast<size_t>(tb) * d.C + r) * d.K + j] & 1;
        }
        v |= bit << (7 - k);
    }
    out[static_cast<size_t>(tb) * nbytes + byte] = static_cast<uint8_t>(v);
}


// Ragged batch: one workgroup per code block of any grant.  The block's
// CRC24B remainder over its K' bits and the remainder of its part of the
// TB (its first K' - crc_cb bits) as the last bits of a message, shifted by
// x^(bits after it in its TB) mod g_TB (the host's per-block `xpow`).  2282
// blocks in 16.5 us; with two table loads per set bit it took 49.
__global__ void __launch_bounds__(kChunkThreads) RaggedCrcKernel(const int8_t *__restrict__ bits,
                                                                const airan::RaggedCb *__restrict__ cbs,
                                                                const uint32_t *__restrict__ pow_b,
                                                                const uint32_t *__restrict__ pow_a,
                                                                const uint32_t *__restrict__ pow_16,
                                                                uint8_t *__restrict__ cb_ok,
                                                                uint32_t *__restrict__ tb_part)
{
    const airan::RaggedCb &c = cbs[blockIdx.x];
    uint32_t rb, ra;
    CrcBlockRemainders(bits + c.bits_off, c.k, c.crc_cb ? c.kprime : 0u, c.kprime - c.crc_cb, pow_b,
                       c.len_tb == 24 ? pow_a : pow_16, c.poly_tb, c.len_tb, &rb, &ra);
    if (threadIdx.x == 0) {
        cb_ok[blockIdx.x] = c.crc_cb ? static_cast<uint8_t>(rb == 0) : static_cast<uint8_t>(1);
        tb_part[blockIdx.x] = airan::CrcMulMod(ra, c.xpow, c.poly_tb, c.len_tb);
    }
}

// tb_ok of TB blockIdx.x (one wave): the parts of its code blocks (first[t] ..
// first[t] + count[t] - 1) XOR to zero.
__global__ void __launch_bounds__(64) RaggedCrcFinishKernel(const uint32_t *__restrict__ tb_part,
                                                            const uint32_t *__restrict__ first,
                                                            const uint32_t *__restrict__ count,
                                                            uint8_t *__restrict__ tb_ok)
{
    const uint32_t t = blockIdx.x, n = count[t];
    const uint32_t *p = tb_part + first[t];
    uint32_t x = 0;
    for (uint32_t r = threadIdx.x; r < n; r += 64) x ^= p[r];
    for (int off = 32; off > 0; off >>= 1) x ^= __shfl_xor(x, off);
    if (threadIdx.x == 0) tb_ok[t] = x == 0 ? 1 : 0;
}

}  // namespace

namespace airan {

uint32_t CrcXpowHost(const AiranTbPlanV1 &p, uint32_t r)
{
    const uint32_t poly = p.crc_tb == 24 ? kPolyA : kPoly16, len = p.crc_tb;
    const uint32_t mask = (1u << len) - 1u;
    uint64_t e = static_cast<uint64_t>(p.C - 1 - r) * (p.Kprime - p.crc_cb);
    // x^e mod g by square-and-multiply on the host.
    auto mul = [&](uint32_t a, uint32_t b) {
        uint32_t res = 0;
        for (int i = static_cast<int>(len) - 1; i >= 0; --i) {
            const uint32_t top = (res >> (len - 1)) & 1u;
            res = (res << 1) & mask;
            if (top) res ^= poly;
            if ((b >> i) & 1u) res ^= a;
        }
        return res;
    };
    uint32_t x = 1u, base = 2u;
    while (e != 0) {
        if (e & 1u) x = mul(x, base);
        base = mul(base, base);
        e >>= 1;
    }
    return x;
}

uint32_t CrcTbPoly(uint32_t crc_tb) { return crc_tb == 24 ? kPolyA : kPoly16; }

int32_t LaunchCrcRagged(const RaggedCb *cbs, uint32_t num_cb, const int8_t *bits, uint8_t *cb_ok, uint32_t *tb_part,
                        const uint32_t *tb_first, const uint32_t *tb_count, uint8_t *tb_ok, uint32_t num_tbs,
                        hipStream_t s)
{
    CrcTables *t = nullptr;
    const int32_t st = EnsureTables(&t);
    if (st != AIRAN_OK) return st;
    if (num_cb == 0 || num_tbs == 0) return AIRAN_INVALID_ARGUMENT;
    hipLaunchKernelGGL(RaggedCrcKernel, dim3(num_cb), dim3(kChunkThreads), 0, s, bits, cbs, t->pow_b, t->pow_a,
                       t->pow_16, cb_ok, tb_part);
    hipLaunchKernelGGL(RaggedCrcFinishKernel, dim3(num_tbs), dim3(64), 0, s, tb_part, tb_first, tb_count, tb_ok);
    return LaunchStatus();
}

int32_t CrcJobSetup(const AiranTbPlanV1 &p, uint8_t *cb_ok, uint32_t *tb_part, CrcJob *out)
{
    if (p.C == 0 || p.C > kCrcMaxCb || p.Kprime > p.K || p.K > 8448 || p.Kprime < p.crc_cb ||
        (p.crc_tb != 24 && p.crc_tb != 16) ||
        (p.crc_cb != 0 && p.crc_cb != 24) ||
        static_cast<uint64_t>(p.C) * (p.Kprime - p.crc_cb) != static_cast<uint64_t>(p.tbs) + p.crc_tb)
        return AIRAN_INVALID_ARGUMENT;
    CrcTables *t = nullptr;
    const int32_t st = EnsureTables(&t);
    if (st != AIRAN_OK) return st;
    *out = CrcJob{t->pow_b, p.crc_tb == 24 ? t->pow_a : t->pow_16, cb_ok, tb_part, nullptr, p.C, p.Kprime, p.crc_cb,
                   p.Kprime - p.crc_cb, p.crc_tb == 24 ? kPolyA : kPoly16, p.crc_tb};
    return AIRAN_OK;
}

// Blocks from which the matrix product (32 blocks per workgroup) is the faster
// check.  A workgroup per block against it, K = 8448: 129 blocks 5.2 / 16.1 us,
// 2064 blocks 15.7 / 19.0 us, 8256 blocks 42.9 / 31.9 us; lines through these
// cross near 3000.
constexpr uint32_t kCrcMfmaMin = 3000;

// The matrix-core path needs whole position pairs and aligned 16-byte loads.
bool CrcMfmaEligible(const void *bits, uint32_t K, uint32_t num_cb, const void *tables)
{
    return num_cb >= kCrcMfmaMin && K % 32 == 0 &&
           ((reinterpret_cast<uintptr_t>(bits) | reinterpret_cast<uintptr_t>(tables)) & 15u) == 0;
}

// The fragment table of the matrix product, where a check of num_cb blocks
// would take it.
void LaunchCrcTables(const CrcJob &c, uint32_t K, uint32_t num_cb, void *tables, hipStream_t s)
{
    if (K % 32 != 0 || num_cb < kCrcMfmaMin) return;
    const uint32_t P = K / 32;
    static_assert(kCrcTableBytes >= 2 * (8448 / 32) * 64 * sizeof(uint4), "fragment table size");
    hipLaunchKernelGGL(CrcFragKernel, dim3(CeilDiv(2 * P * 64, 256)), dim3(256), 0, s, c, P,
                       static_cast<uint4 *>(tables));
}

void LaunchCbCrc(const int8_t *bits, const CrcJob &c, uint32_t K, uint32_t num_cb, const void *tables,
                 hipStream_t s)
{
    if (CrcMfmaEligible(bits, K, num_cb, tables))
        hipLaunchKernelGGL(CrcMfmaKernel, dim3(CeilDiv(num_cb, kCrcCols)), dim3(kCrcWaves * 64), 0, s, bits, c, K,
                           num_cb, static_cast<const uint4 *>(tables));
    else
        hipLaunchKernelGGL(CbCrcKernel, dim3(num_cb), dim3(kChunkThreads), 0, s, bits, c, K);
}

void LaunchCrcFinish(const uint32_t *tb_part, uint8_t *tb_ok, uint32_t num_tbs, uint32_t C, hipStream_t s)
{
    hipLaunchKernelGGL(TbFinishKernel, dim3(num_tbs), dim3(64), 0, s, tb_part, tb_ok, C);
}

}  // namespace airan

extern "C" size_t airan_crc_check_WorkspaceBytes(uint32_t num_tbs)
{
    // Per-block TB remainder parts, then the matrix product's table.
    return airan::CrcTableOffset(num_tbs) + airan::kCrcTableBytes;
}

extern "C" int32_t airan_crc_check_Enqueue(const AiranTbPlanV1 *p, uint32_t num_tbs, const void *bits,
                                           void *cb_ok, void *tb_ok, void *tb_bytes, void *workspace,
                                           size_t workspace_bytes, void *stream)
{
    if (p == nullptr || bits == nullptr || cb_ok == nullptr || tb_ok == nullptr || stream == nullptr ||
        num_tbs == 0 || p->C == 0 || p->C > airan::kCrcMaxCb || p->Kprime > p->K || p->K > 8448 ||
        p->Kprime < p->crc_cb || (p->crc_tb != 24 && p->crc_tb != 16) || (p->crc_cb != 0 && p->crc_cb != 24) ||
        static_cast<uint64_t>(p->C) * (p->Kprime - p->crc_cb) != static_cast<uint64_t>(p->tbs) + p->crc_tb)
        return AIRAN_INVALID_ARGUMENT;
    if (workspace == nullptr || workspace_bytes < airan_crc_check_WorkspaceBytes(num_tbs))
        return AIRAN_RESOURCE_TOO_SMALL;
    CrcTables *t = nullptr;
    int32_t st = EnsureTables(&t);
    if (st != AIRAN_OK) return st;
    CrcDev d{p->C, p->K, p->Kprime, p->crc_cb, p->crc_tb, p->tbs,
             p->crc_tb == 24 ? kPolyA : kPoly16, p->crc_tb};
    airan::CrcJob c{t->pow_b, p->crc_tb == 24 ? t->pow_a : t->pow_16, static_cast<uint8_t *>(cb_ok),
                     static_cast<uint32_t *>(workspace), nullptr, p->C, p->Kprime, p->crc_cb,
                     p->Kprime - p->crc_cb, d.poly_tb, d.len_tb};
    hipStream_t s = static_cast<hipStream_t>(stream);
    void *tables = static_cast<uint8_t *>(workspace) + airan::CrcTableOffset(num_tbs);
    airan::LaunchCrcTables(c, p->K, num_tbs * p->C, tables, s);
    airan::LaunchCbCrc(static_cast<const int8_t *>(bits), c, p->K, num_tbs * p->C, tables, s);
    airan::LaunchCrcFinish(static_cast<const uint32_t *>(workspace), static_cast<uint8_t *>(tb_ok), num_tbs, p->C, s);
    if (tb_bytes != nullptr) {
        dim3 grid(airan::CeilDiv((p->tbs + 7) / 8, 256), num_tbs);
        hipLaunchKernelGGL(PackKernel, grid, dim3(256), 0, s, static_cast<const int8_t *>(bits),
                           static_cast<uint8_t *>(tb_bytes), d);
    }
    return airan::LaunchStatus();
}
