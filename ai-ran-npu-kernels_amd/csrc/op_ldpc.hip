// op_ldpc.hip -- BG1 layered normalized min-sum LDPC decoder for gfx950.
//
// Schedule and arithmetic follow fec/ldpc_decode/ldpc_decode_kernel.cpp:
// rows in order (:533-713), per row gather -> subtract old message ->
// min1/min2/sign product -> alpha = 0.75 (:248-300) -> posterior update and
// scatter; final clamp +-5120, int16 conversion with CAST_RINT and bit =
// (int16 value < 0) (:719-780), i.e. a REF-mode posterior in [-0.5, 0)
// decodes to 0.
//
// Two kernels.  LdpcPairKernel (FP16 messages, at most 8 active rows, Z < 384
// mainly; UsePair has the rule): two code blocks per workgroup, one in each
// fp16 half of every posterior word.  LdpcCheckPairKernel (the rest): one code
// block per workgroup, two checks of it per lane.  In both the posterior lives in LDS, the message state in
// registers, a thread owns the same checks of every row (within a row the
// threads touch a permutation of each column, so nothing conflicts) and a
// barrier separates rows.
#include <algorithm>
#include <mutex>

#include "common.h"
#include "airan_ldpc_bg1.h"
#include "launch.h"
#include "ragged.h"
#include "ratematch.h"

// Posterior of the code blocks owned by a pair decoder workgroup whose
// lifting size is not known at compile time.
extern __shared__ uint16_t airan_ldpc_lam[];

namespace {

// ------------------------------------------------------------------ fast path
// FP16 messages and at most kFastRows active rows (every code rate above
// about 0.75), with:
//  * row degrees fixed at compile time and per-lifting-size edge words
//    (col * Z | (shift mod Z) << 16) in constant memory, so an edge costs a
//    scalar load and three VALU ops of addressing;
//  * fp16 VALU arithmetic on the posterior: a single fp16 add/sub/mul of
//    fp16 operands rounds exactly like the fp32 operation rounded to fp16
//    (fp32 has 24 >= 2*11 + 2 significand bits, so rounding twice is
//    innocuous);
//  * LDS holding only the (22 + rows) columns the active rows touch, so
//    several code blocks share a CU; columns beyond never change.
// With FUSED the decoder input is de-rate-matched on the fly from the
// bit-plane codeword LLRs (the standalone rate-dematch arithmetic).
constexpr int kNumLift = 5;  // Z = 24 << zi
constexpr int kFastRows = 8;
constexpr int kFastDeg[kFastRows] = {19, 19, 19, 19, 3, 8, 9, 7};

constexpr int FastRowStart(int r)
{
    int s = 0;
    for (int i = 0; i < r; ++i) s += kFastDeg[i];
    return s;
}

constexpr int kFastEdges = FastRowStart(kFastRows);

struct Bg1LiftDev {
    uint32_t w[kNumLift][kFastEdges];
};

__constant__ Bg1LiftDev kLift;

// To the current device.
int32_t CopyLiftTable()
{
    for (int r = 0; r < kFastRows; ++r)
        if (AIRAN_BG1_ROW_START[r] != FastRowStart(r) ||
            AIRAN_BG1_ROW_START[r + 1] - AIRAN_BG1_ROW_START[r] != kFastDeg[r])
            return AIRAN_LAUNCH_FAILED;
    Bg1LiftDev t{};
    for (int zi = 0; zi < kNumLift; ++zi) {
        const uint32_t z = 24u << zi;
        for (int e = 0; e < kFastEdges; ++e)
            t.w[zi][e] = static_cast<uint32_t>(AIRAN_BG1_COL[e]) * z |
                         (static_cast<uint32_t>(AIRAN_BG1_SHIFT[e]) % z) << 16;
    }
    return hipMemcpyToSymbol(HIP_SYMBOL(kLift), &t, sizeof(t)) == hipSuccess ? AIRAN_OK : AIRAN_LAUNCH_FAILED;
}

using h16 = _Float16;

__device__ __forceinline__ h16 HBits(uint32_t b) { return __builtin_bit_cast(h16, static_cast<uint16_t>(b)); }
__device__ __forceinline__ uint32_t BitsH(h16 h) { return __builtin_bit_cast(uint16_t, h); }

// Negative and non-zero (fp16 bits), as `value < 0` on the decoded posterior.
__device__ __forceinline__ uint32_t NegBit(uint32_t h) { return (h & 0xffffu) - 0x8001u <= 0x7bffu ? 1u : 0u; }

__device__ __forceinline__ uint32_t LiftAddr(uint32_t w, uint32_t i, uint32_t Z)
{
    uint32_t p = i + (w >> 16);
    p = min(p, p - Z);
    return (w & 0xffffu) + p;
}

// Two code blocks per workgroup: block "A" in the low and block "B" in the
// high fp16 half of every 32-bit posterior word, so one LDS access, one set
// of edge addresses and one packed fp16 add (v_pk_add_f16) serve both.
// Every message of the thread's check lives in a register (one packed pair
// per edge), so the extrinsic is lam - msg with no reconstruction of the old
// message from a compressed state.  Check i of row R, per half:
//   x_k = lam_k - msg_k; min1/min2 of the magnitudes |x_k| (fp16
//   magnitudes order like unsigned integers), sign bits !(x_k >= 0) (bits
//   above 0x7c00: negative, or a NaN), parity p;
//   msg_k = (|x_k| == |min1| ? 0.75 min2 : 0.75 min1) with sign
//   p ^ sign(x_k), and lam_k = x_k + msg_k.
// Selecting the second minimum by magnitude is selecting it by index: an edge whose
// magnitude equals min1 without being min1's index implies min2 == min1, so
// selecting by magnitude instead of index changes no value; and a message's
// sign differs from the recorded sign bit only for a NaN extrinsic, whose
// posterior is NaN and stays NaN (every later extrinsic on it is NaN), so the
// stored message sign is never observed.
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2_t H2(uint32_t x) { return __builtin_bit_cast(h2_t, x); }
__device__ __forceinline__ uint32_t WH(h2_t x) { return __builtin_bit_cast(uint32_t, x); }

// Packed unsigned 16-bit operations on both halves (VOP3P).
__device__ __forceinline__ uint32_t PkMinU16(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_pk_min_u16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint32_t PkMaxU16(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_pk_max_u16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// max(a - b, 0) per half.
__device__ __forceinline__ uint32_t PkSubSatU16(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// (a - b) mod 2^16 per half.
__device__ __forceinline__ uint32_t PkSubU16(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_pk_sub_u16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// (a * b + c) mod 2^16 per half.
__device__ __forceinline__ uint32_t PkMadU16(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Signed 16-bit max / min per half.
__device__ __forceinline__ uint32_t PkMaxI16(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_pk_max_i16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ uint32_t PkMinI16(uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_pk_min_i16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
typedef short s16x2 __attribute__((ext_vector_type(2)));

// Per half: 1 if the fp16 bits exceed 0x7c00 (negative, or a NaN), else 0.
__device__ __forceinline__ uint32_t AboveInf2(uint32_t x) { return PkMinU16(PkSubSatU16(x, 0x7c007c00u), 0x00010001u); }

// Per half: NegBit (negative, non-zero, not NaN) as 0 / 1: x - 0x8001 < 0x7c00.
__device__ __forceinline__ uint32_t NegBit2(uint32_t x)
{
    return PkMinU16(PkSubSatU16(0x7c007c00u, PkSubU16(x, 0x80018001u)), 0x00010001u);
}

// Byte offset in LDS of edge e's posterior word for check i: column base +
// 4 ((i + shift) mod Z), i4 = 4 i, i4m = 4 i - 4 Z (mod 2^32).  With ZT != 0,
// Z = ZT and the edge's column and shift are compile-time constants (callers
// unroll over e): the lanes past the wrap (4 i >= 4 (Z - s)) take i4m, the
// others i4 (a compare and a select), and the constant column base + 4 s
// goes to the LDS instruction's offset field, which the hardware adds to the
// address register modulo 2^32 (so i4m + offset lands on 4 (i + s - Z));
// the posterior must start at LDS address 0 for the offset to hold all of
// it.  Otherwise the edge word comes from the per-lifting-size table.
template <uint32_t ZT>
__device__ __forceinline__ uint32_t EdgeByte(const uint32_t *lw, int e, uint32_t i, uint32_t i4, uint32_t i4m,
                                             uint32_t Z)
{
    if constexpr (ZT != 0) {
        const uint32_t s4 = 4u * (static_cast<uint32_t>(AIRAN_BG1_SHIFT[e]) % ZT);
        const uint32_t base = i4 < 4u * ZT - s4 ? i4 : i4m;
        return base + (4u * static_cast<uint32_t>(AIRAN_BG1_COL[e]) * ZT + s4);
    } else {
        return 4u * LiftAddr(lw[e], i, Z);
    }
}

__device__ __forceinline__ uint32_t &LdsWord(uint32_t *lam2, uint32_t byte)
{
    return *reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(lam2) + byte);
}

// Check i of row R for both blocks.  min1 / min2 are tracked on the fp16
// magnitudes (with duplicates: two edges at the minimum give min2 == min1),
// starting from two virtual edges of magnitude 0x7c00, which is what the
// keys (|x| << 5 | k) from (0x7c00 << 5) give for the magnitudes.  A row
// with an infinite or NaN extrinsic sets *inf_flag.
template <int R, uint32_t ZT>
__device__ __forceinline__ void PairRow(uint32_t *lam2, uint32_t zi, uint32_t i, uint32_t Z, uint32_t *msg,
                                        uint32_t *inf_flag)
{
    constexpr int DEG = kFastDeg[R], E0 = FastRowStart(R);
    const uint32_t *lw = kLift.w[zi];
    // Opaque per row: with compile-time edges the addresses depend on i
    // alone and would otherwise be hoisted out of the iteration loop, every
    // row's at once, in registers.
    uint32_t i4 = 4u * i, i4m = 4u * i - 4u * Z;
    asm volatile("" : "+v"(i4), "+v"(i4m));
    uint32_t m1 = 0x7c007c00u, m2 = 0x7c007c00u;
    // XOR of the extrinsics (bits 15 / 31: the sign parity of each half) and
    // the largest magnitude per half (above 0x7c00 a NaN, 0x7c00 an infinity).
    uint32_t sx = 0, mx = 0;
    // The row's extrinsics and addresses are not held: the message pass
    // reads each posterior again (no other thread writes it within the row)
    // and recomputes its address, and the loads go kChunk at a time, so that
    // the kernel fits 128 VGPRs without spills and a CU holds two workgroups
    // (12 waves) whatever SIMDs their waves land on.
    constexpr int kChunk = 6;
#pragma unroll
    for (int k = 0; k < DEG; ++k) {
        if (k % kChunk == 0 && k > 0) __builtin_amdgcn_sched_barrier(0);
        const uint32_t x = WH(H2(LdsWord(lam2, EdgeByte<ZT>(lw, E0 + k, i, i4, i4m, Z))) - H2(msg[E0 + k]));
        const uint32_t mg = x & 0x7fff7fffu;
        m2 = PkMinU16(m2, PkMaxU16(m1, mg));
        m1 = PkMinU16(m1, mg);
        sx ^= x;
        mx = PkMaxU16(mx, mg);
    }
    const h2_t q = {static_cast<_Float16>(0.75f), static_cast<_Float16>(0.75f)};
    // The parity counts the edges whose bits exceed 0x7c00 (negative, or a
    // NaN of either sign).  Without a NaN in the row that is the sign bit,
    // so the parity is sx's; a row with an infinite or NaN extrinsic (rare,
    // and sticky once a posterior is NaN) counts the extrinsics again and
    // sets the flag.
    uint32_t par = sx & 0x80008000u;
    if (PkSubSatU16(mx, 0x7bff7bffu) != 0) {
        *inf_flag = 1u;
        uint32_t cnt = 0;
#pragma unroll
        for (int k = 0; k < DEG; ++k)
            cnt += AboveInf2(WH(H2(LdsWord(lam2, EdgeByte<ZT>(lw, E0 + k, i, i4, i4m, Z))) - H2(msg[E0 + k])));
        par = (cnt & 1u) << 15 | ((cnt >> 16) & 1u) << 31;
    }
    const uint32_t s1p = WH(q * H2(m1)) | par, s2p = WH(q * H2(m2)) | par;
    const uint32_t d12 = PkSubU16(s2p, s1p);
    // Message pass, kUpd edges at a time: their posteriors are all read
    // before any is written, so the reads of a group are in flight together
    // (within a row every posterior word belongs to one edge of one thread,
    // so no read of the row aliases another edge's write).
    constexpr int kUpd = 6;
#pragma unroll
    for (int k0 = 0; k0 < DEG; k0 += kUpd) {
        constexpr int kMax = kUpd;
        const int n = DEG - k0 < kMax ? DEG - k0 : kMax;
        if (k0 > 0) __builtin_amdgcn_sched_barrier(0);
        uint32_t a[kMax], v[kMax];
#pragma unroll
        for (int k = 0; k < kMax; ++k)
            if (k < n) {
                a[k] = EdgeByte<ZT>(lw, E0 + k0 + k, i, i4, i4m, Z);
                v[k] = LdsWord(lam2, a[k]);
            }
#pragma unroll
        for (int k = 0; k < kMax; ++k)
            if (k < n) {
                const uint32_t x = WH(H2(v[k]) - H2(msg[E0 + k0 + k]));
                // 1 per half where |x_k| == min1, then s1p + that * (s2p - s1p).
                const uint32_t e = PkSubSatU16(0x00010001u, (x & 0x7fff7fffu) ^ m1);
                const uint32_t m = PkMadU16(e, d12, s1p) ^ (x & 0x80008000u);
                msg[E0 + k0 + k] = m;
                LdsWord(lam2, a[k]) = WH(H2(x) + H2(m));
            }
    }
}

template <int R, int ROWS, uint32_t ZT>
__device__ __forceinline__ void PairIteration(uint32_t *lam2, uint32_t zi, uint32_t i, uint32_t Z, uint32_t *msg,
                                              uint32_t *inf_flag)
{
    if constexpr (R < ROWS) {
        if (i < Z) PairRow<R, ZT>(lam2, zi, i, Z, msg, inf_flag);
        __syncthreads();
        PairIteration<R + 1, ROWS, ZT>(lam2, zi, i, Z, msg, inf_flag);
    }
}

// Bit 0: A's check i fails a row's parity; bit 16: B's.  Rows are taken
// one at a time within the 128-VGPR budget of up to 6 active rows, three at
// a time above (their loads in flight together).  A hard decision is
// NegBit (negative, non-zero, not NaN).  No posterior is ever -0 (the
// start values are +0 or non-zero, and round-to-nearest sums and
// differences give -0 only from -0 operands), so without a NaN it is the
// sign bit and a row's parity is the XOR of its posteriors' words (!EXACT);
// EXACT evaluates NegBit per posterior.
template <int R, int ROWS, uint32_t ZT, bool EXACT>
__device__ __forceinline__ uint32_t PairSyndrome(uint32_t *lam2, const uint32_t *lw, uint32_t i, uint32_t Z)
{
    constexpr int G = ROWS <= 6 ? 1 : 3;
    if constexpr (R < ROWS) {
        constexpr int RE = R + G < ROWS ? R + G : ROWS;
        constexpr int E0 = FastRowStart(R), N = FastRowStart(RE) - E0;
        uint32_t i4 = 4u * i, i4m = 4u * i - 4u * Z;
        asm volatile("" : "+v"(i4), "+v"(i4m));
        uint32_t v[N];
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = LdsWord(lam2, EdgeByte<ZT>(lw, E0 + k, i, i4, i4m, Z));
        __builtin_amdgcn_sched_barrier(0);
        uint32_t par = 0;
#pragma unroll
        for (int r = R; r < RE; ++r) {
            uint32_t pr = 0;
#pragma unroll
            for (int k = FastRowStart(r) - E0; k < FastRowStart(r + 1) - E0; ++k) pr ^= EXACT ? NegBit2(v[k]) : v[k];
            par |= EXACT ? pr : (pr >> 15) & 0x00010001u;
        }
        asm volatile("" : "+v"(par) : : "memory");
        return par | PairSyndrome<RE, ROWS, ZT, EXACT>(lam2, lw, i, Z);
    }
    return 0;
}

// Shared words of the pair decoder after its posterior: taken_cb[2],
// syn_bad[8], syn_exact[8], inf_flag[2].
constexpr uint32_t kPairTailWords = 20;

// The pair decoder's LDS: posterior then kPairTailWords.  With Z = ZT known
// at compile time a static array, whose address is a compile-time constant
// (0: the kernel has no other shared variable), so that every edge's column
// base and shift fold into the LDS instructions' offsets; otherwise the
// dynamic allocation.
template <int ROWS, uint32_t ZT>
__device__ __forceinline__ uint32_t *PairLds()
{
    if constexpr (ZT != 0) {
        __shared__ uint32_t buf[(22 + ROWS) * ZT + kPairTailWords];
        return buf;
    } else {
        return reinterpret_cast<uint32_t *>(airan_ldpc_lam);
    }
}

struct LdpcFastDev {
    uint32_t z, zi, k, iters, rows, early_stop, num_cb;
    airan::RateDev rate;  // FUSED: codeword geometry
};

// Decoder input LLR of position t of a block, as the fp16 posterior start
// value (LLR / 256).
__device__ inline uint32_t InputH(int32_t v)
{
    return BitsH(static_cast<h16>(static_cast<float>(v) * (1.0f / 256.0f)));
}

// Loads block cb's posterior start values into half h of lam2 (nl
// positions; cb >= num_cb: a zero block).  FUSED: de-rate-matched from the
// bit-plane codeword LLRs with descriptor desc[cb].
template <bool FUSED>
__device__ inline void PairLoad(uint16_t *lam16, uint32_t h, uint32_t nl, const int16_t *__restrict__ src,
                                const RateMatchDescriptor *__restrict__ desc, const LdpcFastDev &d, uint32_t cb)
{
    const uint32_t i = threadIdx.x;
    if (cb >= d.num_cb) {
        for (uint32_t t = i; t < nl; t += blockDim.x) lam16[2 * t + h] = 0;
        return;
    }
    if constexpr (FUSED) {
        const airan::RateCb rc = airan::RateCbSetup(desc[cb], d.rate);
        if (airan::RateSingle(rc, d.rate)) {
            // Every transmitted bit kk < E lands on its own position (the
            // inverse of RateSingleIndex): q = (q0 + kk) mod (Ncb - filler),
            // position 2Z + (q < fstart ? q : q + filler).  So the block's
            // codeword LLRs -- Qm planes of E/Qm consecutive symbols -- are
            // scattered into LDS after the other positions are set (zero, or
            // +5120 for filler bits).  The symbols of a plane are read in
            // aligned 16-byte chunks of 8 (cw_stride is a multiple of 8) where
            // a chunk lies inside the plane's [rem0, rem0 + eq), and one by one
            // at the plane's two ends (at most 7 each).  A chunk whose 8
            // positions are consecutive (no wrap of q, no filler boundary, all
            // below nl: every chunk but about one per block) is converted with
            // packed int16 clamps and an exact int16 -> fp16 conversion:
            // InputH(clamp(8 x, +-5120)) = fp16(clamp(x, +-640)) / 32, exact.
            const uint32_t two_z = 2u * d.z, fstart = d.rate.kprime - two_z;
            const uint32_t nf = d.rate.ncb - d.rate.filler;
            const int16_t *slot = src + static_cast<size_t>(rc.slot0) * d.rate.qm * d.rate.cw_stride;
            const uint32_t cfirst = (rc.rem0 + 7u) / 8u, clast = (rc.rem0 + rc.eq) / 8u;
            const uint32_t ni = clast > cfirst ? clast - cfirst : 0u;  // whole chunks per plane
            const uint32_t nh = ni ? 8u * cfirst - rc.rem0 : rc.eq;     // symbols before them
            const uint32_t nt = ni ? rc.rem0 + rc.eq - 8u * clast : 0u; // and after them
            const uint32_t total = ni * d.rate.qm;
            const float rcp_ni = 1.0f / static_cast<float>(ni ? ni : 1u);
            // Symbol j (< eq) of plane b, raw codeword LLR v: its position and value.
            auto put = [&](uint32_t b, uint32_t j, int32_t v) {
                uint32_t q = rc.q0 + b * rc.eq + j;
                q = q >= nf ? q - nf : q;
                const uint32_t t = two_z + (q < fstart ? q : q + d.rate.filler);
                if (t >= nl) return;
                v *= 8;
                v = v > 5120 ? 5120 : (v < -5120 ? -5120 : v);
                lam16[2 * t + h] = static_cast<uint16_t>(InputH(v));
            };
            auto chunk_of = [&](uint32_t e, uint32_t &b, uint32_t &cc) {
                b = static_cast<uint32_t>(static_cast<float>(e) * rcp_ni);
                b = b * ni > e ? b - 1u : b;
                b = (b + 1u) * ni <= e ? b + 1u : b;
                cc = cfirst + (e - b * ni);
            };
            constexpr uint32_t kBatch = 2;  // chunk loads of a thread in flight together
            uint4 raw[kBatch];
            auto fetch = [&](uint32_t e0) {
#pragma unroll
                for (uint32_t u = 0; u < kBatch; ++u) {
                    const uint32_t e = e0 + u * blockDim.x;
                    if (e < total) {
                        uint32_t b, cc;
                        chunk_of(e, b, cc);
                        raw[u] = *reinterpret_cast<const uint4 *>(slot + static_cast<size_t>(b) * d.rate.cw_stride +
                                                                  8u * cc);
                    }
                }
            };
            // The first batch is in flight while the other positions are set.
            uint32_t e0 = i;
            fetch(e0);
            const uint32_t fill = InputH(5120);
            for (uint32_t t = i; t < nl; t += blockDim.x)
                lam16[2 * t + h] = static_cast<uint16_t>(
                    t >= two_z + fstart && t < two_z + fstart + d.rate.filler ? fill : 0u);
            __syncthreads();
            // The plane ends, one symbol per thread (at most 14 Qm of them).
            const uint32_t ne = nh + nt;
            for (uint32_t f = i; f < ne * d.rate.qm; f += blockDim.x) {
                const uint32_t b = f / ne, r = f - b * ne;
                const uint32_t j = r < nh ? r : 8u * clast - rc.rem0 + (r - nh);
                put(b, j, slot[static_cast<size_t>(b) * d.rate.cw_stride + rc.rem0 + j]);
            }
            const h2_t scale = {static_cast<_Float16>(1.0f / 32.0f), static_cast<_Float16>(1.0f / 32.0f)};
            while (e0 < total) {
#pragma unroll
                for (uint32_t u = 0; u < kBatch; ++u) {
                    const uint32_t e = e0 + u * blockDim.x;
                    if (e >= total) continue;
                    uint32_t b, cc;
                    chunk_of(e, b, cc);
                    const uint32_t j0 = 8u * cc - rc.rem0;
                    uint32_t q = rc.q0 + b * rc.eq + j0;
                    q = q >= nf ? q - nf : q;
                    const uint32_t t0 = two_z + (q < fstart ? q : q + d.rate.filler);
                    const uint32_t w[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
                    if (q + 8u <= nf && (q >= fstart || q + 8u <= fstart) && t0 + 8u <= nl) {
#pragma unroll
                        for (uint32_t k = 0; k < 4; ++k) {
                            const uint32_t c = PkMinI16(PkMaxI16(w[k], 0xfd80fd80u), 0x02800280u);
                            const h2_t v = __builtin_convertvector(__builtin_bit_cast(s16x2, c), h2_t) * scale;
                            const uint32_t vb = WH(v);
                            lam16[2 * (t0 + 2u * k) + h] = static_cast<uint16_t>(vb);
                            lam16[2 * (t0 + 2u * k + 1u) + h] = static_cast<uint16_t>(vb >> 16);
                        }
                    } else {
#pragma unroll
                        for (uint32_t x = 0; x < 8; ++x)
                            put(b, j0 + x, static_cast<int16_t>(w[x >> 1] >> (16u * (x & 1u))));
                    }
                }
                e0 += kBatch * blockDim.x;
                if (e0 < total) fetch(e0);
            }
        } else {
            for (uint32_t t = i; t < nl; t += blockDim.x)
                lam16[2 * t + h] = static_cast<uint16_t>(InputH(airan::RateDematchValue(t, rc, d.rate, src)));
        }
    } else {
        // nl is a multiple of 4 (Z is a multiple of 24) and the block 8-byte aligned.
        const uint2 *s4 = reinterpret_cast<const uint2 *>(src + static_cast<size_t>(cb) * 68u * d.z);
        for (uint32_t t = i; t < nl / 4u; t += blockDim.x) {
            const uint2 v = s4[t];
            lam16[8 * t + h] = static_cast<uint16_t>(InputH(static_cast<int16_t>(v.x & 0xffffu)));
            lam16[8 * t + 2 + h] = static_cast<uint16_t>(InputH(static_cast<int16_t>(v.x >> 16)));
            lam16[8 * t + 4 + h] = static_cast<uint16_t>(InputH(static_cast<int16_t>(v.y & 0xffffu)));
            lam16[8 * t + 6 + h] = static_cast<uint16_t>(InputH(static_cast<int16_t>(v.y >> 16)));
        }
    }
}

// Writes block cb (half h of lam2): iteration count, hard bits and, when
// lam_out is set, the int16 posterior (positions beyond the LDS part keep
// their input).  Called by the whole workgroup; ends with a barrier, after
// which half h may be overwritten.
template <bool FUSED>
__device__ inline void PairEmit(const uint32_t *lam2, uint32_t h, uint32_t cb, uint32_t it, uint32_t nl,
                                const int16_t *__restrict__ src, const RateMatchDescriptor *__restrict__ desc,
                                int8_t *__restrict__ bits, int16_t *__restrict__ lam_out,
                                uint8_t *__restrict__ iters_out, const LdpcFastDev &d)
{
    const uint32_t i = threadIdx.x;
    const uint16_t *lam16 = reinterpret_cast<const uint16_t *>(lam2);
    if (iters_out != nullptr && i == 0) iters_out[cb] = static_cast<uint8_t>(it);
    int8_t *bo = bits + static_cast<size_t>(cb) * d.k;
    const uint32_t sh = 16u * h;
    if ((d.k & 3u) == 0) {
        const uint4 *l4 = reinterpret_cast<const uint4 *>(lam2);
        for (uint32_t t = i; t < d.k / 4u; t += blockDim.x) {
            const uint4 v = l4[t];
            reinterpret_cast<uint32_t *>(bo)[t] =
                NegBit(v.x >> sh) | NegBit(v.y >> sh) << 8 | NegBit(v.z >> sh) << 16 | NegBit(v.w >> sh) << 24;
        }
    } else {
        for (uint32_t t = i; t < d.k; t += blockDim.x) bo[t] = static_cast<int8_t>(NegBit(lam16[2 * t + h]));
    }
    if (lam_out != nullptr) {
        const uint32_t N = 68u * d.z;
        const airan::RateCb rc = FUSED ? airan::RateCbSetup(desc[cb], d.rate) : airan::RateCb{};
        int16_t *lo = lam_out + static_cast<size_t>(cb) * N;
        for (uint32_t t = i; t < N; t += blockDim.x) {
            float v;
            if (t < nl) {
                v = static_cast<float>(HBits(lam16[2 * t + h]));
            } else {
                const int16_t x = FUSED ? airan::RateDematchValue(t, rc, d.rate, src)
                                        : src[static_cast<size_t>(cb) * N + t];
                v = static_cast<float>(HBits(InputH(x)));
            }
            v = v > 20.0f ? 20.0f : (v < -20.0f ? -20.0f : v);
            lo[t] = static_cast<int16_t>(rintf(v * 256.0f));
        }
    }
    __syncthreads();
}

// Persistent decoder: the G = gridDim.x workgroups decode the blocks two at
// a time, one per half of the posterior words.  When a half's block is done
// (syndrome clear under early stop, or the iteration limit) its outputs are
// written and the next block is loaded into that half (its messages reset)
// while the other half runs on; a half past the last block holds a zero
// block and is never written.  The workgroups take blocks 0, 1, ... from
// the counter queue[0] (two words, zero at launch and left zero) as halves
// free up -- workgroups that start late hold no block meanwhile -- or, with
// queue null, workgroup b walks its static list
// b, b + G, b + 2 G, ...  Blocks are independent of the pairing
// (the halves never interact), so every block's outputs equal a decode of
// that block alone.  src: int16 decoder LLRs [cb][68 Z] (!FUSED) or
// bit-plane codeword LLRs with per-block descriptors (FUSED).  LDS holds the
// (22 + rows) Z posterior pairs the active rows touch.
//
// The refill code (emit, take, load) exists once, in a rolled loop over the
// two halves that also does the first loads.  Up to 6 active rows the kernel
// is held to 4 waves per SIMD (128 VGPRs): a 6-wave workgroup's waves land
// 2, 2, 1, 1 on the SIMDs, and only at 4 waves per SIMD does a second
// workgroup always fit beside it (at 3 the hardware kept one per CU).
template <bool FUSED, int ROWS, uint32_t ZT>
__global__ void __launch_bounds__(384)
    __attribute__((amdgpu_waves_per_eu(ROWS <= 6 ? 4 : 1, ROWS <= 6 ? 4 : 8)))
    LdpcPairKernel(const int16_t *__restrict__ src, const RateMatchDescriptor *__restrict__ desc,
                   int8_t *__restrict__ bits, int16_t *__restrict__ lam_out, uint8_t *__restrict__ iters_out,
                   LdpcFastDev d, uint32_t *__restrict__ queue)
{
    uint32_t *lam2 = PairLds<ROWS, ZT>();
    const uint32_t Z = d.z, i = threadIdx.x;
    const uint32_t nl = (22u + ROWS) * Z;
    // The few shared words live after the posterior (kPairTailWords).  taken_cb: one slot per half (a wave may
    // still be reading half 0's take when thread 0 takes for half 1:
    // PairLoad need not end with a barrier).  syn_bad / syn_exact: per wave,
    // bit h set when half h fails a check.  inf_flag[it0 & 1] (it0 before
    // the pass's increment): some row of the pass saw an infinite or NaN
    // extrinsic, or (harmless: it only selects the exact syndrome) an
    // earlier pass that used the same word did.
    uint32_t *taken_cb = lam2 + nl, *syn_bad = taken_cb + 2, *syn_exact = syn_bad + 8, *inf_flag = syn_exact + 8;
    if (i < 2) inf_flag[i] = 0;  // before the first barrier
    constexpr int kEdges = FastRowStart(ROWS);
    uint32_t msg[kEdges];
#pragma unroll
    for (int e = 0; e < kEdges; ++e) msg[e] = 0;
    uint32_t taken = 0;
    // Per half: its block (>= num_cb: none) and the iterations run on it.
    uint32_t cur0 = ~0u, cur1 = ~0u, it0 = 0, it1 = 0;
    uint32_t refill = 3u;  // bit h: half h is written (if it holds a block) and refilled
    const uint32_t *lw = kLift.w[d.zi];
    for (;;) {
        if (refill != 0) {
#pragma nounroll
            for (uint32_t h = 0; h < 2; ++h) {
                if (((refill >> h) & 1u) == 0) continue;
                const uint32_t cb = h ? cur1 : cur0;
                // The next block is taken before this one's outputs are
                // written, so the queue atomic overlaps the emission, whose
                // closing barrier also publishes the taken index.
                if (queue != nullptr && i == 0) taken_cb[h] = atomicAdd(queue, 1u);
                if (cb < d.num_cb)
                    PairEmit<FUSED>(lam2, h, cb, h ? it1 : it0, nl, src, desc, bits, lam_out, iters_out, d);
                else
                    __syncthreads();
                const uint32_t next =
                    queue == nullptr ? blockIdx.x + taken * gridDim.x : __builtin_amdgcn_readfirstlane(taken_cb[h]);
                ++taken;
                PairLoad<FUSED>(reinterpret_cast<uint16_t *>(lam2), h, nl, src, desc, d, next);
                if (h) {
                    cur1 = next;
                    it1 = 0;
                } else {
                    cur0 = next;
                    it0 = 0;
                }
                const uint32_t keep = h ? 0x0000ffffu : 0xffff0000u;
#pragma unroll
                for (int e = 0; e < kEdges; ++e) msg[e] &= keep;
            }
            __syncthreads();
            if (cur0 >= d.num_cb && cur1 >= d.num_cb) break;
        }
        // Uniform (it0 is the same in every lane): a scalar, so that the
        // flag's address takes no vector register across the pass.
        const uint32_t slot = __builtin_amdgcn_readfirstlane(it0) & 1u;
        PairIteration<0, ROWS, ZT>(lam2, d.zi, i, Z, msg, inf_flag + slot);
        ++it0;
        ++it1;
        uint32_t ok = 0;  // bit h: half h's syndrome is clear
        if (d.early_stop) {
            // Both halves' flags in one barrier: each wave's ballots into
            // syn_bad[wave] (rewritten only after further barriers).  The
            // parity is the sign-bit XOR unless some thread saw an infinite
            // or NaN extrinsic in the iteration: a NaN posterior is created
            // only from an infinite operand, which the row reading it would
            // have seen, and every posterior the syndrome reads was read and
            // rewritten in the iteration.  Then the syndrome is evaluated
            // again with NegBit (rare: saturated blocks only).
            //
            // inf_flag[slot] was set (if at all) before the last row's
            // barrier and is read below; the other word is cleared here for
            // a later pass (this pass writes and reads only inf_flag[slot]):
            // its last reads were in an earlier pass, before this pass's
            // first row barrier, and its next writes follow this pass's
            // syndrome barrier.
            const uint32_t bad = i < Z ? PairSyndrome<0, ROWS, ZT, false>(lam2, lw, i, Z) : 0u;
            const uint32_t wb = (__ballot((bad & 1u) != 0) != 0 ? 1u : 0u) | (__ballot((bad >> 16) != 0) != 0 ? 2u : 0u);
            if ((i & 63u) == 0) syn_bad[i >> 6] = wb;
            if (i == 0) inf_flag[slot ^ 1u] = 0;
            const bool exact = inf_flag[slot] != 0;
            __syncthreads();
            uint32_t any = 0;
            for (uint32_t w = 0; w < blockDim.x / 64u; ++w) any |= syn_bad[w];
            if (exact) {
                const uint32_t bx = i < Z ? PairSyndrome<0, ROWS, ZT, true>(lam2, lw, i, Z) : 0u;
                const uint32_t wx =
                    (__ballot((bx & 1u) != 0) != 0 ? 1u : 0u) | (__ballot((bx >> 16) != 0) != 0 ? 2u : 0u);
                if ((i & 63u) == 0) syn_exact[i >> 6] = wx;
                __syncthreads();
                any = 0;
                for (uint32_t w = 0; w < blockDim.x / 64u; ++w) any |= syn_exact[w];
            }
            ok = ~any & 3u;
        }
        refill = 0;
        if (cur0 < d.num_cb && ((ok & 1u) || it0 >= d.iters)) refill |= 1u;
        if (cur1 < d.num_cb && ((ok & 2u) || it1 >= d.iters)) refill |= 2u;
    }
    // The last workgroup to finish leaves the queue zeroed for the next
    // launch: every take (queue[0]) precedes its workgroup's count in queue[1].
    if (queue != nullptr && i == 0) {
        __threadfence();
        if (atomicAdd(queue + 1, 1u) == gridDim.x - 1) {
            atomicExch(queue, 0u);
            atomicExch(queue + 1, 0u);
        }
    }
}

// ------------------------------------------------------------------ any rows
// One code block per workgroup, two checks per lane: lane i of the first Z/2
// owns checks i and i + Z/2 of every row.  Word j of a column in LDS holds
// positions j (low half) and j + Z/2 (high half), so an edge with shift s
// takes one word -- that of (i + s) mod Z/2 -- its halves exchanged where i + s
// mod Z lands in the upper half (a rotate by 16 on the read and the write),
// and every operation of the row is a packed one on both checks.  Unlike two
// blocks per workgroup (LdpcPairKernel) this halves the LDS and the waves of a
// block, so blocks of any rows, lifting size and iteration count share a CU.
//
// Message state, all in registers: the messages themselves for the four
// degree-19 rows (76 words) and, up to kFewRows rows, for the others; beyond,
// an extension row keeps its two scaled magnitudes and the signs and
// minimum flags of its edges (one bit per edge and check), from which the old
// message is rebuilt as it was computed.  Rows kStaticRows .. 45 (degrees 4 to
// 8) run in one rolled loop over a table of edge words with their state in
// register arrays indexed by the row (s_set_gpr_idx): unrolled, the code of
// 316 edges would not fit the instruction cache.
//
// The arithmetic is that of PairRow (see there: values, parity, infinities and
// NaN).  In MODE_REF the message that is kept (and subtracted in the next
// iteration) is the reference's int8 one, its magnitude rounded half to even
// and clamped to 127, while the posterior takes the fp16 one, so posteriors
// grow from iteration to iteration and may become infinite.
//
// Bound by VALU issue (about 21 instructions per edge and two checks with
// kept messages, 30 with rebuilt ones) and, with fewer blocks than CUs, by a
// row's latency.  Against one check per lane with a compressed state that
// went through memory every row, Z = 384: 200 blocks of 46 rows, 8
// iterations at most 1029 -> 277 us; 143 blocks of 46 rows, 3 iterations, REF
// 378 -> 135 us; 6 blocks of 9 rows 238 -> 49 us; 2282 ragged blocks, with the
// rate dematch that was a pass of its own before, 1564 -> 438 us.
constexpr int kRows = AIRAN_BG1_ROWS;
constexpr int kFewRows = 10;     // rows of the kernel that keeps every message
constexpr int kStaticRows = 10;  // rows unrolled; the rest have degrees 4 .. 8
constexpr int kMinLoopDeg = 4, kMaxLoopDeg = 8;

// Edge words per lifting size: LDS byte of the column's word (shift mod Z/2)
// in bits 0 .. 15, 4 (Z/2 - shift mod Z/2) in bits 16 .. 25 (the lanes' 4 i
// from which on the word index wraps), bit 31: shift >= Z/2.  A row's info:
// first edge | degree << 16.  Padded for reads of kMaxLoopDeg words.
struct Bg1EdgeDev {
    uint32_t w[kNumLift][AIRAN_BG1_EDGES + kMaxLoopDeg];
    uint32_t row[kRows + 2];
};

__constant__ Bg1EdgeDev kEdges;

// To the current device, under g_table_mutex.
int32_t CopyEdgeTable()
{
    static Bg1EdgeDev t;
    t = Bg1EdgeDev{};
    for (int r = 0; r < kRows; ++r) {
        const uint32_t e0 = AIRAN_BG1_ROW_START[r], deg = AIRAN_BG1_ROW_START[r + 1] - e0;
        if (r >= kStaticRows && (deg < kMinLoopDeg || deg > kMaxLoopDeg)) return AIRAN_LAUNCH_FAILED;
        t.row[r] = e0 | deg << 16;
    }
    for (int zi = 0; zi < kNumLift; ++zi) {
        const uint32_t z = 24u << zi, zh = z / 2;
        for (int e = 0; e < AIRAN_BG1_EDGES; ++e) {
            const uint32_t s = AIRAN_BG1_SHIFT[e] % z, sh = s % zh;
            t.w[zi][e] = 4u * (AIRAN_BG1_COL[e] * zh + sh) | 4u * (zh - sh) << 16 | (s >= zh ? 1u << 31 : 0u);
        }
    }
    return hipMemcpyToSymbol(HIP_SYMBOL(kEdges), &t, sizeof(t)) == hipSuccess ? AIRAN_OK : AIRAN_LAUNCH_FAILED;
}

// Per-device "constant tables loaded" flags, guarded by a mutex (callers on
// several host threads may load them at once).
std::mutex g_table_mutex;
bool g_tables_loaded[64] = {};

// Both tables on the current device, whichever kernel the call takes: that
// depends on the number of blocks and their alignment, and a caller who has
// decoded once may capture the next call, where nothing can be copied.
int32_t LoadTables()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return AIRAN_LAUNCH_FAILED;
    std::lock_guard<std::mutex> lock(g_table_mutex);
    if (g_tables_loaded[dev]) return AIRAN_OK;
    int32_t st = CopyLiftTable();
    if (st == AIRAN_OK) st = CopyEdgeTable();
    g_tables_loaded[dev] = st == AIRAN_OK;
    return st;
}

// Lifting sizes other than 24 << zi (plans made by hand may have any of 24 ..
// 384): one check per lane, word j of a column holds position j in its low
// half and zero in the high one, so that odd sizes work and no rotation is
// needed.  Their edge words (word index col Z + shift mod Z in bits 0 .. 15,
// Z - shift mod Z above) are made by each workgroup, in LDS.
// Half of every packed operation is idle and each edge word is an LDS read and a
// readfirstlane: one kernel for all of them, not the fastest for any.  Ragged
// batches of one size, against the kernel with a compressed state in memory that
// decoded them before: 600 blocks of Z = 383, 25 rows 1795 -> 1090 us, 2000 of
// Z = 36, 45 rows 4211 -> 3539, 200 of Z = 340 898 -> 438.
constexpr uint32_t kAnyZ = 1;  // as ZT
constexpr uint32_t kMaxZ = 384;
// As ZT: a size below 384 read from the arguments; one of at most 96, with the
// lanes and the LDS of 96.
constexpr uint32_t kLowZ = 0, kZ96 = 2;

constexpr bool IsLiftSize(uint32_t z)
{
    for (int zi = 0; zi < kNumLift; ++zi)
        if (z == 24u << zi) return true;
    return false;
}

// LDS byte of an edge's word for the lane (4 i = i4) and the rotation that
// puts check i's position into the low half.
struct EdgeAt {
    uint32_t byte, rot;
};

// Edge e with Z = ZT: column and shift are compile-time constants, in the LDS
// instruction's offset (the posterior starts at LDS address 0; the hardware
// adds modulo 2^32, see EdgeByte).
template <uint32_t ZT>
__device__ __forceinline__ EdgeAt StaticEdge(int e, uint32_t i4)
{
    constexpr uint32_t zh = ZT / 2;
    const uint32_t s = static_cast<uint32_t>(AIRAN_BG1_SHIFT[e]) % ZT, sh = s % zh;
    const bool hi = s >= zh, wrap = sh != 0 && i4 >= 4u * (zh - sh);
    return {(wrap ? i4 - 4u * zh : i4) + 4u * (AIRAN_BG1_COL[e] * zh + sh), wrap != hi ? 16u : 0u};
}

// The edge of table word w; zh4 = 2 Z (4 Z with one check per lane).
template <uint32_t ZT>
__device__ __forceinline__ EdgeAt TableEdge(uint32_t w, uint32_t i4, uint32_t zh4)
{
    if constexpr (ZT == kAnyZ) return {i4 + 4u * (w & 0xffffu) - (i4 >= 4u * (w >> 16) ? zh4 : 0u), 0u};
    const bool hi = (w >> 31) != 0, wrap = i4 >= ((w >> 16) & 0x3ffu);
    return {i4 + (w & 0xffffu) - (wrap ? zh4 : 0u), wrap != hi ? 16u : 0u};
}

// Word e of a table: scalar, also from LDS.
template <uint32_t ZT>
__device__ __forceinline__ uint32_t TableWord(const uint32_t *tab, uint32_t e)
{
    if constexpr (ZT == kAnyZ) return __builtin_amdgcn_readfirstlane(tab[e]);
    return tab[e];
}

__device__ __forceinline__ uint32_t Rot16(uint32_t v, uint32_t rot) { return __builtin_amdgcn_alignbit(v, v, rot); }

// The row's parity in the sign bits (PairRow's, with its exact count).
template <int DEG>
__device__ __forceinline__ uint32_t RowParity(const uint32_t (&x)[DEG], uint32_t sx, uint32_t mx, uint32_t *inf_flag)
{
    if (PkSubSatU16(mx, 0x7bff7bffu) != 0) {
        *inf_flag = 1u;
        uint32_t cnt = 0;
#pragma unroll
        for (int k = 0; k < DEG; ++k) cnt += AboveInf2(x[k]);
        return (cnt & 1u) << 15 | ((cnt >> 16) & 1u) << 31;
    }
    return sx & 0x80008000u;
}

// int8 magnitude of an fp16 one: round half to even, at most 127 (0x57f0).
__device__ __forceinline__ uint32_t Int8Magnitude2(uint32_t v)
{
    return PkMinU16(WH(__builtin_elementwise_rint(H2(v))), 0x57f057f0u);
}

// One row: edge(k, i4) places edge k, old(k) is its message (both checks),
// put(k, x, e, m) takes the new one (e: 1 per half where the edge is at the
// minimum); s1p and d12 return the kept messages' two magnitudes with the
// row's parity in the sign bits, as s1p and s2p - s1p (mod 2^16 per half).  The
// addresses are computed anew for the second pass (three instructions an edge,
// against two registers and a mask), and a long row is taken kChunk edges at a
// time, both to stay within the registers.
template <int MODE, int DEG, typename Edge, typename Old, typename Put>
__device__ __forceinline__ void CheckRow(uint32_t *lam, uint32_t i4, uint32_t *inf_flag, uint32_t &s1p, uint32_t &d12,
                                         Edge edge, Old old, Put put)
{
    constexpr int kChunk = 7;
    uint32_t x[DEG];
    uint32_t m1 = 0x7c007c00u, m2 = 0x7c007c00u, sx = 0, mx = 0;
#pragma unroll
    for (int k = 0; k < DEG; ++k) {
        if (k > 0 && k % kChunk == 0) __builtin_amdgcn_sched_barrier(0);
        const EdgeAt a = edge(k, i4);
        x[k] = WH(H2(Rot16(LdsWord(lam, a.byte), a.rot)) - H2(old(k)));
        const uint32_t mg = x[k] & 0x7fff7fffu;
        m2 = PkMinU16(m2, PkMaxU16(m1, mg));
        m1 = PkMinU16(m1, mg);
        sx ^= x[k];
        mx = PkMaxU16(mx, mg);
    }
    const uint32_t par = RowParity<DEG>(x, sx, mx, inf_flag);
    const h2_t q = {static_cast<_Float16>(0.75f), static_cast<_Float16>(0.75f)};
    const uint32_t f1 = WH(q * H2(m1)), f2 = WH(q * H2(m2)), f1p = f1 | par, fd = PkSubU16(f2 | par, f1p);
    s1p = f1p;
    d12 = fd;
    if constexpr (MODE == AIRAN_LDPC_MODE_REF) {
        s1p = Int8Magnitude2(f1) | par;
        d12 = PkSubU16(Int8Magnitude2(f2) | par, s1p);
    }
    asm volatile("" : "+v"(i4));
#pragma unroll
    for (int k = 0; k < DEG; ++k) {
        if (k > 0 && k % kChunk == 0) __builtin_amdgcn_sched_barrier(0);
        const EdgeAt a = edge(k, i4);
        const uint32_t e = PkSubSatU16(0x00010001u, (x[k] & 0x7fff7fffu) ^ m1);
        const uint32_t sg = x[k] & 0x80008000u, m = PkMadU16(e, fd, f1p) ^ sg;
        put(k, x[k], e, MODE == AIRAN_LDPC_MODE_REF ? PkMadU16(e, d12, s1p) ^ sg : m);
        LdsWord(lam, a.byte) = Rot16(WH(H2(x[k]) + H2(m)), a.rot);
    }
}

constexpr int StaticDeg(int r) { return AIRAN_BG1_ROW_START[r + 1] - AIRAN_BG1_ROW_START[r]; }

// Unrolled row R with every message kept (msg: this row's words).
template <int MODE, uint32_t ZT, int R>
__device__ __forceinline__ void FullRow(uint32_t *lam, const uint32_t *tab, uint32_t i4, uint32_t zh4, uint32_t *msg,
                                        uint32_t *inf_flag)
{
    constexpr int E0 = AIRAN_BG1_ROW_START[R], DEG = StaticDeg(R);
    uint32_t s1p, d12;
    auto edge = [&](int k, uint32_t i4) {
        if constexpr (ZT == kMaxZ)
            return StaticEdge<ZT>(E0 + k, i4);
        else
            return TableEdge<ZT>(TableWord<ZT>(tab, E0 + k), i4, zh4);
    };
    CheckRow<MODE, DEG>(
        lam, i4, inf_flag, s1p, d12, edge, [&](int k) { return msg[k]; },
        [&](int k, uint32_t, uint32_t, uint32_t m) { msg[k] = m; });
}

// Unrolled row R (degree at most 10) with compressed state st: s1p, d12,
// minimum flags (bit k / 16 + k of edge k), signs (the same).
template <int MODE, uint32_t ZT, int R>
__device__ __forceinline__ void PackedRow(uint32_t *lam, const uint32_t *tab, uint32_t i4, uint32_t zh4, uint32_t *st,
                                          uint32_t *inf_flag)
{
    constexpr int E0 = AIRAN_BG1_ROW_START[R], DEG = StaticDeg(R);
    static_assert(DEG <= 16, "one bit per edge and check");
    const uint32_t o1 = st[0], od = st[1], oe = st[2], os = st[3];
    uint32_t ne = 0, ns = 0;
    auto edge = [&](int k, uint32_t i4) {
        if constexpr (ZT == kMaxZ)
            return StaticEdge<ZT>(E0 + k, i4);
        else
            return TableEdge<ZT>(TableWord<ZT>(tab, E0 + k), i4, zh4);
    };
    CheckRow<MODE, DEG>(
        lam, i4, inf_flag, st[0], st[1], edge,
        [&](int k) { return PkMadU16((oe >> k) & 0x00010001u, od, o1) ^ ((os << (15 - k)) & 0x80008000u); },
        [&](int k, uint32_t x, uint32_t e, uint32_t) {
            ne |= e << k;
            ns |= (x >> (15 - k)) & (0x00010001u << k);
        });
    st[2] = ne;
    st[3] = ns;
}

// A row of the loop: state s1p, d12 and meta (edge k: sign bit k, minimum
// flag bit 8 + k, and 16 above for the other check).  w: its edge words.
template <int MODE, uint32_t ZT, int DEG>
__device__ __forceinline__ void LoopRow(uint32_t *lam, const uint32_t *w, uint32_t i4, uint32_t zh4, uint32_t &s1p,
                                        uint32_t &d12, uint32_t &meta, uint32_t *inf_flag)
{
    const uint32_t o1 = s1p, od = d12, om = meta;
    uint32_t nm = 0;
    CheckRow<MODE, DEG>(
        lam, i4, inf_flag, s1p, d12, [&](int k, uint32_t i4) { return TableEdge<ZT>(w[k], i4, zh4); },
        [&](int k) { return PkMadU16((om >> (8 + k)) & 0x00010001u, od, o1) ^ ((om << (15 - k)) & 0x80008000u); },
        [&](int k, uint32_t x, uint32_t e, uint32_t) {
            nm |= e << (8 + k);
            nm |= (x >> (15 - k)) & (0x00010001u << k);
        });
    meta = nm;
}

// The unrolled rows from R on, a barrier after each.
template <int MODE, uint32_t ZT, bool FULL, int R>
__device__ __forceinline__ void StaticRows(uint32_t *lam, const uint32_t *tab, uint32_t i4, uint32_t zh4, bool mine,
                                           int rows, uint32_t *core, uint32_t *ext, uint32_t *inf_flag)
{
    if constexpr (R < kStaticRows) {
        // Opaque per row: the addresses depend on the lane alone and would
        // otherwise be hoisted out of the iteration, every row's at once.
        asm volatile("" : "+v"(i4));
        if (R < 4 || R < rows) {
            if (mine) {
                if constexpr (R < 4)
                    FullRow<MODE, ZT, R>(lam, tab, i4, zh4, core + AIRAN_BG1_ROW_START[R], inf_flag);
                else if constexpr (FULL)
                    FullRow<MODE, ZT, R>(lam, tab, i4, zh4, ext + (AIRAN_BG1_ROW_START[R] - AIRAN_BG1_ROW_START[4]),
                                         inf_flag);
                else
                    PackedRow<MODE, ZT, R>(lam, tab, i4, zh4, ext + 4 * (R - 4), inf_flag);
            }
            __syncthreads();
        }
        StaticRows<MODE, ZT, FULL, R + 1>(lam, tab, i4, zh4, mine, rows, core, ext, inf_flag);
    }
}

// Words of N rows' state, indexed by the (uniform) row.
template <int N>
struct RowState {
    typedef uint32_t vec __attribute__((ext_vector_type(N)));
    vec s1p, d12, meta;
};

// Rows r0 .. r0 + count - 1 of the loop.
template <int MODE, uint32_t ZT, int N>
__device__ __forceinline__ void LoopRows(uint32_t *lam, const uint32_t *tab, int r0, int count, bool mine, uint32_t i4,
                                         uint32_t zh4, RowState<N> &st, uint32_t *inf_flag)
{
    if (count <= 0) return;
    uint32_t info = kEdges.row[r0];
    uint32_t w[kMaxLoopDeg];
#pragma unroll
    for (int k = 0; k < kMaxLoopDeg; ++k) w[k] = TableWord<ZT>(tab, (info & 0xffffu) + k);
#pragma nounroll
    for (int j = 0; j < count; ++j) {
        // The next row's words, on their way while this row is worked on.
        const uint32_t ninfo = kEdges.row[r0 + j + 1];
        uint32_t nw[kMaxLoopDeg];
        const uint32_t ne0 = (info & 0xffffu) + (info >> 16);
#pragma unroll
        for (int k = 0; k < kMaxLoopDeg; ++k) nw[k] = TableWord<ZT>(tab, ne0 + k);
        if (mine) {
            uint32_t a = st.s1p[j], b = st.d12[j], c = st.meta[j];
            switch (info >> 16) {
            case 4: LoopRow<MODE, ZT, 4>(lam, w, i4, zh4, a, b, c, inf_flag); break;
            case 5: LoopRow<MODE, ZT, 5>(lam, w, i4, zh4, a, b, c, inf_flag); break;
            case 6: LoopRow<MODE, ZT, 6>(lam, w, i4, zh4, a, b, c, inf_flag); break;
            case 7: LoopRow<MODE, ZT, 7>(lam, w, i4, zh4, a, b, c, inf_flag); break;
            default: LoopRow<MODE, ZT, 8>(lam, w, i4, zh4, a, b, c, inf_flag); break;
            }
            st.s1p[j] = a;
            st.d12[j] = b;
            st.meta[j] = c;
        }
        __syncthreads();
        info = ninfo;
#pragma unroll
        for (int k = 0; k < kMaxLoopDeg; ++k) w[k] = nw[k];
    }
}

// Hard decisions per half as 0 / 1.  FP16: NegBit (negative, non-zero, not
// NaN).  REF: the reference's rint(clamp(v, +-5120)) < 0, which for an fp16
// posterior is v < -0.5 (a NaN gives 0), bits 0xb801 .. 0xfc00.
template <int MODE>
__device__ __forceinline__ uint32_t HardBits2(uint32_t v)
{
    if constexpr (MODE == AIRAN_LDPC_MODE_REF)
        return PkMinU16(PkSubSatU16(0x44004400u, PkSubU16(v, 0xb801b801u)), 0x00010001u);
    return NegBit2(v);
}

// Bit 0 / 16 set where check i / i + Z/2 of one of the rows [r0, r1) fails.
// FP16 without EXACT: the sign-bit XOR (no posterior is -0, and without an
// infinite or NaN extrinsic none is a NaN; see PairSyndrome).
template <int MODE, uint32_t ZT, bool EXACT>
__device__ __forceinline__ uint32_t TableSyndrome(uint32_t *lam, const uint32_t *tab, int r0, int r1, uint32_t i4,
                                                  uint32_t zh4)
{
    uint32_t bad = 0;
#pragma nounroll
    for (int r = r0; r < r1; ++r) {
        const uint32_t info = kEdges.row[r];
        const int deg = static_cast<int>(info >> 16);
        uint32_t p = 0;
#pragma unroll 4
        for (int k = 0; k < deg; ++k) {
            const EdgeAt a = TableEdge<ZT>(TableWord<ZT>(tab, (info & 0xffffu) + k), i4, zh4);
            const uint32_t v = Rot16(LdsWord(lam, a.byte), a.rot);
            p ^= EXACT || MODE == AIRAN_LDPC_MODE_REF ? HardBits2<MODE>(v) : (v >> 15);
        }
        bad |= p & 0x00010001u;
    }
    return bad;
}

template <int MODE, uint32_t ZT, int R, int RE>
__device__ __forceinline__ uint32_t StaticSyndrome(uint32_t *lam, uint32_t i4)
{
    uint32_t bad = 0;
    if constexpr (R < RE) {
        uint32_t p = 0;
        asm volatile("" : "+v"(i4));  // as in StaticRows
#pragma unroll
        for (int k = 0; k < StaticDeg(R); ++k) {
            if (k > 0 && k % 7 == 0) __builtin_amdgcn_sched_barrier(0);
            const EdgeAt a = StaticEdge<ZT>(AIRAN_BG1_ROW_START[R] + k, i4);
            const uint32_t v = Rot16(LdsWord(lam, a.byte), a.rot);
            p ^= MODE == AIRAN_LDPC_MODE_REF ? HardBits2<MODE>(v) << 15 : v;
        }
        bad = (p >> 15) & 0x00010001u;
        return bad | StaticSyndrome<MODE, ZT, R + 1, RE>(lam, i4);
    }
    return bad;
}

struct LdpcDev {
    uint32_t z, zi, k, iters, rows, early_stop;
};

// Posterior start value (fp16) of a decoder input LLR.
template <int MODE>
__device__ __forceinline__ uint32_t StartH(int32_t v)
{
    return MODE == AIRAN_LDPC_MODE_REF ? BitsH(static_cast<h16>(static_cast<float>(v))) : InputH(v);
}

// Half-word index in LDS of posterior position t.
__device__ __forceinline__ uint32_t HalfIndex(uint32_t t, uint32_t z, uint32_t zh)
{
    const uint32_t col = t / z, q = t - col * z;
    return q < zh ? 2u * (col * zh + q) : 2u * (col * zh + q - zh) + 1u;
}

// Loads a ragged block's posterior start values from its grant's bit-plane
// codeword LLRs: positions below nl, word j of a column = positions j and
// j + Z/2 (the rate-dematch arithmetic of ratematch.h).  Where every
// transmitted bit lands on its own position (RateSingle), the planes are read
// in aligned 16-byte chunks of 8 symbols and scattered (see PairLoad);
// otherwise each position gathers its LLRs.  Ends before the barrier that
// makes the posterior visible.  ONE: word t holds position t alone, gathered.
template <bool ONE>
__device__ inline void CheckLoadCodeword(uint32_t *lam, uint32_t z, uint32_t nl, const int16_t *__restrict__ cw,
                                         const airan::RateCb &rc, const airan::RateDev &r)
{
    const uint32_t i = threadIdx.x, nt = blockDim.x, zh = z / 2;
    uint16_t *lam16 = reinterpret_cast<uint16_t *>(lam);
    if constexpr (ONE) {
        for (uint32_t t = i; t < nl; t += nt) lam[t] = InputH(airan::RateDematchValue(t, rc, r, cw));
        return;
    }
    if (!airan::RateSingle(rc, r)) {
        for (uint32_t t = i; t < nl; t += nt)
            lam16[HalfIndex(t, z, zh)] = static_cast<uint16_t>(InputH(airan::RateDematchValue(t, rc, r, cw)));
        return;
    }
    const uint32_t two_z = 2u * z, fstart = r.kprime - two_z, nf = r.ncb - r.filler;
    const int16_t *slot = cw + static_cast<size_t>(rc.slot0) * r.qm * r.cw_stride;
    for (uint32_t t = i; t < nl / 2u; t += nt) lam[t] = 0;
    __syncthreads();
    for (uint32_t t = two_z + fstart + i; t < min(nl, two_z + fstart + r.filler); t += nt)
        lam16[HalfIndex(t, z, zh)] = static_cast<uint16_t>(InputH(5120));
    // Symbol j of plane b: its position.
    auto position = [&](uint32_t b, uint32_t j) {
        uint32_t q = rc.q0 + b * rc.eq + j;
        q = q >= nf ? q - nf : q;
        return two_z + (q < fstart ? q : q + r.filler);
    };
    auto put = [&](uint32_t b, uint32_t j, int32_t v) {
        const uint32_t t = position(b, j);
        if (t >= nl) return;
        v *= 8;
        v = v > 5120 ? 5120 : (v < -5120 ? -5120 : v);
        lam16[HalfIndex(t, z, zh)] = static_cast<uint16_t>(InputH(v));
    };
    // Chunks of 8 symbols at multiples of 8 of the slot's planes, the block's
    // symbols [rem0, rem0 + eq) of each plane inside them.
    const uint32_t c0 = rc.rem0 / 8u, nc = (rc.rem0 + rc.eq + 7u) / 8u - c0;
    for (uint32_t b = 0; b < r.qm; ++b) {
        const int16_t *plane = slot + static_cast<size_t>(b) * r.cw_stride;
        for (uint32_t e = i; e < nc; e += nt) {
            const uint32_t s0 = 8u * (c0 + e);
            const uint4 raw = *reinterpret_cast<const uint4 *>(plane + s0);
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
            const uint32_t j0 = s0 - rc.rem0;  // below zero (wrapped) in a first partial chunk
            const bool whole = s0 >= rc.rem0 && s0 + 8u <= rc.rem0 + rc.eq;
            const uint32_t q = whole ? rc.q0 + b * rc.eq + j0 : 0u, qn = q >= nf ? q - nf : q;
            const uint32_t t0 = two_z + (qn < fstart ? qn : qn + r.filler);
            const uint32_t half = t0 / zh, q0 = t0 - half * zh;  // runs of Z/2: even ones are low halves
            if (whole && qn + 8u <= nf && (qn >= fstart || qn + 8u <= fstart) && t0 + 8u <= nl && q0 + 8u <= zh) {
                const h2_t scale = {static_cast<_Float16>(1.0f / 32.0f), static_cast<_Float16>(1.0f / 32.0f)};
                uint16_t *dst = lam16 + 2u * ((half >> 1) * zh + q0) + (half & 1u);
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const uint32_t cl = PkMinI16(PkMaxI16(w[k], 0xfd80fd80u), 0x02800280u);
                    const uint32_t vb = WH(__builtin_convertvector(__builtin_bit_cast(s16x2, cl), h2_t) * scale);
                    dst[4u * k] = static_cast<uint16_t>(vb);
                    dst[4u * k + 2u] = static_cast<uint16_t>(vb >> 16);
                }
            } else {
#pragma unroll
                for (uint32_t x = 0; x < 8; ++x) {
                    const uint32_t sym = s0 + x;
                    if (sym >= rc.rem0 && sym < rc.rem0 + rc.eq)
                        put(b, sym - rc.rem0, static_cast<int16_t>(w[x >> 1] >> (16u * (x & 1u))));
                }
            }
        }
    }
}

constexpr uint32_t CheckThreads(uint32_t zt) { return zt == kAnyZ ? kMaxZ : zt == kZ96 ? 64 : kMaxZ / 2; }
// Words of a column's posterior.
constexpr uint32_t ColWords(uint32_t zt) { return zt == kZ96 ? 48 : CheckThreads(zt); }

// Where a block's LLRs come from: decoder LLRs [cb][68 Z] in src; or bit-plane
// codeword LLRs (the standalone rate-dematch arithmetic, no lam_out), of code
// block list[b] of a ragged batch with that block's Z, K and rows, or of block
// b of a chain's batch by its descriptor.
constexpr int kSrcLlr = 0, kSrcRagged = 1, kSrcChain = 2;

// MAXROWS: kFewRows or kRows.
template <int MODE, int MAXROWS, uint32_t ZT, int SRC>
__global__ void __launch_bounds__(CheckThreads(ZT)) __attribute__((amdgpu_waves_per_eu(MAXROWS <= kFewRows ? 3 : 2)))
    LdpcCheckPairKernel(const int16_t *__restrict__ src, int8_t *__restrict__ bits, int16_t *__restrict__ lam_out,
                        uint8_t *__restrict__ iters_out, LdpcDev d, const airan::RaggedCb *__restrict__ cbs,
                        const airan::RaggedGrant *__restrict__ grants, const uint32_t *__restrict__ list,
                        const RateMatchDescriptor *__restrict__ desc, airan::RateDev rate)
{
    constexpr bool RAGGED = SRC == kSrcRagged, kOne = ZT == kAnyZ;
    static_assert(!kOne || SRC != kSrcLlr, "no operator call reaches it");
    constexpr uint32_t kCheckThreads = CheckThreads(ZT);
    constexpr bool kFull = MAXROWS <= kFewRows;  // every message of rows 4 .. 9 kept
    constexpr int kCoreEdges = AIRAN_BG1_ROW_START[4];
    constexpr int kExtEdges = AIRAN_BG1_ROW_START[kStaticRows] - kCoreEdges;
    // The posterior, then the waves' syndrome votes (two words) and the flag
    // of an infinite or NaN extrinsic (sticky: it only selects the exact
    // syndrome).  One array, so that the posterior is at LDS address 0.
    constexpr uint32_t kTabWords = kOne ? AIRAN_BG1_EDGES + kMaxLoopDeg : 0;
    __shared__ __align__(16) uint32_t lam[(22 + MAXROWS) * ColWords(ZT) + 4 + kTabWords];
    uint32_t *vote = lam + (22 + MAXROWS) * ColWords(ZT), *inf_flag = vote + 2;
    const uint32_t i = threadIdx.x;
    uint32_t cb = blockIdx.x;
    size_t bits_off;
    if constexpr (RAGGED) {
        cb = list[blockIdx.x];
        const airan::RaggedCb &c = cbs[cb];
        d.z = c.z;
        d.k = c.k;
        d.rows = c.rows;
        if constexpr (!kOne) {
            d.zi = 0;
            while ((24u << d.zi) < d.z) ++d.zi;
        }
        bits_off = c.bits_off;
    } else {
        bits_off = static_cast<size_t>(cb) * d.k;
    }
    const uint32_t Z = ZT == kMaxZ ? ZT : d.z, zh = kOne ? Z : Z / 2, zh4 = 4u * zh;
    const int rows = static_cast<int>(d.rows);
    const uint32_t nl = (22u + d.rows) * Z;  // positions the active rows touch
    uint16_t *lam16 = reinterpret_cast<uint16_t *>(lam);
    if (i < 3) vote[i] = 0;
    if constexpr (kOne)
        for (uint32_t e = i; e < kTabWords; e += kCheckThreads) {
            const uint32_t s = e < AIRAN_BG1_EDGES ? AIRAN_BG1_SHIFT[e] % Z : 0u;
            vote[4 + e] = (e < AIRAN_BG1_EDGES ? AIRAN_BG1_COL[e] * Z + s : 0u) | (Z - s) << 16;
        }
    if constexpr (RAGGED) {
        const airan::RaggedCb &c = cbs[cb];
        const airan::RaggedGrant &gr = grants[c.grant];
        const airan::RateDev r{gr.g.qm, gr.g.cw_symbols, gr.g.cw_stride, Z, c.kprime, c.filler, c.ncb, 1};
        const airan::RateCb rc = airan::RateCbSetup({c.e, c.k0, c.ncb, c.cw_symbol_offset}, r);
        CheckLoadCodeword<kOne>(lam, Z, nl, src + gr.cw_off, rc, r);
    } else if constexpr (SRC == kSrcChain) {
        CheckLoadCodeword<kOne>(lam, Z, nl, src, airan::RateCbSetup(desc[cb], rate), rate);
    } else {
        const int16_t *s = src + static_cast<size_t>(cb) * 68u * Z;
        if ((reinterpret_cast<uintptr_t>(src) & 7u) == 0) {
            // Four words at a time: positions j .. j + 3 and their partners
            // (Z is a multiple of 24: runs of 4 never cross a half).
            const uint32_t per = zh / 4u, total = (22u + d.rows) * per;
            for (uint32_t t = i; t < total; t += kCheckThreads) {
                const uint32_t col = t / per, j = 4u * (t - col * per);
                const uint2 a = *reinterpret_cast<const uint2 *>(s + col * Z + j);
                const uint2 b = *reinterpret_cast<const uint2 *>(s + col * Z + zh + j);
                auto word = [&](uint32_t x, uint32_t y, uint32_t sh) {
                    return StartH<MODE>(static_cast<int16_t>(x >> sh)) |
                           StartH<MODE>(static_cast<int16_t>(y >> sh)) << 16;
                };
                *reinterpret_cast<uint4 *>(lam + col * zh + j) =
                    make_uint4(word(a.x, b.x, 0), word(a.x, b.x, 16), word(a.y, b.y, 0), word(a.y, b.y, 16));
            }
        } else {
            for (uint32_t t = i; t < nl; t += kCheckThreads)
                lam16[HalfIndex(t, Z, zh)] = static_cast<uint16_t>(StartH<MODE>(s[t]));
        }
    }
    const uint32_t *tab = kOne ? vote + 4 : kEdges.w[d.zi];
    uint32_t core[kCoreEdges];
#pragma unroll
    for (int e = 0; e < kCoreEdges; ++e) core[e] = 0;
    uint32_t ext[kFull ? kExtEdges : 4 * (kStaticRows - 4)];
#pragma unroll
    for (uint32_t &v : ext) v = 0;
    RowState<32> sa;  // rows kStaticRows .. + 31
    RowState<4> sb;   // and the last four
    static_assert(kStaticRows + 32 + 4 == kRows, "row states");
    sa.s1p = sa.d12 = sa.meta = 0;
    sb.s1p = sb.d12 = sb.meta = 0;
    __syncthreads();
    const bool mine = i < zh;
    uint32_t it = 0;
    while (it < d.iters) {
        uint32_t i4 = 4u * i;
        StaticRows<MODE, ZT, kFull, 0>(lam, tab, i4, zh4, mine, rows, core, ext, inf_flag);
        if constexpr (MAXROWS > kStaticRows) {
            LoopRows<MODE, ZT, 32>(lam, tab, kStaticRows, min(rows - kStaticRows, 32), mine, i4, zh4, sa, inf_flag);
            LoopRows<MODE, ZT, 4>(lam, tab, kStaticRows + 32, rows - kStaticRows - 32, mine, i4, zh4, sb, inf_flag);
        }
        ++it;
        if (d.early_stop) {
            // The core rows first: a block that has not converged nearly
            // always fails one of them.  Votes: a failing wave sets the word;
            // it is cleared below, before the barriers of the next iteration.
            const bool exact = MODE == AIRAN_LDPC_MODE_FP16 && *inf_flag != 0;
            uint32_t bad = 0;
            if (mine && !exact) {
                if constexpr (ZT == kMaxZ)
                    bad = StaticSyndrome<MODE, ZT, 0, 4>(lam, i4);
                else
                    bad = TableSyndrome<MODE, ZT, false>(lam, tab, 0, 4, i4, zh4);
            } else if (mine) {
                bad = TableSyndrome<MODE, ZT, true>(lam, tab, 0, 4, i4, zh4);
            }
            if (__ballot(bad != 0) != 0 && (i & 63u) == 0) vote[0] = 1u;
            __syncthreads();
            bool ok = vote[0] == 0;
            if (ok) {
                bad = 0;
                if (mine && !exact) {
                    if constexpr (ZT == kMaxZ && MAXROWS <= kFewRows) {
                        // Unrolled up to the few rows; a row beyond the
                        // block's is not read (its column is not loaded).
                        if (rows > 4) bad |= StaticSyndrome<MODE, ZT, 4, 5>(lam, i4);
                        if (rows > 5) bad |= StaticSyndrome<MODE, ZT, 5, 6>(lam, i4);
                        if (rows > 6) bad |= StaticSyndrome<MODE, ZT, 6, 7>(lam, i4);
                        if (rows > 7) bad |= StaticSyndrome<MODE, ZT, 7, 8>(lam, i4);
                        if (rows > 8) bad |= StaticSyndrome<MODE, ZT, 8, 9>(lam, i4);
                        if (rows > 9) bad |= StaticSyndrome<MODE, ZT, 9, 10>(lam, i4);
                    } else {
                        bad = TableSyndrome<MODE, ZT, false>(lam, tab, 4, rows, i4, zh4);
                    }
                } else if (mine) {
                    bad = TableSyndrome<MODE, ZT, true>(lam, tab, 4, rows, i4, zh4);
                }
                if (__ballot(bad != 0) != 0 && (i & 63u) == 0) vote[1] = 1u;
                __syncthreads();
                ok = vote[1] == 0;
            }
            if (ok) break;
            __syncthreads();
            if (i < 2) vote[i] = 0;
        }
    }
    // (every posterior is final: the last row and the votes ended in barriers)
    if (iters_out != nullptr && i == 0) iters_out[cb] = static_cast<uint8_t>(it);
    int8_t *bo = bits + bits_off;
    if (kOne) {
        for (uint32_t t = i; t < d.k; t += kCheckThreads) bo[t] = static_cast<int8_t>(HardBits2<MODE>(lam[t]) & 1u);
    } else if ((d.k & 3u) == 0 && (reinterpret_cast<uintptr_t>(bo) & 3u) == 0) {
        for (uint32_t t = 4u * i; t < d.k; t += 4u * kCheckThreads) {
            const uint32_t h = HalfIndex(t, Z, zh), sh = h & 1u;
            const uint4 v = *reinterpret_cast<const uint4 *>(lam + h / 2u);
            auto bit = [&](uint32_t x) { return (HardBits2<MODE>(x) >> (16u * sh)) & 1u; };
            *reinterpret_cast<uint32_t *>(bo + t) = bit(v.x) | bit(v.y) << 8 | bit(v.z) << 16 | bit(v.w) << 24;
        }
    } else {
        for (uint32_t t = i; t < d.k; t += kCheckThreads)
            bo[t] = static_cast<int8_t>(HardBits2<MODE>(lam16[HalfIndex(t, Z, zh)]) & 1u);
    }
    if (SRC == kSrcLlr && lam_out != nullptr) {
        const int16_t *s = src + static_cast<size_t>(cb) * 68u * Z;
        int16_t *lo = lam_out + static_cast<size_t>(cb) * 68u * Z;
        const float clip = MODE == AIRAN_LDPC_MODE_REF ? 5120.0f : 20.0f;
        const float out_scale = MODE == AIRAN_LDPC_MODE_REF ? 1.0f : 256.0f;
        for (uint32_t t = i; t < 68u * Z; t += kCheckThreads) {
            // Columns beyond the active rows keep their input.
            const uint32_t h = t < nl ? lam16[HalfIndex(t, Z, zh)] : StartH<MODE>(s[t]);
            float v = static_cast<float>(HBits(h));
            v = v > clip ? clip : (v < -clip ? -clip : v);
            lo[t] = static_cast<int16_t>(rintf(v * out_scale));
        }
    }
}

// Workgroups resident on the device at once for a pair-decoder launch shape
// (0 when the runtime cannot tell).
uint32_t PairCapacity(const void *kernel, uint32_t threads, size_t lds)
{
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, static_cast<int>(threads), lds) != hipSuccess)
        return 0;
    return static_cast<uint32_t>(std::max(cus, 0)) * static_cast<uint32_t>(std::max(per_cu, 0));
}

// Launches LdpcPairKernel<FUSED, rows, ZT> (rows 4 .. kFastRows); lds: the
// posterior's bytes (the shared words after it are added here; at Z = 384
// the kernel's LDS is static and none is allocated at launch).
template <bool FUSED>
void LaunchPair(uint32_t rows, uint32_t threads, size_t lds, hipStream_t s, const int16_t *src,
                const RateMatchDescriptor *desc, int8_t *bits, int16_t *lam_out, uint8_t *iters_out,
                const LdpcFastDev &d, uint32_t *queue)
{
    using Kern = void (*)(const int16_t *, const RateMatchDescriptor *, int8_t *, int16_t *, uint8_t *, LdpcFastDev,
                          uint32_t *);
    // Z = 384: edges folded at compile time (UsePair: 7 and 8 rows only).
    const bool z384 = d.z == 384;
    Kern k = rows <= 4 ? LdpcPairKernel<FUSED, 4, 0>
           : rows == 5 ? LdpcPairKernel<FUSED, 5, 0>
           : rows == 6 ? LdpcPairKernel<FUSED, 6, 0>
           : rows == 7 ? (z384 ? LdpcPairKernel<FUSED, 7, 384> : LdpcPairKernel<FUSED, 7, 0>)
                       : (z384 ? LdpcPairKernel<FUSED, 8, 384> : LdpcPairKernel<FUSED, 8, 0>);
    lds = z384 ? 0 : lds + kPairTailWords * sizeof(uint32_t);
    // One resident wave of workgroups, each walking its list of blocks.
    uint32_t grid = (d.num_cb + 1u) / 2u;
    const uint32_t cap = PairCapacity(reinterpret_cast<const void *>(k), threads, lds);
    if (cap > 0) grid = std::min(grid, cap);
    hipLaunchKernelGGL(k, dim3(grid), dim3(threads), lds, s, src, desc, bits, lam_out, iters_out, d, queue);
}

bool FastEligible(uint32_t mode, uint32_t z, uint32_t rows)
{
    return mode == AIRAN_LDPC_MODE_FP16 && rows <= static_cast<uint32_t>(kFastRows) && z >= 24 && z <= 384;
}

// FP16 messages, at most kFastRows rows: two blocks a workgroup (the pair
// decoder) or one block with two checks a lane (LdpcCheckPairKernel).
// Z < 384: the pair, whose lanes are all at work where a check pair's Z / 2 are
// few (8 iterations, pair / check pair: 2048 blocks of Z = 96, 6 rows 81 / 88 us,
// 4000 of Z = 24, 8 rows 81 / 178).  Z = 384: the check pair, whose blocks take and
// leave a compute unit one by one: us without early stop, pair / check pair,
//   rows   128 blocks  600      4000      (8 iterations, launch included)
//    4      61 / 52     90 / 81   -
//    6      72 / 59    105 / 93   -
//    8      81 / 70    156 / 110  635 / 435
// and with early stop ahead at every count (8 rows, 300 blocks: 54 / 51).
// The exception is between one and two blocks a compute unit with every
// iteration run, where the pair's one workgroup a unit is the shorter of two
// equal waits (7 rows, 300 blocks: 75 / 79; 8 rows 82 / 85; 6 rows 73 / 71).
bool UsePair(uint32_t z, uint32_t rows, uint32_t num_cb, bool early_stop)
{
    if (z != 384) return true;
    if (early_stop || rows < 7) return false;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return false;
    const uint32_t n = static_cast<uint32_t>(std::max(cus, 0));
    return num_cb > n && num_cb <= 2u * n;
}

uint32_t LiftIndex(uint32_t z)
{
    uint32_t zi = 0;
    while ((24u << zi) < z) ++zi;
    return zi;
}

// Check pair decoder, Z <= 96: one wave and the LDS of Z = 96 per block, where
// the blocks outnumber what is resident with 192 lanes each (registers allow 2
// workgroups of 3 waves a compute unit, 4 up to kFewRows rows; below that the
// idle lanes only help to load).  4000 blocks, 8 iterations at most, Z = 24 /
// 48 / 96: 46 rows, FP16 484 / 483 / 500 us against 1599 / 1436 / 1491 with 192
// lanes and the LDS of 384, REF 746 / 647 / 668 against 2069 / 1849 / 1909; 9
// rows, FP16 207 / 187 / 199 against 359 / 333 / 357.  1200 blocks of Z = 48: 46
// rows 261 / 537, 9 rows 120 / 154.
bool SmallBlocks(uint32_t z, uint32_t num_cb, bool few)
{
    int dev = 0, cus = 0;
    if (z > 96 || hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return false;
    return num_cb > static_cast<uint32_t>(std::max(cus, 0)) * (few ? 4u : 2u);
}

template <int MODE>
void LaunchCheckPair(const LdpcDecodeOpArgsV1 *a, hipStream_t s)
{
    const LdpcDev d{a->z, LiftIndex(a->z), a->k, a->max_iterations, a->active_rows, a->early_stop ? 1u : 0u};
    using Kern = void (*)(const int16_t *, int8_t *, int16_t *, uint8_t *, LdpcDev, const airan::RaggedCb *,
                          const airan::RaggedGrant *, const uint32_t *, const RateMatchDescriptor *, airan::RateDev);
    const bool few = a->active_rows <= static_cast<uint32_t>(kFewRows);
    const uint32_t zt = a->z == kMaxZ ? kMaxZ : SmallBlocks(a->z, a->num_cb, few) ? kZ96 : kLowZ;
    const Kern k = few ? (zt == kMaxZ   ? LdpcCheckPairKernel<MODE, kFewRows, kMaxZ, kSrcLlr>
                          : zt == kZ96  ? LdpcCheckPairKernel<MODE, kFewRows, kZ96, kSrcLlr>
                                        : LdpcCheckPairKernel<MODE, kFewRows, kLowZ, kSrcLlr>)
                       : (zt == kMaxZ   ? LdpcCheckPairKernel<MODE, kRows, kMaxZ, kSrcLlr>
                          : zt == kZ96  ? LdpcCheckPairKernel<MODE, kRows, kZ96, kSrcLlr>
                                        : LdpcCheckPairKernel<MODE, kRows, kLowZ, kSrcLlr>);
    hipLaunchKernelGGL(k, dim3(a->num_cb), dim3(CheckThreads(zt)), 0, s, static_cast<const int16_t *>(a->lam_in),
                       static_cast<int8_t *>(a->bits), static_cast<int16_t *>(a->lam_out),
                       static_cast<uint8_t *>(a->iterations_out), d, nullptr, nullptr, nullptr, nullptr,
                       airan::RateDev{});
}

// The decoder operator (validated arguments).
int32_t LaunchDecode(const LdpcDecodeOpArgsV1 *a)
{
    const int32_t st = LoadTables();
    if (st != AIRAN_OK) return st;
    hipStream_t s = static_cast<hipStream_t>(a->stream);
    const auto *in = static_cast<const int16_t *>(a->lam_in);
    auto *bits = static_cast<int8_t *>(a->bits);
    const bool aligned = (reinterpret_cast<uintptr_t>(in) & 7u) == 0 && (reinterpret_cast<uintptr_t>(bits) & 3u) == 0;
    if (aligned && FastEligible(a->mode, a->z, a->active_rows) &&
        UsePair(a->z, a->active_rows, a->num_cb, a->early_stop != 0)) {
        const uint32_t rows = a->active_rows;  // validated >= 4
        LdpcFastDev fd{a->z, LiftIndex(a->z), a->k, a->max_iterations, rows, a->early_stop ? 1u : 0u, a->num_cb, {}};
        const size_t fast_lds = static_cast<size_t>(22 + rows) * a->z * sizeof(uint32_t);
        LaunchPair<false>(rows, airan::AlignUp(a->z, 64), fast_lds, s, in, nullptr, bits,
                          static_cast<int16_t *>(a->lam_out), static_cast<uint8_t *>(a->iterations_out), fd, nullptr);
        return airan::LaunchStatus();
    }
    if (a->mode == AIRAN_LDPC_MODE_FP16)
        LaunchCheckPair<AIRAN_LDPC_MODE_FP16>(a, s);
    else
        LaunchCheckPair<AIRAN_LDPC_MODE_REF>(a, s);
    return airan::LaunchStatus();
}

// Largest workspace that airan_ldpc_decode_EnqueueNoAlloc stands in for (the
// reference's 143-block transport block at 46 rows, Z = 384: 20.2 MB).
constexpr size_t kNoAllocMaxBytes = size_t{32} << 20;

}  // namespace

extern "C" {

int32_t airan_ldpc_decode_ValidateOpArgs(const LdpcDecodeOpArgsV1 *a)
{
    if (!airan::HeaderOk(a, sizeof(LdpcDecodeOpArgsV1)) || a->lam_in == nullptr ||
        a->bits == nullptr || a->stream == nullptr || a->num_cb == 0)
        return AIRAN_INVALID_ARGUMENT;
    if (a->lam_in == a->bits || a->lam_in == a->lam_out || a->bits == a->lam_out)
        return AIRAN_INVALID_ARGUMENT;
    bool z_ok = false;
    for (uint32_t z = 3; z <= 384; z *= 2) z_ok |= a->z == z;
    if (!z_ok || a->z < 24) return AIRAN_UNSUPPORTED_PROFILE;
    if (a->k == 0 || a->k > 22 * a->z || a->max_iterations == 0 || a->max_iterations > 100 ||
        a->active_rows < 4 || a->active_rows > AIRAN_BG1_ROWS ||
        (a->mode != AIRAN_LDPC_MODE_REF && a->mode != AIRAN_LDPC_MODE_FP16) || a->num_cb > 1u << 20)
        return AIRAN_INVALID_ARGUMENT;
    return AIRAN_OK;
}

// The caller's part of the contract: a workspace of 8 bytes per (block, row,
// check) above kFastRows rows.  The decoder keeps its message state in
// registers and does not touch it.
size_t airan_ldpc_decode_WorkspaceBytes(uint32_t num_cb, uint32_t z, uint32_t active_rows)
{
    if (active_rows <= static_cast<uint32_t>(kFastRows)) return 0;
    return static_cast<size_t>(num_cb) * active_rows * z * sizeof(uint2);
}

size_t airan_ldpc_decode_NoAllocMaxWorkspaceBytes(void) { return kNoAllocMaxBytes; }

int32_t airan_ldpc_decode_EnqueueNoAlloc(const LdpcDecodeOpArgsV1 *a)
{
    const int32_t st = airan_ldpc_decode_ValidateOpArgs(a);
    if (st != AIRAN_OK) return st;
    if (airan_ldpc_decode_WorkspaceBytes(a->num_cb, a->z, a->active_rows) > kNoAllocMaxBytes)
        return AIRAN_RESOURCE_TOO_SMALL;
    return LaunchDecode(a);
}

int32_t airan_ldpc_decode_Enqueue(const LdpcDecodeOpArgsV1 *a, void *workspace, size_t workspace_bytes)
{
    const int32_t st = airan_ldpc_decode_ValidateOpArgs(a);
    if (st != AIRAN_OK) return st;
    const size_t need = airan_ldpc_decode_WorkspaceBytes(a->num_cb, a->z, a->active_rows);
    if (need > 0 && (workspace == nullptr || workspace_bytes < need)) return AIRAN_RESOURCE_TOO_SMALL;
    return LaunchDecode(a);
}

}  // extern "C"

namespace airan {

int32_t LaunchLdpcRagged(const RaggedCb *cbs, const RaggedGrant *grants, const RaggedLdpcList &many,
                         const RaggedLdpcList &few, const RaggedLdpcList &other, const RaggedLdpcList &any,
                         uint32_t iters, bool early_stop, const int16_t *cw, int8_t *bits, uint8_t *iters_out,
                         hipStream_t s)
{
    const int32_t st = LoadTables();
    if (st != AIRAN_OK) return st;
    const LdpcDev d{0, LiftIndex(384), 0, iters, 0, early_stop ? 1u : 0u};
    constexpr int kMode = AIRAN_LDPC_MODE_FP16;
    auto launch = [&](auto kernel, const RaggedLdpcList &l, uint32_t threads = CheckThreads(kMaxZ)) {
        if (l.count > 0)
            hipLaunchKernelGGL(kernel, dim3(l.count), dim3(threads), 0, s, cw, bits, nullptr, iters_out, d, cbs,
                               grants, l.list, nullptr, RateDev{});
    };
    launch(LdpcCheckPairKernel<kMode, kRows, 384, kSrcRagged>, many);
    launch(LdpcCheckPairKernel<kMode, kFewRows, 384, kSrcRagged>, few);
    launch(LdpcCheckPairKernel<kMode, kRows, kLowZ, kSrcRagged>, other);
    launch(LdpcCheckPairKernel<kMode, kRows, kAnyZ, kSrcRagged>, any, CheckThreads(kAnyZ));
    return LaunchStatus();
}

int32_t LaunchLdpc(const LdpcDecodeOpArgsV1 &a)
{
    const int32_t st = airan_ldpc_decode_ValidateOpArgs(&a);
    return st == AIRAN_OK ? LaunchDecode(&a) : st;
}

uint32_t LdpcFewRows() { return kFewRows; }

bool LdpcLiftSize(uint32_t z) { return IsLiftSize(z); }

int32_t InitLdpcTables()
{
    // So that a caller who ran airan_InitDevice launches nothing but the
    // decoder afterwards.
    return LoadTables();
}

int32_t LaunchLdpcFromCodeword(const Geom &g, const AiranTbPlanV1 &p, const RateMatchDescriptor *desc,
                               const int16_t *cw, uint32_t num_cb, uint32_t rows, uint32_t iters, bool early_stop,
                               int8_t *bits, uint8_t *iters_out, uint32_t *queue,
                               hipStream_t s)
{
    if (num_cb == 0 || !FastEligible(AIRAN_LDPC_MODE_FP16, p.Z, rows) || rows < 4 || iters == 0 || iters > 100 ||
        (p.Z % 24) != 0 || p.K == 0 || p.K > 22 * p.Z || p.Ncb <= p.filler || (reinterpret_cast<uintptr_t>(bits) & 3u) ||
        p.E_low >= (1u << 22) || p.E_high >= (1u << 22))
        return AIRAN_UNSUPPORTED_PROFILE;
    const int32_t st = LoadTables();
    if (st != AIRAN_OK) return st;
    const bool any = !IsLiftSize(p.Z);
    if (any || !UsePair(p.Z, rows, num_cb, early_stop)) {
        const LdpcDev d{p.Z, LiftIndex(p.Z), p.K, iters, rows, early_stop ? 1u : 0u};
        const RateDev r{g.qm, g.cw_symbols, g.cw_stride, p.Z, p.Kprime, p.filler, p.Ncb, num_cb};
        constexpr int kMode = AIRAN_LDPC_MODE_FP16;
        const auto k = any ? LdpcCheckPairKernel<kMode, kRows, kAnyZ, kSrcChain>
                           : LdpcCheckPairKernel<kMode, kFewRows, 384, kSrcChain>;
        hipLaunchKernelGGL(k, dim3(num_cb), dim3(CheckThreads(any ? kAnyZ : kMaxZ)), 0, s, cw, bits, nullptr, iters_out,
                           d, nullptr, nullptr, nullptr, desc, r);
        return LaunchStatus();
    }
    LdpcFastDev fd{p.Z, LiftIndex(p.Z), p.K, iters, rows, early_stop ? 1u : 0u, num_cb,
                   {g.qm, g.cw_symbols, g.cw_stride, p.Z, p.Kprime, p.filler, p.Ncb, num_cb}};
    const size_t lds = static_cast<size_t>(22 + rows) * p.Z * sizeof(uint32_t);
    LaunchPair<true>(rows, AlignUp(p.Z, 64), lds, s, cw, desc, bits, nullptr, iters_out, fd, queue);
    return LaunchStatus();
}

}  // namespace airan

extern "C" {

// Rows 0..3 always; extension row r >= 4 only when its parity column 22 + r
// holds a transmitted circular-buffer position.
uint32_t airan_ldpc_ActiveRows(const AiranTbPlanV1 *p)
{
    if (p == nullptr || p->Z == 0) return AIRAN_BG1_ROWS;
    const uint32_t nf = p->Ncb - p->filler;
    const uint32_t e_max = p->E_high > p->E_low ? p->E_high : p->E_low;
    if (p->k0 != 0 || e_max >= nf) return AIRAN_BG1_ROWS;
    const uint32_t fstart = p->Kprime - 2 * p->Z;
    const uint32_t last = e_max - 1;
    const uint32_t pos = last < fstart ? last : last + p->filler;
    const uint32_t col = (pos + 2 * p->Z) / p->Z;
    int rows = static_cast<int>(col) - 22 + 1;
    rows = rows < 4 ? 4 : (rows > AIRAN_BG1_ROWS ? AIRAN_BG1_ROWS : rows);
    return static_cast<uint32_t>(rows);
}

}  // extern "C"
