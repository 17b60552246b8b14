// Poseidon permutation over Goldilocks, width 12 (rate 8, capacity 4),
// 8 full rounds + 22 partial rounds, S-box x^7, and the Plonky2 sponge
// ("hash_or_noop" and two-to-one compression) used by okx/zeknox's
// PoseidonHasher (native/poseidon/poseidon.cu:771-780,834-838,
// native/poseidon/poseidon_permutation.cuh:83-134).
//
// One permutation per lane: the 12-element state lives in 24 VGPRs; MDS
// coefficients are immediates, round constants come from constant memory.
// Inside the permutation values are kept "relaxed" (any u64 congruent mod p)
// and canonicalised once at the digest, which keeps every Goldilocks
// multiplication at 4 v_mad_u64_u32 for the product plus 2 for the reduction.
#pragma once
#include "gl64.hpp"
#include "poseidon_gl_constants.h"

namespace zk {

struct PoseidonConsts {
    static constexpr u64 circ[12] = ZK_POSEIDON_MDS_CIRC;
    static constexpr u64 diag[12] = ZK_POSEIDON_MDS_DIAG;
};

// Round constants (30 rounds x 12, then 12 zeros so the last round's MDS can
// fold "the next round's constants" uniformly): scalar loads on the device.
#define ZK_RC_WITH_TAIL { ZK_POSEIDON_RC_TABLE_BODY 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 }
static __constant__ const u64 kRoundConstDev[372] = ZK_RC_WITH_TAIL;
static const u64 kRoundConstHost[372] = ZK_RC_WITH_TAIL;

ZK_HD const u64 *round_constants()
{
#ifdef __HIP_DEVICE_COMPILE__
    return kRoundConstDev;
#else
    return kRoundConstHost;
#endif
}

// x^7 = x^3 * x^4 with relaxed (any u64) operands and result.  The squares
// use the general product: the three-product square (gl_sqr_nc) issues fewer
// instructions but its carry chain measured 1.27x slower per square on gfx950.
ZK_HD u64 sbox7(u64 x, bool &rare)
{
    const u64 x2 = gl_mul_nc<true>(x, x, rare);
    const u64 x4 = gl_mul_nc<true>(x2, x2, rare);
    const u64 x3 = gl_mul_nc<true>(x, x2, rare);
    return gl_mul_nc<true>(x3, x4, rare);
}

// a + 2^32 b mod p (relaxed) for a, b < 2^42: with b = b0 + 2^32 b1,
// a + 2^32 b == (a + b1 (2^32 - 1)) + 2^32 b0.  The first sum stays below
// 2^43 (one multiply-add), adding 2^32 b0 wraps past 2^64 at most once and
// the wrap is worth 2^32 - 1, which cannot wrap again (the wrapped value is
// below 2^43).
ZK_HD u64 reduce_lohi42(u64 a, u64 b)
{
    const u64 t = (u64)(u32)(b >> 32) * ZK_EPS + a;
    unsigned c;
    const u32 hi = __builtin_addc((u32)(t >> 32), (u32)b, 0u, &c);
    const u64 r = ((u64)hi << 32) | (u32)t;
    return r + (c ? ZK_EPS : 0);
}

// The same sum with the wrap entered as a borrow of the low word (the rare
// case when it goes below zero) and a carry of the high word: no mask to
// select, no zero-extended pair to build (4 instructions instead of 7).
ZK_HD u64 reduce_lohi42_nc(u64 a, u64 b, bool &rare)
{
    const u64 t = (u64)(u32)(b >> 32) * ZK_EPS + a;
    unsigned c, r;
    const u32 hi = __builtin_addc((u32)(t >> 32), (u32)b, 0u, &c);
    const u32 lo = __builtin_subc((u32)t, opaque_zero(), c, &r);
    rare |= r != 0;
    return ((u64)(hi + c) << 32) | lo;
}

// The same for a, b < 2^64 - 2^32: the multiply-add can wrap too, to at most
// 2^64 - 2^33; each wrap is worth 2^32 - 1 and both enter as above.
ZK_HD u64 reduce_lohi64(u64 a, u64 b, bool &rare)
{
    u64 t;
#ifdef __HIP_DEVICE_COMPILE__
    u64 k;  // carry-out of the multiply-add, as gl_reduce_small_mad_nc
    asm("v_mad_u64_u32 %0, %1, %2, -1, %3\n\ts_nop 1" : "=v"(t), "=s"(k) : "v"((u32)(b >> 32)), "v"(a));
    const bool c1 = __builtin_amdgcn_inverse_ballot_w64(k);
#else
    const bool c1 = __builtin_add_overflow((u64)(u32)(b >> 32) * ZK_EPS, a, &t);
#endif
    unsigned c2, r1, r2;
    const u32 hi = __builtin_addc((u32)(t >> 32), (u32)b, (unsigned)c1, &c2);
    u32 lo = __builtin_subc((u32)t, opaque_zero(), (unsigned)c1, &r1);
    lo = __builtin_subc(lo, opaque_zero(), c2, &r2);
    rare |= (r1 | r2) != 0;
    return ((u64)(hi + c2) << 32) | lo;
}

// The same with no rare case, the wraps entered as selected 2^32 - 1: three
// instructions more, but none waits for a carry of the one before it.  Faster
// where a wave runs alone (16 lanes per permutation: 7.17 -> 6.82 us), slower
// at four waves per SIMD.
ZK_HD u64 reduce_lohi64_exact(u64 a, u64 b)
{
    const u64 t = gl_reduce_small_mad_nc(a, (u32)(b >> 32));
    unsigned c;
    const u32 hi = __builtin_addc((u32)(t >> 32), (u32)b, 0u, &c);
    const u64 r = ((u64)hi << 32) | (u32)t;
    return r + (c ? ZK_EPS : 0);
}

// state <- M state + rcn (the next round's constants), M circulant (first row
// circ) plus diag.  Row r is rcn[r] + sum of 13 products of a state element
// with a constant below 2^6: the low and high 32-bit halves are accumulated
// separately (the sums start at the constant's halves and stay below 2^42),
// then reduced once by reduce_lohi42_nc.  Inputs and outputs
// are relaxed (any u64).  The coefficients come from mds_coeff:
//
// the MDS coefficients as multiplier operands.  The powers of two among them
// (16 and 2) are passed through an opaque scalar register on the device: as
// literals the compiler turns c * x into a 64-bit shift of x, which first
// needs x zero-extended into a register pair (two moves) and so costs more
// than the multiply-add it replaces.
ZK_HD u32 mds_coeff(int i)
{
    const u32 c = (u32)PoseidonConsts::circ[i];
#ifdef __HIP_DEVICE_COMPILE__
    if ((c & (c - 1)) == 0) {
        u32 r;
        asm("s_mov_b32 %0, %1" : "=s"(r) : "i"(c));
        return r;
    }
#endif
    return c;
}

// `need` (uniform across the wave): bit q set when rows 4q .. 4q + 3 are
// wanted; the others are left unspecified.
ZK_HD void mds_fold(u64 s[12], const u64 *rcn, u32 need, bool &rare)
{
    u32 lo[12], hi[12];
#pragma unroll
    for (int j = 0; j < 12; j++) {
        lo[j] = (u32)s[j];
        hi[j] = (u32)(s[j] >> 32);
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
        if (!(need >> q & 1)) continue;
#pragma unroll
        for (int r = 4 * q; r < 4 * q + 4; r++) {
            const u64 k = rcn[r];
            u64 a = (u32)k, b = k >> 32;
#pragma unroll
            for (int i = 0; i < 12; i++) {
                const u64 c = i == 0 ? PoseidonConsts::circ[0] + PoseidonConsts::diag[r] : mds_coeff(i);
                a += c * lo[(i + r) % 12];
                b += c * hi[(i + r) % 12];
            }
            s[r] = reduce_lohi42_nc(a, b, rare);
        }
    }
}

ZK_HD void full_round(u64 s[12], const u64 *rcn, u32 need, bool &rare)
{
#pragma unroll
    for (int i = 0; i < 12; i++) s[i] = sbox7(s[i], rare);
    mds_fold(s, rcn, need, rare);
}

constexpr u32 kAllRows = 7;

// ---- partial rounds in blocks ---------------------------------------------
// Between two S-boxes of a partial round only element 0 is not linear, so K
// consecutive linear layers need not be applied one by one.  A block takes the
// state y[0..12) after an S-box layer, and with M the MDS matrix, Z the
// projection that clears element 0 and y_i the S-box output of the block's
// i-th inner round, the state after its j-th layer is
//   s_j = (M Z)^(j-1) M y + sum_{i<j} (M Z)^(j-1-i) M e0 y_i,
// a combination of 12 + j - 1 known values with non-negative coefficients.
// Element 0 of s_1 .. s_(K-1) is all the inner S-boxes need; the other eleven
// elements are formed once, for s_K.
template <int K>
struct PartialBlock {
    static constexpr int IN = 12 + K - 1;  // y[0..12), then y_1 .. y_(K-1)
    u64 v[K][IN];                          // row 0 of s_(j+1), j < K - 1
    u64 f[12][IN];                         // s_K
};

template <int K>
__host__ __device__ constexpr PartialBlock<K> make_partial_block()
{
    PartialBlock<K> t{};
    constexpr int IN = PartialBlock<K>::IN;
    u64 s[12][IN] = {};  // s_0: y itself
    for (int i = 0; i < 12; i++) s[i][i] = 1;
    for (int j = 0; j < K; j++) {
        if (j)  // element 0 is replaced by the inner S-box output y_j
            for (int c = 0; c < IN; c++) s[0][c] = c == 12 + j - 1;
        u64 n[12][IN] = {};
        for (int r = 0; r < 12; r++)
            for (int i = 0; i < 12; i++) {
                const u64 m = PoseidonConsts::circ[i] + (i == 0 ? PoseidonConsts::diag[r] : 0);
                for (int c = 0; c < IN; c++) n[r][c] += m * s[(i + r) % 12][c];
            }
        for (int r = 0; r < 12; r++)
            for (int c = 0; c < IN; c++) s[r][c] = n[r][c];
        for (int c = 0; c < IN; c++) t.v[j][c] = s[0][c];
    }
    for (int r = 0; r < 12; r++)
        for (int c = 0; c < IN; c++) t.f[r][c] = s[r][c];
    return t;
}

// The round constants with those of elements 1 .. 11 in the partial rounds
// moved through the linear layers: rows 4 .. 25 keep only element 0, what is
// left joins row 26.  Row 30 (zeros) follows the last round.
struct FoldedConsts {
    u64 rc[31 * 12];
};

__host__ __device__ constexpr FoldedConsts make_folded_consts()
{
    constexpr u64 rc[360] = ZK_POSEIDON_RC_TABLE;
    FoldedConsts t{};
    for (int i = 0; i < 360; i++)
        if (i < 60 || i >= 12 * 27) t.rc[i] = rc[i];
    u64 e[12] = {};
    for (int i = 0; i < 12; i++) e[i] = rc[48 + i];
    for (int r = 4; r < 26; r++) {
        t.rc[12 * r] = e[0];
        for (int i = 1; i < 12; i++) t.rc[12 * r + i] = 0;
        e[0] = 0;
        u64 n[12] = {};
        for (int row = 0; row < 12; row++) {
            unsigned __int128 acc = rc[12 * (r + 1) + row];
            for (int i = 0; i < 12; i++)
                acc += (unsigned __int128)(PoseidonConsts::circ[i] + (i == 0 ? PoseidonConsts::diag[row] : 0)) *
                       e[(i + row) % 12];
            n[row] = (u64)(acc % ZK_P);
        }
        for (int i = 0; i < 12; i++) e[i] = n[i];
    }
    for (int i = 0; i < 12; i++) t.rc[12 * 26 + i] = e[i];
    return t;
}

static __constant__ const FoldedConsts kFoldedConstDev = make_folded_consts();
static const FoldedConsts kFoldedConstHost = make_folded_consts();

ZK_HD const u64 *folded_constants()
{
#ifdef __HIP_DEVICE_COMPILE__
    return kFoldedConstDev.rc;
#else
    return kFoldedConstHost.rc;
#endif
}

// x^7 of a value that neighbouring lanes (l and l ^ 1) both hold, in three
// products instead of four: the even lane forms x^2 x, the odd one x^2 x^2,
// and both multiply their own by the other's (swap(r) is the neighbour's r).
template <typename Swap>
ZK_HD u64 sbox7_pair(u64 x, bool odd, Swap swap, bool &rare)
{
    const u64 x2 = gl_mul_nc<true>(x, x, rare);
    const u64 r = gl_mul_nc<true>(x2, odd ? x2 : x, rare);
    return gl_mul_nc<true>(r, swap(r), rare);
}

// The neighbouring lane's value (DPP quad_perm 1, 0, 3, 2).
struct LaneSwap {
    ZK_HD u64 operator()(u64 x) const
    {
#ifdef __HIP_DEVICE_COMPILE__
        const u32 lo = (u32)__builtin_amdgcn_mov_dpp((int)(u32)x, 0xB1, 0xF, 0xF, false);
        const u32 hi = (u32)__builtin_amdgcn_mov_dpp((int)(u32)(x >> 32), 0xB1, 0xF, 0xF, false);
        return ((u64)hi << 32) | lo;
#else
        return x;  // device-only; a host emulation passes its own
#endif
    }
};

// A coefficient as a multiplier operand: small ones are instruction
// immediates, the others scalar registers; powers of two are hidden from the
// compiler (see mds_coeff).
template <u64 C>
ZK_HD u32 block_coeff()
{
    static_assert(C < (1ull << 32), "coefficient exceeds 32 bits");
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (C > 1 && (C & (C - 1)) == 0) {
        u32 r;
        asm("s_mov_b32 %0, %1" : "=s"(r) : "i"((u32)C));
        return r;
    }
#endif
    return (u32)C;
}

// One block: s is the state after an S-box layer; k (folded constants) row j
// holds the constant of element 0 after layer j.  Returns the state before
// the next S-box.
template <int K>
ZK_HD void partial_block(u64 s[12], const u64 *k, bool &rare)
{
    using T = PartialBlock<K>;
    u32 lo[T::IN], hi[T::IN];
#pragma unroll
    for (int i = 0; i < 12; i++) {
        lo[i] = (u32)s[i];
        hi[i] = (u32)(s[i] >> 32);
    }
    static_for<0, K - 1>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        u64 a = (u32)k[12 * j], b = k[12 * j] >> 32;
        static_for<0, 12 + j>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            constexpr PartialBlock<K> tab = make_partial_block<K>();
            a += (u64)block_coeff<tab.v[j][c]>() * lo[c];
            b += (u64)block_coeff<tab.v[j][c]>() * hi[c];
        });
        const u64 y = sbox7(reduce_lohi64(a, b, rare), rare);
        lo[12 + j] = (u32)y;
        hi[12 + j] = (u32)(y >> 32);
    });
    static_for<0, 12>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        u64 a = r ? 0 : (u32)k[12 * (K - 1)], b = r ? 0 : k[12 * (K - 1)] >> 32;
        static_for<0, T::IN>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            constexpr PartialBlock<K> tab = make_partial_block<K>();
            a += (u64)block_coeff<tab.f[r][c]>() * lo[c];
            b += (u64)block_coeff<tab.f[r][c]>() * hi[c];
        });
        s[r] = reduce_lohi64(a, b, rare);
    });
}

// Layers per block.  The rate of the permutation alone with blocks of 1 (one
// layer at a time), 2, 3 and 4 layers on an MI355X: 2.29, 2.91, 3.18 and
// 3.26 G/s (68.8 k, 54.0 k, 49.5 k and 48.3 k SIMD-cycles per wave).  Five
// layers would need coefficients of 37 bits, i.e. two multiply-adds more per
// product; four reach 2^28.3, with rows whose sum is below 2^31.8, so the
// 32-bit halves' sums stay below 2^63.8.
constexpr int kBlock = 4;
constexpr int kBlock0 = 3;               // layers of the first block: those of rounds 3, 4, 5
constexpr int kBlocks = (23 - kBlock0) / kBlock;  // the others': from round kBlockStart on
constexpr int kBlockStart = 3 + kBlock0;
static_assert(kBlock0 + kBlocks * kBlock == 23, "the layers of rounds 3 .. 25");

// 4 full rounds, 22 partial rounds (S-box on element 0), 4 full rounds; the
// constants of rounds 1 .. 3 and 27 .. 29 are added by the layer before
// (round 0's explicitly).  The layer of the fourth full round opens the first
// block.  The loops are not unrolled, so the whole permutation stays resident
// in the instruction cache.  Input: relaxed; output: relaxed (canonicalise
// with gl_canon), only the rows of `need` (mds_fold).
ZK_HD void poseidon_permute(u64 s[12], bool &rare, u32 need = kAllRows)
{
    const u64 *rc = folded_constants();
#pragma unroll
    for (int i = 0; i < 12; i++) s[i] = gl_add_nc(s[i], rc[i], rare);
#pragma unroll 1
    for (int r = 0; r < 3; r++) full_round(s, rc + 12 * (r + 1), kAllRows, rare);
#pragma unroll
    for (int i = 0; i < 12; i++) s[i] = sbox7(s[i], rare);
    partial_block<kBlock0>(s, rc + 12 * 4, rare);
#pragma unroll 1
    for (int b = 0; b < kBlocks; b++) {
        s[0] = sbox7(s[0], rare);
        partial_block<kBlock>(s, rc + 12 * (4 + kBlock0 + kBlock * b), rare);
    }
#pragma unroll
    for (int i = 1; i < 12; i++) s[i] = gl_add_nc(s[i], rc[12 * 26 + i], rare);
#pragma unroll 1
    for (int r = 26; r < 30; r++) full_round(s, rc + 12 * (r + 1), r < 29 ? kAllRows : need, rare);
}

// Coefficient rows of the lane-parallel forms (poseidon_quad.hpp,
// poseidon_hex.hpp).  block: rows 0 .. 11 the elements after a block of kBlock
// layers, rows 12 .. 14 element 0 after its first three; columns the 15
// inputs.  mds: row r of one layer (rows 12 .. 15 repeat 0 .. 3).
struct LaneRows {
    u32 block[16][16], mds[16][12];
};

__host__ __device__ constexpr LaneRows make_lane_rows()
{
    constexpr PartialBlock<kBlock> t = make_partial_block<kBlock>();
    constexpr PartialBlock<1> m = make_partial_block<1>();
    static_assert(kBlock == 4, "three inner rows, 15 inputs");
    LaneRows l{};
    for (int c = 0; c < 15; c++) {
        for (int r = 0; r < 12; r++) l.block[r][c] = (u32)t.f[r][c];
        for (int j = 0; j < 3; j++) l.block[12 + j][c] = (u32)t.v[j][c];
    }
    for (int r = 0; r < 16; r++)
        for (int c = 0; c < 12; c++) l.mds[r][c] = (u32)m.f[r % 12][c];
    return l;
}

static __constant__ const LaneRows kLaneRowsDev = make_lane_rows();
static const LaneRows kLaneRowsHost = make_lane_rows();

ZK_HD const LaneRows &lane_rows()
{
#ifdef __HIP_DEVICE_COMPILE__
    return kLaneRowsDev;
#else
    return kLaneRowsHost;
#endif
}

// sum_i c[i] t[i] for i in [FIRST, 12) on top of (a, b), by 32-bit halves.
template <int FIRST>
ZK_HD void row_sum(const u32 *c, const u64 t[12], u64 &a, u64 &b)
{
#pragma unroll
    for (int i = FIRST; i < 12; i++) {
        a += (u64)c[i] * (u32)t[i];
        b += (u64)c[i] * (u32)(t[i] >> 32);
    }
}

ZK_HD void row_add(u32 c, u64 y, u64 &a, u64 &b)
{
    a += (u64)c * (u32)y;
    b += (u64)c * (u32)(y >> 32);
}

// The same permutation with canonical arithmetic only (no rare cases): the
// recomputation path when a relaxed permutation reported a rare case.
ZK_HD void poseidon_permute_safe(u64 s[12])
{
    const u64 *rc = round_constants();
#pragma unroll 1
    for (int r = 0; r < 30; r++) {
        const bool full = r < 4 || r >= 26;
#pragma unroll
        for (int i = 0; i < 12; i++) s[i] = gl_add(gl_canon(s[i]), rc[12 * r + i]);
#pragma unroll
        for (int i = 0; i < 12; i++) {
            if (full || i == 0) {
                const u64 x2 = gl_mul(s[i], s[i]), x4 = gl_mul(x2, x2);
                s[i] = gl_mul(gl_mul(s[i], x2), x4);
            }
        }
        u64 o[12];
#pragma unroll
        for (int row = 0; row < 12; row++) {
            u64 lo = 0, hi = 0;
#pragma unroll
            for (int i = 0; i < 12; i++) {
                const u64 c = PoseidonConsts::circ[i] + (i == 0 ? PoseidonConsts::diag[row] : 0);
                u64 pl, ph;
                gl_mul_wide(s[(i + row) % 12], c, pl, ph);
                lo += pl;
                hi += ph + (lo < pl ? 1 : 0);
            }
            o[row] = gl_reduce128(lo, hi);
        }
#pragma unroll
        for (int i = 0; i < 12; i++) s[i] = o[i];
    }
}

// The relaxed permutation as the sponges take it: perm(state, rare, rows
// wanted).  (MfmaPermute in poseidon_mfma.hpp is the other.)
struct PlainPermute {
    ZK_HD void operator()(u64 s[12], bool &rare, u32 need) const { poseidon_permute(s, rare, need); }
};

// Two-to-one compression: state = [a, b, 0, 0, 0, 0] -> permute -> state[0..4).
template <typename Perm = PlainPermute>
ZK_HD void hash_two(const u64 a[4], const u64 b[4], u64 out[4], const Perm &perm = Perm())
{
    u64 s[12];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        s[i] = a[i];
        s[4 + i] = b[i];
        s[8 + i] = 0;
    }
    bool rare = false;
    perm(s, rare, 1u);  // the digest is rows 0 .. 3
    if (rare) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] = a[i];
            s[4 + i] = b[i];
            s[8 + i] = 0;
        }
        poseidon_permute_safe(s);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = gl_canon(s[i]);
}

// The rows of the state that are read after a sponge's permutation with `rem`
// elements left before it: the digest after the last, else the capacity and
// the rate elements that the next chunk does not overwrite.
ZK_HD u32 sponge_rows(u32 rem)
{
    if (rem <= 8) return 1u;
    const u32 m = rem - 8;  // elements of the next chunk and after
    return 4u | (m < 8 ? 2u : 0u) | (m < 4 ? 1u : 0u);
}

// hash_or_noop over n elements fetched by `get(i)`: n <= 4 copies the input,
// zero-padded; otherwise the overwrite-mode sponge (a final short chunk leaves
// the stale rate lanes in place), digest = state[0..4).  `chunk(idx, m, v)` sees
// each chunk of input once, right after it is fetched: elements idx .. idx+m-1
// in v[0..m) (the exact recompute of a rare case fetches again, unseen).  Rare
// cases are redone at once, one permutation: redoing the whole sponge at its
// end kept one wave busy for another 17 permutations of a 135-element leaf,
// 0.1 to 0.4 ms of a 5.7 ms launch of 2^20 leaves in every third one.
template <typename Get, typename Chunk, typename Perm = PlainPermute>
ZK_HD void hash_one_chunks(Get get, u32 n, u64 out[4], Chunk chunk, const Perm &perm = Perm())
{
    if (n <= 4) {
#pragma unroll
        for (u32 i = 0; i < 4; i++) out[i] = i < n ? get(i) : 0;
        chunk(0u, n, (const u64 *)out);
        return;
    }
    u64 s[12];
#pragma unroll
    for (int i = 0; i < 12; i++) s[i] = 0;
    for (u32 idx = 0; idx < n; idx += 8) {
        const u32 rem = n - idx;
#pragma unroll
        for (u32 i = 0; i < 8; i++)
            if (i < rem) s[i] = get(idx + i);
        chunk(idx, rem < 8 ? rem : 8u, (const u64 *)s);
        u64 cap[4];
#pragma unroll
        for (int i = 0; i < 4; i++) cap[i] = s[8 + i];
        bool rare = false;
        perm(s, rare, sponge_rows(rem));
        if (rare) {
            // This lane hit a rare relaxed case: redo the permutation exactly
            // from its inputs, the chunk (fetched again) and the capacity; a
            // short chunk leaves rate elements of the state before it in
            // place, which are not kept, so there the sponge is redone.
            const u32 from = rem < 8 ? 0 : idx;
#pragma unroll
            for (int i = 0; i < 12; i++) s[i] = from && i >= 8 ? cap[i - 8] : 0;
            for (u32 k = from; k <= idx; k += 8) {
#pragma unroll
                for (u32 i = 0; i < 8; i++)
                    if (i < n - k) s[i] = get(k + i);
                poseidon_permute_safe(s);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = gl_canon(s[i]);
}

template <typename Get, typename Perm = PlainPermute>
ZK_HD void hash_one(Get get, u32 n, u64 out[4], const Perm &perm = Perm())
{
    hash_one_chunks(get, n, out, [](u32, u32, const u64 *) {}, perm);
}

}  // namespace zk
