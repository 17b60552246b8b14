// Poseidon permutation, one per lane, with the linear layers of its full
// rounds on the matrix cores: same function as poseidon_permute.
//
// A layer's 144 products of a 64-bit state element with a constant below 2^6
// are eight times as many of its bytes, exact in the i32 sums of an i8 MFMA.
// v_mfma_i32_32x32x32_i8 takes 16 bytes of B from a lane (column lane % 32, k
// half lane / 32) and gives it 16 of the 32 rows of that column; with a row of
// A nonzero only in the k half of the lanes that receive the row, every lane
// gets its own 16 x 16 matrix times its own 16 bytes, so the states need no
// exchange between lanes.  The 16 bytes are the low (high) halves of four
// state elements, the 16 rows the four bytes' sums of four output elements
// (the matrix is block-diagonal in the byte index): 18 MFMAs a layer.  Half
// of A is zero, and of the rest three quarters, but the matrix cores are
// otherwise idle; the alternative, a byte transpose of the state, costs as
// much VALU time as it saves in MFMAs.
//
// Bytes enter as signed (x ^ 0x80), i.e. 128 too small; 128 times the row sum
// is part of the constants that start the recombination of a row's byte sums
// s_0 + 2^8 s_1 + 2^16 s_2 + 2^24 s_3 for either half.
//
// An MFMA is not free beside VALU work of other waves (a 32x32x32 costs them
// about 20 cycles, alone it takes 32 to 44), so a layer falls from about 1490
// to 1130 SIMD-cycles: the permutation alone 46.2 k -> 43.8 k, leaf hashing of
// 2^20 rows of 135 elements 5.83 -> 5.60 ms.  In the blocks of the partial
// rounds the coefficients are four bytes wide and 48 MFMAs would replace 360
// multiply-adds, with no gain.
#pragma once
#include "poseidon.hpp"

namespace zk {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Starting values of a row's two 64-bit sums after each full round's layer:
// the halves of the next round's constant plus the bias of the signed bytes.
struct MfmaConsts {
    u64 k[31 * 12][2];
};

__host__ __device__ constexpr MfmaConsts make_mfma_consts()
{
    const FoldedConsts f = make_folded_consts();
    MfmaConsts m{};
    u64 sum = 0;
    for (int i = 0; i < 12; i++) sum += PoseidonConsts::circ[i];
    for (int i = 0; i < 31 * 12; i++) {
        const u64 bias = (sum + PoseidonConsts::diag[i % 12]) * 0x80808080ull;
        m.k[i][0] = (u32)f.rc[i] + bias;
        m.k[i][1] = (f.rc[i] >> 32) + bias;
    }
    return m;
}

static __constant__ const MfmaConsts kMfmaConstDev = make_mfma_consts();

// This lane's part of A: block (R, Q) of the layer's matrix (output elements
// 4R .. 4R+3, input elements 4Q .. 4Q+3) is w[(Q - R) mod 3], the matrix being
// circulant, but w[3] for block (0, 0) with its diagonal entry.  Word j of
// the row (element e, byte b) holds the coefficient of input 4Q + j at byte b.
struct MfmaTiles {
    v4i w[4];
};

ZK_HD void mfma_tiles(u32 lane, MfmaTiles &t)
{
    const LaneRows &l = lane_rows();
    const u32 m = lane & 31, e = m >> 3, b = m & 3;
    const bool mine = ((m >> 2) & 1) == lane >> 5;
#pragma unroll
    for (u32 d = 0; d < 4; d++)
#pragma unroll
        for (u32 j = 0; j < 4; j++) {
            // rows 4 .. 7 for the blocks without the diagonal entry
            const u32 c = d == 3 ? l.mds[e][j] : l.mds[4 + e][(4 + 4 * d + j) % 12];
            t.w[d][j] = mine ? (int)(c << (8 * b)) : 0;
        }
}

// A multiplier the compiler must not turn into shifts or adds.
ZK_HD int opaque_int(int c)
{
#ifdef __HIP_DEVICE_COMPILE__
    int r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "i"(c));
    return r;
#else
    return c;
#endif
}

// s_0 + 2^8 s_1 + 2^16 s_2 + 2^24 s_3 + k for byte sums below 2^17 in
// magnitude.  The constant enters as the addend of the first multiply-add, in
// scalar registers (the compiler would add it by an instruction of its own).
ZK_HD u64 mfma_half(int s0, int s1, int s2, int s3, u64 k, int c65536, int c1)
{
    const int u0 = s0 + (s1 << 8), u1 = s2 + (s3 << 8);
#ifdef __HIP_DEVICE_COMPILE__
    int64_t a;
    u64 carry;
    asm("v_mad_i64_i32 %0, %1, %2, %3, %4" : "=v"(a), "=s"(carry) : "v"(u1), "v"(c65536), "s"(k));
#else
    const int64_t a = (int64_t)u1 * c65536 + (int64_t)k;
#endif
    return (u64)((int64_t)u0 * c1 + a);
}

// state <- M state + the constants k (12 pairs, MfmaConsts); rows as mds_fold.
// All lanes of the wave must call it together.
ZK_DEV void mds_mfma(u64 s[12], const u64 (*k)[2], const MfmaTiles &t, u32 need, bool &rare)
{
#ifdef __HIP_DEVICE_COMPILE__
    v4i lo[3], hi[3];
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lo[q][j] = (int)((u32)s[4 * q + j] ^ 0x80808080u);
            hi[q][j] = (int)((u32)(s[4 * q + j] >> 32) ^ 0x80808080u);
        }
    const int c65536 = opaque_int(65536), c1 = opaque_int(1);
#pragma unroll
    for (int r = 0; r < 3; r++) {
        if (!(need >> r & 1)) continue;
        // this group's constants, loaded before the MFMAs are issued
        u64 kr[4][2];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            kr[e][0] = k[4 * r + e][0];
            kr[e][1] = k[4 * r + e][1];
        }
        __builtin_amdgcn_sched_barrier(0);
        v16i dl = {}, dh = {};
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const v4i &w = t.w[r == 0 && q == 0 ? 3 : (q + 3 - r) % 3];
            dl = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, lo[q], dl, 0, 0, 0);
            dh = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, hi[q], dh, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const u64 a = mfma_half(dl[4 * e], dl[4 * e + 1], dl[4 * e + 2], dl[4 * e + 3], kr[e][0], c65536, c1);
            const u64 b = mfma_half(dh[4 * e], dh[4 * e + 1], dh[4 * e + 2], dh[4 * e + 3], kr[e][1], c65536, c1);
            s[4 * r + e] = reduce_lohi42_nc(a, b, rare);
        }
    }
#endif
}

// poseidon_permute on the relaxed path; all lanes of the wave must call it
// together.
ZK_DEV void poseidon_permute_mfma(u64 s[12], const MfmaTiles &t, bool &rare, u32 need = kAllRows)
{
    const u64 *rc = folded_constants();
    const u64(*k)[2] = kMfmaConstDev.k;
#pragma unroll
    for (int i = 0; i < 12; i++) s[i] = gl_add_nc(s[i], rc[i], rare);
#pragma unroll 1
    for (int r = 0; r < 3; r++) {
#pragma unroll
        for (int i = 0; i < 12; i++) s[i] = sbox7(s[i], rare);
        mds_mfma(s, k + 12 * (r + 1), t, kAllRows, rare);
    }
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
    for (int r = 26; r < 30; r++) {
#pragma unroll
        for (int i = 0; i < 12; i++) s[i] = sbox7(s[i], rare);
        mds_mfma(s, k + 12 * (r + 1), t, r < 29 ? kAllRows : need, rare);
    }
}

// poseidon_permute_mfma for the sponges of poseidon.hpp, which then need all
// lanes of the wave: a lane without work of its own hashes another's input.
struct MfmaPermute {
    MfmaTiles t;
    ZK_DEV MfmaPermute() { mfma_tiles(threadIdx.x & 63, t); }
    ZK_DEV void operator()(u64 s[12], bool &rare, u32 need) const { poseidon_permute_mfma(s, t, rare, need); }
};

}  // namespace zk
