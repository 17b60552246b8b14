// Poseidon permutation spread over a quad of lanes, for latency-bound callers
// (levels of a Merkle tree, small trees): same function as poseidon_permute.
//
// Lane j (= lane & 3) of a quad holds state elements 3j, 3j+1, 3j+2.  A full
// round is: S-box on the lane's elements, then the lane gathers the other nine
// elements of its quad with DPP quad permutes, t[e] = s[(3j + e) mod 12], and
// computes its three MDS rows: row 3j + k = sum_i c_i t[(i + k) mod 12] (+ 8
// t[0] for row 0) + the next round's constant.  Because 3 * 4 = 12, the
// rotated index needs no per-lane fix-up, so the MDS coefficients stay
// immediates.  The partial rounds go in blocks of four layers as in
// partial_block: the state is broadcast once a block, each lane accumulates
// its three rows of the block's result and, lanes 0 .. 2, one of the three
// inner values of element 0 (coefficients in registers), and every lane pair
// runs the block's four S-boxes (sbox7_pair).
//
// The S-box and row phases are host-callable (a host emulation runs the four
// lanes in lock step); only the gathers are device code.
#pragma once
#include "poseidon.hpp"

namespace zk {

// Phase A of a round: S-box on the lane's elements (all three in a full
// round, element 0 of lane 0 in a partial round).
template <bool SAFE>
ZK_HD void quad_sbox(u64 s[3], u32 j, bool full, bool &rare)
{
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (full || k == 0) {
            const u64 x = s[k];
            u64 y;
            if (SAFE) {
                const u64 x2 = gl_mul(x, x), x4 = gl_mul(x2, x2);
                y = gl_mul(gl_mul(x, x2), x4);
            } else {
                bool r = false;
                y = sbox7(x, r);
                if (full || j == 0) rare |= r;
            }
            if (full || j == 0) s[k] = y;
        }
    }
}

// Phase B: the lane's three MDS rows from the gathered state t[e] =
// s[(3j + e) mod 12], plus the next round's constants rk[k] (= constant
// 3j + k of that round).  Exact
// (the limb sums stay below 2^42 and the reduction has no rare case); SAFE
// canonicalises the outputs.
template <bool SAFE>
ZK_HD void quad_mds(const u64 t[12], u32 j, const u64 rk[3], u64 s[3])
{
    u32 lo[12], hi[12];
#pragma unroll
    for (int e = 0; e < 12; e++) {
        lo[e] = (u32)t[e];
        hi[e] = (u32)(t[e] >> 32);
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
        u64 a = (u32)rk[k], b = rk[k] >> 32;
#pragma unroll
        for (int i = 0; i < 12; i++) {
            const u64 c = mds_coeff(i);
            a += c * lo[(i + k) % 12];
            b += c * hi[(i + k) % 12];
        }
        if (k == 0) {  // diag[0] = 8 on row 0 (lane 0), 0 elsewhere
            const u64 dg = j == 0 ? PoseidonConsts::diag[0] : 0;
            a += dg * lo[0];
            b += dg * hi[0];
        }
        const u64 v = reduce_lohi42(a, b);
        s[k] = SAFE ? gl_canon(v) : v;
    }
}

// Value of x held by lane (j + D) & 3 of the same quad (DPP quad_perm).
template <int D>
ZK_DEV u64 quad_fetch(u64 x)
{
#ifdef __HIP_DEVICE_COMPILE__
    constexpr int ctrl = ((0 + D) & 3) | (((1 + D) & 3) << 2) | (((2 + D) & 3) << 4) | (((3 + D) & 3) << 6);
    const u32 lo = (u32)__builtin_amdgcn_mov_dpp((int)(u32)x, ctrl, 0xF, 0xF, false);
    const u32 hi = (u32)__builtin_amdgcn_mov_dpp((int)(u32)(x >> 32), ctrl, 0xF, 0xF, false);
    return ((u64)hi << 32) | lo;
#else
    return x;  // device-only function; the host pass never runs it
#endif
}

// A lane's coefficients in a block (lane_rows): its three rows of the result,
// and the row of the inner value it computes (lane 3: zeros).
struct QuadCoefs {
    u32 f[3][15], v[15];
};

ZK_HD void quad_coefs(u32 j, QuadCoefs &c)
{
    const LaneRows &l = lane_rows();
#pragma unroll
    for (int i = 0; i < 15; i++) {
#pragma unroll
        for (int k = 0; k < 3; k++) c.f[k][i] = l.block[3 * j + k][i];
        c.v[i] = l.block[12 + j][i];
    }
}

// x of lane K of the quad, on every lane of it.
template <int K>
ZK_DEV u64 quad_bcast(u64 x)
{
#ifdef __HIP_DEVICE_COMPILE__
    constexpr int ctrl = K | (K << 2) | (K << 4) | (K << 6);
    const u32 lo = (u32)__builtin_amdgcn_mov_dpp((int)(u32)x, ctrl, 0xF, 0xF, false);
    const u32 hi = (u32)__builtin_amdgcn_mov_dpp((int)(u32)(x >> 32), ctrl, 0xF, 0xF, false);
    return ((u64)hi << 32) | lo;
#else
    return x;  // device-only function; the host emulation gathers itself
#endif
}

// Rounds [r0, r1) one by one, constants from rc (row r + 1 added by round r).
template <bool SAFE>
ZK_DEV void quad_rounds(u64 s[3], u32 j, const u64 *rc, int r0, int r1, bool &rare)
{
    // this lane's constants are vector loads (lane-dependent index): fetch
    // them one round ahead so their latency hides behind the S-box
    u64 rk[3];
#pragma unroll
    for (int k = 0; k < 3; k++) rk[k] = rc[12 * (r0 + 1) + 3 * j + k];
#pragma unroll 1
    for (int r = r0; r < r1; r++) {
        const int rn = r + 2 < 31 ? r + 2 : 30;  // row 30 is the all-zero tail
        u64 rk_next[3];
#pragma unroll
        for (int k = 0; k < 3; k++) rk_next[k] = rc[12 * rn + 3 * j + k];
        quad_sbox<SAFE>(s, j, r < 4 || r >= 26, rare);
        u64 t[12];
        t[0] = s[0];
        t[1] = s[1];
        t[2] = s[2];
        t[3] = quad_fetch<1>(s[0]);
        t[4] = quad_fetch<1>(s[1]);
        t[5] = quad_fetch<1>(s[2]);
        t[6] = quad_fetch<2>(s[0]);
        t[7] = quad_fetch<2>(s[1]);
        t[8] = quad_fetch<2>(s[2]);
        t[9] = quad_fetch<3>(s[0]);
        t[10] = quad_fetch<3>(s[1]);
        t[11] = quad_fetch<3>(s[2]);
        quad_mds<SAFE>(t, j, rk, s);
#pragma unroll
        for (int k = 0; k < 3; k++) rk[k] = rk_next[k];
    }
}

// The permutation on the relaxed path for lane j of a quad (all four lanes
// must execute it together).
ZK_DEV void poseidon_permute_quad_nc(u64 s[3], u32 j, const QuadCoefs &c, bool &rare)
{
    const u64 *rc = folded_constants();
#pragma unroll
    for (int k = 0; k < 3; k++) s[k] = gl_add_nc(s[k], rc[3 * j + k], rare);
    quad_rounds<false>(s, j, rc, 0, kBlockStart, rare);
    // constants of a block: element 0 after its layers; lane j < 3 takes layer
    // j's for its inner value, lane 0 the last for its row 0
    const u64 *kp = rc + 12 * (kBlockStart + 1);
#pragma unroll 1
    for (int blk = 0; blk < kBlocks; blk++, kp += 12 * kBlock) {
        const u64 kv = kp[12 * j], kf = j ? 0 : kp[12 * 3];
        u64 t[12];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            t[k] = quad_bcast<0>(s[k]);
            t[3 + k] = quad_bcast<1>(s[k]);
            t[6 + k] = quad_bcast<2>(s[k]);
            t[9 + k] = quad_bcast<3>(s[k]);
        }
        u64 av = (u32)kv, bv = kv >> 32, a[3] = {(u32)kf, 0, 0}, b[3] = {kf >> 32, 0, 0};
        row_sum<1>(c.v, t, av, bv);
        u64 y = sbox7_pair(t[0], j & 1, LaneSwap(), rare);
        row_add(c.v[0], y, av, bv);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            row_sum<1>(c.f[k], t, a[k], b[k]);
            row_add(c.f[k][0], y, a[k], b[k]);
        }
        static_for<0, kBlock - 1>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            y = sbox7_pair(quad_bcast<q>(reduce_lohi64(av, bv, rare)), j & 1, LaneSwap(), rare);
            if constexpr (q < kBlock - 2) row_add(c.v[12 + q], y, av, bv);
#pragma unroll
            for (int k = 0; k < 3; k++) row_add(c.f[k][12 + q], y, a[k], b[k]);
        });
#pragma unroll
        for (int k = 0; k < 3; k++) s[k] = reduce_lohi64(a[k], b[k], rare);
    }
#pragma unroll
    for (int k = 0; k < 3; k++) s[k] = gl_add_nc(s[k], 3 * j + k ? rc[12 * 26 + 3 * j + k] : 0, rare);
    quad_rounds<false>(s, j, rc, 26, 30, rare);
}

// The permutation on the exact path (canonical in and out).
ZK_DEV void poseidon_permute_quad_safe(u64 s[3], u32 j)
{
    const u64 *rc = round_constants();
    bool unused = false;
#pragma unroll
    for (int k = 0; k < 3; k++) s[k] = gl_add(s[k], rc[3 * j + k]);
    quad_rounds<true>(s, j, rc, 0, 30, unused);
}

// State element 3j + k of a two-to-one compression [a, b, 0, 0, 0, 0].
ZK_DEV u64 quad_two_input(const u64 *a, const u64 *b, u32 j, int k)
{
    const u32 e = 3 * j + (u32)k;
    return e < 4 ? a[e] : (e < 8 ? b[e - 4] : 0);
}

// H(a, b) by a quad: every lane of the quad calls it (a, b read by the lanes
// that need them); lane 0 returns digest elements 0..2 in out[0..2], lane 1
// element 3 in out[0].  All lanes of the wave must call it together (the
// rare-case recomputation is wave-uniform).
ZK_DEV void hash_two_quad(const u64 *a, const u64 *b, u32 j, const QuadCoefs &c, u64 out[3])
{
    u64 s[3];
#pragma unroll
    for (int k = 0; k < 3; k++) s[k] = quad_two_input(a, b, j, k);
    bool rare = false;
    poseidon_permute_quad_nc(s, j, c, rare);
    if (__any(rare)) {
#pragma unroll
        for (int k = 0; k < 3; k++) s[k] = gl_canon(quad_two_input(a, b, j, k));
        poseidon_permute_quad_safe(s, j);
    }
#pragma unroll
    for (int k = 0; k < 3; k++) out[k] = gl_canon(s[k]);
}

// hash_or_noop of n elements fetched by get(i), by a quad: lane j absorbs
// the rate elements 3j..3j+2 of each chunk of 8 (lane 2 only 6 and 7, lane 3
// none), overwrite mode.  Lane 0 returns digest elements 0..2 in out[0..2],
// lane 1 element 3 in out[0].  n <= 4 copies the input (zero padded).  All
// lanes of the wave must call it together with the same n.
template <typename Get>
ZK_DEV void hash_one_quad(Get get, u32 n, u32 j, const QuadCoefs &c, u64 out[3])
{
    if (n <= 4) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const u32 e = 3 * j + (u32)k;
            out[k] = e < n ? get(e) : 0;
        }
        return;
    }
    // the next chunk is fetched before the current one is permuted: two waves
    // on a SIMD do not hide its latency
    const auto fetch = [&](u32 idx, u64 v[3]) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const u32 e = 3 * j + (u32)k;
            if (e < 8 && idx + e < n) v[k] = get(idx + e);
        }
    };
    u64 s[3] = {0, 0, 0};
    fetch(0, s);
    for (u32 idx = 0; idx < n; idx += 8) {
        u64 v[3], in[3];
        fetch(idx + 8, v);
#pragma unroll
        for (int k = 0; k < 3; k++) in[k] = s[k];
        bool rare = false;
        poseidon_permute_quad_nc(s, j, c, rare);
        if (__any(rare)) {  // redo this permutation exactly
#pragma unroll
            for (int k = 0; k < 3; k++) s[k] = gl_canon(in[k]);
            poseidon_permute_quad_safe(s, j);
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const u32 e = 3 * j + (u32)k;
            if (e < 8 && idx + 8 + e < n) s[k] = v[k];
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++) out[k] = gl_canon(s[k]);
}

}  // namespace zk
