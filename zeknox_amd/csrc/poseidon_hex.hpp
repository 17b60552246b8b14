// Poseidon permutation spread over 16 lanes, one state element per lane, for
// the latency-bound narrow levels of a Merkle tree: same function as
// poseidon_permute.
//
// Lane j (= lane & 15) of a group holds state element j for j < 12.  A lone
// wave issues one instruction every 7 to 8 cycles, so what a level costs is the
// number of instructions on a lane.  A full round is one S-box, a broadcast of
// the twelve elements to every lane of the group (DPP row_newbcast: a group is
// a DPP row, and unlike a lane exchange through LDS it has no latency to wait
// for) and the lane's row of the layer, its coefficients in registers.  The
// partial rounds go in blocks of four layers as in partial_block: lanes 0 .. 11
// accumulate the rows of the block's result and lanes 12 .. 14, idle otherwise,
// the three inner values of element 0 in the same instructions; every lane pair
// runs the block's four S-boxes on the broadcast value (sbox7_pair).
//
// The recomputation of a rare case (SAFE) runs round by round with the lanes'
// elements exchanged by ds_bpermute, lanes 12 .. 15 holding copies.
//
// The S-box and row phases are host-callable, so a host emulation can run the
// 16 lanes of a group in lock step (tests/native/poseidon_lanes_test.cpp,
// tests/native/poseidon_block_test.cpp); only the gathers are device code.
#pragma once
#include "poseidon.hpp"

namespace zk {

constexpr u32 kHexLanes = 16;

// Phase A of a round for the lane holding element j: the S-box (every lane
// in a full round, element 0 in a partial round).
template <bool SAFE>
ZK_HD u64 hex_sbox(u64 x, u32 j, bool full, bool &rare)
{
    u64 y;
    if (SAFE) {
        const u64 x2 = gl_mul(x, x), x4 = gl_mul(x2, x2);
        y = gl_mul(gl_mul(x, x2), x4);
    } else {
        bool r = false;
        y = sbox7(x, r);
        if (full || j == 0) rare |= r;
    }
    return (full || j == 0) ? y : x;
}

// Phase B: row j of the MDS from the gathered state t[k] = s[(j + k) mod 12]
// plus the next round's constant rk.  Exact (the half sums stay below 2^42 and
// the reduction has no rare case); SAFE canonicalises the output.
template <bool SAFE>
ZK_HD u64 hex_mds(const u64 t[12], u32 j, u64 rk)
{
    u64 a = (u32)rk, b = rk >> 32;
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const u64 c = mds_coeff(k);
        a += c * (u32)t[k];
        b += c * (u32)(t[k] >> 32);
    }
    const u64 dg = j == 0 ? PoseidonConsts::diag[0] : 0;  // diag[0] = 8, 0 on every other row
    a += dg * (u32)t[0];
    b += dg * (u32)(t[0] >> 32);
    const u64 v = reduce_lohi42(a, b);
    return SAFE ? gl_canon(v) : v;
}

// x of lane `src` (a lane of the same wave), through the LDS crossbar.
ZK_DEV u64 hex_fetch(u64 x, u32 src)
{
#ifdef __HIP_DEVICE_COMPILE__
    const int addr = (int)(src << 2);
    const u32 lo = (u32)__builtin_amdgcn_ds_bpermute(addr, (int)(u32)x);
    const u32 hi = (u32)__builtin_amdgcn_ds_bpermute(addr, (int)(u32)(x >> 32));
    return ((u64)hi << 32) | lo;
#else
    (void)src;
    return x;  // device-only function; the host emulation gathers itself
#endif
}

// A lane's coefficients: row j of the layer and of a block (lane_rows).
struct HexCoefs {
    u32 m[12], b[15];
};

ZK_HD void hex_coefs(u32 j, HexCoefs &c)
{
    const LaneRows &l = lane_rows();
#pragma unroll
    for (int i = 0; i < 12; i++) c.m[i] = l.mds[j][i];
#pragma unroll
    for (int i = 0; i < 15; i++) c.b[i] = l.block[j][i];
}

// x of lane K of the group, on every lane of it.
template <int K>
ZK_DEV u64 hex_bcast(u64 x)
{
#ifdef __HIP_DEVICE_COMPILE__
    const u32 lo = (u32)__builtin_amdgcn_mov_dpp((int)(u32)x, 0x150 + K, 0xF, 0xF, false);
    const u32 hi = (u32)__builtin_amdgcn_mov_dpp((int)(u32)(x >> 32), 0x150 + K, 0xF, 0xF, false);
    return ((u64)hi << 32) | lo;
#else
    return x;  // device-only function; the host emulation gathers itself
#endif
}

ZK_DEV void hex_gather(u64 s, u64 t[12])
{
    static_for<0, 12>([&](auto ic) { t[decltype(ic)::value] = hex_bcast<decltype(ic)::value>(s); });
}

// The permutation on the relaxed path for lane j of a 16-lane group (all 16
// lanes must run it together); lanes 12 .. 15 return nothing of use.
ZK_DEV void poseidon_permute_hex_nc(u64 &s, u32 j, const HexCoefs &c, bool &rare)
{
    const u64 *rc = folded_constants();
    const u32 e = j < 12 ? j : j - 12;
    s = gl_add_nc(s, rc[e], rare);
    u64 t[12];
    auto rounds = [&](int r0, int r1) {
        u64 rk = rc[12 * (r0 + 1) + e];
#pragma unroll 1
        for (int r = r0; r < r1; r++) {
            const u64 rk_next = rc[12 * (r + 2 < 31 ? r + 2 : 30) + e];
            s = hex_sbox<false>(s, e, r < 4 || r >= 26, rare);
            hex_gather(s, t);
            u64 a = (u32)rk, b = rk >> 32;
            row_sum<0>(c.m, t, a, b);
            s = reduce_lohi42(a, b);
            rk = rk_next;
        }
    };
    rounds(0, kBlockStart);
    // constants of a block: element 0 after its layers, on lanes 12, 13, 14 and 0
    const u64 *kp = rc + 12 * (kBlockStart + 1 + (j >= 12 ? j - 12 : 3));
    const bool has_k = j == 0 || (j >= 12 && j < 15);
#pragma unroll 1
    for (int blk = 0; blk < kBlocks; blk++) {
        const u64 kk = kp[12 * kBlock * blk];
        const u64 k = has_k ? kk : 0;
        u64 a = (u32)k, b = k >> 32;
        hex_gather(s, t);
        row_sum<1>(c.b, t, a, b);
        u64 y = sbox7_pair(t[0], j & 1, LaneSwap(), rare);
        row_add(c.b[0], y, a, b);
        static_for<0, kBlock - 1>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            y = sbox7_pair(hex_bcast<12 + q>(reduce_lohi64_exact(a, b)), j & 1, LaneSwap(), rare);
            row_add(c.b[12 + q], y, a, b);
        });
        s = reduce_lohi64_exact(a, b);
    }
    s = gl_add_nc(s, e ? rc[12 * 26 + e] : 0, rare);
    rounds(26, 30);
}

// The permutation on the exact path (canonical in and out), round by round;
// `base` is the wave lane of the group's lane 0.
ZK_DEV void poseidon_permute_hex_safe(u64 &s, u32 j, u32 base)
{
    const u64 *rc = round_constants();
    const u32 e = j < 12 ? j : j - 12;  // the element this lane holds
    s = gl_add(s, rc[e]);
    u32 src[12];
#pragma unroll
    for (int k = 1; k < 12; k++) src[k] = base + (e + (u32)k) % 12;
#pragma unroll 1
    for (int r = 0; r < 30; r++) {
        bool unused = false;
        s = hex_sbox<true>(s, e, r < 4 || r >= 26, unused);
        u64 t[12];
        t[0] = s;
#pragma unroll
        for (int k = 1; k < 12; k++) t[k] = hex_fetch(s, src[k]);
        s = hex_mds<true>(t, e, rc[12 * (r + 1) + e]);
    }
}

// H(a, b) by a 16-lane group: every lane calls it (lane j reads the element
// it holds) with its coefficients; lanes 0..3 return digest element j.  All
// lanes of the wave must call it together (the rare-case recomputation is
// wave-uniform).
ZK_DEV u64 hash_two_hex(const u64 *a, const u64 *b, u32 j, u32 base, const HexCoefs &c)
{
    const u32 e = j < 12 ? j : j - 12;
    const u64 in = e < 4 ? a[e] : (e < 8 ? b[e - 4] : 0);
    u64 s = in;
    bool rare = false;
    poseidon_permute_hex_nc(s, j, c, rare);
    if (__any(rare)) {
        s = gl_canon(in);
        poseidon_permute_hex_safe(s, j, base);
    }
    return gl_canon(s);
}

// hash_or_noop of n elements fetched by get(i), by a 16-lane group: lane j < 8
// absorbs element j of each chunk of 8, overwrite mode.  Lanes 0..3 return
// digest element j.  n <= 4 copies the input (zero padded).  All lanes of the
// wave must call it together with the same n.
template <typename Get>
ZK_DEV u64 hash_one_hex(Get get, u32 n, u32 j, u32 base, const HexCoefs &c)
{
    if (n <= 4) return j < n ? get(j) : 0;
    const auto fetch = [&](u32 idx, u64 old) { return j < 8 && idx + j < n ? get(idx + j) : old; };
    u64 s = fetch(0, 0);
    for (u32 idx = 0; idx < n; idx += 8) {
        const u64 next = fetch(idx + 8, 0);  // in flight during the permutation
        const u64 in = s;
        bool rare = false;
        poseidon_permute_hex_nc(s, j, c, rare);
        if (__any(rare)) {
            // redo this permutation exactly; lanes 12 .. 15 take their copies
            const u64 copy = hex_fetch(in, base + (j < 12 ? j : j - 12));
            s = gl_canon(copy);
            poseidon_permute_hex_safe(s, j, base);
        }
        if (j < 8 && idx + 8 + j < n) s = next;
    }
    return gl_canon(s);
}

}  // namespace zk
