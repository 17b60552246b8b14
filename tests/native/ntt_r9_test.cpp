// The 9-bit and 8-bit forms of the 16-element pass (r16_*<1>, <0>), run thread by thread in
// kernel order, against the general pass (fast_phase) on the same plans: both
// computations of each transform must agree bit for bit.  Usage: ntt_r9_test;
// prints "ok, N transforms".
#include <stdio.h>
#include <string.h>

#include <random>
#include <vector>

#include "../../zeknox_amd/csrc/ntt_pass.hpp"

using namespace zk;

template <int XB, bool INV>
static void run_r16(const PassArgs &a, u64 ntiles)
{
    std::vector<u64> lds((size_t)R16<XB>::G * R16<XB>::GP);
    std::vector<u64> out(16 * kR10Threads);
    for (u64 b = 0; b < ntiles; b++) {
        u32 col;
        u64 jhi, fast0;
        Pass<8 + XB>::tile_decode(a, xcd_tile(b, ntiles), col, jhi, fast0);
        const bool last = (a.S + 8 + XB) == a.L;
        bool any = (a.flags & F_FORCE_EXACT) != 0;
        for (u32 t = 0; t < kR10Threads; t++) r16_step_a<XB, INV, false>(a, col, jhi, fast0, t, lds.data(), any);
        if constexpr (XB > 0)
            for (u32 t = 0; t < kR10Threads; t++) r16_step_b<XB, INV, false>(a, t, lds.data(), any);
        for (u32 t = 0; t < kR10Threads; t++) r16_step_c<XB, INV, false>(a, t, lds.data(), last, &out[16 * t], any);
        if (any) {
            for (u32 t = 0; t < kR10Threads; t++) r16_step_a<XB, INV, true>(a, col, jhi, fast0, t, lds.data(), any);
            if constexpr (XB > 0)
                for (u32 t = 0; t < kR10Threads; t++) r16_step_b<XB, INV, true>(a, t, lds.data(), any);
            for (u32 t = 0; t < kR10Threads; t++) r16_step_c<XB, INV, true>(a, t, lds.data(), last, &out[16 * t], any);
        }
        for (u32 t = 0; t < kR10Threads; t++) r16_store<XB>(a, col, jhi, fast0, t, last, &out[16 * t]);
    }
}

template <int B, bool INV>
static void run_fast(const PassArgs &a, u64 ntiles)
{
    std::vector<u64> lds(fast_lds_bytes<B>(1u << a.Gbits) / sizeof(u64) + 1);
    for (u64 b = 0; b < ntiles; b++)
        for (int phase = 0; phase < 2; phase++)
            for (u32 t = 0; t < kThreads; t++)
                fast_phase<(B + 1) / 2, B / 2, INV>(a, xcd_tile(b, ntiles), phase, t, kThreads, lds.data());
}

template <bool INV>
static void run_pass(const PassPlan &pp)
{
    if (pp.r9) return run_r16<1, INV>(pp.a, pp.ntiles);
    if (pp.r8) return run_r16<0, INV>(pp.a, pp.ntiles);
    switch (pp.B) {
    case 4: return run_fast<4, INV>(pp.a, pp.ntiles);
    case 5: return run_fast<5, INV>(pp.a, pp.ntiles);
    case 8: return run_fast<8, INV>(pp.a, pp.ntiles);
    case 9: return run_fast<9, INV>(pp.a, pp.ntiles);
    default: printf("pass of %u bits not run here\n", pp.B);
    }
}

static std::vector<u64> pw[2], tb[2], gpw;

static void fill_powers(u64 x, u64 *row, int n)
{
    u64 v = 1;
    for (int i = 0; i < n; i++) {
        row[i] = v;
        v = gl_mul(v, x);
    }
}

// One transform through the plan `bits` with the 9-bit kernel allowed or not.
static std::vector<u64> transform(u32 lg, u32 lg_in, u32 ncols, bool inv, bool coset, bool force, bool table, bool place,
                                  std::vector<u32> bits, bool r9, const std::vector<u64> &in, int &nr9)
{
    NttTune t{};
    t.np = (u32)bits.size();
    for (u32 p = 0; p < t.np; p++) {
        t.bits[p] = bits[p];
        t.gbits[p] = kTuneAuto;
        t.r10[p] = r9;
    }
    ntt_tune_table()[lg] = t;
    const u64 N = 1ull << lg;
    std::vector<u64> out(ncols * N, 0xDEADBEEFull), scratch(ncols * N);
    NttJob job;
    job.src = in.data();
    job.dst = out.data();
    job.src_stride = 1ull << lg_in;
    job.dst_stride = N;
    job.ncols = ncols;
    job.lg = lg;
    job.lg_in = lg_in;
    job.inverse = inv;
    job.coset_in = coset && !inv;
    job.coset_out = coset && inv;
    job.scale_out = inv;
    auto passes = plan_passes(job, pw[inv].data(), gpw.data(), place ? nullptr : scratch.data(), 66560);
    std::vector<std::vector<u64>> tws;
    tws.reserve(passes.size());
    for (PassPlan &pp : passes) {
        pp.a.tb = tb[inv].data();
        if (force) pp.a.flags |= F_FORCE_EXACT;
        if (pp.a.S > 0 && table) {
            tws.emplace_back(1ull << (pp.a.L - pp.a.Sprev));
            for (u64 i = 0; i < tws.back().size(); i++)
                tws.back()[i] = twiddle_entry(pw[inv].data(), pp.a.L, pp.a.S, pp.a.Sprev, i);
            pp.a.tw = tws.back().data();
        }
        // the rule takes the 8-bit form for launches that fill the chip; its
        // arithmetic is run here on small ones
        if (r9 && pp.B == 8 && pp.a.S == 0 && pp.a.Jbits >= kR8Gbits && !pp.r8) {
            pp.r8 = true;
            f16_retile(pp, kR8Gbits);
        }
        nr9 += pp.r9 || pp.r8;
        inv ? run_pass<true>(pp) : run_pass<false>(pp);
    }
    ntt_tune_table()[lg] = NttTune{};
    return out;
}

int main()
{
    gpw.resize(3 * kPowLen);
    u64 base = 7;
    for (int k = 0; k < 3; k++) {
        fill_powers(base, gpw.data() + k * kPowLen, kPowLen);
        base = gl_pow(base, (u64)kPowLen);
    }
    for (int d = 0; d < 2; d++) {
        pw[d].resize((size_t)(kMaxLg + 1) * kPowLen);
        tb[d].resize(16 * 64);
        for (int L = 0; L <= kMaxLg; L++) fill_powers(d ? gl_inv(gl_omega(L)) : gl_omega(L), &pw[d][(size_t)L * kPowLen], kPowLen);
        for (u32 v = 0; v < 16; v++) fill_powers(gl_pow(pw[d][(size_t)10 * kPowLen + 1], zk_bitrev(v, 4)), &tb[d][64 * v], 64);
    }
    std::mt19937_64 g(9);
    int runs = 0, fails = 0, nr9 = 0;
    // first, middle and last passes; 16 (32) groups exactly and more
    const std::vector<std::vector<u32>> plans = {{9, 4}, {4, 9}, {9, 5}, {5, 9}, {4, 9, 4},
                                                 {8, 5}, {8, 9}};
    for (const auto &bits : plans) {
        u32 lg = 0;
        for (u32 b : bits) lg += b;
        for (int inv = 0; inv < 2; inv++)
            for (u32 r = 0; r < (inv ? 1u : 7u); r += r < 3 ? 1 : 3)
                for (int form = 0; form < 4; form++) {
                    if (lg >= 16 && (form == 1 || form == 2 || r > 1)) continue;  // the larger plans: fewer forms
                    const u32 ncols = form == 2 ? 3 : 1;
                    const bool coset = form != 1, force = form == 3, table = form < 2, place = form == 2;
                    std::vector<u64> in((size_t)ncols << (lg - r));
                    for (u64 &x : in) x = g() % ZK_P;
                    int none = 0;
                    const auto want = transform(lg, lg - r, ncols, inv, coset, force, table, place, bits, false, in, none);
                    const auto got = transform(lg, lg - r, ncols, inv, coset, force, table, place, bits, true, in, nr9);
                    runs++;
                    if ((none || got != want) && fails++ < 10)
                        printf("plan %u,%u.. inv %d r %u form %d: differs\n", bits[0], bits[1], inv, r, form);
                }
    }
    if (!nr9) fails++;
    printf("%s, %d transforms, %d 16-element passes\n", fails ? "FAIL" : "ok", runs, nr9);
    return fails ? 1 : 0;
}
