// Host emulation of a whole transform through the kernels ntt_launch picks:
// as ntt_host_test.cpp, whose kernels and arguments it takes, with the
// dispatch of launch_f16 (the 16-element kernel's 10-, 9- and 8-bit forms).
// Prints each pass's form; with no columns' file ("-") it only prints the plan.
//
// usage: ntt_forms_test lg lg_in ncols inverse coset force_exact table in.bin out.bin
//        [np b1 b2 b3 g1 g2 g3 r1 r2 r3]
#define main ntt_host_test_main
#include "ntt_host_test.cpp"
#undef main

template <int XB, bool INV, bool SAFE>
static bool r16_steps(const PassArgs &a, u32 col, u64 jhi, u64 fast0, u64 *lds, bool last, u64 *out)
{
    bool rare = (a.flags & F_FORCE_EXACT) != 0;
    for (u32 t = 0; t < kR10Threads; t++) r16_step_a<XB, INV, SAFE>(a, col, jhi, fast0, t, lds, rare);
    if constexpr (XB > 0)
        for (u32 t = 0; t < kR10Threads; t++) r16_step_b<XB, INV, SAFE>(a, t, lds, rare);
    for (u32 t = 0; t < kR10Threads; t++) r16_step_c<XB, INV, SAFE>(a, t, lds, last, out + 16 * t, rare);
    return rare;
}

// ntt_r16_kernel; returns the tiles that took the exact path
template <int XB, bool INV>
static u64 run_r16(const PassArgs &a, u64 ntiles)
{
    using R = R16<XB>;
    std::vector<u64> lds((size_t)R::G * R::GP), out(16 * kR10Threads);
    u64 exact = 0;
    for (u64 b = 0; b < ntiles; b++) {
        u32 col;
        u64 jhi, fast0;
        Pass<R::B>::tile_decode(a, xcd_tile(b, ntiles), col, jhi, fast0);
        const bool last = (a.S + R::B) == a.L;
        if (r16_steps<XB, INV, false>(a, col, jhi, fast0, lds.data(), last, out.data())) {
            exact++;
            r16_steps<XB, INV, true>(a, col, jhi, fast0, lds.data(), last, out.data());
        }
        for (u32 t = 0; t < kR10Threads; t++) r16_store<XB>(a, col, jhi, fast0, t, last, &out[16 * t]);
    }
    return exact;
}

template <bool INV>
static u64 run_pass(const PassPlan &pp)
{
    if (pp.r10) return run_r16<2, INV>(pp.a, pp.ntiles);
    if (pp.r9) return run_r16<1, INV>(pp.a, pp.ntiles);
    if (pp.r8) return run_r16<0, INV>(pp.a, pp.ntiles);
    run_fast_b<INV>(pp.B, pp.a, pp.ntiles);
    return 0;
}

int main(int argc, char **argv)
{
    if (argc != 10 && argc != 20) return 2;
    const u32 lg = atoi(argv[1]), lg_in = atoi(argv[2]), ncols = atoi(argv[3]);
    const bool inv = atoi(argv[4]) != 0, coset = atoi(argv[5]) != 0, force = atoi(argv[6]) != 0;
    const bool table = atoi(argv[7]) != 0, run = strcmp(argv[8], "-") != 0;
    const u64 N = 1ull << lg, n = 1ull << lg_in;
    if (argc > 10) {
        NttTune t{};
        t.np = (u32)atoi(argv[10]);
        for (int p = 0; p < 3; p++) {
            const int g = atoi(argv[14 + p]);
            t.bits[p] = (u32)atoi(argv[11 + p]);
            t.gbits[p] = g < 0 ? kTuneAuto : (u32)g;
            t.r10[p] = (u32)atoi(argv[17 + p]);
        }
        if (!ntt_tune_valid(lg, t)) return 6;
        ntt_tune_table()[lg] = t;
    }
    std::vector<u64> in(run ? ncols * n : 1), out(run ? ncols * N : 1, 0xDEADBEEFull), scratch(out.size());
    FILE *f;
    if (run) {
        f = fopen(argv[8], "rb");
        if (!f || fread(in.data(), 8, in.size(), f) != in.size()) return 3;
        fclose(f);
    }
    // the device context's tables, on the host
    std::vector<u64> pw((size_t)(kMaxLg + 1) * kPowLen), gpw(3 * kPowLen), tb(16 * 64);
    for (int L = 0; L <= kMaxLg; L++) {
        const u64 w = gl_omega((u32)L);
        fill_powers(inv ? gl_inv(w) : w, pw.data() + (size_t)L * kPowLen, kPowLen);
    }
    for (int k = 0; k < 3; k++)
        fill_powers(k == 0 ? 7 : gl_pow(gpw[(k - 1) * kPowLen + 1], (u64)kPowLen), gpw.data() + k * kPowLen, kPowLen);
    const u64 w1024 = pw[(size_t)10 * kPowLen + 1];
    for (u32 v = 0; v < 16; v++) fill_powers(gl_pow(w1024, zk_bitrev(v, 4)), tb.data() + 64 * v, 64);

    NttJob job;
    job.src = in.data();
    job.dst = out.data();
    job.src_stride = n;
    job.dst_stride = N;
    job.ncols = ncols;
    job.lg = lg;
    job.lg_in = lg_in;
    job.inverse = inv;
    job.coset_in = coset && !inv;
    job.coset_out = coset && inv;
    job.scale_out = inv;
    auto passes = plan_passes(job, pw.data(), gpw.data(), scratch.data(), 66560);
    std::vector<std::vector<u64>> tws(passes.size());
    for (size_t p = 0; p < passes.size(); p++) {
        PassPlan &pp = passes[p];
        if (!pp.fast || pp.r10 + pp.r9 + pp.r8 > 1) return 7;
        pp.a.tb = tb.data();
        if (force) pp.a.flags |= F_FORCE_EXACT;
        if (run && table && pp.a.S > 0) {
            tws[p].resize(1ull << (pp.a.L - pp.a.Sprev));
            for (u64 i = 0; i < tws[p].size(); i++)
                tws[p][i] = twiddle_entry(pw.data(), pp.a.L, pp.a.S, pp.a.Sprev, i);
            pp.a.tw = tws[p].data();
        }
        const u64 exact = !run ? 0 : (inv ? run_pass<true>(pp) : run_pass<false>(pp));
        const char *form = pp.r10 ? "r10" : (pp.r9 ? "r9" : (pp.r8 ? "r8" : "general"));
        printf("pass S=%u B=%u tiles=%llu exact=%llu form=%s\n", pp.a.S, pp.B, (unsigned long long)pp.ntiles,
               (unsigned long long)exact, form);
    }
    if (!run) return 0;
    f = fopen(argv[9], "wb");
    if (!f || fwrite(out.data(), 8, out.size(), f) != out.size()) return 4;
    fclose(f);
    return 0;
}
