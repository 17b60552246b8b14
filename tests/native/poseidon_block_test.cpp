// The blocked permutation (poseidon_permute) against the exact one
// (poseidon_permute_safe) on random and edge states, with every set of wanted
// rows; the relaxed permutations of 16 lanes and of a quad, their lanes run in
// lock step with the broadcasts done here; the block reductions against 128-bit arithmetic at the limits of their
// ranges; and the block tables' row sums against the limit the 64-bit sums
// need.  Prints "ok, N states, M rare".
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../zeknox_amd/csrc/poseidon_hex.hpp"
#include "../../zeknox_amd/csrc/poseidon_mfma.hpp"
#include "../../zeknox_amd/csrc/poseidon_quad.hpp"

using namespace zk;
typedef unsigned __int128 u128;

static int fails = 0;

static void expect(const char *what, u64 got, u128 want)
{
    if (gl_canon(got) != (u64)(want % ZK_P) && fails++ < 10) printf("%s: wrong value\n", what);
}

// sbox7_pair on the even and the odd lane of a pair, which must agree
static u64 sbox_pair(u64 x, bool &rare)
{
    u64 y[2];
    for (int odd = 0; odd < 2; odd++)
        y[odd] = sbox7_pair(x, odd, [&](u64) {
            u64 other = 0;  // what the other lane passes to its exchange
            (void)sbox7_pair(x, !odd, [&](u64 r) { return other = r; }, rare);
            return other;
        }, rare);
    if (y[0] != y[1] && fails++ < 10) printf("sbox7_pair: the lanes differ\n");
    return y[0];
}

// poseidon_permute_hex_nc, lane by lane
static void permute_hex(u64 st[12], bool &rare)
{
    const u64 *rc = folded_constants();
    HexCoefs c[16];
    u64 s[16], t[12], a[16], b[16];
    for (u32 j = 0; j < 16; j++) {
        hex_coefs(j, c[j]);
        const u32 e = j < 12 ? j : j - 12;
        s[j] = gl_add_nc(st[e], rc[e], rare);
    }
    auto gather = [&] {
        for (int i = 0; i < 12; i++) t[i] = s[i];
    };
    auto rounds = [&](int r0, int r1) {
        for (int r = r0; r < r1; r++) {
            for (u32 j = 0; j < 16; j++) s[j] = hex_sbox<false>(s[j], j < 12 ? j : j - 12, r < 4 || r >= 26, rare);
            gather();
            for (u32 j = 0; j < 16; j++) {
                const u64 k = rc[12 * (r + 1) + (j < 12 ? j : j - 12)];
                u64 x = (u32)k, y = k >> 32;
                row_sum<0>(c[j].m, t, x, y);
                s[j] = reduce_lohi42(x, y);
            }
        }
    };
    rounds(0, kBlockStart);
    for (int blk = 0; blk < kBlocks; blk++) {
        const u64 *kp = rc + 12 * (kBlockStart + 1 + kBlock * blk);
        gather();
        const u64 y0 = sbox_pair(t[0], rare);
        for (u32 j = 0; j < 16; j++) {
            const u64 k = j >= 12 && j < 15 ? kp[12 * (j - 12)] : (j == 0 ? kp[36] : 0);
            a[j] = (u32)k;
            b[j] = k >> 32;
            row_sum<1>(c[j].b, t, a[j], b[j]);
            row_add(c[j].b[0], y0, a[j], b[j]);
        }
        for (int q = 0; q < kBlock - 1; q++) {
            u64 v[16];
            for (u32 j = 0; j < 16; j++) v[j] = reduce_lohi64_exact(a[j], b[j]);
            const u64 y = sbox_pair(v[12 + q], rare);
            for (u32 j = 0; j < 16; j++) row_add(c[j].b[12 + q], y, a[j], b[j]);
        }
        for (u32 j = 0; j < 16; j++) s[j] = reduce_lohi64_exact(a[j], b[j]);
    }
    for (u32 e = 1; e < 12; e++) s[e] = gl_add_nc(s[e], rc[12 * 26 + e], rare);
    rounds(26, 30);
    for (int e = 0; e < 12; e++) st[e] = s[e];
}

// poseidon_permute_quad_nc, lane by lane
static void permute_quad(u64 st[12], bool &rare)
{
    const u64 *rc = folded_constants();
    QuadCoefs c[4];
    u64 s[4][3];
    for (u32 j = 0; j < 4; j++) {
        quad_coefs(j, c[j]);
        for (u32 k = 0; k < 3; k++) s[j][k] = gl_add_nc(st[3 * j + k], rc[3 * j + k], rare);
    }
    auto rounds = [&](int r0, int r1) {
        for (int r = r0; r < r1; r++) {
            for (u32 j = 0; j < 4; j++) quad_sbox<false>(s[j], j, r < 4 || r >= 26, rare);
            u64 n[4][3];
            for (u32 j = 0; j < 4; j++) {
                u64 t[12];
                for (u32 e = 0; e < 12; e++) t[e] = s[(3 * j + e) % 12 / 3][(3 * j + e) % 3];
                quad_mds<false>(t, j, rc + 12 * (r + 1) + 3 * j, n[j]);
            }
            for (u32 j = 0; j < 4; j++)
                for (int k = 0; k < 3; k++) s[j][k] = n[j][k];
        }
    };
    rounds(0, kBlockStart);
    for (int blk = 0; blk < kBlocks; blk++) {
        const u64 *kp = rc + 12 * (kBlockStart + 1 + kBlock * blk);
        u64 t[12], a[4][4], b[4][4];  // [lane][three rows, inner value]
        for (u32 e = 0; e < 12; e++) t[e] = s[e / 3][e % 3];
        const u64 y0 = sbox_pair(t[0], rare);
        for (u32 j = 0; j < 4; j++)
            for (int k = 0; k < 4; k++) {
                const u32 *cc = k < 3 ? c[j].f[k] : c[j].v;
                const u64 kk = k == 3 ? kp[12 * j] : (j + k == 0 ? kp[36] : 0);
                a[j][k] = (u32)kk;
                b[j][k] = kk >> 32;
                row_sum<1>(cc, t, a[j][k], b[j][k]);
                row_add(cc[0], y0, a[j][k], b[j][k]);
            }
        for (int q = 0; q < kBlock - 1; q++) {
            const u64 y = sbox_pair(reduce_lohi64(a[q][3], b[q][3], rare), rare);
            for (u32 j = 0; j < 4; j++) {
                row_add(c[j].v[12 + q], y, a[j][3], b[j][3]);
                for (int k = 0; k < 3; k++) row_add(c[j].f[k][12 + q], y, a[j][k], b[j][k]);
            }
        }
        for (u32 j = 0; j < 4; j++)
            for (int k = 0; k < 3; k++) s[j][k] = reduce_lohi64(a[j][k], b[j][k], rare);
    }
    for (u32 e = 1; e < 12; e++) s[e / 3][e % 3] = gl_add_nc(s[e / 3][e % 3], rc[12 * 26 + e], rare);
    rounds(26, 30);
    for (u32 e = 0; e < 12; e++) st[e] = s[e / 3][e % 3];
}

// One layer as mds_mfma computes it for 64 lanes, with the MFMA's sums formed
// here from its operand layout (A row m and B column m of lane m + 32 k are the
// k half's 16 bytes; result register i of lane n + 32 g is row 8 (i / 4) + 4 g
// + i % 4 of column n), against the layer by multiply-adds.
static void check_mfma_layer(std::mt19937_64 &g)
{
    static const MfmaConsts mc = make_mfma_consts();
    MfmaTiles t[64];
    u64 s[64][12];
    for (u32 l = 0; l < 64; l++) {
        mfma_tiles(l, t[l]);
        for (int i = 0; i < 12; i++) s[l][i] = l % 3 ? g() : (l & 1 ? ~0ull : 0);
    }
    auto byte = [](const v4i &v, int k) { return (int)(signed char)(v[k / 4] >> (8 * (k % 4))); };
    const int round = (int)(g() % 3) + 1;
    for (u32 l = 0; l < 64; l++) {
        u64 want[12];
        for (int i = 0; i < 12; i++) want[i] = s[l][i];
        bool rare = false;
        mds_fold(want, folded_constants() + 12 * round, kAllRows, rare);
        for (int r = 0; r < 3; r++) {
            int d[2][16] = {};
            for (int half = 0; half < 2; half++)
                for (int q = 0; q < 3; q++)
                    for (int i = 0; i < 16; i++) {
                        const u32 m = 8 * (i / 4) + 4 * (l >> 5) + i % 4;
                        for (u32 kh = 0; kh < 2; kh++) {  // both k halves of column l % 32
                            const u32 bl = (l & 31) + 32 * kh;
                            v4i b;
                            for (int j = 0; j < 4; j++) b[j] = (int)((u32)(s[bl][4 * q + j] >> (32 * half)) ^ 0x80808080u);
                            const v4i &a = t[m + 32 * kh].w[r == 0 && q == 0 ? 3 : (q + 3 - r) % 3];
                            for (int k = 0; k < 16; k++) d[half][i] += byte(a, k) * byte(b, k);
                        }
                    }
            for (int e = 0; e < 4; e++) {
                const u64 *k = mc.k[12 * round + 4 * r + e];
                const u64 a = mfma_half(d[0][4 * e], d[0][4 * e + 1], d[0][4 * e + 2], d[0][4 * e + 3], k[0], 65536, 1);
                const u64 b = mfma_half(d[1][4 * e], d[1][4 * e + 1], d[1][4 * e + 2], d[1][4 * e + 3], k[1], 65536, 1);
                const u64 got = reduce_lohi42_nc(a, b, rare);
                if (!rare && gl_canon(got) != gl_canon(want[4 * r + e]) && fails++ < 10)
                    printf("mfma layer: lane %u row %d differs\n", l, 4 * r + e);
            }
        }
    }
}

template <int K>
static void row_sums()
{
    constexpr PartialBlock<K> t = make_partial_block<K>();
    // halves below 2^32 times a row sum s, plus a constant below 2^32, stay
    // below (s + 1) 2^32; reduce_lohi64 needs sums below 2^64 - 2^32
    const u64 limit = (1ull << 32) - 2;
    for (int r = 0; r < 12; r++) {
        u64 s = 0;
        for (int c = 0; c < PartialBlock<K>::IN; c++) s += t.f[r][c];
        if (s > limit && fails++ < 10) printf("K %d row %d: sum too large\n", K, r);
    }
}

int main(int argc, char **argv)
{
    const int n = argc > 1 ? atoi(argv[1]) : 20000;
    std::mt19937_64 g(11);
    const u64 edges[] = {0, 1, 0xFFFFFFFFull, 1ull << 32, ZK_P - 1, ZK_P, ZK_P + 1, ~0ull, ~0ull - 1, ~0ull << 32};
    long rares = 0;
    for (int it = 0; it < n; it++) {
        u64 in[12], want[12];
        for (int i = 0; i < 12; i++) want[i] = in[i] = it % 3 ? g() : edges[g() % 10];
        poseidon_permute_safe(want);
        for (int lanes = 0; lanes < 2; lanes++) {
            u64 s[12];
            for (int i = 0; i < 12; i++) s[i] = in[i];
            bool rare = false;
            lanes ? permute_quad(s, rare) : permute_hex(s, rare);
            if (rare) {
                rares++;
                continue;
            }
            for (int i = 0; i < 12; i++)
                if (gl_canon(s[i]) != want[i] && fails++ < 10)
                    printf("state %d %s: element %d differs\n", it, lanes ? "quad" : "hex", i);
        }
        for (u32 need = 1; need < 8; need++) {
            u64 s[12];
            for (int i = 0; i < 12; i++) s[i] = in[i];
            bool rare = false;
            poseidon_permute(s, rare, need);
            if (rare) {
                rares++;
                continue;
            }
            for (int i = 0; i < 12; i++)
                if ((need >> (i / 4) & 1) && gl_canon(s[i]) != want[i] && fails++ < 10)
                    printf("state %d need %u: element %d differs\n", it, need, i);
        }
    }
    const u64 amax = 0xFFFFFFFF00000000ull;
    for (int it = 0; it < n; it++) {
        const u64 a = it % 4 ? g() % amax : amax - 1 - g() % 3, b = it % 4 ? g() % amax : amax - 1 - (g() % 3 << 31);
        bool rare = false;
        const u64 r = reduce_lohi64(a, b, rare);
        expect("reduce_lohi64_exact", reduce_lohi64_exact(a, b), (u128)a % ZK_P + ((u128)(b % ZK_P) << 32) % ZK_P);
        if (!rare) expect("reduce_lohi64", r, (u128)a % ZK_P + ((u128)(b % ZK_P) << 32) % ZK_P);
        rare = false;
        const u64 c = a >> 22, d = b >> 22;
        const u64 q = reduce_lohi42_nc(c, d, rare);
        if (!rare) expect("reduce_lohi42_nc", q, (u128)c + ((u128)d << 32));
    }
    for (int it = 0; it < 6; it++) check_mfma_layer(g);
    row_sums<kBlock0>();
    row_sums<kBlock>();
    if (fails) return 1;
    printf("ok, %d states, %ld rare\n", n, rares);
    return 0;
}
