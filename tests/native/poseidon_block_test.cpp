// The blocked permutation (poseidon_permute) against the exact one
// (poseidon_permute_safe) on random and edge states, with every set of wanted
// rows; the block reductions against 128-bit arithmetic at the limits of their
// ranges; and the block tables' row sums against the limit the 64-bit sums
// need.  Prints "ok, N states, M rare".
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../zeknox_amd/csrc/poseidon.hpp"

using namespace zk;
typedef unsigned __int128 u128;

static int fails = 0;

static void expect(const char *what, u64 got, u128 want)
{
    if (gl_canon(got) != (u64)(want % ZK_P) && fails++ < 10) printf("%s: wrong value\n", what);
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
        if (!rare) expect("reduce_lohi64", r, (u128)a % ZK_P + ((u128)(b % ZK_P) << 32) % ZK_P);
        rare = false;
        const u64 c = a >> 22, d = b >> 22;
        const u64 q = reduce_lohi42_nc(c, d, rare);
        if (!rare) expect("reduce_lohi42_nc", q, (u128)c + ((u128)d << 32));
    }
    row_sums<kBlock0>();
    row_sums<kBlock>();
    if (fails) return 1;
    printf("ok, %d states, %ld rare\n", n, rares);
    return 0;
}
