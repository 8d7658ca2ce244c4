// Host build of the product that four lanes form (half_mul, half_join,
// half_round of mdz_amd/csrc/mp_rn.h) at every word count that k_quad.h uses
// it at, bit for bit against mul_rn: the product from its two halves, the
// squares from one.  Operands with few bits and all ones bring the short
// product's window onto midpoints (the exact path), random ones do not.
//
// usage: mp_half_selftest <seed> <cases-per-config>
#include <stdio.h>
#include <stdlib.h>

#define MDZG_CUTS_BOUNDED
#define MDZG_COUNT_SHORT_FALLBACK 1
#include "../mdz_amd/csrc/mp_rn.h"

long mdzg::mdzg_short_fallbacks = 0;
using namespace mdzg;

static uint64_t state;
static uint64_t rnd()
{
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

template <int N>
static mp<N> value(int kclr)
{
    mp<N> v;
    const int kind = (int)(rnd() % 6);
    for (int j = 0; j < N; ++j)
        v.m[j] = kind == 0 ? ~0u : (kind <= 2 ? 0u : (uint32_t)rnd());
    for (int k = 0; k < kind; ++k)
        if (kind <= 2) v.m[rnd() % N] |= 1u << (rnd() % 32);
    v.m[N - 1] |= 0x80000000u;
    if (rnd() % 16 == 0)
        for (int j = 0; j < N; ++j) v.m[j] = 0;
    for (int j = 0; j < N; ++j)
        v.m[j] &= 32 * j >= kclr ? ~0u : (32 * (j + 1) <= kclr ? 0u : ~0u << (kclr & 31));
    v.e = is_zero(v) ? EZERO : (int)(rnd() % 9) - 4;
    v.s = (uint32_t)(rnd() & 1);
    return v;
}

template <int N>
static bool same(const mp<N>& a, const mp<N>& b)
{
    for (int j = 0; j < N; ++j)
        if (a.m[j] != b.m[j]) return false;
    return is_zero(a) || (a.e == b.e && a.s == b.s);
}

static long no_exact;      // word counts whose operands never met the exact path

template <int N>
static long run(long cases)
{
    long bad = 0;
    const long before = mdzg_short_fallbacks;
    for (long i = 0; i < cases; ++i) {
        const int kclr = i % 3 == 0 ? 0 : (int)(rnd() % (32 * cut_words<N>()));
        const mp<N> a = value<N>(kclr), b = value<N>(kclr);
        limb_value<N> x, y;
        to_limbs<N>(x, a);
        to_limbs<N>(y, b);
        mp<N> r, ref;
        uint32_t H[N + 1], H3[N + 1];
        uint64_t low = 0, low3 = 0;
        half_mul<N>(x.m, y.m, 0u, ~0u, H, low);
        half_mul<N>(y.m, x.m, 0u, 0u, H3, low3);
        half_join<N>(H, low, [&](uint32_t, int j) {
            return j == -2 ? (uint32_t)low3 : (j == -1 ? (uint32_t)(low3 >> 32) : H3[j]);
        });
        half_round<N>(r, x, y, H, low, ~0u, kclr);
        mul_rn<N, false>(ref, a, b, kclr);
        if (!same(r, ref) && bad++ < 4) printf("N=%d kclr=%d product, case %ld\n", N, kclr, i);
        low = 0;
        half_mul<N>(x.m, x.m, 1u, ~0u, H, low);
        half_join<N>(H, low, [](uint32_t, int) { return 0u; });
        half_round<N>(r, x, x, H, low, ~0u, kclr);
        mul_rn<N, true>(ref, a, a, kclr);
        if (!same(r, ref) && bad++ < 4) printf("N=%d kclr=%d square, case %ld\n", N, kclr, i);
    }
    if (mdzg_short_fallbacks == before) ++no_exact;
    return bad;
}

int main(int argc, char** argv)
{
    state = argc > 1 ? strtoull(argv[1], 0, 10) : 1;
    const long c = argc > 2 ? atol(argv[2]) : 20000;
    const long bad = run<10>(c) + run<12>(c) + run<14>(c) + run<16>(c) + run<20>(c) + run<24>(c) +
                     run<28>(c) + run<32>(c);
    printf("%ld mismatches, %ld word counts without an exact product\n", bad, no_exact);
    return bad != 0 || no_exact != 0;
}
