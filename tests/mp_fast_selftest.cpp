// Host build of mdz_amd/csrc/mp_fast.h checked against mp_rn.h (which
// mp_selftest checks against MPFR): the whole iteration, bit for bit, over
// states at every alignment distance from 0 to past the guard word, equal and
// nearly equal operands, all-ones and few-bit significands, zeros, squares
// near the escape threshold, the four formulas, and every precision
// p = 32N - kclr with kclr < 32.
//
// usage: mp_fast_selftest <seed> <cases-per-config>
#include <stdio.h>
#include <stdlib.h>

#include "../mdz_amd/csrc/mp_fast.h"

using namespace mdzg;

static uint64_t state;
static uint64_t rnd()
{
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// a p-bit value of exponent e: random, all ones, a power of two, few bits
template <int N>
static mp<N> value(int kclr, int e)
{
    mp<N> v;
    const int kind = (int)(rnd() % 8);
    for (int j = 0; j < N; ++j)
        v.m[j] = kind == 0 ? 0xffffffffu : (kind <= 2 ? 0u : (uint32_t)rnd());
    if (kind == 2) v.m[rnd() % N] |= 1u << (rnd() % 32);
    if (kind == 3) v.m[0] = (rnd() & 1) ? 0xffffffffu : 0u;
    v.m[N - 1] |= 0x80000000u;
    v.m[0] &= 0u - (1u << kclr);
    v.e = e;
    v.s = (uint32_t)(rnd() & 1);
    if (rnd() % 32 == 0) set_zero(v), v.e = EZF;
    return v;
}

template <int N>
static bool same(const mp<N>& a, const mp<N>& b)
{
    if (is_zero(a) && is_zero(b)) return true;
    if (a.e != b.e || a.s != b.s) return false;
    for (int j = 0; j < N; ++j)
        if (a.m[j] != b.m[j]) return false;
    return true;
}

template <int N, bool FULL>
static long run(int kclr, long cases)
{
    long bad = 0;
    rn_prec<FULL> pr;
    set_prec(pr, kclr);
    for (long i = 0; i < cases; ++i) {
        const int far = (int)(rnd() % 4);
        const int span = far == 0 ? 2 : (far == 1 ? 40 : 32 * (N + 2) + 3);
        mp<N> wre = value<N>(kclr, 1 - (int)(rnd() % span)), wim = value<N>(kclr, 1 - (int)(rnd() % span));
        mp<N> cre = value<N>(kclr, 1 - (int)(rnd() % span)), cim = value<N>(kclr, 1 - (int)(rnd() % span));
        if (rnd() % 8 == 0) wim = wre;
        if (rnd() % 16 == 0) { wim = wre; wim.m[0] ^= 1u << (kclr ? kclr : (int)(rnd() % 32)); }
        // start from squares as the loop holds them
        mp<N> wre2, wim2;
        mul_rn<N, true>(wre2, wre, wre, kclr);
        mul_rn<N, true>(wim2, wim, wim, kclr);
        if (rnd() % 8 == 0) { cre = wre2; cre.s = 1; cre.e += (int)(rnd() % 3) - 1; }
        const int formula = (int)(rnd() % 4), wz = (int)(rnd() % 7) + 1;
        rn_form f = { formula == 1 ? 0u : 1u, formula == 2 ? 0u : 1u, formula == 3 ? 1u : 0u };
        mp<N> are = wre, aim = wim, are2 = wre2, aim2 = wim2;
        // several steps, so that computed values meet computed values
        for (int k = 0; k < 4; ++k) {
            mp<N> t;
            mul_rn<N, false>(t, wre, wim, kclr);
            if (formula == 1) t.s = 0;
            twice(t);
            add_rn<N>(wim, t, cim, 0u, kclr);
            add_rn<N, SUB_NONNEG>(t, wre2, wim2, 1u, kclr);
            if (formula == 2 || (formula == 3 && ((wz + k) & 1))) t.s = 0;
            add_rn<N>(wre, t, cre, 0u, kclr);
            mul_rn<N, true>(wim2, wim, wim, kclr);
            mul_rn<N, true>(wre2, wre, wre, kclr);
            add_rn<N>(t, wim2, wre2, 0u, kclr);
            const bool esc = gt4<N>(t);
            const bool got = step_fast<N, FULL>(are, aim, are2, aim2, cre, cim, f, pr, wz + k, 1) != 0;
            if (got != esc || !same(are, wre) || !same(aim, wim) || !same(are2, wre2) ||
                !same(aim2, wim2)) {
                if (bad++ < 5)
                    printf("N=%d kclr=%d case %ld step %d formula %d esc %d/%d\n", N, kclr, i, k,
                           formula, got, esc);
                break;
            }
            // past the escape, or exponents no orbit reaches (c = 0)
            if (esc || wre2.e < -100000 || wim2.e < -100000) break;
        }
    }
    return bad;
}

template <int N>
static long all(long cases)
{
    long bad = run<N, true>(0, 4 * cases);
    for (int k = 1; k < 32 && 32 * N - k >= 2; ++k) bad += run<N, false>(k, cases / 8 + 1);
    return bad;
}

int main(int argc, char** argv)
{
    state = argc > 1 ? strtoull(argv[1], 0, 10) : 1;
    const long cases = argc > 2 ? atol(argv[2]) : 20000;
    const long bad = all<1>(cases) + all<2>(cases) + all<3>(cases) + all<4>(cases) +
                     all<5>(cases) + all<6>(cases) + all<7>(cases) + all<8>(cases) +
                     run<10, true>(0, 4 * cases);
    printf("%ld mismatches\n", bad);
    return bad != 0;
}
