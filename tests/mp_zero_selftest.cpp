// Zeros in the RN arithmetic (mdz_amd/csrc/mp_rn.h), built with the signed
// overflow check: the escape loop's operations on the real axis and in the
// Julia set of c = 0 keep every exponent inside an int32, and a zero stays
// zero through products, sums and the escape test.
#include <stdio.h>

#define MDZG_CUTS_BOUNDED
#include "../mdz_amd/csrc/mp_fast.h"

using namespace mdzg;

template <int N>
static long run(int kclr)
{
    long bad = 0;
    for (int start = 0; start < 4; ++start) {
        mp<N> wre, wim, cre, cim, wre2, wim2, t, u;
        set_zero(wre);
        set_zero(wim);
        set_zero(cim);
        if (start & 1) wre.m[N - 1] = 0xc0000000u, wre.e = 0, wre.s = 1;   // -3/4
        cre = wre;
        if (start & 2) set_zero(cre);                                      // Julia, c = 0
        clamp_zero(wre), clamp_zero(wim), clamp_zero(cre), clamp_zero(cim);
        mul_rn<N, true>(wre2, wre, wre, kclr);
        mul_rn<N, true>(wim2, wim, wim, kclr);
        const double thresh = 4.0 + ldexp(1.0, 2 - (32 * N - kclr));
        for (int i = 0; i < 40; ++i) {
            mul_rn<N, false>(t, wre, wim, kclr);
            twice(t);
            add_rn<N>(wim, t, cim, 0u, kclr);
            add_rn<N, SUB_NONNEG>(u, wre2, wim2, 1u, kclr);
            add_rn<N>(wre, u, cre, 0u, kclr);
            mul_rn<N, true>(wim2, wim, wim, kclr);
            mul_rn<N, true>(wre2, wre, wre, kclr);
            bad += !is_zero(wim) || !is_zero(wim2) || (!(start & 1) && !is_zero(wre)) ||
                   escaped<N>(wim2, wre2, thresh, kclr);
        }
    }
    return bad;
}

template <int N>
static long both() { return run<N>(0) + run<N>(N <= 8 ? 7 : 32 * cut_words<N>() - 1); }

int main()
{
    const long bad = both<1>() + both<2>() + both<4>() + both<8>() + both<10>() + both<12>() +
                     both<16>() + both<20>() + both<24>() + both<32>();
    printf("%ld mismatches\n", bad);
    return bad != 0;
}
