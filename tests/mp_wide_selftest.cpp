// Host build of the wide RN arithmetic of mdz_amd/csrc/mp_rn.h as the kernels
// compile it (MDZG_CUTS_BOUNDED): products in 29-bit limbs and the rounding
// at a cut in the lowest words, bit for bit against a schoolbook product and
// a rounding done bit by bit.  Operands with few bits and all ones bring the
// short product's window onto midpoints and run the increment through every
// word.
//
// usage: mp_wide_selftest <seed> <cases-per-config>
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

// P (L words, top bit set) rounded to nearest even at p bits into N words
template <int N>
static void round_ref(const uint32_t* P, int L, int p, uint32_t* R, int& e)
{
    const int cut = 32 * L - p;                  // bits below the kept part
    auto bit = [&](int i) { return (P[i >> 5] >> (i & 31)) & 1u; };
    bool low = false;
    for (int i = 0; i < cut - 1; ++i) low |= bit(i);
    const bool up = cut > 0 && bit(cut - 1) && (low || bit(cut));
    uint64_t c = up ? 1 : 0;
    uint32_t Q[2 * N + 2];
    for (int j = 0; j < L; ++j) {
        uint32_t keep = 32 * j >= cut ? ~0u : (32 * (j + 1) <= cut ? 0u : ~0u << (cut & 31));
        uint64_t t = (uint64_t)(P[j] & keep);
        if (up && j == cut >> 5) t += (uint64_t)1 << (cut & 31);
        else if (j > cut >> 5) t += c;
        Q[j] = (uint32_t)t;
        c = j >= cut >> 5 ? t >> 32 : 0;
    }
    if (c) {
        Q[L - 1] = 0x80000000u;
        e += 1;
    }
    for (int j = 0; j < N; ++j) R[j] = Q[L - N + j];
}

template <int N>
static mp<N> value(int kclr)
{
    mp<N> v;
    const int kind = (int)(rnd() % 6);
    for (int j = 0; j < N; ++j)
        v.m[j] = kind == 0 ? ~0u : (kind <= 3 ? 0u : (uint32_t)rnd());
    for (int k = 0; kind > 0 && kind < kind % 4 * 2 && k < kind; ++k)
        v.m[rnd() % N] |= 1u << (rnd() % 32);
    v.m[N - 1] |= 0x80000000u;
    for (int j = 0; j < N; ++j)
        v.m[j] &= 32 * j >= kclr ? ~0u : (32 * (j + 1) <= kclr ? 0u : ~0u << (kclr & 31));
    v.e = (int)(rnd() % 9) - 4;
    v.s = (uint32_t)(rnd() & 1);
    return v;
}

template <int N>
static long run(long cases)
{
    long bad = 0;
    const int most = N <= 8 ? 31 : 32 * cut_words<N>() - 1;
    for (long i = 0; i < cases; ++i) {
        const int kclr = i % 3 == 0 ? 0 : (int)(rnd() % (most + 1)), p = 32 * N - kclr;
        const mp<N> a = value<N>(kclr), b = i % 4 ? value<N>(kclr) : a;
        uint32_t P[2 * N] = { 0 };
        for (int x = 0; x < N; ++x) {
            uint64_t c = 0;
            for (int y = 0; y < N; ++y) {
                const uint64_t t = (uint64_t)a.m[x] * b.m[y] + P[x + y] + c;
                P[x + y] = (uint32_t)t;
                c = t >> 32;
            }
            P[x + N] = (uint32_t)c;
        }
        int e = a.e + b.e;
        if (!(P[2 * N - 1] >> 31)) {
            for (int j = 2 * N - 1; j > 0; --j) P[j] = P[j] << 1 | P[j - 1] >> 31;
            P[0] <<= 1;
            e -= 1;
        }
        mp<N> r;
        if (i % 4)
            mul_rn<N, false>(r, a, b, kclr);
        else
            mul_rn<N, true>(r, a, a, kclr);
        uint32_t R[N];
        round_ref<N>(P, 2 * N, p, R, e);
        bool ok = r.e == e;
        for (int j = 0; j < N; ++j) ok = ok && r.m[j] == R[j];
        if (!ok && bad++ < 4) printf("N=%d kclr=%d product, case %ld\n", N, kclr, i);
        // a value in limbs and back
        if constexpr (limb_product<N>()) {
            limb_value<N> l;
            mp<N> w;
            to_limbs<N>(l, a);
            from_limbs<N>(w, l);
            for (int j = 0; j < N; ++j)
                if (w.m[j] != a.m[j] && bad++ < 4) printf("N=%d limbs, case %ld\n", N, i);
        }
        // rounding alone: random words, guard word and sticky bit
        if (kclr) {
            uint32_t X[N + 2], Y[N], G = (rnd() & 3) ? (uint32_t)rnd() : 0u, S = (uint32_t)(rnd() & 1);
            const mp<N> v = value<N>(0);
            X[0] = S;
            X[1] = G;
            for (int j = 0; j < N; ++j) X[j + 2] = Y[j] = v.m[j];
            int e1 = 0, e2 = 0;
            round_masked<N>(Y, G, S, e1, kclr);
            round_ref<N>(X, N + 2, p, R, e2);
            ok = e1 == e2;
            for (int j = 0; j < N; ++j) ok = ok && Y[j] == R[j];
            if (!ok && bad++ < 4) printf("N=%d kclr=%d rounding, case %ld\n", N, kclr, i);
        }
    }
    return bad;
}

int main(int argc, char** argv)
{
    state = argc > 1 ? strtoull(argv[1], 0, 10) : 1;
    const long c = argc > 2 ? atol(argv[2]) : 20000;
    const long bad = run<1>(c) + run<4>(c) + run<8>(c) + run<10>(c) + run<16>(c) + run<20>(c) +
                     run<24>(c) + run<28>(c) + run<32>(c);
    printf("%ld mismatches, %ld exact products\n", bad, mdzg_short_fallbacks);
    return bad != 0;
}
