/*
 * mp_fast.h -- the escape loop's iteration for up to 8 words (p <= 256), and
 * for 10 whole ones (p = 320), with few branches.
 *
 * add_rn and mul_rn (mp_rn.h) skip every step that no lane of the wave needs
 * behind a wave vote: about 30 votes an iteration.  With several waves per SIMD
 * that is the cheapest form; but a vote is a compare, a scalar test and a
 * branch, 43 cycles on a wave that has its SIMD to itself against 4.5 for a
 * VALU instruction, and the frames MDZ draws (480x360 = 2700 waves on 1024
 * SIMDs, and every frame's last, longest orbits) leave a SIMD one to three
 * waves.  There an iteration of the 4-word loop took 2900 cycles, half of
 * them votes and the wait states of the carry chains.  The forms here do the same arithmetic without
 * branches and collect the conditions that need more in lane masks, tested
 * once for several operations.  Where one holds (probability about 2^-26 a
 * lane on random significands) the operations concerned are done again by
 * add_rn / mul_rn.
 *
 *   product  short product, the one-bit normalisation under the exec mask,
 *            rounding; again when the short product's window reaches a
 *            midpoint or the increment leaves the lowest word
 *   sum      both operands are shifted right by two bits of headroom plus
 *            their exponent's distance to the larger one: no swap, no carry
 *            out of the top, and the leading zeros of the sum are 1 to 31, so
 *            that one funnel shift by 32 - lz a word normalises.  The smaller
 *            magnitude of a subtraction, by its aligned top word, enters
 *            complemented, so the sum is never negative unless the top words
 *            are equal; again in that case, when the top word cancels, or
 *            when the rounding leaves the lowest word
 *   escape   sum of the squares in units of 2^-27 from the top words; again by
 *            escaped() within 4 units of the threshold
 *
 * Cycles an iteration on one wave alone / pixel rate of a full chip, interior
 * frames, add_rn and mul_rn -> these forms:
 *    64 bits   2375 -> 1272      210 -> 212 G pixel-iter/s
 *    80 bits   3517 -> 1575      141 -> 170
 *   128 bits   2928 -> 1718      135 -> 146
 *   176 bits   4369 -> 2279       89 -> 102
 *   256 bits   3967 -> 2740       83 -> 81 (frames of escaping pixels: 75 -> 78)
 * What is left is VALU issue: 309 instructions an iteration at 4 words, 39 of
 * them multiply-accumulates.  Where all lanes of a wave agree and the chip is
 * full, the votes were the cheaper form at 6 and 8 whole words: 517
 * instructions an iteration at 8 words against 541 here.  A 1920x1080 frame of
 * orbits that settle too slowly to be found periodic (300 iterations) takes
 * 5.9 ms at 192 bits and 7.9 at 256, with votes 5.7 and 7.1; frames with
 * escaping pixels gain 2 to 39 %.  add_rn in the waves whose lanes agree took
 * 6.6 and 8.0 ms.
 * An exact zero is rare here: a wave with a pixel on the real axis does its
 * iterations twice.  256x256 frames of the set, whose middle row lies there,
 * take 1.06 (64 bits), 1.34 (80), 1.23 (128) and 1.27 (256) times what they took
 * with votes; with that row elsewhere 0.5 to 0.7 times.  Telling zeros from rare
 * lanes gave most of that back, but slowed other frames by up to 2 % and, by
 * an uneven second round of waves, a 640x480 frame of escaping pixels at 128
 * bits from 12.1 to 14.5 ms.
 * At 320 bits an iteration alone takes 3,300 cycles against 4,800 (a 480x360
 * frame of a saved scene 26.1 -> 21.3 ms); the ragged 10-word kernel, whose cut
 * may lie in the second word, and those from 12 words up keep add_rn and
 * mul_rn (this form was not measured there).
 *
 * A precision of p = 32N - kclr bits with 0 <= kclr < 32 is covered: rounding
 * at bit kclr of the lowest word is one add with carry and a mask.
 *
 * Zeros keep M == 0 and an exponent of at most 2 EZF (EZF below): products
 * of zeros need no case of their own, the sums shift them out.
 */
#ifndef MDZG_MP_FAST_H
#define MDZG_MP_FAST_H

#include "mp_rn.h"

namespace mdzg {

/* word counts whose kernels use these forms */
template <int N, bool FULL>
constexpr bool rn_fast() { return N <= 8 || (N == 10 && FULL); }

/* exponent of a zero that enters an iteration: twice it, and its distance to
   any other, fit an int32 */
static constexpr int32_t EZF = -(1 << 28);

/* lane mask on the device, 0 or 1 on the host */
typedef uint64_t lanes;

MP_HD lanes lanes_of(bool c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(c);
#else
    return c ? 1u : 0u;
#endif
}

/* a | b by the scalar unit (the compiler moves masks it cannot prove uniform
   to vector registers) */
MP_HD lanes join(lanes a, lanes b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    lanes r;
    asm("s_or_b64 %0, %1, %2" : "=s"(r) : "s"(a), "s"(b) : "scc");
    return r;
#else
    return a | b;
#endif
}

template <int N>
MP_HD mp<N> again(const mp<N>& v)
{
    mp<N> r = v;
    r.e = again(v.e);
    return r;
}

/* what rounding at p = 32N - kclr bits needs of kclr (FULL: kclr = 0) */
template <bool FULL>
struct rn_prec {
    uint32_t k, half, keep;       /* kclr, 2^(kclr-1), ~(2^kclr - 1) */
};
template <>
struct rn_prec<true> {};

MP_HD void set_prec(rn_prec<true>&, int) {}
MP_HD void set_prec(rn_prec<false>& p, int kclr)
{
    p.k = (uint32_t)kclr;
    p.half = 1u << ((p.k - 1u) & 31u);
    p.keep = 0u - (p.half << 1);
}
MP_HD int kclr_of(const rn_prec<true>&) { return 0; }
MP_HD int kclr_of(const rn_prec<false>& p) { return (int)p.k; }

/* A += B, K words with a carry in and out of lane mask c, where the words of
   A and B are first exclusive-ored with mA and mB.  gfx950 needs two wait
   states between the write of a carry and its use by the next
   v_addc_co_u32; the exclusive-ors of the next word fill them. */
template <int K>
MP_HD void sum_words(uint32_t* A, uint32_t* B, uint32_t mA, uint32_t mB, lanes& c)
#if defined(__HIP_DEVICE_COMPILE__)
    ;
template <>
MP_HD void sum_words<2>(uint32_t* A, uint32_t* B, uint32_t mA, uint32_t mB, lanes& c)
{
    lanes co;
    asm("v_xor_b32 %0, %5, %0\n\t"
        "v_xor_b32 %2, %6, %2\n\t"
        "v_addc_co_u32 %0, %4, %0, %2, %7\n\t"
        "v_xor_b32 %1, %5, %1\n\t"
        "v_xor_b32 %3, %6, %3\n\t"
        "v_addc_co_u32 %1, %4, %1, %3, %4"
        : "+&v"(A[0]), "+&v"(A[1]),
          "+&v"(B[0]), "+&v"(B[1]), "=&s"(co)
        : "v"(mA), "v"(mB), "s"(c));
    c = co;
}
template <>
MP_HD void sum_words<3>(uint32_t* A, uint32_t* B, uint32_t mA, uint32_t mB, lanes& c)
{
    lanes co;
    asm("v_xor_b32 %0, %7, %0\n\t"
        "v_xor_b32 %3, %8, %3\n\t"
        "v_addc_co_u32 %0, %6, %0, %3, %9\n\t"
        "v_xor_b32 %1, %7, %1\n\t"
        "v_xor_b32 %4, %8, %4\n\t"
        "v_addc_co_u32 %1, %6, %1, %4, %6\n\t"
        "v_xor_b32 %2, %7, %2\n\t"
        "v_xor_b32 %5, %8, %5\n\t"
        "v_addc_co_u32 %2, %6, %2, %5, %6"
        : "+&v"(A[0]), "+&v"(A[1]), "+&v"(A[2]),
          "+&v"(B[0]), "+&v"(B[1]), "+&v"(B[2]), "=&s"(co)
        : "v"(mA), "v"(mB), "s"(c));
    c = co;
}
template <>
MP_HD void sum_words<4>(uint32_t* A, uint32_t* B, uint32_t mA, uint32_t mB, lanes& c)
{
    lanes co;
    asm("v_xor_b32 %0, %9, %0\n\t"
        "v_xor_b32 %4, %10, %4\n\t"
        "v_addc_co_u32 %0, %8, %0, %4, %11\n\t"
        "v_xor_b32 %1, %9, %1\n\t"
        "v_xor_b32 %5, %10, %5\n\t"
        "v_addc_co_u32 %1, %8, %1, %5, %8\n\t"
        "v_xor_b32 %2, %9, %2\n\t"
        "v_xor_b32 %6, %10, %6\n\t"
        "v_addc_co_u32 %2, %8, %2, %6, %8\n\t"
        "v_xor_b32 %3, %9, %3\n\t"
        "v_xor_b32 %7, %10, %7\n\t"
        "v_addc_co_u32 %3, %8, %3, %7, %8"
        : "+&v"(A[0]), "+&v"(A[1]), "+&v"(A[2]), "+&v"(A[3]),
          "+&v"(B[0]), "+&v"(B[1]), "+&v"(B[2]), "+&v"(B[3]), "=&s"(co)
        : "v"(mA), "v"(mB), "s"(c));
    c = co;
}
template <>
MP_HD void sum_words<5>(uint32_t* A, uint32_t* B, uint32_t mA, uint32_t mB, lanes& c)
{
    lanes co;
    asm("v_xor_b32 %0, %11, %0\n\t"
        "v_xor_b32 %5, %12, %5\n\t"
        "v_addc_co_u32 %0, %10, %0, %5, %13\n\t"
        "v_xor_b32 %1, %11, %1\n\t"
        "v_xor_b32 %6, %12, %6\n\t"
        "v_addc_co_u32 %1, %10, %1, %6, %10\n\t"
        "v_xor_b32 %2, %11, %2\n\t"
        "v_xor_b32 %7, %12, %7\n\t"
        "v_addc_co_u32 %2, %10, %2, %7, %10\n\t"
        "v_xor_b32 %3, %11, %3\n\t"
        "v_xor_b32 %8, %12, %8\n\t"
        "v_addc_co_u32 %3, %10, %3, %8, %10\n\t"
        "v_xor_b32 %4, %11, %4\n\t"
        "v_xor_b32 %9, %12, %9\n\t"
        "v_addc_co_u32 %4, %10, %4, %9, %10"
        : "+&v"(A[0]), "+&v"(A[1]), "+&v"(A[2]), "+&v"(A[3]), "+&v"(A[4]),
          "+&v"(B[0]), "+&v"(B[1]), "+&v"(B[2]), "+&v"(B[3]), "+&v"(B[4]), "=&s"(co)
        : "v"(mA), "v"(mB), "s"(c));
    c = co;
}
#else
{
    for (int j = 0; j < K; ++j) {
        uint32_t co;
        A[j] = add_cc(A[j] ^ mA, B[j] ^ mB, (uint32_t)c, co);
        c = co;
    }
}
#endif

/* sum_words over W words in blocks of at most five */
template <int W>
MP_HD void sum_chain(uint32_t* A, uint32_t* B, uint32_t mA, uint32_t mB, lanes& c)
{
    constexpr int K = W <= 5 ? W : (W <= 10 ? (W + 1) / 2 : 4);
    sum_words<K>(A, B, mA, mB, c);
    if constexpr (W > K)
        sum_chain<W - K>(A + K, B + K, mA, mB, c);
}

/* H (N+1 words) <<= 1 and e -= 1 on the lanes whose top bit is clear, under
   the exec mask: one instruction a word where a select of the shifted word
   takes two */
template <int N>
MP_HD void norm1(uint32_t* H, int32_t& e)
#if defined(__HIP_DEVICE_COMPILE__)
    ;
template <>
MP_HD void norm1<1>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %3, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %1\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %2, -1, %2\n\t"
        "s_mov_b64 exec, %3"
        : "+&v"(H[0]), "+&v"(H[1]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<2>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %4, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %2\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %3, -1, %3\n\t"
        "s_mov_b64 exec, %4"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<3>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %5, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %3\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %4, -1, %4\n\t"
        "s_mov_b64 exec, %5"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<4>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %6, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %4\n\t"
        "v_alignbit_b32 %4, %4, %3, 31\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %5, -1, %5\n\t"
        "s_mov_b64 exec, %6"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]), "+&v"(H[4]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<5>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %7, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %5\n\t"
        "v_alignbit_b32 %5, %5, %4, 31\n\t"
        "v_alignbit_b32 %4, %4, %3, 31\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %6, -1, %6\n\t"
        "s_mov_b64 exec, %7"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]), "+&v"(H[4]), "+&v"(H[5]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<6>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %8, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %6\n\t"
        "v_alignbit_b32 %6, %6, %5, 31\n\t"
        "v_alignbit_b32 %5, %5, %4, 31\n\t"
        "v_alignbit_b32 %4, %4, %3, 31\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %7, -1, %7\n\t"
        "s_mov_b64 exec, %8"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]), "+&v"(H[4]), "+&v"(H[5]), "+&v"(H[6]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<7>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %9, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %7\n\t"
        "v_alignbit_b32 %7, %7, %6, 31\n\t"
        "v_alignbit_b32 %6, %6, %5, 31\n\t"
        "v_alignbit_b32 %5, %5, %4, 31\n\t"
        "v_alignbit_b32 %4, %4, %3, 31\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %8, -1, %8\n\t"
        "s_mov_b64 exec, %9"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]), "+&v"(H[4]), "+&v"(H[5]), "+&v"(H[6]), "+&v"(H[7]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<8>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %10, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %8\n\t"
        "v_alignbit_b32 %8, %8, %7, 31\n\t"
        "v_alignbit_b32 %7, %7, %6, 31\n\t"
        "v_alignbit_b32 %6, %6, %5, 31\n\t"
        "v_alignbit_b32 %5, %5, %4, 31\n\t"
        "v_alignbit_b32 %4, %4, %3, 31\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %9, -1, %9\n\t"
        "s_mov_b64 exec, %10"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]), "+&v"(H[4]), "+&v"(H[5]), "+&v"(H[6]), "+&v"(H[7]), "+&v"(H[8]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
template <>
MP_HD void norm1<10>(uint32_t* H, int32_t& e)
{
    uint64_t sv;
    asm("s_mov_b64 %12, exec\n\t"
        "v_cmpx_le_i32 vcc, 0, %10\n\t"
        "v_alignbit_b32 %10, %10, %9, 31\n\t"
        "v_alignbit_b32 %9, %9, %8, 31\n\t"
        "v_alignbit_b32 %8, %8, %7, 31\n\t"
        "v_alignbit_b32 %7, %7, %6, 31\n\t"
        "v_alignbit_b32 %6, %6, %5, 31\n\t"
        "v_alignbit_b32 %5, %5, %4, 31\n\t"
        "v_alignbit_b32 %4, %4, %3, 31\n\t"
        "v_alignbit_b32 %3, %3, %2, 31\n\t"
        "v_alignbit_b32 %2, %2, %1, 31\n\t"
        "v_alignbit_b32 %1, %1, %0, 31\n\t"
        "v_lshlrev_b32 %0, 1, %0\n\t"
        "v_add_u32 %11, -1, %11\n\t"
        "s_mov_b64 exec, %12"
        : "+&v"(H[0]), "+&v"(H[1]), "+&v"(H[2]), "+&v"(H[3]), "+&v"(H[4]), "+&v"(H[5]), "+&v"(H[6]), "+&v"(H[7]), "+&v"(H[8]), "+&v"(H[9]), "+&v"(H[10]),
          "+&v"(e), "=&s"(sv)
        :
        : "vcc");
}
#else
{
    if (!(H[N] >> 31)) {
        for (int j = N; j >= 1; --j) H[j] = funnel_r(H[j], H[j - 1], 31u);
        H[0] <<= 1;
        e -= 1;
    }
}
#endif

/* R0 + (G > t), carry lanes to co; d = a - b and x = p ^ q fill the two wait
   states between the compare and the add */
MP_HD void round_gt(uint32_t& R0, uint32_t G, uint32_t t, int32_t& d, int32_t a, uint32_t b,
                    uint32_t& x, uint32_t p, uint32_t q, lanes& co)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_cmp_gt_u32 vcc, %4, %5\n\t"
        "v_sub_u32 %1, %6, %7\n\t"
        "v_xor_b32 %2, %8, %9\n\t"
        "v_addc_co_u32 %0, %3, 0, %0, vcc"
        : "+v"(R0), "=&v"(d), "=&v"(x), "=&s"(co)
        : "v"(G), "v"(t), "v"(a), "v"(b), "v"(p), "v"(q)
        : "vcc");
#else
    const uint32_t inc = G > t ? 1u : 0u;
    d = (int32_t)((uint32_t)a - b);
    x = p ^ q;
    R0 += inc;
    co = (inc && R0 == 0) ? 1u : 0u;
#endif
}

/* {R1, R0} + h + (z != 0) with R0 masked by keep; carry lanes to co,
   otherwise as round_gt.  The lowest word holds only 32 - kclr bits of the
   significand, so the increment leaves it too often (every 512th sum at kclr
   = 24) to leave R1 to the rare path; N == 1 has no R1. */
template <int N>
MP_HD void round_ne(uint32_t* R, uint32_t z, uint32_t h, uint32_t keep, int32_t& d, int32_t a,
                    uint32_t b, uint32_t& x, uint32_t p, uint32_t q, lanes& co)
{
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (N == 1)
        asm("v_cmp_ne_u32 vcc, 0, %4\n\t"
            "v_sub_u32 %1, %7, %8\n\t"
            "v_xor_b32 %2, %9, %10\n\t"
            "v_addc_co_u32 %0, %3, %0, %5, vcc\n\t"
            "v_and_b32 %0, %6, %0"
            : "+v"(R[0]), "=&v"(d), "=&v"(x), "=&s"(co)
            : "v"(z), "v"(h), "v"(keep), "v"(a), "v"(b), "v"(p), "v"(q)
            : "vcc");
    else
        asm("v_cmp_ne_u32 vcc, 0, %5\n\t"
            "v_sub_u32 %2, %8, %9\n\t"
            "s_nop 0\n\t"
            "v_addc_co_u32 %0, vcc, %0, %6, vcc\n\t"
            "v_xor_b32 %3, %10, %11\n\t"
            "v_and_b32 %0, %7, %0\n\t"
            "v_addc_co_u32 %1, %4, 0, %1, vcc"
            : "+&v"(R[0]), "+&v"(R[1]), "=&v"(d), "=&v"(x), "=&s"(co)
            : "v"(z), "v"(h), "v"(keep), "v"(a), "v"(b), "v"(p), "v"(q)
            : "vcc");
#else
    uint32_t c;
    R[0] = add_cc(R[0], h, z ? 1u : 0u, c) & keep;
    if (N > 1)
        R[N > 1 ? 1 : 0] = add_cc(R[N > 1 ? 1 : 0], 0u, c, c);
    d = (int32_t)((uint32_t)a - b);
    x = p ^ q;
    co = c;
#endif
}

/* R (N words, guard word G below, sticky S in {0, 1}) rounded to nearest even
   at p bits; co gets the lanes whose increment is not carried far enough */
template <int N, bool FULL>
MP_HD void round_fast(uint32_t* R, uint32_t G, uint32_t S, const rn_prec<FULL>& pr, int32_t& d,
                      int32_t a, uint32_t b, uint32_t& x, uint32_t p, uint32_t q, lanes& co)
{
    if constexpr (FULL) {
        const uint32_t o = (R[0] & 1u) | S;
        round_gt(R[0], G, 0x80000000u - o, d, a, b, x, p, q, co);
    } else {
        /* {R0 mod 2^k, G, S} + 2^(k-1) - 1 + lsb carries into bit k exactly
           where nearest even rounds up */
        const uint32_t lsb = (R[0] >> pr.k) & 1u;
        round_ne<N>(R, G | lsb | S, pr.half - 1u, pr.keep, d, a, b, x, p, q, co);
    }
}

/* as round_ne for N > 1 with z != 0 on every lane; y = v + u fills a wait
   state */
MP_HD void round_half(uint32_t& R0, uint32_t& R1, uint32_t half, uint32_t keep, uint32_t& y,
                      uint32_t v, uint32_t u, lanes& co)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm("v_add_co_u32 %0, vcc, %0, %4\n\t"
        "v_add_u32 %2, %7, %6\n\t"
        "v_and_b32 %0, %5, %0\n\t"
        "v_addc_co_u32 %1, %3, 0, %1, vcc"
        : "+&v"(R0), "+&v"(R1), "=&v"(y), "=&s"(co)
        : "v"(half), "v"(keep), "v"(v), "i"(u)
        : "vcc");
#else
    uint32_t c;
    R0 = add_cc(R0, half, 0u, c) & keep;
    R1 = add_cc(R1, 0u, c, c);
    y = v + u;
    co = c;
#endif
}

/* r = RN_p(a * b) (SQR: a * a); rare: lanes whose result may be wrong.  r
   may not be a or b. */
template <int N, bool FULL, bool SQR>
MP_HD void mul_fast(mp<N>& r, const mp<N>& a, const mp<N>& b, const rn_prec<FULL>& pr, lanes& rare)
{
    constexpr int K0 = short_col<N>();
    uint32_t H[N + 1];
    uint32_t S;
    mant_product<N, SQR, K0>(a.m, b.m, H, S);
    int32_t e = SQR ? (a.e + a.e) : (a.e + b.e);
    norm1<N>(H, e);
    lanes co;
    int32_t d;
    uint32_t s;
    const uint32_t sa = SQR ? 0u : a.s, sb = SQR ? 0u : b.s;
    if constexpr (K0 == 0) {
        round_fast<N, FULL>(H + 1, H[0], S, pr, d, 0, 0u, s, sa, sb, co);
    } else {
        /* the product lies within U units of the guard word above H: unsure
           when a midpoint is in reach (mul_rn), else its sticky bit is 1 */
        constexpr uint32_t U = 2u * N;
        if constexpr (FULL) {
            round_gt(H[1], H[0], 0x7fffffffu, d, (int32_t)0x80000000u, H[0], s, sa, sb, co);
            rare = join(rare, lanes_of((uint32_t)d < U));
        } else {
            uint32_t y;
            round_half(H[1], H[2], pr.half, pr.keep, y, H[0], U - 1u, co);
            s = sa ^ sb;
            rare = join(rare, lanes_of(y < U));
        }
    }
    rare = join(rare, co);
#pragma unroll
    for (int j = 0; j < N; ++j) r.m[j] = H[j + 1];
    r.e = e;
    r.s = SQR ? 0u : s;
}

/* N words of v, shifted right by sh (mod 32), into N+1 words */
template <int N>
MP_HD void align_words(uint32_t* X, const uint32_t* v, uint32_t sh)
{
    X[N] = v[N - 1] >> (sh & 31u);
#pragma unroll
    for (int j = N - 1; j >= 1; --j) X[j] = funnel_r(v[j], v[j - 1], sh);
    X[0] = funnel_r(v[0], 0u, sh);
}

/* X (N+1 words) shifted right by w words, S |= anything lost */
template <int N>
MP_HD void shift_words(uint32_t* X, uint32_t w, uint32_t& S)
{
    uint32_t lost = 0;
    if (wave_all((w == 0) | (w > (uint32_t)N))) {
        /* each lane's operand stays or goes as a whole */
#pragma unroll
        for (int j = 0; j <= N; ++j) {
            lost |= X[j];
            X[j] = w ? 0u : X[j];
        }
        lost = w ? lost : 0u;
    } else {
#pragma unroll
        for (int st = 0; st < stages(N + 1); ++st) {
            const int t = 1 << st;
            const bool c = (w & (uint32_t)t) != 0;
            if (wave_any(c)) {
                uint32_t l = 0;
#pragma unroll
                for (int j = 0; j < t && j <= N; ++j) l |= X[j];
#pragma unroll
                for (int j = 0; j <= N; ++j) X[j] = c ? (j + t <= N ? X[j + t] : 0u) : X[j];
                lost |= c ? l : 0u;
            }
        }
    }
    S |= lost ? 1u : 0u;
}

/* operands of a sum aligned under a common exponent e */
template <int N>
struct aligned {
    uint32_t A[N + 1], B[N + 1];
    uint32_t da, db;              /* how far each was shifted */
    int32_t e;
};

template <int N>
MP_HD void align_fast(aligned<N>& x, const mp<N>& a, const mp<N>& b)
{
    const int32_t mx = a.e > b.e ? a.e : b.e;
    x.e = mx + 2;
    x.da = (uint32_t)x.e - (uint32_t)a.e;
    x.db = (uint32_t)x.e - (uint32_t)b.e;
    align_words<N>(x.A, a.m, x.da);
    align_words<N>(x.B, b.m, x.db);
}

/* lanes whose exponents lie a word or more apart */
template <int N>
MP_HD bool is_far(const aligned<N>& x)
{
    return (x.da | x.db) >= 32u;
}

/* the words' part of the shifts: each lane's smaller operand, which near the
   real axis is b (wim^2, c_im) on every lane */
template <int N>
MP_HD void align_far(aligned<N>& x, uint32_t& S, lanes live)
{
    constexpr uint32_t MOST = 32u * (N + 1);
    const bool fa = x.da > x.db;
    const uint32_t d = fa ? x.da : x.db;
    const bool any = (lanes_of(fa) & live) != 0;
    uint32_t X[N + 1];
#pragma unroll
    for (int j = 0; j <= N; ++j) X[j] = x.B[j];
    if (any) {
#pragma unroll
        for (int j = 0; j <= N; ++j) X[j] = fa ? x.A[j] : X[j];
    }
    shift_words<N>(X, (d < MOST ? d : MOST) >> 5, S);
    if (any) {
#pragma unroll
        for (int j = 0; j <= N; ++j) {
            const uint32_t b = x.B[j];
            x.B[j] = fa ? b : X[j];
            x.A[j] = fa ? X[j] : x.A[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j <= N; ++j) x.B[j] = X[j];
    }
}

/* leading zeros of a positive x (anything for another) */
MP_HD uint32_t lead_zeros(uint32_t x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    uint32_t r;
    asm("v_ffbh_u32 %0, %1" : "=v"(r) : "v"(x));
    return r;
#else
    return clz32(x) & 31u;
#endif
}

/* r = RN_p(a + b) of the aligned operands x with signs sa and sb (NONNEG: a - b
   of nonnegative values), S a sticky bit of the smaller; rare as in mul_fast */
template <int N, bool FULL, bool NONNEG>
MP_HD void sum_fast(mp<N>& r, aligned<N>& x, uint32_t sa, uint32_t sb, uint32_t S,
                    const rn_prec<FULL>& pr, lanes& rare)
{
    const bool lt = x.A[N] < x.B[N];
    const uint32_t sub = NONNEG ? 1u : (sa ^ sb);
    /* complement the smaller operand of a subtraction; a sticky bit stands
       for the fraction that its complement does not reach */
    const uint32_t msk = 0u - sub;
    const uint32_t mA = lt ? msk : 0u;
    const uint32_t mB = msk ^ mA;
    lanes c = lanes_of(sub > S);
    sum_chain<N + 1>(x.A, x.B, mA, mB, c);
    uint32_t* T = x.A;
    /* 0 or, where the top words were equal, negative: not decided here */
    rare = join(rare, lanes_of((int32_t)T[N] <= 0));
    const uint32_t lz = lead_zeros(T[N]);
    const uint32_t sh = 32u - lz;
    uint32_t R[N];
#pragma unroll
    for (int j = N; j >= 1; --j) R[j - 1] = funnel_r(T[j], T[j - 1], sh);
    const uint32_t G = T[0] << (lz & 31u);
    lanes co;
    round_fast<N, FULL>(R, G, S, pr, r.e, x.e, lz, r.s, NONNEG ? 0u : sa, mA & 1u, co);
    rare = join(rare, co);
#pragma unroll
    for (int j = 0; j < N; ++j) r.m[j] = R[j];
}

/* RN_p(wim2 + wre2) > 4, decided from the top words in units of 2^-27 (each
   term within a unit or two of its value) unless within 4 units of the threshold
   4 + 2^(2-p) (escaped()), then in unsure.  Shifts of 5 - e clamped to 1..31:
   an exponent above 4 leaves at least 2^30 units, past any threshold. */
template <int N, bool FULL>
MP_HD lanes escaped_fast(const mp<N>& wim2, const mp<N>& wre2, const rn_prec<FULL>& pr,
                        lanes& unsure)
{
    const int32_t ai = 5 - wim2.e, ar = 5 - wre2.e;
    const uint32_t si = (uint32_t)(ai < 1 ? 1 : (ai > 31 ? 31 : ai));
    const uint32_t sr = (uint32_t)(ar < 1 ? 1 : (ar > 31 ? 31 : ar));
    const uint32_t est = (wim2.m[N - 1] >> si) + (wre2.m[N - 1] >> sr);
    uint32_t thr = 1u << 29;
    if (!FULL && N == 1)          /* p >= 30 otherwise: less than a unit */
        thr += (1u << 29) >> ((32u - (uint32_t)kclr_of(pr)) & 31u);
    unsure = join(unsure, lanes_of(est - thr + 4u <= 8u));
    return lanes_of(est > thr);
}

/* a formula's signs: wim's product loses its sign (Burning Ship), the
   squares' difference its own (Celtic, or the hybrid at odd iterations) */
struct rn_form {
    uint32_t bs;                  /* 0: |t1|, else 1                          */
    uint32_t ce;                  /* 0: |t1|, else 1                          */
    uint32_t va;                  /* 1: hybrid                                */
};

/* an operand as loaded: a zero's exponent raised to EZF.  In a sum with a zero
   c (a Julia set of c = 0) values below 2^EZF then become 0 or, in add_rn, at
   most a unit of the guard word below 2^EZF; their squares' exponents would
   otherwise pass the end of an int32 after 30 iterations. */
template <int N>
MP_HD void clamp_zero(mp<N>& v)
{
    if (is_zero<N>(v))
        v.e = EZF;
}

/* One iteration of src/frac_mandel.c:36-48 (and siblings) for the lanes of
   live: z and z^2 advance; returns the lanes that escape.  The
   votes: one for the alignment distances of the first two sums, one for
   their and the product's rare lanes, one for the distance of the third sum,
   one for everything after it. */
template <int N, bool FULL>
MP_HD lanes step_fast(mp<N>& wre, mp<N>& wim, mp<N>& wre2, mp<N>& wim2, const mp<N>& cre,
                     const mp<N>& cim, const rn_form& f, const rn_prec<FULL>& pr, int32_t wz,
                     lanes live)
{
    mp<N> t, u, w;
    lanes rare = 0;
    uint32_t su = 0, sw = 0;
    {
        aligned<N> xu, xw;
        mul_fast<N, FULL, false>(t, wre, wim, pr, rare);           /* t1 = wre * wim   */
        t.e += 1;                                                  /* t1 *= 2          */
        t.s &= f.bs;                                               /* Burning Ship     */
        align_fast<N>(xu, wre2, wim2);
        align_fast<N>(xw, t, cim);
        const lanes far = lanes_of(is_far<N>(xu) | is_far<N>(xw)) & live;
        if (far != 0) {
            if ((lanes_of(is_far<N>(xu)) & live) != 0) align_far<N>(xu, su, live);
            if ((lanes_of(is_far<N>(xw)) & live) != 0) align_far<N>(xw, sw, live);
        }
        sum_fast<N, FULL, true>(u, xu, 0u, 1u, su, pr, rare);      /* t1 = wre2 - wim2 */
        sum_fast<N, FULL, false>(w, xw, t.s, cim.s, sw, pr, rare); /* wim = t1 + c_im  */
    }
    if (__builtin_expect((rare & live) != 0, 0)) {
        mul_rn<N, false>(t, again(wre), again(wim), kclr_of(pr));
        t.e += 1;
        t.s &= f.bs;
        add_rn<N>(w, t, again(cim), 0u, kclr_of(pr));
        add_rn<N, SUB_NONNEG>(u, again(wre2), again(wim2), 1u, kclr_of(pr));
        clamp_zero<N>(w);
    }
    u.s &= f.ce ^ ((uint32_t)wz & f.va);                           /* Celtic           */
    wim = w;
    lanes rare2 = 0;
    uint32_t sr = 0;
    {
        aligned<N> xr;
        align_fast<N>(xr, u, cre);
        const lanes far = lanes_of(is_far<N>(xr)) & live;
        if (far != 0)
            align_far<N>(xr, sr, live);
        sum_fast<N, FULL, false>(wre, xr, u.s, cre.s, sr, pr, rare2);  /* wre = t1 + c_re */
    }
    mul_fast<N, FULL, true>(wim2, wim, wim, pr, rare2);            /* wim2 = wim^2     */
    mul_fast<N, FULL, true>(wre2, wre, wre, pr, rare2);            /* wre2 = wre^2     */
    lanes esc = escaped_fast<N, FULL>(wim2, wre2, pr, rare2);
    if (__builtin_expect((rare2 & live) != 0, 0)) {
        add_rn<N>(wre, again(u), again(cre), 0u, kclr_of(pr));
        clamp_zero<N>(wre);
        mul_rn<N, true>(wim2, again(wim), wim, kclr_of(pr));
        mul_rn<N, true>(wre2, again(wre), wre, kclr_of(pr));
        const double thresh = 4.0 + ldexp(1.0, 2 - (32 * N - kclr_of(pr)));
        esc = lanes_of(escaped<N>(wim2, wre2, thresh, kclr_of(pr)));
    }
    return esc;
}

}  // namespace mdzg

#endif
