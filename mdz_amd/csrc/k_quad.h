#ifndef MDZG_K_QUAD_H
#define MDZG_K_QUAD_H
/*
 * k_quad.h -- four lanes a pixel for the RN loops of 10 words (ragged) and more,
 * for launches that leave most of the chip idle.
 *
 * A lane that has a pixel to itself issues one instruction per 4.5 cycles
 * however empty the chip is: 7,500 cycles an iteration at 512 bits, 16,700 at
 * 1024.  A 64x64 tile is 64 waves for 1024 SIMDs, and it takes as long as
 * 65,536 pixels do.  Here the lanes q = 0..3 of an aligned quad share a
 * pixel:
 *
 *   products   q1 squares wim, q2 squares wre, q0 and q3 form half of wre *
 *              wim each.  All run the same columns, the sums of x[i] y[k-i]
 *              over i < k-i in 29-bit limbs with (x, y) = (re, im), (im, im),
 *              (re, re), (im, re): a square doubles its sums and adds the
 *              diagonal, q0 adds the diagonal of the product, and q3's half
 *              joins q0's.
 *   sums       q0 forms wim = 2 t + c_im while q2 forms u = wre2 - wim2, then
 *              q2 forms wre = u + c_re
 *   exchange   quad_perm moves (DPP), one instruction a word
 *
 * About 0.45 of the instructions in a lane's iteration, for four times the
 * lanes: 64x64 tiles at 300, 512 and 1024 bits take 1.18, 2.48 and 8.4 ms
 * against 1.95, 4.35 and 16.7 with one lane a pixel.  Up to 32768 pixels
 * (rule and figures: mdzg_dev_quad_pays).  At that size every pixel of a
 * launch has its quad where two blocks fit a CU, as they do: the persistent
 * form then claims once, and only the slices refill.
 *
 * The loop's state between iterations: v = z (wim on q0, wre on q2) and p =
 * the products of z (2 t's product on q0, wim2 on q1, wre2 on q2).  A pixel
 * that starts, or resumes from a slice's saved z, enters as `fresh`: its
 * first pass forms the products of the z in v and leaves the sums and the
 * escape test out.
 */
#include "k_escape.h"

/* not where the one-lane loop has few votes (mp_fast.h): at 320 bits that
   takes 1.16 ms for the 256x256 pixels of a wave per SIMD, four lanes 1.24 for
   128x128 */
template <int N, bool FULL>
constexpr bool rn_quad() { return N >= 10 && !rn_fast<N, FULL>(); }

/* lane `p_q` of each quad to lane q */
template <int P0, int P1, int P2, int P3>
__device__ __forceinline__ uint32_t qperm(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, P0 | P1 << 2 | P2 << 4 | P3 << 6, 0xf, 0xf,
                                              true);
}

/* a lane's c (c_im on q0, c_re on q2): registers, or from 20 words the
   block's LDS, as c_src keeps both */
template <int N, bool LDS>
struct quad_c;
template <int N>
struct quad_c<N, false> {
    mp<N> v;
    __device__ __forceinline__ void init(uint32_t*) {}
    __device__ __forceinline__ void put(const mp<N>& c) { v = c; }
    __device__ __forceinline__ mp<N> get() const { return v; }
};
template <int N>
struct quad_c<N, true> {
    uint32_t* base;
    __device__ __forceinline__ void init(uint32_t* lds) { base = lds + threadIdx.x; }
    __device__ __forceinline__ void put(const mp<N>& c)
    {
#pragma unroll
        for (int j = 0; j < N; ++j) base[j * 256] = c.m[j];
        base[N * 256] = (uint32_t)c.e;
        base[(N + 1) * 256] = c.s;
    }
    __device__ __forceinline__ mp<N> get() const
    {
        mp<N> v;
#pragma unroll
        for (int j = 0; j < N; ++j) v.m[j] = base[j * 256];
        v.e = (int32_t)base[N * 256];
        v.s = base[(N + 1) * 256];
        return v;
    }
};

template <int N>
struct quad_state {
    mp<N> v, p;
    quad_c<N, (N >= 20)> c;
};

/* a lane's role as the numbers its code uses */
struct quad_role {
    uint32_t q;
    uint32_t dbl;    /* shift of the column sums: 1 for the squares */
    uint32_t diag;   /* all ones where the diagonal is added (not q3) */
    uint32_t join;   /* all ones where q3's half is added (q0) */
};

__device__ __forceinline__ quad_role quad_role_of()
{
    quad_role r;
    r.q = threadIdx.x & 3u;
    r.dbl = (r.q == 1 || r.q == 2) ? 1u : 0u;
    r.diag = r.q == 3 ? 0u : ~0u;
    r.join = r.q == 0 ? ~0u : 0u;
    return r;
}

/* r.p = the rounded products of z in s.v (on q3: nothing) */
template <int N>
__device__ __forceinline__ void quad_products(quad_state<N>& s, const quad_role& r, int kclr)
{
    limb_value<N> x, y;
    {
        limb_value<N> z;
        to_limbs<N>(z, s.v);
#pragma unroll
        for (int i = 0; i < limb_count<N>(); ++i) {
            x.m.l[i] = qperm<2, 0, 2, 0>(z.m.l[i]);
            y.m.l[i] = qperm<0, 0, 2, 2>(z.m.l[i]);
        }
        x.e = (int32_t)qperm<2, 0, 2, 0>((uint32_t)z.e);
        y.e = (int32_t)qperm<0, 0, 2, 2>((uint32_t)z.e);
        x.s = qperm<2, 0, 2, 0>(z.s);
        y.s = qperm<0, 0, 2, 2>(z.s);
    }
    uint32_t H[N + 1];
    uint64_t low = 0;
    half_mul<N>(x.m, y.m, r.dbl, r.diag, H, low);
    /* q0: its half and q3's */
    half_join<N>(H, low, [&](uint32_t v, int) { return qperm<3, 3, 3, 3>(v) & r.join; });
    half_round<N>(s.p, x, y, H, low, r.diag, kclr);
}

/* Up to n passes of the quads of live, fewer once none is left: the sums
   (not for fresh pixels), the products, the escape test.  As rn_run. */
template <int N, bool FULL>
__device__ __forceinline__ void quad_run(quad_state<N>& s, const quad_role& r, const rn_form& f,
                                         int kc, int32_t& wz, lanes& live, lanes& fresh, int n)
{
    const int kclr = FULL ? 0 : kc;
    for (int it = 0; it < n && live != 0; ++it) {
        const lanes go = live & ~fresh;
        wz = add_lanes(wz, scalar_copy(go));
        const bool on = (go >> __lane_id()) & 1u;
        /* q0: 2 t + c_im, q2: wre2 - wim2 */
        mp<N> b = s.c.get();
        const mp<N> cre = b;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint32_t w = qperm<1, 1, 1, 1>(s.p.m[j]);
            b.m[j] = r.q == 2 ? w : b.m[j];
        }
        {
            const uint32_t we = qperm<1, 1, 1, 1>((uint32_t)s.p.e);
            b.e = r.q == 2 ? (int32_t)we : b.e;
            b.s = r.q == 2 ? 1u : b.s;
        }
        if (on && !(r.q & 1u)) {
            mp<N> a = s.p;
            if (r.q == 0) {
                twice<N>(a);
                a.s &= f.bs;
            }
            add_rn<N>(s.v, a, b, 0u, kclr);
        }
        if (on && r.q == 2) {
            s.v.s &= f.ce ^ ((uint32_t)wz & f.va);
            mp<N> u = s.v;
            add_rn<N>(s.v, u, cre, 0u, kclr);
        }
        quad_products<N>(s, r, kclr);
        /* q2: RN(wim2 + wre2) > 4, as escaped_fast (p >= 257 here) */
        const uint32_t ti = qperm<1, 1, 1, 1>(s.p.m[N - 1]);
        const int32_t ei = (int32_t)qperm<1, 1, 1, 1>((uint32_t)s.p.e);
        const int32_t er = s.p.e;
        const int32_t ai = 5 - (ei < -64 ? -64 : ei), ar = 5 - (er < -64 ? -64 : er);
        const uint32_t si = (uint32_t)(ai < 1 ? 1 : (ai > 31 ? 31 : ai));
        const uint32_t sr = (uint32_t)(ar < 1 ? 1 : (ar > 31 ? 31 : ar));
        const uint32_t est = (ti >> si) + (s.p.m[N - 1] >> sr);
        bool esc = est > (1u << 29);
        const bool unsure = (r.q == 2) & (est - (1u << 29) + 4u <= 8u);
        if (__builtin_expect(wave_any(unsure), 0)) {
            mp<N> w, sum;
#pragma unroll
            for (int j = 0; j < N; ++j) w.m[j] = qperm<1, 1, 1, 1>(s.p.m[j]);
            w.e = ei;
            w.s = 0;
            if (unsure) {
                add_rn<N>(sum, w, s.p, 0u, kclr);
                esc = gt4<N>(sum);
            }
        }
        lanes m = lanes_of(esc & (r.q == 2)) & go;
        m |= m >> 2;
        m |= m << 1;                  /* lanes 0, 1 from 0; 2, 3 from 2 */
        live &= ~m;
        fresh = 0;
    }
}

/* lane masks: all lanes of a quad agree on active, wz, depth, ... */
template <int N, bool FULL>
__device__ __forceinline__ void quad_load(quad_state<N>& s, const quad_role& r,
                                          const mdzg_dtile& t, int row, int col,
                                          const uint32_t* state)
{
    const bool re = r.q == 2 || r.q == 3;
    const uint32_t* z = re ? t.xs + (size_t)col * MDZG_VS(N) : t.ys + (size_t)row * MDZG_VS(N);
    mp<N> c;
    load_mp<N>(c, t.family == 1 ? t.jc + (re ? 0 : MDZG_VS(N)) : z);
    s.c.put(c);
    load_mp<N>(s.v, state ? state + (re ? 0 : MDZG_VS(N)) : z);
}

template <int N, bool FULL>
__global__ __launch_bounds__(256, 2) void k_rn_quad(const mdzg_dtile* tiles, int ntiles,
                                                    uint64_t total, unsigned long long* counter,
                                                    const volatile int* cancel, int chunk)
{
    __shared__ uint32_t c_lds[N >= 20 ? (N + 2) * 256 : 1];
    const quad_role r = quad_role_of();
    quad_state<N> s;
    s.c.init(c_lds);
    set_zero<N>(s.v);
    set_zero<N>(s.p);
    bool active = false, drained = false;
    int kclr = 0;
    uint32_t round = 0;
    const uint32_t often = cancel_mask<12>(chunk);
    int32_t wz = 0, depth = 0;
    uint32_t* out = nullptr;
    rn_form fm = { 1u, 1u, 0u };
    lanes fresh = 0;
    wave_run run = { 0, 0u };
    for (;;) {
        if (!drained) {
            const bool need = !active;
            const uint64_t g0 = claim<0u>(need && r.q == 0, counter, run);
            const uint64_t g = (uint64_t)qperm<0, 0, 0, 0>((uint32_t)g0) |
                               (uint64_t)qperm<0, 0, 0, 0>((uint32_t)(g0 >> 32)) << 32;
            const bool got = need && g < total;
            fresh = lanes_of(got);
            if (got) {
                const int ti = find_tile(tiles, ntiles, g);
                const mdzg_dtile& t = tiles[ti];
                const uint32_t local = (uint32_t)(g - t.pix_begin);
                const int row = (int)(local / (uint32_t)t.ncols);
                const int col = (int)(local % (uint32_t)t.ncols);
                quad_load<N, FULL>(s, r, t, row, col, nullptr);
                fm = form_of(t.fractal);
                kclr = t.kclr;
                depth = t.depth;
                out = t.out + local;
                wz = 0;
                active = true;
                asm volatile("" ::"v"(kclr), "v"(depth), "v"(out));
            }
            drained = __any(need && g >= total);
        }
        if (!__any(active))
            break;
        const int stop = ((++round & often) == 0) ? read_cancel(cancel) : 0;
        /* passes that no lane's depth ends; a fresh pixel's first makes no
           iteration */
        const int todo = depth - wz < chunk ? depth - wz : chunk;
        const int n = __builtin_amdgcn_readfirstlane(__ockl_wfred_min_i32(
            active ? todo + (int)((fresh >> __lane_id()) & 1u) : 0x7fffffff));
        const lanes start = scalar_copy(__ballot(active));
        lanes live = start;
        quad_run<N, FULL>(s, r, fm, kclr, wz, live, fresh, n);
        const bool esc = ((start & ~live) >> __lane_id()) & 1u;
        if (active && (esc || wz >= depth)) {
            if (r.q == 0)
                put_count(out, esc ? (uint32_t)wz : 0u);
            active = false;
        }
        if (stop)
            break;
    }
}

/* Resumable slice (serving): see k_fp64_slice.  The saved state is the one
   that the one-lane slices save and resume. */
template <int N, bool FULL>
__global__ __launch_bounds__(256, 2) void k_rn_quad_slice(const mdzg_dtile* tiles, int ntiles,
                                                          uint64_t total,
                                                          unsigned long long* counter, int budget,
                                                          int lane_budget)
{
    __shared__ uint32_t c_lds[N >= 20 ? (N + 2) * 256 : 1];
    const quad_role r = quad_role_of();
    quad_state<N> s;
    s.c.init(c_lds);
    set_zero<N>(s.v);
    set_zero<N>(s.p);
    bool active = false, drained = false;
    int kclr = 0;
    int32_t wz = 0, depth = 0;
    int32_t left = 0;           /* this pixel's iterations left in the slice */
    int32_t lb = lane_budget;   /* this quad's iterations left in the slice */
    uint32_t local = 0;
    const mdzg_dtile* tp = tiles;
    rn_form fm = { 1u, 1u, 0u };
    lanes fresh = 0;
    wave_run run = { 0, 0u };
    for (;;) {
        fresh = 0;
        do {
            if (drained)
                break;
            const bool need = !active && lb > 0;
            const uint64_t g0 = claim<0u>(need && r.q == 0, counter, run);
            const uint64_t g = (uint64_t)qperm<0, 0, 0, 0>((uint32_t)g0) |
                               (uint64_t)qperm<0, 0, 0, 0>((uint32_t)(g0 >> 32)) << 32;
            bool got = need && g < total;
            if (got) {
                tp = &tiles[find_tile(tiles, ntiles, g)];
                local = (uint32_t)(g - tp->pix_begin);
                got = tp->out[local] == 0xffffffffu;
            }
            if (got) {
                const int row = (int)(local / (uint32_t)tp->ncols);
                const int col = (int)(local % (uint32_t)tp->ncols);
                wz = tp->wzs[local];
                quad_load<N, FULL>(s, r, *tp, row, col,
                                   wz == 0 ? nullptr
                                           : tp->state + (size_t)local * 4 * MDZG_VS(N));
                fm = form_of(tp->fractal);
                kclr = tp->kclr;
                depth = tp->depth;
                left = budget;
                active = true;
            }
            fresh |= lanes_of(got);
            drained = __any(need && g >= total) || !__any(lb > 0);
        } while (!__any(active));
        if (!__any(active))
            break;
        /* passes that no lane's depth or budget ends, at most about 8 */
        int32_t todo = depth - wz < 8 ? depth - wz : 8;
        todo = todo < left ? todo : left;
        todo = todo < lb ? todo : lb;
        const int n = __builtin_amdgcn_readfirstlane(__ockl_wfred_min_i32(
            active ? todo + (int)((fresh >> __lane_id()) & 1u) : 0x7fffffff));
        const int32_t wz0 = wz;
        const lanes start = scalar_copy(__ballot(active));
        lanes live = start;
        quad_run<N, FULL>(s, r, fm, kclr, wz, live, fresh, n);
        const bool esc = ((start & ~live) >> __lane_id()) & 1u;
        if (active) {
            left -= wz - wz0;
            lb -= wz - wz0;
            if (esc || wz >= depth) {
                if (r.q == 0) {
                    put_count(tp->out + local, esc ? (uint32_t)wz : 0u);
                    atomicSub(tp->remaining, 1u);
                }
                active = false;
            } else if (left == 0 || lb == 0) {
                /* z from q0 (im) and q2 (re), z^2 from q1 and q2 */
                uint32_t* st = tp->state + (size_t)local * 4 * MDZG_VS(N);
                if (!(r.q & 1u))
                    store_mp<N>(st + (r.q == 0 ? MDZG_VS(N) : 0), s.v);
                if (r.q == 1 || r.q == 2)
                    store_mp<N>(st + (r.q == 1 ? 3 : 2) * MDZG_VS(N), s.p);
                if (r.q == 0)
                    tp->wzs[local] = wz;
                active = false;
            }
        }
    }
}

#endif
