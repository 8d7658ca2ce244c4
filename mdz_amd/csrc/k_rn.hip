/* k_rn.hip -- the RN<N> kernels of k_escape.h for one word count, selected by
 * -DMDZG_N=<N> at compile time (one object per N, built in parallel).
 * Exports mdzg_kget_rn<N>(full, &tile, &persist, &slice) and, from 10 words up,
 * for the four-lanes-a-pixel forms mdzg_kquad_rn<N>(full, &persist, &slice) to
 * the launch table. */
#include "k_escape.h"
#include "k_quad.h"

#ifndef MDZG_N
#error "build with -DMDZG_N=<words>"
#endif

#define KGET_NAME2(n) mdzg_kget_rn##n
#define KGET_NAME(n) KGET_NAME2(n)
#define KQUAD_NAME2(n) mdzg_kquad_rn##n
#define KQUAD_NAME(n) KQUAD_NAME2(n)

#if MDZG_N >= 10
extern "C" void KQUAD_NAME(MDZG_N)(int full, const void** persist, const void** slice)
{
    *persist = *slice = nullptr;
    if (full) {
        if constexpr (rn_quad<MDZG_N, true>()) {
            *persist = (const void*)k_rn_quad<MDZG_N, true>;
            *slice = (const void*)k_rn_quad_slice<MDZG_N, true>;
        }
    } else {
        if constexpr (rn_quad<MDZG_N, false>()) {
            *persist = (const void*)k_rn_quad<MDZG_N, false>;
            *slice = (const void*)k_rn_quad_slice<MDZG_N, false>;
        }
    }
}
#endif

extern "C" void KGET_NAME(MDZG_N)(int full, const void** tile, const void** persist,
                                  const void** slice)
{
    if (full) {
        *tile = (const void*)k_rn_tile<MDZG_N, true>;
        *persist = (const void*)k_rn_persist<MDZG_N, true>;
        *slice = (const void*)k_rn_slice<MDZG_N, true>;
    } else {
        *tile = (const void*)k_rn_tile<MDZG_N, false>;
        *persist = (const void*)k_rn_persist<MDZG_N, false>;
        *slice = (const void*)k_rn_slice<MDZG_N, false>;
    }
}

