/*
 * launch.hip -- kernel table and launch wrappers called by the C host runtime.
 *
 * Kernel id: 0 = FP64; MDZG_RN_KID[i] + full for the RN kernels of word count
 * MDZG_NWORDS[i] (full = the tile precision is exactly 32N bits);
 * MDZG_KID_GMP0 + j for the GMP-path kernels of storage bucket j.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include "mdzg_dev.h"

extern "C" {
void mdzg_kget_fp64(const void** tile, const void** persist, const void** slice);
void mdzg_kget_rn1(int, const void**, const void**, const void**);
void mdzg_kget_rn2(int, const void**, const void**, const void**);
void mdzg_kget_rn3(int, const void**, const void**, const void**);
void mdzg_kget_rn4(int, const void**, const void**, const void**);
void mdzg_kget_rn5(int, const void**, const void**, const void**);
void mdzg_kget_rn6(int, const void**, const void**, const void**);
void mdzg_kget_rn7(int, const void**, const void**, const void**);
void mdzg_kget_rn8(int, const void**, const void**, const void**);
void mdzg_kget_rn10(int, const void**, const void**, const void**);
void mdzg_kget_rn12(int, const void**, const void**, const void**);
void mdzg_kget_rn14(int, const void**, const void**, const void**);
void mdzg_kget_rn16(int, const void**, const void**, const void**);
void mdzg_kget_rn20(int, const void**, const void**, const void**);
void mdzg_kget_rn24(int, const void**, const void**, const void**);
void mdzg_kget_rn28(int, const void**, const void**, const void**);
void mdzg_kget_rn32(int, const void**, const void**, const void**);
void mdzg_kquad_rn10(int, const void**, const void**);
void mdzg_kquad_rn12(int, const void**, const void**);
void mdzg_kquad_rn14(int, const void**, const void**);
void mdzg_kquad_rn16(int, const void**, const void**);
void mdzg_kquad_rn20(int, const void**, const void**);
void mdzg_kquad_rn24(int, const void**, const void**);
void mdzg_kquad_rn28(int, const void**, const void**);
void mdzg_kquad_rn32(int, const void**, const void**);
void mdzg_kget_gmp(int bucket, const void**, const void**, const void**);
const void* mdzg_kprobe_rn4(void);
const void* mdzg_kprobe_rn32(void);
}

typedef void (*kget_fn)(int, const void**, const void**, const void**);
static const kget_fn kget_rn[MDZG_NCLASS_N] = {
    mdzg_kget_rn1,  mdzg_kget_rn2,  mdzg_kget_rn3,  mdzg_kget_rn4,
    mdzg_kget_rn5,  mdzg_kget_rn6,  mdzg_kget_rn7,  mdzg_kget_rn8,
    mdzg_kget_rn10, mdzg_kget_rn12, mdzg_kget_rn14, mdzg_kget_rn16,
    mdzg_kget_rn20, mdzg_kget_rn24, mdzg_kget_rn28, mdzg_kget_rn32,
};
typedef void (*kquad_fn)(int, const void**, const void**);
static const kquad_fn kquad_rn[MDZG_NCLASS_N] = {
    nullptr,         nullptr,         nullptr,         nullptr,
    nullptr,         nullptr,         nullptr,         nullptr,
    mdzg_kquad_rn10, mdzg_kquad_rn12, mdzg_kquad_rn14, mdzg_kquad_rn16,
    mdzg_kquad_rn20, mdzg_kquad_rn24, mdzg_kquad_rn28, mdzg_kquad_rn32,
};
static const int rn_kid[MDZG_NCLASS_N] = MDZG_RN_KID_INIT;

/* RN class of an RN kernel id */
static int class_of_kid(int kid)
{
    int i = 0;
    while (i < MDZG_NCLASS_N - 1 && kid != rn_kid[i] && kid != rn_kid[i] + 1)
        ++i;
    return i;
}

/* form: 0 = per-tile, 1 = persistent, 2 = resumable slice, 3 and 4 = persistent
   and slice with four lanes a pixel (null where a kernel has none) */
static void lookup(int kid, int form, const void** f)
{
    const void* t = nullptr;
    const void* p = nullptr;
    const void* sl = nullptr;
    if (form >= 3) {
        *f = nullptr;
        if (kid == 0 || (kid >= MDZG_KID_GMP0 && kid < MDZG_KID_GMP0 + MDZG_NGMP))
            return;
        if (kquad_rn[class_of_kid(kid)])
            kquad_rn[class_of_kid(kid)]((kid - 1) & 1, &p, &sl);
        *f = form == 3 ? p : sl;
        return;
    }
    if (kid == 0)
        mdzg_kget_fp64(&t, &p, &sl);
    else if (kid >= MDZG_KID_GMP0 && kid < MDZG_KID_GMP0 + MDZG_NGMP)
        mdzg_kget_gmp(kid - MDZG_KID_GMP0, &t, &p, &sl);
    else
        kget_rn[class_of_kid(kid)]((kid - 1) & 1, &t, &p, &sl);
    *f = form == 2 ? sl : (form == 1 ? p : t);
}

/* counts to the UINT_MAX sentinel, queue counters to zero: a kernel, so
   that a graph holds no memset node */
__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        p[i] = v;
}

/* Issue-rate probes for the roofline peak: every lane runs four independent
   chains of one instruction, v_mad_u64_u32 (32x32+64, the multiply-accumulate
   of the RN products) or v_fma_f64, `iters` times.  The chains never stop on
   a data value; the result is stored so nothing is removed. */
__global__ __launch_bounds__(256) void k_probe_mad(uint32_t* out, int iters)
{
    uint64_t a0 = threadIdx.x, a1 = a0 + 1, a2 = a0 + 2, a3 = a0 + 3;
    const uint32_t x = blockIdx.x | 1u, y = threadIdx.x | 3u;
    for (int i = 0; i < iters; ++i) {
        uint64_t c0, c1, c2, c3;
        asm volatile("v_mad_u64_u32 %0, %4, %8, %9, %0\n\t"
                     "v_mad_u64_u32 %1, %5, %8, %9, %1\n\t"
                     "v_mad_u64_u32 %2, %6, %8, %9, %2\n\t"
                     "v_mad_u64_u32 %3, %7, %8, %9, %3"
                     : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "=&s"(c0), "=&s"(c1), "=&s"(c2),
                       "=&s"(c3)
                     : "v"(x), "v"(y));
    }
    out[blockIdx.x * blockDim.x + threadIdx.x] = (uint32_t)(a0 ^ a1 ^ a2 ^ a3);
}

__global__ __launch_bounds__(256) void k_probe_fma(uint32_t* out, int iters)
{
    double a0 = threadIdx.x, a1 = a0 + 1.0, a2 = a0 + 2.0, a3 = a0 + 3.0;
    const double x = 0.999999, y = 1e-9 * (blockIdx.x + 1);
    for (int i = 0; i < iters; ++i) {
        asm volatile("v_fma_f64 %0, %4, %0, %5\n\t"
                     "v_fma_f64 %1, %4, %1, %5\n\t"
                     "v_fma_f64 %2, %4, %2, %5\n\t"
                     "v_fma_f64 %3, %4, %3, %5"
                     : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
                     : "v"(x), "v"(y));
    }
    out[blockIdx.x * blockDim.x + threadIdx.x] = (uint32_t)(int)(a0 + a1 + a2 + a3);
}

static void node_init(mdzg_gnode* n, const void* f, unsigned grid, unsigned block)
{
    memset(n, 0, sizeof *n);
    n->func = f;
    n->grid = grid;
    n->block = block;
}

template <class T>
static void node_arg(mdzg_gnode* n, const T& v)
{
    static_assert(sizeof(T) <= MDZG_GNODE_BUF, "argument too large");
    const int o = (n->used + 7) & ~7;
    memcpy((char*)n->buf + o, &v, sizeof v);
    n->off[n->nargs++] = o;
    n->used = o + (int)sizeof v;
}

extern "C" {

int mdzg_dev_nkernels(void) { return MDZG_NKERNELS; }

/* Four lanes a pixel (k_quad.h) up to two of its waves per SIMD, 32768 pixels
   on 256 CUs.  Times of a deep zoom, one lane a pixel / four, up to one wave
   per SIMD of the latter (128x128) and up to two (181x181): 1024 bits 17.2 /
   8.5 and 13.2 ms, 512 bits 4.30 / 2.56 and 3.65, 300 bits 1.96 / 1.25 and
   1.70; with more (221x221) 17.9, 4.97 and 2.14 ms, slower than one lane. */
int mdzg_dev_quad_pays(int kid, uint64_t total, int ncu)
{
    if (kid < 0 || kid >= mdzg_dev_nkernels() || total > (uint64_t)ncu * 128u)
        return 0;
    const void* f;
    lookup(kid, 3, &f);
    return f != nullptr;
}

/* dynamic LDS with which a persistent launch's blocks take more than half of a
   CU's 160 KB each */
unsigned mdzg_dev_spread(int kid)
{
    const void* f;
    lookup(kid, 1, &f);
    hipFuncAttributes a;
    if (!f || hipFuncGetAttributes(&a, f) != hipSuccess)
        return 0;
    const size_t want = (size_t)81 << 10;
    return a.sharedSizeBytes < want ? (unsigned)(want - a.sharedSizeBytes) : 0u;
}

/* blocks of a persistent (slice) launch: one lane a pixel, four with quad,
   at most blocks_per_cu a CU */
int mdzg_dev_grid(uint64_t total, int quad, int ncu, int blocks_per_cu)
{
    const uint64_t want = ((quad ? 4 * total : total) + 255) / 256;
    const uint64_t cap = (uint64_t)ncu * (uint64_t)(blocks_per_cu > 0 ? blocks_per_cu : 1);
    return (int)(want < cap ? (want ? want : 1) : cap);
}

/* kind 0: v_mad_u64_u32, 1: v_fma_f64.  blocks of 256 lanes (4 waves, one
   per SIMD) per CU x ncu, iters x 4 instructions per lane; *ms the kernel
   time by HIP events on a stream of its own. */
int mdzg_dev_rate_probe(int kind, int ncu, int blocks_per_cu, int iters, double* ms)
{
    if ((kind != 0 && kind != 1) || ncu < 1 || blocks_per_cu < 1 || iters < 1 || !ms)
        return -1;
    const unsigned grid = (unsigned)ncu * (unsigned)blocks_per_cu;
    uint32_t* out = nullptr;
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = -3;
    if (hipMalloc((void**)&out, (size_t)grid * 256 * 4) == hipSuccess &&
        hipStreamCreateWithFlags(&st, hipStreamNonBlocking) == hipSuccess &&
        hipEventCreate(&e0) == hipSuccess && hipEventCreate(&e1) == hipSuccess) {
        const void* f = kind == 0 ? (const void*)k_probe_mad : (const void*)k_probe_fma;
        void* args[] = { (void*)&out, (void*)&iters };
        float t = 0.f;
        if (hipLaunchKernel(f, dim3(grid), dim3(256), args, 0, st) == hipSuccess &&   /* warm-up */
            hipEventRecord(e0, st) == hipSuccess &&
            hipLaunchKernel(f, dim3(grid), dim3(256), args, 0, st) == hipSuccess &&
            hipEventRecord(e1, st) == hipSuccess && hipStreamSynchronize(st) == hipSuccess &&
            hipEventElapsedTime(&t, e0, e1) == hipSuccess) {
            *ms = t;
            rc = 0;
        }
    }
    if (st) hipStreamSynchronize(st);
    if (e0) hipEventDestroy(e0);
    if (e1) hipEventDestroy(e1);
    if (st) hipStreamDestroy(st);
    if (out) hipFree(out);
    return rc;
}

int mdzg_dev_node_fill(mdzg_gnode* n, uint32_t* p, uint64_t count, uint32_t v)
{
    if (!n || !p || count == 0)
        return -1;
    uint64_t g = (count + 255) / 256;
    if (g > 2048)
        g = 2048;
    node_init(n, (const void*)k_fill_u32, (unsigned)g, 256);
    node_arg(n, p);
    node_arg(n, count);
    node_arg(n, v);
    return 0;
}

/* The RN loops up to 10 words read the cancel flag every 16 chunks: with at most
   32 iterations a chunk, every 512.  Nothing tuned is longer. */
static int launch_chunk(int kid, int chunk)
{
    if (kid == 0 || (kid >= MDZG_KID_GMP0 && kid < MDZG_KID_GMP0 + MDZG_NGMP) || chunk <= 32)
        return chunk;
    return class_of_kid(kid) <= 8 /* 10 words */ ? 32 : chunk;
}

int mdzg_dev_node_persist(mdzg_gnode* n, int kid, const mdzg_dtile* d_tiles, int ntiles,
                          uint64_t total, unsigned long long* d_counter, const int* d_cancel,
                          int quad, int grid, int chunk)
{
    if (!n || kid < 0 || kid >= mdzg_dev_nkernels() || ntiles <= 0 || grid <= 0 || chunk <= 0)
        return -1;
    const void* f;
    lookup(kid, quad ? 3 : 1, &f);
    if (!f)
        return -1;
    chunk = launch_chunk(kid, chunk);
    node_init(n, f, (unsigned)grid, 256);
    node_arg(n, d_tiles);
    node_arg(n, ntiles);
    node_arg(n, total);
    node_arg(n, d_counter);
    node_arg(n, d_cancel);
    node_arg(n, chunk);
    return 0;
}

int mdzg_dev_node_slice(mdzg_gnode* n, int kid, const mdzg_dtile* d_tiles, int ntiles,
                        uint64_t total, unsigned long long* d_counter, int quad, int grid,
                        int budget, int lane_budget)
{
    if (!n || kid < 0 || kid >= mdzg_dev_nkernels() || ntiles <= 0 || grid <= 0 || budget <= 0 ||
        lane_budget <= 0)
        return -1;
    const void* f;
    lookup(kid, quad ? 4 : 2, &f);
    if (!f)
        return -1;
    node_init(n, f, (unsigned)grid, 256);
    node_arg(n, d_tiles);
    node_arg(n, ntiles);
    node_arg(n, total);
    node_arg(n, d_counter);
    node_arg(n, budget);
    node_arg(n, lane_budget);
    return 0;
}

int mdzg_dev_occupancy(int kid, int persist)
{
    if (kid < 0 || kid >= mdzg_dev_nkernels())
        return 0;
    const void* f;
    lookup(kid, persist, &f);
    int nb = 0;
    if (!f)
        return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 256, 0) != hipSuccess)
        return 0;
    return nb;
}

int mdzg_dev_launch_tile(int kid, const mdzg_dtile* d_tile, uint32_t npix, hipStream_t st)
{
    if (kid < 0 || kid >= mdzg_dev_nkernels() || npix == 0)
        return -1;
    const void* f;
    lookup(kid, 0, &f);
    void* args[] = { (void*)&d_tile };
    return hipLaunchKernel(f, dim3((npix + 255u) / 256u), dim3(256), args, 0, st) == hipSuccess
               ? 0 : -3;
}

/* the per-operation probe of the RN kernel of nwords (4 or 32) words, one
   lane per pixel of the tile */
int mdzg_dev_launch_op_probe(int nwords, const mdzg_dtile* d_tile, uint32_t npix, int op,
                             int warm, int reps, hipStream_t st)
{
    const void* f = nwords == 4 ? mdzg_kprobe_rn4() : (nwords == 32 ? mdzg_kprobe_rn32() : nullptr);
    if (!f || npix == 0 || op < 0 || op >= MDZG_NOPP)
        return -1;
    void* args[] = { (void*)&d_tile, (void*)&op, (void*)&warm, (void*)&reps };
    return hipLaunchKernel(f, dim3((npix + 255u) / 256u), dim3(256), args, 0, st) == hipSuccess
               ? 0 : -3;
}

int mdzg_dev_launch_persist(int kid, const mdzg_dtile* d_tiles, int ntiles, uint64_t total,
                            unsigned long long* d_counter, const int* d_cancel, int quad,
                            int grid, int chunk, hipStream_t st)
{
    if (kid < 0 || kid >= mdzg_dev_nkernels() || ntiles <= 0 || grid <= 0 || chunk <= 0)
        return -1;
    const void* f;
    lookup(kid, quad ? 3 : 1, &f);
    if (!f)
        return -1;
    chunk = launch_chunk(kid, chunk);
    void* args[] = { (void*)&d_tiles, (void*)&ntiles, (void*)&total, (void*)&d_counter,
                     (void*)&d_cancel, (void*)&chunk };
    return hipLaunchKernel(f, dim3(grid), dim3(256), args, 0, st) == hipSuccess ? 0 : -3;
}

int mdzg_dev_occupancy_slice(int kid)
{
    if (kid < 0 || kid >= mdzg_dev_nkernels())
        return 0;
    const void* f;
    lookup(kid, 2, &f);
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 256, 0) != hipSuccess)
        return 0;
    return nb;
}

} /* extern "C" */
