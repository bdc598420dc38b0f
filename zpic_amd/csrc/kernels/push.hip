/*
 * push.hip - particle push and charge-conserving current deposit (gfx950).
 *
 * Replaces the particle loop of the reference spec_advance
 * (em2d/particles.c:1125-1259) with interpolate_fld (:1029-1071), the
 * Boris push (:1137-1192), ltrim (:1081-1084) and dep_current_zamb
 * (:773-924).  The per-particle arithmetic follows the reference operation
 * by operation; with -ffp-contract=off and IEEE division/square root the
 * new momenta, positions and cell indices are bit-identical to the
 * reference given the same fields.
 *
 * Layout of one launch: one workgroup per tile of TX x TY cells.  The
 * workgroup stages the E and B values of its window (the tile plus an H
 * cell drift margin plus the 1-below/2-above stencil) into LDS, pushes the
 * particles of its tile range with gathers from LDS, accumulates the
 * current of its window in LDS (64-bit fixed point with ds_add_u64 by
 * default, float ds_add_f32 on request), and finally stores the window to
 * its own slot of `region` with plain coalesced stores.  No two
 * workgroups write the same address, so no global atomics are needed; the
 * windows are summed into J afterwards by current.hip in a fixed order.
 *
 * A particle that has drifted more than H cells out of its tile since the
 * last sort is listed, and pushed on the global path by the same workgroup
 * after the others: gathers from the guard-inclusive field buffers exactly
 * as the reference indexes them, and deposits into the raw overflow grid
 * `Jov` with 64-bit fixed-point atomics (exact, order-free sums).  The
 * unsorted tail (particles injected by the moving window since the last
 * sort) takes the same path, in workgroups of its own.
 */
#include "push_core.h"

using namespace zk;

/* waves per SIMD of the single-species tile push: 5 allow 96 VGPRs, of which
 * it takes 85 or 86 (LWFA 4000 x 256: 0.2537 -> 0.2505 ms per step against 4
 * waves, when the 96 still left a few values spilled outside the loop) */
#ifndef ZK_PUSH_OCC
#define ZK_PUSH_OCC 5
#endif
/* waves per SIMD of the fused multi-species push: 5 allow 96 VGPRs, of which
 * it takes 87; the extra wave hides more latency (2048^2 Weibel: 5 waves
 * 1.727 ms per launch against 1.750 with 4, when the 5-wave build still
 * reloaded two spilled address terms in the loop) */
#ifndef ZK_SPECIES_OCC
#define ZK_SPECIES_OCC 5
#endif

namespace {


/* Threads per tile workgroup.  256 where the tiles fill the GPU: five such
 * workgroups share a CU's LDS and registers.  With fewer tiles than that the
 * waves of a tile decide how many the CU runs: up to one tile per CU, 1024
 * threads. */
constexpr int ZK_CUS = 256;

inline int tile_threads(int ntiles) { return ntiles <= ZK_CUS ? 1024 : ntiles <= 2 * ZK_CUS ? 512 : 256; }

/* The first global_blocks blocks push the unsorted tail (the global pass)
 * in the same launch: the two touch disjoint particles, deposit into
 * disjoint windows or with exact atomics into the overflow grid, and write
 * their own energy partials, so they may run side by side (one launch and
 * its gap less per step while a moving window's injected columns wait for a
 * sort).  They come first because each is a long chain of dependent global
 * accesses. */
template <int MIN_WAVES, int PAIR, bool FX, int WC = 0, int NT = 256>
__global__ void __launch_bounds__(NT, MIN_WAVES) push_tile_kernel(zk_push_args a)
{
    zk_stamp_first(a.stamp);
    const int b = (int)blockIdx.x - a.global_blocks;
    if (b < 0)
        push_global_body(a, blockIdx.x, a.global_blocks);
    else
        push_tile_body<PAIR, FX, OneSpecies, WC, NT>(OneSpecies{a}, zk_xcd_item(b, a.t.ntiles));
    zk_stamp_last(a.stamp);
}

/* every species of a simulation in one launch (shared staging and window) */
template <int WC, int NT>
__global__ void __launch_bounds__(NT, NT == 256 ? ZK_SPECIES_OCC : 4) push_species_kernel(zk_push_multi m)
{
    zk_stamp_first(m.s[0].stamp);
    push_tile_body<1, true, SpeciesSet, WC, NT>(SpeciesSet{m}, zk_xcd_item(blockIdx.x, m.s[0].t.ntiles));
    zk_stamp_last(m.s[0].stamp);
}

__global__ void __launch_bounds__(256) push_global_kernel(zk_push_args a)
{
    zk_stamp_first(a.stamp);
    push_global_body(a, blockIdx.x, gridDim.x);
    zk_stamp_last(a.stamp);
}

__global__ void stamp_kernel(zk_stamp st) { zk_stamp_last(st); }

/* a thread per slot: start to end of the phases of slots 0 .. n - 1 */
__global__ void __launch_bounds__(ZK_CLOCK_SLOTS) clock_fold_kernel(zk_clock *clk, int n)
{
    __shared__ unsigned long long part[ZK_CLOCK_SLOTS];
    const int k = threadIdx.x;
    unsigned long long t = 0;
    if (k < n) {
        auto &a = clk->at[k];
        unsigned long long e = 0;
        for (int x = 0; x < ZK_XCDS; x++) {
            e = max(e, a.end[x]);
            a.end[x] = 0;
        }
        if (a.start != 0 && e > a.start) t = e - a.start;
        a.start = 0;
    }
    part[k] = t;
    __syncthreads();
    if (k > 0) return;
    for (int i = 1; i < ZK_CLOCK_SLOTS; i++) t += part[i];
    clk->total += t;
}

/* one block per species */
__global__ void __launch_bounds__(1024) finalize_set_kernel(zk_finalize_set f)
{
    const int k = blockIdx.x;
    finalize_set_body(f, k);
}

/* For every float x of [first, first + n) (as bit patterns): whether
 * rcp_ge1, sqrt_ge1 and div_ge1(a, x) differ from the correctly rounded
 * results of the compiler's own division and square root. */
__global__ void rounding_kernel(unsigned first, unsigned n, float a, unsigned long long *bad)
{
    unsigned long long r = 0, s = 0, d = 0;
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float x = __uint_as_float(first + i);
        r += rcp_ge1(x) != 1.0f / x;
        s += sqrt_ge1(x) != sqrtf(x);
        d += div_ge1(a, x) != a / x;
    }
    if (r) atomicAdd(&bad[0], r);
    if (s) atomicAdd(&bad[1], s);
    if (d) atomicAdd(&bad[2], d);
}

__global__ void rescale_fx_kernel(long long *p, size_t n, int shift)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] >>= shift;
}

__global__ void fill_kernel(float *p, size_t n, float v)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

} // namespace

namespace {

typedef void (*tile_kernel)(zk_push_args);
typedef void (*species_kernel)(zk_push_multi);

template <int WC>
tile_kernel fixed_kernel(int nt)
{
    return nt == 1024  ? push_tile_kernel<4, 1, true, WC, 1024>
           : nt == 512 ? push_tile_kernel<4, 1, true, WC, 512>
                       : push_tile_kernel<ZK_PUSH_OCC, 1, true, WC, 256>;
}

template <int WC>
species_kernel set_kernel(int nt)
{
    return nt == 1024 ? push_species_kernel<WC, 1024>
           : nt == 512 ? push_species_kernel<WC, 512>
                       : push_species_kernel<WC, 256>;
}

/* windows of large tiles need more than the default 64 KiB of LDS */
int allow_lds(const void *fn, size_t lds)
{
    return lds > 65536 ? (int)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) : 0;
}

} // namespace

extern "C" int zk_push(const zk_push_args *a, zk_stream_t s)
{
    const int n = a->t.WX * a->t.WY;
    /* E, B window (6 n floats) and the current window: 3 n floats, or 3 n
     * 64-bit integers with the fixed-point deposit */
    const size_t lds = (size_t)6 * n * sizeof(float) + (size_t)3 * n * (a->fixed ? 8 : 4);
    if (a->t.ntiles > 0) {
        /* float-deposit variants: 0 lets the compiler keep every value in
         * registers (about 6 waves per SIMD); 8 asks for 8 waves per SIMD at
         * the price of a few register spills; 2 pushes two particles per
         * thread and iteration */
        const int nt = a->fixed ? tile_threads(a->t.ntiles) : 256;
        const tile_kernel fn = a->fixed ? (default_window(a->t) ? fixed_kernel<ZK_WIN_DEFAULT>(nt) : fixed_kernel<0>(nt))
                               : a->waves == 8 ? (tile_kernel)push_tile_kernel<8, 1, false>
                               : a->waves == 2 ? (tile_kernel)push_tile_kernel<1, 2, false>
                                               : (tile_kernel)push_tile_kernel<1, 1, false>;
        const int e = allow_lds((const void *)fn, lds);
        if (e) return e;
        /* the tail's blocks, then the tiles */
        hipLaunchKernelGGL(fn, dim3(a->global_blocks + a->t.ntiles), dim3(nt), lds, s, *a);
    } else if (a->global_blocks > 0) {
        hipLaunchKernelGGL(push_global_kernel, dim3(a->global_blocks), dim3(256), 0, s, *a);
    }
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_push_species(const zk_push_multi *m, zk_stream_t s)
{
    const zk_push_args *a = &m->s[0];
    if (m->n < 1 || m->n > ZK_FUSE_MAX || !a->fixed) return (int)hipErrorInvalidValue;
    const int n = a->t.WX * a->t.WY;
    const size_t lds = (size_t)6 * n * sizeof(float) + (size_t)3 * n * 8;
    if (a->t.ntiles > 0) {
        const int nt = tile_threads(a->t.ntiles);
        const species_kernel fn = default_window(a->t) ? set_kernel<ZK_WIN_DEFAULT>(nt) : set_kernel<0>(nt);
        const int e = allow_lds((const void *)fn, lds);
        if (e) return e;
        hipLaunchKernelGGL(fn, dim3(a->t.ntiles), dim3(nt), lds, s, *m);
    }
    for (int k = 0; k < m->n; k++) {
        if (m->s[k].global_blocks <= 0) continue;
        zk_push_args g = m->s[k];
        if (a->t.ntiles > 0) g.stamp.open = 0; /* the tile launch began the phase */
        hipLaunchKernelGGL(push_global_kernel, dim3(g.global_blocks), dim3(256), 0, s, g);
    }
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_spec_finalize_set(const zk_finalize_set *f, zk_stream_t s)
{
    if (f->n < 1 || f->n > ZK_FUSE_MAX) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(finalize_set_kernel, dim3(f->n), dim3(1024), 0, s, *f);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_fill_f32(float *p, size_t n, float v, zk_stream_t s)
{
    if (n == 0) return 0;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_stamp_end(zk_stamp st, zk_stream_t s)
{
    hipLaunchKernelGGL(stamp_kernel, dim3(1), dim3(64), 0, s, st);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_clock_fold(zk_clock *clk, int n, zk_stream_t s)
{
    if (n < 0 || n > ZK_CLOCK_SLOTS) return (int)hipErrorInvalidValue;
    if (n > 0) hipLaunchKernelGGL(clock_fold_kernel, dim3(1), dim3(ZK_CLOCK_SLOTS), 0, s, clk, n);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_rounding_check(unsigned first, unsigned n, float a, unsigned long long bad[3])
{
    unsigned long long *d = nullptr;
    int e = (int)hipMalloc((void **)&d, 3 * sizeof(*d));
    if (e) return e;
    e = (int)hipMemcpy(d, bad, 3 * sizeof(*d), hipMemcpyHostToDevice);
    if (!e) {
        hipLaunchKernelGGL(rounding_kernel, dim3(4096), dim3(256), 0, nullptr, first, n, a, d);
        e = (int)hipGetLastError();
    }
    if (!e) e = (int)hipMemcpy(bad, d, 3 * sizeof(*d), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return e;
}

extern "C" int zk_rescale_fx(long long *p, size_t n, int shift, zk_stream_t s)
{
    if (n == 0 || shift <= 0) return 0;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(rescale_fx_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, n, shift);
    ZK_LAUNCH_CHECK();
}
