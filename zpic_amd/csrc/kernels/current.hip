/*
 * current.hip - current density after deposition (gfx950).
 *
 * zk_current_reduce turns the per-tile current windows written by the
 * push kernel (plus the raw current of out-of-window pushes) into the final
 * guard-inclusive J.  It reproduces the reference's deposit-then-fold
 * semantics (em2d/current.c:118-159): deposits are accumulated at raw
 * node positions in [-1, n+1], and every node of a periodic axis receives
 * the sum of all its periodic images, guard copies included.  Along x with
 * a moving window, and along y with open boundaries, there is no fold and
 * the raw guard columns (rows) are kept.
 * One thread per output node; contributions are summed in a fixed order,
 * so the result does not depend on scheduling.
 *
 * zk_smooth applies [sa, sb, sa] passes along x and then y with the guard
 * handling of kernel_x / kernel_y (em2d/current.c:316-413).
 */
#include "current_core.h"
#include "finalize_core.h"

using namespace zk;

namespace {

/* The first RED_FIN blocks finish the push's bookkeeping (energy and push
 * count of a.fin's species, one block each), which was a launch of its own
 * (4 us of a small grid's step) and has nothing to do with J; the others
 * take 32 x 8 nodes each, in contiguous runs per XCD like the tiles that
 * wrote the windows.  RED_FIN is 8 so that it does not shift those runs. */
constexpr int RED_FIN = 8;

template <int N>
__global__ void __launch_bounds__(256) reduce_kernel(zk_reduce_args a, int nbx, int nblocks)
{
    const int b = (int)blockIdx.x - RED_FIN;
    if (b < 0) {
        const int k = blockIdx.x;
        if (k < a.fin.n) finalize_set_body(a.fin, k);
        return;
    }
    if constexpr (N == 0) {
        reduce_node(a, b * blockDim.x + threadIdx.x);
    } else {
        const int item = zk_xcd_item(b, nblocks);
        reduce_block<N>(a, item % nbx, item / nbx);
    }
}

/* Filter passes of one launch: n1 along x, then n2 along y. */
struct SmoothPasses {
    float sa[ZK_MAX_PASSES + ZK_MAX_Y_PASSES], sb[ZK_MAX_PASSES + ZK_MAX_Y_PASSES];
    int n1, n2;
};

/* All filter passes of a step (kernel_x and kernel_y passes,
 * em2d/current.c:316-459) in one launch and in registers: a wave holds ROWS
 * rows of 64 columns, a column per lane, and applies the x passes with lane
 * shifts and the y passes along the rows.  Every pass spends one column or
 * row of margin on each side, so 64 - 2 n1 columns and ROWS - 2 n2 rows are
 * written.
 *
 * The passes are a few operations on J, which the caches hold on all but the
 * largest grids: what they cost is launches and, inside one, waiting; the
 * lane shifts need neither LDS nor barriers.  97 x 61 cells, 3 x and 3 y
 * passes: 5.1 us, where x passes in LDS and a launch per y pass took 19.3;
 * 1500 x 128, 5 x passes: 4.4 us instead of 15.4; 2048 x 2048, one of each:
 * 24.7 us for 100 MB.
 *
 * The arithmetic and guard handling are those of the passes one after the
 * other, so J is the same bit for bit.  x passes filter interior rows only,
 * and there every column of a periodic axis is the image of an interior one;
 * with a moving window, or without x passes, the guard columns keep their
 * values (after y passes of an earlier launch they are no images: y passes
 * leave them unfiltered).  y passes filter
 * interior columns only; on a periodic axis every row is the image of an
 * interior one, except that the first y pass reads the guard rows -1 and ny
 * as the x passes left them, unfiltered; with open y boundaries the guard
 * rows keep their values. */
template <int ROWS>
__global__ void __launch_bounds__(64) smooth_kernel(const float *__restrict__ in, float *__restrict__ out, int nx,
                                                    int ny, int nrow, SmoothPasses ps, int periodic_x, int open_y)
{
    const int lane = threadIdx.x;
    const int n1 = ps.n1, n2 = ps.n2;
    const bool ring = !open_y && n2 > 0; /* rows are images of interior rows */
    const int b = (int)blockIdx.x * (64 - 2 * n1) - n1 + lane, i = b - 1;
    const int r0 = (int)blockIdx.y * (ROWS - 2 * n2); /* first output buffer row */
    const int jt = r0 - 1 - n2;                       /* raw row of v[0] */
    const int c0 = ring ? zk_wrap(jt, ny) : jt;       /* and its image */
    const bool in_x = i >= 0 && i < nx;
    const bool col = b >= 0 && b < nx + 3;
    const bool images = periodic_x && n1 > 0; /* columns of inner rows are images of interior columns */
    const int bi = images ? zk_wrap(i, nx) + 1 : b;
    float v[ROWS][3];
#pragma unroll
    for (int r = 0, c = c0; r < ROWS; r++, c = ring && c + 1 == ny ? 0 : c + 1) {
        const bool inner = c >= 0 && c < ny;
        const bool ok = inner ? images || col : c >= -1 && c <= ny + 1 && col;
        const float *q = in + (ok ? 3 * ((size_t)(inner ? bi : b) + (size_t)(c + 1) * nrow) : 0);
        v[r][0] = ok ? q[0] : 0.0f;
        v[r][1] = ok ? q[1] : 0.0f;
        v[r][2] = ok ? q[2] : 0.0f;
    }
    /* the guard rows the first y pass reads, if it reaches the seam */
    float lo[3] = {0.0f, 0.0f, 0.0f}, up[3] = {0.0f, 0.0f, 0.0f};
    const bool seam = ring && (c0 == 0 || c0 + ROWS >= ny);
    if (seam && in_x) {
        const float *q = in + 3 * (size_t)b, *w = in + 3 * ((size_t)b + (size_t)(ny + 1) * nrow);
        for (int c = 0; c < 3; c++) {
            lo[c] = q[c];
            up[c] = w[c];
        }
    }
    for (int p = 0; p < n1; p++) {
        const float sa = ps.sa[p], sb = ps.sb[p];
        const bool live = periodic_x || in_x;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const float l[3] = {lane_below(v[r][0]), lane_below(v[r][1]), lane_below(v[r][2])};
            const float u[3] = {lane_above(v[r][0]), lane_above(v[r][1]), lane_above(v[r][2])};
            float o[3];
            stencil(sa, sb, l, v[r], u, o);
            const bool f = live && (ring || (jt + r >= 0 && jt + r < ny));
#pragma unroll
            for (int c = 0; c < 3; c++) v[r][c] = f ? o[c] : v[r][c];
        }
    }
    for (int p = 0; p < n2; p++) {
        const float sa = ps.sa[n1 + p], sb = ps.sb[n1 + p];
        const bool guards = p == 0 && seam;
        float below[3] = {v[0][0], v[0][1], v[0][2]};
        int cr = c0;
#pragma unroll
        for (int r = 1; r < ROWS - 1; r++) {
            cr = ring && cr + 1 == ny ? 0 : cr + 1;
            float l[3] = {below[0], below[1], below[2]}, u[3] = {v[r + 1][0], v[r + 1][1], v[r + 1][2]};
            if (guards) {
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    l[c] = cr == 0 ? lo[c] : l[c];
                    u[c] = cr == ny - 1 ? up[c] : u[c];
                }
            }
            float o[3];
            stencil(sa, sb, l, v[r], u, o);
            const bool f = in_x && (ring || (jt + r >= 0 && jt + r < ny));
#pragma unroll
            for (int c = 0; c < 3; c++) {
                below[c] = v[r][c];
                v[r][c] = f ? o[c] : v[r][c];
            }
        }
    }
    if (lane < n1 || lane >= 64 - n1 || !col) return;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        const int bj = jt + r + 1;
        if (r < n2 || r >= ROWS - n2 || bj >= ny + 3) continue;
        float *o = out + 3 * ((size_t)b + (size_t)bj * nrow);
        o[0] = v[r][0];
        o[1] = v[r][1];
        o[2] = v[r][2];
    }
}

template <int ROWS>
void smooth_launch(const float *in, float *out, int nx, int ny, int nrow, const SmoothPasses &ps, int periodic_x,
                   int open_y, hipStream_t s)
{
    const int w = 64 - 2 * ps.n1, h = ROWS - 2 * ps.n2;
    hipLaunchKernelGGL(smooth_kernel<ROWS>, dim3((nx + 3 + w - 1) / w, (ny + 3 + h - 1) / h), dim3(64), 0, s, in, out,
                       nx, ny, nrow, ps, periodic_x, open_y);
}

} // namespace

extern "C" int zk_current_clears(const zk_tiles *t) { return reduce_span(*t) != 0; }

extern "C" int zk_current_reduce(const zk_reduce_args *a, zk_stream_t s)
{
    const int span = reduce_span(a->t);
    const int nbx = zk_red_blocks_x(a->t.nx), nodes = (a->t.nx + 3) * (a->t.ny + 3);
    const int nb = span ? nbx * zk_red_blocks_y(a->t.ny) : (nodes + 255) / 256;
    const dim3 grid(RED_FIN + nb);
    if (span == 2) hipLaunchKernelGGL(reduce_kernel<2>, grid, dim3(256), 0, s, *a, nbx, nb);
    else if (span == 3) hipLaunchKernelGGL(reduce_kernel<3>, grid, dim3(256), 0, s, *a, nbx, nb);
    else hipLaunchKernelGGL(reduce_kernel<0>, grid, dim3(256), 0, s, *a, nbx, nb);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_smooth(const float *in, float *out, int nx, int ny, int nrow, int n1, int n2, const float *sa,
                         const float *sb, int periodic_x, int open_y, zk_stream_t s)
{
    if (n1 < 0 || n2 < 0 || n1 > ZK_MAX_PASSES || n2 > ZK_MAX_Y_PASSES || n1 + n2 < 1)
        return (int)hipErrorInvalidValue;
    SmoothPasses ps;
    ps.n1 = n1;
    ps.n2 = n2;
    for (int k = 0; k < n1 + n2; k++) {
        ps.sa[k] = sa[k];
        ps.sb[k] = sb[k];
    }
    /* the fewest rows a wave that leave at least `least` to write: a wave's
     * time grows with its rows, so two where the GPU has waves to spare (97 x
     * 61 cells, 3 y passes: 5.1 us with 8 rows, 9.2 with 16), four where the
     * rows of the margin are read and filtered in time that other waves could
     * use (from about 2500 waves on) */
    const int least = (size_t)(nx + 3) * (ny + 3) < (1u << 18) ? 2 : 4;
    const int rows = 2 * n2 + least;
    if (rows <= 4) smooth_launch<4>(in, out, nx, ny, nrow, ps, periodic_x, open_y, s);
    else if (rows <= 8) smooth_launch<8>(in, out, nx, ny, nrow, ps, periodic_x, open_y, s);
    else if (rows <= 16) smooth_launch<16>(in, out, nx, ny, nrow, ps, periodic_x, open_y, s);
    else smooth_launch<32>(in, out, nx, ny, nrow, ps, periodic_x, open_y, s);
    ZK_LAUNCH_CHECK();
}
