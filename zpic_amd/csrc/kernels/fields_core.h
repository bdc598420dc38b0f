/*
 * fields_core.h - device code of the field kernels, shared by fields.hip
 * and the batched kernels of batch.hip.
 */
#ifndef ZK_FIELDS_CORE_H
#define ZK_FIELDS_CORE_H

#include "common.h"

namespace zk {


typedef zk_yee_k YeeK; /* (dt/2)/dx, (dt/2)/dy, dt/dx, dt/dy, dt, Mur coefficient along y */

/* shift: the step ends in a window move (em2d/emf.c:646-676): every node
 * is written one column to the left, the leftmost guard column's values
 * are dropped and raw columns nx - 1 .. nx + 1 are zeroed, as the
 * reference's shift after the step leaves them (the y guards commute with
 * the shift). */
/* Guard cells (emf_update_gc, em2d/emf.c:573-637): a node that is the
 * periodic image of guards is also written to those guards, and guards
 * with an image are written by it alone, so no copy pass follows the step
 * (a launch of 3.5-4.5 us at any grid size: 11 % of a 32 x 32 step's
 * kernels, 5 % of a vacuum step at 2000 x 512).  Tiles away from the edges
 * keep the plain store. */
/* ext: the fields the particles see, E and B plus the external ones
 * (em2d/emf.c:432-470), are written with them (a launch of 2.6 us for each
 * of the two, and one for the phase's clock, on a 97 x 61 grid). */
__device__ inline void yee_store(float *__restrict__ Eo, float *__restrict__ Bo, int nx, int nrow, int bi, int bj,
                                 const float *e, const float *b, int shift, const zk_ext &ext)
{
    for (int f = 0; f < 2; f++) {
        if (!ext.out[f]) continue;
        const size_t g = 3 * ((size_t)bi + (size_t)bj * nrow);
        for (int c = 0; c < 3; c++)
            ext.out[f][g + c] = (f ? b[c] : e[c]) + (ext.grid[f] ? ext.grid[f][g + c] : ext.uniform[f][c]);
    }
    if (shift) {
        /* buffer column bi goes to bi - 1 (raw i - 1); raw columns from
         * nx - 1 on are zero, the last one written by the last node */
        if (bi == 0) return;
        const size_t g = 3 * ((size_t)(bi - 1) + (size_t)bj * nrow);
        const bool zero = bi - 1 >= nx;
        for (int c = 0; c < 3; c++) {
            Bo[g + c] = zero ? 0.0f : b[c];
            Eo[g + c] = zero ? 0.0f : e[c];
        }
        if (bi == nx + 2)
            for (int c = 0; c < 3; c++) Bo[g + 3 + c] = Eo[g + 3 + c] = 0.0f;
        return;
    }
    const size_t g = 3 * ((size_t)bi + (size_t)bj * nrow);
    for (int c = 0; c < 3; c++) {
        Bo[g + c] = b[c];
        Eo[g + c] = e[c];
    }
}

/* One field step of R rows of the buffer from row bj0 on, by one wave: a
 * column per lane (buffer column bi), the rows in registers.  A half step of
 * B reaches one column right and one row up, the whole step of E one left
 * and one down, so the wave reads one column and row below its outputs and
 * two above; X = 1: one more row below.
 *
 * The step is a few operations per byte: what bounds it is the reads and
 * writes on large grids and the latency of one read elsewhere.  Lane shifts
 * need neither LDS nor barriers, and all loads are under way before the
 * first is used.  2000 x 512 cells: 14.3 us for 62 MB (20.3 with tiles in
 * LDS), 256 x 256: 5.4 (6.4), 2048 x 2048: 67.7 for 252 MB (73.4).
 *
 * The half and whole steps update B and E in place: a node's new value
 * depends on its own old value and on neighbours of the other field.
 *
 * open_y: first-order Mur absorbing boundaries at the y edges, after the
 * whole step of E and before the second half step of B, as the reference's
 * one-dimensional code applies them along x (em1d/emf.c:379-406, 548-561):
 * the tangential components Ex, Ez of the guard rows j = -1 and j = ny
 * become E_in(n) + S (E_in(n+1) - E_guard(n)) with E_in the adjacent
 * interior row (0, ny - 1) and S = (dt - dy) / (dt + dy); the old values
 * are read from the input buffer E, which the kernel does not write.  A wave
 * that writes row ny needs the whole step on row ny - 1: either the row is
 * one of its own or X is 1. */
template <int R, int X>
struct YeeRows {
    float e[R + 3 + X][3], b[R + 2 + X][3], jj[R + 2 + X][3]; /* row v is buffer row bj0 - 1 - X + v */

    __device__ void load(const float *__restrict__ E, const float *__restrict__ B, int nx, int ny, int nrow, int bi,
                         int bj0)
    {
#pragma unroll
        for (int v = 0; v < R + 3 + X; v++) {
            const int bj = bj0 - 1 - X + v;
            const bool in = bi >= 0 && bi < nx + 3 && bj >= 0 && bj < ny + 3;
            const size_t g = in ? 3 * ((size_t)bi + (size_t)bj * nrow) : 0;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                e[v][c] = in ? E[g + c] : 0.0f;
                if (v < R + 2 + X) b[v][c] = in ? B[g + c] : 0.0f;
            }
        }
    }

    /* J NULL: zero */
    __device__ void load_j(const float *__restrict__ J, int nx, int ny, int nrow, int bi, int bj0)
    {
#pragma unroll
        for (int v = 1; v < R + 2 + X; v++) {
            const int bj = bj0 - 1 - X + v;
            const bool in = J && bi >= 0 && bi < nx + 3 && bj >= 0 && bj < ny + 3;
            const size_t g = in ? 3 * ((size_t)bi + (size_t)bj * nrow) : 0;
#pragma unroll
            for (int c = 0; c < 3; c++) jj[v][c] = in ? J[g + c] : 0.0f;
        }
    }

    /* the step, and the R rows of lanes [l0, l0 + w), whose first holds
     * buffer column c0, to Eo and Bo */
    __device__ void step(const float *__restrict__ E, float *__restrict__ Eo, float *__restrict__ Bo, int nx, int ny,
                         int nrow, const YeeK &k, int bi, int bj0, int l0, int w, int c0, int periodic_x, int open_y,
                         int shift, const zk_ext &ext)
    {
        const int lane = __lane_id();
        const int bw = nx + 3, bh = ny + 3;
        const int i = bi - 1, j0 = bj0 - 2 - X; /* raw column, raw row of e[0] */
        const bool half_x = i >= -1 && i <= nx, whole_x = i >= 0 && i <= nx + 1;
        /* B1 = B + dt/2 * (-curl E) */
#pragma unroll
        for (int v = 0; v < R + 2 + X; v++) {
            const bool f = half_x && j0 + v >= -1 && j0 + v <= ny;
            const float ea1 = lane_above(e[v][1]), ea2 = lane_above(e[v][2]);
            const float x = b[v][0] + (-k.dty2 * (e[v + 1][2] - e[v][2]));
            const float y = b[v][1] + (k.dtx2 * (ea2 - e[v][2]));
            const float z = b[v][2] + (-k.dtx2 * (ea1 - e[v][1]) + k.dty2 * (e[v + 1][0] - e[v][0]));
            b[v][0] = f ? x : b[v][0];
            b[v][1] = f ? y : b[v][1];
            b[v][2] = f ? z : b[v][2];
        }
        /* E1 = E + dt * (curl B1 - J) */
#pragma unroll
        for (int v = 1; v < R + 2 + X; v++) {
            const bool f = whole_x && j0 + v >= 0 && j0 + v <= ny + 1;
            const float bb1 = lane_below(b[v][1]), bb2 = lane_below(b[v][2]);
            const float x = e[v][0] + ((+k.dty * (b[v][2] - b[v - 1][2])) - k.dt * jj[v][0]);
            const float y = e[v][1] + ((-k.dtx * (b[v][2] - bb2)) - k.dt * jj[v][1]);
            const float z = e[v][2] + ((+k.dtx * (b[v][1] - bb1) - k.dty * (b[v][0] - b[v - 1][0])) - k.dt * jj[v][2]);
            e[v][0] = f ? x : e[v][0];
            e[v][1] = f ? y : e[v][1];
            e[v][2] = f ? z : e[v][2];
        }
        if (open_y && (bj0 <= X || bj0 + R >= ny + 1)) {
#pragma unroll
            for (int v = 1; v < R + 2 + X; v++) {
                const int jb = j0 + v;
                if ((jb != -1 && jb != ny) || bi < 0 || bi >= bw) continue;
                const int d = jb == -1 ? 1 : -1; /* towards the interior */
                const size_t gb = 3 * ((size_t)bi + (size_t)(jb + 1) * nrow);
                const size_t gi = 3 * ((size_t)bi + (size_t)(jb + 1 + d) * nrow);
                const float up0 = e[v + 1][0], up2 = e[v + 1][2], dn0 = e[v - 1][0], dn2 = e[v - 1][2];
                e[v][0] = E[gi + 0] + k.mur_y * ((d > 0 ? up0 : dn0) - E[gb + 0]);
                e[v][2] = E[gi + 2] + k.mur_y * ((d > 0 ? up2 : dn2) - E[gb + 2]);
            }
        }
        /* rows holding guards, or nodes that guards are images of */
        const bool edge = (periodic_x && (c0 <= 2 || c0 + w > nx)) || (!open_y && (bj0 <= 2 || bj0 + R > ny));
        /* B2 = B1 + dt/2 * (-curl E1) and outputs */
#pragma unroll
        for (int v = 1 + X; v < R + 1 + X; v++) {
            const int bj = bj0 - 1 - X + v, j = bj - 1;
            const bool f = half_x && j >= -1 && j <= ny;
            const float ea1 = lane_above(e[v][1]), ea2 = lane_above(e[v][2]);
            const float x = b[v][0] + (-k.dty2 * (e[v + 1][2] - e[v][2]));
            const float y = b[v][1] + (k.dtx2 * (ea2 - e[v][2]));
            const float z = b[v][2] + (-k.dtx2 * (ea1 - e[v][1]) + k.dty2 * (e[v + 1][0] - e[v][0]));
            if (lane < l0 || lane >= l0 + w || bi >= bw || bj >= bh) continue;
            const float bn[3] = {f ? x : b[v][0], f ? y : b[v][1], f ? z : b[v][2]};
            const float en[3] = {e[v][0], e[v][1], e[v][2]};
            if (!edge) {
                yee_store(Eo, Bo, nx, nrow, bi, bj, en, bn, shift, ext);
                continue;
            }
            /* the images of an interior index c on a periodic axis of n cells:
             * c - n when that is the lower guard, c, and c + n, ... up to n + 1 */
            const bool cy = !open_y;
            if ((periodic_x && (i < 0 || i >= nx)) || (cy && (j < 0 || j >= ny))) continue;
            for (int gj = cy && j - ny >= -1 ? j - ny : j; gj <= ny + 1; gj += ny) {
                for (int gi = periodic_x && i - nx >= -1 ? i - nx : i; gi <= nx + 1; gi += nx) {
                    yee_store(Eo, Bo, nx, nrow, gi + 1, gj + 1, en, bn, shift, ext);
                    if (!periodic_x) break;
                }
                if (!cy) break;
            }
        }
    }
};

/* Unit u of the buffer: R rows by ZK_YEE_W columns, units in rows of
 * zk_yee_units_x(nx).  With open y the top units end at the last row (and
 * repeat rows of those below), which keeps rows ny - 1 and ny together. */
template <int R>
__device__ inline void yee_rows(const float *__restrict__ E, const float *__restrict__ B, const float *__restrict__ J,
                                float *__restrict__ Eo, float *__restrict__ Bo, int nx, int ny, int nrow,
                                const YeeK &k, const int u, const int periodic_x, const int open_y = 0,
                                const int shift = 0, const zk_ext &ext = zk_ext())
{
    const int ux = zk_yee_units_x(nx);
    const int c0 = u % ux * ZK_YEE_W, bi = c0 - 1 + (int)__lane_id();
    const int bj0 = open_y ? max(0, min(u / ux * R, ny + 3 - R)) : u / ux * R;
    YeeRows<R, 0> y;
    y.load(E, B, nx, ny, nrow, bi, bj0);
    y.load_j(J, nx, ny, nrow, bi, bj0);
    y.step(E, Eo, Bo, nx, ny, nrow, k, bi, bj0, 1, ZK_YEE_W, c0, periodic_x, open_y, shift, ext);
}

/* Guard nodes take the value of their image: x (unless the window moves)
 * and y (unless the y boundaries are open).  One thread per guard node. */
__device__ inline void guard_node(float *E, float *B, int nx, int ny, int nrow, int periodic_x, const int k,
                                  const int open_y = 0)
{
    const int bw = nx + 3;
    const int nrows_g = 3 * bw;       /* guard rows: j = -1, ny, ny+1 */
    const int ncols_g = 3 * ny;       /* guard columns of interior rows */
    int i, j;
    if (k < nrows_g) {
        i = k % bw - 1;
        const int r = k / bw;
        j = (r == 0) ? -1 : ny + r - 1;
    } else if (k < nrows_g + ncols_g) {
        const int q = k - nrows_g;
        const int c = q % 3;
        j = q / 3;
        i = (c == 0) ? -1 : nx + c - 1;
    } else {
        return;
    }
    const int ci = periodic_x ? zk_wrap(i, nx) : i;
    const int cj = open_y ? j : zk_wrap(j, ny);
    if (ci == i && cj == j) return;
    const size_t d = 3 * ((size_t)(i + 1) + (size_t)(j + 1) * nrow);
    const size_t s = 3 * ((size_t)(ci + 1) + (size_t)(cj + 1) * nrow);
    for (int c = 0; c < 3; c++) {
        E[d + c] = E[s + c];
        B[d + c] = B[s + c];
    }
}

} // namespace zk

#endif
