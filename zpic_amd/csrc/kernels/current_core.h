/*
 * current_core.h - device code of the current reduction and filters, shared
 * by current.hip and the batched kernels of batch.hip.
 */
#ifndef ZK_CURRENT_CORE_H
#define ZK_CURRENT_CORE_H

#include "common.h"
#include "reduce_index.h"

namespace zk {


__device__ inline int floor_div(int a, int b)
{
    int q = a / b;
    return (a % b != 0 && ((a < 0) != (b < 0))) ? q - 1 : q;
}

/* One node by itself, for any tiling and any grid: the windows one after
 * the other.  reduce_block below is its faster form. */
__device__ inline void reduce_node(const zk_reduce_args &a, const int node)
{
    const zk_tiles &t = a.t;
    const int bw = t.nx + 3, bh = t.ny + 3;
    if (node >= bw * bh) return;
    const int i = node % bw - 1, j = node / bw - 1;
    const int ci = a.periodic_x ? zk_wrap(i, t.nx) : i;
    const int cj = a.open_y ? j : zk_wrap(j, t.ny);
    const int n = t.WX * t.WY;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    for (int ky = -1; ky <= 1; ky++) {
        if (a.open_y && ky != 0) continue;
        const int ry = cj + ky * t.ny;
        if (ry < -1 || ry > t.ny + 1) continue;
        const int ty_lo = max(0, floor_div(ry + 1 + t.H - t.WY, t.TY) + 1);
        const int ty_hi = min(t.nty - 1, floor_div(ry + 1 + t.H, t.TY));
        for (int kx = -1; kx <= 1; kx++) {
            if (!a.periodic_x && kx != 0) continue;
            const int rx = ci + kx * t.nx;
            if (rx < -1 || rx > t.nx + 1) continue;
            const int tx_lo = max(0, floor_div(rx + 1 + t.H - t.WX, t.TX) + 1);
            const int tx_hi = min(t.ntx - 1, floor_div(rx + 1 + t.H, t.TX));
            for (int ty = ty_lo; a.region && ty <= ty_hi; ty++) {
                const int v = ry - (ty * t.TY - 1 - t.H);
                for (int tx = tx_lo; tx <= tx_hi; tx++) {
                    const int u = rx - (tx * t.TX - 1 - t.H);
                    const float *w = a.region + (size_t)(tx + ty * t.ntx) * 3 * n + u + v * t.WX;
                    sx += w[0];
                    sy += w[n];
                    sz += w[2 * n];
                }
            }
            const long long *o = a.Jov + 3 * ((rx + 1) + (ry + 1) * a.nrow);
            sx += (float)o[0] * a.jov_unscale;
            sy += (float)o[1] * a.jov_unscale;
            sz += (float)o[2] * a.jov_unscale;
        }
    }
    float *out = a.J + 3 * (size_t)node;
    out[0] = sx;
    out[1] = sy;
    out[2] = sz;
}

/* The sum of reduce_node for raw node (i, j) of the buffer, for grids of at
 * least 3 x 3 cells whose windows span at most N tiles per axis (W <= N T).
 *
 * The work is a handful of loads per node, and what bounds it is their
 * latency: reduce_node walks the windows with integer divisions and waits
 * for each load before the next (10 us on grids of any size up to 256 x
 * 256).  Here the N x N candidate windows are found with one product per
 * axis, all their loads are issued together, and the sums are then taken in
 * reduce_node's order, so J is the same bit for bit: a window that does not
 * cover the node adds 0 to a sum that starts at +0.  (The images of a node
 * in turn: their loads side by side as well gain 0.3 us on 128 x 128 cells
 * and lose 1.3 on a 1500 x 128 moving window.) */
template <int N>
__device__ inline void reduce_sum(const zk_reduce_args &a, const int i, const int j, float s[3])
{
    const zk_tiles &t = a.t;
    const int fx = a.periodic_x, fy = !a.open_y;
    const int ci = !fx ? i : i < 0 ? i + t.nx : i >= t.nx ? i - t.nx : i;
    const int cj = !fy ? j : j < 0 ? j + t.ny : j >= t.ny ? j - t.ny : j;
    const float invx = 1.0f / t.TX, invy = 1.0f / t.TY;
    const int n = t.WX * t.WY;
    int rxs[2], rys[2];
    const int nix = axis_images(ci, t.nx, fx, rxs), niy = axis_images(cj, t.ny, fy, rys);
    s[0] = s[1] = s[2] = 0.0f;
    for (int gy = 0; gy < niy; gy++) {
        const int ry = gy ? rys[1] : rys[0];
        const int ky = last_tile(ry, t.H, invy);
        for (int gx = 0; gx < nix; gx++) {
            const int rx = gx ? rxs[1] : rxs[0];
            const int kx = last_tile(rx, t.H, invx);
            long long o0 = 0, o1 = 0, o2 = 0;
            if (a.jflag[(rx + 1) / ZK_RED_BX + (ry + 1) / ZK_RED_BY * zk_red_blocks_x(t.nx)]) {
                const long long *o = a.Jov + 3 * ((rx + 1) + (size_t)(ry + 1) * a.nrow);
                o0 = o[0];
                o1 = o[1];
                o2 = o[2];
            }
            if (a.region) {
                float v[N * N][3];
#pragma unroll
                for (int d = 0; d < N * N; d++) {
                    const int ty = ky - (N - 1) + d / N, tx = kx - (N - 1) + d % N;
                    const int w = window_offset(ry, t.H, t.TY, ty), u = window_offset(rx, t.H, t.TX, tx);
                    const bool ok = window_covers(ty, t.nty, w, t.WY) && window_covers(tx, t.ntx, u, t.WX);
                    const float *p = a.region + (ok ? (size_t)(tx + ty * t.ntx) * 3 * n + u + w * t.WX : 0);
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const float q = p[c * n];
                        v[d][c] = ok ? q : 0.0f;
                    }
                }
#pragma unroll
                for (int d = 0; d < N * N; d++)
#pragma unroll
                    for (int c = 0; c < 3; c++) s[c] += v[d][c];
            }
            s[0] += (float)o0 * a.jov_unscale;
            s[1] += (float)o1 * a.jov_unscale;
            s[2] += (float)o2 * a.jov_unscale;
        }
    }
}

/* Nodes [32 bx, 32 bx + 32) x [8 by, 8 by + 8) of the buffer, one thread
 * each. */
template <int N>
__device__ inline void reduce_block(const zk_reduce_args &a, const int bx, const int by)
{
    const zk_tiles &t = a.t;
    /* the other overflow grid, deposited to in the step before: its flagged
     * blocks are cleared for the next step */
    bool clear = false;
    if (a.jflag_next) {
        unsigned char *f = a.jflag_next + bx + by * zk_red_blocks_x(t.nx);
        clear = *f != 0;
        __syncthreads();
        if (clear && threadIdx.x == 0) *f = 0;
    }
    const int i = bx * ZK_RED_BX + (int)(threadIdx.x % ZK_RED_BX) - 1;
    const int j = by * ZK_RED_BY + (int)(threadIdx.x / ZK_RED_BX) - 1;
    if (i > t.nx + 1 || j > t.ny + 1) return;
    if (clear) {
        long long *z = a.Jov_next + 3 * ((size_t)(i + 1) + (size_t)(j + 1) * a.nrow);
        z[0] = z[1] = z[2] = 0;
    }
    float s[3];
    reduce_sum<N>(a, i, j, s);
    float *out = a.J + 3 * ((size_t)(i + 1) + (size_t)(j + 1) * (t.nx + 3));
    out[0] = s[0];
    out[1] = s[1];
    out[2] = s[2];
}

/* the N that reduce_sum needs (0: only reduce_node can take the grid or
 * the tiling; it reads the whole overflow grid and clears none) */
__host__ __device__ inline int reduce_span(const zk_tiles &t)
{
    if (t.nx < 3 || t.ny < 3) return 0;
    if (t.WX <= 2 * t.TX && t.WY <= 2 * t.TY) return 2;
    return t.WX <= 3 * t.TX && t.WY <= 3 * t.TY ? 3 : 0;
}

__device__ inline void stencil(float sa, float sb, const float *l, const float *m, const float *u, float *o)
{
    o[0] = sa * l[0] + sb * m[0] + sa * u[0];
    o[1] = sa * l[1] + sb * m[1] + sa * u[1];
    o[2] = sa * l[2] + sb * m[2] + sa * u[2];
}

__device__ inline void smooth_node(const float *__restrict__ in, float *__restrict__ out, int nx, int ny,
                                   int nrow, int axis, float sa, float sb, int periodic_x, const int node,
                                   const int open_y = 0)
{
    const int bw = nx + 3, bh = ny + 3;
    if (node >= bw * bh) return;
    const int i = node % bw - 1, j = node / bw - 1;
#define AT(a, b) (in + 3 * ((size_t)((a) + 1) + (size_t)((b) + 1) * nrow))
    float *o = out + 3 * (size_t)node;
    const bool ix_in = (i >= 0 && i < nx), jy_in = (j >= 0 && j < ny);
    if (axis == 0) {
        /* kernel_x: interior rows only; x guards of those rows are copies
         * unless the window moves */
        if (jy_in && (ix_in || periodic_x)) {
            const int c = ix_in ? i : zk_wrap(i, nx);
            stencil(sa, sb, AT(c - 1, j), AT(c, j), AT(c + 1, j), o);
            return;
        }
    } else if (jy_in || !open_y) {
        /* kernel_y: interior nodes; then y guards of every column copy the
         * final value of their image row (with open y boundaries the guard
         * rows keep their values, below) */
        const int c = jy_in ? j : zk_wrap(j, ny);
        if (ix_in) {
            stencil(sa, sb, AT(i, c - 1), AT(i, c), AT(i, c + 1), o);
            return;
        }
        const float *s = AT(i, c);
        o[0] = s[0];
        o[1] = s[1];
        o[2] = s[2];
        return;
    }
    const float *s = AT(i, j);
    o[0] = s[0];
    o[1] = s[1];
    o[2] = s[2];
#undef AT
}

} // namespace zk

#endif
