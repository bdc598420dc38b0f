/*
 * fields.hip - Yee field solver and field bookkeeping (gfx950).
 *
 * zk_yee fuses the three half/whole steps of the reference emf_advance
 * (em2d/emf.c:688-698): B += dt/2 curl E over i,j in [-1,n] (yee_b,
 * :500-522), E += dt (curl B - J) over [0,n+1] (yee_e, :531-562), and
 * B += dt/2 curl E again, into one pass with rows in registers.  Each node
 * is computed with the reference's expressions and update ranges, so with
 * the same J the result is bit-identical.  Inputs and outputs are distinct
 * buffers (the host swaps them).  The guard cells of the outputs are
 * written by the nodes they are images of (emf_update_gc, :573-637), and
 * with external fields the same pass writes the fields seen by particles
 * (emf_update_part_fld, :838-914).  zk_field_step folds and filters the
 * current in the same launch (current.hip's kernels on their own).
 *
 * zk_field_guards copies guard cells from their periodic images on its own
 * (grids edited outside the step); zk_move_window shifts the grid one cell left
 * and clears the last columns (emf_move_window, :648-675); zk_add_ext
 * forms the fields seen by particles on its own (grids edited outside the
 * step);
 * zk_emf_energy sums E_c^2 and B_c^2 in FP64 (emf_get_energy, :729-750);
 * zk_charge deposits the CIC charge density (spec_deposit_charge,
 * em2d/particles.c:1289-1324, before its boundary fold).
 */
#include <mutex>

#include "current_core.h"
#include "fields_core.h"
#include "finalize_core.h"

using namespace zk;

/* Scratch of spec_deposit_charge_noalloc: the deposit (first half) and the
 * caller's density (second half), ZK_NOALLOC_CHARGE_MAX nodes each.  Every
 * device holds its own copy for the life of the process. */
static __device__ __align__(256) float scratch[2 * ZK_NOALLOC_CHARGE_MAX];

namespace {

template <int R, bool EXT>
__global__ void __launch_bounds__(256) yee_kernel(const float *__restrict__ E, const float *__restrict__ B,
                                                  const float *__restrict__ J, float *__restrict__ Eo,
                                                  float *__restrict__ Bo, int nx, int ny, int nrow, YeeK k,
                                                  int periodic_x, int open_y, int shift, int units, zk_ext ext,
                                                  zk_stamp st)
{
    zk_stamp_first(st);
    /* contiguous runs of units per XCD: neighbours share their margins in L2 */
    const int u = zk_xcd_item(blockIdx.x, gridDim.x) * (blockDim.x / 64) + threadIdx.x / 64;
    if (u < units) yee_rows<R>(E, B, J, Eo, Bo, nx, ny, nrow, k, u, periodic_x, open_y, shift, EXT ? ext : zk_ext());
    /* the units are alike: the last end with the last */
    if (blockIdx.x + 512 >= gridDim.x) zk_stamp_last_waves(st);
}

/* Waves of a workgroup of field_step_kernel, a staged row each, and the rows
 * that leaves to write: fewer waves start sooner, more spend fewer on the
 * rows of the margin. */
__host__ __device__ inline int field_rows(int waves, int n2, int open_y) { return waves - 1 - open_y - 2 * n2; }
inline int field_waves(int n2, int open_y) { return field_rows(8, n2, open_y) >= 4 ? 8 : 16; }
__host__ __device__ inline int field_cols(int n1) { return 64 - (n1 > 1 ? n1 : 1) - (n1 > 1 ? n1 + 1 : 2); }

/* Current fold, filter passes and field step in one launch, bit for bit the
 * separate kernels' results.
 *
 * On grids of up to a few hundred cells a side each of those kernels takes 4
 * to 6 us, of which its loads and arithmetic are a fraction: the rest is
 * starting, waiting for one chain of loads and draining, and about 3.5 us
 * pass between two launches.  Here the chains run once and side by side: a
 * wave starts the loads of E and B, sums the windows for its row of J (a
 * column per lane), filters along x by lane shifts, along y through LDS, and
 * takes the field step of its row.  Rows and columns of the margins are
 * computed by every workgroup that needs them, which is why larger grids
 * keep the separate launches.  32 x 32 cells: 8.9 us for fold and step, 11.7
 * and a gap in two launches; 256 x 256, a pass each way: 10.0 us, 16.1 and
 * two gaps in three; 1500 x 128, 5 x passes: 12.3 us instead of 15.9.
 *
 * Workgroups in order: one per species whose push is to be finished, those
 * that clear the flagged blocks of the next overflow grid (a wave per
 * block), and the field_cols x field_rows units of the buffer.
 *
 * The passes' guard handling is smooth_kernel's; the raw guard rows that the
 * first y pass reads equal their images' raw rows (both are folded alike),
 * which the neighbouring waves hold. */
template <int N, int X>
__global__ void __launch_bounds__(1024) field_step_kernel(zk_field_args f)
{
    extern __shared__ float fs[];
    const int waves = blockDim.x / 64, lane = threadIdx.x % 64;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
    int u = (int)blockIdx.x - f.r.fin.n;
    if (u < 0) {
        finalize_set_body(f.r.fin, blockIdx.x);
        return;
    }
    const int nx = f.r.t.nx, ny = f.r.t.ny, nrow = f.r.nrow;
    if (u < f.clears) {
        const int nbx = zk_red_blocks_x(nx), b = u * waves + w;
        if (b >= nbx * zk_red_blocks_y(ny) || !f.r.jflag_next[b]) return;
        for (int k = lane; k < ZK_RED_BX * ZK_RED_BY; k += 64) {
            const int bi = b % nbx * ZK_RED_BX + k % ZK_RED_BX, bj = b / nbx * ZK_RED_BY + k / ZK_RED_BX;
            if (bi >= nx + 3 || bj >= ny + 3) continue;
            long long *z = f.r.Jov_next + 3 * ((size_t)bi + (size_t)bj * nrow);
            z[0] = z[1] = z[2] = 0;
        }
        if (lane == 0) f.r.jflag_next[b] = 0;
        return;
    }
    u -= f.clears;
    const int n1 = f.n1, n2 = f.n2, px = f.r.periodic_x, oy = f.r.open_y;
    const int l0 = n1 > 1 ? n1 : 1, cols = field_cols(n1), rows = field_rows(waves, n2, X);
    const int ux = (nx + 3 + cols - 1) / cols;
    const int c0 = u % ux * cols, bi = c0 - l0 + lane, i = bi - 1;
    const int r0 = u / ux * rows;            /* first buffer row to write */
    const int j = r0 - 1 - n2 - X + w;       /* this wave's raw row */
    const bool ring = !oy && n2 > 0;         /* rows are images of interior rows */
    const int cr = ring ? zk_wrap(j, ny) : j;
    const bool inner = cr >= 0 && cr < ny, in_x = i >= 0 && i < nx, col = bi >= 0 && bi < nx + 3;
    const bool out = w >= n2 + X && w < n2 + X + rows && j + 1 < ny + 3;
    YeeRows<1, X> y;
    if (out) y.load(f.E, f.B, nx, ny, nrow, bi, j + 1);
    float s[3] = {0.0f, 0.0f, 0.0f};
    if (inner ? px || col : cr >= -1 && cr <= ny + 1 && col)
        reduce_sum<N>(f.r, inner && px ? zk_wrap(i, nx) : i, cr, s);
    /* LDS: the rows before the x passes (for the first y pass), then two
     * buffers in turn */
    const int plane = 3 * 64 * waves, own = 3 * (64 * w + lane);
    float *raw = fs, *cur = fs + plane, *nxt = fs + 2 * plane;
    if (n2 > 0)
        for (int c = 0; c < 3; c++) raw[own + c] = s[c];
    const bool live_x = (px || in_x) && (ring || inner);
    for (int p = 0; p < n1; p++) {
        const float l[3] = {lane_below(s[0]), lane_below(s[1]), lane_below(s[2])};
        const float a[3] = {lane_above(s[0]), lane_above(s[1]), lane_above(s[2])};
        float o[3];
        stencil(f.sa[p], f.sb[p], l, s, a, o);
        for (int c = 0; c < 3; c++) s[c] = live_x ? o[c] : s[c];
    }
    for (int c = 0; c < 3; c++) cur[own + c] = s[c];
    __syncthreads();
    const bool live_y = in_x && (ring || inner) && w > 0 && w < waves - 1;
    for (int p = 0; p < n2; p++) {
        if (live_y) {
            const float *l = (p == 0 && ring && cr == 0 ? raw : cur) + own - 3 * 64;
            const float *a = (p == 0 && ring && cr == ny - 1 ? raw : cur) + own + 3 * 64;
            float o[3];
            stencil(f.sa[n1 + p], f.sb[n1 + p], l, s, a, o);
            for (int c = 0; c < 3; c++) s[c] = o[c];
        }
        for (int c = 0; c < 3; c++) nxt[own + c] = s[c];
        __syncthreads();
        float *t = cur;
        cur = nxt;
        nxt = t;
    }
    if (!out) return;
    if (u == 0 && w == n2 + X && lane == 0) zk_stamp_open(f.stamp);
    for (int c = 0; c < 3; c++) {
        if (X) y.jj[1][c] = cur[own - 3 * 64 + c];
        y.jj[1 + X][c] = s[c];
        y.jj[2 + X][c] = cur[own + 3 * 64 + c];
    }
    if (lane >= l0 && lane < l0 + cols && col) {
        float *o = f.r.J + 3 * ((size_t)bi + (size_t)(j + 1) * nrow);
        o[0] = s[0];
        o[1] = s[1];
        o[2] = s[2];
    }
    y.step(f.E, f.Eo, f.Bo, nx, ny, nrow, f.k, bi, j + 1, l0, cols, c0, px, oy, f.shift, f.ext);
    if (w == n2 + X && lane == 0) zk_stamp_close(f.stamp);
}

YeeK yee_constants(float dt, float dx, float dy)
{
    YeeK k;
    const float dt2 = dt / 2.0f;
    k.dtx2 = dt2 / dx;
    k.dty2 = dt2 / dy;
    k.dtx = dt / dx;
    k.dty = dt / dy;
    k.dt = dt;
    k.mur_y = (dt - dy) / (dt + dy);
    return k;
}

__global__ void guard_kernel(float *E, float *B, int nx, int ny, int nrow, int periodic_x, int open_y)
{
    guard_node(E, B, nx, ny, nrow, periodic_x, blockIdx.x * blockDim.x + threadIdx.x, open_y);
}

__global__ void move_window_kernel(const float *E, const float *B, float *Eo, float *Bo, int nx, int ny, int nrow)
{
    const int bw = nx + 3, bh = ny + 3;
    const int node = blockIdx.x * blockDim.x + threadIdx.x;
    if (node >= bw * bh) return;
    const int i = node % bw - 1;
    const size_t d = 3 * (size_t)node;
    if (i >= nx - 1) {
        for (int c = 0; c < 3; c++) Eo[d + c] = Bo[d + c] = 0.0f;
    } else {
        for (int c = 0; c < 3; c++) {
            Eo[d + c] = E[d + 3 + c];
            Bo[d + c] = B[d + 3 + c];
        }
    }
}

/* ---- laser pulse (em2d/emf.c:158-350), on the device ----
 * The reference's expressions: float operands, the C library's double
 * functions (sin, cos, exp, atan2, sqrt) with the results rounded to float
 * where the reference assigns them; the device's double functions agree
 * with the host's to within an ulp of double, so a float result can differ
 * only where the double value lies that close to a float rounding
 * boundary. */
__device__ inline float laser_envelope(const zk_laser_k &L, const float z)
{
    if (z > L.start) return 0.0f;
    if (z > L.start - L.rise) {
        const float u = z - L.start;
        const float e = (float)sin(1.5707963267948966 * u / L.rise);
        return e * e;
    }
    if (z > L.start - (L.rise + L.flat)) return 1.0f;
    if (z > L.start - (L.rise + L.flat + L.fall)) {
        const float u = z - (L.start - L.rise - L.flat - L.fall);
        const float e = (float)sin(1.5707963267948966 * u / L.fall);
        return e * e;
    }
    return 0.0f;
}

__device__ inline float laser_phase(const zk_laser_k &L, const float zpos, const float r)
{
    const float z = zpos - L.focus;
    const float zr = L.omega0 * (L.W0 * L.W0) / 2;
    const float r2 = r * r;
    const float curv = r2 * z / (zr * zr + z * z);
    const float w2 = (zr * zr) / (zr * zr + z * z);
    const float gouy = (float)atan2((double)z, (double)zr);
    return (float)(sqrt(sqrt((double)w2)) * exp((double)(-r2 * w2 / (L.W0 * L.W0))) *
                   cos((double)(L.omega0 * (z + curv) - gouy)));
}

/* one thread per interior node; E, B from the buffer origin */
__global__ void laser_kernel(float *E, float *B, int nx, int ny, int nrow, zk_laser_k L)
{
    const int node = blockIdx.x * blockDim.x + threadIdx.x;
    if (node >= nx * ny) return;
    const int i = node % nx, j = node / nx;
    const size_t g = 3 * ((size_t)(i + 1) + (size_t)(j + 1) * nrow);
    const float z = i * L.hx;
    const float zh = z + L.hx / 2;
    const float env = L.amp * laser_envelope(L, z);
    const float envh = L.amp * laser_envelope(L, zh);
    if (L.type == 0) { /* plane: the products and the sums in double, as in the reference */
        const double c = cos((double)(L.omega0 * z)), ch = cos((double)(L.omega0 * zh));
        E[g + 1] = (float)((double)E[g + 1] + (double)env * c * (double)L.cp);
        E[g + 2] = (float)((double)E[g + 2] + (double)env * c * (double)L.sp);
        B[g + 1] = (float)((double)B[g + 1] + (double)(-envh) * ch * (double)L.sp);
        B[g + 2] = (float)((double)B[g + 2] + (double)envh * ch * (double)L.cp);
    } else {
        const float r = j * L.hy - L.axis;
        const float rh = r + L.hy / 2;
        E[g + 1] += +env * laser_phase(L, z, rh) * L.cp;
        E[g + 2] += +env * laser_phase(L, z, r) * L.sp;
        B[g + 1] += -envh * laser_phase(L, zh, r) * L.sp;
        B[g + 2] += +envh * laser_phase(L, zh, rh) * L.cp;
    }
}

/* E_x, B_x from div E = div B = 0, integrated in double from the right
 * edge of each row (em2d/emf.c:213-231): one thread per row */
__global__ void laser_div_kernel(float *E, float *B, int nx, int ny, int nrow, double ratio)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ny) return;
#define AT(a, b) (3 * ((size_t)((a) + 1) + (size_t)((b) + 1) * nrow))
    double ex = 0.0, bx = 0.0;
    for (int i = nx - 1; i >= 0; i--) {
        ex += ratio * (E[AT(i + 1, j) + 1] - E[AT(i + 1, j - 1) + 1]);
        E[AT(i, j)] = (float)ex;
        bx += ratio * (B[AT(i, j + 1) + 1] - B[AT(i, j) + 1]);
        B[AT(i, j)] = (float)bx;
    }
#undef AT
}

__global__ void add_ext_kernel(const float *F, const float *ext, float ux, float uy, float uz, float *out,
                               size_t nodes)
{
    for (size_t n = blockIdx.x * (size_t)blockDim.x + threadIdx.x; n < nodes; n += (size_t)gridDim.x * blockDim.x) {
        float a0 = ext ? ext[3 * n + 0] : ux;
        float a1 = ext ? ext[3 * n + 1] : uy;
        float a2 = ext ? ext[3 * n + 2] : uz;
        out[3 * n + 0] = F[3 * n + 0] + a0;
        out[3 * n + 1] = F[3 * n + 1] + a1;
        out[3 * n + 2] = F[3 * n + 2] + a2;
    }
}

__global__ void energy_partial(const float *E, const float *B, int nx, int ny, int nrow, double *partial)
{
    __shared__ double red[16];
    double s[6] = {0, 0, 0, 0, 0, 0};
    const int cells = nx * ny;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < cells; c += gridDim.x * blockDim.x) {
        const int i = c % nx, j = c / nx;
        const size_t g = 3 * ((size_t)(i + 1) + (size_t)(j + 1) * nrow);
        for (int q = 0; q < 3; q++) {
            const float e = E[g + q], b = B[g + q];
            s[q] += (double)(e * e);
            s[3 + q] += (double)(b * b);
        }
    }
    for (int q = 0; q < 6; q++) {
        const double v = zk_block_sum(s[q], red);
        if (threadIdx.x == 0) partial[6 * blockIdx.x + q] = v;
    }
}

/* Sums the workgroups' partials, one wave per component: four loads a lane
 * at 256 partials.  Bound by the latency of one load; one thread per
 * component, which loads and adds 256 partials one after another, took
 * 32 us instead of 5. */
__global__ __launch_bounds__(6 * 64) void energy_final(const double *partial, int nblk, double *out6, double scale)
{
    const int q = threadIdx.x / 64, lane = threadIdx.x % 64;
    double s = 0.0;
    for (int b = lane; b < nblk; b += 64) s += partial[6 * b + q];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o);
    if (lane == 0) out6[q] = s * scale;
}

/* CIC charge of one particle added with global float atomics. */
__device__ inline void charge_global(float *rho, int c, int nrow, float wx, float wy, float q)
{
    unsafeAtomicAdd(&rho[c], (1.0f - wx) * (1.0f - wy) * q);
    unsafeAtomicAdd(&rho[c + 1], (wx) * (1.0f - wy) * q);
    unsafeAtomicAdd(&rho[c + nrow], (1.0f - wx) * (wy) * q);
    unsafeAtomicAdd(&rho[c + 1 + nrow], (wx) * (wy) * q);
}

/* One weight: to window node w where its float is an integer at the fixed
 * point's scale, 2^44 / Q with Q the power of two at or above |q|, which the
 * floats of [2^-21 Q, |q|] are; sums of ZK_FX_TILE_MAX of them fit.  Smaller
 * weights (one corner in some 10^5) would be cut, and a NaN or a weight
 * beyond |q|, of a particle that is not in its cell, lost: they go to the
 * grid as they are. */
__device__ inline void charge_add(const zk_charge_args &a, unsigned long long *w, float *rho, float v)
{
    const unsigned lo = __float_as_uint(a.fx_min), hi = __float_as_uint(a.fx_max);
    if (__float_as_uint(fabsf(v)) - lo <= hi - lo) atomicAdd(w, zk_fx(v, a.fx_scale));
    else if (v != 0.0f) unsafeAtomicAdd(rho, v);
}

/* Charge density from tile-sorted particles.  With four global atomics per
 * particle the atomics set the time (512 x 512, 4.2 M particles: 395 us,
 * where reading the particles takes 11 us).  Here `splits` workgroups per
 * tile sum their share in an LDS window of the tile and its H-cell drift
 * margin, in fixed point, and add each window node to the grid once (20 us).
 * Particles outside the window, the unsorted tail (the last `tail`
 * workgroups), weights outside [fx_min, fx_max] (charge_add) and tiles beyond
 * the fixed point's range use the global atomics. */
__global__ void __launch_bounds__(256) charge_kernel(zk_charge_args a)
{
    extern __shared__ unsigned long long win[];
    const zk_tiles &t = a.t;
    const zk_parts &p = a.p;
    const int nrow = t.nx + 1;
    const int b = (int)blockIdx.x - t.ntiles * a.splits;
    if (b >= 0) {
        const int n = a.ctr->np_total;
        for (int i = a.ctr->n_sorted + b * blockDim.x + threadIdx.x; i < n; i += a.tail * blockDim.x) {
            const int cell = p.cell[i];
            if (cell < 0) continue;
            const int c = zk_cell_ix(cell, p.cbits) + nrow * zk_cell_iy(cell, p.cbits);
            charge_global(a.rho, c, nrow, p.x[i], p.y[i], a.q);
        }
        return;
    }
    const int tile = (int)blockIdx.x / a.splits, part = (int)blockIdx.x % a.splits;
    const int W = t.TX + 2 * t.H + 1, V = t.TY + 2 * t.H + 1; /* nodes: one more than cells */
    const int x0 = tile % t.ntx * t.TX - t.H, y0 = tile / t.ntx * t.TY - t.H;
    for (int m = threadIdx.x; m < W * V; m += blockDim.x) win[m] = 0ull;
    const int i0 = a.tile_off[tile], i1 = a.tile_n ? i0 + a.tile_n[tile] : a.tile_off[tile + 1];
    const bool exact = i1 - i0 <= ZK_FX_TILE_MAX;
    const int piece = (i1 - i0 + a.splits - 1) / a.splits;
    const int lo = i0 + part * piece, hi = min(i1, lo + piece);
    __syncthreads();
    for (int i = lo + (int)threadIdx.x; i < hi; i += blockDim.x) {
        const int cell = p.cell[i];
        const float wx = p.x[i], wy = p.y[i];
        if (cell < 0) continue;
        const int ix = zk_cell_ix(cell, p.cbits), iy = zk_cell_iy(cell, p.cbits);
        const unsigned u = ix - x0, v = iy - y0;
        if (exact && u < (unsigned)(W - 1) && v < (unsigned)(V - 1)) {
            unsigned long long *w = win + u + v * W;
            float *r = a.rho + ix + nrow * iy;
            charge_add(a, &w[0], &r[0], (1.0f - wx) * (1.0f - wy) * a.q);
            charge_add(a, &w[1], &r[1], (wx) * (1.0f - wy) * a.q);
            charge_add(a, &w[W], &r[nrow], (1.0f - wx) * (wy) * a.q);
            charge_add(a, &w[W + 1], &r[nrow + 1], (wx) * (wy) * a.q);
        } else {
            charge_global(a.rho, ix + nrow * iy, nrow, wx, wy, a.q);
        }
    }
    __syncthreads();
    for (int m = threadIdx.x; m < W * V; m += blockDim.x) {
        const long long r = (long long)win[m];
        if (r != 0) unsafeAtomicAdd(&a.rho[x0 + m % W + nrow * (y0 + m / W)], (float)((double)r * a.fx_unscale));
    }
}

/* phase-space quantity code (X1 1, X2 2, U1 4, U2 5, U3 6) of particle i,
 * as em2d/particles.c:1569-1632 forms it */
__device__ inline float pha_quantity(const zk_parts &p, int i, int q, float dx0, float dx1)
{
    switch (q) {
    case 1: return (p.x[i] + zk_cell_ix(p.cell[i], p.cbits)) * dx0;
    case 2: return (p.y[i] + zk_cell_iy(p.cell[i], p.cbits)) * dx1;
    case 4: return p.ux[i];
    case 5: return p.uy[i];
    case 6: return p.uz[i];
    }
    return 0.0f;
}

/* The reference's bins and weights of one particle's quantities in bins
 * (va, vb) of an na x nb grid, added with add(bin, weight). */
template <class Add>
__device__ inline void pha_bins(float va, float vb, int na, int nb, float q, Add add)
{
    const int ia = (int)(va + 0.5f), ib = (int)(vb + 0.5f);
    const float wa = va - ia + 0.5f, wb = vb - ib + 0.5f;
    int c = ia + na * ib;
    if (ib >= 0 && ib < nb) {
        if (ia >= 0 && ia < na) add(c, (1.0f - wa) * (1.0f - wb) * q);
        if (ia + 1 >= 0 && ia + 1 < na) add(c + 1, wa * (1.0f - wb) * q);
    }
    c += na;
    if (ib + 1 >= 0 && ib + 1 < nb) {
        if (ia >= 0 && ia < na) add(c, (1.0f - wa) * wb * q);
        if (ia + 1 >= 0 && ia + 1 < na) add(c + 1, wa * wb * q);
    }
}

/* Bilinear phase-space density of quantities (qa, qb), straight into the
 * grid with global atomics. */
__global__ void pha_kernel(zk_parts p, const zk_spec_ctr *ctr, int qa, int qb, float dx0, float dx1, int na, int nb,
                           float amin, float bmin, float ra, float rb, float q, float *out)
{
    const int n = ctr->np_total;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (p.cell[i] < 0) continue;
        const float va = (pha_quantity(p, i, qa, dx0, dx1) - amin) * ra;
        const float vb = (pha_quantity(p, i, qb, dx0, dx1) - bmin) * rb;
        pha_bins(va, vb, na, nb, q, [&](int c, float v) { atomicAdd(&out[c], v); });
    }
}

/* The same without global atomics, which set the time above (4.2 M
 * particles on 256 x 256 bins: 990 us).  The grid is cut into `chunks` runs
 * of at most PHA_BINS bins; workgroup (r, k) sums every r-th share of the
 * particles into an LDS copy of run k and stores it as replica r of the
 * grid in `rep`; pha_sum_kernel adds the replicas in order.  Each particle
 * is read once per run: 12 bytes against the four atomics it replaces.  On
 * those 256 x 256 bins 155 + 12 us, 128 x 128 bins 91 + 12 us; the LDS float
 * atomics set it (four particles' loads in flight per thread: no change). */
constexpr int PHA_BINS = 16 * 1024; /* 64 KB of LDS: two workgroups per CU */
constexpr int PHA_THREADS = 1024;

__global__ void __launch_bounds__(PHA_THREADS) pha_lds_kernel(zk_parts p, const zk_spec_ctr *ctr, int qa, int qb,
                                                              float dx0, float dx1, int na, int nb, float amin,
                                                              float bmin, float ra, float rb, float q, float *rep)
{
    extern __shared__ float hist[];
    const int nbins = na * nb, c0 = (int)blockIdx.y * PHA_BINS, nc = min(PHA_BINS, nbins - c0);
    for (int m = threadIdx.x; m < nc; m += blockDim.x) hist[m] = 0.0f;
    __syncthreads();
    const int n = ctr->np_total;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int cell = p.cell[i];
        const float va = (pha_quantity(p, i, qa, dx0, dx1) - amin) * ra;
        const float vb = (pha_quantity(p, i, qb, dx0, dx1) - bmin) * rb;
        if (cell < 0) continue;
        pha_bins(va, vb, na, nb, q, [&](int c, float v) {
            const unsigned m = (unsigned)(c - c0);
            if (m < (unsigned)nc) atomicAdd(&hist[m], v);
        });
    }
    __syncthreads();
    for (int m = threadIdx.x; m < nc; m += blockDim.x) rep[(size_t)blockIdx.x * nbins + c0 + m] = hist[m];
}

/* 32 bins per workgroup, every eighth replica per thread: one thread per
 * bin walked up to 512 replicas in a row (75 us; the replicas are 32 MB) */
__global__ void __launch_bounds__(256) pha_sum_kernel(const float *rep, int nrep, int nbins, float *out)
{
    __shared__ float part[8][32];
    const int l = threadIdx.x % 32, g = threadIdx.x / 32, m = blockIdx.x * 32 + l;
    float s = 0.0f;
    if (m < nbins)
        for (int r = g; r < nrep; r += 8) s += rep[(size_t)r * nbins + m];
    part[g][l] = s;
    __syncthreads();
    if (g > 0 || m >= nbins) return;
    for (int k = 1; k < 8; k++) s += part[k][l];
    out[m] = s;
}

__global__ void add_kernel(float *acc, const float *v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        acc[i] += v[i];
}

#define ZK_MAX_DEVICES 64
float *g_scratch[ZK_MAX_DEVICES];
std::mutex g_scratch_lock;

} // namespace

/* The array's name is not a device address in host code: its address on a
 * device comes from hipGetSymbolAddress, called once per device with that
 * device current, and only that address is passed to kernels and copies. */
extern "C" int zk_noalloc_scratch(float **ptr)
{
    int dev = 0;
    int e = (int)hipGetDevice(&dev);
    if (e) return e;
    if (dev < 0 || dev >= ZK_MAX_DEVICES) return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        e = (int)hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e) return e;
        g_scratch[dev] = (float *)p;
    }
    *ptr = g_scratch[dev];
    return 0;
}

extern "C" int zk_add_f32(float *acc, const float *v, size_t n, zk_stream_t s)
{
    if (n == 0) return 0;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(add_kernel, dim3((unsigned)blocks), dim3(256), 0, s, acc, v, n);
    ZK_LAUNCH_CHECK();
}

/* Replicas of the phase-space grid the LDS path keeps, 0 where it does not
 * pay: beyond 16 runs the particles are read more often than the atomics
 * cost.  About two workgroups per CU over all runs, and no more than one per
 * 4096 particles. */
static int pha_replicas(int np, int na, int nb)
{
    const long long runs = ((long long)na * nb + PHA_BINS - 1) / PHA_BINS;
    if (runs > 16) return 0;
    const long long r = 512 / runs, want = ((long long)np + 4095) / 4096;
    return (int)(want < 1 ? 1 : want < r ? want : r);
}

extern "C" size_t zk_pha_scratch(int np_upper, int na, int nb)
{
    return (size_t)pha_replicas(np_upper, na, nb) * (size_t)na * (size_t)nb * sizeof(float);
}

extern "C" int zk_pha(const zk_parts *p, int np_upper, const zk_spec_ctr *ctr, int qa, int qb, float dx0, float dx1,
                      int na, int nb, float amin, float bmin, float ra, float rb, float q, float *out, float *scratch,
                      zk_stream_t s)
{
    if (na <= 0 || nb <= 0) return 0;
    const int rep = pha_replicas(np_upper, na, nb), nbins = na * nb;
    if (rep > 0) {
        const size_t lds = (size_t)(nbins < PHA_BINS ? nbins : PHA_BINS) * sizeof(float);
        hipLaunchKernelGGL(pha_lds_kernel, dim3(rep, (nbins + PHA_BINS - 1) / PHA_BINS), dim3(PHA_THREADS), lds, s, *p,
                           ctr, qa, qb, dx0, dx1, na, nb, amin, bmin, ra, rb, q, scratch);
        hipLaunchKernelGGL(pha_sum_kernel, dim3((nbins + 31) / 32), dim3(256), 0, s, scratch, rep, nbins, out);
    } else {
        long long b = (np_upper + 255) / 256;
        if (b < 1) b = 1;
        if (b > 4096) b = 4096;
        const int e = zk_fill_f32(out, (size_t)nbins, 0.0f, s);
        if (e) return e;
        hipLaunchKernelGGL(pha_kernel, dim3((unsigned)b), dim3(256), 0, s, *p, ctr, qa, qb, dx0, dx1, na, nb, amin,
                           bmin, ra, rb, q, out);
    }
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_yee_ext(const float *E, const float *B, const float *J, float *Eo, float *Bo, int nx, int ny,
                          int nrow, float dt, float dx, float dy, int periodic_x, int open_y, int shift,
                          const zk_ext *ext, zk_stamp st, zk_stream_t s)
{
    if (shift && (ext->out[0] || ext->out[1])) return (int)hipErrorInvalidValue;
    const YeeK k = yee_constants(dt, dx, dy);
    const int r = zk_yee_rows(nx, ny), units = zk_yee_units(nx, ny, r);
    const bool x = ext->out[0] || ext->out[1];
#define YEE(R, X, WAVES)                                                                                              \
    hipLaunchKernelGGL((yee_kernel<R, X>), dim3((units + WAVES - 1) / WAVES), dim3(64 * WAVES), 0, s, E, B, J, Eo,    \
                       Bo, nx, ny, nrow, k, periodic_x, open_y, shift, units, *ext, st)
    if (r == ZK_YEE_R_SMALL && x) YEE(ZK_YEE_R_SMALL, true, 1);
    else if (r == ZK_YEE_R_SMALL) YEE(ZK_YEE_R_SMALL, false, 1);
    else if (x) YEE(ZK_YEE_R, true, 4);
    else YEE(ZK_YEE_R, false, 4);
#undef YEE
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_yee(const float *E, const float *B, const float *J, float *Eo, float *Bo, int nx, int ny, int nrow,
                      float dt, float dx, float dy, int periodic_x, int open_y, int shift, zk_stamp st, zk_stream_t s)
{
    const zk_ext none = {};
    return zk_yee_ext(E, B, J, Eo, Bo, nx, ny, nrow, dt, dx, dy, periodic_x, open_y, shift, &none, st, s);
}

/* From here on the separate launches read each window and node once and cost
 * no more: 256 x 256 cells 10.0 us in one launch, 16.1 in three; 512 x 512
 * the same with the gap between two; 2000 x 512 22.2 and 22.0, the run 1.5 %
 * longer in one; 2048 x 2048 210 and 175. */
#define ZK_FIELD_STEP_NODES (1 << 19)

extern "C" int zk_field_step_ok(const zk_tiles *t, int n1, int n2, int open_y)
{
    return reduce_span(*t) != 0 && n1 <= ZK_MAX_PASSES && n2 <= ZK_MAX_Y_PASSES && field_rows(16, n2, open_y) >= 4 &&
           (long long)(t->nx + 3) * (t->ny + 3) < ZK_FIELD_STEP_NODES;
}

extern "C" int zk_field_step(const zk_field_args *args, float dt, float dx, float dy, zk_stream_t s)
{
    zk_field_args f = *args;
    const int nx = f.r.t.nx, ny = f.r.t.ny, oy = f.r.open_y != 0;
    if (!zk_field_step_ok(&f.r.t, f.n1, f.n2, oy) || f.n1 < 0 || f.n2 < 0 ||
        (f.shift && (f.ext.out[0] || f.ext.out[1])))
        return (int)hipErrorInvalidValue;
    f.k = yee_constants(dt, dx, dy);
    const int waves = field_waves(f.n2, oy), rows = field_rows(waves, f.n2, oy), cols = field_cols(f.n1);
    f.clears = f.r.jflag_next ? (zk_red_blocks_x(nx) * zk_red_blocks_y(ny) + waves - 1) / waves : 0;
    const int units = (nx + 3 + cols - 1) / cols * ((ny + 3 + rows - 1) / rows);
    const dim3 grid(f.r.fin.n + f.clears + units), block(64 * waves);
    const size_t lds = sizeof(float) * 3 * 3 * 64 * waves;
    const int span = reduce_span(f.r.t);
    if (span == 2 && !oy) hipLaunchKernelGGL((field_step_kernel<2, 0>), grid, block, lds, s, f);
    else if (span == 2) hipLaunchKernelGGL((field_step_kernel<2, 1>), grid, block, lds, s, f);
    else if (!oy) hipLaunchKernelGGL((field_step_kernel<3, 0>), grid, block, lds, s, f);
    else hipLaunchKernelGGL((field_step_kernel<3, 1>), grid, block, lds, s, f);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_field_guards(float *E, float *B, int nx, int ny, int nrow, int periodic_x, int open_y,
                               zk_stream_t s)
{
    /* a moving window (no x copies) with open y (no y copies): nothing to do */
    if (!periodic_x && open_y) return 0;
    const int n = 3 * (nx + 3) + 3 * ny;
    hipLaunchKernelGGL(guard_kernel, dim3((n + 255) / 256), dim3(256), 0, s, E, B, nx, ny, nrow, periodic_x,
                       open_y);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_move_window(const float *E, const float *B, float *Eo, float *Bo, int nx, int ny, int nrow,
                                     zk_stream_t s)
{
    const int nodes = (nx + 3) * (ny + 3);
    hipLaunchKernelGGL(move_window_kernel, dim3((nodes + 255) / 256), dim3(256), 0, s, E, B, Eo, Bo, nx, ny, nrow);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_add_ext(const float *F, const float *ext, float ux, float uy, float uz, float *out,
                                 size_t nodes, zk_stream_t s)
{
    size_t blocks = (nodes + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(add_ext_kernel, dim3((unsigned)blocks), dim3(256), 0, s, F, ext, ux, uy, uz, out, nodes);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_emf_energy(const float *E, const float *B, int nx, int ny, int nrow, double *partial,
                                    int nblk, double *out6, double scale, zk_stream_t s)
{
    hipLaunchKernelGGL(energy_partial, dim3(nblk), dim3(256), 0, s, E, B, nx, ny, nrow, partial);
    hipLaunchKernelGGL(energy_final, dim3(1), dim3(6 * 64), 0, s, partial, nblk, out6, scale);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_charge(zk_charge_args a, int tail_upper, zk_stream_t s)
{
    /* a few workgroups per CU also on grids of few tiles */
    a.splits = a.t.ntiles > 0 ? 1024 / a.t.ntiles : 1;
    a.splits = a.splits < 1 ? 1 : a.splits > 16 ? 16 : a.splits;
    long long b = (tail_upper + 255) / 256;
    a.tail = (int)(b < 0 ? 0 : b > 4096 ? 4096 : b);
    const unsigned grid = (unsigned)(a.t.ntiles * a.splits + a.tail);
    const size_t lds = (size_t)(a.t.TX + 2 * a.t.H + 1) * (size_t)(a.t.TY + 2 * a.t.H + 1) * 8;
    if (grid > 0) hipLaunchKernelGGL(charge_kernel, dim3(grid), dim3(256), lds, s, a);
    ZK_LAUNCH_CHECK();
}

extern "C" int zk_laser(float *E, float *B, int nx, int ny, int nrow, const zk_laser_k *L, double ratio, zk_stream_t s)
{
    const int nodes = nx * ny;
    if (nodes <= 0) return 0;
    hipLaunchKernelGGL(laser_kernel, dim3((nodes + 255) / 256), dim3(256), 0, s, E, B, nx, ny, nrow, *L);
    if (L->type != 0) hipLaunchKernelGGL(laser_div_kernel, dim3((ny + 63) / 64), dim3(64), 0, s, E, B, nx, ny, nrow, ratio);
    ZK_LAUNCH_CHECK();
}
