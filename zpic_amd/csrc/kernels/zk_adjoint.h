/*
 * zk_adjoint.h - launchers of the reverse-mode kernels (adjoint.hip).
 *
 * Layouts are those of zk.h: guard-inclusive float3 grids of
 * (nx + 3) x (ny + 3) nodes with row stride nrow, particles as seven
 * arrays grouped by tile.  Particle adjoints are five arrays: the
 * adjoints of the cell offsets x, y (equal to those of the continuous
 * positions) and of the momenta ux, uy, uz.
 */
#ifndef ZK_ADJOINT_H
#define ZK_ADJOINT_H

#include "zk.h"

#ifdef __cplusplus
extern "C" {
#endif

typedef struct zk_adj_vec {
    float *lx, *ly, *lux, *luy, *luz;
} zk_adj_vec;

typedef struct zk_adj_spec {
    zk_parts p;                 /* particle state at the start of the step (read) */
    const int *tile_off;        /* [ntiles + 1] tile ranges of p */
    zk_adj_vec lin;             /* particle adjoints after the step (read) */
    zk_adj_vec lout;            /* particle adjoints before the step (written) */
    int *ovf_list;              /* slots outside their tile window, listed at the start
                                   of the listing workgroup's share of the tile range */
    float tem, dt_dx, dt_dy, qnx, qny, q;
} zk_adj_spec;

typedef struct zk_adj_push_args {
    zk_adj_spec s[ZK_FUSE_MAX];
    int ns;                     /* species (1 to ZK_FUSE_MAX) */
    const float *E, *B;         /* fields at the start of the step */
    const float *lam;           /* adjoint of the raw current, per buffer node */
    int nrow;
    float *region;              /* [ns * ntiles * splits][6][WY][WX] field-adjoint windows */
    float *lE, *lB;             /* field adjoints (accumulated) */
    zk_tiles t;
    int splits;                 /* workgroups per tile (>= 1) */
    unsigned *amax;             /* [ns * ntiles * splits] float bits: running maximum of the
                                   gathered-field adjoints of a window slot (0 at the start) */
} zk_adj_push_args;

/* dst = src for the seven particle arrays (and ids when both have them) */
int zk_copy_parts(const zk_parts *dst, const zk_parts *src, int n, zk_stream_t s);
/* a = sa and b = sb, n floats each */
int zk_copy_pair(float *a, const float *sa, float *b, const float *sb, size_t n, zk_stream_t s);
/* lB(interior) += scale * B(interior) */
int zk_adj_loss(float *lB, const float *B, int nx, int ny, int nrow, float scale, zk_stream_t s);
/* Reverse of the field step (periodic) and of the periodic current fold: lE,
 * lB hold the adjoints of the step's output fields, lE_in, lB_in (other
 * buffers) receive those of its input fields, lJ that of the current and lam
 * that of the raw current (per buffer node).  F: NULL, or the step's output B, whose loss term
 * scale * B is first added to lB on the interior. */
int zk_adj_fields(const float *lE, const float *lB, const float *F, float scale, float *lE_in, float *lB_in,
                  float *lJ, float *lam, int nx, int ny, int nrow, float dt, float dx, float dy, zk_stream_t s);
/* Reverse of the particle push of a set of species (tile pass, listed
 * particles, field-adjoint windows added into lE, lB) */
/* workgroups of zk_adj_push that the GPU holds at once */
#define ZK_ADJ_RESIDENT 768
int zk_adj_push(const zk_adj_push_args *a, zk_stream_t s);
/* dst[i] = src[pos[ids_dst[i]]] with pos[ids_src[k]] = k: particle
 * adjoints carried from one particle order to another */
int zk_adj_permute(const zk_adj_vec *src, const zk_adj_vec *dst, const int64_t *ids_src, const int64_t *ids_dst,
                   int *pos, int n, zk_stream_t s);
/* out[5 id + c] = component c of slot i (x, y, ux, uy, uz) */
int zk_adj_by_id(const zk_adj_vec *v, const int64_t *ids, int n, float *out, zk_stream_t s);

#ifdef __cplusplus
}
#endif

#endif
