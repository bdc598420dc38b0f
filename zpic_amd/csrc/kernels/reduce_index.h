/*
 * reduce_index.h - which current windows cover a node (integer arithmetic
 * only, compiled for the device and, in the tests, for the host).
 */
#ifndef ZK_REDUCE_INDEX_H
#define ZK_REDUCE_INDEX_H

#ifdef __HIP__
#define ZK_HD __host__ __device__
#else
#define ZK_HD
#endif

namespace zk {

/* Raw positions in [-1, n + 1] that fold onto interior index c of an axis
 * of n >= 3 cells, ascending; an axis that is not folded has c alone.
 * Returns how many (at most 2). */
ZK_HD inline int axis_images(int c, int n, int fold, int r[2])
{
    r[0] = r[1] = c;
    if (!fold) return 1;
    if (c == n - 1) {
        r[0] = -1;
        return 2;
    }
    if (c <= 1) {
        r[1] = c + n;
        return 2;
    }
    return 1;
}

/* The last tile of T cells whose window (T + 2 H + 3 nodes from H + 1 below
 * the tile) starts at or below raw position r >= -1; inv = 1.0f / T.  With
 * a + 0.5 at least 0.5 from any multiple of T, the float product rounds
 * down to the right quotient for a < 2^22. */
ZK_HD inline int last_tile(int r, int H, float inv) { return (int)(((float)(r + 1 + H) + 0.5f) * inv); }

/* Offset of raw position r in the window of tile k, and whether tile k
 * exists and its window covers r (k at or below last_tile(r)). */
ZK_HD inline int window_offset(int r, int H, int T, int k) { return r + 1 + H - k * T; }
ZK_HD inline bool window_covers(int k, int nt, int u, int W) { return k >= 0 && k < nt && u < W; }

} // namespace zk

#endif
