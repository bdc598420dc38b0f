/* Windows summed into each node by the current reduction: the list that
 * reduce_index.h forms, against a plain search over every image and tile. */
#include <cstdio>
#include <vector>

#include "reduce_index.h"

struct Term { int r, k, u; };
static bool same(const std::vector<Term> &a, const std::vector<Term> &b)
{
    if (a.size() != b.size()) return false;
    for (size_t m = 0; m < a.size(); m++)
        if (a[m].r != b[m].r || a[m].k != b[m].k || a[m].u != b[m].u) return false;
    return true;
}

int main()
{
    long long nodes = 0, bad = 0;
    const int sizes[] = {3, 4, 5, 7, 8, 15, 16, 17, 31, 33, 61, 97, 128, 250, 1500};
    const int tiles[] = {2, 3, 5, 7, 8, 12, 13, 16, 20, 24, 32, 48};
    for (int n : sizes)
        for (int T : tiles)
            for (int H = 1; H <= 6; H++)
                for (int fold = 0; fold < 2; fold++) {
                    if (T > n) continue;
                    const int W = T + 2 * H + 3, nt = (n + T - 1) / T;
                    const int N = W <= 2 * T ? 2 : W <= 3 * T ? 3 : 0;
                    if (!N) continue;
                    for (int i = -1; i <= n + 1; i++) {
                        const int c = !fold ? i : ((i % n) + n) % n;
                        std::vector<Term> want, got;
                        for (int s = fold ? -1 : 0; s <= (fold ? 1 : 0); s++) {
                            const int r = c + s * n;
                            if (r < -1 || r > n + 1) continue;
                            for (int k = 0; k < nt; k++) {
                                const int u = r - (k * T - 1 - H);
                                if (u >= 0 && u < W) want.push_back({r, k, u});
                            }
                        }
                        int rs[2];
                        const int m = zk::axis_images(c, n, fold, rs);
                        for (int g = 0; g < m; g++) {
                            const int last = zk::last_tile(rs[g], H, 1.0f / T);
                            for (int k = last - (N - 1); k <= last; k++) {
                                const int u = zk::window_offset(rs[g], H, T, k);
                                if (zk::window_covers(k, nt, u, W)) {
                                    if (u < 0) bad++;
                                    got.push_back({rs[g], k, u});
                                }
                            }
                        }
                        nodes++;
                        if (!same(want, got)) bad++;
                    }
                }
    printf("{\"nodes\": %lld, \"bad\": %lld}\n", nodes, bad);
    return 0;
}
