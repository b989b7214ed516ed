// The cut of the slab Gram kernel against a count of every block's tiles, and its
// cost in time.
#include <chrono>
#include <cstdio>

#include "gram_shape.h"

using namespace gh;

static int counted(int p16, int q16, int MB, int NB, bool upper)
{
    int most = 0;
    for (int i = 0; i < p16; i += MB)
        for (int j = 0; j < q16; j += NB) {
            int live = 0;
            for (int x = i; x < std::min(p16, i + MB); x++)
                for (int y = j; y < std::min(q16, j + NB); y++) live += !upper || x <= y;
            most = std::max(most, live);
        }
    return most;
}

int main()
{
    for (int upper = 0; upper < 2; upper++)
        for (int p = 1; p <= 24; p++)
            for (int q = upper ? p : 1; q <= (upper ? p : 24); q++) {
                for (int MB = 1; MB <= p; MB++)
                    for (int NB = 1; NB <= q; NB++)
                        if (slab_live(p, q, MB, NB, upper) != counted(p, q, MB, NB, upper))
                            return printf("%d x %d tiles in %d x %d, upper %d\n", p, q, MB, NB, upper), 1;
                const SlabShape s = slab_shape(p, q, upper);
                if (s.bp * s.MB < p || s.bq * s.NB < q || s.MB + s.NB > kSlabTiles || s.NT > kSlabMaxNT ||
                    8 * s.NT < counted(p, q, s.MB, s.NB, upper))
                    return printf("%d x %d tiles: no cut\n", p, q), 1;
            }
    // 2,000 columns, symmetric: the cut must not cost what the products do
    double us = 1e9;
    for (int i = 0; i < 10; i++) {
        const auto t = std::chrono::steady_clock::now();
        volatile int bp = slab_shape(125, 125, true).bp;
        (void)bp;
        us = std::min(us, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t).count());
    }
    if (us > 2000.0) return printf("2,000 columns: %.0f us\n", us), 1;
    return 0;
}
