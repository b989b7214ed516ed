// Blocks of the slab Gram kernel (hip_tiles.hip): p16 x q16 tiles of 16 columns
// cut into bp x bq blocks of MB x NB tiles, NT of them per wavefront.  Host code
// without HIP.
#ifndef GRAM_SHAPE_H_
#define GRAM_SHAPE_H_

#include <algorithm>
#include <cstdint>

namespace gh {

constexpr int kSlabTiles = 28;  // most 16-column tiles of V and W together in a block (7 units per thread)
constexpr int kSlabMaxNT = 17;  // most output tiles per wavefront

struct SlabShape {
    int bp, bq, MB, NB, NT;
};

// Most tiles that a block computes.  Of the blocks that reach above the diagonal
// those of the first block row have the most, and there the last whole block or
// the part beside it: tile column y holds min(MB, p16, y + 1) tiles.
inline int slab_live(int p16, int q16, int MB, int NB, bool upper)
{
    if (!upper) return std::min(MB, p16) * std::min(NB, q16);
    const int x = std::min(MB, p16);
    const auto left_of = [x](int64_t y) {  // tiles in the columns 0 .. y - 1
        return y <= x ? y * (y + 1) / 2 : (int64_t)x * (x + 1) / 2 + (y - x) * x;
    };
    const int last = (q16 - 1) / NB * NB;
    int64_t most = left_of(q16) - left_of(last);
    if (last > 0) most = std::max(most, left_of(last) - left_of(last - NB));
    return (int)most;
}

// The cheapest cut: per row, a tile of products costs about 1, a tile's 16
// columns 3.5 to load (67 TF and 5 TB/s in FP64, 153 TF in FP32).
inline SlabShape slab_shape(int p16, int q16, bool upper)
{
    SlabShape best{0, 0, 0, 0, 0};
    double least = 0.0;
    for (int bp = 1; bp <= p16; bp++)
        for (int bq = 1; bq <= q16; bq++) {
            // many more blocks than some cut needs only load more
            if (best.bp > 0 && bp * bq > 4 * best.bp * best.bq) break;
            const int MB = (p16 + bp - 1) / bp, NB = (q16 + bq - 1) / bq;
            const int NT = (slab_live(p16, q16, MB, NB, upper) + 7) / 8;
            if (MB + NB > kSlabTiles || NT > kSlabMaxNT) continue;
            const double cost = (double)bp * bq * (8.0 * NT + 3.5 * (MB + NB));
            if (best.bp == 0 || cost < least) {
                least = cost;
                best = {(p16 + MB - 1) / MB, (q16 + NB - 1) / NB, MB, NB, NT};
            }
        }
    return best;
}

}  // namespace gh
#endif
