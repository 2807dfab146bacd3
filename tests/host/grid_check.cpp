// Host check of wide_grid: every block once, fewer than 2^32 threads along x.
#include "common.hpp"

int main()
{
    for (long blocks : {1L, 2L, 255L, (1L << 23) - 1, 1L << 23, (1L << 23) + 1, (1L << 24) + 5,
                        67108865L, 134217728L}) {
        const dim3 g = regot::wide_grid(blocks);
        const long x = g.x, y = g.y;
        // at most one row of blocks past the end, y within the 65536 of a launch
        if (x * 256 >= 1L << 32 || x * y < blocks || x * (y - 1) >= blocks || y > 65535 ||
            g.z != 1) {
            std::printf("%ld blocks: %ld x %ld\n", blocks, x, y);
            return 1;
        }
    }
    return 0;
}
