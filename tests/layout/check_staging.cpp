// check_staging.cpp -- host check of the columns that the plane-tiled kernels stage
// (stage_column in grid_tile.hpp), compiled for the host only and run by
// tests/test_staging.py: for every layout that can be instantiated, every grid axis from
// the shortest one up to four tiles, every tile and every unit of a row, the unit's cells
// lie on the axis, and the units of the used cells are the ones that the wrapped window
// needs.  Prints "STAGING_OK" and the number of layouts whose spare units needed care.
#include <cstdio>
#include <cstdlib>

#include "grid_tile.hpp"

using namespace cunfft;

static int g_layouts = 0, g_short = 0;

template <typename T, int D, int W, int V> void check()
{
    using L = TileLayout<T, D, W, 1, V>;
    if constexpr (L::fits) {
        ++g_layouts;
        bool past = false;
        for (int n = L::TL; n <= 4 * L::TL; n += L::TL) {
            if (n < W) continue;
            for (int o = 0; o < n; o += L::TL)
                for (int un = 0; un < L::RP / L::CPL; ++un) {
                    const int plain = o + L::CPL * un;
                    past = past || plain - n >= n;
                    const int c = (int)stage_column<L>((uint32_t)o, un, (uint32_t)n);
                    if (c < 0 || c + L::CPL > n) {
                        printf("%zu D%d W%d V%d n %d o %d unit %d: column %d\n", sizeof(T), D, W, V, n, o, un, c);
                        exit(1);
                    }
                    if (L::CPL * un < L::PL && c != plain % n) {
                        printf("%zu D%d W%d V%d n %d o %d unit %d: column %d of %d\n", sizeof(T), D, W, V, n, o, un,
                               c, plain % n);
                        exit(1);
                    }
                }
        }
        g_short += past;
    }
}

template <typename T, int D, int V> void widths()
{
    check<T, D, 4, V>();
    check<T, D, 6, V>();
    check<T, D, 8, V>();
    check<T, D, 10, V>();
    check<T, D, 12, V>();
    check<T, D, 14, V>();
    check<T, D, 16, V>();
    check<T, D, 18, V>();
}

template <typename T> void all()
{
    widths<T, 2, 0>();
    widths<T, 2, 1>();
    widths<T, 2, 2>();
    widths<T, 3, 0>();
    widths<T, 3, 1>();
    widths<T, 3, 2>();
}

int main()
{
    all<float>();
    all<double>();
    printf("%d layouts, %d with spare units past a second copy of the axis\nSTAGING_OK\n", g_layouts, g_short);
    return 0;
}
