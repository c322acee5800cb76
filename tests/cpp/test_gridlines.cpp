// The lines that the tiles of the multigrid kernels read (gf_gridlines.hpp), for every lane of every tile of
// grids narrower and wider than a tile: in range, and the right one wherever a result depends on it.
#include <cstdio>
#include <cstdlib>

#include "../../goosefem_amd/csrc/gf_gridlines.hpp"

static long checked = 0;

template <int W, int H, class F>
static void sweep(const char* what, int ring, F line)
{
    for (int per = 0; per < 2; ++per)
        for (int m = per ? 3 : 4; m <= 300; ++m) {
            const int own = W - 2 * H;
            for (int b = 0; b < (m + own - 1) / own; ++b)
                for (int t = 0; t < W; ++t) {
                    const int raw = gf::tile_raw<W, H>(b, t), got = line(b, t, m, per);
                    const int want = per ? ((raw % m) + m) % m : raw >= 0 && raw < m ? raw : -1;
                    const bool used = ring < 0 || (raw >= -ring && raw < m + ring);
                    ++checked;
                    if (got < -1 || got >= m || (got == -1 && per) || (used && got != want)) {
                        std::printf("%s: %d lines%s, tile %d lane %d: %d (line %d)\n", what, m, per ? " wrapped" : "", b,
                                    t, got, raw);
                        std::exit(1);
                    }
                }
        }
}

int main()
{
    // the smoothing tiles (every lane's line feeds an owned one), the product's tiles (one ring)
    sweep<32, 6>("down x", -1, gf::tile_line<32, 6>);
    sweep<16, 6>("down y", -1, gf::tile_line<16, 6>);
    sweep<32, 5>("up x", -1, gf::tile_line<32, 5>);
    sweep<16, 5>("up y", -1, gf::tile_line<16, 5>);
    sweep<34, 1>("product x", 1, gf::tile_line_ring<34, 1>);
    sweep<10, 1>("product y", 1, gf::tile_line_ring<10, 1>);
    std::printf("%ld lanes: ALL OK\n", checked);
    return 0;
}
