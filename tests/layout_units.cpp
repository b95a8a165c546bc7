// The lattices' layout (kernels.h tile_geom, tiles_serve, LatGeom), checked on the host.
#include <cstdio>
#include <vector>

#include "../imexlb_amd/csrc/kernels.h"

using namespace imx;

static int failures = 0;
#define CHECK(c)                                                    \
    do {                                                            \
        if (!(c)) {                                                 \
            if (++failures < 20) printf("line %d: %s\n", __LINE__, #c); \
        }                                                           \
    } while (0)

static uint64_t plane_elems(const LatGeom &g) { return g.zs / Q; }

int main()
{
    const uint64_t elems[3] = {8, 4, 2};
    for (uint64_t elem : elems) {
        const uint64_t line = 128 / elem;
        for (uint32_t plane = 64; plane < 5000; ++plane) {
            LatGeom g;
            CHECK(tile_geom(plane, 1, elem, false, g));
            const uint64_t t = uint64_t(1) << g.tl, held = plane_elems(g);
            CHECK(t >= line && t * elem <= 32768 && held % t == 0 && held >= plane && held - plane < t);
            // at most a sixteenth unused, or what rounding up to lines leaves
            CHECK((held - plane) * 16 <= plane || (t == line && held == (plane + line - 1) / line * line));
            for (bool aa : {false, true})
                for (uint64_t cells : {uint64_t(20000), uint64_t(100000), uint64_t(1000000), uint64_t(10000000)}) {
                    const uint32_t nz = (uint32_t)(cells / plane) + 2;
                    if (!tiles_serve(g, plane, 1, nz, elem, aa)) continue;
                    const uint64_t bytes = lattice_elems(g, nz) * elem * (aa ? 1 : 2);
                    const uint64_t part = bytes > LAST_LEVEL ? 12 : bytes > LAST_LEVEL / 2 ? 4 : 1;
                    CHECK((held - plane) * part <= plane);
                }
        }
        for (uint32_t plane = 0; plane < 64; ++plane) {
            LatGeom g;
            CHECK(!tile_geom(plane, 1, elem, true, g));
        }
        // every population of every cell has a place of its own
        for (uint32_t plane : {64u, 65u, 80u, 130u, 144u, 400u, 529u, 1665u, 4097u})
            for (bool aa : {false, true}) {
                LatGeom g;
                CHECK(tile_geom(plane, 1, elem, aa, g));
                const uint32_t nz = 3;
                std::vector<bool> seen(lattice_elems(g, nz), false);
                for (int i = 0; i < Q; ++i)
                    for (uint32_t z = 0; z < nz; ++z)
                        for (uint32_t p = 0; p < plane; ++p) {
                            const uint64_t o = g.off(g.pos(i), z, p);
                            CHECK(o < seen.size() && !seen[o]);
                            if (o < seen.size()) seen[o] = true;
                        }
            }
    }
    if (!failures) printf("ok\n");
    return failures != 0;
}
