// complete_level(): the places of a level's tiles in the cube of its root, wherever the root lies, and
// no answer for tiles that are not exactly that cube.
#include <cstdio>

#include "cmg_host.hpp"

using namespace cmg;

static int failures = 0;
#define CHECK(...)                                              \
    do {                                                        \
        if (!(__VA_ARGS__)) {                                   \
            std::printf("line %d: %s\n", __LINE__, #__VA_ARGS__); \
            ++failures;                                         \
        }                                                       \
    } while (0)

static Topology tree(const Coord& root, int levels)
{
    const uint32_t log2[5] = {4, 6, 9, 12, 12};
    Topology t(0.125f, 5, log2);
    t.set_tile(0, root, LEAF);
    t.compress();
    t.iterative_refine([levels](int, const Coord&) { return levels; });
    t.finalize();
    return t;
}

int main()
{
    // uniform trees under roots at, beside, before and far from the origin
    for (const Coord& r : {Coord{0, 0, 0}, Coord{1, 0, 0}, Coord{-1, 2, 0}, Coord{0, -3, -1}, Coord{100000, -70000, 9}}) {
        Topology t = tree(r, 3);
        for (int l = 1; l <= 3; ++l) {
            const int e = 1 << l;
            const std::vector<int32_t> at = complete_level(t, t.level_start[0], l);
            CHECK(at.size() == size_t(e) * e * e);
            for (size_t p = 0; p < at.size(); ++p) {
                const int x = int(p) / (e * e), y = int(p) / e % e, z = int(p) % e;
                CHECK(at[p] == t.tile_at(l, Coord{r[0] * e + x, r[1] * e + y, r[2] * e + z}));
            }
        }
        CHECK(complete_level(t, t.level_start[0], 4).empty());
    }
    // eight tiles of level 1 that are not the root's cube: one of them beside it, on each side of each axis
    for (int a = 0; a < 3; ++a)
        for (int far : {-1, 2, 4}) {
            const uint32_t log2[2] = {4, 6};
            Topology t(0.125f, 2, log2);
            t.set_tile(0, Coord{0, 0, 0}, NONLEAF);
            for (int o = 1; o < 8; ++o) t.set_tile(1, Coord{o & 1, (o >> 1) & 1, (o >> 2) & 1}, LEAF);
            Coord c{0, 0, 0};
            c[a] = far;
            t.set_tile(1, c, LEAF);
            t.finalize();
            CHECK(t.level_start[2] - t.level_start[1] == 8);
            CHECK(complete_level(t, 0, 1).empty());
        }
    // a GHOST tile among the eight, and fewer or more than eight
    for (int extra : {0, 1, 2}) {
        const uint32_t log2[2] = {4, 6};
        Topology t(0.125f, 2, log2);
        t.set_tile(0, Coord{0, 0, 0}, NONLEAF);
        for (int o = 0; o < 8 - (extra == 1); ++o)
            t.set_tile(1, Coord{o & 1, (o >> 1) & 1, (o >> 2) & 1}, extra == 0 && o == 5 ? GHOST : LEAF);
        if (extra == 2) t.set_tile(1, Coord{2, 0, 0}, GHOST);
        t.finalize();
        CHECK(complete_level(t, 0, 1).empty());
    }
    // at the ends of the coordinates' range: root << level does not fit 32 bits
    {
        const uint32_t log2[2] = {4, 6};
        Topology t(0.125f, 2, log2);
        t.set_tile(0, Coord{0x40000000, 0, 0}, NONLEAF);
        for (int o = 0; o < 8; ++o) t.set_tile(1, Coord{o & 1, (o >> 1) & 1, (o >> 2) & 1}, LEAF);
        t.finalize();
        CHECK(complete_level(t, 0, 1).empty());
    }
    if (!failures) std::printf("complete_level OK\n");
    return failures != 0;
}
