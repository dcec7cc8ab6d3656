// Every load that batch_q8_pipe_kernel makes of a workgroup's weights and
// scales, by its own offsets (q8_pipe.hpp), against the bytes of its views:
// for every count of row tiles a workgroup can have and group pairs up to
// those of 16,384 columns, the scalar offset lies in the view and the furthest
// lane's read ends in it; row tiles that are there are read in their place.
// Likewise the vectors' halves, for even and odd counts of groups.  The plans'
// splits cover the groups without an empty one and, as a partial-sum buffer is
// sized by tiles of 16 vectors, kernel and splits change with those only.
// "choice TILES GROUPS N" prints which kernel takes a product.
#include "q8_pipe.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>

using namespace tvara_amd;

int main(int argc, char** argv) {
    if (argc == 5 && !std::strcmp(argv[1], "choice")) {
        std::printf("%d\n", pipe_choice(std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4])));
        return 0;
    }
    long bad = 0, seen = 0;
    for (int tiles = 1; tiles <= kPipeRowTiles; ++tiles)
        for (int pairs = 1; pairs <= 256; ++pairs)
            for (int pair = 0; pair < pairs; ++pair)
                for (int t = 0; t < kPipeRowTiles; ++t) {
                    const int w = pipe_weight_offset(t, tiles, pairs, pair), wview = tiles * pairs * kQ8PairBytes;
                    const int d = pipe_scale_offset(t, tiles, pairs, pair), dview = tiles * pairs * kQ8PairScales;
                    bad += w < 0 || w >= wview || w + 63 * 16 + 16 > wview;
                    bad += d < 0 || d >= dview || d + 15 * 4 + 4 > dview;
                    if (t < tiles) bad += w != (t * pairs + pair) * 1024 || d != (t * pairs + pair) * 64;
                    ++seen;
                }
    for (int groups = 1; groups <= 512; ++groups)
        for (int tiles : {1, 2, 5, 128})
            for (int vt = 0; vt < tiles; ++vt)
                for (int group = 0; group < (groups + 1) / 2 * 2; ++group)
                    for (int part = 0; part < 2; ++part) {
                        const int x = pipe_vector_offset(vt, groups, group, part), view = tiles * groups * 2048;
                        bad += x < 0 || x >= view || x + 15 * 128 + 3 * 16 + 16 > view;
                        if (group < groups) bad += x != (vt * groups + group) * 2048 + part * 64;
                        ++seen;
                    }
    for (int tiles : {1, 2, 15, 16, 17, 36, 64, 128, 257, 1024, 2050, 8016})
        for (int groups : {1, 2, 3, 8, 18, 65, 256, 257, 512}) {
            const Q8Plan c = q8_plan(tiles, groups);
            bad += c.per % 4 || c.splits * c.per < groups || (c.splits - 1) * c.per >= groups || c.gx * c.rt < tiles;
            for (int n = 1; n <= 2100; ++n) {
                const int vt = pipe_choice(tiles, groups, n), first = (n - 1) / 16 * 16 + 1;
                bad += (vt != 0 && vt != 2 && vt != 4) || (vt && n <= 64) || vt != pipe_choice(tiles, groups, first);
                for (int most : {1, 8}) {
                    const PipePlan p = pipe_plan(tiles, groups, n, vt ? vt : 2, most);
                    bad += p.per % 2 || p.splits > most || p.splits * p.per < groups || (p.splits - 1) * p.per >= groups;
                    bad += p.splits != pipe_plan(tiles, groups, first, vt ? vt : 2, most).splits;
                }
                ++seen;
            }
        }
    std::printf("%s: %ld loads and plans, %ld wrong\n", bad ? "failed" : "passed", seen, bad);
    return bad != 0;
}
