// Every load that batch_q8_pipe_kernel makes of a workgroup's weights and
// scales, by its own offsets (q8_pipe.hpp), against the bytes of its views:
// for every count of row tiles a workgroup can have and group pairs up to
// those of 16,384 columns, the scalar offset lies in the view and the furthest
// lane's read ends in it; row tiles that are there are read in their place.
// Likewise the vectors' halves, for even and odd counts of groups.
#include "q8_pipe.hpp"

#include <cstdio>
#include <initializer_list>

using namespace tvara_amd;

int main() {
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
    std::printf("%s: %ld loads, %ld outside their view\n", bad ? "failed" : "passed", seen, bad);
    return bad != 0;
}
