// How the products of a Q8_0 matrix by many vectors are laid out over the GPU,
// which kernel takes them, and where the tiled one (batch_q8_pipe_kernel) reads
// its operands: plain arithmetic, shared with a host test that walks the shapes.
//
// The tiled kernel's buffer views cover one workgroup's row tiles, and all
// vectors; a load's tile is part of its scalar offset.  A raw buffer load compares
// its vector offset with what the view has left after the scalar one, which says
// nothing once the scalar offset is past the view; so a scalar offset always lies
// in it: row tiles past the matrix read its last one again, and their rows are
// not stored.
#pragma once

#include <algorithm>

namespace tvara_amd {

constexpr int kPipeRowTiles = 16;                      // of a workgroup
constexpr int kQ8PairBytes = 1024, kQ8PairScales = 64;  // int8 weights and scales of a row tile's group pair

// row tile of the workgroup's `tiles` that stands for its tile `t`
constexpr int pipe_row_tile(int t, int tiles) { return t < tiles ? t : tiles - 1; }

// scalar offsets of group pair `pair` of row tile t in the views of the weights
// and of the scales; a lane adds 16 bytes times itself, or four times its row
constexpr int pipe_weight_offset(int t, int tiles, int pairs, int pair) {
    return (pipe_row_tile(t, tiles) * pairs + pair) * kQ8PairBytes;
}
constexpr int pipe_scale_offset(int t, int tiles, int pairs, int pair) {
    return (pipe_row_tile(t, tiles) * pairs + pair) * kQ8PairScales;
}

// scalar offset of the halves (part 0: hi, 1: lo) of a group of vector tile vt,
// which must exist; lane l adds 128 bytes times l%16 and 16 times l/16
constexpr int pipe_vector_offset(int vt, int groups, int group, int part) {
    return (vt * groups + (group < groups ? group : groups - 1)) * 2048 + part * 64;
}

// row tiles per workgroup and groups per K split of the batched Q8_0
// product: four row tiles from 1,024 tiles up, else two (more workgroups for
// the smaller matrices); the groups are split while the launch has fewer than
// 512 workgroups (two per CU), in whole chunks of four groups, never below
// eight groups and into at most eight splits (the epilogues read every split)
struct Q8Plan {
    int rt, gx, per, splits;
};
inline Q8Plan q8_plan(int tiles, int groups) {
    Q8Plan p{};
    p.rt = tiles >= 1024 ? 4 : 2;
    p.gx = (tiles + p.rt - 1) / p.rt;
    const int want = p.gx >= 512 ? 1 : std::min({(512 + p.gx - 1) / p.gx, std::max(1, groups / 8), 8});
    p.per = (groups + want - 1) / want;
    p.per = (p.per + 3) / 4 * 4;  // whole chunks, so splits start on a group pair
    p.splits = (groups + p.per - 1) / p.per;
    return p;
}

// Plan of the tiled GEMM with vt vector tiles a wave: K split while the launch
// has fewer than 256 workgroups (one a CU), into at most eight splits of at
// least eight groups
struct PipePlan {
    int vt, gx, per, splits;  // vector tiles a wave, workgroups per split, groups per split, splits
};
inline PipePlan pipe_plan(int tiles, int groups, int n, int vt, int most_splits = 8) {
    PipePlan p{};
    const int vtiles = (n + 15) / 16;
    p.vt = vt;
    p.gx = ((tiles + 15) / 16) * ((vtiles + 2 * vt - 1) / (2 * vt));
    const int want = std::min({std::max(1, 256 / p.gx), std::max(1, groups / 8), most_splits});
    p.per = ((groups + want - 1) / want + 1) / 2 * 2;  // whole pairs
    p.splits = (groups + p.per - 1) / p.per;
    return p;
}

// What multiplies n vectors: 0 for the chunked kernel, else the tiled GEMM's
// vector tiles a wave.  Above 64 vectors the one whose estimated time, in us, is
// the least.  The GEMM takes 1.0 (vt = 2) or 1.7 (vt = 4) a group pair of its
// split and round of the CUs, however few CUs there is work for, and 9 or 11
// around them; the chunked kernel 2 a thousand of its small workgroups and 0.2 a
// thousand row tiles x groups, for every block of 64 vectors, and 4 around
// them.  Each also pays for its partial sums (read at 4 TB/s by the epilogue),
// and the chunked one for halves written by lane.  MI355X, chunked / vt = 2 / vt
// = 4: 960 x 576 at 128 vectors 4.8 / 11.8 / 19.2, 2,048 x 2,048 at 128 8.6 /
// 12.0 / 18.2 and at 512 24.5 / 17.8 / 19.5, 16,384 x 2,048 at 128 30.1 / 25.8 /
// 28.4 and at 512 104.5 / 77.3 / 65.2.  Over 360 shapes from 512 x 512 to 28,672 x
// 4,096 at 65-2,048 vectors the choice is within 0.1% of the fastest in the
// geometric mean, 5% at worst; the GEMM for all, vt = 4 above 256 vectors, 37%.
// (Decided by the count of 16-vector tiles, for batch_part_floats.)
inline int pipe_choice(int tiles, int groups, int n) {
    if (n <= 64) return 0;
    const int vtiles = (n + 15) / 16, blocks = (vtiles + 3) / 4;
    const double sums = 1024e-6 / 4 * vtiles * tiles;
    auto partial = [&](int splits) { return splits > 1 ? splits * sums : 0.0; };
    const Q8Plan c = q8_plan(tiles, groups);
    double best = 4 + 0.02 * c.per + blocks * (2e-4 * tiles * groups + 2e-3 * c.gx * c.splits) + partial(c.splits) +
                  0.3e-6 * 2048 * vtiles * groups;
    int choice = 0;
    for (int vt : {2, 4}) {
        const PipePlan p = pipe_plan(tiles, groups, n, vt);
        const int rounds = (p.gx * p.splits + 255) / 256;
        const double us = (vt == 2 ? 9 + 1.0 * rounds * p.per / 2 : 11 + 1.7 * rounds * p.per / 2) + partial(p.splits);
        if (us < best) {
            best = us;
            choice = vt;
        }
    }
    return choice;
}

}  // namespace tvara_amd
