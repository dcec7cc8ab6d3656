// Where the tiled Q8_0 product (batch_q8_pipe_kernel) reads its weights and
// vectors: plain arithmetic, shared with a host test that walks every shape.
//
// The kernel's buffer views cover one workgroup's row tiles, and all vectors; a
// load's tile is part of its scalar offset.  A raw buffer load compares its vector offset
// with what the view has left after the scalar one, which says nothing once
// the scalar offset is past the view; so a scalar offset always lies in it:
// row tiles past the matrix read its last one again, and their rows are not
// stored.
#pragma once

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

}  // namespace tvara_amd
