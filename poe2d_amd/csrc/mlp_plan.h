// Host arithmetic of the network's transfers and launches (no device code, no HIP types).
#pragma once

#include <algorithm>
#include <cstddef>

namespace poe2d {
namespace mlp {

// The piece of a rows x cols copy that goes through `floats` values of staging at a time: as many whole
// rows as fit, or, where a row is longer than that (a network without hidden layers has little workspace),
// part of one.
struct Piece {
    int rows, cols;
};
inline Piece staging_piece(size_t floats, int rows, int cols)
{
    if (floats >= (size_t)cols) return {(int)std::min<size_t>(rows, floats / cols), cols};
    return {1, (int)floats};
}

// Rows of a prediction whose inputs (`in` values each) are on the device at a time: all n, or as many
// batches as kInputFloats hold, at least one.
constexpr size_t kInputFloats = size_t(16) << 20;
inline int predict_stretch(int n, int in, int batch)
{
    const size_t batches = std::max<size_t>(kInputFloats / in / batch, 1);
    return (int)std::min<size_t>(n, batches * batch);
}

}  // namespace mlp
}  // namespace poe2d
