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

// The longest rows the kernels of direct loads take: their offsets within a tile's 256 rows have 32 bits.
constexpr int kRingRow = 1 << 23;

// Whether an ensemble's output layer (M x N over K inputs per member; alone: of one member) and its statistics are formed in one
// kernel, a block's members and k tiles one after the other, or member by member from products split over
// K.  The chain costs 0.22 to 0.32 us per 64 inputs whatever the tiles; a member's split product and
// statistics 12 us, 17 with their launches where the host bounds them, and more with every output, since
// its partials pass through memory.  us per prediction, one kernel / split (64 x 64 tiles in brackets): five
// members, 4096 inputs 128 / 145 (5), 8192 204 / 148 (5), 209 / 178 (32), 400 / 523 (99), 16384 361 / 189 (5),
// 606 / 369 (32), 859 / 650 (128), 707 / 900 (313), 65536 1848 / 316 (5), 2390 / 1128 (128); one member, 2048
// inputs 90 / 93 (1), 3072 101 / 86 (1), 4096 105 / 98 (1).
constexpr int kOutputChain = 4096, kOutputChainAlone = 2048, kOutputChainTile = 64;
inline bool ensemble_in_registers(int M, int N, int K, bool alone = false)
{
    const long long tiles = ((M + 63) / 64) * (long long)((N + 63) / 64);
    return K <= kRingRow && K <= (alone ? kOutputChainAlone : kOutputChain) + kOutputChainTile * tiles;
}

}  // namespace mlp
}  // namespace poe2d
