// Host arithmetic of one-dimensional launches (no device code).
#pragma once
#include <cstddef>
#include <cstdint>

namespace vx {

// A launch dimension holds fewer than 2^32 threads: this many blocks of 256.
constexpr uint64_t kMaxBlocks256 = (1ull << 32) / 256 - 1;

// f(first, count) for the launches that `blocks` blocks of 256 threads take, in
// order, until one returns false; whether none did.
template <class F>
bool launch_pieces(uint64_t blocks, F f) {
    for (uint64_t first = 0; first < blocks; first += kMaxBlocks256) {
        const uint64_t left = blocks - first;
        if (!f((uint32_t)first, (uint32_t)(left < kMaxBlocks256 ? left : kMaxBlocks256))) return false;
    }
    return true;
}

// Blocks of k_clear_volume: 512 words of an array, 256 words of the march grid.
constexpr uint64_t clear_blocks(size_t words) { return ((uint64_t)words + 511) / 512; }
constexpr uint64_t clear_grid_blocks(size_t words) { return ((uint64_t)words + 255) / 256; }

}  // namespace vx
