// Grid of the depth-first kernel (enum.hip k_extend) and the launch setting dfs_blocks, which is its blocks.
#pragma once
#include <cstdint>

namespace csm {

constexpr uint32_t kDfsWaves = 2;  // waves per block: their LDS stacks stay under 64 KB at 16 depths
// By default 2,048 waves, what is resident when two launches share the chip; waves that start when the items are
// used up only contend for them.  Strategy 0, 8,192-edge batches on a 50K-vertex graph, per round trip: 64 blocks
// 23.7 ms, 128 18.7, 256 16.2, 512 16.5, 1024 17.2, 2048 20.0, 4096 25.5, 16384 56.
constexpr uint32_t kDfsBlocks = 1024, kMinDfsBlocks = 64, kMaxDfsBlocks = 16384;

// Blocks of a launch over `items` items at most: no more waves than items, unless an item is only a
// part of the work that its waves share (`whole`).
constexpr uint32_t dfs_grid(uint32_t blocks, uint64_t items, bool whole) {
    const uint64_t most = blocks < kMaxDfsBlocks ? blocks : kMaxDfsBlocks;
    const uint64_t need = (items + kDfsWaves - 1) / kDfsWaves;
    return static_cast<uint32_t>(whole || need > most ? most : need ? need : 1);
}

}  // namespace csm
