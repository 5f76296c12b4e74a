// Grids of blocks (block_grid): every block numbered, each dimension below 2^32
// lanes of 512 and 2^16 rows, no row wholly past the blocks.
#include <cstdio>

#include "../../exactdiagonalization.jl_amd/csrc/host_logic.hpp"

int main() {
  for (uint64_t columns : {0ull, 1ull, 3ull, 4ull, 1ull << 24, (1ull << 24) + 1, (1ull << 26) - 1, 1ull << 26, (1ull << 26) + 1,
                           77558760ull, 1ull << 32, 1ull << 34})
    for (uint64_t per_block : {4ull, 256ull}) {
      const uint64_t blocks = (columns + per_block - 1) / per_block;
      const edhip::BlockGrid g = edhip::block_grid(blocks);
      if ((uint64_t)g.x * g.y < blocks || (uint64_t)g.x * 512 >= 1ull << 32 || g.y >= 1u << 16 ||
          (g.y > 0 && (uint64_t)g.x * (g.y - 1) >= std::max<uint64_t>(blocks, 1)))
        return std::printf("%llu blocks: %u x %u\n", (unsigned long long)blocks, g.x, g.y), 1;
    }
  std::printf("ok\n");
  return 0;
}
