// Host check of block_of_piece (zfp_block.h) over every piece of a workgroup's blocks at every rate it serves.
#include <stdio.h>
#include "../cswap_amd/csrc/zfp_block.h"

int main()
{
  for (unsigned maxbits = 64; maxbits <= 4096; maxbits += 64) {
    const uint32_t by = cswap::piece_multiplier(maxbits), per_block = maxbits / 128;
    if (maxbits % 128) {
      if (by) return printf("%u bits\n", maxbits), 1;
      continue;
    }
    for (uint32_t p = 0; p < 64 * per_block; p++)
      if (cswap::block_of_piece(p, by) != p / per_block) return printf("%u bits, piece %u\n", maxbits, p), 1;
  }
  return 0;
}
