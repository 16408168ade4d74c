// Host check of zfp_runs.h: over whole fields, every element is stored once, from its own place in the image, and
// every index stays inside the image and the field.
#include <stdio.h>
#include <vector>
#include "../cswap_amd/csrc/zfp_runs.h"

using namespace cswap;

static bool field(uint32_t nx, uint32_t ny, uint32_t nz, uintptr_t base)
{
  const Runs p = make_runs(nx, ny, nz, base);
  const size_t plane = (size_t)nx * ny;
  std::vector<unsigned char> seen(plane * nz, 0);
  for (uint32_t g = 0; g < (p.block_rows + p.rows - 1) / p.rows; g++) {
    const RunsWave w = runs_wave(p, g);
    if (w.blocks < 1 || w.blocks > 64 || w.total < 1 || w.total > kRunsImageDwords / p.unit) return false;
    for (uint32_t z = 0; z < 4; z++) {
      std::vector<size_t> image(kRunsImageDwords, ~(size_t)0);
      for (uint32_t l = 0; l < 64; l++) {
        const uint32_t b = l < w.blocks ? l : w.blocks - 1, q = (w.first + b) / p.mx, s = q / p.my;
        for (uint32_t y = 0; y < 4; y++)
          for (uint32_t x = 0; x < 4; x++) {
            const size_t at = 4 * (runs_block(p, b) + y * p.mx) + x;
            if (at >= image.size()) return false;
            image[at] = (4 * s + z) * plane + (size_t)(4 * (q % p.my) + y) * nx + 4 * ((w.first + b) % p.mx) + x;
          }
      }
      const bool cut = z >= p.planes_last && w.cut != ~0u;
      if (cut && w.cut == 0) break;
      for (uint32_t i = 0; i < w.total; i++) {
        uint32_t from, to;
        runs_unit(p, w, i, from, to);
        const bool again = cut && to >= w.cut;
        if (again) from = 0, to = w.skip;
        for (uint32_t e = 0; e < p.unit; e++) {
          const size_t at = (4 * w.slab + z) * plane + (size_t)to * p.unit + e;
          if ((size_t)from * p.unit + e >= image.size() || at >= seen.size() || image[from * p.unit + e] != at) return false;
          if (!again) seen[at]++;
        }
      }
    }
  }
  for (unsigned char n : seen)
    if (n != 1) return false;
  return true;
}

int main()
{
  for (uint32_t v = 0; v < 2048; v++)
    for (uint32_t d = 1; d < 1024; d++)
      if (runs_quotient(v, runs_multiplier(d)) != v / d) return printf("%u / %u\n", v, d), 1;
  for (uint32_t nx = 2; nx <= 256; nx = nx < 37 ? nx + 1 : nx + 31)
    for (uint32_t ny : {1u, 3u, 4u, 7u, 14u, 17u, 35u, 1023u, 1024u, 1025u, 1500u})
      for (uint32_t nz : {1u, 4u, 6u, 63u})
        for (uintptr_t base : {4096u, 4100u, 4104u})
          if (!(nz == 63 && ny > 1000) && !field(nx, ny, nz, base)) return printf("%u x %u x %u at %u\n", nx, ny, nz, (unsigned)base), 1;
  return 0;
}
