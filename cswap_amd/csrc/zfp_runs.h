// zfp_runs.h -- how a wavefront of the decoder stores whole block rows of a packed field as runs of memory.
//
// Host and device: the tests walk the same functions over whole fields on the CPU.
#ifndef CSWAP_ZFP_RUNS_H
#define CSWAP_ZFP_RUNS_H

#include "zfp_block.h"

namespace cswap {

// A wavefront takes `rows` consecutive block rows (mx blocks each, so that at most 64 lanes have a block).
// One plane of them at a time stands in LDS as whole blocks, 4 * mx elements to a row ("the image").  In memory a
// plane of them is a run per slab of four planes that they lie in; the run's elements are counted
// through all slabs, in units of `unit` elements that never cross the end of a row.
struct Runs {
  uint32_t rows, block_rows;         // per wavefront, of the field
  uint32_t mx, my, ny;
  uint32_t lane_mul;                 // lane * lane_mul >> 16 = lane / mx
  uint32_t unit;                     // 4, 2 or 1 elements
  uint32_t width, plane;             // a row and a plane, in units
  uint32_t row_more, slab_more;      // what the image has more than memory, per row and per slab, in units
  uint32_t slab_step;                // from the end of a slab's plane to the start of the same plane of the next, in units
  uint32_t planes_last;              // planes of the last slab that exist, 1 to 4
  uint32_t last_row;                 // the first block row of the last slab
  uint32_t by_width, by_slab;        // multipliers of runs_quotient
  Div31 by_my;
};
constexpr uint32_t kRunsImageDwords = 64 * 16;

// v / d for v < 2^11 and d < 2^10 in one 24-bit multiplication, mul = ceil(2^23 / d): v * mul is above
// v * 2^23 / d by less than v < 2^23 / d, which is how far v / d stays below the next whole number, times 2^23.
inline uint32_t runs_multiplier(uint32_t d) { return ((1u << 23) + d - 1) / d; }
CSWAP_HD uint32_t runs_quotient(uint32_t v, uint32_t mul)
{
  return (uint32_t)(((uint64_t)((v << 9) & 0xffffffu) * (mul & 0xffffffu)) >> 32);
}

constexpr uint32_t kRunsPlaneElements = 1u << 22;  // three planes of fewer are counted in 24 bits

// nx <= 256, nx * ny < kRunsPlaneElements; base: the address of the field, looked at for its alignment
inline Runs make_runs(uint32_t nx, uint32_t ny, uint32_t nz, uintptr_t base)
{
  Runs r;
  r.mx = (nx + 3) / 4;
  r.my = (ny + 3) / 4;
  r.ny = ny;
  const uint32_t mz = (nz + 3) / 4;
  r.rows = 64 / r.mx;
  r.block_rows = r.my * mz;
  r.lane_mul = (65536 + r.mx - 1) / r.mx;
  r.unit = (nx % 4 == 0 && base % 16 == 0) ? 4 : (nx % 2 == 0 && base % 8 == 0) ? 2 : 1;
  r.width = nx / r.unit;
  r.plane = r.width * ny;
  const uint32_t pitch = 4 * r.mx / r.unit;
  r.row_more = pitch - r.width;
  r.slab_more = (4 * r.my - ny) * pitch;
  r.slab_step = 3 * r.plane;
  r.planes_last = nz - 4 * (mz - 1);
  r.last_row = r.my * (mz - 1);
  r.by_width = runs_multiplier(r.width);
  r.by_slab = runs_multiplier(ny < 1024 ? ny : 512);
  r.by_my = make_div31(r.my);
  return r;
}

// One wavefront's share.
struct RunsWave {
  uint32_t slab;           // of its first block row
  uint32_t first, blocks;  // its blocks
  uint32_t skip;           // units of the slab's plane in front of its first row
  uint32_t phase;          // the rows of a plane of the slab that are left reach a multiple of the divisor of by_slab at its end
  uint32_t total;          // units of one plane, through all its slabs
  uint32_t cut;            // if it has rows of the field's last slab: where its planes begin in memory, as runs_unit counts, else ~0
};
CSWAP_HD RunsWave runs_wave(const Runs& p, uint32_t wave)
{
  RunsWave w;
  const uint32_t q0 = wave * p.rows;
  const uint32_t q1 = q0 + p.rows < p.block_rows ? q0 + p.rows : p.block_rows;
  w.slab = div31(q0, p.by_my);
  const uint32_t row = q0 - w.slab * p.my;
  w.first = q0 * p.mx;
  w.blocks = (q1 - q0) * p.mx;
  w.skip = 4 * row * p.width;
  // A wavefront has 256 rows at most.  Planes of 1024 and more are left once or not at all: 512 stands for them,
  // counted so that it is reached where the plane ends.
  w.phase = p.ny < 1024 ? 4 * row : 4 * row + 512 > p.ny ? 4 * row + 512 - p.ny : 0;
  const uint32_t s1 = div31(q1 - 1, p.by_my), y1 = q1 - s1 * p.my;  // the last block row, and the one behind it in that slab
  const uint32_t end = 4 * y1 < p.ny ? 4 * y1 : p.ny;
  w.total = (s1 - w.slab) * p.plane + end * p.width - w.skip;
  w.cut = q1 <= p.last_row ? ~0u : 4 * (s1 - w.slab) * p.plane;
  return w;
}

// a * b + c, a and b below 2^24: a 32-bit multiplication takes the vector unit four times as long, and the compiler
// cannot see that these fit.  b is the same for the whole wavefront.
CSWAP_HD uint32_t runs_mad(uint32_t a, uint32_t b, uint32_t c)
{
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t r;
  asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
#else
  return a * b + c;
#endif
}
// Unit i of a plane: where it stands in the image, and how far behind the first slab's plane in memory.
CSWAP_HD void runs_unit(const Runs& p, const RunsWave& w, uint32_t i, uint32_t& image, uint32_t& memory)
{
  const uint32_t r = runs_quotient(i, p.by_width);  // rows follow each other through the slabs
  const uint32_t k = runs_quotient(r + w.phase, p.by_slab);
  image = runs_mad(k, p.slab_more, runs_mad(r, p.row_more, i));
  memory = runs_mad(k, p.slab_step, i + w.skip);
}
// A block's first row in the image, in pieces of 16 bytes; its row y stands y * mx further
CSWAP_HD uint32_t runs_block(const Runs& p, uint32_t block)
{
  const uint32_t j = (block * p.lane_mul) >> 16;
  return block + 3 * j * p.mx;
}

}  // namespace cswap
#endif
