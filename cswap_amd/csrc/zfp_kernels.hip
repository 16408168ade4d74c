// zfp_kernels.hip -- ZFP fixed-rate fp32 3-D encode / decode for gfx950.
//
// Work decomposition: one wavefront (64 lanes) per group of 64 consecutive
// blocks, ONE LANE PER BLOCK.  A lane keeps its 64 coefficients in registers
// through cast, lifting, reorder, bit transpose and the embedded coder
// (zfp_block.h), so there is no cross-lane traffic at all.  The wave's slice of
// the stream (64 blocks x maxbits bits = maxbits 64-bit words, always a whole
// number of words) is staged in LDS, which the coder addresses bit by bit, and
// moved to/from HBM in 16-byte pieces.  Because the stream is fixed-rate,
// stream offsets are closed-form and no device-wide scan, atomic or memset of
// the stream is needed (the reference pre-zeroes the stream and adds every bit
// with a global atomic, CSWAP+/zfp/encode.cuh:252-299, encode3.cuh:152).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include "../../include/cswap_hip.h"
#include "../../include/cswap_test_hooks.h"
#include "zfp_block.h"
#include "zfp_runs.h"
#include "common.h"

namespace cswap {

struct Field3 {
  uint32_t nx, ny, nz;     // extents in elements
  uint32_t mx, my;         // blocks along x and y
  uint32_t nblocks;
  long long sx, sy, sz;    // strides in elements
  int rows16;              // 1: x-rows of every block are contiguous and 16-byte aligned, rows nest inside
                           //    planes inside the volume, and any 64 consecutive blocks lie within 4 GiB
  int rows4;               // 1: as rows16, but the rows may start at any element, and nx >= 2
  int full;                // 1: rows4, and every block is a full one
  int stream16;            // 1: the stream pointer is 16-byte aligned
  uint32_t by_piece;       // whole-word rates with an even number of words per block, else 0: the multiplier of block_of_piece
  int read_once;           // 1: a field of kReadOnceBytes and more (see make_field)
  int store_hint;          // 1: the 32-bit decoder stores the field's rows with the nontemporal hint (row_store_hint)
  int once64;              // 1: the decoder of 64-bit elements should store its rows with the hint (see make_field)
  Div31 by_mx, by_my;      // block index -> block coordinates without a hardware divide
};

// Fields of at least this many bytes are loaded with the nontemporal hint (make_field)
#ifndef CSWAP_READ_ONCE_BYTES
#define CSWAP_READ_ONCE_BYTES (128ull << 20)
#endif
constexpr unsigned long long kReadOnceBytes = CSWAP_READ_ONCE_BYTES;

// Fields below this many bytes are coded by the pair form (two wavefronts per 64 blocks)
#ifndef CSWAP_PAIR_ENCODE_BYTES
#define CSWAP_PAIR_ENCODE_BYTES (40ull << 20)
#endif
#ifndef CSWAP_PAIR_DECODE_BYTES
#define CSWAP_PAIR_DECODE_BYTES (40ull << 20)   // and only where pair_decode_pays
#endif

// 16 bytes of the field as the compiler's own vector type (what the nontemporal builtins take)
typedef float stream_f4 __attribute__((ext_vector_type(4)));
// the same and its shorter brothers where only 4-byte alignment is known: still one instruction each
typedef float row_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float row_f2 __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned long long stream_u2 __attribute__((ext_vector_type(2)));

// ------------------------------------------------------------- LDS adapter
// The bit region the block codec ORs into / reads from is LDS: it serves as the
// dynamically indexable extension of the register file (a lane cannot index
// its registers with a run-time bit position).  The codec hands over the byte
// offset of a dword as the LDS address itself, so bit positions count from LDS
// address 0: a block's first bit is bit0 + its offset within the region.  (With
// a pointer to the region plus an offset, every access would cost one more
// instruction that adds the region's address.)
typedef __attribute__((address_space(3))) uint32_t lds_u32;
struct LdsBits {
  unsigned bit0;  // bit position of the region's first bit
  __device__ __forceinline__ explicit LdsBits(uint32_t* region)
      : bit0(8u * (unsigned)(size_t)(__attribute__((address_space(3))) void*)region)
  {
  }
  __device__ __forceinline__ static lds_u32* at(unsigned d) { return (lds_u32*)(size_t)d; }
  __device__ __forceinline__ void or32(unsigned d, uint32_t v) const
  {
    __hip_atomic_fetch_or(at(d), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);  // ds_or_b32
  }
  __device__ __forceinline__ uint32_t ld32(unsigned d) const { return *at(d); }
};

// The same with the codec's table of expanded bytes (zfp_block.h: expand8) in front of the region: 512
// bytes per workgroup, a 16-bit read per byte.  Most bytes are zero, so most lanes read one address.
typedef uint16_t table_u16 __attribute__((may_alias));  // the table's pieces are written 8 bytes at a time
struct LdsBitsTable : LdsBits {
  static constexpr bool kExpands = true;
  const table_u16* table;
  __device__ __forceinline__ LdsBitsTable(uint32_t* region, const uint2* pieces)
      : LdsBits(region), table(reinterpret_cast<const table_u16*>(pieces))
  {
  }
  __device__ __forceinline__ uint32_t expanded(uint32_t word, int k) const { return table[(word >> (8 * k)) & 0xffu]; }
};
__constant__ const ExpandTable kExpandTable = make_expand_table();
// A lane's 8 bytes of the table: asked for before anything else, written to LDS when the region is cleared.
__device__ __forceinline__ uint2 table_piece(unsigned lane)
{
  uint2 piece;
  __builtin_memcpy(&piece, kExpandTable.v + 4 * lane, sizeof piece);
  return piece;
}

// For decoding, with the table of collapsed bytes: 256 bytes.
struct LdsBitsCollapse : LdsBits {
  static constexpr bool kCollapses = true;
  const uint8_t* table;
  __device__ __forceinline__ LdsBitsCollapse(uint32_t* region, const uint32_t* t)
      : LdsBits(region), table(reinterpret_cast<const uint8_t*>(t))
  {
  }
  __device__ __forceinline__ uint32_t collapsed(uint32_t word, int k) const { return table[(word >> (8 * k)) & 0xffu]; }
};
__constant__ const CollapseTable kCollapseTable = make_collapse_table();
__device__ __forceinline__ uint32_t collapse_piece(unsigned lane)
{
  uint32_t piece;
  __builtin_memcpy(&piece, kCollapseTable.v + 4 * lane, sizeof piece);
  return piece;
}
// What stands behind every block in the decoder's region.  A one, for the run that the budget cuts short, and zeros.
constexpr uint64_t kFence = 1;

// Layout of the wave's LDS bit region.
//  whole-word rates (maxbits % 64 == 0): every lane owns a private slot of
//    maxbits + slack bits (slot a multiple of 128 bits), so the coder needs no
//    end-of-block guards and each lane moves its own words to/from HBM;
//  other rates: the 64 blocks are packed back to back exactly as in the stream
//    (always a whole number of words per wave) and moved cooperatively.
__host__ __device__ inline unsigned slot_bits(unsigned maxbits)
{
  return (maxbits & 63u) ? maxbits : ((maxbits + 128u + 127u) & ~127u);
}
__host__ __device__ inline unsigned region_dwords(unsigned maxbits)
{
  return ((2u * slot_bits(maxbits) + 4u) + 3u) & ~3u;  // + padding of 128 bits for what reads and OR-ed zeros reach past the last slot
}
// The 32-bit decoder's slot is the block and its fence (kFence), nothing more: its
// reads reach up to 128 bits further, into the next lane's block (or the region's
// padding of as many bits), and those bits are never looked at.  The stride is then 2 (mod 4)
// dwords at even word counts.  Against slots as the encoder's: 10 bits per value 50 MB 16.0 / 16.7 us,
// 100 MB 26.9 / 27.5; at 4, 8, 16, 24 and 32 level or up to 1 % ahead.  Slots are 8-byte aligned only.
__host__ __device__ inline unsigned dec_slot_bits(unsigned maxbits)
{
  return (maxbits & 63u) ? maxbits : maxbits + 64u;
}
__host__ __device__ inline unsigned dec_region_dwords(unsigned maxbits)
{
  return ((2u * dec_slot_bits(maxbits) + 4u) + 3u) & ~3u;
}

// ------------------------------------------------------------- block <-> field
__device__ __forceinline__ void block_origin(const Field3& fd, uint32_t b, uint32_t& x0, uint32_t& y0,
                                             uint32_t& z0)
{
  uint32_t q = div31(b, fd.by_mx);
  x0 = (b - q * fd.mx) * 4;
  uint32_t r = div31(q, fd.by_my);
  y0 = (q - r * fd.my) * 4;
  z0 = r * 4;
}

// Addressing of the fast path (Field3::rows16): the wavefront's first block gives
// a wave-uniform 64-bit base, every lane adds a 32-bit byte offset to it.  Block
// order is x, then y, then z and the strides nest, so offsets grow with the block
// index; the host only sets rows16 when 64 consecutive blocks span less than 4 GiB.
struct WaveBase {
  long long origin;  // element offset of the first block's corner
  uint32_t fx, fy, fz;
};
__device__ __forceinline__ WaveBase wave_base(const Field3& fd, uint32_t first)
{
  WaveBase w;
  block_origin(fd, first, w.fx, w.fy, w.fz);
  w.origin = (long long)w.fx + (long long)w.fy * fd.sy + (long long)w.fz * fd.sz;
  return w;
}
__device__ __forceinline__ uint32_t lane_bytes(const Field3& fd, const WaveBase& w, uint32_t x0, uint32_t y0,
                                               uint32_t z0)
{
  return ((x0 - w.fx) + (y0 - w.fy) * (uint32_t)fd.sy + (z0 - w.fz) * (uint32_t)fd.sz) * 4u;  // mod 2^32
}

template <bool ONCE>
__device__ __forceinline__ void load_block(const float* __restrict__ in, const Field3& fd, uint32_t first,
                                           uint32_t b, float (&f)[64])
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  if (fd.rows16 && bx == 4 && by == 4 && bz == 4) {
    const WaveBase w = wave_base(fd, first);
    const char* base = reinterpret_cast<const char*>(in + w.origin);
    const uint32_t mine = lane_bytes(fd, w, x0, y0, z0);
    const uint32_t sy4 = (uint32_t)fd.sy * 4u, sz4 = (uint32_t)fd.sz * 4u;
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++) {
        const stream_f4* src = reinterpret_cast<const stream_f4*>(base + (size_t)(mine + (y * sy4 + z * sz4)));
        const stream_f4 v = ONCE ? __builtin_nontemporal_load(src) : *src;
        f[16 * z + 4 * y + 0] = v.x;
        f[16 * z + 4 * y + 1] = v.y;
        f[16 * z + 4 * y + 2] = v.z;
        f[16 * z + 4 * y + 3] = v.w;
      }
  } else {
    const float* p = in + (long long)x0 * fd.sx + (long long)y0 * fd.sy + (long long)z0 * fd.sz;
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int x = 0; x < 4; x++) {
          bool ok = (uint32_t)x < bx && (uint32_t)y < by && (uint32_t)z < bz;
          f[16 * z + 4 * y + x] = ok ? p[x * fd.sx + y * fd.sy + z * fd.sz] : 0.0f;
        }
    if (bx < 4 || by < 4 || bz < 4) pad_block3(f, bx, by, bz);
  }
}

// Where the four rows (planes) of a block that has only n of them along this axis are read
// from, in bytes from the first one at a distance of s bytes: the padding rule (pad4) as
// addresses.  n = 1: a,a,a,a; 2: a,b,b,a; 3: a,b,c,a.
__device__ __forceinline__ void padded_offsets(uint32_t n, uint32_t s, uint32_t (&off)[4])
{
  off[0] = 0;
  off[1] = n >= 2 ? s : 0;
  off[2] = n >= 3 ? 2 * s : off[1];
  off[3] = n >= 4 ? 3 * s : 0;
}

// Fields of contiguous rows that are not all full blocks of aligned rows (odd feature maps and
// the like) take the same 16-byte loads and stores, with two changes.  A row may start at any
// element: the instruction needs 4-byte alignment only.  Where a block is cut off along y or z
// its padding is read from the addresses the padding rule names; along x the row is read whole
// -- its end is the start of the next row, or what lies between rows -- and the padding is
// selected in registers.  Only blocks whose reads would leave the field (the last block along
// all three axes) go element by element.  nx = 1 stays out: four elements are up to four rows
// there, and other blocks than the last could leave the field.  Against one predicated 4-byte
// access per element with its own 64-bit address, at 8 bits per value and with the coders that step from
// run to run: 60 MB in 35x35 planes encoded in 26.2 instead of 28.1 us and decoded in 26.4 instead of 39.8,
// 321 MB of them in 90 instead of 108 and 119 instead of 166; 26 MB in 14x14 planes 16.9 / 19.6 and 18.7 / 26.5.
// Now: 60 MB in 35x35 planes 21.9 and 22.9, 26 MB in 14x14 13.3 and 16.2.  (Packed fields are decoded by zfp_decode3_runs_kernel where
// that is faster.)
__device__ __forceinline__ void load_row(const char* src, float (&f)[64], int row)
{
  const row_f4* p = reinterpret_cast<const row_f4*>(src);
  const row_f4 v = *p;
  f[4 * row + 0] = v.x;
  f[4 * row + 1] = v.y;
  f[4 * row + 2] = v.z;
  f[4 * row + 3] = v.w;
}

__device__ __forceinline__ void load_block_rows(const float* __restrict__ in, const Field3& fd, uint32_t first, uint32_t b,
                                                float (&f)[64])
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  const uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  const bool leaves = bx < 4 && y0 + by == fd.ny && z0 + bz == fd.nz;  // its last row is the field's, and is cut off
  if (leaves) {
    load_block<false>(in, fd, first, b, f);
    return;
  }
  const WaveBase w = wave_base(fd, first);
  const char* base = reinterpret_cast<const char*>(in + w.origin);
  const uint32_t mine = lane_bytes(fd, w, x0, y0, z0);
  uint32_t yo[4], zo[4];
  padded_offsets(by, (uint32_t)fd.sy * 4u, yo);
  padded_offsets(bz, (uint32_t)fd.sz * 4u, zo);
#pragma unroll
  for (int z = 0; z < 4; z++)
#pragma unroll
    for (int y = 0; y < 4; y++) load_row(base + (size_t)(mine + yo[y] + zo[z]), f, y + 4 * z);
  if (fd.nx & 3u) {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      f[4 * r + 1] = bx >= 2 ? f[4 * r + 1] : f[4 * r];
      f[4 * r + 2] = bx >= 3 ? f[4 * r + 2] : f[4 * r + 1];
      f[4 * r + 3] = bx >= 4 ? f[4 * r + 3] : f[4 * r];
    }
  }
}

// one x-row of an int32 block: last lifting pass, values handed on as bit patterns
__device__ __forceinline__ void decode_row_i32(int32_t (&ib)[64], int row, float (&f)[4])
{
  inv_lift4(ib[4 * row], ib[4 * row + 1], ib[4 * row + 2], ib[4 * row + 3]);
#pragma unroll
  for (int x = 0; x < 4; x++) f[x] = __int_as_float(ib[4 * row + x]);
}

// Finishes the block (inverse lifting along x, cast) and stores it.  Every
// x-row is finished and stored on its own, so the finished values never all
// sit in registers at once.
template <bool INT>
__device__ __forceinline__ void finish_and_store_block(float* __restrict__ out, const Field3& fd, uint32_t first,
                                                       uint32_t b, int32_t (&ib)[64], float w)
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  if (fd.rows16 && bx == 4 && by == 4 && bz == 4) {
    const WaveBase wb = wave_base(fd, first);
    char* base = reinterpret_cast<char*>(out + wb.origin);
    const uint32_t mine = lane_bytes(fd, wb, x0, y0, z0);
    const uint32_t sy4 = (uint32_t)fd.sy * 4u, sz4 = (uint32_t)fd.sz * 4u;
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++) {
        float r[4];
        if (INT) decode_row_i32(ib, y + 4 * z, r);
        else decode_row(ib, y + 4 * z, w, r);
        const stream_f4 v = {r[0], r[1], r[2], r[3]};
        __builtin_nontemporal_store(v, reinterpret_cast<stream_f4*>(base + (size_t)(mine + (y * sy4 + z * sz4))));
      }
  } else {
    float* p = out + (long long)x0 * fd.sx + (long long)y0 * fd.sy + (long long)z0 * fd.sz;
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++) {
        float r[4];
        if (INT) decode_row_i32(ib, y + 4 * z, r);
        else decode_row(ib, y + 4 * z, w, r);
#pragma unroll
        for (int x = 0; x < 4; x++)
          if ((uint32_t)x < bx && (uint32_t)y < by && (uint32_t)z < bz) p[x * fd.sx + y * fd.sy + z * fd.sz] = r[x];
      }
  }
}

// The same where rows start at any element or end inside a block.  The hint is for aligned rows:
// elsewhere it leaves partial lines to memory (60 MB in 35x35 planes 27.9 us with it, 26.4 without; 321 MB 149 and 119).
template <bool INT, bool HINT>
__device__ __forceinline__ void finish_and_store_rows(float* __restrict__ out, const Field3& fd, uint32_t first, uint32_t b,
                                                      int32_t (&ib)[64], float w)
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  const uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  const WaveBase wb = wave_base(fd, first);
  char* base = reinterpret_cast<char*>(out + wb.origin);
  const uint32_t mine = lane_bytes(fd, wb, x0, y0, z0);
  const uint32_t sy4 = (uint32_t)fd.sy * 4u, sz4 = (uint32_t)fd.sz * 4u;
#pragma unroll
  for (int z = 0; z < 4; z++)
#pragma unroll
    for (int y = 0; y < 4; y++) {
      float r[4];
      if (INT) decode_row_i32(ib, y + 4 * z, r);
      else decode_row(ib, y + 4 * z, w, r);
      if ((uint32_t)y < by && (uint32_t)z < bz) {
        float* dst = reinterpret_cast<float*>(base + (size_t)(mine + (y * sy4 + z * sz4)));
        if (bx == 4) {
          const row_f4 v = {r[0], r[1], r[2], r[3]};
          if (HINT) __builtin_nontemporal_store(v, reinterpret_cast<row_f4*>(dst));
          else *reinterpret_cast<row_f4*>(dst) = v;
        } else if (fd.nx & 2u) {
          const row_f2 v = {r[0], r[1]};
          *reinterpret_cast<row_f2*>(dst) = v;
          if (fd.nx & 1u) dst[2] = r[2];
        } else {
          dst[0] = r[0];
        }
      }
    }
}

// ------------------------------------------------------------- LDS region <-> stream
__device__ __forceinline__ void zero_region(uint4* lds_raw, unsigned lane, unsigned maxbits)
{
  const unsigned n16 = region_dwords(maxbits) / 4;
  for (unsigned i = lane; i < n16; i += 64) lds_raw[i] = make_uint4(0, 0, 0, 0);
}

// The blocks of a workgroup lie one behind the other in the stream, so its threads can move them as one
// run of 16-byte pieces, thread t the pieces t, t + threads, ...: every instruction covers whole lines,
// where lanes that move the words of their own block touch another line than their neighbour in each of
// their instructions (64 lines at 16 bits per value, 32 at 8).  Four pieces at a time, all asked for
// before the first is used: one by one, a stream that comes from memory costs its latency four times
// (402.7 MB at 8 bits, from a cold stream, decoded in 104 us by own words, 109 one piece at a time, 92 four).
// The decoder, own words -> pieces: 402.7 MB at 8 bits 88.9 -> 83.1 us (104 -> 92 cold), 201.3 MB 49.4 -> 45.0, at 16
// bits 75.9 -> 62.7 (85 -> 71 cold), 50.3 MB 17.9 -> 17.3, at 16 bits 24.4 -> 20.3.  The encoder: 201.3 MB at 8 bits
// 49.3 -> 47.2, at 16 bits 72.2 -> 65.5, 402.7 MB 92.7 -> 89.3, 50.3 MB 17.8 -> 17.5.
// PAD: dwords between the blocks of the region.
template <unsigned PAD>
__device__ __forceinline__ uint32_t piece_dword(uint32_t p, uint32_t by)
{
  return 4 * p + PAD * (__umul24(p, by) >> 16);  // block_of_piece
}

// stream: the workgroup's first block.  B pieces of every thread; past the last piece all move that one.
template <unsigned B, unsigned THREADS, unsigned PAD>
__device__ __forceinline__ void store_batch(const uint32_t* lds, unsigned p0, unsigned last, uint32_t by, char* __restrict__ dst)
{
  ulonglong2 v[B];
  unsigned p[B];
#pragma unroll
  for (unsigned k = 0; k < B; k++) {
    p[k] = min(p0 + k * THREADS, last);
    v[k] = *reinterpret_cast<const ulonglong2*>(lds + piece_dword<PAD>(p[k], by));
  }
#pragma unroll
  for (unsigned k = 0; k < B; k++) *reinterpret_cast<ulonglong2*>(dst + (size_t)(16u * p[k])) = v[k];
}

template <unsigned B, unsigned THREADS, unsigned PAD>
__device__ __forceinline__ void load_batch(uint32_t* lds, unsigned p0, unsigned last, uint32_t by, const char* __restrict__ src)
{
  ulonglong2 v[B];
  unsigned p[B];
#pragma unroll
  for (unsigned k = 0; k < B; k++) {
    p[k] = min(p0 + k * THREADS, last);
    v[k] = *reinterpret_cast<const ulonglong2*>(src + (size_t)(16u * p[k]));
  }
#pragma unroll
  for (unsigned k = 0; k < B; k++) {
    uint64_t* dst = reinterpret_cast<uint64_t*>(lds + piece_dword<PAD>(p[k], by));
    dst[0] = v[k].x;
    dst[1] = v[k].y;
  }
}

template <unsigned THREADS, unsigned PAD>
__device__ __forceinline__ void store_pieces(const uint32_t* lds, unsigned t, uint32_t valid, unsigned maxbits, uint32_t by,
                                             uint64_t* __restrict__ stream)
{
  const unsigned all = 64 * (maxbits >> 7), last = valid * (maxbits >> 7) - 1;
  char* dst = reinterpret_cast<char*>(stream);
  unsigned i = 0;
  for (; i + 4 * THREADS <= all; i += 4 * THREADS) store_batch<4, THREADS, PAD>(lds, i + t, last, by, dst);
  for (; i < all; i += THREADS) store_batch<1, THREADS, PAD>(lds, i + t, last, by, dst);
}

template <unsigned THREADS, unsigned PAD>
__device__ __forceinline__ void load_pieces(uint32_t* lds, unsigned t, uint32_t valid, unsigned maxbits, uint32_t by,
                                            const uint64_t* __restrict__ stream)
{
  const unsigned all = 64 * (maxbits >> 7), last = valid * (maxbits >> 7) - 1;
  const char* src = reinterpret_cast<const char*>(stream);
  unsigned i = 0;
  for (; i + 4 * THREADS <= all; i += 4 * THREADS) load_batch<4, THREADS, PAD>(lds, i + t, last, by, src);
  for (; i + 2 * THREADS <= all; i += 2 * THREADS) load_batch<2, THREADS, PAD>(lds, i + t, last, by, src);
  for (; i < all; i += THREADS) load_batch<1, THREADS, PAD>(lds, i + t, last, by, src);
}
constexpr unsigned kSlackDwords = 4, kFenceDwords = 2;  // slot_bits and dec_slot_bits at whole-word rates of even word counts

// the wave's coded blocks from LDS to the stream
template <bool WHOLE>
__device__ __forceinline__ void store_region(const uint32_t* lds, unsigned lane, uint32_t first, uint32_t valid,
                                             unsigned maxbits, const Field3& fd, uint64_t* __restrict__ stream)
{
  if (WHOLE) {
    const unsigned W = maxbits >> 6;
    if (fd.by_piece && fd.stream16) {
      store_pieces<64, kSlackDwords>(lds, lane, valid, maxbits, fd.by_piece, stream + (size_t)first * W);
    } else if (lane < valid) {  // an odd number of words, or a stream off 16 bytes: each lane stores its own block's
      const uint64_t* src = reinterpret_cast<const uint64_t*>(lds + lane * (slot_bits(maxbits) / 32));
      uint64_t* dst = stream + (size_t)(first + lane) * W;
      for (unsigned j = 0; j < W; j++) dst[j] = src[j];
    }
  } else {
    const unsigned nwords = (valid * maxbits + 63u) >> 6;
    const uint64_t* src = reinterpret_cast<const uint64_t*>(lds);
    uint64_t* dst = stream + (size_t)(first >> 6) * maxbits;
    for (unsigned i = lane; i < nwords; i += 64) dst[i] = src[i];
  }
}

// the wave's coded blocks from the stream into LDS; whole-word rates get the
// fence behind every block that the fenced decoder relies on
template <bool WHOLE, unsigned PAD>
__device__ __forceinline__ void load_region(uint32_t* lds, unsigned lane, uint32_t first, uint32_t valid,
                                            unsigned maxbits, unsigned slot, const Field3& fd,
                                            const uint64_t* __restrict__ stream)
{
  if (WHOLE) {
    const unsigned W = maxbits >> 6;
    uint64_t* dst = reinterpret_cast<uint64_t*>(lds + lane * (slot / 32));
    if (fd.by_piece && fd.stream16) {
      load_pieces<64, PAD>(lds, lane, valid, maxbits, fd.by_piece, stream + (size_t)first * W);
    } else if (lane < valid) {
      const uint64_t* src = stream + (size_t)(first + lane) * W;
      for (unsigned j = 0; j < W; j++) dst[j] = src[j];
    }
    if (lane < valid) dst[W] = kFence;
  } else {
    const unsigned nwords = (valid * maxbits + 63u) >> 6;
    const uint64_t* src = stream + (size_t)(first >> 6) * maxbits;
    uint64_t* dst = reinterpret_cast<uint64_t*>(lds);
    for (unsigned i = lane; i < nwords + 2; i += 64) dst[i] = i < nwords ? src[i] : 0;
  }
}

// ------------------------------------------------------------- kernels
// grid.x = ceil(nblocks/64) workgroups of one wavefront; dynamic LDS =
// region_dwords(maxbits) dwords.
// INT: the field holds int32 values (moved as 32-bit patterns through the same loads and stores)
// ONCE: the field is loaded with the nontemporal hint (Field3::read_once)
// WPE: wavefronts per SIMD the kernel is built for and held to.  Five, except from 16 bits
// per value on: there a wavefront's LDS region (9 KB and more) lets 16 or 17 wavefronts
// into a compute unit, unevenly over its SIMDs.  The encoder, three / four / five per SIMD, us, one tensor over
// and over (several in turn): 16 bits 100 MB 32.0 / 30.9 / 33.2 (35.2 / 34.8 / 35.7), 201 MB 57.2 / 55.4 / 57.8 (59.1 / 58.5 / 60.1); 24 bits 37.7 / 39.4 /
// 41.0 (42.2 / 43.4 / 44.4), 66.2 / 67.6 / 68.6; 32 bits 45.7 / 47.0 / 47.3, 79.4 / 80.8 / 81.0; in 35x35 planes the same.  Three for all of
// these rates (84 registers, so it is the attribute that holds it there).  The decoder, three / four / five: 16 bits 100 MB 34.9 /
// 34.1 / 35.6, 201 MB 62.8 / 57.2 / 60.1 (70.2 / 65.9 / 67.0); 24 and 32 bits within 1.5 %.  Four.  Below 36 MB all are level.
// ROWS: a field for load_block_rows
template <bool WHOLE, bool INT, bool ONCE, bool ROWS>
__device__ __forceinline__ void encode3_f32(const float* __restrict__ in, const Field3& fd, unsigned maxbits,
                                            uint64_t* __restrict__ stream)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  const unsigned slot = slot_bits(maxbits);

  // A wavefront in one of its memory phases (the loads here, the stores at the end) goes before
  // the ones that are coding when both have an instruction to issue: its requests are what the
  // compute unit's other wavefronts will be computing behind (201.3 MB, nothing cached: 51.7 -> 49.9 us at
  // 8 bits per value, 61.8 -> 59.1 at 16; 402.7 MB 94.0 and 93.9).
  __shared__ uint2 table[WHOLE ? 64 : 1];
  float f[64];
  __builtin_amdgcn_s_setprio(3);
  uint2 piece;
  if (WHOLE) piece = table_piece(lane);
  if (lane < valid) {  // in flight while the region is cleared
    if (ROWS) load_block_rows(in, fd, first, first + lane, f);
    else load_block<ONCE>(in, fd, first, first + lane, f);
  }
  zero_region(lds_raw, lane, maxbits);
  if (WHOLE) table[lane] = piece;
  __syncthreads();
  __builtin_amdgcn_s_setprio(0);

  if (lane < valid) {
    LdsBitsTable mem(lds, table);
    if (INT) {
      int32_t v[64];
#pragma unroll
      for (int i = 0; i < 64; i++) v[i] = __float_as_int(f[i]);
      encode_block_i32<!WHOLE>(v, mem.bit0 + lane * slot, maxbits, mem);
    } else {
      encode_block<!WHOLE>(f, mem.bit0 + lane * slot, maxbits, mem);
    }
  }
  __syncthreads();
  __builtin_amdgcn_s_setprio(3);
  store_region<WHOLE>(lds, lane, first, valid, maxbits, fd, stream);
}

template <bool WHOLE, bool INT = false, bool ONCE = false, int WPE = 5>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void zfp_encode3_f32_kernel(
    const float* __restrict__ in, Field3 fd, unsigned maxbits, uint64_t* __restrict__ stream)
{
  encode3_f32<WHOLE, INT, ONCE, false>(in, fd, maxbits, stream);
}
// Kernels of their own for these fields: one kernel with both kinds of rows decoded full fields 2-6 %
// slower (100 MB 29.2 instead of 27.5 us, 403 MB 89.7 instead of 87.4; measured with a step per run).
template <bool WHOLE, bool INT = false, int WPE = 5>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void zfp_encode3_rows_kernel(
    const float* __restrict__ in, Field3 fd, unsigned maxbits, uint64_t* __restrict__ stream)
{
  encode3_f32<WHOLE, INT, false, true>(in, fd, maxbits, stream);
}

// Five wavefronts per SIMD (at most 96 registers, which the row-wise finish
// and the late block coordinates below reach without spilling): measured
// 2.5 % faster than the four that the unconstrained 105 registers allow; six
// (80 registers) spills and is slower again.
template <bool WHOLE, bool INT, bool ROWS>
__device__ __forceinline__ void decode3_f32(const uint64_t* __restrict__ stream, const Field3& fd, unsigned maxbits,
                                            float* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  const unsigned slot = dec_slot_bits(maxbits);

  // Issue priorities: the load of the stream and the bit planes (a dependent chain through LDS
  // reads) go first, the lifting along z and y inside decode_block_zy fills the slots that are
  // left, and the last part -- lifting along x, cast, the row stores -- sits between the two.
  // Measured on 402.7 MB, with a step per run: 97.5 us with one priority for everything, 94.3 us with the planes
  // above the rest, 87.8 us with the last part below the planes as well (16 bits per value:
  // 137 -> 129 us); the last part below the lifting: 110 us.
  __shared__ uint32_t table[WHOLE ? 64 : 1];
  __builtin_amdgcn_s_setprio(3);
  if (WHOLE) table[lane] = collapse_piece(lane);
  load_region<WHOLE, kFenceDwords>(lds, lane, first, valid, maxbits, slot, fd, stream);
  __syncthreads();

  if (lane < valid) {
    int32_t ib[64];
    float w;
    LdsBitsCollapse mem(lds, table);
    if (INT) {
      w = 0.0f;
      decode_block_i32_zy<WHOLE>(mem, mem.bit0 + lane * slot, maxbits, ib);
    } else {
      decode_block_zy<WHOLE>(mem, mem.bit0 + lane * slot, maxbits, ib, w);
    }
    // block coordinates and addresses are worked out only now, from a lane id
    // that is recomputed here and tied to a decoded value: otherwise they (or
    // the thread index they come from) are held in registers through the whole
    // decode, or spilled
    uint32_t zero = 0;
    asm volatile("" : "+v"(zero) : "v"(ib[0]));
    const uint32_t b = first + __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));  // lane id again
    __builtin_amdgcn_s_setprio(1);
    // (as one variant with the hint decided row by row, the compiler finishes all rows ahead and spills)
    if (ROWS && fd.store_hint) finish_and_store_rows<INT, true>(out, fd, first, b, ib, w);
    else if (ROWS) finish_and_store_rows<INT, false>(out, fd, first, b, ib, w);
    else finish_and_store_block<INT>(out, fd, first, b, ib, w);
  }
}

template <bool WHOLE, bool INT = false, int WPE = 5>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void zfp_decode3_f32_kernel(
    const uint64_t* __restrict__ stream, Field3 fd, unsigned maxbits, float* __restrict__ out)
{
  decode3_f32<WHOLE, INT, false>(stream, fd, maxbits, out);
}
template <bool WHOLE, bool INT = false, int WPE = 5>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void zfp_decode3_rows_kernel(
    const uint64_t* __restrict__ stream, Field3 fd, unsigned maxbits, float* __restrict__ out)
{
  decode3_f32<WHOLE, INT, true>(stream, fd, maxbits, out);
}

// ------------------------------------------------------------- rows that are not made of whole lines
// The decoder for packed fields whose rows are no multiple of 128 bytes (zfp_runs.h).  One lane per block and a row store
// per lane, as above, leaves rows of 28 bytes in parts of a line that are 16 bytes long, and one instruction touches
// as many lines as it has rows: 160 MB in 7x7 planes took three times as long as in 32x32.  Here a wavefront takes whole
// block rows, and one plane of them at a time goes through LDS (4 KB in the place of the decoded stream, so as many
// wavefronts are resident as before): written as whole blocks, 16 bytes a lane without conflicts, read and stored
// in the order of memory.  Where a unit stands and goes is worked out once and holds for all four planes.  What it
// costs: two trips through LDS a plane, and lanes that are left over (64 / mx block rows fit).  Lanes without a block decode the
// last one once more, units past the end store the last one again.  Bound by memory where rows are whole
// 16 bytes (28x28: 160 MB and its stream at 5.1 TB/s, 32x32 5.4), by the 4-byte stores and the vector unit at odd lengths.  8 bits per
// value, one tensor over and over (several in turn), row stores -> this, us:
//   units of 16 bytes  4x4 20 MB 16.1 -> 13.0 (16.6 -> 12.2), 60 MB 28.6 -> 21.8 (29.5 -> 21.9), 160 MB 57 -> 48 (68 -> 49) · 28x28 20 MB 13.3 -> 12.6
//     (14.8 -> 11.8), 60 MB 20.1 -> 18.8 (23.9 -> 19.0), 160 MB 40.4 -> 38.5 (54.3 -> 38.9) · 56x56 60 MB 19.7 -> 18.9 (23.5 -> 19.1)
//   of 8  14x14 20 MB 15.2 -> 13.1 (16.2 -> 12.8), 60 MB 27.2 -> 22.8 (28.1 -> 24.6), 160 MB 51 -> 46 (65 -> 51)
//   of 4  7x7 20 MB 21.4 -> 14.9 (21.7 -> 15.9), 60 MB 44 -> 24.5 (45 -> 26.2), 160 MB 97 -> 51 (106 -> 58) · 35x35 20 MB 14.2 -> 14.4 (15.6 ->
//     13.2), 60 MB 22.8 -> 21.3 (26.5 -> 23.9), 160 MB 44 -> 43 (60 -> 51)
//   4 bits per value, 100 MB  28x28 26.4 -> 25.6 (35.4 -> 25.9); 16 bits 38.4 -> 36.3 (48.9 -> 40.6), 35x35 41.8 -> 41.2 (52.9 -> 49.3)
template <int V>
struct RunUnit;
template <>
struct RunUnit<4> {
  typedef stream_f4 type;
};
template <>
struct RunUnit<2> {
  typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct RunUnit<1> {
  typedef float type;
};

// Computes these sixteen values where this stands
__device__ __forceinline__ void pin16(int32_t (&ib)[64], int i)
{
  asm volatile(""
               : "+v"(ib[i]), "+v"(ib[i + 1]), "+v"(ib[i + 2]), "+v"(ib[i + 3]), "+v"(ib[i + 4]), "+v"(ib[i + 5]), "+v"(ib[i + 6]),
                 "+v"(ib[i + 7]), "+v"(ib[i + 8]), "+v"(ib[i + 9]), "+v"(ib[i + 10]), "+v"(ib[i + 11]), "+v"(ib[i + 12]),
                 "+v"(ib[i + 13]), "+v"(ib[i + 14]), "+v"(ib[i + 15]));
}

// The last lifting pass, the cast and the stores, a plane at a time.  V: elements of a unit.  The pins keep the compiler
// from working ahead on later planes, whose values it would hold twice over: without them it spills at 96 registers.
template <int V, bool HINT>
__device__ __forceinline__ void finish_and_store_runs(float* __restrict__ out, const Runs& p, const RunsWave& wave, char* image,
                                                      int32_t (&ib)[64], float w)
{
  typedef typename RunUnit<V>::type unit_t;
  constexpr int kUnits = 16 / V;
  uint32_t src[kUnits], dst[kUnits];
  uint32_t zero = 0;
  asm volatile("" : "+v"(zero) : "v"(ib[0]));
  const uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
  char* mine = image + 16 * runs_block(p, min(lane, wave.blocks - 1));
  const uint32_t row = 16 * p.mx;
  char* plane = reinterpret_cast<char*>(out) + (size_t)wave.slab * 16u * V * p.plane;
#pragma unroll
  for (int z = 0; z < 4; z++) {
    if (z) pin16(ib, 16 * z);
#pragma unroll
    for (int y = 0; y < 4; y++) {
      float r[4];
      decode_row(ib, y + 4 * z, w, r);
      const stream_f4 v = {r[0], r[1], r[2], r[3]};
      *reinterpret_cast<stream_f4*>(mine + y * row) = v;
    }
    if (z == 0) {
      uint32_t l = lane;
      asm volatile("" : "+v"(l) : "v"(ib[0]));
#pragma unroll
      for (int j = 0; j < kUnits; j++) {
        runs_unit(p, wave, min(l + 64u * j, wave.total - 1), src[j], dst[j]);
        src[j] *= 4 * V;
        dst[j] *= 4 * V;
      }
    } else if (z == p.planes_last && wave.cut != ~0u) {  // from here on without the last slab: its units store the first one again
      if (wave.cut == 0) return;
#pragma unroll
      for (int j = 0; j < kUnits; j++) {
        const bool gone = dst[j] >= wave.cut * (4 * V);
        src[j] = gone ? 0 : src[j];
        dst[j] = gone ? wave.skip * (4 * V) : dst[j];
      }
    }
    __syncthreads();
    constexpr int kBatch = kUnits < 8 ? kUnits : 4;
#pragma unroll
    for (int b = 0; b < kUnits; b += kBatch) {
      if (b) __builtin_amdgcn_sched_barrier(0);
      unit_t v[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; j++) v[j] = *reinterpret_cast<const unit_t*>(image + src[b + j]);
#pragma unroll
      for (int j = 0; j < kBatch; j++) {
        asm volatile("" : "+v"(dst[b + j]));  // a 32-bit offset to the plane's address, not a 64-bit one per unit
        unit_t* to = reinterpret_cast<unit_t*>(plane + (size_t)dst[b + j]);
        if (HINT) __builtin_nontemporal_store(v[j], to);
        else *to = v[j];
      }
    }
    __syncthreads();
    plane += (size_t)4u * V * p.plane;
  }
}

template <int V, bool HINT, int WPE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void zfp_decode3_runs_kernel(
    const uint64_t* __restrict__ stream, Field3 fd, Runs runs, unsigned maxbits, float* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const RunsWave wave = runs_wave(runs, blockIdx.x);
  const unsigned slot = dec_slot_bits(maxbits);
  __shared__ uint32_t table[64];
  __builtin_amdgcn_s_setprio(3);
  table[lane] = collapse_piece(lane);
  load_region<true, kFenceDwords>(lds, lane, wave.first, wave.blocks, maxbits, slot, fd, stream);
  __syncthreads();
  int32_t ib[64];
  float w;
  LdsBitsCollapse mem(lds, table);
  decode_block_zy<true>(mem, mem.bit0 + min(lane, wave.blocks - 1) * slot, maxbits, ib, w);
#pragma unroll
  for (int i = 0; i < 64; i += 16) pin16(ib, i);
  __builtin_amdgcn_s_setprio(1);
  __syncthreads();  // the image takes the stream's place
  finish_and_store_runs<V, HINT>(out, runs, wave, reinterpret_cast<char*>(lds), ib, w);
}

// ------------------------------------------------------------- the pair form: two wavefronts per 64 blocks
// For fields that are too small to fill the chip with one lane per block.  A workgroup is two
// wavefronts; lane l of both works on block first + l, each doing its half of every phase
// (zfp_block.h: pair_encode_half), so that a field keeps twice as many wavefronts in flight,
// each with half the serial work.  Fast path only: whole-word rates with an even number of
// 16-byte pieces per block, full blocks, 16-byte aligned contiguous rows.
//
// Dynamic LDS, in dwords: [region: region_dwords(maxbits)] [maxima: 128] [flag: 4]
// [U0: 1280] [U1: 1280].  U0 and U1 carry all three later exchanges in turn, and the rule
// that makes this safe without barriers of its own is that a half only ever writes into the
// one it was the last to read:
//   z exchange   half h writes U_h (lane * 20 + j, four 16-byte pieces)        barrier  reads U_(1-h)
//   reorder      writes the 13 coefficients it sends into U_(1-h) (slot * 64 + lane)
//                                                                               barrier  reads U_h
//   planes       writes its 32 bits of 16 planes into U_h (k * 64 + lane)      barrier  reads both
constexpr unsigned kPairMaxima = 128, kPairFlag = 4, kPairU = 1280;
__host__ __device__ inline unsigned pair_lds_dwords(unsigned maxbits)  // without the table of expanded bytes
{
  return region_dwords(maxbits) + kPairMaxima + kPairFlag + 2 * kPairU;
}

template <int H>
struct LdsExchange {
  float* maxima;
  uint32_t* flag;
  uint32_t* mine;    // U_H
  uint32_t* theirs;  // U_(1-H)
  unsigned lane;
  __device__ __forceinline__ float other_max(float m)
  {
    maxima[H * 64 + lane] = m;
    __syncthreads();
    return maxima[(1 - H) * 64 + lane];
  }
  __device__ __forceinline__ void swap16(const int32_t (&out)[16], int32_t (&in)[16])
  {
    uint4* dst = reinterpret_cast<uint4*>(mine + lane * 20);
#pragma unroll
    for (int j = 0; j < 4; j++)
      dst[j] = make_uint4((uint32_t)out[4 * j], (uint32_t)out[4 * j + 1], (uint32_t)out[4 * j + 2], (uint32_t)out[4 * j + 3]);
    __syncthreads();
    const uint4* src = reinterpret_cast<const uint4*>(theirs + lane * 20);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint4 v = src[j];
      in[4 * j] = (int32_t)v.x;
      in[4 * j + 1] = (int32_t)v.y;
      in[4 * j + 2] = (int32_t)v.z;
      in[4 * j + 3] = (int32_t)v.w;
    }
  }
  __device__ __forceinline__ void seq_put(int slot, uint32_t v) { theirs[slot * 64 + lane] = v; }
  __device__ __forceinline__ void seq_sync() { __syncthreads(); }
  __device__ __forceinline__ uint32_t seq_get(int slot) { return mine[slot * 64 + lane]; }
  __device__ __forceinline__ void plane_put(int k, uint32_t v) { mine[k * 64 + lane] = v; }
  __device__ __forceinline__ void plane_sync() { __syncthreads(); }
  __device__ __forceinline__ uint64_t plane_get(int k)
  {
    const uint32_t* u0 = H == 0 ? mine : theirs;
    const uint32_t* u1 = H == 0 ? theirs : mine;
    return ((uint64_t)u1[k * 64 + lane] << 32) | u0[k * 64 + lane];
  }
  // Half 0 answers for both, so that the two can never disagree about the barriers ahead.
  __device__ __forceinline__ bool more(bool any)
  {
    if (H == 0 && lane == 0) *flag = any ? 1u : 0u;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*flag) != 0;
  }
  __device__ __forceinline__ void done() { __syncthreads(); }
};

template <int H>
__device__ __forceinline__ void pair_encode_body(const float* __restrict__ in, const Field3& fd, unsigned maxbits,
                                                 uint32_t* lds, const uint2* table, unsigned lane, uint32_t first)
{
  const bool live = first + lane < fd.nblocks;
  const uint32_t b = live ? first + lane : fd.nblocks - 1;
  float p[16], q[16];
  {
    uint32_t x0, y0, z0;
    block_origin(fd, b, x0, y0, z0);
    const WaveBase w = wave_base(fd, first);
    const char* base = reinterpret_cast<const char*>(in + w.origin);
    const uint32_t me = lane_bytes(fd, w, x0, y0, z0);
    const uint32_t sy4 = (uint32_t)fd.sy * 4u, sz4 = (uint32_t)fd.sz * 4u;
    constexpr int ZP = H == 0 ? 0 : 2, ZQ = H == 0 ? 3 : 1;
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const stream_f4 vp = *reinterpret_cast<const stream_f4*>(base + (size_t)(me + (y * sy4 + ZP * sz4)));
      const stream_f4 vq = *reinterpret_cast<const stream_f4*>(base + (size_t)(me + (y * sy4 + ZQ * sz4)));
      p[4 * y] = vp.x; p[4 * y + 1] = vp.y; p[4 * y + 2] = vp.z; p[4 * y + 3] = vp.w;
      q[4 * y] = vq.x; q[4 * y + 1] = vq.y; q[4 * y + 2] = vq.z; q[4 * y + 3] = vq.w;
    }
  }
  const unsigned region = region_dwords(maxbits);
  LdsExchange<H> ex;
  ex.maxima = reinterpret_cast<float*>(lds + region);
  ex.flag = lds + region + kPairMaxima;
  ex.mine = lds + region + kPairMaxima + kPairFlag + H * kPairU;
  ex.theirs = lds + region + kPairMaxima + kPairFlag + (1 - H) * kPairU;
  ex.lane = lane;
  LdsBitsTable mem(lds, table);
  pair_encode_half<H>(p, q, live, mem.bit0 + lane * slot_bits(maxbits), maxbits, mem, ex);
}

// Seven wavefronts per SIMD (72 registers; 75 without the limit) leave the LDS to bound how many are resident.
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(7, 8))) void zfp_encode3_f32_pair_kernel(
    const float* __restrict__ in, Field3 fd, unsigned maxbits, uint64_t* __restrict__ stream)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned tid = threadIdx.x, lane = tid & 63u;
  const uint32_t first = blockIdx.x * 64u;
  __shared__ uint2 table[64];
  if (tid < 64) table[tid] = table_piece(tid);
  {  // the region starts out zero; the first exchange's barrier orders this before any coder's OR
    const unsigned n16 = region_dwords(maxbits) / 4;
    for (unsigned i = tid; i < n16; i += 128) lds_raw[i] = make_uint4(0, 0, 0, 0);
  }
  if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) pair_encode_body<0>(in, fd, maxbits, lds, table, lane, first);
  else pair_encode_body<1>(in, fd, maxbits, lds, table, lane, first);
  // Both halves are past the barrier of more() or done(): every block is coded.
  store_pieces<128, kSlackDwords>(lds, tid, min(64u, fd.nblocks - first), maxbits, fd.by_piece,
                                  stream + (size_t)first * (maxbits >> 6));
}

// The pair form of the decoder (zfp_block.h: pair_decode_half).  Dynamic LDS, in dwords:
// [region: dec_region_dwords(maxbits)] [scales: 64] [flag: 4] [U0: 1024] [U1: 1024].
//   planes     half 0 writes the low words of 16 plane words into U0 and the high words into U1
//              (k * 64 + lane)                                                barrier  half h reads U_h
//              (the same again for the low 16 planes, between two more barriers, when they follow)
//   reorder    half h writes the 13 coefficients it sends into U_h (slot * 64 + lane)
//                                                                              barrier  reads U_(1-h)
//   z exchange half h writes into U_(1-h) (j * 64 + lane)                     barrier  reads U_h
// again a half only ever writes into the one it was the last to read.
constexpr unsigned kPairScales = 64, kPairDecU = 1024;
__host__ __device__ inline unsigned pair_dec_lds_dwords(unsigned maxbits)
{
  return dec_region_dwords(maxbits) + kPairScales + kPairFlag + 2 * kPairDecU;
}

template <int H>
struct LdsDecExchange {
  float* scales;
  uint32_t* flag;
  uint32_t* u0;
  uint32_t* u1;
  unsigned lane;
  __device__ __forceinline__ uint32_t* mine() const { return H == 0 ? u0 : u1; }
  __device__ __forceinline__ uint32_t* theirs() const { return H == 0 ? u1 : u0; }
  __device__ __forceinline__ void plane_put(int k, uint64_t x)
  {
    u0[k * 64 + lane] = (uint32_t)x;
    u1[k * 64 + lane] = (uint32_t)(x >> 32);
  }
  __device__ __forceinline__ void scale_put(float w) { scales[lane] = w; }
  __device__ __forceinline__ bool planes_sync(bool any)
  {
    if (H == 0 && lane == 0) *flag = any ? 1u : 0u;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*flag) != 0;
  }
  __device__ __forceinline__ uint32_t plane_get(int k) { return mine()[k * 64 + lane]; }
  __device__ __forceinline__ float scale_get() { return scales[lane]; }
  __device__ __forceinline__ void consumed() { __syncthreads(); }
  __device__ __forceinline__ void low_sync() { __syncthreads(); }
  __device__ __forceinline__ void seq_put(int slot, uint32_t v) { mine()[slot * 64 + lane] = v; }
  __device__ __forceinline__ void seq_sync() { __syncthreads(); }
  __device__ __forceinline__ uint32_t seq_get(int slot) { return theirs()[slot * 64 + lane]; }
  __device__ __forceinline__ void swap16(const int32_t (&out)[16], int32_t (&in)[16])
  {
#pragma unroll
    for (int j = 0; j < 16; j++) theirs()[j * 64 + lane] = (uint32_t)out[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16; j++) in[j] = (int32_t)mine()[j * 64 + lane];
  }
};

template <int H, bool HINT>
__device__ __forceinline__ void pair_decode_body(const Field3& fd, unsigned maxbits, uint32_t* lds, const uint32_t* table,
                                                 unsigned lane, uint32_t first, float* __restrict__ out)
{
  const unsigned region = dec_region_dwords(maxbits);
  LdsDecExchange<H> ex;
  ex.scales = reinterpret_cast<float*>(lds + region);
  ex.flag = lds + region + kPairScales;
  ex.u0 = lds + region + kPairScales + kPairFlag;
  ex.u1 = ex.u0 + kPairDecU;
  ex.lane = lane;
  LdsBitsCollapse mem(lds, table);
  float p[16], q[16];
  pair_decode_half<H>(mem, mem.bit0 + lane * dec_slot_bits(maxbits), maxbits, ex, p, q);
  if (first + lane < fd.nblocks) {
    uint32_t x0, y0, z0;
    block_origin(fd, first + lane, x0, y0, z0);
    const WaveBase w = wave_base(fd, first);
    char* base = reinterpret_cast<char*>(out + w.origin);
    const uint32_t me = lane_bytes(fd, w, x0, y0, z0);
    const uint32_t sy4 = (uint32_t)fd.sy * 4u, sz4 = (uint32_t)fd.sz * 4u;
    constexpr int ZP = H == 0 ? 0 : 2, ZQ = H == 0 ? 3 : 1;
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const stream_f4 vp = {p[4 * y], p[4 * y + 1], p[4 * y + 2], p[4 * y + 3]};
      const stream_f4 vq = {q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3]};
      stream_f4* dp = reinterpret_cast<stream_f4*>(base + (size_t)(me + (y * sy4 + ZP * sz4)));
      stream_f4* dq = reinterpret_cast<stream_f4*>(base + (size_t)(me + (y * sy4 + ZQ * sz4)));
      if (HINT) {
        __builtin_nontemporal_store(vp, dp);
        __builtin_nontemporal_store(vq, dq);
      } else {
        *dp = vp;
        *dq = vq;
      }
    }
  }
}

template <bool HINT>
__device__ __forceinline__ void pair_decode(const uint64_t* __restrict__ stream, const Field3& fd, unsigned maxbits,
                                            float* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned tid = threadIdx.x, lane = tid & 63u;
  const uint32_t first = blockIdx.x * 64u;
  __shared__ uint32_t table[64];
  if (tid < 64) table[tid] = collapse_piece(tid);
  {  // the fence goes behind every block; the slots past the end of the field read as empty blocks
    const unsigned W = maxbits >> 6, slot = dec_slot_bits(maxbits);
    const uint32_t valid = min(64u, fd.nblocks - first);
    load_pieces<128, kFenceDwords>(lds, tid, valid, maxbits, fd.by_piece, stream + (size_t)first * W);
    uint64_t* own = reinterpret_cast<uint64_t*>(lds + lane * (slot / 32));
    if (tid < 64) own[W] = kFence;
    else if (lane >= valid) own[0] = 0;
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) pair_decode_body<0, HINT>(fd, maxbits, lds, table, lane, first, out);
  else pair_decode_body<1, HINT>(fd, maxbits, lds, table, lane, first, out);
}

__global__ __launch_bounds__(128) void zfp_decode3_f32_pair_kernel(const uint64_t* __restrict__ stream, Field3 fd,
                                                                   unsigned maxbits, float* __restrict__ out)
{
  pair_decode<true>(stream, fd, maxbits, out);
}
// without the hint (Field3::store_hint): 11 MB in 8x8 planes at 16 bits per value, several in turn, 13.7 us, 15.6 with it,
// in 4x4 planes 14.6 and 31
__global__ __launch_bounds__(128) void zfp_decode3_f32_pair_plain_kernel(const uint64_t* __restrict__ stream, Field3 fd,
                                                                         unsigned maxbits, float* __restrict__ out)
{
  pair_decode<false>(stream, fd, maxbits, out);
}

// ------------------------------------------------------------- the quad form: four lanes per block
// For the smallest fields.  A wavefront codes 16 blocks: lane 4 * block + q holds z-slice q, so
// a lane's share of every phase but the coder is a quarter of a block's, and a field keeps four
// times as many wavefronts in flight as with one lane per block.  Through LDS the lanes of a
// block turn its values (along z the lines y = q), put the coefficients in coding order and
// hand out the bit planes.
//   encoder  lane q codes every fourth plane, q first: where a plane starts is a prefix over the
//            planes before it (plane_bits), a quad of lanes at a time with data-parallel-primitive
//            moves, so four planes are coded at once and nobody steps through a plane twice
//   decoder  where a plane starts is only known when the one before is decoded: all four lanes
//            decode every plane, each keeps its quarter, and the exchange that the encoder needs falls away
// A lane's rows are loaded by the padding rule's addresses, so the form takes every field of
// floats at a whole-word rate.  What bounds it is the chain left in a wavefront: the encoder's
// four rounds of planes, the decoder's 13 to 16 planes one after the other.  4.2 MB at 8 bits per value,
// quad / one lane per block: encode 5.2 / 7.8 us (pair form 6.4), decode 8.1 / 9.5; the rule is at quad_pays.
constexpr unsigned kQuadBlocks = 16;   // blocks of a wavefront
constexpr unsigned kQuadStride = 68;   // dwords of a block's exchange area: 64 and four to spread the banks
__host__ __device__ inline unsigned quad_region_dwords(unsigned slot) { return (kQuadBlocks * slot / 32 + 4u + 3u) & ~3u; }
__host__ __device__ inline unsigned quad_lds_dwords(unsigned slot) { return quad_region_dwords(slot) + kQuadBlocks * kQuadStride; }

__constant__ const QuadOrder kQuadOrder = make_quad_order();

template <int CTRL>
__device__ __forceinline__ uint32_t quad_move(uint32_t v)  // value of the quad's lane that CTRL names for mine
{
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kQuadDown1 = 0x90, kQuadDown2 = 0x44, kQuadLast = 0xff;
template <int CTRL>
__device__ __forceinline__ uint64_t quad_move64(uint64_t v)
{
  return ((uint64_t)quad_move<CTRL>((uint32_t)(v >> 32)) << 32) | quad_move<CTRL>((uint32_t)v);
}

// index inside a block of n elements along an axis that the padding rule (pad4) puts at i
__device__ __forceinline__ uint32_t padded_index(uint32_t n, uint32_t i)
{
  return i < n ? i : (n == 2 && i == 2 ? 1u : 0u);
}

// the four rows of z-slice q of block b
__device__ __forceinline__ void quad_load(const float* __restrict__ in, const Field3& fd, uint32_t b, uint32_t q,
                                          float (&f)[16])
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  const float* p = in + ((long long)x0 * fd.sx + (long long)y0 * fd.sy + (long long)z0 * fd.sz);
  if (fd.full) {
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const row_f4 v = *reinterpret_cast<const row_f4*>(p + ((long long)q * fd.sz + y * fd.sy));
      f[4 * y] = v.x; f[4 * y + 1] = v.y; f[4 * y + 2] = v.z; f[4 * y + 3] = v.w;
    }
    return;
  }
  const uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  const bool leaves = bx < 4 && y0 + by == fd.ny && z0 + bz == fd.nz;  // as in load_block
  p += (long long)padded_index(bz, q) * fd.sz;
  if (fd.rows4 && !leaves) {
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const row_f4 v = *reinterpret_cast<const row_f4*>(p + (long long)padded_index(by, y) * fd.sy);
      f[4 * y] = v.x;
      f[4 * y + 1] = bx >= 2 ? v.y : v.x;
      f[4 * y + 2] = bx >= 3 ? v.z : f[4 * y + 1];
      f[4 * y + 3] = bx >= 4 ? v.w : v.x;
    }
  } else {
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
      for (int x = 0; x < 4; x++)
        f[4 * y + x] = p[(long long)padded_index(bx, x) * fd.sx + (long long)padded_index(by, y) * fd.sy];
  }
}

// One round of the coder: four planes, lane q's is x; acc and base (the OR of the planes so far
// and the bit position behind them) are the same in the four lanes.
__device__ __forceinline__ void quad_round(TableEncoder<LdsBitsTable>& enc, uint64_t x, uint32_t q, uint64_t& acc,
                                           unsigned& base)
{
  const uint32_t from1 = q >= 1 ? ~0u : 0u, from2 = q >= 2 ? ~0u : 0u;
  const uint64_t from1w = ((uint64_t)from1 << 32) | from1, from2w = ((uint64_t)from2 << 32) | from2;
  uint64_t all = x | (quad_move64<kQuadDown1>(x) & from1w);
  all |= quad_move64<kQuadDown2>(all) & from2w;  // planes of the lanes up to mine
  const uint64_t before = acc | (quad_move64<kQuadDown1>(all) & from1w);
  const unsigned n = known_after(before);
  const unsigned bits = plane_bits(x, n, known_after(acc | all));
  unsigned sum = bits + (quad_move<kQuadDown1>(bits) & from1);
  sum += quad_move<kQuadDown2>(sum) & from2;
  enc.pos = base + sum - bits;
  enc.n = n;
  acc |= quad_move64<kQuadLast>(all);
  base += quad_move<kQuadLast>(sum);
  if (CSWAP_ANY(x != 0 || n != 0)) enc.plane(x);  // an empty plane of a block without known coefficients is one zero bit
}

// 16 planes: t as quad_planes leaves it, exchange: the block's exchange area
__device__ __forceinline__ void quad_code16(const uint32_t (&t)[8], uint32_t* exchange, uint32_t q,
                                            TableEncoder<LdsBitsTable>& enc, uint64_t& acc, unsigned& base)
{
#pragma unroll
  for (int j = 0; j < 8; j++) exchange[4 * j + q] = t[j];
  __syncthreads();
  const uint4 u = *reinterpret_cast<const uint4*>(exchange + 4 * (7 - q));
  const uint4 v = *reinterpret_cast<const uint4*>(exchange + 4 * (3 - q));
  constexpr uint32_t kHigh = 0x07060302u, kLow = 0x05040100u;  // the high / low halves of two words
  const uint64_t r0 = ((uint64_t)byte_perm(u.w, u.z, kHigh) << 32) | byte_perm(u.y, u.x, kHigh);
  const uint64_t r1 = ((uint64_t)byte_perm(v.w, v.z, kHigh) << 32) | byte_perm(v.y, v.x, kHigh);
  const uint64_t r2 = ((uint64_t)byte_perm(u.w, u.z, kLow) << 32) | byte_perm(u.y, u.x, kLow);
  const uint64_t r3 = ((uint64_t)byte_perm(v.w, v.z, kLow) << 32) | byte_perm(v.y, v.x, kLow);
  quad_round(enc, r0, q, acc, base);
  if (CSWAP_ANY(base < enc.limit)) quad_round(enc, r1, q, acc, base);
  if (CSWAP_ANY(base < enc.limit)) quad_round(enc, r2, q, acc, base);
  if (CSWAP_ANY(base < enc.limit)) quad_round(enc, r3, q, acc, base);
}

__global__ __launch_bounds__(64) void zfp_encode3_f32_quad_kernel(const float* __restrict__ in, Field3 fd,
                                                                  unsigned maxbits, uint64_t* __restrict__ stream)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x, bl = lane >> 2, q = lane & 3u;
  const uint32_t b = blockIdx.x * kQuadBlocks + bl;
  const bool live = b < fd.nblocks;
  const unsigned slot = slot_bits(maxbits);
  uint32_t* ex = lds + quad_region_dwords(slot) + bl * kQuadStride;

  __shared__ uint2 table[64];
  const uint2 piece = table_piece(lane);
  float f[16];
  quad_load(in, fd, live ? b : fd.nblocks - 1, q, f);
  table[lane] = piece;
  uint32_t to_seq[4];
#pragma unroll
  for (int i = 0; i < 4; i++) to_seq[i] = kQuadOrder.to_seq[q][i];
  {
    const unsigned n16 = quad_region_dwords(slot) / 4;
    for (unsigned i = lane; i < n16; i += 64) lds_raw[i] = make_uint4(0, 0, 0, 0);
  }
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) m = fmaxf(m, fabsf(f[i]));
  m = fmaxf(m, f32_from_bits(quad_move<kQuadXor1>(f32_bits(m))));
  m = fmaxf(m, f32_from_bits(quad_move<kQuadXor2>(f32_bits(m))));
  const uint32_t mb = f32_bits(m);
  const uint32_t e = (live && mb) ? (mb >> 23) + 1 : 0;  // as block_header_e
  const float s = e ? pow2f(30 - ((int)e - 127)) : 0.0f;

  int32_t c[16];  // x + 4y of slice q, then x + 4z of the plane y = q
#pragma unroll
  for (int i = 0; i < 16; i++) c[i] = (int32_t)(s * f[i]);
#pragma unroll
  for (int y = 0; y < 4; y++) fwd_lift4(c[4 * y], c[4 * y + 1], c[4 * y + 2], c[4 * y + 3]);
#pragma unroll
  for (int x = 0; x < 4; x++) fwd_lift4(c[x], c[x + 4], c[x + 8], c[x + 12]);
#pragma unroll
  for (int y = 0; y < 4; y++)
    *reinterpret_cast<int4*>(ex + 16 * q + 4 * y) = make_int4(c[4 * y], c[4 * y + 1], c[4 * y + 2], c[4 * y + 3]);
  __syncthreads();
#pragma unroll
  for (int z = 0; z < 4; z++) {
    const int4 v = *reinterpret_cast<const int4*>(ex + 16 * z + 4 * q);
    c[4 * z] = v.x; c[4 * z + 1] = v.y; c[4 * z + 2] = v.z; c[4 * z + 3] = v.w;
  }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < 4; x++) fwd_lift4(c[x], c[x + 4], c[x + 8], c[x + 12]);
#pragma unroll
  for (int i = 0; i < 16; i++)  // negabinary: the add here, the xor inside the transpose
    *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(ex) + ((to_seq[i / 4] >> (8 * (i % 4))) & 0xffu)) =
        (uint32_t)c[i] + kNegabinary;
  __syncthreads();
  uint32_t a[16];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint4 v = *reinterpret_cast<const uint4*>(ex + 16 * q + 4 * i);
    a[4 * i] = v.x; a[4 * i + 1] = v.y; a[4 * i + 2] = v.z; a[4 * i + 3] = v.w;
  }
  __syncthreads();

  LdsBitsTable mem(lds, table);
  TableEncoder<LdsBitsTable> enc(mem, mem.bit0 + bl * slot, maxbits);
  unsigned base = e ? enc.pos + 9 : enc.limit;  // an all-zero block or one past the end: nothing is written
  if (e && q == 0) enc.put(2 * e + 1, 9);
  uint64_t acc = 0;
  uint32_t t[8];
  quad_planes<true>(a, t);
  quad_code16(t, ex, q, enc, acc, base);
  if (CSWAP_ANY(base < enc.limit)) {
    quad_planes<false>(a, t);
    __syncthreads();
    quad_code16(t, ex, q, enc, acc, base);
  }
  __syncthreads();

  if (live) {  // the four lanes of a block move its words
    const unsigned W = maxbits >> 6;
    const uint64_t* src = reinterpret_cast<const uint64_t*>(lds + bl * (slot / 32));
    uint64_t* dst = stream + (size_t)b * W;
    if ((W & 1u) == 0 && fd.stream16) {
      for (unsigned j = 2 * q; j < W; j += 8)
        *reinterpret_cast<ulonglong2*>(dst + j) = *reinterpret_cast<const ulonglong2*>(src + j);
    } else {
      for (unsigned j = q; j < W; j += 4) dst[j] = src[j];
    }
  }
}

__global__ __launch_bounds__(64) void zfp_decode3_f32_quad_kernel(const uint64_t* __restrict__ stream, Field3 fd,
                                                                  unsigned maxbits, float* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x, bl = lane >> 2, q = lane & 3u;
  const uint32_t b = blockIdx.x * kQuadBlocks + bl;
  const bool live = b < fd.nblocks;
  const unsigned slot = dec_slot_bits(maxbits);
  uint32_t* ex = lds + quad_region_dwords(slot) + bl * kQuadStride;
  __shared__ uint32_t table[64];
  table[lane] = collapse_piece(lane);
  {  // the four lanes of a block bring its words; blocks past the end read as empty
    const unsigned W = maxbits >> 6;
    uint64_t* dst = reinterpret_cast<uint64_t*>(lds + bl * (slot / 32));
    const uint64_t* src = stream + (size_t)b * W;
    if (!live) {
      for (unsigned j = q; j < W; j += 4) dst[j] = 0;
    } else if ((W & 1u) == 0 && fd.stream16) {
      for (unsigned j = 2 * q; j < W; j += 8) {
        const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(src + j);
        dst[j] = v.x;
        dst[j + 1] = v.y;
      }
    } else {
      for (unsigned j = q; j < W; j += 4) dst[j] = src[j];
    }
    if (q == 0) dst[W] = kFence;
  }
  uint32_t to_xyz[4];
#pragma unroll
  for (int i = 0; i < 4; i++) to_xyz[i] = kQuadOrder.to_xyz[q][i];
  __syncthreads();

  LdsBitsCollapse mem(lds, table);
  TableDecoder<LdsBitsCollapse> dec(mem, mem.bit0 + bl * slot, maxbits);
  const uint32_t h = (uint32_t)dec.window(dec.pos);
  const bool coded = (h & 1) != 0;
  dec.pos = coded ? dec.pos + 9 : dec.limit;
  const uint32_t mine = (q & 1u) ? 0x07060302u : 0x05040100u;  // my half of the word that has my quarter of a plane
  uint32_t t[8], l[8];
#pragma unroll
  for (int k = 15; k >= 0; k--) {
    uint64_t x = 0;
    if (CSWAP_ANY(dec.active())) x = k >= 12 ? dec.leading_plane() : dec.plane();
    const uint32_t word = (q & 2u) ? (uint32_t)(x >> 32) : (uint32_t)x;
    if (k >= 8) t[k - 8] = word;
    else t[k] = byte_perm(t[k], word, mine);
  }
  quad_untranspose(t);
  uint32_t bias = kNegabinary;
  if (CSWAP_ANY(dec.active())) {
#pragma unroll
    for (int k = 15; k >= 0; k--) {
      const uint64_t x = dec.low_plane();
      const uint32_t word = (q & 2u) ? (uint32_t)(x >> 32) : (uint32_t)x;
      if (k >= 8) l[k - 8] = word;
      else l[k] = byte_perm(l[k], word, mine);
    }
    quad_untranspose(l);
  } else {
#pragma unroll
    for (int k = 0; k < 8; k++) l[k] = 0;
    bias = kNegabinary & 0xffff0000u;
  }
  uint32_t a[16];
  quad_coefficients(t, l, a);
#pragma unroll
  for (int i = 0; i < 16; i++)
    *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(ex) + ((to_xyz[i / 4] >> (8 * (i % 4))) & 0xffu)) = a[i];
  __syncthreads();
  int32_t c[16];  // x + 4z of the plane y = q, then x + 4y of slice q
#pragma unroll
  for (int z = 0; z < 4; z++) {
    const int4 v = *reinterpret_cast<const int4*>(ex + 16 * z + 4 * q);
    c[4 * z] = v.x; c[4 * z + 1] = v.y; c[4 * z + 2] = v.z; c[4 * z + 3] = v.w;
  }
#pragma unroll
  for (int x = 0; x < 4; x++) inv_lift4_biased(c[x], c[x + 4], c[x + 8], c[x + 12], bias);
#pragma unroll
  for (int z = 0; z < 4; z++)
    *reinterpret_cast<int4*>(ex + 16 * z + 4 * q) = make_int4(c[4 * z], c[4 * z + 1], c[4 * z + 2], c[4 * z + 3]);
  __syncthreads();
#pragma unroll
  for (int y = 0; y < 4; y++) {
    const int4 v = *reinterpret_cast<const int4*>(ex + 16 * q + 4 * y);
    c[4 * y] = v.x; c[4 * y + 1] = v.y; c[4 * y + 2] = v.z; c[4 * y + 3] = v.w;
  }
#pragma unroll
  for (int x = 0; x < 4; x++) inv_lift4(c[x], c[x + 4], c[x + 8], c[x + 12]);
  const float w = coded ? decode_scale((h >> 1) & 0xffu) : 0.0f;
  float r[16];
#pragma unroll
  for (int y = 0; y < 4; y++) {
    inv_lift4(c[4 * y], c[4 * y + 1], c[4 * y + 2], c[4 * y + 3]);
#pragma unroll
    for (int x = 0; x < 4; x++) r[4 * y + x] = w * (float)c[4 * y + x];
  }

  uint32_t x0, y0, z0;
  block_origin(fd, live ? b : 0u, x0, y0, z0);
  const uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  if (!live || q >= bz) return;
  float* p = out + ((long long)x0 * fd.sx + (long long)y0 * fd.sy + (long long)(z0 + q) * fd.sz);
  if (fd.full && fd.rows16) {  // few enough lines for the hint whatever the rows are (4.2 MB in 4x4 planes 7.5 us, 7.8 without)
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const stream_f4 v = {r[4 * y], r[4 * y + 1], r[4 * y + 2], r[4 * y + 3]};
      __builtin_nontemporal_store(v, reinterpret_cast<stream_f4*>(p + y * fd.sy));
    }
  } else if (fd.rows4 && bx == 4) {
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const row_f4 v = {r[4 * y], r[4 * y + 1], r[4 * y + 2], r[4 * y + 3]};
      if ((uint32_t)y < by) *reinterpret_cast<row_f4*>(p + y * fd.sy) = v;
    }
  } else {
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
      for (int x = 0; x < 4; x++)
        if ((uint32_t)x < bx && (uint32_t)y < by) p[x * fd.sx + y * fd.sy] = r[4 * y + x];
  }
}

// ------------------------------------------------------------- 64-bit elements
// Fields of doubles or int64 (zfp_type_double, zfp_type_int64): the same
// decomposition, values moved as 64-bit patterns.  Fast path: full block whose
// x-rows are contiguous and 16-byte aligned (two 16-byte accesses per row).
__device__ __forceinline__ void load_block_w64(const uint64_t* __restrict__ in, const Field3& fd, uint32_t b,
                                               uint64_t (&q)[64])
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  const uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  const uint64_t* p = in + (long long)x0 * fd.sx + (long long)y0 * fd.sy + (long long)z0 * fd.sz;
  if (fd.rows16 && bx == 4 && by == 4 && bz == 4) {
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++) {
        const ulonglong2* r = reinterpret_cast<const ulonglong2*>(p + y * fd.sy + z * fd.sz);
        const ulonglong2 a = r[0], c = r[1];
        q[16 * z + 4 * y + 0] = a.x;
        q[16 * z + 4 * y + 1] = a.y;
        q[16 * z + 4 * y + 2] = c.x;
        q[16 * z + 4 * y + 3] = c.y;
      }
  } else {
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int x = 0; x < 4; x++) {
          bool ok = (uint32_t)x < bx && (uint32_t)y < by && (uint32_t)z < bz;
          q[16 * z + 4 * y + x] = ok ? p[x * fd.sx + y * fd.sy + z * fd.sz] : 0ull;
        }
    if (bx < 4 || by < 4 || bz < 4) pad_block3(q, bx, by, bz);
  }
}

template <bool ONCE>
__device__ __forceinline__ void store_block_w64(uint64_t* __restrict__ out, const Field3& fd, uint32_t b,
                                                const uint64_t (&q)[64])
{
  uint32_t x0, y0, z0;
  block_origin(fd, b, x0, y0, z0);
  const uint32_t bx = min(4u, fd.nx - x0), by = min(4u, fd.ny - y0), bz = min(4u, fd.nz - z0);
  uint64_t* p = out + (long long)x0 * fd.sx + (long long)y0 * fd.sy + (long long)z0 * fd.sz;
  if (fd.rows16 && bx == 4 && by == 4 && bz == 4) {
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++) {
        stream_u2* r = reinterpret_cast<stream_u2*>(p + y * fd.sy + z * fd.sz);
        const stream_u2 a = {q[16 * z + 4 * y + 0], q[16 * z + 4 * y + 1]};
        const stream_u2 c = {q[16 * z + 4 * y + 2], q[16 * z + 4 * y + 3]};
        if (ONCE) {
          __builtin_nontemporal_store(a, r);
          __builtin_nontemporal_store(c, r + 1);
        } else {
          r[0] = a;
          r[1] = c;
        }
      }
  } else {
#pragma unroll
    for (int z = 0; z < 4; z++)
#pragma unroll
      for (int y = 0; y < 4; y++)
#pragma unroll
        for (int x = 0; x < 4; x++)
          if ((uint32_t)x < bx && (uint32_t)y < by && (uint32_t)z < bz)
            p[x * fd.sx + y * fd.sy + z * fd.sz] = q[16 * z + 4 * y + x];
  }
}

template <bool WHOLE, bool INT>
__global__ __launch_bounds__(64) void zfp_encode3_w64_kernel(const uint64_t* __restrict__ in, Field3 fd,
                                                             unsigned maxbits, uint64_t* __restrict__ stream)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  __shared__ uint2 table[WHOLE ? 64 : 1];
  uint2 piece;
  if (WHOLE) piece = table_piece(lane);
  uint64_t q[64];
  if (lane < valid) load_block_w64(in, fd, first + lane, q);  // in flight while the region is cleared
  zero_region(lds_raw, lane, maxbits);
  if (WHOLE) table[lane] = piece;
  __syncthreads();
  if (lane < valid) {
    LdsBitsTable mem(lds, table);
    encode_block_w64<!WHOLE, INT>(q, mem.bit0 + lane * slot_bits(maxbits), maxbits, mem);
  }
  __syncthreads();
  store_region<WHOLE>(lds, lane, first, valid, maxbits, fd, stream);
}

// ONCE: rows stored with the nontemporal hint (Field3::once64)
template <bool WHOLE, bool INT, bool ONCE = false>
__global__ __launch_bounds__(64) void zfp_decode3_w64_kernel(const uint64_t* __restrict__ stream, Field3 fd,
                                                             unsigned maxbits, uint64_t* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  __builtin_amdgcn_s_setprio(3);  // the 32-bit decoder's priorities (here, at two wavefronts per SIMD, worth 2.6 %)
  __shared__ uint32_t table[WHOLE ? 64 : 1];
  if (WHOLE) table[lane] = collapse_piece(lane);
  load_region<WHOLE, kSlackDwords>(lds, lane, first, valid, maxbits, slot_bits(maxbits), fd, stream);
  __syncthreads();
  if (lane < valid) {
    uint64_t q[64];
    LdsBitsCollapse mem(lds, table);
    decode_block_w64<INT, WHOLE>(mem, mem.bit0 + lane * slot_bits(maxbits), maxbits, q);
    __builtin_amdgcn_s_setprio(1);
    store_block_w64<ONCE>(out, fd, first + lane, q);
  }
}

// ------------------------------------------------------------- 2-D / 1-D fields
// Same decomposition (one lane per block of 16 or 4 values, 64 blocks per
// wave, LDS bit region); element accesses are predicated scalars.
struct FieldLow {
  uint32_t nx, ny;   // ny = 1 for a 1-D field
  uint32_t mx;       // blocks along x
  uint32_t nblocks;
  long long sx, sy;
};

template <int DIMS>
__device__ __forceinline__ void load_block_low(const float* __restrict__ in, const FieldLow& fd, uint32_t b,
                                               float (&f)[16])
{
  const uint32_t q = b / fd.mx;
  const uint32_t x0 = (b - q * fd.mx) * 4, y0 = DIMS == 2 ? q * 4 : 0;
  const float* p = in + (long long)x0 * fd.sx + (long long)y0 * fd.sy;
  const uint32_t bx = min(4u, fd.nx - x0), by = DIMS == 2 ? min(4u, fd.ny - y0) : 1u;
#pragma unroll
  for (int y = 0; y < 4; y++)
#pragma unroll
    for (int x = 0; x < 4; x++) {
      bool ok = (uint32_t)x < bx && (uint32_t)y < by;
      f[4 * y + x] = ok ? p[x * fd.sx + y * fd.sy] : 0.0f;
    }
#pragma unroll
  for (int y = 0; y < (DIMS == 2 ? 4 : 1); y++) pad4(f[4 * y], f[4 * y + 1], f[4 * y + 2], f[4 * y + 3], bx);
  if (DIMS == 2) {
#pragma unroll
    for (int x = 0; x < 4; x++) pad4(f[x], f[x + 4], f[x + 8], f[x + 12], by);
  }
}

template <int DIMS>
__device__ __forceinline__ void store_block_low(float* __restrict__ out, const FieldLow& fd, uint32_t b,
                                                const float (&f)[16])
{
  const uint32_t q = b / fd.mx;
  const uint32_t x0 = (b - q * fd.mx) * 4, y0 = DIMS == 2 ? q * 4 : 0;
  float* p = out + (long long)x0 * fd.sx + (long long)y0 * fd.sy;
  const uint32_t bx = min(4u, fd.nx - x0), by = DIMS == 2 ? min(4u, fd.ny - y0) : 1u;
#pragma unroll
  for (int y = 0; y < 4; y++)
#pragma unroll
    for (int x = 0; x < 4; x++)
      if ((uint32_t)x < bx && (uint32_t)y < by) p[x * fd.sx + y * fd.sy] = f[4 * y + x];
}

// The wave's 64 blocks are packed back to back in LDS exactly as in the stream
// (64 * maxbits bits = maxbits whole words) and moved cooperatively.
template <int DIMS, bool INT = false>
__global__ __launch_bounds__(64) void zfp_encode_low_f32_kernel(const float* __restrict__ in, FieldLow fd,
                                                                unsigned maxbits, uint64_t* __restrict__ stream)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  const unsigned n16 = (2u * maxbits + 4u + 3u) / 4u;
  for (unsigned i = lane; i < n16; i += 64) lds_raw[i] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  if (lane < valid) {
    float f[16];
    load_block_low<DIMS>(in, fd, first + lane, f);
    LdsBits mem(lds);
    encode_block_low<DIMS, true, INT>(f, mem.bit0 + lane * maxbits, maxbits, mem);
  }
  __syncthreads();
  const unsigned nwords = (valid * maxbits + 63u) >> 6;
  const uint64_t* src = reinterpret_cast<const uint64_t*>(lds);
  uint64_t* dst = stream + (size_t)blockIdx.x * maxbits;
  for (unsigned i = lane; i < nwords; i += 64) dst[i] = src[i];
}

template <int DIMS, bool INT = false>
__global__ __launch_bounds__(64) void zfp_decode_low_f32_kernel(const uint64_t* __restrict__ stream, FieldLow fd,
                                                                unsigned maxbits, float* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  const unsigned nwords = (valid * maxbits + 63u) >> 6;
  const uint64_t* src = stream + (size_t)blockIdx.x * maxbits;
  uint64_t* dst = reinterpret_cast<uint64_t*>(lds);
  for (unsigned i = lane; i < nwords + 2; i += 64) dst[i] = i < nwords ? src[i] : 0;
  __syncthreads();
  if (lane < valid) {
    float f[16];
    LdsBits mem(lds);
    decode_block_low<DIMS, INT>(mem, mem.bit0 + lane * maxbits, maxbits, f);
    store_block_low<DIMS>(out, fd, first + lane, f);
  }
}

// 64-bit elements, 2-D / 1-D
template <int DIMS, bool INT>
__global__ __launch_bounds__(64) void zfp_encode_low_w64_kernel(const uint64_t* __restrict__ in, FieldLow fd,
                                                                unsigned maxbits, uint64_t* __restrict__ stream)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  const unsigned n16 = (2u * maxbits + 4u + 3u) / 4u;
  for (unsigned i = lane; i < n16; i += 64) lds_raw[i] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  if (lane < valid) {
    const uint32_t b = first + lane;
    const uint32_t r = b / fd.mx;
    const uint32_t x0 = (b - r * fd.mx) * 4, y0 = DIMS == 2 ? r * 4 : 0;
    const uint64_t* p = in + (long long)x0 * fd.sx + (long long)y0 * fd.sy;
    const uint32_t bx = min(4u, fd.nx - x0), by = DIMS == 2 ? min(4u, fd.ny - y0) : 1u;
    uint64_t q[16];
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
      for (int x = 0; x < 4; x++) {
        bool ok = (uint32_t)x < bx && (uint32_t)y < by;
        q[4 * y + x] = ok ? p[x * fd.sx + y * fd.sy] : 0ull;
      }
#pragma unroll
    for (int y = 0; y < (DIMS == 2 ? 4 : 1); y++) pad4(q[4 * y], q[4 * y + 1], q[4 * y + 2], q[4 * y + 3], bx);
    if (DIMS == 2) {
#pragma unroll
      for (int x = 0; x < 4; x++) pad4(q[x], q[x + 4], q[x + 8], q[x + 12], by);
    }
    LdsBits mem(lds);
    encode_block_low_w64<DIMS, true, INT>(q, mem.bit0 + lane * maxbits, maxbits, mem);
  }
  __syncthreads();
  const unsigned nwords = (valid * maxbits + 63u) >> 6;
  const uint64_t* src = reinterpret_cast<const uint64_t*>(lds);
  uint64_t* dst = stream + (size_t)blockIdx.x * maxbits;
  for (unsigned i = lane; i < nwords; i += 64) dst[i] = src[i];
}

template <int DIMS, bool INT>
__global__ __launch_bounds__(64) void zfp_decode_low_w64_kernel(const uint64_t* __restrict__ stream, FieldLow fd,
                                                                unsigned maxbits, uint64_t* __restrict__ out)
{
  extern __shared__ uint4 lds_raw[];
  uint32_t* lds = reinterpret_cast<uint32_t*>(lds_raw);
  const unsigned lane = threadIdx.x;
  const uint32_t first = blockIdx.x * 64u;
  const uint32_t valid = min(64u, fd.nblocks - first);
  const unsigned nwords = (valid * maxbits + 63u) >> 6;
  const uint64_t* src = stream + (size_t)blockIdx.x * maxbits;
  uint64_t* dst = reinterpret_cast<uint64_t*>(lds);
  for (unsigned i = lane; i < nwords + 2; i += 64) dst[i] = i < nwords ? src[i] : 0;
  __syncthreads();
  if (lane < valid) {
    uint64_t q[16];
    LdsBits mem(lds);
    decode_block_low_w64<DIMS, INT>(mem, mem.bit0 + lane * maxbits, maxbits, q);
    const uint32_t b = first + lane;
    const uint32_t r = b / fd.mx;
    const uint32_t x0 = (b - r * fd.mx) * 4, y0 = DIMS == 2 ? r * 4 : 0;
    uint64_t* p = out + (long long)x0 * fd.sx + (long long)y0 * fd.sy;
    const uint32_t bx = min(4u, fd.nx - x0), by = DIMS == 2 ? min(4u, fd.ny - y0) : 1u;
#pragma unroll
    for (int y = 0; y < 4; y++)
#pragma unroll
      for (int x = 0; x < 4; x++)
        if ((uint32_t)x < bx && (uint32_t)y < by) p[x * fd.sx + y * fd.sy] = q[4 * y + x];
  }
}

static int make_field_low(FieldLow& fd, int dims, const void* base, const void* stream, size_t nx, size_t ny,
                          ptrdiff_t sx, ptrdiff_t sy, unsigned maxbits, unsigned elem)
{
  if (dims == 1) ny = 1;
  if (!nx || !ny || maxbits < 16 || maxbits > 4096) return CSWAP_E_ARG;
  if (nx > 0x7fffffffu || ny > 0x7fffffffu) return CSWAP_E_ARG;
  if (((uintptr_t)stream % 8) != 0 || ((uintptr_t)base % elem) != 0) return CSWAP_E_ARG;
  size_t mx = (nx + 3) / 4, my = dims == 2 ? (ny + 3) / 4 : 1;
  size_t nb = mx * my;
  if (nb > 0xfffffff0ull) return CSWAP_E_ARG;
  fd.nx = (uint32_t)nx; fd.ny = (uint32_t)ny; fd.mx = (uint32_t)mx; fd.nblocks = (uint32_t)nb;
  fd.sx = sx ? sx : 1;
  fd.sy = sy ? sy : (ptrdiff_t)nx;
  return CSWAP_OK;
}

// ------------------------------------------------------------- host side
// Whether the decoder stores a field's aligned rows with the nontemporal hint: base, pitch (row to row) and plane
// (plane to plane) in bytes.  Where every row starts on a 128-byte line one instruction writes whole lines, and the hint
// pays at any size: 402.7 MB decode in 107 us instead of 117, and the kernel that runs next no longer waits behind those
// lines draining from the memory-side cache (33.6 MB: 14.5 instead of 17.6 us, a reader of the result right after it
// no slower).  A line that several instructions write in parts leaves the cache in those parts, each a write of its own to
// memory; without the hint it is put together there.  That hurts where the parts are small or many; a field of some 20 MB
// is through before it does.  Microseconds at 8 bits per value, one tensor over and over / several in turn, hint : none --
//   half lines: 64 bytes a row 18 MB 12.2 : 13.0 / 11.6 : 14.1 · 36: 15.3 : 16.2 / 16.5 : 17.3 · 43: 17.7 : 16.6 / 18.4 : 17.9 ·
//     110: 38.4 : 29.7 / 38.3 : 35.8 · 140: 45.5 : 36.0 / 45.0 : 45.7 (268 MB 75.8 : 79.8); 192 bytes 36: 13.7 : 15.9 / 14.5 : 17.1 ·
//     58: 18.9 : 19.1 / 19.1 : 20.5 · 110: 31.9 : 29.1 / 32.3 : 35.3; 320 bytes 58: 18.3 : 19.0 / 18.4 : 20.5 · 110: 29.9 : 29.1 / 30.2 : 35.2 ·
//     140: 35.8 : 35.4 / 35.8 : 43.5
//   smaller parts: 16 bytes 11 MB 12.7 : 12.4 / 23.9 : 12.6; 32 bytes 15: 11.3 : 12.0 / 16.2 : 12.5; 112 bytes 15: 11.9 : 12.0 / 13.2 : 12.7 · 43: 25.6 :
//     17.0 / 27.0 : 19.8; 160 bytes 25: 13.5 : 13.8 / 14.8 : 15.9 · 30: 15.5 : 14.2 / 16.8 : 16.6; 784 bytes 21: 13.2 : 13.3 / 13.1 : 15.3 · 30: 15.3 : 14.3 /
//     15.5 : 17.1 · 50: 22.2 : 17.7 / 22.5 : 22.9; 1552 to 6160 bytes 50: 19.7-22.4 : 17.4-18.0 / 20.1-22.5 : 21.3-22.2 · 100: 36-40 : 28-30 /
//     36-40 : 37-39 · 200, in turn: 68.4 : 65.3.  They take more at 4 bits (24 MB of 160 bytes 12.3 : 12.2 / 13.1 : 14.1) and less at 16 (36: 21.3 :
//     20.4 / 22.3 : 23.5; 18 MB of 96 bytes 14.9 : 15.7 / 16.3 : 18.5)
//   rows of whole lines that start 16 bytes into one: 128 bytes 21 MB 12.9 : 13.3 / 14.4 : 15.1 · 50: 26.8 : 17.6 / 27.8 : 19.4 · 140: 73.1 : 36.0 / 73.4 :
//     46.7; 512 bytes 36: 15.1 : 16.2 / 15.9 : 17.9 · 50: 19.9 : 17.5 / 20.1 : 19.4; 3072 bytes 50: 20.2 : 17.3 / 20.5 : 21.0 · 200: 66 : 47 / 66 : 62
static bool row_store_hint(unsigned long long base, unsigned long long pitch, unsigned long long plane, unsigned long long bytes,
                           unsigned maxbits)
{
  const unsigned long long starts = base | pitch | plane;
  const unsigned long long mib = bytes >> 20;
  if (starts % 128 == 0) return true;
  if (starts % 64 == 0) return bytes >= kReadOnceBytes || pitch >= 320 || mib < (pitch >= 192 ? 56u : 38u);
  if (bytes >= kReadOnceBytes) return false;
  if (pitch >= 1536) return true;
  if (pitch >= 256 && pitch % 64 == 0) return mib < 36;
  const unsigned rate = maxbits / 64;  // bits per value
  if (pitch >= 160) return mib < (rate < 20 ? 16 + rate : 36);
  return pitch >= 96 && pitch * maxbits >= 128 * 512 && mib < 20;
}

static int make_field(Field3& fd, const void* base, const void* stream, size_t nx, size_t ny, size_t nz,
                      ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, unsigned elem)
{
  if (((uintptr_t)stream % 8) != 0 || ((uintptr_t)base % elem) != 0) return CSWAP_E_ARG;
  if (!nx || !ny || !nz) return CSWAP_E_ARG;
  if (maxbits < 16 || maxbits > 4096) return CSWAP_E_ARG;
  if (nx > 0x7fffffffu || ny > 0x7fffffffu || nz > 0x7fffffffu) return CSWAP_E_ARG;
  size_t mx = (nx + 3) / 4, my = (ny + 3) / 4, mz = (nz + 3) / 4;
  size_t nb = mx * my * mz;
  if (nb / mz != mx * my || nb > 0x7fffffffull) return CSWAP_E_ARG;  // block indices stay below 2^31
  fd.nx = (uint32_t)nx; fd.ny = (uint32_t)ny; fd.nz = (uint32_t)nz;
  fd.mx = (uint32_t)mx; fd.my = (uint32_t)my;
  fd.nblocks = (uint32_t)nb;
  fd.sx = sx ? sx : 1;
  fd.sy = sy ? sy : (ptrdiff_t)nx;
  fd.sz = sz ? sz : (ptrdiff_t)(nx * ny);
  fd.by_mx = make_div31(fd.mx);
  fd.by_my = make_div31(fd.my);
  // fast path: aligned contiguous rows; rows inside planes inside the volume (so
  // element offsets grow with the block index); and the slabs of four planes that
  // 64 consecutive blocks can touch (one more than they fill) stay below 4 GiB, so
  // every block of a wavefront is within a 32-bit byte offset of its first block
  const size_t slabs = (64 + mx * my - 1) / (mx * my) + 1;
  const ptrdiff_t per16 = (ptrdiff_t)(16 / elem);  // elements in 16 bytes
  fd.rows16 = fd.sx == 1 && (fd.sy % per16) == 0 && (fd.sz % per16) == 0 && ((uintptr_t)base % 16) == 0 &&
              fd.sy >= (ptrdiff_t)nx && fd.sz >= fd.sy * (ptrdiff_t)ny &&
              (unsigned long long)fd.sz * 4ull * elem * slabs < 0xfff00000ull;
  fd.rows4 = fd.sx == 1 && nx >= 2 && fd.sy >= (ptrdiff_t)nx && fd.sz >= fd.sy * (ptrdiff_t)ny &&
             (unsigned long long)fd.sz * 4ull * elem * slabs < 0xfff00000ull;
  fd.full = fd.rows4 && ((nx | ny | nz) & 3u) == 0;
  fd.stream16 = ((uintptr_t)stream % 16) == 0;
  fd.by_piece = piece_multiplier(maxbits);
  // Cache policy of the field's 16-byte rows.
  // The decoder's stores: row_store_hint.
  // The encoder loads with the hint only when the field is large against that cache (256 MB): a smaller
  // tensor is still cached from the kernel that produced it, and hinted loads of cached lines are slower.
  // Producer kernel + encoder, hinted / plain loads: 402.7 MB 205 / 220 us, 201.3 MB
  // 95 / 109 us, 100.7 MB 43.6 / 43.2 us, 50.3 MB 26.1 / 24.5 us.  Rows shorter than a line and not made of half lines
  // are fetched once per instruction that wants a part of it: hint / none, 32 bytes 268 MB 90 / 68 cold, 96: 151 MB 41.6 /
  // 37.0 warm, 112: 411 MB 107 / 100; from a line on the hint is ahead again (224: 206 MB 51.8 / 54.8).
  // The stream keeps the default policy: the decoder or the copy engine reads it next.
  fd.read_once = (unsigned long long)nx * ny * nz * elem >= kReadOnceBytes;
  fd.store_hint = fd.rows16 && row_store_hint((uintptr_t)base, (unsigned long long)fd.sy * elem, (unsigned long long)fd.sz * elem,
                                             (unsigned long long)nx * ny * nz * elem, maxbits);
  // 64-bit elements: a lane's row is two 16-byte pieces, half a line per store instruction.  The
  // hint on those stores gains 15 % at 537 MB and loses 20 % at 134 MB: only for fields of 256 MiB
  // and more (the memory-side cache's size).
  fd.once64 = elem == 8 && (unsigned long long)nx * ny * nz * elem >= (256ull << 20);
  return CSWAP_OK;
}

}  // namespace cswap

using namespace cswap;

extern "C" size_t cswap_zfp_stream_bytes(size_t nx, size_t ny, size_t nz, unsigned maxbits)
{
  size_t nb = ((nx + 3) / 4) * ((ny + 3) / 4) * ((nz + 3) / 4);
  return (nb * maxbits / 64) * 8;
}

extern "C" size_t cswap_zfp_stream_capacity(size_t nx, size_t ny, size_t nz, unsigned maxbits)
{
  size_t nb = ((nx + 3) / 4) * ((ny + 3) / 4) * ((nz + 3) / 4);
  return ((nb * maxbits + 63) / 64) * 8;
}

// element kinds of a field
enum Elem { kF32 = 0, kI32 = 1, kF64 = 2, kI64 = 3 };
// whole-word rates from this many bits per block of 64 values on run the 32-bit kernels built for fewer wavefronts per SIMD
constexpr unsigned kFewerWavesFrom = 1024;
static unsigned elem_bytes(Elem e) { return e == kF32 || e == kI32 ? 4u : 8u; }

// Fields below this many bytes are coded by the pair form where their shape allows
// (cswap_zfp_set_pair_bytes).
static std::atomic<unsigned long long> g_pair_encode_bytes{CSWAP_PAIR_ENCODE_BYTES};

// what the pair kernels take: the fast path of the field (aligned contiguous rows, an aligned
// stream), full blocks only, and a whole-word rate whose blocks split into two halves of
// whole 16-byte pieces
static bool pair_shape(const Field3& fd, unsigned maxbits)
{
  return fd.rows16 && fd.stream16 && (maxbits & 255u) == 0 && ((fd.nx | fd.ny | fd.nz) & 3u) == 0;
}

// Whether the encoder loads with the nontemporal hint (make_field: read_once); the variants that do are
// those of whole-word rates.
static bool load_hint(const Field3& fd, bool whole)
{
  return fd.read_once && fd.rows16 && whole && (fd.sy % 16 == 0 || fd.sy >= 32);  // (elements; make_field has the reasons)
}

// Which fields the kernels for contiguous rows at any element take.  The encoder's: all that are not
// whole blocks of aligned rows.  Both leave fields whose rows are aligned and whole along x to the other
// kernel where that one has the hint: only the last block rows are cut off there, and the hint on the
// others' whole lines is worth more.  The decoder's has it always, and takes no other fields (39 MB in 197 rows of 768: encode
// 20.8 us either way, decode 16.2 with the other kernel, 17.1 with this; 57 MB in 197 rows of 196: encode
// 28.1 and 26.3, decode 28.3 both), the encoder's on large fields (producer kernel + encoder, other kernel
// / this, 197 rows of 768 or 3072: 201 MB at 8 bits per value 116 / 123 us, 290 MB 156 / 172, 402 MB
// 220 / 232; the encoder by itself, over and over on what is cached, 59.9 / 58.8, 74.1 / 75.8 and 101.1 /
// 100.7, at 16 bits 71.2 / 73.7, 96.0 / 103.9 and 127 / 140).  Cut off along x, the hint gains less
// than the rows (203 MB in 197 rows of 771 at a pitch of 772: 130 / 124).
static bool encode_rows(const Field3& fd, bool whole)
{
  return fd.rows4 && !(fd.full && fd.rows16) && !(load_hint(fd, whole) && (fd.nx & 3u) == 0);
}
static bool decode_rows(const Field3& fd) { return fd.rows4 && !(fd.store_hint && (fd.nx & 3u) == 0); }

// Which packed fields of floats the decoder stores as runs through LDS, and whether with the hint; us at 8 bits per value,
// one tensor over and over (several in turn).
//  - Rows of whole 16 bytes: with the hint, at all sizes and down to 48 lanes of 64 with a block (52x52 52 lanes, 60 MB
//    20.0 -> 19.5 (24.7 -> 19.4); 100x100 50 lanes, 150 MB 37.8 -> 38.1 (52.8 -> 39.4)).  Not where rows are whole lines, nor where row stores
//    do as well: half lines from 320 bytes a row on (80x80 60 MB 18.4 and 18.4 (18.7 and 18.6); 112x112 19 MB 11.2 and 12.6 (11.6 and
//    11.8)), 192 bytes below 38 MiB (20 MB 11.3 and 12.7 (11.7 and 12.0); 60 MB 19.6 -> 18.6 (21.1 -> 18.7)).
//  - Other rows: their runs end inside lines.  Below 40 MiB the hint pays all the same (plain / hint: 35x35 20 MB 14.3 / 14.4 (15.6 /
//    13.2), 31x31 36 MB 17.6 / 15.9 (19.2 / 16.3), 33x33 36 MB 21.2 / 19.6 (23.1 / 20.0; row stores 21.0 and 23.5)) unless a plane is
//    shorter than two lines (6x6 36 MB 20.3 / 24.3 (21.6 / 25.6)); fewer than 56 lanes only below 24 MiB (softmax values: 49x49 22 MB row
//    stores 17.4, runs 17.0 (17.6, 16.2), 39 MB at 4 bits 17.8 and 18.9).  From there on it costs (35x35 60 MB 21.3 / 25.7 (23.9 / 26.2)),
//    and without it lanes left over and padding tell.  A last block of one column never pays: 5x5 150 MB 101 -> 105 (108 -> 107), 13x13
//    64 -> 67 (73 -> 70), 17x17 60 MB 30.6 -> 33.4 (33.1 -> 35.9), 33x33 27.7 -> 28.7 (30.5 -> 31.2).  Other rows of 16 elements and more are asked
//    to fill 7/8 of what a wavefront can hold (30x30 0.88: 22.8 -> 22.2 (24.1 -> 23.8); 50x50 0.75: 21.4 -> 22.1 (25.9 -> 24.5)), shorter
//    ones gain whatever they fill (15x15 30 -> 24 (31 -> 25), 6x6 38 -> 30 (41 -> 33), 3x3 58 -> 33 (60 -> 42)), and rows from
//    252 bytes on gain nothing (63x63 60 MB 20.8 -> 20.9 (22.8 -> 23.3), 127x127 20.0 -> 20.5 (22.3 -> 22.6)).
//  - Either only where blocks are full enough: most of the image is padding with one row to a plane (28x1 150 MB 97 -> 106 (97 -> 109),
//    15x1 30 MB 1.19 times), and with two in rows of more than 8 (100x2 150 MB 1.23 times (1.10), 35x2 30 MB 1.04 (1.07)).
//    With the hint a plane that is not whole 64-byte sectors ends inside one, which is then written twice, and a short plane is little
//    else: 150 MB in 4x2 3.0 times (2.3), 8x7 1.59 (1.14), 12x3 2.2 (1.6), 28x7 1.32 (1.01), 24x7 1.22 (0.96); from 1 KB on 28x10 1.01 (0.75),
//    100x3 1.18 (0.87), 252x9 0.99 (0.75); whole sectors 8x6 1.01 (0.76), 16x3 0.58 (0.49).
enum RunsRoute { kNoRuns, kRunsPlain, kRunsHint };
static RunsRoute decode_runs(const Field3& fd, uintptr_t base)
{
  const bool packed = fd.rows4 && fd.sy == (long long)fd.nx && fd.sz == fd.sy * (long long)fd.ny;
  if (!packed || fd.mx > 64 || fd.sz >= (long long)kRunsPlaneElements || fd.nx % 32 == 0) return kNoRuns;
  const unsigned lanes = 64 / fd.mx * fd.mx;
  if (lanes < 48 || fd.ny == 1 || (fd.ny == 2 && fd.nx > 8 && fd.nx % 16 != 0)) return kNoRuns;
  const unsigned long long bytes = 4ull * fd.nx * fd.ny * fd.nz;
  if (fd.nx % 4 == 0 && base % 16 == 0) {
    if (fd.sz % 16 != 0 && 4 * fd.sz < 1024) return kNoRuns;
    if (fd.nx % 16 == 0 && base % 64 == 0 && (fd.nx >= 80 || (fd.nx == 48 && bytes < (38ull << 20)))) return kNoRuns;
    return kRunsHint;
  }
  if (bytes < ((lanes < 56 ? 24ull : 40ull) << 20)) return 4 * fd.sz >= 256 ? kRunsHint : kRunsPlain;
  const unsigned long long held = (unsigned long long)lanes * fd.nx * fd.ny, room = 64ull * 16 * fd.mx * fd.my;
  return fd.nx % 4 != 1 && (fd.nx < 16 || (fd.nx < 63 && 8 * held >= 7 * room)) ? kRunsPlain : kNoRuns;
}

static std::atomic<unsigned long long> g_pair_decode_bytes{CSWAP_PAIR_DECODE_BYTES};

// The pair form pays while all of a field's workgroups are on the chip at once (twice the
// wavefronts, each with half the serial work); a field that needs a second round of them is
// faster with one lane per block.  How many workgroups a compute unit holds is set by their
// LDS: measured, 88 % of what its 160 KB divided by the workgroup's bytes allows.  A limit of
// SIZE_MAX takes the form for every field it can code (tests, measurements).
static bool pair_fits(unsigned grid, size_t lds_bytes, unsigned long long limit)
{
  if (limit == ~0ull) return true;
  const double per_cu = 0.88 * 160.0 * 1024.0 / (double)lds_bytes;
  return (double)grid <= per_cu * (double)device_compute_units();
}
// The decoder's pair form, whose planes one half decodes alone, pays while every workgroup has a SIMD of
// its own -- then what the halves share is worth its barriers -- and the planes are not all of the time.  One lane
// per block / pair form, us, one tensor over and over (several in turn), 16.5 MB: 16 bits per value in 64x64 planes 12.3 / 11.9 (13.0 /
// 12.7), 28x28 16.1 / 15.0 (16.5 / 15.3), 8x8 14.7 / 14.1 (16.7 / 16.0); 20 bits 12.5 / 12.4 (13.3 / 13.4), 16.2 / 15.4 (16.9 / 16.4), 14.9 / 14.6;
// 24 bits 12.5 / 12.6 (13.6 / 14.0), 16.2 / 15.8 (17.0 / 16.8), 14.9 / 14.9; 28 bits 12.6 / 13.0 (14.0 / 14.5), 16.4 / 16.2 (17.4 / 17.5), 15.2 / 15.3; 10 MB
// alike.  Beyond one workgroup per SIMD, at 16 bits: 21 MB 14.6 / 14.6, 25.2 MB 14.3 / 15.2, 41.9 MB 17.1 / 23.3.  At 8 bits 12.6 MB 11.1 /
// 10.8, 16.8 MB 10.9 / 10.9.
constexpr unsigned kPairDecodeFromBits = 1024, kPairDecodeBelowBits = 1792;
static bool pair_decode_pays(unsigned grid, unsigned maxbits, unsigned long long limit)
{
  if (limit == ~0ull) return true;
  return maxbits >= kPairDecodeFromBits && maxbits < kPairDecodeBelowBits && grid <= 4u * (unsigned)device_compute_units();
}

// The quad form pays while its wavefronts (16 blocks each) are few per compute unit: it trades
// instructions (half as many again as the pair form's, for the same blocks) for short chains.
// Microseconds, quad / pair / one lane per block at 8 bits per value by wavefronts per compute unit:
//   encode  1 (1 MB) 4.5 / 6.1 / 7.6 · 4: 5.2 / 6.4 / 7.8 · 8: 6.6 / 7.6 / 8.5 · 12: 7.8 / 7.9 / 8.9 ·
//           16: 9.2 / 8.2 / 9.3; where the pair form does not apply (odd planes): 8: 6.7 / - / 9.2 ·
//           19: 10.7 / - / 11.9 · 23: 12.5 / - / 12.5 · 25: 14.1 / - / 13.1
//   decode  1: 7.4 / 8.5 / 9.1 · 4: 8.1 / 8.9 / 9.5 · 8: 9.3 / 10.4 / 10.4 · 10: 10.8 / 10.6 / 10.8 · 14: 12.9 / 10.9 / 11.1;
//           odd planes 8: 10.7 / - / 11.7 · 10: 12.8 / - / 12.2 · 15: 15.2 / - / 12.8
// The decoder's lines cross at the same place at 4, 16 and 32 bits per value (9.6 / 9.5 / 9.6, 13.4 / 12.5 / 13.2 and
// 13.6 / 13.2 / 13.1 at 10 wavefronts).  The encoder's against the pair form cross between 11 and 14 (12: 7.0 / 6.9 at 4
// bits, 9.7 / 10.6 at 16, 11.8 / 13.4 at 32); of odd planes at 16 bits 19: 13.9 / 14.9 · 20: 15.3 / 15.2 · 21: 16.3 / 15.5, at 32 bits
// 18: 18.1 / 18.4 · 25: 23.2 / 22.2.  The steps are where the wavefronts' LDS no longer lets all of them onto the chip at once;
// from 30 bits per value on one lane per block meets that limit, too.
constexpr unsigned kQuadWaves = 11;        // per compute unit, the encoder's where the pair form applies
constexpr unsigned kQuadWavesNoPair = 22;  // where it does not
constexpr unsigned kQuadWavesDecode = 9;  // the decoder's; kQuadWaves in rows of at most 32 bytes, where no other form stores with the hint
constexpr unsigned kQuadOneRoundBelow = 1920;
static double quad_waves_encode(const Field3& fd, unsigned maxbits)
{
  if (pair_shape(fd, maxbits)) return kQuadWaves;
  const double fit = 0.92 * 160.0 * 1024.0 / (4.0 * (double)quad_lds_dwords(slot_bits(maxbits)));
  return maxbits < kQuadOneRoundBelow && fit < kQuadWavesNoPair ? fit : kQuadWavesNoPair;
}
// Rows of 16 and 32 bytes: the quad form, whose stores have the hint at any length of row, against what else takes the
// field, one tensor over and over (several in turn), us, 10.4 MB: 16 bytes 8 bits per value 11.2 / 12.0 (11.1 / 12.5), 4 bits 10.0 /
// 10.8 (11.7 / 11.1), 32 bits 13.7 / 14.9 (14.5 / 16.8); 32 bytes 11.0 / 11.2 (10.7 / 11.6), 10.0 / 9.9 (9.5 / 10.2), 13.5 / 14.2 (14.5 / 16.4); 80 bytes
// 12.5 / 11.3 (11.1 / 11.7).  Where the pair form applies 16 bytes at 16 bits 13.7 / 13.9 (13.8 / 14.6), 32 bytes 13.7 / 12.7 (13.8 / 13.6).
static double quad_waves_decode(const Field3& fd, unsigned maxbits)
{
  const bool pair = pair_shape(fd, maxbits) && maxbits >= kPairDecodeFromBits && maxbits < kPairDecodeBelowBits;
  return fd.full && fd.rows16 && fd.sy <= 8 && !pair ? kQuadWaves : kQuadWavesDecode;
}
static bool quad_pays(uint32_t nblocks, double waves, unsigned long long bytes, unsigned long long pair_below, int compute_units)
{
  return pair_below != ~0ull && bytes < pair_below && (double)nblocks <= (double)kQuadBlocks * waves * (double)compute_units;
}

extern "C" void cswap_zfp_set_pair_bytes(size_t encode_below, size_t decode_below, size_t* previous)
{
  const size_t e = (size_t)g_pair_encode_bytes.exchange(encode_below, std::memory_order_relaxed);
  const size_t d = (size_t)g_pair_decode_bytes.exchange(decode_below, std::memory_order_relaxed);
  if (previous) {
    previous[0] = e;
    previous[1] = d;
  }
}

extern "C" int cswap_test_zfp_encode_route(size_t nx, size_t ny, size_t nz, ptrdiff_t sy, ptrdiff_t sz, unsigned misaligned,
                                           unsigned maxbits, int compute_units)
{
  Field3 fd;
  const uintptr_t base = 4096 + 4 * (uintptr_t)misaligned;  // looked at for its alignment only
  int rc = make_field(fd, reinterpret_cast<const void*>(base), reinterpret_cast<const void*>(4096), nx, ny, nz, 1, sy, sz,
                      maxbits, 4);
  if (rc) return rc;
  const bool whole = (maxbits & 63u) == 0;
  if (compute_units > 0 && whole && quad_pays(fd.nblocks, quad_waves_encode(fd, maxbits), (unsigned long long)nx * ny * nz * 4ull,
                                              CSWAP_PAIR_ENCODE_BYTES, compute_units))
    return 3;
  return encode_rows(fd, whole) ? 1 : load_hint(fd, whole) ? 2 : 0;
}

extern "C" int cswap_test_zfp_decode_quad(size_t nx, size_t ny, size_t nz, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits,
                                          int compute_units)
{
  Field3 fd;
  const void* aligned = reinterpret_cast<const void*>((uintptr_t)4096);
  int rc = make_field(fd, aligned, aligned, nx, ny, nz, 1, sy, sz, maxbits, 4);
  if (rc) return rc;
  return (maxbits & 63u) == 0 && quad_pays(fd.nblocks, quad_waves_decode(fd, maxbits), (unsigned long long)nx * ny * nz * 4ull,
                                           CSWAP_PAIR_DECODE_BYTES, compute_units);
}

extern "C" int cswap_test_zfp_decode_runs(size_t nx, size_t ny, size_t nz, ptrdiff_t sy, ptrdiff_t sz, unsigned base)
{
  Field3 fd;
  const void* at = reinterpret_cast<const void*>((uintptr_t)4096 + base);
  int rc = make_field(fd, at, reinterpret_cast<const void*>((uintptr_t)4096), nx, ny, nz, 1, sy, sz, 512, 4);
  return rc ? rc : (int)decode_runs(fd, (uintptr_t)at);
}

extern "C" int cswap_test_zfp_store_hint(unsigned long long base, unsigned long long pitch, unsigned long long plane,
                                         unsigned long long bytes, unsigned maxbits)
{
  return row_store_hint(base, pitch, plane, bytes, maxbits);
}

#define CSWAP_LAUNCH3(KERNEL_, T_, ARG0_, ARG3_)                                                                   \
  do {                                                                                                              \
    if (whole && !is_int)                                                                                           \
      hipLaunchKernelGGL((KERNEL_<true, false>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);   \
    else if (!whole && !is_int)                                                                                     \
      hipLaunchKernelGGL((KERNEL_<false, false>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);  \
    else if (whole)                                                                                                 \
      hipLaunchKernelGGL((KERNEL_<true, true>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);    \
    else                                                                                                            \
      hipLaunchKernelGGL((KERNEL_<false, true>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);   \
  } while (0)

// quad: false leaves out the form with four lanes per block
static int compress3(const void* d_in, Elem elem, size_t nx, size_t ny, size_t nz, ptrdiff_t sx, ptrdiff_t sy,
                     ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream, cswap_stream_t stream, bool quad = true)
{
  if (!d_in || !d_stream) return CSWAP_E_ARG;
  Field3 fd;
  int rc = make_field(fd, d_in, d_stream, nx, ny, nz, sx, sy, sz, maxbits, elem_bytes(elem));
  if (rc) return rc;
  unsigned grid = (fd.nblocks + 63) / 64;
  size_t lds_bytes = (size_t)region_dwords(maxbits) * 4;
  hipStream_t st = (hipStream_t)stream;
  const bool whole = (maxbits & 63u) == 0;
  const bool is_int = elem == kI32 || elem == kI64;
  const unsigned long long pair_below = g_pair_encode_bytes.load(std::memory_order_relaxed);
  if (quad && elem == kF32 && whole && quad_pays(fd.nblocks, quad_waves_encode(fd, maxbits),
                                          (unsigned long long)nx * ny * nz * 4ull, pair_below, device_compute_units())) {
    hipLaunchKernelGGL(zfp_encode3_f32_quad_kernel, dim3((fd.nblocks + kQuadBlocks - 1) / kQuadBlocks), dim3(64),
                       (size_t)quad_lds_dwords(slot_bits(maxbits)) * 4, st, static_cast<const float*>(d_in), fd, maxbits,
                       d_stream);
    return check_launch();
  }
  if (elem == kF32 && pair_shape(fd, maxbits) && (unsigned long long)nx * ny * nz * 4ull < pair_below &&
      pair_fits(grid, (size_t)pair_lds_dwords(maxbits) * 4 + sizeof(ExpandTable), pair_below)) {
    hipLaunchKernelGGL(zfp_encode3_f32_pair_kernel, dim3(grid), dim3(128), (size_t)pair_lds_dwords(maxbits) * 4, st,
                       static_cast<const float*>(d_in), fd, maxbits, d_stream);
    return check_launch();
  }
  if (elem_bytes(elem) == 4) {
    const float* in = static_cast<const float*>(d_in);
    const bool once = load_hint(fd, whole);
    if (encode_rows(fd, whole)) {
      if (whole && maxbits >= kFewerWavesFrom && !is_int)
        hipLaunchKernelGGL((zfp_encode3_rows_kernel<true, false, 3>), dim3(grid), dim3(64), lds_bytes, st, in, fd, maxbits,
                           d_stream);
      else if (whole && maxbits >= kFewerWavesFrom)
        hipLaunchKernelGGL((zfp_encode3_rows_kernel<true, true, 3>), dim3(grid), dim3(64), lds_bytes, st, in, fd, maxbits,
                           d_stream);
      else
        CSWAP_LAUNCH3(zfp_encode3_rows_kernel, float, in, d_stream);
    } else if (whole && maxbits >= kFewerWavesFrom) {
      if (once && !is_int)
        hipLaunchKernelGGL((zfp_encode3_f32_kernel<true, false, true, 3>), dim3(grid), dim3(64), lds_bytes, st, in,
                           fd, maxbits, d_stream);
      else if (once)
        hipLaunchKernelGGL((zfp_encode3_f32_kernel<true, true, true, 3>), dim3(grid), dim3(64), lds_bytes, st, in,
                           fd, maxbits, d_stream);
      else if (!is_int)
        hipLaunchKernelGGL((zfp_encode3_f32_kernel<true, false, false, 3>), dim3(grid), dim3(64), lds_bytes, st, in,
                           fd, maxbits, d_stream);
      else
        hipLaunchKernelGGL((zfp_encode3_f32_kernel<true, true, false, 3>), dim3(grid), dim3(64), lds_bytes, st, in,
                           fd, maxbits, d_stream);
    } else if (once && !is_int)
      hipLaunchKernelGGL((zfp_encode3_f32_kernel<true, false, true>), dim3(grid), dim3(64), lds_bytes, st, in, fd,
                         maxbits, d_stream);
    else if (once)
      hipLaunchKernelGGL((zfp_encode3_f32_kernel<true, true, true>), dim3(grid), dim3(64), lds_bytes, st, in, fd,
                         maxbits, d_stream);
    else
      CSWAP_LAUNCH3(zfp_encode3_f32_kernel, float, in, d_stream);
  } else {
    const uint64_t* in = static_cast<const uint64_t*>(d_in);
    CSWAP_LAUNCH3(zfp_encode3_w64_kernel, uint64_t, in, d_stream);
  }
  return check_launch();
}

static int decompress3(const uint64_t* d_stream, Elem elem, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                       ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, void* d_out, cswap_stream_t stream,
                       bool quad = true)
{
  if (!d_out || !d_stream) return CSWAP_E_ARG;
  Field3 fd;
  int rc = make_field(fd, d_out, d_stream, nx, ny, nz, sx, sy, sz, maxbits, elem_bytes(elem));
  if (rc) return rc;
  unsigned grid = (fd.nblocks + 63) / 64;
  size_t lds_bytes = (size_t)region_dwords(maxbits) * 4;
  hipStream_t st = (hipStream_t)stream;
  const bool whole = (maxbits & 63u) == 0;
  const bool is_int = elem == kI32 || elem == kI64;
  const unsigned long long pair_below = g_pair_decode_bytes.load(std::memory_order_relaxed);
  if (quad && elem == kF32 && whole && quad_pays(fd.nblocks, quad_waves_decode(fd, maxbits), (unsigned long long)nx * ny * nz * 4ull,
                                                 pair_below, device_compute_units())) {
    hipLaunchKernelGGL(zfp_decode3_f32_quad_kernel, dim3((fd.nblocks + kQuadBlocks - 1) / kQuadBlocks), dim3(64),
                       (size_t)quad_lds_dwords(dec_slot_bits(maxbits)) * 4, st, d_stream, fd, maxbits,
                       static_cast<float*>(d_out));
    return check_launch();
  }
  if (elem == kF32 && pair_shape(fd, maxbits) && (unsigned long long)nx * ny * nz * 4ull < pair_below &&
      pair_decode_pays(grid, maxbits, pair_below)) {
    const auto kernel = fd.store_hint ? zfp_decode3_f32_pair_kernel : zfp_decode3_f32_pair_plain_kernel;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(128), (size_t)pair_dec_lds_dwords(maxbits) * 4, st, d_stream, fd, maxbits,
                       static_cast<float*>(d_out));
    return check_launch();
  }
  if (elem_bytes(elem) == 4) {
    float* out = static_cast<float*>(d_out);
    lds_bytes = (size_t)dec_region_dwords(maxbits) * 4;
    const RunsRoute route = elem == kF32 && whole ? decode_runs(fd, (uintptr_t)d_out) : kNoRuns;
    if (route != kNoRuns) {
      const Runs runs = make_runs(fd.nx, fd.ny, fd.nz, (uintptr_t)d_out);
      const bool fewer = maxbits >= kFewerWavesFrom;
      const auto kernel =
          runs.unit == 4 ? (fewer ? zfp_decode3_runs_kernel<4, true, 4> : zfp_decode3_runs_kernel<4, true, 5>)
          : runs.unit == 2
              ? (route == kRunsHint ? (fewer ? zfp_decode3_runs_kernel<2, true, 4> : zfp_decode3_runs_kernel<2, true, 5>)
                                    : (fewer ? zfp_decode3_runs_kernel<2, false, 4> : zfp_decode3_runs_kernel<2, false, 5>))
              : (route == kRunsHint ? (fewer ? zfp_decode3_runs_kernel<1, true, 4> : zfp_decode3_runs_kernel<1, true, 5>)
                                    : (fewer ? zfp_decode3_runs_kernel<1, false, 4> : zfp_decode3_runs_kernel<1, false, 5>));
      lds_bytes = std::max(lds_bytes, (size_t)kRunsImageDwords * 4);
      hipLaunchKernelGGL(kernel, dim3((runs.block_rows + runs.rows - 1) / runs.rows), dim3(64), lds_bytes, st, d_stream, fd,
                         runs, maxbits, out);
      return check_launch();
    }
    if (decode_rows(fd)) {
      if (whole && maxbits >= kFewerWavesFrom && !is_int)
        hipLaunchKernelGGL((zfp_decode3_rows_kernel<true, false, 4>), dim3(grid), dim3(64), lds_bytes, st, d_stream, fd,
                           maxbits, out);
      else if (whole && maxbits >= kFewerWavesFrom)
        hipLaunchKernelGGL((zfp_decode3_rows_kernel<true, true, 4>), dim3(grid), dim3(64), lds_bytes, st, d_stream, fd,
                           maxbits, out);
      else
        CSWAP_LAUNCH3(zfp_decode3_rows_kernel, float, d_stream, out);
    } else if (whole && maxbits >= kFewerWavesFrom && !is_int)
      hipLaunchKernelGGL((zfp_decode3_f32_kernel<true, false, 4>), dim3(grid), dim3(64), lds_bytes, st, d_stream, fd,
                         maxbits, out);
    else if (whole && maxbits >= kFewerWavesFrom)
      hipLaunchKernelGGL((zfp_decode3_f32_kernel<true, true, 4>), dim3(grid), dim3(64), lds_bytes, st, d_stream, fd,
                         maxbits, out);
    else
      CSWAP_LAUNCH3(zfp_decode3_f32_kernel, float, d_stream, out);
  } else {
    uint64_t* out = static_cast<uint64_t*>(d_out);
    if (fd.once64 && fd.rows16 && whole && !is_int)
      hipLaunchKernelGGL((zfp_decode3_w64_kernel<true, false, true>), dim3(grid), dim3(64), lds_bytes, st, d_stream,
                         fd, maxbits, out);
    else if (fd.once64 && fd.rows16 && whole)
      hipLaunchKernelGGL((zfp_decode3_w64_kernel<true, true, true>), dim3(grid), dim3(64), lds_bytes, st, d_stream,
                         fd, maxbits, out);
    else
      CSWAP_LAUNCH3(zfp_decode3_w64_kernel, uint64_t, d_stream, out);
  }
  return check_launch();
}
#undef CSWAP_LAUNCH3

extern "C" int cswap_zfp_compress_f32(const float* d_in, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                                      ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream,
                                      cswap_stream_t stream)
{
  return compress3(d_in, kF32, nx, ny, nz, sx, sy, sz, maxbits, d_stream, stream);
}

extern "C" int cswap_zfp_decompress_f32(const uint64_t* d_stream, size_t nx, size_t ny, size_t nz,
                                        ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits,
                                        float* d_out, cswap_stream_t stream)
{
  return decompress3(d_stream, kF32, nx, ny, nz, sx, sy, sz, maxbits, d_out, stream);
}

// A packed field through the forms that fields of every size share (common.h).
int cswap::zfp_compress_f32_no_quad(const float* d_in, size_t nx, size_t ny, size_t nz, unsigned maxbits, uint64_t* d_stream,
                                    hipStream_t stream)
{
  return compress3(d_in, kF32, nx, ny, nz, 0, 0, 0, maxbits, d_stream, stream, false);
}
int cswap::zfp_decompress_f32_no_quad(const uint64_t* d_stream, size_t nx, size_t ny, size_t nz, unsigned maxbits, float* d_out,
                                      hipStream_t stream)
{
  return decompress3(d_stream, kF32, nx, ny, nz, 0, 0, 0, maxbits, d_out, stream, false);
}

// ------------------------------------------------------------- any dimensionality
static size_t blocks_nd(int dims, size_t nx, size_t ny, size_t nz)
{
  size_t nb = (nx + 3) / 4;
  if (dims >= 2) nb *= (ny + 3) / 4;
  if (dims >= 3) nb *= (nz + 3) / 4;
  return nb;
}

extern "C" size_t cswap_zfp_stream_capacity_nd(int dims, size_t nx, size_t ny, size_t nz, unsigned maxbits)
{
  if (dims < 1 || dims > 3) return 0;
  return ((blocks_nd(dims, nx, ny, nz) * maxbits + 63) / 64) * 8;
}

extern "C" size_t cswap_zfp_stream_bytes_nd(int dims, size_t nx, size_t ny, size_t nz, unsigned maxbits)
{
  if (dims < 1 || dims > 3) return 0;
  if (dims == 3) return cswap_zfp_stream_bytes(nx, ny, nz, maxbits);
  return cswap_zfp_stream_capacity_nd(dims, nx, ny, nz, maxbits);  // 1-D and 2-D round up (zfp/shared.h:42-71)
}

#define CSWAP_LAUNCH_LOW(KERNEL_, ARG0_, ARG3_)                                                                  \
  do {                                                                                                             \
    if (dims == 2 && !is_int)                                                                                      \
      hipLaunchKernelGGL((KERNEL_<2, false>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);     \
    else if (dims == 2)                                                                                            \
      hipLaunchKernelGGL((KERNEL_<2, true>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);      \
    else if (!is_int)                                                                                              \
      hipLaunchKernelGGL((KERNEL_<1, false>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);     \
    else                                                                                                           \
      hipLaunchKernelGGL((KERNEL_<1, true>), dim3(grid), dim3(64), lds_bytes, st, ARG0_, fd, maxbits, ARG3_);      \
  } while (0)

static int compress_nd(const void* d_in, Elem elem, int dims, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                       ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream, cswap_stream_t stream)
{
  if (dims == 3) return compress3(d_in, elem, nx, ny, nz, sx, sy, sz, maxbits, d_stream, stream);
  if (!d_in || !d_stream || (dims != 1 && dims != 2)) return CSWAP_E_ARG;
  FieldLow fd;
  int rc = make_field_low(fd, dims, d_in, d_stream, nx, ny, sx, sy, maxbits, elem_bytes(elem));
  if (rc) return rc;
  unsigned grid = (fd.nblocks + 63) / 64;
  size_t lds_bytes = (size_t)((2u * maxbits + 4u + 3u) / 4u) * 16;
  hipStream_t st = (hipStream_t)stream;
  const bool is_int = elem == kI32 || elem == kI64;
  if (elem_bytes(elem) == 4) {
    const float* in = static_cast<const float*>(d_in);
    CSWAP_LAUNCH_LOW(zfp_encode_low_f32_kernel, in, d_stream);
  } else {
    const uint64_t* in = static_cast<const uint64_t*>(d_in);
    CSWAP_LAUNCH_LOW(zfp_encode_low_w64_kernel, in, d_stream);
  }
  return check_launch();
}

static int decompress_nd(const uint64_t* d_stream, Elem elem, int dims, size_t nx, size_t ny, size_t nz,
                         ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, void* d_out,
                         cswap_stream_t stream)
{
  if (dims == 3) return decompress3(d_stream, elem, nx, ny, nz, sx, sy, sz, maxbits, d_out, stream);
  if (!d_out || !d_stream || (dims != 1 && dims != 2)) return CSWAP_E_ARG;
  FieldLow fd;
  int rc = make_field_low(fd, dims, d_out, d_stream, nx, ny, sx, sy, maxbits, elem_bytes(elem));
  if (rc) return rc;
  unsigned grid = (fd.nblocks + 63) / 64;
  size_t lds_bytes = (size_t)((2u * maxbits + 4u + 3u) / 4u) * 16;
  hipStream_t st = (hipStream_t)stream;
  const bool is_int = elem == kI32 || elem == kI64;
  if (elem_bytes(elem) == 4) {
    float* out = static_cast<float*>(d_out);
    CSWAP_LAUNCH_LOW(zfp_decode_low_f32_kernel, d_stream, out);
  } else {
    uint64_t* out = static_cast<uint64_t*>(d_out);
    CSWAP_LAUNCH_LOW(zfp_decode_low_w64_kernel, d_stream, out);
  }
  return check_launch();
}
#undef CSWAP_LAUNCH_LOW

extern "C" int cswap_zfp_compress_f32_nd(const float* d_in, int dims, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                                         ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream,
                                         cswap_stream_t stream)
{
  return compress_nd(d_in, kF32, dims, nx, ny, nz, sx, sy, sz, maxbits, d_stream, stream);
}

extern "C" int cswap_zfp_decompress_f32_nd(const uint64_t* d_stream, int dims, size_t nx, size_t ny, size_t nz,
                                           ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, float* d_out,
                                           cswap_stream_t stream)
{
  return decompress_nd(d_stream, kF32, dims, nx, ny, nz, sx, sy, sz, maxbits, d_out, stream);
}

extern "C" int cswap_zfp_compress_i32_nd(const int32_t* d_in, int dims, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                                         ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream,
                                         cswap_stream_t stream)
{
  return compress_nd(d_in, kI32, dims, nx, ny, nz, sx, sy, sz, maxbits, d_stream, stream);
}

extern "C" int cswap_zfp_decompress_i32_nd(const uint64_t* d_stream, int dims, size_t nx, size_t ny, size_t nz,
                                           ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits,
                                           int32_t* d_out, cswap_stream_t stream)
{
  return decompress_nd(d_stream, kI32, dims, nx, ny, nz, sx, sy, sz, maxbits, d_out, stream);
}

extern "C" int cswap_zfp_compress_f64_nd(const double* d_in, int dims, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                                         ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream,
                                         cswap_stream_t stream)
{
  return compress_nd(d_in, kF64, dims, nx, ny, nz, sx, sy, sz, maxbits, d_stream, stream);
}

extern "C" int cswap_zfp_decompress_f64_nd(const uint64_t* d_stream, int dims, size_t nx, size_t ny, size_t nz,
                                           ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, double* d_out,
                                           cswap_stream_t stream)
{
  return decompress_nd(d_stream, kF64, dims, nx, ny, nz, sx, sy, sz, maxbits, d_out, stream);
}

extern "C" int cswap_zfp_compress_i64_nd(const int64_t* d_in, int dims, size_t nx, size_t ny, size_t nz, ptrdiff_t sx,
                                         ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits, uint64_t* d_stream,
                                         cswap_stream_t stream)
{
  return compress_nd(d_in, kI64, dims, nx, ny, nz, sx, sy, sz, maxbits, d_stream, stream);
}

extern "C" int cswap_zfp_decompress_i64_nd(const uint64_t* d_stream, int dims, size_t nx, size_t ny, size_t nz,
                                           ptrdiff_t sx, ptrdiff_t sy, ptrdiff_t sz, unsigned maxbits,
                                           int64_t* d_out, cswap_stream_t stream)
{
  return decompress_nd(d_stream, kI64, dims, nx, ny, nz, sx, sy, sz, maxbits, d_out, stream);
}
