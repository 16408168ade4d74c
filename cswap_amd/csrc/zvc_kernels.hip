// zvc_kernels.hip -- zero-value compaction (ZVC) of fp32 tensors for gfx950, in
// the reference's on-the-wire format (CSWAP+/zfp/compression.cu): the tensor is
// cut into `process` contiguous chunks of E = ceil(n/process) elements; chunk i
// owns W = ceil(E/32) mask words at word i*W (bit k%32 of word k/32 <=> element
// E*i+k != 0) and its packed non-zeros start at values[begin[i]].
//
// Work decomposition: ONE WAVEFRONT PER CHUNK (the reference uses one thread
// per chunk, which makes every access strided by E).  Lane l of iteration t
// looks at chunk element 64t+l, so loads are contiguous 256-byte rows, one
// __ballot gives the two mask words of the iteration directly in the
// reference's bit order, mbcnt gives each non-zero its slot, and the packed
// stores of a wave are contiguous.  The chunk-granular exclusive scan the
// format carries anyway (`begin`) is the device-wide scan; no finer scan is
// needed.
#include <hip/hip_runtime.h>
#include <atomic>

#include <mutex>

#include "../../include/cswap_hip.h"
#include "../../include/cswap_test_hooks.h"
#include "common.h"
#include "zfp_block.h"  // Div31

namespace cswap {

constexpr int kWavesPerGroup = 4;

__device__ __forceinline__ unsigned lane_id() { return threadIdx.x & 63u; }
__device__ __forceinline__ unsigned popc64(unsigned long long v) { return (unsigned)__popcll(v); }
// number of set bits of m below this lane
__device__ __forceinline__ unsigned rank_below(unsigned long long m)
{
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

__device__ __forceinline__ int wave_sum(int v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Inclusive prefix sum over the 64 lanes of a wavefront with data-parallel-primitive
// moves (row shifts inside rows of 16 lanes, then the row broadcasts): six additions, no
// trip through the LDS crossbar that a shuffle takes.
__device__ __forceinline__ unsigned wave_inclusive_scan(unsigned v)
{
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
  v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
  return v;
}

// 16-byte store with the nontemporal hint, for output that is written once in whole lines
typedef float stream_f4 __attribute__((ext_vector_type(4)));
// 16 bytes at any element: chunks of a length that is no multiple of four start on no 16-byte boundary
typedef float any_f4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void st_stream4(float4* p, float4 v)
{
  stream_f4 t = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(t, reinterpret_cast<stream_f4*>(p));
}

// The same where the address may be any element's.  The wavefront then writes partial lines at both
// ends, and the hint does not always pay.  Long chunks: below kPackedHintBelow, one tensor over and over (several in turn), us, without ->
// with it 16 MB 7.0 -> 6.7 (7.9 -> 7.2), 20 MB 8.1 -> 7.6 (9.6 -> 8.1), 24 MB 8.2 -> 8.2 (9.1 -> 9.0); from there on it takes from one tensor what it gives
// to several (30 MB 10.0 -> 10.6 (13.9 -> 11.4), 45 MB 12.9 -> 14.3 (19.7 -> 16.5), 60 MB 15.8 -> 18.9 (24.3 -> 22.9)).  Short chunks: packed_hint.
template <bool ALIGNED, bool HINT = false>
__device__ __forceinline__ void st_row4(float* p, float4 v)
{
  if (ALIGNED) {
    st_stream4(reinterpret_cast<float4*>(p), v);
  } else {
    any_f4 t = {v.x, v.y, v.z, v.w};
    if (HINT) __builtin_nontemporal_store(t, reinterpret_cast<any_f4*>(p));
    else *reinterpret_cast<any_f4*>(p) = t;
  }
}

// A tensor's elements as the single-pass kernels read them, each of them once.  ONCE: with the nontemporal hint, which leaves the
// memory-side cache (256 MB) to the values that go out and to what other kernels have there.  Tensors of kReadOnceFrom bytes and more: below
// that the next reader of the tensor itself, the layer that it is the input of, finds it evicted.  Plain loads -> hint, us, tensors in turn:
// compaction and expansion (half zeros) 67 MB 49.4 -> 50.6, 100 MB 70.1 -> 67.0, 201 MB 133.8 -> 119.0, 268 MB 169.5 -> 163.3, odd chunks 89 MB 61.4 -> 57.2,
// 180 MB 125.3 -> 117.4; producer, compaction and a reader behind it 60 MB 60.6 -> 64.6, 89 MB 90.2 -> 90.3, 134 MB 137.6 -> 132.9, 241 MB 247 -> 233.
// One tensor over and over, which the cache holds, loses up to 160 MB, and that is the price: the compaction by itself (in turn) 94 MB
// 37.5 -> 41.0 (43.0 -> 41.1), 120 MB 43.7 -> 47.8 (50.3 -> 47.8), 159 MB 52.9 -> 57.0 (60.6 -> 58.4), 199 MB 68.9 -> 66.5 (70.4 -> 68.8).
constexpr unsigned long long kReadOnceFrom = 80ull << 20;
template <bool ONCE>
__device__ __forceinline__ float ld_once(const float* p)
{
  return ONCE ? __builtin_nontemporal_load(p) : *p;
}

struct Geometry {
  int n;        // elements
  int E;        // elements per chunk
  int W;        // mask words per chunk
  int process;  // chunks in the layout
  int active;   // chunks that hold data
  int backwards;  // compaction order, see zvc_compact_kernel
};

// ------------------------------------------------------------------ count
__global__ __launch_bounds__(64 * kWavesPerGroup) void zvc_count_kernel(const float* __restrict__ in,
                                                                         Geometry g, int* __restrict__ count)
{
  const int c = blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6);
  if (c >= g.active) return;
  const unsigned lane = lane_id();
  const long long b = (long long)g.E * c;
  const int len = (int)min((long long)g.E, (long long)g.n - b);
  const float* p = in + b;
  int acc = 0;
  const any_f4* p4 = reinterpret_cast<const any_f4*>(p);
  const int n4 = len >> 2;
  for (int i = lane; i < n4; i += 64) {
    const any_f4 v = p4[i];
    acc += (v.x != 0.0f) + (v.y != 0.0f) + (v.z != 0.0f) + (v.w != 0.0f);
  }
  for (int i = (n4 << 2) + lane; i < len; i += 64) acc += (p[i] != 0.0f);
  acc = wave_sum(acc);
  if (lane == 0) count[c] = acc;
}

// ------------------------------------------------------------------ scan
// In-place exclusive scan of k ints by one workgroup of 1024 threads; total to
// *nnz.  Each thread owns 16 consecutive entries per 16384-entry tile.
__global__ __launch_bounds__(1024) void zvc_scan_kernel(int* __restrict__ v, int k, int* __restrict__ nnz)
{
  __shared__ int wave_tot[16];
  const unsigned tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
  int carry = 0;
  for (int base = 0; base < k; base += 16384) {
    const int i0 = base + (int)tid * 16;
    int x[16];
    if (i0 + 16 <= k) {
      const int4* p = reinterpret_cast<const int4*>(v + i0);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        int4 q = p[j];
        x[4 * j] = q.x; x[4 * j + 1] = q.y; x[4 * j + 2] = q.z; x[4 * j + 3] = q.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 16; j++) x[j] = i0 + j < k ? v[i0 + j] : 0;
    }
    int tsum = 0;
#pragma unroll
    for (int j = 0; j < 16; j++) tsum += x[j];
    int s = tsum;  // inclusive scan of thread sums inside the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      int t = __shfl_up(s, o, 64);
      if ((int)lane >= o) s += t;
    }
    __syncthreads();  // wave_tot of the previous tile has been consumed
    if (lane == 63) wave_tot[wv] = s;
    __syncthreads();
    int wave_off = 0, total = 0;
#pragma unroll
    for (unsigned w = 0; w < 16; w++) {
      int t = wave_tot[w];
      if (w < wv) wave_off += t;
      total += t;
    }
    int run = carry + wave_off + s - tsum;
    if (i0 + 16 <= k) {
      int4* p = reinterpret_cast<int4*>(v + i0);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        int4 q;
        q.x = run; run += x[4 * j];
        q.y = run; run += x[4 * j + 1];
        q.z = run; run += x[4 * j + 2];
        q.w = run; run += x[4 * j + 3];
        p[j] = q;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 16; j++) {
        if (i0 + j < k) v[i0 + j] = run;
        run += x[j];
      }
    }
    carry += total;
  }
  if (tid == 0) *nnz = carry;
}

// ------------------------------------------------------------------ compact
// Two forms.  zvc_compact_kernel (the one that normally runs) collects a chunk's
// non-zeros in a per-wave LDS ring of two 256-float halves and writes a half out
// whenever it is full: every lane stores 16 bytes of one aligned 1 KB run, with the
// nontemporal hint -- whole lines per store instruction, like the expansion's
// output.  The first and the last 16-byte group of a chunk may be shared with the
// neighbouring chunks and are written element by element.  It needs a 16-byte
// aligned values pointer; zvc_compact_rows_kernel below stores each row's non-zeros
// straight from the lanes that hold them and runs otherwise.
constexpr int kUnroll = 8;  // independent 256-byte rows in flight per wave
constexpr int kHalf = 256;  // floats per half of a wave's ring
// Tensors of at least this many bytes take the staged form.  Compaction alone / count + scan +
// compact, staged against row-wise, in microseconds: 512 MiB 177 / 240 against 166 / 254,
// 256 MiB 72 / 115 against 83 / 121, 128 MiB 33.6 / 57.9 against 32.1 / 56.5, 64 MiB 17.9 / 33.6
// against 17.0 / 32.7 (below the size of the memory-side cache the hint only costs: the
// next reader of the values finds them in HBM instead of the cache).
#ifndef CSWAP_STAGED_COMPACT_BYTES
#define CSWAP_STAGED_COMPACT_BYTES (192ull << 20)
#endif
static std::atomic<unsigned long long> g_staged_compact_bytes{CSWAP_STAGED_COMPACT_BYTES};  // cswap_zvc_set_staged_compact_bytes

__device__ __forceinline__ void lds_order()
{
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

__global__ __launch_bounds__(64 * kWavesPerGroup) void zvc_compact_kernel(
    const float* __restrict__ in, Geometry g, const int* __restrict__ begin, float* __restrict__ values,
    uint32_t* __restrict__ mask)
{
  __shared__ __attribute__((aligned(16))) float ring_all[kWavesPerGroup][2 * kHalf];
  int c = (int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6));
  if (c >= g.process) return;
  if (g.backwards) c = g.process - 1 - c;  // see zvc_compact_rows_kernel
  const unsigned lane = lane_id();
  float* ring = ring_all[threadIdx.x >> 6];
  uint32_t* mrow = mask + (size_t)c * g.W;
  if (c >= g.active) {
    for (int w = lane; w < g.W; w += 64) mrow[w] = 0;
    return;
  }
  const long long b = (long long)g.E * c;
  const int len = (int)min((long long)g.E, (long long)g.n - b);
  const float* p = in + b;
  const unsigned out0 = (unsigned)begin[c];
  unsigned skip = out0 & 3u;     // slots at the front of the next write-out that belong to the chunk before
  unsigned base = out0 - skip;   // index in values of the slot at `head` (a multiple of four)
  unsigned head = 0;             // 0 or kHalf
  unsigned fill = skip;          // slots in use, counted from head
  const int iters = (g.E + 63) >> 6;
  uint32_t held = 0;  // lane l holds mask word (64*(t/32) + l) of the chunk until flushed
  for (int t0 = 0; t0 < iters; t0 += kUnroll) {
    float x[kUnroll];
#pragma unroll
    for (int j = 0; j < kUnroll; j++) {
      const int k = (t0 + j) * 64 + (int)lane;
      x[j] = k < len ? p[k] : 0.0f;  // out-of-range elements read as zero: no bit, no value
    }
#pragma unroll
    for (int j = 0; j < kUnroll; j++) {
      const int t = t0 + j;
      const bool nz = x[j] != 0.0f;
      const unsigned long long m = __ballot(nz);
      if (nz) ring[(head + fill + rank_below(m)) & (2 * kHalf - 1)] = x[j];
      fill += popc64(m);
      if (fill >= (unsigned)kHalf) {  // wave-uniform: the half at head is complete
        lds_order();
        const stream_f4 v = *reinterpret_cast<const stream_f4*>(ring + head + 4 * lane);
        float* dst = values + base + 4 * lane;
        if (skip == 0) {
          __builtin_nontemporal_store(v, reinterpret_cast<stream_f4*>(dst));
        } else {
          const unsigned j0 = 4 * lane;
          if (j0 + 0 >= skip) dst[0] = v.x;
          if (j0 + 1 >= skip) dst[1] = v.y;
          if (j0 + 2 >= skip) dst[2] = v.z;
          if (j0 + 3 >= skip) dst[3] = v.w;
          skip = 0;
        }
        lds_order();
        base += kHalf;
        head ^= (unsigned)kHalf;
        fill -= (unsigned)kHalf;
      }
      if (t >= iters) continue;  // tail of the unrolled group: nothing left in this chunk
      const unsigned slot = (unsigned)(2 * t) & 63u;
      if (lane == slot) held = (uint32_t)m;
      if (lane == slot + 1) held = (uint32_t)(m >> 32);
      if ((t & 31) == 31 || t == iters - 1) {
        const int w = (t >> 5) * 64 + (int)lane;
        const int filled = 2 * (t & 31) + 2;
        if ((int)lane < filled && w < g.W) mrow[w] = held;
        held = 0;
      }
    }
  }
  // what is left in the ring: slots [skip, fill) of the half at head
  lds_order();
  const unsigned j0 = 4 * lane;
  if (j0 < fill) {
    const stream_f4 v = *reinterpret_cast<const stream_f4*>(ring + head + j0);
    float* dst = values + base + j0;
    if (j0 >= skip && j0 + 4 <= fill) {
      *reinterpret_cast<stream_f4*>(dst) = v;
    } else {
      if (j0 + 0 >= skip && j0 + 0 < fill) dst[0] = v.x;
      if (j0 + 1 >= skip && j0 + 1 < fill) dst[1] = v.y;
      if (j0 + 2 >= skip && j0 + 2 < fill) dst[2] = v.z;
      if (j0 + 3 >= skip && j0 + 3 < fill) dst[3] = v.w;
    }
  }
}


__global__ __launch_bounds__(64 * kWavesPerGroup) void zvc_compact_rows_kernel(
    const float* __restrict__ in, Geometry g, const int* __restrict__ begin, float* __restrict__ values,
    uint32_t* __restrict__ mask)
{
  // Tensors larger than the memory-side cache are walked from the last chunk
  // to the first: the counting pass that ran just before went first to last, so
  // the chunks it touched last are the ones still cached (measured: count + scan
  // + compact 6-7 % faster at 256 and 512 MiB; smaller tensors stay cached
  // either way and are walked forwards).
  int c = (int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6));
  if (c >= g.process) return;
  if (g.backwards) c = g.process - 1 - c;
  const unsigned lane = lane_id();
  uint32_t* mrow = mask + (size_t)c * g.W;
  if (c >= g.active) {  // chunk without data: the reference leaves these words untouched; define them
    for (int w = lane; w < g.W; w += 64) mrow[w] = 0;
    return;
  }
  const long long b = (long long)g.E * c;
  const int len = (int)min((long long)g.E, (long long)g.n - b);
  const float* p = in + b;
  unsigned off = (unsigned)begin[c];
  const int iters = (g.E + 63) >> 6;
  uint32_t held = 0;  // lane l holds mask word (64*(t/32) + l) of the chunk until flushed
  for (int t0 = 0; t0 < iters; t0 += kUnroll) {
    float x[kUnroll];
#pragma unroll
    for (int j = 0; j < kUnroll; j++) {
      const int k = (t0 + j) * 64 + (int)lane;
      x[j] = k < len ? p[k] : 0.0f;  // out-of-range elements read as zero: no bit, no value
    }
#pragma unroll
    for (int j = 0; j < kUnroll; j++) {
      const int t = t0 + j;
      const bool nz = x[j] != 0.0f;
      const unsigned long long m = __ballot(nz);
      if (nz) values[off + rank_below(m)] = x[j];
      off += popc64(m);
      if (t >= iters) continue;  // tail of the unrolled group: nothing left in this chunk
      const unsigned slot = (unsigned)(2 * t) & 63u;
      if (lane == slot) held = (uint32_t)m;
      if (lane == slot + 1) held = (uint32_t)(m >> 32);
      if ((t & 31) == 31 || t == iters - 1) {
        const int w = (t >> 5) * 64 + (int)lane;
        const int filled = 2 * (t & 31) + 2;
        if ((int)lane < filled && w < g.W) mrow[w] = held;
        held = 0;
      }
    }
  }
}

// ------------------------------------------------------------------ expand
// One wavefront expands one chunk, one lane four consecutive elements with one 16-byte
// store (with the nontemporal hint: 256 MiB expand in 63 instead of 88 us, 32 MiB in
// 10.9 instead of 12.3 us, a reader of the result right after it no slower;
// the same hint on the loads of the counting and compacting passes gains nothing).
// With a 4-byte store per element the instruction stream bounds it, not the bytes.
// A row is 256 elements = 8 mask words; lane l keeps mask word 64*(row/8) + l of the
// chunk, together with the number of set bits in the words before it inside its row,
// so a lane finds its nibble and the rank of its first element with two cross-lane reads.
// ALIGNED: E % 4 == 0 and a 16-byte aligned destination, so every chunk starts on a
// 16-byte boundary.  Otherwise the same 16-byte stores at any element, without the hint from 28 MiB on:
// 60 MB in chunks of 1838 elements 16.3 us, against 18.6 us with a 4-byte store per element.
constexpr int kRowsInFlight = 8;  // divides the 8 rows one refill covers

template <bool ALIGNED, bool HINT>
__global__ __launch_bounds__(64 * kWavesPerGroup) void zvc_expand4_kernel(
    const float* __restrict__ values, const uint32_t* __restrict__ mask, const int* __restrict__ begin,
    Geometry g, float* __restrict__ out)
{
  const int c = blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6);
  if (c >= g.active) return;
  const unsigned lane = lane_id();
  const long long b = (long long)g.E * c;
  const int len = (int)min((long long)g.E, (long long)g.n - b);
  const uint32_t* mrow = mask + (size_t)c * g.W;
  float* q = out + b;
  unsigned off = (unsigned)begin[c];
  const int rows = (len + 255) >> 8;
  const unsigned sub = lane & 7u;  // my nibble inside the word I read
  const uint32_t below = (1u << (4u * sub)) - 1u;
  uint32_t held = 0, pre = 0;  // pre: low half = set bits before my word in its row, high half = through it
  for (int r0 = 0; r0 < rows; r0 += kRowsInFlight) {
    {  // refill: 64 words = 8 rows
      const int w = (r0 >> 3) * 64 + (int)lane;
      held = w < g.W ? mrow[w] : 0u;
      const int first = w * 32;  // bits past the end of the chunk carry no data
      if (first + 32 > len) held = first >= len ? 0u : (held & ((1u << (len - first)) - 1u));
      const uint32_t cnt = (uint32_t)__popc(held);
      uint32_t s = cnt;
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)s, o, 64);
        if (sub >= (unsigned)o) s += t;
      }
      pre = (s - cnt) | (s << 16);
    }
    float4 x[kRowsInFlight];
#pragma unroll
    for (int j = 0; j < kRowsInFlight; j++) {
      const int src = (j << 3) + (int)(lane >> 3);
      const uint32_t w = (uint32_t)__shfl((int)held, src, 64);
      const uint32_t p = (uint32_t)__shfl((int)pre, src, 64);
      const uint32_t row_total = (uint32_t)__builtin_amdgcn_readlane((int)pre, (j << 3) + 7) >> 16;
      const uint32_t nib = (w >> (4u * sub)) & 15u;
      unsigned rk = off + (p & 0xffffu) + (unsigned)__popc(w & below);
      float4 v;
      v.x = (nib & 1u) ? values[rk] : 0.0f;
      rk += nib & 1u;
      v.y = (nib & 2u) ? values[rk] : 0.0f;
      rk += (nib >> 1) & 1u;
      v.z = (nib & 4u) ? values[rk] : 0.0f;
      rk += (nib >> 2) & 1u;
      v.w = (nib & 8u) ? values[rk] : 0.0f;
      x[j] = v;
      off += row_total;
    }
#pragma unroll
    for (int j = 0; j < kRowsInFlight; j++) {
      const int k = (r0 + j) * 256 + 4 * (int)lane;
      if (k + 4 <= len) {
        st_row4<ALIGNED, HINT>(q + k, x[j]);
      } else {  // ragged end of the last chunk
        if (k < len) q[k] = x[j].x;
        if (k + 1 < len) q[k + 1] = x[j].y;
        if (k + 2 < len) q[k + 2] = x[j].z;
      }
    }
  }
}

// Short chunks.  A wavefront per chunk is bound by the wavefronts there are to start: 16384 of
// them take 8.8 us with three elements each.  Here one wavefront takes as many of them as 64 words hold.  Lane l
// keeps one word together with where its values start and where its elements go, so a word
// finds its chunk's end and offset by itself and the eight rows of a refill are full.
// 16384 chunks, one wavefront per chunk -> this: 7 MB 11.3 -> 5.9 us, 25.7 MB 11.1 -> 8.4,
// 33.6 MB (512 elements per chunk) 11.0 -> 8.7.
// It takes chunks of at most kPackedWords mask words where there are more than kPackedFrom of
// them: three or more to a wavefront.  Two to a wavefront measure the same as one each, and few
// chunks are all in flight at once either way.
constexpr int kPackedWords = 21, kPackedFrom = 2048;
// Whether its stores at any element carry the nontemporal hint.  Compaction and expansion of one tensor over and over
// / of several in turn, us, hint against none.  16384 chunks: 19 MB 23.4 : 24.0 / 22.4 : 24.2 · 24 MB 24.4 : 24.2 / 25.1 : 26.6 ·
// 29 MB 26.4 : 25.0 / 28.9 : 29.2 · 32 MB 26.4 : 25.4 / 29.6 : 30.0 · 42 MB 36.8 : 34.4 / 39.8 : 40.3; 32768 chunks: 24 MB 24.4 : 24.6 /
// 25.4 : 27.1 · 30.5 MB 24.5 : 25.1 / 27.8 : 30.0 · 38 MB 35.9 : 34.1 / 38.7 : 38.5; 65536 chunks: 34 MB 35.2 : 33.5 / 37.9 : 36.5 · 87 MB
// 83.9 : 79.5 / 91.9 : 91.8 · 168 MB 134 : 154 / 150 : 158.  Expansion with a reader right behind it gains from the
// lines that plain stores leave in the cache: 17 MB 25.7 : 26.3 / 25.1 : 24.0, 42 MB 34.0 : 30.1 / 39.1 : 35.8.
constexpr size_t kPackedHintBelow = 28u << 20, kPackedHintFrom = 128u << 20;
static bool packed_hint(size_t bytes) { return bytes < kPackedHintBelow || bytes >= kPackedHintFrom; }
template <bool ALIGNED, bool HINT>
__global__ __launch_bounds__(64 * kWavesPerGroup) void zvc_expand_packed_kernel(
    const float* __restrict__ values, const uint32_t* __restrict__ mask, const int* __restrict__ begin,
    Geometry g, int per, float* __restrict__ out)
{
  const int c0 = (int)(blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6)) * per;
  if (c0 >= g.active) return;
  const unsigned lane = lane_id();
  const unsigned W = (unsigned)g.W;
  const unsigned cl = lane * ((65536u + W - 1) / W) >> 16;  // lane / W
  const unsigned k = lane - cl * W, c = (unsigned)c0 + cl;
  const bool live = (int)cl < per && c < (unsigned)g.active;
  uint32_t held = 0;
  unsigned first = 0, dst = 0;
  int valid = 0;  // elements of my word that exist
  if (live) {
    held = mask[(size_t)c0 * W + lane];
    first = (unsigned)begin[c];
    dst = (unsigned)g.E * c + 32u * k;
    const int len = (int)min((unsigned)g.E, (unsigned)g.n - (unsigned)g.E * c);
    valid = min(max(len - 32 * (int)k, 0), 32);
    if (valid < 32) held &= (1u << valid) - 1u;  // bits past the end of the chunk carry no data
  }
  const unsigned cnt = (unsigned)__popc(held);
  const unsigned before = wave_inclusive_scan(cnt) - cnt;
  const unsigned rank = first + before - (unsigned)__shfl((int)before, (int)(cl * W), 64);
  const unsigned sub = lane & 7u;
  const uint32_t below = (1u << (4u * sub)) - 1u;
  const int rows = ((int)W * per + 7) >> 3;
  float4 x[8];
  unsigned to[8];
  int left[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    if (j >= rows) break;
    const int src = (j << 3) + (int)(lane >> 3);
    const uint32_t w = (uint32_t)__shfl((int)held, src, 64);
    unsigned rk = (unsigned)__shfl((int)rank, src, 64);
    to[j] = (unsigned)__shfl((int)dst, src, 64) + 4u * sub;
    left[j] = __shfl(valid, src, 64) - 4 * (int)sub;
    const uint32_t nib = (w >> (4u * sub)) & 15u;
    rk += (unsigned)__popc(w & below);
    float4 v;
    v.x = (nib & 1u) ? values[rk] : 0.0f;
    rk += nib & 1u;
    v.y = (nib & 2u) ? values[rk] : 0.0f;
    rk += (nib >> 1) & 1u;
    v.z = (nib & 4u) ? values[rk] : 0.0f;
    rk += (nib >> 2) & 1u;
    v.w = (nib & 8u) ? values[rk] : 0.0f;
    x[j] = v;
  }
#pragma unroll
  for (int j = 0; j < 8; j++) {
    if (j >= rows) break;
    float* q = out + to[j];
    if (left[j] >= 4) {
      st_row4<ALIGNED, HINT>(q, x[j]);
    } else {
      if (left[j] > 0) q[0] = x[j].x;
      if (left[j] > 1) q[1] = x[j].y;
      if (left[j] > 2) q[2] = x[j].z;
    }
  }
}

// How many elements of its line lie in front of a chunk that goes to q
__device__ __forceinline__ unsigned line_phase(const float* q) { return (unsigned)(reinterpret_cast<uintptr_t>(q) >> 2) & 31u; }

// The mask words of a chunk moved up by `phase` bits: lane l's word behind the one of the lane before, whose
// last lane's word of the refill before is `carry`.  Returns the shifted word and steps carry.
__device__ __forceinline__ uint32_t shifted_words(uint32_t word, unsigned phase, unsigned lane, uint32_t& carry)
{
  uint32_t before = (uint32_t)__shfl_up((int)word, 1, 64);
  if (lane == 0) before = carry;
  carry = (uint32_t)__builtin_amdgcn_readlane((int)word, 63);
  return (uint32_t)((((uint64_t)word << 32) | before) >> (32u - phase));
}

// Mask word w of a chunk of len elements: bits past its end carry no data
__device__ __forceinline__ uint32_t chunk_word(uint32_t word, int w, unsigned len)
{
  const unsigned first = (unsigned)w * 32u;
  return first + 32 <= len ? word : first >= len ? 0u : word & ((1u << (len - first)) - 1u);
}

// Four elements at place k of rows that start `phase` elements before the chunk and end with it at `end`; q: the start of the rows
__device__ __forceinline__ void store_lane(float* q, unsigned k, unsigned phase, unsigned end, float4 v)
{
  if (k >= phase && k + 4 <= end) {
    st_stream4(reinterpret_cast<float4*>(q + k), v);
  } else {
    if (k >= phase && k < end) q[k] = v.x;
    if (k + 1 >= phase && k + 1 < end) q[k + 1] = v.y;
    if (k + 2 >= phase && k + 2 < end) q[k + 2] = v.z;
    if (k + 3 >= phase && k + 3 < end) q[k + 3] = v.w;
  }
}

// zvc_expand4_kernel once more, for tensors larger than the memory-side cache (the size from which
// the compaction is staged, too): the packed values of four rows (1024 elements) are first
// brought into an LDS region of the wavefront with aligned 16-byte loads -- whole lines per
// instruction -- and picked from there, and the mask words of the next eight rows are asked
// for while the current eight are expanded.  Fetching the values one by one from global
// memory, four partly filled load instructions per row, is 15 % slower where they come from
// HBM (512 MiB: 0.151 against 0.178 ms; staging eight rows at a time 0.167, two 0.163: less
// LDS per wavefront means more wavefronts per compute unit to hide the two loads each group
// waits for, fewer rows per group means more groups) and the same where they come from the
// cache; on small tensors the LDS costs more occupancy than the loads gain, so those keep
// the kernels above.
// The rows start where the line starts that the chunk begins in, whatever the chunk's length: its mask is moved up by as many
// bits (shifted_words), and every store but a chunk's first and last is one of whole lines.  Rows that started with
// the chunk put every line together from two instructions, each part a write of its own to memory.  One tensor over and
// over (several in turn), us: chunks of 3308 elements 217 MB 57.9 -> 52.1 (73.2 -> 70.5), 3675 241 MB 64.6 -> 57.1 (67.0 -> 61.2), 4738 311 MB
// 82.8 -> 74.6 (105.4 -> 99.2), 5025 329 MB 87.0 -> 78.5 (110.2 -> 102.9); 4096 (always a line's start) 268 MB 62.5 and 62.4 (77.0 and 76.8).
// The same in zvc_expand4_kernel gains nothing reliable below that size (60 MB 16.4 -> 16.7 (24.7 -> 25.7), 188 MB 52.7 -> 45.3 (64 -> 65)
// but whole lines 34 MB 8.2 -> 8.7 (9.7 -> 10.4)).
constexpr int kRowsStaged = 4;  // divides kRowsInFlight

__global__ __launch_bounds__(64 * kWavesPerGroup) void zvc_expand4_staged_kernel(
    const float* __restrict__ values, const uint32_t* __restrict__ mask, const int* __restrict__ begin,
    Geometry g, float* __restrict__ out)
{
  __shared__ __attribute__((aligned(16))) float lds_all[kWavesPerGroup][256 * kRowsStaged + 8];
  const int c = blockIdx.x * kWavesPerGroup + (threadIdx.x >> 6);
  if (c >= g.active) return;
  float* lds = lds_all[threadIdx.x >> 6];
  const unsigned lane = lane_id();
  const long long b = (long long)g.E * c;
  const int len = (int)min((long long)g.E, (long long)g.n - b);
  const uint32_t* mrow = mask + (size_t)c * g.W;
  const unsigned phase = line_phase(out + b), end = phase + (unsigned)len;  // below 2^31 + 32
  float* q = out + b - phase;
  unsigned off = (unsigned)begin[c];
  const int rows = (int)((end + 255u) >> 8);
  const unsigned sub = lane & 7u;  // my nibble inside the word I read
  const uint32_t below = (1u << (4u * sub)) - 1u;
  uint32_t held_next = (int)lane < g.W ? mrow[lane] : 0u, carry = 0;
  for (int r0 = 0; r0 < rows; r0 += kRowsInFlight) {
    uint32_t held, pre;  // pre: low half = set bits before my word in its row, high half = through it
    {  // 64 words = 8 rows; the next 64 are asked for now
      const int w = (r0 >> 3) * 64 + (int)lane;
      held = shifted_words(chunk_word(held_next, w, (unsigned)len), phase, lane, carry);
      held_next = w + 64 < g.W ? mrow[w + 64] : 0u;
      const uint32_t cnt = (uint32_t)__popc(held);
      uint32_t s = cnt;
#pragma unroll
      for (int o = 1; o < 8; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)s, o, 64);
        if (sub >= (unsigned)o) s += t;
      }
      pre = (s - cnt) | (s << 16);
    }
#pragma unroll
    for (int h = 0; h < kRowsInFlight; h += kRowsStaged) {
      // where each row's values start inside the group of four, and how many the group has
      unsigned row_start[kRowsStaged], total = 0;
#pragma unroll
      for (int j = 0; j < kRowsStaged; j++) {
        row_start[j] = total;
        total += (uint32_t)__builtin_amdgcn_readlane((int)pre, ((h + j) << 3) + 7) >> 16;
      }
      // values[off, off + total) to lds[shift ...] with loads aligned in global memory (shift = off % 4);
      // the last group of four is fetched element by element so that nothing past the values is read
      const unsigned shift = off & 3u;
      const float* src = values + (off - shift);
      const unsigned until = shift + total;
      lds_order();  // the picks of the previous group are done
      for (unsigned k = 4u * lane; k < until; k += 256u) {
        if (k + 4u <= until) {
          *reinterpret_cast<float4*>(lds + k) = *reinterpret_cast<const float4*>(src + k);
        } else {
          for (unsigned e = k; e < until; e++) lds[e] = src[e];
        }
      }
      lds_order();
      float4 x[kRowsStaged];
#pragma unroll
      for (int j = 0; j < kRowsStaged; j++) {
        const int from = ((h + j) << 3) + (int)(lane >> 3);
        const uint32_t w = (uint32_t)__shfl((int)held, from, 64);
        const uint32_t p = (uint32_t)__shfl((int)pre, from, 64);
        const uint32_t nib = (w >> (4u * sub)) & 15u;
        unsigned rk = shift + row_start[j] + (p & 0xffffu) + (unsigned)__popc(w & below);
        float4 v;
        v.x = (nib & 1u) ? lds[rk] : 0.0f;
        rk += nib & 1u;
        v.y = (nib & 2u) ? lds[rk] : 0.0f;
        rk += (nib >> 1) & 1u;
        v.z = (nib & 4u) ? lds[rk] : 0.0f;
        rk += (nib >> 2) & 1u;
        v.w = (nib & 8u) ? lds[rk] : 0.0f;
        x[j] = v;
      }
      off += total;
#pragma unroll
      for (int j = 0; j < kRowsStaged; j++) {
        store_lane(q, 256u * (unsigned)(r0 + h + j) + 4u * lane, phase, end, x[j]);
      }
    }
  }
}

// ------------------------------------------------------------------ status words
// The single-pass kernel below exchanges counts between workgroups through status words
// in global memory, read and written with relaxed atomics of agent scope (they travel past
// the per-XCD L2 caches, which are not coherent with each other).
// How often a wavefront may ask again for status words it is waiting for, summed over the whole
// kernel (not per word: once the budget is spent every later wait of that wavefront returns at
// once, and a wavefront that sees the failure flag up stops waiting as well, so a run that cannot
// finish -- the grid's workgroups are not all resident at the same time, say -- ends after one
// budget, not after one per tile).  A turn is a sleep and a trip to memory, 1-2 us: the default
// is some tens of milliseconds, two orders of magnitude above what the kernel takes for 1 GiB.
constexpr unsigned kSpinLimit = 1u << 15;
constexpr unsigned kFlagEvery = 32;  // a waiting wavefront looks at the failure flag every so many turns
// cswap_zvc_debug_set_lookback: the bound of the waits, and what is left out
static std::atomic<unsigned> g_spin_limit{kSpinLimit}, g_skip{0};
constexpr unsigned kSkipFirstCount = 1, kSkipFirstMark = 2, kRefuseLastTile = 4;

// Head of a workspace.  ws[0]: kWsMagic once cswap_zvc_workspace_clear has prepared it;
// ws[1]: not 0 after a run whose bounded waits ran out (stays until the next clear, and
// every run that finds it reports failure); ws[3]: number of runs whose scanner has
// finished.  The status words proper start at ws[16].  A run that succeeds leaves them
// zero again: whoever consumes a status word clears it.
//
// Who reports what.  The scanner is ahead of everybody else by two stages, so the
// checks and the result are its business and cost the data workgroups nothing: it looks
// at ws[0] and ws[1] when it starts, and when it has published the last offset it writes
// *nnz (the total, or -1 if the flag is up by then) and only then steps ws[3].  A wavefront
// whose wait ran out raises the flag at once; before it ends it waits (bounded) for ws[3]
// to move and then writes -1 itself, so its -1 lands after whatever the scanner wrote, and
// a scanner that is late finds the flag.  A workspace that is refused (never prepared, or
// left behind by a failed run) makes the scanner write -1 and hand out offsets of zero, so
// that every workgroup runs through without waiting; the data workgroups keep every offset
// they are given inside the tensor, whatever the word held.
constexpr uint32_t kWsMagic = 0x5a564331u;
constexpr int kWsFlag = 1, kWsRuns = 3;

__global__ void zvc_ws_clear_kernel(uint32_t* ws, int words)
{
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < words) ws[i] = i == 0 ? kWsMagic : 0u;
}

__device__ __forceinline__ uint32_t ld_status(const uint32_t* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_status(uint32_t* p, uint32_t v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------------ stream
// count + scan + compact in one pass, as a pipeline that never holds data while it
// waits.  The tensor is cut into tiles of 192 rows (a row = 64 elements = two mask
// words); a grid of G resident workgroups (one per compute unit) walks them round
// robin: workgroup w takes tiles w, w+G, w+2G, ...  Each of its sixteen wavefronts keeps
// 12 rows of five consecutive tiles of the workgroup in registers: while tile i is
// compacted, tiles i+1 and i+2 wait counted, tile i+3 is counted and its count published,
// and the loads of tile i+4 are issued one row at a time between the rows of tile i, so
// that memory sees a steady stream of requests instead of bursts.  One more workgroup,
// the scanner, reads the published counts in tile order and publishes each tile's offset;
// a count is published two stages before its tile's offset is needed, which covers the two
// trips through memory (count to the scanner, offset back) that take about a stage each on
// this part, so a workgroup that asks for the offset of its next tile at the start of a
// stage has it when the stage ends, and nobody waits for anybody's latest step.  The
// compacted values go through an LDS stage per tile and leave as whole 16-byte groups
// aligned in the values array.
//
// Needs: chunk length a multiple of 32 (the mask is then the flat bit mask and a chunk
// starts on a half row), two status words per tile in the workspace, a 16-byte aligned
// values pointer, and all G+1 workgroups resident at once (the waits are bounded).
// Workspace (prepared once by cswap_zvc_workspace_clear; a run leaves it as it found it):
// ws[status_at + t] = kTileReady | count of tile t, ws[offset_at + t] = kTileReady | number of
// non-zeros before tile t (place_status_words says where); the scanner clears a count when it
// has read it, a workgroup the offsets of its tiles when it is through, so no launch is spent on
// clearing.
//
// Measured on one MI355X, half of the elements zero (this kernel / count + scan + compact):
// 512 MiB 0.157 / 0.241 ms, 256 MiB 0.085 / 0.115 ms, 128 MiB 0.051 / 0.057, 64 MiB 0.032 /
// 0.033, 32 MiB 0.022 / 0.020 ms (a tensor of a few rounds of the grid does not fill the
// pipeline).
constexpr int kSWaves = 16, kSRows = 12;
constexpr int kSTileRows = kSWaves * kSRows, kSTileElems = kSTileRows * 64;
constexpr int kSSlots = 5;   // tiles of a workgroup in registers
constexpr int kSAhead = kSSlots - 1;  // the loads run this many tiles ahead of the compaction
constexpr uint32_t kTileReady = 1u << 31;

struct StreamGeometry {
  int n, E, W, process, active;
  int rows;    // rows that exist in the mask layout: process * W / 2 rounded up
  int tiles;   // rows / 192 rounded up
  int mask_words;
  int status_at, offset_at;  // pipeline kernel: where the counts and the offsets of the tiles start in the workspace
};

// The scanner: one wavefront turns counts into offsets, 256 tiles at a time, in tile order.
__device__ void zvc_stream_scanner(uint32_t* ws, const StreamGeometry& g, int step, int* nnz, unsigned spin_limit)
{
  const int tiles = g.tiles;
  if (threadIdx.x >= 64) return;
  const unsigned lane = lane_id();
  uint32_t* status = ws + g.status_at;
  uint32_t* offset = ws + g.offset_at;
  const uint32_t magic = ld_status(&ws[0]), flag0 = ld_status(&ws[kWsFlag]);
  const bool refused = magic != kWsMagic || flag0 != 0u;
  if (refused && lane == 0) *nnz = -1;
  unsigned carry = 0;
  unsigned spins = 0;    // turns of waiting so far, over all steps
  bool flagged = false;  // the failure flag is up: no more waiting, the offsets from here on are garbage below n
  // `step` tiles at a time (at most 256): the tiles that the data workgroups count in the same
  // stage, so that a step never waits for a count that is published a stage later than the rest
  for (int t0 = 0; t0 < tiles; t0 += step) {
    // lane l owns tiles t0 + 4l .. t0 + 4l + 3
    const int stop = t0 + step < tiles ? t0 + step : tiles;
    uint32_t v[4] = {kTileReady, kTileReady, kTileReady, kTileReady};
    while (!refused) {
      bool missing = false;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int t = t0 + 4 * (int)lane + r;
        v[r] = t < stop ? ld_status(&status[t]) : kTileReady;
        missing |= (v[r] & kTileReady) == 0u;
      }
      if (__ballot(missing) == 0ull || flagged) break;
      if (++spins > spin_limit) {  // give up: flag it; the offsets that follow are garbage below n
        if (lane == 0) atomicOr(&ws[kWsFlag], 1u);
        flagged = true;
        break;
      }
      if (spins % kFlagEvery == 0 && ld_status(&ws[kWsFlag]) != 0u) {  // a data workgroup gave up
        flagged = true;
        break;
      }
      __builtin_amdgcn_s_sleep(4);
    }
    // these counts have been read: clear them for the next run
    if (!refused) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int t = t0 + 4 * (int)lane + r;
        if (t < stop) st_status(&status[t], 0u);
      }
    }
    unsigned c[4], mine = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      c[r] = v[r] & ~kTileReady;
      mine += c[r];
    }
    const unsigned incl = wave_inclusive_scan(mine);
    unsigned run = carry + incl - mine;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = t0 + 4 * (int)lane + r;
      if (t < stop) st_status(&offset[t], kTileReady | run);
      run += c[r];
    }
    carry += (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
  }
  if (lane == 0) {
    if (!refused) *nnz = ld_status(&ws[kWsFlag]) != 0u ? -1 : (int)carry;
    __threadfence();
    __hip_atomic_fetch_add(&ws[kWsRuns], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// HINT: the values leave with the nontemporal hint, from 5/3 of the size from which the three kernels' compaction is staged on (320 MiB).  Below,
// whoever reads them next finds them in the memory-side cache.  The compaction by itself is within 3 % either way.  With the expansion behind
// it, with the hint / without, us over one tensor (in turn): 268 MB 170 / 148 (170 / 163), 302 194 / 167 (194 / 195), 346 216 / 186 (217 / 208), 417 262 /
// 222 (262 / 243), 470 286 / 245 (288 / 261), 537 317 / 328 (319 / 323): the line could lie at 480 MiB.
template <bool ONCE, bool HINT>
__global__ __launch_bounds__(64 * kSWaves) void zvc_stream_kernel(
    const float* __restrict__ in, StreamGeometry g, uint32_t* __restrict__ ws, int* __restrict__ begin,
    int* __restrict__ nnz, float* __restrict__ values, uint32_t* __restrict__ mask, unsigned spin_limit,
    unsigned skip)
{
  __shared__ __attribute__((aligned(16))) float stage[kSTileElems + 8];
  __shared__ unsigned s_cnt[kSSlots][kSWaves];
  const int G = (int)gridDim.x - 1, w = (int)blockIdx.x;
  if (w == G) {
    zvc_stream_scanner(ws, g, G, nnz, spin_limit);
    return;
  }
  const unsigned lane = lane_id();
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  uint32_t* status = ws + g.status_at;
  uint32_t* offset = ws + g.offset_at;
  const int iters = (g.tiles - w + G - 1) / G;  // >= 1: the grid has no more data workgroups than there are tiles
  // chunk index = half row / W by multiply and shift (exact while half rows * W < 2^40)
  const unsigned long long w_magic = ((1ull << 40) + (unsigned)g.W - 1) / (unsigned)g.W;

  float x[kSSlots][kSRows];
  unsigned woff[kSSlots];   // non-zeros of the workgroup's tile in the wavefronts before mine
  unsigned total[kSSlots];  // non-zeros of the workgroup's tile
  // The registers of a slot hold what the loads brought, also for rows that do not exist; `have[slot]`
  // says how many elements do, and whoever looks at the values applies it (a select right after the
  // load would be a use of the value and would make the load's latency part of the stage that issued it).
  int have[kSSlots];
  uint32_t ov = 0;          // the offset word of the workgroup's next tile, once it has arrived (every
                            // wavefront reads it for itself: one more branch-free load per stage)

  // Where my rows of tile t start, as a base that is the same for the whole wavefront and
  // the number of elements that exist from there on (0..768).  Rows that do not exist -- past
  // the end of the tensor, tiles past the last one -- are read from the start of the tensor
  // instead and ignored: every wavefront issues the same loads on every path, so that the
  // compiler's count of loads in flight is exact and a wait for one tile does not also wait
  // for the tile whose loads were issued after it.
  auto rows_of = [&](int t, const float*& base, int& exist) {
    const long long first = ((long long)t * kSTileRows + wv * kSRows) * 64;
    long long left = (long long)g.n - first;
    left = left < 0 ? 0 : (left > kSRows * 64 ? kSRows * 64 : left);
    exist = (int)left;
    base = in + (left > 0 ? first : 0);
  };
  auto count_tile = [&](const float (&src)[kSRows], int slot) {
    unsigned cnt = 0;
    if (have[slot] == kSRows * 64) {
#pragma unroll
      for (int j = 0; j < kSRows; j++) cnt += popc64(__ballot(src[j] != 0.0f));
    } else {
#pragma unroll
      for (int j = 0; j < kSRows; j++) cnt += popc64(__ballot(src[j] != 0.0f && (int)lane < have[slot] - 64 * j));
    }
    if (lane == 0) s_cnt[slot][wv] = cnt;
  };
  // after the barrier that follows count_tile: my offset inside the tile and the tile's total; wave 0 publishes it
  auto share_counts = [&](int slot, int t, bool exists) {
    const unsigned mine = lane < (unsigned)kSWaves ? s_cnt[slot][lane] : 0u;
    const unsigned incl = wave_inclusive_scan(mine);
    total[slot] = (unsigned)__builtin_amdgcn_readlane((int)incl, kSWaves - 1);
    woff[slot] = (unsigned)__builtin_amdgcn_readlane((int)(incl - mine), wv);
    if (wv == 0 && exists && lane == 0 && !((skip & kSkipFirstCount) && t == 0)) st_status(&status[t], kTileReady | total[slot]);
  };
  // waits (bounded) until the scanner has published the offset of tile t
  bool gave_up = false;
  uint32_t runs0 = 0;  // ws[kWsRuns] when this wavefront gave up
  unsigned spins = 0;   // turns of waiting so far, over all tiles
  auto await_offset = [&](int t) {
    while ((ov & kTileReady) == 0u && !gave_up) {
      const bool spent = ++spins > spin_limit;
      if (spent || (spins % kFlagEvery == 0 && ld_status(&ws[kWsFlag]) != 0u)) {
        // give up (my budget is spent, or somebody else's was): flag it and go on with what is
        // there, so that every workgroup still reaches its end (offsets are kept inside the
        // tensor, the output is garbage); no later tile waits again
        if (spent && lane == 0) atomicOr(&ws[kWsFlag], 1u);
        runs0 = ld_status(&ws[kWsRuns]);  // the scanner has not finished: it still owes this offset
        gave_up = true;
        break;
      }
      __builtin_amdgcn_s_sleep(2);
      ov = ld_status(&offset[t]);
    }
  };
  // what the write-out of a tile needs, kept from its scatter to the next stage
  unsigned out_prefix = 0, out_total = 0;
  uint32_t out_held = 0;
  int out_begin_idx = -1, out_begin_val = 0;
  long long out_word = 0;
  unsigned prev_prefix = 0, prev_total = 0;
  auto write_out = [&](unsigned tile_prefix, unsigned tile_total) {
    const unsigned shift = tile_prefix & 3u;
    const unsigned end = shift + tile_total;           // stage slots [shift, end) hold data
    float* base = values + (tile_prefix - shift);      // 16-byte aligned
    for (unsigned q = threadIdx.x; 4u * q < end; q += 64 * kSWaves) {
      const stream_f4 v = *reinterpret_cast<const stream_f4*>(stage + 4u * q);
      float* dst = base + 4u * q;
      if (4u * q >= shift && 4u * q + 4u <= end) {
        if (HINT) __builtin_nontemporal_store(v, reinterpret_cast<stream_f4*>(dst));
        else *reinterpret_cast<stream_f4*>(dst) = v;
      } else {  // the first and the last group of a tile are shared with its neighbours
        if (4u * q + 0u >= shift && 4u * q + 0u < end) dst[0] = v.x;
        if (4u * q + 1u >= shift && 4u * q + 1u < end) dst[1] = v.y;
        if (4u * q + 2u >= shift && 4u * q + 2u < end) dst[2] = v.z;
        if (4u * q + 3u >= shift && 4u * q + 3u < end) dst[3] = v.w;
      }
    }
    if (lane < 2u * kSRows && out_word < (long long)g.mask_words) mask[out_word] = out_held;
    if (out_begin_idx >= 0) begin[out_begin_idx] = out_begin_val;
  };

  // ---- fill the pipeline: four tiles on their way, the first three counted and published
  {
    const float* base;
    int exist;
#pragma unroll
    for (int k = 0; k < kSAhead; k++) {
      rows_of(w + k * G, base, exist);
      have[k] = exist;
#pragma unroll
      for (int j = 0; j < kSRows; j++) x[k][j] = ld_once<ONCE>(base + min(lane + 64u * j, (unsigned)max(exist - 1, 0)));
    }
  }
#pragma unroll
  for (int k = 0; k < kSAhead - 1; k++) count_tile(x[k], k);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kSAhead - 1; k++) share_counts(k, w + k * G, k < iters);
  ov = ld_status(&offset[w]);

  for (int i0 = 0; i0 < iters; i0 += kSSlots) {
#pragma unroll
    for (int s = 0; s < kSSlots; s++) {
      const int i = i0 + s;
      if (i >= iters) break;
      const int t = i * G + w;
      // ---- this tile's offset was asked for a stage ago; ask for the next one
      await_offset(t);
      out_total = total[s];
      // whatever the word held (a workspace that was never prepared, a wait that ran out): what this
      // tile writes stays inside the tensor
      // (in a vector register on purpose: as a scalar the compiler fetches the word's value the
      // moment it was asked for, which waits for every load in flight)
      {
        uint32_t given = ov & ~kTileReady;
        asm volatile("" : "+v"(given));
        out_prefix = min(given, (unsigned)g.n - out_total);
      }
      // ---- the previous tile leaves
      if (i > 0) write_out(prev_prefix, prev_total);
      prev_prefix = out_prefix;
      prev_total = out_total;
      __syncthreads();
      ov = ld_status(&offset[i + 1 < iters ? t + G : t]);
      // ---- non-zeros of this tile into the LDS stage, one row at a time, and after each row the
      // load of the same row of the tile four ahead, so that the requests to memory are spread
      // over the whole stage instead of arriving in a burst
      {
        const int r0 = t * kSTileRows + wv * kSRows;  // my first row
        unsigned at = (out_prefix & 3u) + woff[s];    // stage slot of the next non-zero
        const unsigned at0 = at;
        uint32_t held = 0;
        const float* base;
        int exist;
        rows_of(t + kSAhead * G, base, exist);
        have[(s + kSAhead) % kSSlots] = exist;
        const unsigned last = (unsigned)max(exist - 1, 0);
        // the same loop twice: with every row of both tiles there (nearly always), and with the checks
        // for rows that are not; both issue the same twelve loads
        if (have[s] == kSRows * 64 && exist == kSRows * 64) {
#pragma unroll
          for (int j = 0; j < kSRows; j++) {
            const float v = x[s][j];
            const bool nz = v != 0.0f;
            const unsigned long long m = __ballot(nz);
            const unsigned slot =
                __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, at));
            if (nz) stage[slot] = v;
            at += popc64(m);
            if (lane == 2u * j) held = (uint32_t)m;
            if (lane == 2u * j + 1u) held = (uint32_t)(m >> 32);
            x[(s + kSAhead) % kSSlots][j] = ld_once<ONCE>(base + lane + 64u * j);
          }
        } else {
#pragma unroll
          for (int j = 0; j < kSRows; j++) {
            const float v = x[s][j];
            const bool nz = v != 0.0f && (int)lane < have[s] - 64 * j;
            const unsigned long long m = __ballot(nz);
            const unsigned slot =
                __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, at));
            if (nz) stage[slot] = v;
            at += popc64(m);
            if (lane == 2u * j) held = (uint32_t)m;
            if (lane == 2u * j + 1u) held = (uint32_t)(m >> 32);
            x[(s + kSAhead) % kSSlots][j] = ld_once<ONCE>(base + min(lane + 64u * j, last));
          }
        }
        // lane k < 32 holds mask word k of my rows = half row 2*r0 + k; a chunk starts there
        // if the half row index is a multiple of W
        const unsigned in_word = (unsigned)__popc(held);
        const unsigned before = wave_inclusive_scan(in_word) - in_word;
        const unsigned half = 2u * (unsigned)r0 + lane;
        const unsigned c = (unsigned)(((unsigned long long)half * w_magic) >> 40);
        const bool starts = lane < 2u * kSRows && c * (unsigned)g.W == half && (int)c < g.active;
        out_begin_idx = starts ? (int)c : -1;
        out_begin_val = (int)(out_prefix - (out_prefix & 3u) + at0 + before);
        out_held = held;
        out_word = (long long)r0 * 2 + lane;
      }
      // ---- the tile three ahead arrived during the previous stage: count it (in the same
      // straight line as the loads above, so that the wait for it knows which loads are younger)
      count_tile(x[(s + kSAhead - 1) % kSSlots], (s + kSAhead - 1) % kSSlots);
      __syncthreads();
      share_counts((s + kSAhead - 1) % kSSlots, t + (kSAhead - 1) * G, i + kSAhead - 1 < iters);
    }
  }
  write_out(prev_prefix, prev_total);
  // ---- the offsets of my tiles have all been read: clear them for the next run (here and not tile by
  // tile: a store per stage from one wavefront, small as it is, costs the pipeline 4 % at 256 MiB)
  for (int i = (int)threadIdx.x; i < iters; i += 64 * kSWaves) st_status(&offset[i * G + w], 0u);
  // ---- a wavefront whose wait ran out says so after the scanner has written its result
  if (gave_up) {
    for (unsigned spins = 0; ld_status(&ws[kWsRuns]) == runs0 && spins < spin_limit; spins++)
      __builtin_amdgcn_s_sleep(2);
    if (lane == 0) *nnz = -1;
  }
}

// ------------------------------------------------------------------ one kernel for small tensors
// Below 64 MiB the whole tensor fits in the registers of one grid.  It is cut into tiles of consecutive
// elements, a workgroup each: W wavefronts of R rows of 64 elements.  A workgroup loads its tile, counts it,
// publishes the count, reads the counts of the workgroups before it (one trip through memory), takes their sum as
// its offset and stores its non-zeros straight from the registers (at these sizes the values array stays in the
// memory-side cache, where whole-line stores through an LDS stage gain nothing).  The last workgroup, which has read
// every count but its own, writes the total.  Nobody waits for a workgroup with a higher number than its own, so the
// grid makes progress however few of its workgroups the hardware runs at a time (they are started in order).
//
// Rows are rows of the tensor, whatever the chunks are: a row's ballot is 64 bits of the flat bit mask.  Where
// chunks are whole half rows that is the mask layout.  Elsewhere (RAGGED) the tile's bits go to LDS, and a lane makes a
// mask word from the 32 bits at its first element; a word belongs to the tile that has its first element, and the last
// wavefront looks one row further than the tile for the bits of the tile's last words.
//
// Groups of 64 tiles.  A tile's count is read by every later tile of its group; the last tile of a group, when it has
// read them all, publishes the group's total, which every tile of later groups reads.  So an offset takes two trips
// through memory, 1 us each.  Every count has 32 bytes to itself: what workgroups on different dies store into one
// line is stored one after the other, 5 ns and more a store, and with the counts side by side those were the time (33.6 MB in
// 512 tiles 13.6 -> 11.7 us, 60 MB in 919 tiles 22.1 -> 18.8; how often they are read, and that 64 tiles read one, does
// not show).  A tile that has its offset marks its own count, and the counts of a group in which all are marked are
// cleared: by the last tile of the group after next, those of the last three groups by the last tile.  (A counter per group on
// which the tiles add, and whose last adder clears: 33.6 MB 2.4 us more, 60 MB 3.3.)
//
// The totals live in two arrays of 256 words, used in turns: run k publishes into array k & 1 and clears the other one, which
// nobody reads any more; ws[kWsSmallRuns] counts the runs.  The entries that a run has no group for are its
// last workgroup's, so every entry is written and cleared every time.  The arrays have one
// place in every workspace (status words 65024 to 65535, which the pipeline kernel leaves out; the counts are in front of
// them), whatever chunk count a call comes with.  The last workgroup alone steps the run counter, and only when it has
// its offset, so that everybody has taken the same array: had it stepped past a workgroup that is still to
// start, that one would publish into the next run's array.
//
// Failure works as in the pipeline kernel for the shapes that take_single_pass says 2 for (MAY_FAIL): a wait that runs
// out, for a count or before a clearing, raises the sticky flag, the offsets are kept inside the tensor, and the wavefront
// that gave up writes -1 after the last workgroup has stepped the run counter; a workgroup that starts when the flag is up leaves,
// and if it is the last one it writes -1.  The other shapes must not fail.  A workgroup whose wait runs out counts the elements
// before its own by itself; the flag goes up all the same, since counts that nobody clears would be the next run's.  Where the
// workspace is found unusable the last tile of every group compacts the whole group, and the others write their mask words and leave:
// they have published nothing, so that tile is refused as well or its wait for them runs out.  What it costs, until the workspace is
// cleared, is to read what is in front of a group at one workgroup's rate: 60 MB 1.6 ms, 92 MB 2.3, 235 MB 9.6 (20, 34 and 79 us with
// the workspace; with every tile on its own, the square of the size: 7.3, 19 and 86 ms).
//
// Bound by the two trips (some 2 us), by the loads before and the stores behind them, which overlap only as far as tiles
// differ in when they get their offset, and by instruction issue (14 a row).  Against one workgroup of sixteen wavefronts on
// every compute unit, whatever the size, with one trip for 256 counts side by side, us alone / with the expansion behind it: 1 MB 7.5 -> 4.8 /
// 11.9 -> 9.4, 4.2 MB 8.0 -> 5.8 / 13.0 -> 11.1, 16.8 MB 10.2 -> 8.1 / 18.2 -> 16.7, 33.6 MB 13.2 -> 12.4 / 24.4 -> 23.6, 50 MB 21.5 -> 17.3 / 34.8 -> 31.0;
// chunks of any length: 22 MB 13.5 -> 9.7 / 24.1 -> 21.3, 60 MB 24.4 -> 20.5 / 40.4 -> 36.3.
constexpr unsigned kGroupTiles = 64, kGroupsMax = 64;  // a lane for each
constexpr unsigned kCountWords = 8;                    // from one count to the next
constexpr uint32_t kTileThrough = 1u << 30;            // the tile has its offset
constexpr int kWsSmallRuns = 4;
constexpr int kStatusWordsMin = 65536;  // status words of the smallest workspace
constexpr int kSmallTotals = 256;
constexpr int kSmallWords = 2 * kSmallTotals;
constexpr int kSmallCounts = kStatusWordsMin - kSmallWords;  // status word at which the two arrays start
static_assert(kGroupsMax * kGroupTiles * kCountWords <= (unsigned)kSmallCounts, "the counts are in front of the totals");

struct SmallGeometry {
  unsigned n, E, W, process;
  unsigned tiles;
  unsigned spread;            // log2 of the words from one group's total to the next
  unsigned mask_words, tail;  // words of the mask, and the first of those that hold no element
  unsigned clearers;          // workgroups behind the tiles that clear those; 0: the tiles do
  Div31 by_E, by_W;
};

// How many workgroups of `threads` clear the mask words that hold no element, where the tiles would take more than
// eight turns each.  Few elements in many chunks: the one tile of 8192 elements took 8.0 us with 65536 chunks, 15.0 with 262144
// and 43 with 2^20; with these workgroups 5.7, 5.6 and 6.0 (16384 chunks, cleared by the tile, 6.0).
static unsigned small_clearers(const SmallGeometry& g, unsigned threads)
{
  const unsigned words = g.mask_words - g.tail;
  if (words <= 8ull * threads * g.tiles) return 0;
  const unsigned groups = (words + 4 * threads - 1) / (4 * threads);
  return groups < 1024 ? groups : 1024;
}

// old with lane `lane` replaced by the uniform v
__device__ uint32_t write_lane(uint32_t v, uint32_t lane, uint32_t old) __asm("llvm.amdgcn.writelane.i32");

// What a workgroup does without the others' counts: counts the elements before `from` by itself, and compacts from there to
// `end`, all but the mask.  Returns the count of non-zeros before `end`.  `from` is a multiple of 64 * W * 8.
template <int W>
__device__ __forceinline__ unsigned compact_alone(const float* __restrict__ in, unsigned from, unsigned end, Div31 by_E, unsigned E,
                                                  unsigned* s_cnt, int* __restrict__ begin, float* __restrict__ values)
{
  const unsigned lane = lane_id(), wv = threadIdx.x >> 6;
  constexpr unsigned kStep = 4 * 64 * W;
  auto nonzero = [](any_f4 v) { return (unsigned)(v.x != 0.0f) + (v.y != 0.0f) + (v.z != 0.0f) + (v.w != 0.0f); };
  unsigned mine = 0, i = 4 * threadIdx.x;
  for (; i + 7 * kStep < from; i += 8 * kStep) {  // 8 loads on their way: one workgroup's rate is what this takes
    any_f4 v[8];
#pragma unroll
    for (unsigned j = 0; j < 8; j++) v[j] = *reinterpret_cast<const any_f4*>(in + i + j * kStep);
#pragma unroll
    for (unsigned j = 0; j < 8; j++) mine += nonzero(v[j]);
  }
  for (; i < from; i += kStep) mine += nonzero(*reinterpret_cast<const any_f4*>(in + i));
  mine = (unsigned)wave_sum((int)mine);
  if (lane == 0) s_cnt[wv] = mine;
  __syncthreads();
  unsigned offset = 0;
  for (int k = 0; k < W; k++) offset += s_cnt[k];
  for (unsigned base = from; base < end; base += 64 * W * 8) {
    const unsigned e = base + 512 * wv + lane;
    float v[8];
#pragma unroll
    for (unsigned j = 0; j < 8; j++) {
      v[j] = in[min(e + 64 * j, end - 1)];
      if (e + 64 * j >= end) v[j] = 0.0f;
    }
    unsigned cnt = 0;
#pragma unroll
    for (unsigned j = 0; j < 8; j++) cnt += popc64(__ballot(v[j] != 0.0f));
    __syncthreads();  // s_cnt has been read
    if (lane == 0) s_cnt[wv] = cnt;
    __syncthreads();
    unsigned at = offset;
    for (unsigned k = 0; k < (unsigned)W; k++) {
      at += k < wv ? s_cnt[k] : 0u;
      offset += s_cnt[k];
    }
#pragma unroll
    for (unsigned j = 0; j < 8; j++) {
      const unsigned long long m = __ballot(v[j] != 0.0f);
      const unsigned slot = at + rank_below(m), me = e + 64 * j, c = div31(me, by_E);
      if (v[j] != 0.0f) values[slot] = v[j];
      if (me < end && c * E == me) begin[c] = (int)slot;
      at += popc64(m);
    }
  }
  return offset;
}

template <int W, int R, bool RAGGED, bool ONCE, bool MAY_FAIL>
__global__ __launch_bounds__(64 * W, 8) void zvc_small_kernel(
    const float* __restrict__ in, SmallGeometry g, uint32_t* __restrict__ ws, int* __restrict__ begin, int* __restrict__ nnz,
    float* __restrict__ values, uint32_t* __restrict__ mask, unsigned spin_limit, unsigned skip)
{
  constexpr unsigned kElems = 64u * W * R, kHalves = 2u * W * R;
  static_assert(R <= 32, "64 half rows to a wavefront");
  __shared__ uint32_t bits[kHalves + 2];  // the tile's bits, and those of the row behind it
  __shared__ uint16_t pre[kHalves];       // set bits of the wavefront's half rows before this one
  __shared__ unsigned s_cnt[W], s_before[W];  // set bits of each wavefront's rows, and of the rows before them
  __shared__ unsigned s_head[4];              // refused, offset, gave up, failure flag
  const unsigned t = blockIdx.x, lane = lane_id();
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned first = t * kElems, mine = first + 64u * R * wv;  // my tile's first element, my wavefront's
  const unsigned end = min(first + kElems, g.n);

  // is the workspace usable, and which count array is this run's: asked for together with the data
  uint32_t magic = kWsMagic, flag = 0, runs = 0;
  if (wv == 0) {
    magic = ld_status(&ws[0]);
    flag = ld_status(&ws[kWsFlag]);
    runs = ld_status(&ws[kWsSmallRuns]);
  }

  // ---- my rows
  float x[R];
  const int left = mine < g.n ? (int)min(g.n - mine, 64u * R) : 0;  // elements that exist
  if (left == 64 * R) {
#pragma unroll
    for (int j = 0; j < R; j++) x[j] = ld_once<ONCE>(in + (mine + lane + 64u * j));
  } else {  // what does not exist is read from an element that does, and is a zero from here on
    const float* base = in + (left > 0 ? mine : 0u);
    const unsigned last = (unsigned)max(left - 1, 0);
#pragma unroll
    for (int j = 0; j < R; j++) x[j] = base[min(lane + 64u * j, last)];
#pragma unroll
    for (int j = 0; j < R; j++) x[j] = (int)lane < left - 64 * j ? x[j] : 0.0f;
  }
  float behind = 0.0f;
  if (RAGGED && wv == W - 1 && first + kElems + lane < g.n) behind = in[first + kElems + lane];

  if (__builtin_expect(t >= g.tiles, 0)) {  // no tile (and element 0 loaded for it): a share of the mask words that hold no element
    for (unsigned f = g.tail + (t - g.tiles) * 64u * W + threadIdx.x; f < g.mask_words; f += g.clearers * 64u * W) mask[f] = 0;
    return;
  }

  // ---- count: lane l < 2R keeps half row l of my rows
  uint32_t held = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    asm volatile("" : "+v"(x[j]));  // row after row: the ballots are made again below, 32 scalar pairs would not last
    const unsigned long long m = __ballot(x[j] != 0.0f);
    held = write_lane((uint32_t)m, 2 * j, held);
    held = write_lane((uint32_t)(m >> 32), 2 * j + 1, held);
  }
  const unsigned in_half = (unsigned)__popc(held), upto = wave_inclusive_scan(in_half);
  if (lane < 2u * R) {
    if (RAGGED) bits[2 * R * wv + lane] = held;
    pre[2 * R * wv + lane] = (uint16_t)(upto - in_half);
    if (!RAGGED && mine / 32 + lane < g.tail) mask[mine / 32 + lane] = held;
  }
  if (RAGGED && wv == W - 1) {
    const unsigned long long m = __ballot(behind != 0.0f);
    if (lane == 0) {
      bits[kHalves] = (uint32_t)m;
      bits[kHalves + 1] = (uint32_t)(m >> 32);
    }
  }
  if (lane == 63) s_cnt[wv] = upto;
  const bool last_tile = t == g.tiles - 1;
  if (wv == 0 && lane == 0) s_head[0] = (magic != kWsMagic || flag != 0u || ((skip & kRefuseLastTile) && last_tile)) ? 1u : 0u;
  __syncthreads();
  const bool refused = __builtin_amdgcn_readfirstlane((int)s_head[0]) != 0;
  static_assert(kElems % (64 * W * 8) == 0, "compact_alone");
  if (MAY_FAIL && refused) {  // nothing is published, no value written
    // The last tile says so whatever the first one found: the flag may have gone up since.
    if ((t == 0 || last_tile) && threadIdx.x == 0) *nnz = -1;
    return;
  }
  const unsigned wave_cnt = lane < (unsigned)W ? s_cnt[lane] : 0u, wave_upto = wave_inclusive_scan(wave_cnt);
  const unsigned total = (unsigned)__builtin_amdgcn_readlane((int)wave_upto, W - 1);
  const unsigned before_wave = (unsigned)__builtin_amdgcn_readlane((int)(wave_upto - wave_cnt), wv);
  if (wv == 1 && lane < (unsigned)W) s_before[lane] = wave_upto - wave_cnt;

  bool gave_up = false;
  if (wv == 0) {
    // ---- publish, and collect what is before me
    const unsigned group = t / kGroupTiles, place = t % kGroupTiles;
    uint32_t* const counts = ws + 16 + (size_t)group * (kGroupTiles * kCountWords);  // my group's
    uint32_t* const totals = ws + 16 + kSmallCounts + (runs & 1u) * kSmallTotals;
    uint32_t* const others = ws + 16 + kSmallCounts + ((runs & 1u) ^ 1u) * kSmallTotals;
    const bool ends_group = place == kGroupTiles - 1, silent = (skip & kSkipFirstCount) && t == 0;
    unsigned in_group = 0, groups_before = 0, spins = 0;
    bool need_count = lane < place, need_total = lane < group;
    bool counts_open = !refused;
    if (!refused) {
      if (lane == 0 && !silent) st_status(&counts[place * kCountWords], kTileReady | total);
      if (last_tile)  // the other array, and the entries of this one that are no whole group's total
        for (unsigned k = lane; k < (unsigned)kSmallTotals; k += 64) {
          if (k % (1u << g.spread) != 0u || k >> g.spread >= (t + 1) / kGroupTiles) st_status(&totals[k], kTileReady);
          st_status(&others[k], 0u);
        }
    }
    while (!refused) {
      uint32_t count = 0, group_total = 0;
      if (need_count) count = ld_status(&counts[lane * kCountWords]);
      if (need_total) group_total = ld_status(&totals[lane << g.spread]);
      if (count & kTileReady) {
        in_group = count & (kTileThrough - 1u);
        need_count = false;
      }
      if (group_total & kTileReady) {
        groups_before = group_total & ~kTileReady;
        need_total = false;
      }
      if (counts_open && __ballot(need_count) == 0ull) {
        counts_open = false;
        if (ends_group) {
          const unsigned sum = (unsigned)__builtin_amdgcn_readlane((int)wave_inclusive_scan(in_group), 63);
          if (lane == 0) st_status(&totals[group << g.spread], kTileReady | (sum + total));
        }
      }
      if (!counts_open && __ballot(need_total) == 0ull) break;
      spins++;
      if (spins > spin_limit || (spins % kFlagEvery == 0 && ld_status(&ws[kWsFlag]) != 0u)) {
        if (lane == 0) atomicOr(&ws[kWsFlag], 1u);
        gave_up = true;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    if (refused) gave_up = true;
    if (!gave_up && lane == 0 && !silent && !((skip & kSkipFirstMark) && t == 0)) st_status(&counts[place * kCountWords], kTileReady | kTileThrough | total);
    const unsigned before = (unsigned)__builtin_amdgcn_readlane((int)wave_inclusive_scan(in_group + groups_before), 63);
    if (lane == 0) {
      s_head[1] = min(before, g.n - total);  // whatever the words held: what this workgroup writes stays inside the tensor
      s_head[2] = gave_up ? 1u : 0u;
      if (MAY_FAIL && last_tile) s_head[3] = ld_status(&ws[kWsFlag]);
    }
  } else {
    // ---- meanwhile the mask words that start in my tile, and my share of those that hold no element
    if (RAGGED) {
      const unsigned c0 = div31(first, g.by_E), c1 = div31(end, g.by_E);
      const unsigned from = c0 * g.W + (first - c0 * g.E + 31u) / 32u;
      const unsigned stop = end == g.n ? g.tail : c1 * g.W + (end - c1 * g.E + 31u) / 32u;
      for (unsigned f = from + threadIdx.x - 64u; f < stop; f += 64u * (W - 1)) {
        const unsigned c = div31(f, g.by_W), e = c * g.E + 32u * (f - c * g.W), at = e - first;
        const unsigned len = min(c * g.E + g.E, g.n) - e;  // elements of the chunk from here on
        uint32_t w = __builtin_amdgcn_alignbit(bits[at / 32u + 1], bits[at / 32u], at & 31u);
        if (len < 32u) w &= (1u << len) - 1u;
        mask[f] = w;
      }
    }
    if (g.clearers == 0)
      for (unsigned f = g.tail + t * 64u * (W - 1) + threadIdx.x - 64u; f < g.mask_words; f += g.tiles * 64u * (W - 1)) mask[f] = 0;
  }
  __syncthreads();
  // Two ifs, and not one with an else: the compiler lays both sides out one behind the other and would keep the rows in registers
  // through compact_alone, 36 bytes a lane of them in scratch memory (92 MB in chunks of any length 34.2 -> 36.5 us).
  int alone = !MAY_FAIL && __builtin_amdgcn_readfirstlane((int)s_head[2]) != 0;
  if (!alone) {
    const unsigned offset = s_head[1];

    // ---- where the chunks that start in my tile start among the values
    {
      const unsigned c0 = div31(first + g.E - 1u, g.by_E), c1 = div31(end + g.E - 1u, g.by_E);
      for (unsigned c = c0 + threadIdx.x; c < c1; c += 64u * W) {
        const unsigned at = c * g.E - first, h = at / 32u, w = h / (2u * R);
        unsigned o = offset + s_before[w] + pre[h];
        if (RAGGED) o += (unsigned)__popc(bits[h] & ((1u << (at & 31u)) - 1u));
        begin[c] = (int)o;
      }
    }
    // ---- the counts that I clear, if I clear any: asked for now, looked at when my rows are out
    const unsigned group = t / kGroupTiles, groups = (g.tiles + kGroupTiles - 1) / kGroupTiles;
    const bool clears = wv == 0 && !gave_up && (last_tile || ((t + 1) % kGroupTiles == 0 && group >= 2 && group + 1 < groups));
    const unsigned clear_at = (group < 2 ? 0u : group - 2u) * kGroupTiles + lane;
    const unsigned clear_end = last_tile ? g.tiles : (group < 2 ? 0u : group - 1u) * kGroupTiles;
    uint32_t* const clear = ws + 16 + (size_t)clear_at * kCountWords;
    uint32_t through[3] = {kTileThrough, kTileThrough, kTileThrough};
    auto ask = [&] {
#pragma unroll
      for (unsigned k = 0; k < 3; k++)
        if (clear_at + k * kGroupTiles < clear_end) through[k] = ld_status(clear + (size_t)k * kGroupTiles * kCountWords);
    };
    if (clears) ask();
    // ---- my non-zeros, row by row, straight from the lanes that hold them
    float* const out = values + (offset + before_wave);
    unsigned at = 0;
#pragma unroll
    for (int j = 0; j < R; j++) {
      asm volatile("" : "+v"(x[j]));
      const bool nz = x[j] != 0.0f;
      const unsigned long long m = __ballot(nz);
      const unsigned slot = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, at));
      if (nz) *reinterpret_cast<float*>(reinterpret_cast<char*>(out) + (size_t)(4u * slot)) = x[j];
      at += popc64(m);
    }

    if (clears) {
      for (unsigned spins = 0; __ballot((through[0] & through[1] & through[2] & kTileThrough) == 0u) != 0ull; spins++) {
        if (spins > spin_limit || (spins % kFlagEvery == kFlagEvery - 1 && ld_status(&ws[kWsFlag]) != 0u)) {
          if (lane == 0) atomicOr(&ws[kWsFlag], 1u);
          gave_up = true;  // my rows are out, but what is left in the workspace makes this a failed run like any other
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        ask();
      }
#pragma unroll
      for (unsigned k = 0; k < 3; k++)
        if (clear_at + k * kGroupTiles < clear_end) st_status(clear + (size_t)k * kGroupTiles * kCountWords, 0u);
    }

    // ---- the result
    if (last_tile && threadIdx.x == 0) {
      const bool failed = MAY_FAIL && (gave_up || s_head[3] != 0u);
      *nnz = failed ? -1 : (int)(offset + total);
      __threadfence();
      __hip_atomic_fetch_add(&ws[kWsSmallRuns], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (MAY_FAIL && gave_up && !last_tile) {  // (wavefront 0 of another workgroup) after the last workgroup has spoken
      for (unsigned spins = 0; ld_status(&ws[kWsSmallRuns]) == runs && spins < spin_limit; spins++) __builtin_amdgcn_s_sleep(2);
      if (lane == 0) *nnz = -1;
    }
  }
  asm volatile("" : "+v"(alone));
  if (!MAY_FAIL && __builtin_amdgcn_readfirstlane(alone) != 0) {
    const bool ends_group = (t + 1) % kGroupTiles == 0 || last_tile;
    // (a refused tile that does not end its group leaves: the one that does is refused or gives up, too)
    if (refused && !ends_group) return;
    const unsigned from = ends_group ? t / kGroupTiles * kGroupTiles * kElems : first;
    const unsigned count = compact_alone<W>(in, from, end, g.by_E, g.E, s_cnt, begin, values);
    if (last_tile && threadIdx.x == 0) *nnz = (int)count;
  }
}

// ------------------------------------------------------------------ probe
__global__ void zero_u64_kernel(unsigned long long* p) { *p = 0ull; }

__global__ __launch_bounds__(1024) void probe_nnz_kernel(const float* __restrict__ in, size_t n,
                                                        unsigned long long* __restrict__ nnz)
{
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t nthreads = (size_t)gridDim.x * blockDim.x;
  unsigned acc = 0;
  // head up to 16-byte alignment, body in float4, tail
  size_t head = (16 - ((uintptr_t)in & 15u)) & 15u;
  head = min(head >> 2, n);
  for (size_t i = tid; i < head; i += nthreads) acc += (in[i] != 0.0f);
  const float4* p4 = reinterpret_cast<const float4*>(in + head);
  const size_t n4 = (n - head) >> 2;
  size_t i = tid;
  for (; i + 3 * nthreads < n4; i += 4 * nthreads) {  // four independent 16-byte loads in flight per lane
    float4 v0 = p4[i], v1 = p4[i + nthreads], v2 = p4[i + 2 * nthreads], v3 = p4[i + 3 * nthreads];
    acc += (v0.x != 0.0f) + (v0.y != 0.0f) + (v0.z != 0.0f) + (v0.w != 0.0f);
    acc += (v1.x != 0.0f) + (v1.y != 0.0f) + (v1.z != 0.0f) + (v1.w != 0.0f);
    acc += (v2.x != 0.0f) + (v2.y != 0.0f) + (v2.z != 0.0f) + (v2.w != 0.0f);
    acc += (v3.x != 0.0f) + (v3.y != 0.0f) + (v3.z != 0.0f) + (v3.w != 0.0f);
  }
  for (; i < n4; i += nthreads) {
    float4 v = p4[i];
    acc += (v.x != 0.0f) + (v.y != 0.0f) + (v.z != 0.0f) + (v.w != 0.0f);
  }
  for (size_t i = head + (n4 << 2) + tid; i < n; i += nthreads) acc += (in[i] != 0.0f);
  acc = (unsigned)wave_sum((int)acc);
  // one atomic per workgroup, and few workgroups: same-address atomics from
  // different XCDs serialise at the memory side (~12 ns each)
  __shared__ unsigned part[16];
  if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (unsigned w = 0; w < (blockDim.x >> 6); w++) s += part[w];
    if (s) atomicAdd(nnz, s);
  }
}

static int make_geometry(Geometry& g, int n, int process)
{
  if (n <= 0 || process <= 0 || process > (1 << 20)) return CSWAP_E_ARG;
  g.n = n;
  g.process = process;
  g.E = n / process + (n % process != 0);
  g.W = g.E / 32 + (g.E % 32 != 0);
  g.active = n / g.E + (n % g.E != 0);
  g.backwards = n > (48 << 20);  // more than 192 MB of fp32
  return CSWAP_OK;
}

}  // namespace cswap

using namespace cswap;

extern "C" int cswap_zvc_chunk_elems(int n, int process)
{
  Geometry g;
  return make_geometry(g, n, process) ? 0 : g.E;
}
extern "C" int cswap_zvc_chunk_words(int n, int process)
{
  Geometry g;
  return make_geometry(g, n, process) ? 0 : g.W;
}
extern "C" int cswap_zvc_active_chunks(int n, int process)
{
  Geometry g;
  return make_geometry(g, n, process) ? 0 : g.active;
}
extern "C" size_t cswap_zvc_mask_bytes(int n, int process)
{
  Geometry g;
  return make_geometry(g, n, process) ? 0 : (size_t)g.W * (size_t)g.process * sizeof(uint32_t);
}

extern "C" int cswap_zvc_count(const float* d_in, int n, int process, int* d_count, cswap_stream_t stream)
{
  if (!d_in || !d_count) return CSWAP_E_ARG;
  Geometry g;
  int rc = make_geometry(g, n, process);
  if (rc) return rc;
  unsigned grid = (g.active + kWavesPerGroup - 1) / kWavesPerGroup;
  hipLaunchKernelGGL(zvc_count_kernel, dim3(grid), dim3(64 * kWavesPerGroup), 0, (hipStream_t)stream, d_in, g,
                     d_count);
  return check_launch();
}

extern "C" int cswap_zvc_scan(int* d_count, int k, int* d_nnz, cswap_stream_t stream)
{
  if (!d_count || !d_nnz || k <= 0) return CSWAP_E_ARG;
  hipLaunchKernelGGL(zvc_scan_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, d_count, k, d_nnz);
  return check_launch();
}

extern "C" size_t cswap_zvc_set_staged_compact_bytes(size_t bytes)
{
  return (size_t)g_staged_compact_bytes.exchange(bytes);
}

extern "C" int cswap_zvc_compact(const float* d_in, int n, int process, const int* d_begin, float* d_values,
                                 uint32_t* d_mask, cswap_stream_t stream)
{
  if (!d_in || !d_begin || !d_values || !d_mask) return CSWAP_E_ARG;
  Geometry g;
  int rc = make_geometry(g, n, process);
  if (rc) return rc;
  unsigned grid = (g.process + kWavesPerGroup - 1) / kWavesPerGroup;
  if ((reinterpret_cast<uintptr_t>(d_values) & 15u) == 0 && 4ull * (unsigned long long)n >= g_staged_compact_bytes)
    hipLaunchKernelGGL(zvc_compact_kernel, dim3(grid), dim3(64 * kWavesPerGroup), 0, (hipStream_t)stream, d_in,
                       g, d_begin, d_values, d_mask);
  else
    hipLaunchKernelGGL(zvc_compact_rows_kernel, dim3(grid), dim3(64 * kWavesPerGroup), 0, (hipStream_t)stream,
                       d_in, g, d_begin, d_values, d_mask);
  return check_launch();
}

extern "C" int cswap_test_zvc_packed_hint(size_t bytes) { return packed_hint(bytes); }

extern "C" int cswap_zvc_expand(const float* d_values, const uint32_t* d_mask, const int* d_begin, int n,
                                int process, float* d_out, cswap_stream_t stream)
{
  if (!d_values || !d_mask || !d_begin || !d_out) return CSWAP_E_ARG;
  Geometry g;
  int rc = make_geometry(g, n, process);
  if (rc) return rc;
  unsigned grid = (g.active + kWavesPerGroup - 1) / kWavesPerGroup;
  const bool aligned = g.E % 4 == 0 && (reinterpret_cast<uintptr_t>(d_out) & 15u) == 0;
  const bool staged = (reinterpret_cast<uintptr_t>(d_values) & 15u) == 0 &&
                      4ull * (unsigned long long)n >= g_staged_compact_bytes;
#define CSWAP_EXPAND(KERNEL_)                                                                                     \
  hipLaunchKernelGGL(KERNEL_, dim3(grid), dim3(64 * kWavesPerGroup), 0, (hipStream_t)stream, d_values, d_mask, d_begin, \
                     g, d_out)
  if (!staged && g.W <= kPackedWords && g.active > kPackedFrom) {
    const int per = 64 / g.W;
    const unsigned waves = (unsigned)((g.active + per - 1) / per);
    const dim3 packed_grid((waves + kWavesPerGroup - 1) / kWavesPerGroup);
    const auto kernel = aligned                   ? zvc_expand_packed_kernel<true, true>
                        : packed_hint(4 * (size_t)n) ? zvc_expand_packed_kernel<false, true>
                                                     : zvc_expand_packed_kernel<false, false>;
    hipLaunchKernelGGL(kernel, packed_grid, dim3(64 * kWavesPerGroup), 0, (hipStream_t)stream, d_values, d_mask, d_begin, g,
                       per, d_out);
  } else if (staged) CSWAP_EXPAND(zvc_expand4_staged_kernel);
  else if (aligned) CSWAP_EXPAND((zvc_expand4_kernel<true, true>));
  else if (4 * (size_t)n < kPackedHintBelow) CSWAP_EXPAND((zvc_expand4_kernel<false, true>));
  else CSWAP_EXPAND((zvc_expand4_kernel<false, false>));
#undef CSWAP_EXPAND
  return check_launch();
}

extern "C" int cswap_zvc_compress(const float* d_in, int n, int process, int* d_begin, int* d_nnz,
                                  float* d_values, uint32_t* d_mask, cswap_stream_t stream)
{
  if (!d_nnz) return CSWAP_E_ARG;
  int rc = cswap_zvc_count(d_in, n, process, d_begin, stream);
  if (rc) return rc;
  rc = cswap_zvc_scan(d_begin, cswap_zvc_active_chunks(n, process), d_nnz, stream);
  if (rc) return rc;
  return cswap_zvc_compact(d_in, n, process, d_begin, d_values, d_mask, stream);
}

// Chunk count for a tensor of n elements when the caller is free to choose:
// about 1024 elements per chunk, as a power of two between 1024 and 16384.
// Measured on one MI355X (count + scan + compact, then expand, half-zero data):
// 1 and 4 MiB tensors run 40 % / 60 % faster with 1024 chunks than with the
// reference's 16384, 16 MiB is best at 4096, 32 MiB at 8192, 128 MiB and above
// at 16384 and more; below ~1000 elements per chunk the wavefronts are too short
// to cover their start-up, above ~4000 too few are in flight.
extern "C" int cswap_zvc_pick_process(size_t n)
{
  size_t target = n / 1024;
  int p = 1024;
  while (p < 16384 && (size_t)p * 2 <= target) p *= 2;
  return p;
}

// status words of a workspace for `process` chunks
static int status_words(int process) { return process > kStatusWordsMin ? process : kStatusWordsMin; }

extern "C" size_t cswap_zvc_workspace_bytes(int process)
{
  return process > 0 ? ((size_t)status_words(process) + 16) * sizeof(uint32_t) : 0;
}

extern "C" void cswap_zvc_debug_set_lookback(unsigned spin_limit, unsigned skip)
{
  g_spin_limit.store(spin_limit ? spin_limit : kSpinLimit);
  g_skip.store(skip);
}

// Tensors of at least this many bytes take the pipeline kernel in cswap_zvc_compress_fused; smaller ones,
// which do not fill the pipeline (a few rounds of the grid), finish sooner in the one-kernel form that
// holds the whole tensor in registers: 60 MiB 21 us, the pipeline 32.
static std::atomic<unsigned long long> g_single_pass_bytes{64ull << 20};  // cswap_zvc_set_single_pass_bytes

extern "C" size_t cswap_zvc_set_single_pass_bytes(size_t bytes)
{
  return (size_t)g_single_pass_bytes.exchange(bytes);
}

// Data workgroups of the pipeline kernel: one per compute unit but one (the scanner's), no more
// than there are tiles, and no more than the 256 tiles whose counts the scanner's one wavefront
// turns into offsets per step (four per lane) -- on a part with more compute units than that the
// tiles past the 256th of every step would never get an offset.
static int stream_data_groups(int tiles, int compute_units)
{
  int g = compute_units - 1;
  if (g > tiles) g = tiles;
  if (g > 4 * 64) g = 4 * 64;
  return g < 0 ? 0 : g;
}
extern "C" int cswap_test_zvc_stream_groups(int tiles, int compute_units) { return stream_data_groups(tiles, compute_units); }

// Where the pipeline kernel's two arrays of one word per tile go: around the small form's words, which
// hold the counts of its last run.  In front of them; with many tiles behind them, if the workspace is
// one for enough chunks; or one array on either side.  False: no room.
static bool place_status_words(StreamGeometry& sg, int process)
{
  const int behind = status_words(process) - kStatusWordsMin;
  const bool front = 2 * sg.tiles <= kSmallCounts, back = 2 * sg.tiles <= behind;
  sg.status_at = 16 + (!front && back ? kStatusWordsMin : 0);
  sg.offset_at = front || back ? sg.status_at + sg.tiles : 16 + kStatusWordsMin;
  return front || back || (sg.tiles <= kSmallCounts && sg.tiles <= behind);
}

// whether the single pass takes a tensor of this shape; fills its geometry
static bool single_pass_shape(const Geometry& g, int n, int process, StreamGeometry& sg)
{
  sg.n = n; sg.E = g.E; sg.W = g.W; sg.process = process; sg.active = g.active;
  const long long mask_words = (long long)g.W * process;
  sg.mask_words = (int)mask_words;
  sg.rows = (int)((mask_words + 1) / 2);
  sg.tiles = (sg.rows + kSTileRows - 1) / kSTileRows;
  // whole half rows per chunk, two status words per tile in the workspace, a compute unit for
  // every workgroup, and a tensor large enough to fill the pipeline
  return g.E % 32 == 0 && mask_words < (1ll << 31) - 64 && place_status_words(sg, process) &&
         device_compute_units() > 1 && 4ull * (unsigned long long)n >= g_single_pass_bytes;
}

// Whether the one-kernel form for small tensors takes a shape that the pipeline kernel does not: up to kGroupsMax groups of its
// largest tiles, 256 MiB.  Chunks of any length from 64 MiB on, three kernels -> this form, us alone / on tensors in turn / with the
// expansion behind it: 68 MB 35.9 -> 22.5 / 42.2 -> 30.3 / 53.8 -> 40.4, 120 MB 54.2 -> 34.9 / 64.3 -> 44.3 / 87.2 -> 71.6, 241 MB 102.9 -> 85.9 /
// 113 -> 85 / 183 -> 146.  Whole half rows stay with the pipeline there, 241 MB of which take 73.  Fills the geometry but for its tiles.
static bool small_pass_shape(const Geometry& g, int n, SmallGeometry& sg)
{
  const unsigned long long single_from = g_single_pass_bytes.load();
  const long long mask_words = (long long)g.W * g.process;
  if (single_from == 0 || single_from == ~0ull || n > (int)(kGroupsMax * kGroupTiles * 64 * 8 * 32) || mask_words >= (1ll << 31) - 64) return false;
  sg.n = (unsigned)n; sg.E = (unsigned)g.E; sg.W = (unsigned)g.W; sg.process = (unsigned)g.process;
  sg.mask_words = (unsigned)mask_words;
  const unsigned in_last = (unsigned)(n - (long long)(g.active - 1) * g.E);  // elements of the last chunk that has any
  sg.tail = (unsigned)(g.active - 1) * sg.W + (in_last + 31u) / 32u;
  sg.by_E = make_div31(sg.E);
  sg.by_W = make_div31(sg.W);
  return true;
}
// Whether a run of it reports failure where the workspace fails it (zvc_small_kernel: MAY_FAIL): whole half rows per
// chunk, at most 131072 rows of the mask layout on a part of 256 compute units.
static bool small_pass_may_fail(const Geometry& g)
{
  const int cus = device_compute_units();
  const long long rows = ((long long)g.W * g.process + 1) / 2;
  return g.E % 32 == 0 && cus > 0 && rows <= (long long)(cus < 256 ? cus : 256) * 512;
}

extern "C" int cswap_zvc_takes_single_pass(int n, int process)
{
  Geometry g;
  StreamGeometry sg;
  SmallGeometry small;
  if (make_geometry(g, n, process) != CSWAP_OK) return 0;
  if (single_pass_shape(g, n, process, sg)) return 1;
  return small_pass_shape(g, n, small) && small_pass_may_fail(g) ? 2 : 0;
}

bool cswap::zvc_small_any_chunk(int n, int process)
{
  Geometry g;
  SmallGeometry small;
  return make_geometry(g, n, process) == CSWAP_OK && cswap_zvc_takes_single_pass(n, process) == 0 && small_pass_shape(g, n, small);
}

// report: the small form reports failure whatever the shape
static int compress_fused(const float* d_in, int n, int process, void* d_ws, int* d_begin, int* d_nnz, float* d_values,
                          uint32_t* d_mask, bool report, cswap_stream_t stream)
{
  if (!d_in || !d_ws || !d_begin || !d_nnz || !d_values || !d_mask) return CSWAP_E_ARG;
  Geometry g;
  int rc = make_geometry(g, n, process);
  if (rc) return rc;
  uint32_t* ws = (uint32_t*)d_ws;
  const int cus = device_compute_units();
  StreamGeometry sg;
  // what neither one-kernel form takes runs the three kernels (the pipeline needs a 16-byte aligned output, too)
  const bool single_pass = single_pass_shape(g, n, process, sg) && (reinterpret_cast<uintptr_t>(d_values) & 15u) == 0;
  SmallGeometry small;
  if (!single_pass && small_pass_shape(g, n, small)) {
    const bool may_fail = report || (small_pass_may_fail(g) && 4ull * (unsigned long long)n < g_single_pass_bytes.load());
#define CSWAP_SMALL_AS(W, R, RAGGED, ONCE)                                                                          \
  hipLaunchKernelGGL((may_fail ? zvc_small_kernel<W, R, RAGGED, ONCE, true> : zvc_small_kernel<W, R, RAGGED, ONCE, false>), \
                     dim3(small.tiles + small.clearers), dim3(64 * W), 0, (hipStream_t)stream, d_in, small, ws, d_begin, d_nnz, \
                     d_values, d_mask, g_spin_limit.load(), g_skip.load())
#define CSWAP_SMALL(W, R, ONCE)                                 \
  do {                                                          \
    small.tiles = ((unsigned)n + 64 * W * R - 1) / (64 * W * R); \
    small.spread = 2; \
    while (small.spread < 7 && (small.tiles + kGroupTiles - 1) / kGroupTiles <= (unsigned)kSmallTotals >> (small.spread + 1)) small.spread++; \
    small.clearers = small_clearers(small, 64 * W);             \
    if (g.E % 32 != 0) CSWAP_SMALL_AS(W, R, true, ONCE);        \
    else CSWAP_SMALL_AS(W, R, false, ONCE);                     \
  } while (0)
    // The tile by size, us for the compaction alone / with the expansion behind it, tiles of 16 x 8 rows : 16 x 16 : 8 x 32: 1 MB 4.8 : 5.5 :
    // 6.2 / 9.4 : 10.1 : 10.5 · 4.2 MB 5.8 : 6.2 : 6.9 / 11.1 : 11.2 : 11.6 · 8.4 MB 6.3 : 6.6 : 7.2 / 12.9 : 13.4 : 13.8 · 16.8 MB 8.2 : 8.1 : 8.8 /
    // 17.7 : 16.7 : 17.5 · 33.6 MB 16.8 : 12.4 : 12.7 / 26.4 : 23.6 : 24.2 · 50 MB 22.3 : 19.3 : 17.3 / 35.8 : 33.0 : 31.0.  Small tiles while each has a compute
    // unit to itself; then those of sixteen wavefronts while two on every compute unit hold the tensor, then
    // those of eight with twice the rows, four to a compute unit: all of them at once up to 64 MiB.
    if (n <= 256 * 64 * 16 * 8) CSWAP_SMALL(16, 8, false);
    else if (n <= 512 * 64 * 16 * 16) CSWAP_SMALL(16, 16, false);
    else if (4ull * (unsigned long long)n < kReadOnceFrom) CSWAP_SMALL(8, 32, false);
    else CSWAP_SMALL(8, 32, true);
#undef CSWAP_SMALL
#undef CSWAP_SMALL_AS
    return check_launch();
  }
  if (!single_pass) return cswap_zvc_compress(d_in, n, process, d_begin, d_nnz, d_values, d_mask, stream);
  // one workgroup per compute unit, the last of them the scanner
  const int data_groups = stream_data_groups(sg.tiles, cus);
  const unsigned long long bytes = 4ull * (unsigned long long)n;
  const auto kernel = bytes * 3 >= g_staged_compact_bytes.load() * 5 ? zvc_stream_kernel<true, true>
                      : bytes >= kReadOnceFrom                       ? zvc_stream_kernel<true, false>
                                                                     : zvc_stream_kernel<false, false>;
  hipLaunchKernelGGL(kernel, dim3(data_groups + 1), dim3(64 * kSWaves), 0, (hipStream_t)stream, d_in, sg, ws, d_begin, d_nnz,
                     d_values, d_mask, g_spin_limit.load(), g_skip.load());
  return check_launch();
}

extern "C" int cswap_zvc_compress_fused(const float* d_in, int n, int process, void* d_ws, int* d_begin,
                                        int* d_nnz, float* d_values, uint32_t* d_mask, cswap_stream_t stream)
{
  return compress_fused(d_in, n, process, d_ws, d_begin, d_nnz, d_values, d_mask, false, stream);
}

int cswap::zvc_compress_fused_reporting(const float* d_in, int n, int process, void* d_ws, int* d_begin, int* d_nnz,
                                        float* d_values, uint32_t* d_mask, hipStream_t stream)
{
  return compress_fused(d_in, n, process, d_ws, d_begin, d_nnz, d_values, d_mask, true, stream);
}

// ------------------------------------------------------------------ no allocation
// The single-pass compression once more, for callers that cannot bring a workspace
// because they cannot allocate one: the status words live in this array, one copy
// per GPU, held until the process ends.
constexpr int kStaticProcessMax = 65536;
static __device__ __align__(256) uint32_t scratch[kStaticProcessMax + 16] = {kWsMagic};  // prepared from the start

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
uint32_t* g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each GPU, once looked up
}  // namespace

// device address of this GPU's copy of `scratch` (looked up on first use), or an error code
static int static_workspace(uint32_t** ws)
{
  int dev = -1;
  CSWAP_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return CSWAP_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {  // first call on this GPU: where its copy of the array lives
    void* p = nullptr;
    CSWAP_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = static_cast<uint32_t*>(p);
  }
  *ws = g_scratch_ptr[dev];
  return CSWAP_OK;
}

extern "C" int cswap_zvc_compress_fused_static(const float* d_in, int n, int process, int* d_begin, int* d_nnz,
                                               float* d_values, uint32_t* d_mask, cswap_stream_t stream)
{
  if (process > kStaticProcessMax) return CSWAP_E_NOMEM;
  uint32_t* ws = nullptr;
  int rc = static_workspace(&ws);
  if (rc) return rc;
  return cswap_zvc_compress_fused(d_in, n, process, ws, d_begin, d_nnz, d_values, d_mask, stream);
}

extern "C" int cswap_zvc_workspace_clear(void* d_ws, int process, cswap_stream_t stream)
{
  uint32_t* ws = static_cast<uint32_t*>(d_ws);
  if (!ws) {  // the static array of the current GPU
    int rc = static_workspace(&ws);
    if (rc) return rc;
    process = kStaticProcessMax;
  }
  if (process <= 0) return CSWAP_E_ARG;
  const int words = status_words(process) + 16;
  hipLaunchKernelGGL(zvc_ws_clear_kernel, dim3((words + 255) / 256), dim3(256), 0, (hipStream_t)stream, ws, words);
  return check_launch();
}

extern "C" int cswap_probe_nnz(const float* d_in, size_t n, unsigned long long* d_nnz, cswap_stream_t stream)
{
  if (!d_in || !d_nnz || !n) return CSWAP_E_ARG;
  hipLaunchKernelGGL(zero_u64_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, d_nnz);
  size_t want = (n / 16 + 1023) / 1024;  // 4 float4 per thread and pass
  unsigned grid = (unsigned)(want < 1 ? 1 : (want > 512 ? 512 : want));
  hipLaunchKernelGGL(probe_nnz_kernel, dim3(grid), dim3(1024), 0, (hipStream_t)stream, d_in, n, d_nnz);
  return check_launch();
}
