// Host check of the block codec's forms for planes with many runs (zfp_block.h) against the ones
// that take a step per run.  Exits with 1 and a line of text at the first difference.
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <random>
#include <vector>
#include "../cswap_amd/csrc/zfp_block.h"

namespace {
using namespace cswap;

constexpr unsigned kBefore = 8, kAfter = 8;  // dwords in front of and behind a block's slot that are watched

struct Bits {
  std::vector<uint32_t> dw;
  explicit Bits(unsigned maxbits) : dw(kBefore + maxbits / 32 + 4 + kAfter, 0u) {}
  void or32(unsigned d, uint32_t v) { dw.at(d / 4) |= v; }  // .at: no access outside, not even with zeros
};
constexpr ExpandTable kTable = make_expand_table();
struct TableBits : Bits {
  static constexpr bool kExpands = true;
  using Bits::Bits;
  uint32_t expanded(uint32_t word, int k) const { return kTable.v[(word >> (8 * k)) & 0xffu]; }
};

constexpr CollapseTable kCollapse = make_collapse_table();
struct ReadBits {
  std::vector<uint32_t> dw;
  uint32_t ld32(unsigned d) const { return dw.at(d / 4); }
};
struct TableReadBits : ReadBits {
  static constexpr bool kCollapses = true;
  uint32_t collapsed(uint32_t word, int k) const { return kCollapse.v[(word >> (8 * k)) & 0xffu]; }
};

// the block's bits and the 128 behind them, and that nothing else was written
template <class A, class B>
bool same(const A& a, const B& b, unsigned maxbits, const char* what)
{
  for (unsigned d = 0; d < a.dw.size(); d++) {
    const bool slack = d >= kBefore + maxbits / 32;
    if (a.dw[d] != b.dw[d] && !slack) return printf("%s: dword %u differs: %08x %08x\n", what, d, a.dw[d], b.dw[d]), false;
    if ((d < kBefore || d >= kBefore + maxbits / 32 + 4) && b.dw[d])
      return printf("%s: wrote dword %u of a slot of %u bits\n", what, d, maxbits), false;
  }
  return true;
}

uint64_t sparse(std::mt19937_64& g, int kind)
{
  uint64_t x = g();
  for (int i = 0; i < kind; i++) x &= g();
  if (kind == 7) x = ~(uint64_t)0;
  if (kind == 8) x = (uint64_t)0xffffffffu << (g() % 33);
  if (kind == 9) x = (uint64_t)1 << (g() % 64);
  return x;
}

bool encoder_planes(std::mt19937_64& g)
{
  for (int it = 0; it < 300000; it++) {
    const unsigned maxbits = 64 * (1 + g() % 5), n = g() % 65;
    Bits a(maxbits);
    TableBits b(maxbits);
    BlockEncoder<Bits, false> ea(a, 32 * kBefore, maxbits);
    TableEncoder<TableBits> eb(b, 32 * kBefore, maxbits);
    ea.n = eb.n = n;
    ea.pos = eb.pos = 32 * kBefore + g() % maxbits;
    for (int k = 0; k < 3; k++) {
      const uint64_t x = sparse(g, (int)(g() % 10));
      ea.plane(x);
      if (k == 1 && eb.active()) eb.plane_with_runs(x, eb.n < 64 ? x >> eb.n : 0);  // (also where there are none)
      else eb.plane(x);
      if (ea.active() != eb.active() || (ea.active() && (ea.pos != eb.pos || ea.n != eb.n)))
        return printf("plane %016llx: at %u, %u known; by table at %u, %u known\n", (unsigned long long)x, ea.pos, ea.n, eb.pos,
                      eb.n),
               false;
    }
    if (!same(a, b, maxbits, "encoder plane")) return false;
  }
  return true;
}

bool encoder_blocks(std::mt19937_64& g)
{
  std::normal_distribution<float> normal(0.0f, 1.0f);
  for (int it = 0; it < 20000; it++) {
    const unsigned maxbits = 64 * (1 + g() % 64);
    float f[64];
    const int kind = it % 4;
    for (int i = 0; i < 64; i++)
      f[i] = kind == 0 ? normal(g) : kind == 1 ? std::max(normal(g), 0.0f) : kind == 2 ? ldexpf(normal(g), (int)(g() % 40) - 20)
                                                                                      : 1.0f + 0.001f * (float)i;
    Bits a(maxbits);
    TableBits b(maxbits);
    encode_block<false>(f, 32 * kBefore, maxbits, a);
    encode_block<false>(f, 32 * kBefore, maxbits, b);
    if (!same(a, b, maxbits, "encoder block")) return false;
  }
  return true;
}
// Any bits are a plane to the decoder: words of random bits, sparse, dense or from the encoder, with
// whatever follows the fence, read by both decoders from every position, up to the end of the budget.
bool decoder_planes(std::mt19937_64& g)
{
  for (int it = 0; it < 300000; it++) {
    const unsigned words = 1 + g() % 5, maxbits = 64 * words;
    ReadBits a;
    TableReadBits b;
    const int kind = (int)(g() % 10);
    Bits coded(maxbits);
    if (it % 2) {
      BlockEncoder<Bits, false> e(coded, 32 * kBefore, maxbits);
      while (e.active()) e.plane(sparse(g, (int)(g() % 10)));
    }
    for (unsigned d = 0; d < 2 * words; d += 2) {
      const uint64_t r = it % 2 ? ((uint64_t)coded.dw[kBefore + d + 1] << 32) | coded.dw[kBefore + d] : sparse(g, kind);
      a.dw.push_back((uint32_t)r);
      a.dw.push_back((uint32_t)(r >> 32));
    }
    b.dw = a.dw;
    a.dw.insert(a.dw.end(), {~0u, ~0u});
    b.dw.insert(b.dw.end(), {1u, 0u});
    for (int d = 0; d < 4; d++) {  // the decoders read up to 128 bits past the fence
      a.dw.push_back((uint32_t)g());
      b.dw.push_back((uint32_t)g());
    }
    BlockDecoder<ReadBits, 64, true> da(a, 0, maxbits);
    TableDecoder<TableReadBits> db(b, 0, maxbits);
    if (it % 2 == 0) {
      da.nrem = db.nrem = 63 - (int)(g() % 65);
      da.pos = db.pos = g() % maxbits;
    }
    for (int k = 0; k < 64 && da.active(); k++) {
      const unsigned pos = da.pos;
      const int nrem = da.nrem;
      const uint64_t xa = da.plane(), xb = k % 3 == 2 ? db.low_plane() : db.plane();
      if (xa != xb || da.active() != db.active() || (da.active() && (da.pos != db.pos || da.nrem != db.nrem)))
        return printf("decoder plane at %u of %u, %d to find: %016llx to %u, %d; by table %016llx to %u, %d\n", pos, maxbits,
                      nrem, (unsigned long long)xa, da.pos, da.nrem, (unsigned long long)xb, db.pos, db.nrem),
               false;
    }
    if (!db.active() && db.plane() != 0) return puts("a plane past the budget is not empty"), false;
  }
  return true;
}

bool decoder_blocks(std::mt19937_64& g)
{
  std::normal_distribution<float> normal(0.0f, 1.0f);
  for (int it = 0; it < 20000; it++) {
    const unsigned words = 1 + g() % 64, maxbits = 64 * words;
    float f[64], fa[64], fb[64];
    for (int i = 0; i < 64; i++) f[i] = it % 3 == 0 ? normal(g) : it % 3 == 1 ? std::max(normal(g), 0.0f) : 1.0f + 0.001f * (float)i;
    Bits coded(maxbits);
    encode_block<false>(f, 32 * kBefore, maxbits, coded);
    ReadBits a;
    TableReadBits b;
    a.dw.assign(coded.dw.begin() + kBefore, coded.dw.begin() + kBefore + 2 * words);
    b.dw = a.dw;
    a.dw.insert(a.dw.end(), {~0u, ~0u, 0x12345678u, 0x9abcdef0u, 0x12345678u, 0x9abcdef0u});
    b.dw.insert(b.dw.end(), {1u, 0u, 0x12345678u, 0x9abcdef0u, 0x12345678u, 0x9abcdef0u});
    decode_block<true>(a, 0, maxbits, fa);
    decode_block<true>(b, 0, maxbits, fb);
    if (memcmp(fa, fb, sizeof fa)) return printf("decoder block of %u bits\n", maxbits), false;
  }
  return true;
}
}  // namespace

int main()
{
  std::mt19937_64 g(20);
  for (unsigned b = 0; b < 256; b++) {  // the way back, from what the encoder's table makes of 4 coefficients, cut off at 8 bits
    for (unsigned i = 0; i < 16; i++)
      if ((kTable.v[i] & 0xffu) == b && kCollapse.v[b] != i) return printf("collapse8(%u)\n", b), 1;
  }
  for (unsigned b = 0; b < 256; b++) {  // the table itself: a value bit, and a one behind it if it is one
    unsigned p = 0, e = 0;
    for (unsigned i = 0; i < 8; i++) {
      const unsigned bit = (b >> i) & 1u;
      e |= bit << p++;
      if (bit) e |= 1u << p++;
    }
    if (e != kTable.v[b]) return printf("expand8(%u)\n", b), 1;
  }
  if (!encoder_planes(g) || !encoder_blocks(g) || !decoder_planes(g) || !decoder_blocks(g)) return 1;
  puts("ok");
  return 0;
}
