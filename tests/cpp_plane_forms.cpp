// Host check of the block codec's forms for planes with many runs (zfp_block.h) against the ones
// that take a step per run.  Exits with 1 and a line of text at the first difference.
#include <stdio.h>
#include <string.h>
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
}  // namespace

int main()
{
  std::mt19937_64 g(20);
  for (unsigned b = 0; b < 256; b++) {  // the table itself: a value bit, and a one behind it if it is one
    unsigned p = 0, e = 0;
    for (unsigned i = 0; i < 8; i++) {
      const unsigned bit = (b >> i) & 1u;
      e |= bit << p++;
      if (bit) e |= 1u << p++;
    }
    if (e != kTable.v[b]) return printf("expand8(%u)\n", b), 1;
  }
  if (!encoder_planes(g) || !encoder_blocks(g)) return 1;
  puts("ok");
  return 0;
}
