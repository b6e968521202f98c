// Host check of the rule that picks the dQ form at head dim 128: longest_q_tile is an upper bound of every query
// tile's blocks (from the union of its queries' intervals, for any run start) over random masks, and
// dq_two_waves on the sizes its comment states. Prints "tiles <n> bad <m>"; non-zero exit on any mismatch.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../sps_amd/csrc/attn_kernels.hpp"

using namespace sps;

int main(int argc, char** argv) {
  const int iters = argc > 1 ? atoi(argv[1]) : 2000;
  std::mt19937 rng(13);
  auto r = [&](int n) { return (int)(rng() % (unsigned)n); };
  long tiles = 0, bad = 0;
  for (int it = 0; it < iters; ++it) {
    MaskSpec m;
    m.family = r(3);
    m.P = m.family == FAMILY_REVERSE_SPS ? 1 : 0;
    m.N = 1 + r(3000);
    if (m.family != FAMILY_FULL) m.N = 2 * ((m.N + 1) / 2);
    m.window = r(6) == 0 ? -1 : r(3) == 0 ? m.N : r(imin(m.N, 700) + 1);
    m.has_pkw = m.family != FAMILY_FULL && r(2) == 0;
    m.pkw = r(6) == 0 ? -1 : r(imin(m.N, 700) + 1);
    m.has_docs = 1;
    const int longest = longest_q_tile(m), run = r(m.N);
    for (int qt = 0; qt < q_tiles(m.N); ++qt) {
      Interval u0, u1;
      q_tile_union(m, qt, [&](int q) { return q >= run ? run : 0; }, u0, u1);
      int first, n0, n1;
      cover_blocks(u0.lo, u0.hi, first, n0);
      cover_blocks(u1.lo, u1.hi, first, n1);
      bad += n0 + n1 > longest;
      ++tiles;
    }
  }
  auto expect = [&](bool want, int family, int N, int window, int pkw, int docs, int64_t n) {
    MaskSpec m{family, family == FAMILY_REVERSE_SPS, N, window, pkw >= 0, pkw, docs};
    bad += dq_two_waves(m, n) != want;
    ++tiles;
  };
  for (int docs = 0; docs < 2; ++docs) {
    expect(false, FAMILY_SPS, 2048, 64, 64, docs, 256);
    expect(true, FAMILY_SPS, 2048, 64, 64, docs, 257);
    expect(docs == 0, FAMILY_SPS, 2048, 128, 512, docs, 311);  // at most 19 + 7 blocks
    expect(true, FAMILY_SPS, 2048, 128, 512, docs, 312);
    expect(docs == 0, FAMILY_FULL, 2048, 0, -1, docs, 512);
    expect(true, FAMILY_FULL, 2048, 0, -1, docs, 513);
    expect(true, FAMILY_SPS, 4096, 4096, -1, docs, 1024);
  }
  printf("tiles %ld bad %ld\n", tiles, bad);
  return bad ? 1 : 0;
}
