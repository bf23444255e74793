// Which tiles a product of the hybrid route's prefill takes: rules of the host, over sizes alone.
#pragma once

#include <algorithm>

namespace qmk {
namespace hybrid {

constexpr int kMaxTickets = 512;                       // tiles of a product that is cut along K
constexpr int kPartialUnits = 256 * 128 * 128 / 4;     // quads its parts leave: 256 of 128 x 128, or as many values

// bf16 portions are computed in one order, whatever their tiles and length: the columns of a product one after the other (no group of waves takes half of
// them, no workgroup a part), an attention's keys by one group of waves, a head's key channels by four waves.  Some tokens are ill-conditioned (the norm over
// a recurrence's first output leaves little but the sign of a sum that may be close to zero, and some later tokens come close to that), so that a sum taken
// in another order is enough to change what they leave in the states.  Largest relative difference of a state, cache or logits between two orders, 24 sets of weights of
// each of four shapes (width 2048): 2 tokens 0.31, 34 0.065, 100 0.077, 256 0.050, 512 0.038, 1000 0.026, 1531 0.024; 192 prompts of 1025 to 3900 tokens:
// 0.053, and in one cache a value that differs by twice its root mean square.  The median is 0.008 to 0.024 at every length.  (With cuts along K, two groups
// in the attention and eight waves in the scan 43 tokens of the 2b shape took 2.72 ms instead of 2.98, 2 x 2048 of the looped 1b shape 14.4 instead of 15.1.)

// The tiles of a bf16 product.  It takes as many rounds as its tiles fill the chip, 256 at a time, each about `step` us for 2048 columns and `fixed` us besides, `streams` us
// more where the epilogue moves the residual's streams, and `overlapped` us once.  Where two workgroups share a CU (`a_cu`) a round that is not full takes its part of one.
// Fitted to every kind's launches in whole portions of 1 to 4096 tokens of the four shapes (90 lengths, 2011 products; weights and streams from memory), each portion with all its
// products on one kind, so that the kind that comes out cheapest is close to the fastest one, which is more than that its price is its time: it takes 0.8 % longer than the fastest
// one on the average, at most 24 % (with prices fitted to single launches 2.1 and 48 %; of lengths that a first fit had not seen 0.7, and 2.0).  Whole portions, those prices / these: 0.99 (200 tokens of
// the looped shapes) to 1.04 (1750 and 2048 of the others), 1.008 on the average of 43 lengths.  Tiles32 ends at 128 tokens, where its price begins to be off.
// us, M x N x K, the kinds around the line: 43 x 2048 x 6144 with the streams Few32 15.0, Few64 20.9; 43 x 5696 x 2048 Tiles32 10.6, Few64 11.8, Tiles64 13.5; 43 x 12288 x 2048 Tiles64 15.2,
// Tiles32 16.7; 520 x 2048 x 6144 with them Tiles64 41.9, Wide64 47.0; 1024 x 2048 x 6144 with them Wide64 54.6, Turns96 56.5, Tiles64 64.8; 520 x 12288 x 2048 Wide256 31.8, Turns128 36.2;
// 1531 x 2048 x 2048 with them Turns96 33.6, Turns128 36.8, Wide64 42.6; 2048 x 2048 x 2048 with them Turns128 42.8, Tall192 49.1, Wide64 53.2; 1531 x 2048 x 8192 with them Turns96 72.6,
// Turns128 84.6; 3000 x 2048 x 8192 Tall192 97.8, Tall256 111.5; 1531 x 16384 x 2048 Tall256 94.9, Wide256 100.1; 2048 x 16384 x 2048 Turns256 123.2, Tall256 125.4.
// Memory is not priced: it bounds all kinds alike where there are many rows for few tokens.  Two kinds of launches have become a tenth faster since the fit and were not fitted again: Few32 (with waves that
// only load) is priced too dear, products into an attention in all kinds.
struct TileCost {
  int most_tokens, bm, bn, bk, a_cu;
  double step, fixed, overlapped, streams;
};
constexpr int kAnyTokens = 0x7fffffff, kTileKinds = 12;
constexpr TileCost kTileCosts[kTileKinds] = {
    {kAnyTokens, 64, 64, 64, 2, 6.7, 2.0, 3.0, 17.2},          // Tiles64
    {kAnyTokens, 128, 256, 64, 1, 21.3, 14.3, 0.0, 42.9},      // Wide256
    {kAnyTokens, 128, 64, 64, 2, 12.4, 1.8, 4.7, 10.0},        // Wide64
    {kAnyTokens, 96, 128, 64, 1, 12.7, 6.8, 0.0, 9.5},         // Turns96
    {kAnyTokens, 128, 128, 64, 1, 13.1, 7.8, 1.6, 13.8},       // Turns128
    {kAnyTokens, 192, 128, 64, 1, 17.3, 9.9, 0.8, 20.2},       // Tall192
    {kAnyTokens, 256, 128, 64, 1, 20.4, 11.4, 1.8, 26.7},      // Tall256
    {kAnyTokens, 192, 256, 32, 1, 38.7, 12.0, 3.5, 57.7},      // Turns192
    {kAnyTokens, 256, 256, 32, 1, 44.5, 16.0, 0.7, 70.4},      // Turns256
    {128, 64, 32, 64, 2, 4.5, 4.5, 0.5, 2.3},                  // Tiles32
    {256, 64, 16, 128, 2, 4.9, 0.8, 2.6, 2.1},                 // Few64
    {64, 32, 16, 256, 1, 3.2, 2.2, 1.6, 1.4},                  // Few32
};
inline int choose_tiles(int M, int N, int K, int groups, bool streams) {
  int best = 0;
  double least = 0.;
  for (int kind = 0; kind < kTileKinds; ++kind) {
    const TileCost& t = kTileCosts[kind];
    if (M > t.most_tokens || K % t.bk != 0) continue;
    const long long tiles = static_cast<long long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * groups;
    const double rounds = t.a_cu > 1 ? std::max(1., tiles / 256.) : static_cast<double>((tiles + 255) / 256);
    const double us = rounds * (t.step * K / 2048. + t.fixed + (streams ? t.streams : 0.)) + t.overlapped;
    if (kind == 0 || us < least) {
      least = us;
      best = kind;
    }
  }
  return best;
}

// The same for products with an fp32 side, or of columns that are no multiple of 64: tiles of 128 x 128 where there are tokens for them and they
// fill the chip already, else of 64 x 64, with an fp32 side cut along K until they fill it four times over (us, 64 -> 128: 1 x 65536 x 2048
// 94 -> 150, 200 x 12288 x 2048 62 -> 76, 2048 x 16384 x 2048 829 -> 589).
struct RegisterTiles {
  bool large = false;
  int splits = 1;
};
inline RegisterTiles choose_register_tiles(int M, int N, int K, int groups, bool cut) {
  RegisterTiles c;
  const long long large = static_cast<long long>((M + 127) / 128) * ((N + 127) / 128) * groups, small = static_cast<long long>((M + 63) / 64) * ((N + 63) / 64) * groups;
  c.large = M >= 512 && large >= 256;
  if (c.large || !cut) return c;
  while (c.splits < 8 && small * c.splits < 512 && K / c.splits >= 512 && small <= kMaxTickets && small * c.splits * 2 * 64 * 64 / 4 <= kPartialUnits) c.splits *= 2;
  return c;
}

// Products whose tokens' side is in three parts: the kind of tile and the number of parts along K, priced like the bf16 ones, an epilogue of the usual mixture
// within `fixed`, and what a cut costs.  What decides is how full the chip is: a workgroup has it 256 at a time, and larger tiles read LDS less often
// for a product.  us by (tokens x rows, cuts), single launches, x 12288 x 2048, 20 tokens: (32 x 128, 2) 15.8, (32 x 128, 4) 21.5, (64 x 128, 2) 19.8; 100: (64 x 128, 1) 27.2, (32 x 128, 1) 37,
// (64 x 192, 1) 34; 200: (64 x 192, 1) 39.6, (64 x 128, 1) 53, (32 x 128, 1) 54; 200 x 2048 x 6144 with the streams: (32 x 128, 2) 34, (64 x 128, 4) 37, (64 x 192, 4) 48; 200 x
// 2048 x 2048: (32 x 128, 2) 19.2, (32 x 128, 4) 28, (64 x 128, 4) 25; 20 x 2048 x 2048: (32 x 128, 4) 13.1, (32 x 128, 8) 13.3, (64 x 128, 4) 17.2.
struct PartCost {
  int bm, bn;
  double step, fixed;
};
constexpr int kPartKinds = 3;
constexpr PartCost kPartCosts[kPartKinds] = {{32, 128, 15.5, 3.0}, {64, 128, 20.5, 9.0}, {64, 192, 29.0, 13.0}};      // Parts32, Parts64, PartsWide
struct PartTiles {
  int kind = 0, splits = 1;
};
inline PartTiles choose_part_tiles(int M, int N, int K, int groups) {
  PartTiles best;
  double least = 0.;
  for (int kind = 0; kind < kPartKinds; ++kind) {
    const PartCost& t = kPartCosts[kind];
    const long long tiles = static_cast<long long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * groups;
    for (int splits = 1; splits <= 8; splits *= 2) {
      // a ticket a tile, room for all parts, columns for every part
      if (splits > 1 && (tiles > kMaxTickets || tiles * splits * t.bm * t.bn / 4 > kPartialUnits || K / splits < 256)) break;
      const double cut = splits == 1 ? 0. : splits == 2 ? 3.5 : splits == 4 ? 6. : 8.;
      const double us = static_cast<double>((tiles * splits + 255) / 256) * (t.step * K / splits / 2048. + t.fixed) + cut;
      if ((kind == 0 && splits == 1) || us < least) {
        least = us;
        best = PartTiles{kind, splits};
      }
    }
  }
  return best;
}

}  // namespace hybrid
}  // namespace qmk
