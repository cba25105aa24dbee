// How the picks of a prefill batch are cut into tiles: arithmetic of host and device without HIP, so that
// it is checked on the CPU, also at sizes that no GPU test has the memory for.
#pragma once

#include <algorithm>
#include <cmath>

#ifdef __HIPCC__
#define AEG_HD __host__ __device__
#else
#define AEG_HD
#endif

namespace aegist {

// First pick of tile j of the n balanced tiles of c picks (j = n: c); the first c % n tiles have one pick
// more than the others. No product of two counts: c j / n leaves 32 bits from 370704 picks of one expert
// in tiles of 64.
AEG_HD constexpr int tile_begin(int c, int j, int n) { return c / n * j + (j < c % n ? j : c % n); }

constexpr int kMoeRows = 512;  // code rows of a prefill tile's workgroup
constexpr int kMoeCus = 256;   // such workgroups on the chip at once (one per CU)

// Picks per prefill tile of moe.hip for T tokens with K of E experts each (D x I): 16, 32, 48 or 64, or 0
// for the tiles of at most 32 picks on 64-row workgroups. A prefill tile reads and converts its codes
// once for all its picks, but its workgroups are large and walk all of a row's groups one after the other
// (60 to 80 us a round of both projections at D = 2048): they pay where they fill the chip. What fills it is
// counted for experts that are drawn alike (the host does not know the picks; where 128 tokens all pick the same 8 of
// 256 experts of 2048 x 512, the smaller tiles would take 69 us instead of 105). Measured (us, 64-row workgroups, then prefill tiles of 64; D x I):
//   few experts, 2048 x 512, 9 tokens with 2 of 8 39.7, 68.7; other widths at decode batches, 2048 x 768, 1
//   token with 8 of 256 34.7, 70.0; 16 tokens 129, 148; 1536 x 768, 4 tokens with 2 of 8 34.4, 66.1
//   2048 x 512, 128 tokens with 8 of 256 231, 182, 2048 tokens 698, 418; 1024 x 256, 64 tokens 88.3, 66.9
// Over 1428 batches of 1 to 2048 tokens, 4 to 512 experts, D 512 to 2048, I 128 to 1536 the rule's choice is
// 1.1% above the fastest of the five on average, and 2 of them more than 3% above the 128-row workgroups before (1.05
// at most). Past them it is up to 1.23 of those: experts twice and more as wide as a model of 512 or 768, and
// sizes that leave a seventh and more of 512 rows idle, at few experts of 64 and more picks.
inline int moe_tile_picks(int T, int K, int E, int D, int I) {
    const double N = (double)T * K, mean = N / E, share = K < E ? (double)K / E : 1.0;
    const double touched = E * (1 - std::pow(1 - share, T));
    const double gu = std::ceil(2.0 * I / kMoeRows), dn = std::ceil((double)D / kMoeRows);  // workgroups of a tile
    if (mean < 16) {
        // one tile per expert, nearly: prefill tiles where the last round of workgroups is nearly full and
        // little of it is padding (full rounds 0.72 to 0.8 of the other's time; an expert of few
        // blocks needs less, its 64-row workgroups reading the shortest runs), in the projection whose
        // rows are the longer walk
        const double blocks = I > D ? dn : gu, pad = (I > D ? D : 2.0 * I) / (kMoeRows * blocks);
        const double rounds = touched * blocks / kMoeCus;
        double least = std::min(0.9, 0.5 + 0.1 * blocks);
        // experts with more than 16 picks: from one on, the 64-row workgroups run as two launches, one per
        // tile size, each of which takes as long as one (2 of 8 experts: 32 tokens 40.7 us, 64 79.5)
        double p = std::pow(1 - share, T), upto16 = p;
        for (int k = 0; k < 16 && k < T; k++) upto16 += p *= (double)(T - k) / (k + 1) * share / (1 - share);
        if (share < 1 && E * (1 - upto16) >= 0.3) least *= 0.6;
        return rounds / std::ceil(rounds) * pad * pad >= least ? 64 : 0;
    }
    // tiles of at most `cap` picks: the last of an expert's is half full on average
    auto tiles = [&](int cap) { return std::max(touched, N / cap + touched / 2); };
    auto rounds = [](double workgroups) { return std::ceil(workgroups / kMoeCus); };
    // all experts at 17 to 32 picks: one launch of the 64-row workgroups again (2 of 16 experts, 192 tokens,
    // 2048 x 768: 66 us, prefill tiles 86)
    if (mean >= 20 && mean <= 28 && tiles(64) * gu < kMoeCus / 2) return 0;
    // the smallest tiles that the chip takes in one round (2048 x 1408, 2 of 8 experts, 512 tokens: 32 picks
    // 111 us, 64 143) or, where every expert has more than one tile of 64 anyway, in no more rounds than
    // those (their last one is nearly empty: 896 x 896, 2 of 8 experts, 2048 tokens, 272 workgroups 131 us,
    // 48 picks 113); past that the least code traffic
    for (int cap = 16; cap < 64; cap += 16)
        if (rounds(tiles(cap) * gu) <= 1) return cap;
    if (mean > 64)
        for (int cap = 16; cap < 64; cap += 16)
            if (rounds(tiles(cap) * gu) <= rounds(tiles(64) * gu) && rounds(tiles(cap) * dn) <= rounds(tiles(64) * dn))
                return cap;
    return 64;
}

}  // namespace aegist
