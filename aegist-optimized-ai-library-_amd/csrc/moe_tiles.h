// How an expert's picks are cut into tiles: integer arithmetic of host and device without HIP, so that
// it is checked on the CPU at sizes that no GPU test has the memory for.
#pragma once

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

}  // namespace aegist
