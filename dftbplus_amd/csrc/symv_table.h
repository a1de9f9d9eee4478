// Choice of the tile counts of the tridiagonalisation's symmetric product from measured times
// (symv_autotune). Plain host code.
#pragma once

#include <utility>
#include <vector>

namespace dftbhip {

constexpr int kTuneBucket = 256;        // trailing sizes of one choice
constexpr int kTuneFixed = 4;           // fixed tile counts timed
constexpr int kTuneOptions[kTuneFixed] = {2, 4, 8, 16};
constexpr double kTuneGain = 0.02;

using TileTable = std::vector<std::pair<int, int>>;   // (first trailing size, tiles), ascending

// t[o nb + b]: seconds of option o in bucket b, the fixed counts first, then the even share (the
// default). fixed: the fastest fixed count of each bucket, switching away from that of the bucket
// below only for a gain of kTuneGain (buckets of small trailing sizes are launch bound and differ
// by noise only). The table to install is the same with 0, the even share, in the buckets whose
// fixed count does not gain kTuneGain over it: no table makes a bucket slower than the default.
inline void symv_choose(const std::vector<double>& t, int nb, TileTable* fixed,
                        TileTable* install) {
  fixed->clear();
  install->clear();
  int cur = -1;
  for (int b = 0; b < nb; ++b) {
    auto at = [&](int o) { return t[(size_t)o * nb + b]; };
    int best = 0;
    for (int o = 1; o < kTuneFixed; ++o)
      if (at(o) < at(best)) best = o;
    if (cur < 0 || at(best) < (1.0 - kTuneGain) * at(cur)) {
      if (best != cur) fixed->push_back({b * kTuneBucket, kTuneOptions[best]});
      cur = best;
    }
    const int tiles = at(cur) < (1.0 - kTuneGain) * at(kTuneFixed) ? kTuneOptions[cur] : 0;
    if (install->empty() || install->back().second != tiles)
      install->push_back({b * kTuneBucket, tiles});
  }
}

}  // namespace dftbhip
