// dps_tune.h -- z chunks of the spreading: which the batch interface takes,
// which launch each names, and what dps_batch_tune times.  Host only.
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace dps {

// 16-byte staging rows of a record of rs_max words (0: too long)
inline int staged_words(int rs_max)
{
  static const int sizes[] = {8, 10, 12, 16, 20, 24, 32};
  for (int npf : sizes)
    if (rs_max + 7 <= 16 * npf) return npf;
  return 0;
}

// whether a fixed-point cell of zc rows (reals of tsz bytes) and its staged
// records fit in LDS
inline bool chunk_fits(size_t tsz, size_t lds_max, int rs_max, int zc)
{
  const int npf = staged_words(rs_max);
  const size_t bytes = (size_t)3 * zc * (8 * 17 + 1) * tsz + (size_t)256 * npf * tsz + 2064;
  return npf > 0 && bytes <= std::min<size_t>(65536, lds_max);
}

// z tiles per wavefront of k_spread that a chunk names: the solver's own
// chunk stands for its own number of tiles (spread_tiles), any other for the
// tiles it covers
inline int chunk_tiles(int chunk, int own_chunk, int own_tiles, int max_tiles)
{
  return chunk == own_chunk ? own_tiles : std::max(1, std::min(max_tiles, (chunk + 15) / 16));
}

struct SpreadLaunch {
  int chunk, tiles;
};

constexpr int TUNE_CHUNKS[] = {8, 12, 16, 24, 32, 48};

// Launches of k_spread to time: the one in use, then every other number of
// tiles that some chunk the interface takes names.
template <class Fits>
std::vector<SpreadLaunch> tile_candidates(int tiles_now, int own_chunk, int own_tiles, int max_tiles, Fits&& fits)
{
  std::vector<SpreadLaunch> out;
  auto name = [&](int tiles) {
    if (tiles == own_tiles) {
      out.push_back({own_chunk, tiles});
      return;
    }
    for (int c : TUNE_CHUNKS)
      if (c != own_chunk && chunk_tiles(c, own_chunk, own_tiles, max_tiles) == tiles && fits(c)) {
        out.push_back({c, tiles});
        return;
      }
  };
  name(tiles_now);
  for (int t = 1; t <= max_tiles; ++t)
    if (t != tiles_now) name(t);
  return out;
}

// Chunks of the fixed-point cells to time: the one in use, then the others.
template <class Fits>
std::vector<int> chunk_candidates(int chunk_now, Fits&& fits)
{
  std::vector<int> out{chunk_now};
  for (int c : TUNE_CHUNKS)
    if (c != chunk_now && fits(c)) out.push_back(c);
  return out;
}

// The launch in use (ms[0]) stays unless another is faster by more than the
// timings of one differ (2 %).
inline int fastest(const std::vector<float>& ms)
{
  int best = 0;
  for (int i = 1; i < (int)ms.size(); ++i)
    if (ms[i] < (best ? 1.0f : 0.98f) * ms[best]) best = i;
  return best;
}

}  // namespace dps
