// dps_tune.h on the host, for ctypes
#include "dps_tune.h"

extern "C" {
int tune_tiles(int chunk, int own_chunk, int own_tiles, int max_tiles)
{
  return dps::chunk_tiles(chunk, own_chunk, own_tiles, max_tiles);
}
int tune_fits(int tsz, int rs_max, int zc) { return dps::chunk_fits(tsz, 163840, rs_max, zc); }
// out: (chunk, tiles) pairs
int tune_tile_candidates(int now, int own_chunk, int own_tiles, int max_tiles, int tsz, int rs_max, int nz, int* out)
{
  int n = 0;
  for (const auto& c : dps::tile_candidates(now, own_chunk, own_tiles, max_tiles, [&](int zc) {
         return zc <= nz && zc >= std::min(own_chunk, 8) && dps::chunk_fits(tsz, 163840, rs_max, zc);
       })) {
    out[n++] = c.chunk;
    out[n++] = c.tiles;
  }
  return n / 2;
}
int tune_chunk_candidates(int now, int tsz, int rs_max, int nz, int* out)
{
  int n = 0;
  for (int c : dps::chunk_candidates(
           now, [&](int zc) { return zc <= nz && zc >= 8 && dps::chunk_fits(tsz, 163840, rs_max, zc); }))
    out[n++] = c;
  return n;
}
int tune_fastest(const float* ms, int n) { return dps::fastest(std::vector<float>(ms, ms + n)); }
}
