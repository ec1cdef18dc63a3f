// The spreading scan (spread.hip) as the host code calls it.
#pragma once
#include <cstddef>

namespace mapx {
namespace spread {

// Device memory a scan of DS0 x DS1 cells works in, beside its output: per 64x64 tile 8192 bytes
// of cell words, 512 of finished bits, a notification word and a queue entry (4 bytes each);
// 64 * 256 bytes of the queues' counters and 64 * 4 of queue entries.
inline size_t scratch_bytes(int DS0, int DS1) {
  const size_t tiles = (size_t)(((long)DS0 + 63) / 64) * (size_t)(((long)DS1 + 63) / 64);
  return tiles * (8192 + 512 + 4 + 4) + 64 * 256 + 64 * 4;
}

// dt: the DataTypeEnum of the raster. Returns the launch count.
int run(void* out, const void* in, const void* dir, void* scratch, int dt, int BS0, int BS1, int NB0, int NB1, int DS0,
        int DS1, void* stream);

}  // namespace spread
}  // namespace mapx
