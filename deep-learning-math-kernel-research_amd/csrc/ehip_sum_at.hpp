// Which 16 bytes a lane reads for the in-place sum.  Plain arithmetic, which a host program can walk as well.
#ifndef EHIP_SUM_AT_HPP
#define EHIP_SUM_AT_HPP
#include <stddef.h>
#include <stdint.h>
#if defined(__HIPCC__)
#define EHIP_SUM_FN __host__ __device__ __forceinline__
#else
#define EHIP_SUM_FN inline
#endif

namespace ehip {

// cell: of the lane's pixel in its first channels; at: bytes to those it reads; own: it has a pixel and these channels are real.
// Otherwise the lane reads `readable` instead, 16 bytes of the handle's: the place of channels that only fill up a tile lies behind the
// image's planes, after the last image behind the output, by up to the tile's share of one (64 -> 1696 channels at 75 x 99: 22 planes,
// 2.6 MB).
EHIP_SUM_FN const uint8_t *sum_operand(const uint8_t *cell, size_t at, bool own, const void *readable)
{
  return own ? cell + at : static_cast<const uint8_t *>(readable);
}

}  // namespace ehip
#endif
