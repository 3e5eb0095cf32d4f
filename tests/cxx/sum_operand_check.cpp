// Walks the reads of the in-place sum's operand by waves of `tiles` x 32 channels, blocked output, some of whose channels only fill
// up the last tiles (CPU tests).
#include "ehip_sum_at.hpp"

// 0: every lane reads its own cell of the output, or the handle's bytes; else 1 + the first wrong (n, pixel, wave, tile, half)
extern "C" __attribute__((visibility("default"))) long long sum_operand_check(int n, int oc2, int ohw, int waves, int tiles)
{
  using namespace ehip;
  const size_t bytes = (size_t)16 * n * oc2 * ohw;
  const uint8_t *const out = reinterpret_cast<const uint8_t *>((uintptr_t)1 << 40), *const handle = reinterpret_cast<const uint8_t *>((uintptr_t)1 << 44);
  const size_t tile_stride = (size_t)2 * ohw * 16;
  long long at = 0;
  for (int i = 0; i < n; ++i)
    for (int r = 0; r < ohw; ++r)
      for (int w = 0; w < waves; ++w)
        for (int mt = 0; mt < tiles; ++mt)
          for (int lh = 0; lh < 2; ++lh, ++at) {
            const int block = w * tiles * 2 + lh, mine = block + 2 * mt;
            const uint8_t *cell = out + (((size_t)i * oc2 + block) * ohw + r) * 16;
            const uint8_t *p = sum_operand(cell, mt * tile_stride, mine < oc2, handle);
            const bool inside = p >= out && p + 16 <= out + bytes;
            if (mine < oc2 ? !inside || p != out + (((size_t)i * oc2 + mine) * ohw + r) * 16 : p != handle) return 1 + at;
          }
  return 0;
}
