// Walks every read of the input that k_gemm_u8s8_split makes for a layer, with the kernel's own address arithmetic (CPU tests).
#include "ehip_convs_at.hpp"

// 0: every lane reads the cell it should, or is past the buffer where there is none; else 1 + the first wrong (n, oh, ow, tap, k-step, half)
extern "C" __attribute__((visibility("default"))) long long conv_split_check(int nhwc, int n, int ic2, int ih, int iw, int oh, int ow,
                                                                             int k, int stride, int pad)
{
  using namespace ehip;
  const SplitStrides s = split_strides(nhwc != 0, ic2, ih * iw);
  const unsigned long long bytes = 16ull * n * ic2 * ih * iw;
  long long at = 0;
  for (int i = 0; i < n; ++i)
    for (int y = 0; y < oh; ++y)
      for (int x = 0; x < ow; ++x)
        for (int tap = 0; tap < k * k; ++tap)
          for (int pr = 0; pr < (ic2 + 1) / 2; ++pr)
            for (int lh = 0; lh < 2; ++lh, ++at) {
              const int h = y * stride - pad + tap / k, w = x * stride - pad + tap % k, unit = 2 * pr + lh;
              const unsigned lane = split_lane(split_tap(s, split_image(s, i, lh, ic2, ih * iw), h, w, ih, iw), pr, lh, ic2);
              const unsigned long long byte = (unsigned long long)lane + split_step(s, pr);
              const bool cell = h >= 0 && h < ih && w >= 0 && w < iw && unit < ic2;
              const unsigned long long want =
                  nhwc ? (((unsigned long long)i * ih + h) * iw + w) * ic2 * 16 + unit * 16
                       : ((((unsigned long long)i * ic2 + unit) * ih + h) * iw + w) * 16;
              // (a range check that takes the lane's offset alone, or the sum)
              if (cell ? byte != want || byte + 16 > bytes : lane < bytes) return 1 + at;
            }
  return 0;
}
