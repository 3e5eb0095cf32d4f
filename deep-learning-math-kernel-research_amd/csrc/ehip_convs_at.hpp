// Where the lanes of k_gemm_u8s8_split (ehip_convs.hip) read the input.  Plain arithmetic, which a host program can walk as well:
// the range check of the kernel's loads can be counted on for the lane's offset alone, not for what is added to it for all lanes, so
// that offset has to say by itself whether there is a cell to read.
#ifndef EHIP_CONVS_AT_HPP
#define EHIP_CONVS_AT_HPP
#if defined(__HIPCC__)
#define EHIP_SPLIT_FN __host__ __device__ __forceinline__
#else
#define EHIP_SPLIT_FN inline
#endif

namespace ehip {

constexpr unsigned kSplitPastEnd = 0x80000000u;   // past every buffer (at most 2^31 - 1 bytes): the load gives zeros

// bytes between neighbouring pixels (px) and units of 16 channels (unit)
struct SplitStrides {
  unsigned px, unit;
};
EHIP_SPLIT_FN SplitStrides split_strides(bool nhwc, int ic2, int ihw)
{
  return SplitStrides{nhwc ? (unsigned)ic2 * 16u : 16u, nhwc ? 16u : (unsigned)ihw * 16u};
}
// the lower half of a wave (lh = 0) takes the even units of a k-step, the upper one the odd ones
EHIP_SPLIT_FN unsigned split_image(const SplitStrides &s, int n, int lh, int ic2, int ihw)
{
  return (unsigned)n * ic2 * ihw * 16u + lh * s.unit;
}
// of one tap; outside the image: past the buffer, code 0
EHIP_SPLIT_FN unsigned split_tap(const SplitStrides &s, unsigned image, int h, int w, int ih, int iw)
{
  const bool inside = (unsigned)h < (unsigned)ih && (unsigned)w < (unsigned)iw;
  return inside ? image + (unsigned)(h * iw + w) * s.px : kSplitPastEnd;
}
// the lane's offset in k-step `pr` (units 2 pr, 2 pr + 1; an odd count has no second unit in the last one) and what is added to
// it for all lanes
EHIP_SPLIT_FN unsigned split_lane(unsigned tap, int pr, int lh, int ic2)
{
  return 2 * pr + lh < ic2 ? tap : kSplitPastEnd;
}
EHIP_SPLIT_FN unsigned split_step(const SplitStrides &s, int pr)
{
  return (unsigned)(2 * pr) * s.unit;
}

}  // namespace ehip
#endif
