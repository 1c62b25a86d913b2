// What 32-bit byte offsets reach of a convolution's tensors, and the runs of images and ranges of depth that follow from it.
// Host arithmetic only.
#pragma once
#include <algorithm>
#include <cstdint>

namespace tsplit {

struct ConvTileGeo {
  int imgs, C, H, W, O, kH, kW, ph, pw, s, oH, oW;
};

// The tile kernel addresses the gathered tensor with 32-bit byte offsets.  One beyond `reach` bytes is taken in runs of whole images,
// one launch each (images are independent in the forward and backward-data passes): -> images per launch, 0 if not even one fits or
// an image has no elements.
inline int images_per_launch(const ConvTileGeo &g, int64_t src_elems_per_img, int64_t reach) {
  if (g.imgs <= 0 || src_elems_per_img <= 0) return 0;
  // what the base is moved back by, so that no offset is negative: the padding (forward), the last tap (data gradient)
  const int64_t back = std::max(static_cast<int64_t>(g.kH + g.ph) * g.W + g.kW + g.pw, static_cast<int64_t>(g.kH - 1) * g.oW + g.kW - 1);
  const int64_t room = reach - 4 * back;
  const int64_t fit = room / (src_elems_per_img * 4);
  if (fit < 1) return 0;
  if (fit >= g.imgs) return g.imgs;
  const int64_t launches = (g.imgs + fit - 1) / fit;          // equal runs rather than a short last one
  return static_cast<int>((g.imgs + launches - 1) / launches);
}

// The filter gradient's depth: images x positions, an image's positions in whole words of 4.
constexpr int kDepthStep = 32;   // of one step of its kernel
inline int depth_per_image(const ConvTileGeo &g) { return (g.oH * g.oW + 3) / 4 * 4; }
inline int64_t padded_depth(const ConvTileGeo &g) { return static_cast<int64_t>(depth_per_image(g)) * g.imgs; }

// images of both tensors that lie within `reach` bytes of the first one, rows past the last channel included
inline int64_t span_images(const ConvTileGeo &g, int64_t reach) {
  const int64_t dy = static_cast<int64_t>(g.O + 128) * g.oH * g.oW * 4, x = static_cast<int64_t>(g.C + 128) * g.H * g.W * 4;
  return reach / std::max<int64_t>(1, std::max(dy, x));
}
// The deepest range whose images, wherever it begins, lie within that span (it begins and ends inside an image at worst); a
// multiple of the step, 0 if not even one step fits.
inline int64_t deepest_range(const ConvTileGeo &g, int64_t reach) {
  const int64_t span = span_images(g, reach);
  const int64_t depth = span < g.imgs ? (span - 2) * depth_per_image(g) : padded_depth(g) + kDepthStep - 1;
  return std::max<int64_t>(0, depth / kDepthStep * kDepthStep);
}
// where the filter gradient's kernel can take the shape
inline bool filter_gradient_in_reach(const ConvTileGeo &g, int64_t reach) {
  return span_images(g, reach) >= 3 && deepest_range(g, reach) >= kDepthStep && padded_depth(g) < (1ll << 31) - 64 &&
         static_cast<int64_t>(g.O) * (g.C + 16) * g.kH * g.kW < (1ll << 31) - 256;
}
// depth of a range where `S` of them are asked for
inline int range_depth(const ConvTileGeo &g, int64_t reach, int S) {
  const int64_t steps = (padded_depth(g) + kDepthStep - 1) / kDepthStep;
  return static_cast<int>(std::min((steps + S - 1) / S * kDepthStep, deepest_range(g, reach)));
}

}  // namespace tsplit
