// Layout changes at the edge of the single-image modules for MI355X (gfx950): images with their channels innermost to and from
// channel planes, several images per launch.  C ABI in include/layout.h.
#include <hip/hip_runtime.h>

#include "../../include/layout.h"
#include "inpaint_common.h"

namespace {

using inpaint::fail;

struct Image {
  const float* src;
  float* dst;
  int channels;
  long long row, column, channel;  // strides of the image, in floats
};
struct Images {
  Image of[LAYOUT_MAX_IMAGES];
};

// One pixel per thread, blockIdx.y the image: the channels of a wavefront's 64 pixels are one contiguous run (of a contiguous
// image), read or written stride by stride while its lines are in the cache; the planes' side is coalesced.  Bound by memory.
// torch's strided copies take a launch for each image, four of them and 29 us of kernels before a TGV pass of 1 x 2 x 375 x 1241;
// 100 iterations forward from the module: 613 us with them, 601 with this launch.
template <bool TO_PLANES>
__global__ __launch_bounds__(256) void move_images(Images images, int W, int P) {
  const Image im = images.of[blockIdx.y];
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= P) return;
  const int y = p / W, x = p - y * W;
  const long long at = y * im.row + x * im.column;
#pragma unroll 4
  for (int c = 0; c < im.channels; c++) {
    const long long plane = (long long)c * P + p, pixel = at + c * im.channel;
    if (TO_PLANES) im.dst[plane] = im.src[pixel];
    else im.dst[pixel] = im.src[plane];
  }
}

template <bool TO_PLANES>
int move(const char* name, const float* const* src, float* const* dst, const int* channels, const long long* strides, int count, int h,
         int w, void* stream) {
  if (!src || !dst || !channels || !strides) return fail(INPAINT_ERR_ARG, "%s: null pointer", name);
  if (count < 1 || count > LAYOUT_MAX_IMAGES) return fail(INPAINT_ERR_ARG, "%s: 1 to %d images, not %d", name, LAYOUT_MAX_IMAGES, count);
  if (h < 1 || w < 1 || (long long)h * w >= (1ll << 31) - 256) return fail(INPAINT_ERR_ARG, "%s: bad size %dx%d", name, h, w);
  Images images{};
  for (int i = 0; i < count; i++) {
    if (!src[i] || !dst[i] || channels[i] < 1) return fail(INPAINT_ERR_ARG, "%s: image %d: null pointer or no channel", name, i);
    images.of[i] = {src[i], dst[i], channels[i], strides[3 * i], strides[3 * i + 1], strides[3 * i + 2]};
  }
  const int P = h * w;
  hipLaunchKernelGGL(move_images<TO_PLANES>, dim3((unsigned)((P + 255) / 256), (unsigned)count), dim3(256), 0, (hipStream_t)stream, images, w, P);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

}  // namespace

extern "C" {

const char* layout_last_error(void) { return inpaint::error_buffer(); }

int layout_to_planes(const float* const* src, float* const* dst, const int* channels, const long long* strides, int count, int h,
                     int w, void* stream) {
  return move<true>("layout_to_planes", src, dst, channels, strides, count, h, w, stream);
}

int layout_to_images(const float* const* src, float* const* dst, const int* channels, const long long* strides, int count, int h,
                     int w, void* stream) {
  return move<false>("layout_to_images", src, dst, channels, strides, count, h, w, stream);
}

}  // extern "C"
