/* C ABI of the layout changes at the edge of the single-image modules (libinpaint_hip.so): images with their channels innermost
 * (H x W x C, any strides) to and from channel planes (C x H x W), several images per launch.
 *
 * Same conventions as tvinpaint.h: device pointers on the current HIP device, float32, `stream` a hipStream_t passed as void*.
 * The calls only enqueue work; the arrays are read before they return.
 */
#ifndef LAYOUT_H_
#define LAYOUT_H_

#include "tvinpaint.h"

#ifdef __cplusplus
extern "C" {
#endif

#define LAYOUT_MAX_IMAGES 8

/* count images of h x w pixels; image i has channels[i] channels, its element (y, x, c) lies at
 * y * strides[3 * i] + x * strides[3 * i + 1] + c * strides[3 * i + 2] floats; its planes are contiguous.
 * layout_to_planes: src images, dst planes.  layout_to_images: src planes, dst images. */
int layout_to_planes(const float* const* src, float* const* dst, const int* channels, const long long* strides, int count, int h,
                     int w, void* stream);
int layout_to_images(const float* const* src, float* const* dst, const int* channels, const long long* strides, int count, int h,
                     int w, void* stream);

const char* layout_last_error(void);

#ifdef __cplusplus
}
#endif

#endif /* LAYOUT_H_ */
