// Quadratic sub-pixel fit of a matching cost and median of a per-pixel displacement histogram for
// MI355X (gfx950): the two small layers upstream of the inpainting layer.  C ABI in
// include/flowaux.h; reference: cudaQuadFit/cudaCode/quadFit.cu (QF.cu below) and
// cudaMedian/cudaCode/medimax.cu (MM.cu).
//
// Arithmetic: every expression keeps the reference's operation order and types (its double
// literals promote the surrounding sub-expression), no contraction, IEEE division -- the per-pixel
// results are bit-equal to a plain C++ evaluation of the reference source.  The one exception is the
// gradient wrt the second feature map, a scatter with float atomics whose order is not defined
// (here or in the reference).
//
// Layout of the work:
//  * quadratic fit: one pixel per lane, lanes along the image row, a loop over the feature
//    channels.  Per channel a wavefront reads one 256-byte row segment of the first map and three
//    (shifted, overlapping) row segments of the second map around the displaced position; the
//    overlaps are served by the vector L1.  HBM sees every feature once: (2C+5) floats per pixel
//    forward, (5C+5) backward (the scatter reads and writes its target).
//  * median: the histogram bins are innermost in memory, so a lane that walked its own pixel's bins
//    would touch a new cache line per step.  The histograms of 64 consecutive pixels are one
//    contiguous run: a wavefront brings it into LDS with full-line loads and each lane walks its
//    pixel's bins there in the reference's sequential order.  Above 255 bins the run comes in pieces
//    of 32 bins (row pitch 33 words: no bank conflicts), and the forward pass stops at the piece in
//    which the last pixel of the block found its median.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdlib>

#include "../../include/flowaux.h"
#include "inpaint_common.h"

namespace {

using inpaint::fail;

// optional timing of the dominant kernel of each backward pass (the bench switches it on)
inpaint::KernelTimer g_timer;
int g_timed_pass = 1;  // quadratic fit, backward: 1 = the per-source pass, 2 = the gather pass

// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Pixels that are close in
// the image read the same lines of the second feature map (the rows above and below, the shifted
// segments), so the blocks are renumbered such that every XCD works through one contiguous band of
// the pixel range.  The grid is a multiple of 8 blocks; blocks past the end return.
__device__ __forceinline__ long long banded_pixel_index() {
  const int per_xcd = gridDim.x >> 3;
  const int logical_block = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  return (long long)logical_block * 256 + threadIdx.x;
}
inline dim3 banded_grid(long long pixels) { return dim3((unsigned)(((pixels + 255) / 256 + 7) / 8 * 8)); }

// ---------------------------------------------------------------------------------------------
// quadratic fit
// ---------------------------------------------------------------------------------------------
struct Fit {
  bool inside;
  int validX, validY;
  unsigned o00, o0p, o0m, op0, om0;  // offsets of the five taps inside one channel plane
  int ix, iy;
  float c00, ax, ay, bx, by, fx, fy;
};

// QF.cu:75-104 == QF.cu:198-226: the two parabolas through the five costs, their validity and vertices
__device__ __forceinline__ void finish_fit(Fit& f, float cost00, float cost0p, float costp0, float cost0m, float costm0,
                                           int iidx, int iidy, int H, int W) {
  f.c00 = cost00;
  f.ax = 0.5 * (cost0p + cost0m - 2. * cost00);  // QF.cu:75-78
  f.ay = 0.5 * (costp0 + costm0 - 2. * cost00);
  f.bx = 0.5 * (cost0p - cost0m);
  f.by = 0.5 * (costp0 - costm0);
  f.validX = (f.ax < 0 && f.ax * f.ax >= 0.25 * f.bx * f.bx);  // QF.cu:83-89
  f.validY = (f.ay < 0 && f.ay * f.ay >= 0.25 * f.by * f.by);
  if (!(iidx < W - 1 && iidx > 0)) f.validX = 0;
  if (!(iidy < H - 1 && iidy > 0)) f.validY = 0;
  f.fx = f.fy = 0.f;
  if (f.validX) f.fx = -0.5 * f.bx / f.ax;  // QF.cu:92-104
  if (f.validY) f.fy = -0.5 * f.by / f.ay;
}

// QF.cu:22-104 (forward) == QF.cu:149-226 (backward): displaced position, the five matching
// costs, the two parabolas and their validity.
__device__ __forceinline__ Fit fit_pixel(const float* __restrict__ a, const float* __restrict__ q,
                                         const float* __restrict__ fl, int d, int H, int W, size_t HW, int h, int w) {
  Fit f;
  const unsigned p = (unsigned)h * W + w;
  const float idx = w + fl[p];       // QF.cu:31-32
  const float idy = h + fl[HW + p];
  f.inside = idx <= W - 1 && idx >= 0 && idy <= H - 1 && idy >= 0;  // QF.cu:35; a NaN displacement counts as outside
  f.validX = f.validY = 0;
  f.c00 = f.ax = f.ay = f.bx = f.by = f.fx = f.fy = 0.f;
  f.ix = f.iy = 0;
  f.o00 = f.o0p = f.o0m = f.op0 = f.om0 = 0;
  if (!f.inside) return f;
  const int iidx = (int)floor(idx + 0.5);  // QF.cu:47-48
  const int iidy = (int)floor(idy + 0.5);
  const int iidx_m = max(iidx - 1, 0), iidy_m = max(iidy - 1, 0);  // QF.cu:50-53
  const int iidx_p = min(iidx + 1, W - 1), iidy_p = min(iidy + 1, H - 1);
  f.ix = iidx; f.iy = iidy;
  f.o00 = (unsigned)iidy * W + iidx;
  f.o0p = (unsigned)iidy * W + iidx_p;
  f.o0m = (unsigned)iidy * W + iidx_m;
  f.op0 = (unsigned)iidy_p * W + iidx;
  f.om0 = (unsigned)iidy_m * W + iidx;
  float cost00 = 0.f, cost0p = 0.f, costp0 = 0.f, cost0m = 0.f, costm0 = 0.f;
#pragma unroll 4
  for (int cc = 0; cc < d; cc++) {  // QF.cu:63-71
    const float I1 = a[(size_t)cc * HW + p];
    const float* qc = q + (size_t)cc * HW;
    cost00 += I1 * qc[f.o00];
    cost0p += I1 * qc[f.o0p];
    costp0 += I1 * qc[f.op0];
    cost0m += I1 * qc[f.o0m];
    costm0 += I1 * qc[f.om0];
  }
  finish_fit(f, cost00, cost0p, costp0, cost0m, costm0, iidx, iidy, H, W);
  return f;
}

// QF.cu:14-139.  Every pixel writes its three outputs (zero outside the image), so no fill pass.
__global__ __launch_bounds__(256) void quadfit_forward_kernel(const float* __restrict__ im0, const float* __restrict__ im1,
                                                              const float* __restrict__ flow, float* __restrict__ out,
                                                              int N, int d, int H, int W, int fc) {
  const size_t HW = (size_t)H * W;
  const long long t = banded_pixel_index();
  if (t >= (long long)N * HW) return;
  const int n = (int)(t / HW);
  const unsigned p = (unsigned)(t - (long long)n * HW);
  const int h = p / W, w = p - h * W;
  const Fit f = fit_pixel(im0 + (size_t)n * d * HW, im1 + (size_t)n * d * HW, flow + (size_t)n * fc * HW, d, H, W, HW, h, w);
  float* o = out + (size_t)n * 3 * HW + p;
  float score = 0.f;
  if (f.inside)  // QF.cu:136 (fx, fy are zero wherever QF.cu:125-133 would not store them)
    score = f.ax * f.fx * f.fx + f.bx * f.fx + f.c00 + f.ay * f.fy * f.fy + f.by * f.fy;
  o[0] = f.fx;
  o[HW] = f.fy;
  o[2 * HW] = score;
}

// QF.cu:145-300.  g0 is written by its own pixel (zero outside the image); g1 is zero-filled
// before the launch and collects the scatter.
__global__ __launch_bounds__(256) void quadfit_backward_kernel(const float* __restrict__ im0, const float* __restrict__ im1,
                                                               const float* __restrict__ flow, const float* __restrict__ gin,
                                                               float* __restrict__ g0, float* __restrict__ g1, int N,
                                                               int d, int H, int W, int fc) {
  const size_t HW = (size_t)H * W;
  const long long t = banded_pixel_index();
  if (t >= (long long)N * HW) return;
  const int n = (int)(t / HW);
  const unsigned p = (unsigned)(t - (long long)n * HW);
  const int h = p / W, w = p - h * W;
  const float* a = im0 + (size_t)n * d * HW;
  const float* q = im1 + (size_t)n * d * HW;
  float* G0 = g0 + (size_t)n * d * HW;
  float* G1 = g1 + (size_t)n * d * HW;
  const Fit f = fit_pixel(a, q, flow + (size_t)n * fc * HW, d, H, W, HW, h, w);
  if (!f.inside) {
    for (int cc = 0; cc < d; cc++) G0[(size_t)cc * HW + p] = 0.f;
    return;
  }
  const int validX = f.validX, validY = f.validY;
  const float ax = f.ax, ay = f.ay, fx = f.fx, fy = f.fy;
  // QF.cu:244-253
  const float dfx_dbx = validX ? -1. / (2. * ax) : 0.;
  const float dfx_dax = validX ? -fx / ax : 0.;
  const float dfy_dby = validY ? -1. / (2. * ay) : 0.;
  const float dfy_day = validY ? -fy / ay : 0.;
  const float ds_dax = validX ? fx * fx : 0.;
  const float ds_dbx = validX ? fx : 0.;
  const float ds_dc = (validX || validY) ? 1. : 0.;
  const float ds_day = validY ? fy * fy : 0.;
  const float ds_dby = validY ? fy : 0.;
  const float dFdfx = gin[(size_t)n * 3 * HW + p];  // QF.cu:261-263
  const float dFdfy = gin[(size_t)n * 3 * HW + HW + p];
  const float dFds = gin[(size_t)n * 3 * HW + 2 * HW + p];
  // the channel-independent factors of QF.cu:279-290, each in the type the source gives it
  const double k00 = -2. * dFdfx * dfx_dax - 2. * dFdfy * dfy_day - 2. * dFds * ds_dax - 2. * dFds * ds_day + 2. * dFds * ds_dc;
  const float k0p = dFdfx * dfx_dax + dFdfx * dfx_dbx + dFds * ds_dax + dFds * ds_dbx;
  const float k0m = dFdfx * dfx_dax - dFdfx * dfx_dbx + dFds * ds_dax - dFds * ds_dbx;
  const float kp0 = dFdfy * dfy_day + dFdfy * dfy_dby + dFds * ds_day + dFds * ds_dby;
  const float km0 = dFdfy * dfy_day - dFdfy * dfy_dby + dFds * ds_day - dFds * ds_dby;
  if (validX || validY) {
#pragma unroll 2
    for (int cc = 0; cc < d; cc++) {
      const float* qc = q + (size_t)cc * HW;
      float* gc = G1 + (size_t)cc * HW;
      const float I1 = a[(size_t)cc * HW + p];
      const float I2 = qc[f.o00], I2_0p = qc[f.o0p], I2_0m = qc[f.o0m], I2_p0 = qc[f.op0], I2_m0 = qc[f.om0];
      unsafeAtomicAdd(gc + f.o00, (float)(0.5 * I1 * k00));
      unsafeAtomicAdd(gc + f.o0p, (float)(0.5 * I1 * k0p));
      unsafeAtomicAdd(gc + f.o0m, (float)(0.5 * I1 * k0m));
      unsafeAtomicAdd(gc + f.op0, (float)(0.5 * I1 * kp0));
      unsafeAtomicAdd(gc + f.om0, (float)(0.5 * I1 * km0));
      G0[(size_t)cc * HW + p] = 0.5 * (I2 * k00 + I2_0p * k0p + I2_0m * k0m + I2_p0 * kp0 + I2_m0 * km0);
    }
  } else {  // QF.cu:293-297: only the centre cost carries a gradient
#pragma unroll 4
    for (int cc = 0; cc < d; cc++) {
      const float I1 = a[(size_t)cc * HW + p];
      const float I2 = q[(size_t)cc * HW + f.o00];
      G0[(size_t)cc * HW + p] = I2 * dFds;
      unsafeAtomicAdd(G1 + (size_t)cc * HW + f.o00, I1 * dFds);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Quadratic fit, backward without float atomics.  Agent-scope float atomics are executed at the
// memory side on this GPU and run two orders of magnitude below HBM speed, so the scatter into the
// gradient of the second feature map is turned into a gather through a per-call inverse map:
//   pass A (per source pixel)  fit, gradient wrt the first map, the five scatter coefficients of the
//                              pixel (they do not depend on the channel) and one integer atomic that
//                              appends the pixel to the list of its displaced position (kSlots entries
//                              per position; what does not fit goes to an overflow list);
//   pass B (per target pixel)  gathers, per channel, I1 * coefficient from the sources listed at the
//                              target and at its four neighbours (a source centred on the left
//                              neighbour reaches the target with its right tap, and so on);
//   pass C (two lists)         after pass B, with float atomics: the sources that found their list full (it takes more
//                              than kSlots pixels landing on one position), and the target pixels that pass B has listed
//                              and left at zero: more sources than it holds in registers, or one outside its window.  A
//                              few pixels in a hundred on a smooth flow, a quarter on one that contracts by two, nearly
//                              all on one that scatters every tile.
// A tap that the image border clamps back onto the centre carries a zero coefficient (the axis is
// not fitted at the border), so the gather leaves it out.
// Workspace (caller provided): count[P] | overflow count, slow count, pad | slots[P*kSlots] | overflow list[P] | coef[5*P] |
// slow list[P].
// ---------------------------------------------------------------------------------------------
constexpr int kSlots = 4;

struct QfWorkspace {
  int* count;      // sources per displaced position
  int* ovf_count;  // one counter
  int* slots;      // [P][kSlots] source pixel (index inside its sample)
  int* slow_count; // one counter
  int* ovf;        // global index of the sources that did not fit
  int* slow;       // global index of the target pixels that pass B leaves to pass C
  float* coef;     // [5][P]: taps 00, 0p, 0m, p0, m0
};
long long qf_workspace_bytes(long long P) { return (long long)sizeof(int) * (P * (8 + kSlots) + 64 + 4); }
QfWorkspace qf_carve(void* base, long long P) {
  QfWorkspace w;
  int* p = reinterpret_cast<int*>(base);
  w.count = p;
  w.ovf_count = p + P;
  w.slow_count = p + P + 1;
  w.slots = p + (P + 64 + 3) / 4 * 4;  // 16-byte aligned: a position's kSlots entries are read as one int4
  w.ovf = w.slots + P * kSlots;
  w.coef = reinterpret_cast<float*>(w.ovf + P);
  w.slow = w.ovf + 6 * P;
  return w;
}

// the channel-independent factors of QF.cu:244-263,279-297 as multipliers of I1 (scatter) and I2 (g0)
struct Factors {
  bool any_valid;
  double k00;
  float k0p, k0m, kp0, km0, dFds;
};
__device__ __forceinline__ Factors scatter_factors(const Fit& f, float dFdfx, float dFdfy, float dFds) {
  Factors k;
  const int validX = f.validX, validY = f.validY;
  const float ax = f.ax, ay = f.ay, fx = f.fx, fy = f.fy;
  const float dfx_dbx = validX ? -1. / (2. * ax) : 0.;  // QF.cu:244-253
  const float dfx_dax = validX ? -fx / ax : 0.;
  const float dfy_dby = validY ? -1. / (2. * ay) : 0.;
  const float dfy_day = validY ? -fy / ay : 0.;
  const float ds_dax = validX ? fx * fx : 0.;
  const float ds_dbx = validX ? fx : 0.;
  const float ds_dc = (validX || validY) ? 1. : 0.;
  const float ds_day = validY ? fy * fy : 0.;
  const float ds_dby = validY ? fy : 0.;
  k.any_valid = validX || validY;
  k.dFds = dFds;
  k.k00 = -2. * dFdfx * dfx_dax - 2. * dFdfy * dfy_day - 2. * dFds * ds_dax - 2. * dFds * ds_day + 2. * dFds * ds_dc;
  k.k0p = dFdfx * dfx_dax + dFdfx * dfx_dbx + dFds * ds_dax + dFds * ds_dbx;
  k.k0m = dFdfx * dfx_dax - dFdfx * dfx_dbx + dFds * ds_dax - dFds * ds_dbx;
  k.kp0 = dFdfy * dfy_day + dFdfy * dfy_dby + dFds * ds_day + dFds * ds_dby;
  k.km0 = dFdfy * dfy_day - dFdfy * dfy_dby + dFds * ds_day - dFds * ds_dby;
  return k;
}

__device__ __forceinline__ Factors scatter_factors(const Fit& f, const float* __restrict__ gin, size_t n, size_t HW, unsigned p) {
  return scatter_factors(f, gin[n * 3 * HW + p], gin[n * 3 * HW + HW + p], gin[n * 3 * HW + 2 * HW + p]);  // QF.cu:261-263
}

// a source's scatter coefficients (contribution to g1 at a tap = I1 * coefficient, QF.cu:279-283,296) and its entry in the list
// of the position it lands on
__device__ __forceinline__ void store_source(const QfWorkspace& ws, const Factors& k, long long P, long long base, long long t,
                                             long long landing, unsigned p) {
  ws.coef[0 * P + t] = k.any_valid ? (float)(0.5 * k.k00) : k.dFds;
  ws.coef[1 * P + t] = k.any_valid ? 0.5f * k.k0p : 0.f;
  ws.coef[2 * P + t] = k.any_valid ? 0.5f * k.k0m : 0.f;
  ws.coef[3 * P + t] = k.any_valid ? 0.5f * k.kp0 : 0.f;
  ws.coef[4 * P + t] = k.any_valid ? 0.5f * k.km0 : 0.f;
  const long long centre = base + landing;
  const int pos = atomicAdd(ws.count + centre, 1);
  if (pos < kSlots) ws.slots[centre * kSlots + pos] = (int)p;
  else ws.ovf[atomicAdd(ws.ovf_count, 1)] = (int)t;
}

__global__ __launch_bounds__(256) void quadfit_backward_sources(const float* __restrict__ im0, const float* __restrict__ im1,
                                                                const float* __restrict__ flow, const float* __restrict__ gin,
                                                                float* __restrict__ g0, QfWorkspace ws, int N, int d, int H,
                                                                int W, int fc) {
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW;
  const long long t = banded_pixel_index();
  if (t >= P) return;
  const int n = (int)(t / HW);
  const unsigned p = (unsigned)(t - (long long)n * HW);
  const int h = p / W, w = p - h * W;
  const float* a = im0 + (size_t)n * d * HW;
  const float* q = im1 + (size_t)n * d * HW;
  float* G0 = g0 + (size_t)n * d * HW;
  const Fit f = fit_pixel(a, q, flow + (size_t)n * fc * HW, d, H, W, HW, h, w);
  if (!f.inside) {
    for (int cc = 0; cc < d; cc++) G0[(size_t)cc * HW + p] = 0.f;
    return;
  }
  const Factors k = scatter_factors(f, gin, n, HW, p);
  store_source(ws, k, P, (long long)n * HW, t, f.o00, p);
  if (k.any_valid) {
#pragma unroll 4
    for (int cc = 0; cc < d; cc++) {  // QF.cu:286-290
      const float* qc = q + (size_t)cc * HW;
      const float I2 = qc[f.o00], I2_0p = qc[f.o0p], I2_0m = qc[f.o0m], I2_p0 = qc[f.op0], I2_m0 = qc[f.om0];
      G0[(size_t)cc * HW + p] = 0.5 * (I2 * k.k00 + I2_0p * k.k0p + I2_0m * k.k0m + I2_p0 * k.kp0 + I2_m0 * k.km0);
    }
  } else {
#pragma unroll 4
    for (int cc = 0; cc < d; cc++) G0[(size_t)cc * HW + p] = q[(size_t)cc * HW + f.o00] * k.dFds;  // QF.cu:295
  }
}

__global__ __launch_bounds__(256) void quadfit_backward_gather(const float* __restrict__ im0, float* __restrict__ g1,
                                                               QfWorkspace ws, int N, int d, int H, int W) {
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW;
  const long long t = banded_pixel_index();
  if (t >= P) return;
  const int n = (int)(t / HW);
  const unsigned p = (unsigned)(t - (long long)n * HW);
  const int h = p / W, w = p - h * W;
  const long long base = (long long)n * HW;
  const float* a = im0 + (size_t)n * d * HW;
  float* G1 = g1 + (size_t)n * d * HW + p;
  // (position whose sources reach this pixel, tap they reach it with); -1: outside the image
  long long ctr[5];
  ctr[0] = base + p;
  ctr[1] = w > 0 ? base + p - 1 : -1;      // right tap of the left neighbour
  ctr[2] = w < W - 1 ? base + p + 1 : -1;  // left tap of the right neighbour
  ctr[3] = h > 0 ? base + p - W : -1;      // lower tap of the upper neighbour
  ctr[4] = h < H - 1 ? base + p + W : -1;  // upper tap of the lower neighbour
  // compact list of the (source, coefficient) pairs that reach this pixel, in registers
  constexpr int kPairs = 8;
  unsigned src[kPairs];
  float cf[kPairs];
#pragma unroll
  for (int j = 0; j < kPairs; j++) {
    src[j] = p;
    cf[j] = 0.f;
  }
  int cnt[5];
  int np = 0;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    cnt[k] = ctr[k] >= 0 ? min(ws.count[ctr[k]], kSlots) : 0;
#pragma unroll
    for (int i = 0; i < kSlots; i++) {
      if (i < cnt[k]) {
        const unsigned sidx = (unsigned)ws.slots[ctr[k] * kSlots + i];
        const float c = ws.coef[(long long)k * P + base + sidx];
#pragma unroll
        for (int j = 0; j < kPairs; j++)
          if (np == j) {
            src[j] = sidx;
            cf[j] = c;
          }
        np++;
      }
    }
  }
  // longest list among the wavefront's active lanes: the unrolled gathers beyond it are skipped by a uniform branch
  unsigned need = 0;
#pragma unroll
  for (int j = 0; j < kPairs; j++)
    if (__ballot(np > j) != 0) need |= 1u << j;
  if (np <= kPairs) {
    for (int cc = 0; cc < d; cc++) {
      const float* ac = a + (size_t)cc * HW;
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < kPairs; j++)
        if (need & (1u << j)) acc += ac[src[j]] * cf[j];
      G1[(size_t)cc * HW] = acc;
    }
    return;
  }
  for (int cc = 0; cc < d; cc++) {  // more pairs than registers: walk the lists per channel
    const float* ac = a + (size_t)cc * HW;
    float acc = 0.f;
#pragma unroll
    for (int k = 0; k < 5; k++)
      for (int i = 0; i < cnt[k]; i++) {
        const unsigned sidx = (unsigned)ws.slots[ctr[k] * kSlots + i];
        acc += ac[sidx] * ws.coef[(long long)k * P + base + sidx];
      }
    G1[(size_t)cc * HW] = acc;
  }
}

// Pass C, after the gather has written g1: the sources whose list was full, one lane per (source, channel), and the target
// pixels the gather has left at zero.  Both add with float atomics.
// Few such pixels -- up to 64 values to write per wavefront of the launch: one wavefront per pixel, one lane per list entry and
// then per channel, so that all reads of a pixel are in flight at once; every read touches as many cache lines as there are
// channels.
// Many: one lane per pixel.  A wavefront takes 64 that follow each other in the list (the gather lists a row's pixels
// together, so their sources are neighbours too) and a share of the channels, as small a share as gives every wavefront work;
// each lane collects its pairs in LDS and sums four channels at a time.  Bound by the reads of the first map either way.
// Backward pass, us, wavefront per pixel / lane per pixel (/ walked inside the gather, one lane per pixel and all channels):
// 1 x 8 x 448 x 1000, a flow that scatters every tile 655 / 316 (/ 350); one that contracts by two 310 / 193 (/ 406);
// 542 such pixels in the image 75 / 95 (/ 116), some 4500 92 / 97 (/ 158); 2 x 64 x 192 x 624, some 4500 of them 279 / 262
// (/ 1076); 4 x 32 x 384 x 1248, 19384 of them 715 / 683 (/ 1436).
constexpr int kEntries = 5 * kSlots, kQuad = 4;  // list entries a pixel can have, channels (and entries) in flight
static_assert(kSlots == 4 && kEntries % kQuad == 0, "four entries per list");

// (first: this wavefront's number in the launch of `waves`)
__device__ __forceinline__ void add_one_pixel_per_wavefront(const float* __restrict__ im0, float* __restrict__ g1, const QfWorkspace& ws,
                                                            int slow, int first, int waves, long long P, int d, int H, int W) {
  const size_t HW = (size_t)H * W;
  const int lane = threadIdx.x & 63;
  for (int r = first; r < slow; r += waves) {
    const int t = __builtin_amdgcn_readfirstlane(ws.slow[r]);
    const int n = t / (int)HW;
    const long long base = (long long)n * HW;
    const unsigned p = (unsigned)(t - base);
    const int y = p / W, x = p - y * W;
    const int k = lane >> 2, e = lane & 3;  // list (tap) and entry of lanes 0..19
    const bool has = k == 0 || (k == 1 && x > 0) || (k == 2 && x < W - 1) || (k == 3 && y > 0) || (k == 4 && y < H - 1);
    const long long ctr = base + (long long)p + (!has ? 0 : (k == 1 ? -1 : (k == 2 ? 1 : (k == 3 ? -W : (k == 4 ? W : 0)))));
    const bool used = has && e < min(ws.count[ctr], kSlots);
    const unsigned sp = used ? (unsigned)ws.slots[ctr * kSlots + e] : 0u;
    const float c = used ? ws.coef[(long long)k * P + base + sp] : 0.f;
    const unsigned long long mask = __ballot(used);
    // (all lanes stay in this loop, the ones past the last channel on that channel: lanes 0..19 hold the entries the others read)
    for (int c0 = 0; c0 < d; c0 += 64) {
      const int cc = min(c0 + lane, d - 1);
      const float* ac = im0 + ((size_t)n * d + cc) * HW;
      float v[5 * kSlots];
#pragma unroll
      for (int j = 0; j < 5 * kSlots; j++) v[j] = ac[(unsigned)__builtin_amdgcn_readlane((int)sp, j)];  // (unused: the plane's first value)
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 5 * kSlots; j++)
        if ((mask >> j) & 1) acc += v[j] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c), j));
      if (c0 + lane < d) unsafeAtomicAdd(g1 + ((size_t)n * d + cc) * HW + p, acc);
    }
  }
}

__device__ __forceinline__ void add_one_pixel_per_lane(const float* __restrict__ im0, float* __restrict__ g1, const QfWorkspace& ws,
                                                       float2 (*front)[64], int slow, int first, int waves, long long P, int d, int H,
                                                       int W) {
  const size_t HW = (size_t)H * W;
  const int lane = threadIdx.x & 63;
  const int groups = (int)((slow + 63ll) / 64), quads = (d + kQuad - 1) / kQuad;
  const int shares = min(quads, max(1, waves / groups)), per = (quads + shares - 1) / shares;  // quads of channels per item
  const long long items = (long long)groups * ((quads + per - 1) / per);
  for (long long item = first; item < items; item += waves) {
    const int share = (int)(item / groups), r = (int)(item - (long long)share * groups) * 64 + lane;
    const bool live = r < slow;
    const int t = ws.slow[min(r, slow - 1)];
    const int n = t / (int)HW;
    const long long base = (long long)n * HW;
    const unsigned p = (unsigned)(t - base);
    const int y = p / W, x = p - y * W;
    const bool has[5] = {live, live && x > 0, live && x < W - 1, live && y > 0, live && y < H - 1};
    const int step[5] = {0, -1, 1, -W, W};
    int cnt[5];
    int4 sl[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {  // (an absent list reads the pixel's own)
      const long long ctr = base + (long long)p + (has[k] ? step[k] : 0);
      cnt[k] = ws.count[ctr];
      sl[k] = *reinterpret_cast<const int4*>(ws.slots + ctr * kSlots);
    }
    float cv[5][kSlots];
    unsigned spv[5][kSlots];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      cnt[k] = has[k] ? min(cnt[k], kSlots) : 0;
      const int e[kSlots] = {sl[k].x, sl[k].y, sl[k].z, sl[k].w};
#pragma unroll
      for (int s = 0; s < kSlots; s++) {
        spv[k][s] = s < cnt[k] ? (unsigned)e[s] : 0u;  // (an entry nobody filled: source 0, not used)
        cv[k][s] = ws.coef[(long long)k * P + base + spv[k][s]];
      }
    }
    // (computed here: all coefficients in one batch of loads, not each behind the branch of its entry)
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
      for (int s = 0; s < kSlots; s++) asm volatile("" : "+v"(cv[k][s]));
    int np = 0;
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
      for (int s = 0; s < kSlots; s++)
        if (s < cnt[k]) front[np++][lane] = make_float2(__uint_as_float(spv[k][s]), cv[k][s]);
    const float* a = im0 + (size_t)n * d * HW;
    float* G1 = g1 + (size_t)n * d * HW + p;
    for (int c0 = share * per * kQuad; c0 < min((share + 1) * per * kQuad, d); c0 += kQuad) {
      float acc[kQuad] = {0.f, 0.f, 0.f, 0.f};
      for (int j0 = 0; __ballot(j0 < np) != 0; j0 += kQuad) {
        float2 e[kQuad];
        float v[kQuad][kQuad];
#pragma unroll
        for (int j = 0; j < kQuad; j++) e[j] = front[j0 + j][lane];
#pragma unroll
        for (int j = 0; j < kQuad; j++) {
          const unsigned sp = j0 + j < np ? __float_as_uint(e[j].x) : 0u;  // (past a pixel's last entry: the plane's first value, not used)
#pragma unroll
          for (int q = 0; q < kQuad; q++) v[q][j] = a[(size_t)min(c0 + q, d - 1) * HW + sp];
        }
#pragma unroll
        for (int j = 0; j < kQuad; j++)
#pragma unroll
          for (int q = 0; q < kQuad; q++) acc[q] = j0 + j < np ? acc[q] + v[q][j] * e[j].y : acc[q];
      }
#pragma unroll
      for (int q = 0; q < kQuad; q++)
        if (live && c0 + q < d) unsafeAtomicAdd(G1 + (size_t)(c0 + q) * HW, acc[q]);
    }
  }
}

__global__ __launch_bounds__(256) void quadfit_backward_overflow(const float* __restrict__ im0, const float* __restrict__ flow,
                                                                 float* __restrict__ g1, QfWorkspace ws, int N, int d, int H,
                                                                 int W, int fc) {
  __shared__ float2 front[4][kEntries][64];
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW;
  const int slow = *ws.slow_count;
  const long long total = (long long)*ws.ovf_count * d;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), first = (int)blockIdx.x * 4 + wave, waves = (int)gridDim.x * 4;
  if ((long long)slow * d > 64ll * waves) add_one_pixel_per_lane(im0, g1, ws, front[wave], slow, first, waves, P, d, H, W);
  else add_one_pixel_per_wavefront(im0, g1, ws, slow, first, waves, P, d, H, W);
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
    const int e = (int)(i / d), cc = (int)(i - (long long)e * d);  // one lane per (source, channel)
    const long long t = ws.ovf[e];
    const int n = (int)(t / HW);
    const unsigned p = (unsigned)(t - (long long)n * HW);
    const int h = p / W, w = p - h * W;
    const float* fl = flow + (size_t)n * fc * HW;
    const float idx = w + fl[p], idy = h + fl[HW + p];  // QF.cu:31-32,47-53 (the pixel is inside the image)
    const int iidx = (int)floor(idx + 0.5), iidy = (int)floor(idy + 0.5);
    const unsigned o[5] = {(unsigned)iidy * W + iidx, (unsigned)iidy * W + min(iidx + 1, W - 1),
                           (unsigned)iidy * W + max(iidx - 1, 0), (unsigned)min(iidy + 1, H - 1) * W + iidx,
                           (unsigned)max(iidy - 1, 0) * W + iidx};
    const float I1 = im0[((size_t)n * d + cc) * HW + p];
    float* gc = g1 + ((size_t)n * d + cc) * HW;
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const float cf = ws.coef[(long long)k * P + t];
      if (cf != 0.f) unsafeAtomicAdd(gc + o[k], I1 * cf);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Tiled kernels.  A lane that reads its five taps straight from memory issues gathers whose
// addresses follow the (jittery) flow; the vector L1 then handles them almost lane by lane and
// becomes the bound.  Here a block owns a 64 x 16 tile of pixels (4 rows per lane), finds the
// bounding box of all taps of the tile, and per channel stages that window of the second feature
// map in LDS with row-wise coalesced loads (double buffered: the next channel's window is in flight
// while the taps of the current one are read from LDS).  A pixel whose taps do not fit the window's
// capacity reads them from memory as before.
// ---------------------------------------------------------------------------------------------
constexpr int kTW = 64;  // tile width: one pixel column per lane
constexpr int kMaxWinW = 128;  // widest window
template <int PX>              // PX pixels per lane (rows PX * wave + i): tile height, window capacity in floats
struct TileCfg {
  static constexpr int TH = 4 * PX, ELEMS = (96 * (4 * PX + 16) + 255) / 256 * 256;
};
constexpr int kPxTile = 2;

struct Box {
  int x0, y0, w, h;
};
struct TilePx {
  bool inside, far;
  int ix, iy, xm, xp, ym, yp;
  unsigned p;     // the pixel's offset inside a channel plane
  unsigned o[5];  // taps 00, 0p, 0m, p0, m0: offsets into the window, or into the plane when far
};

// QF.cu:31-53: displaced position and tap coordinates of pixel (x, y), displacement (u, v); widens the tile's bounding box
__device__ __forceinline__ void locate_at(TilePx& s, float u, float v, int H, int W, int x, int y, bool valid, int& minx, int& maxx,
                                          int& miny, int& maxy) {
  s.inside = s.far = false;
  s.ix = s.iy = s.xm = s.xp = s.ym = s.yp = 0;
  s.p = valid ? (unsigned)y * W + x : 0u;
  if (!valid) return;
  const float idx = x + u;
  const float idy = y + v;
  if (!(idx <= W - 1 && idx >= 0 && idy <= H - 1 && idy >= 0)) return;  // QF.cu:35; NaN counts as outside
  s.inside = true;
  s.ix = (int)floor(idx + 0.5);
  s.iy = (int)floor(idy + 0.5);
  s.xm = max(s.ix - 1, 0); s.ym = max(s.iy - 1, 0);
  s.xp = min(s.ix + 1, W - 1); s.yp = min(s.iy + 1, H - 1);
  minx = min(minx, s.xm); maxx = max(maxx, s.xp);
  miny = min(miny, s.ym); maxy = max(maxy, s.yp);
}
__device__ __forceinline__ void locate(TilePx& s, const float* __restrict__ fl, size_t HW, int H, int W, int x, int y,
                                       bool valid, int& minx, int& maxx, int& miny, int& maxy) {
  const unsigned p = valid ? (unsigned)y * W + x : 0u;
  locate_at(s, fl[p], fl[HW + p], H, W, x, y, valid, minx, maxx, miny, maxy);
}

__device__ __forceinline__ Box block_box(int minx, int maxx, int miny, int maxy, int* red, int capacity) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    minx = min(minx, __shfl_xor(minx, o));
    maxx = max(maxx, __shfl_xor(maxx, o));
    miny = min(miny, __shfl_xor(miny, o));
    maxy = max(maxy, __shfl_xor(maxy, o));
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[wave * 4 + 0] = minx; red[wave * 4 + 1] = maxx; red[wave * 4 + 2] = miny; red[wave * 4 + 3] = maxy;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; k++) {
    minx = min(minx, red[k * 4 + 0]); maxx = max(maxx, red[k * 4 + 1]);
    miny = min(miny, red[k * 4 + 2]); maxy = max(maxy, red[k * 4 + 3]);
  }
  Box b{0, 0, 0, 0};
  if (maxx >= minx) {
    b.x0 = minx; b.y0 = miny;
    b.w = min(maxx - minx + 1, kMaxWinW);
    b.h = min(maxy - miny + 1, capacity / b.w);
  }
  return b;
}

__device__ __forceinline__ void place(TilePx& s, const Box& b, int W) {
  if (!s.inside) return;
  s.far = !(s.xp - b.x0 < b.w && s.yp - b.y0 < b.h);
  if (s.far) {
    s.o[0] = (unsigned)s.iy * W + s.ix; s.o[1] = (unsigned)s.iy * W + s.xp; s.o[2] = (unsigned)s.iy * W + s.xm;
    s.o[3] = (unsigned)s.yp * W + s.ix; s.o[4] = (unsigned)s.ym * W + s.ix;
  } else {
    const int cx = s.ix - b.x0, cy = s.iy - b.y0;
    s.o[0] = cy * b.w + cx; s.o[1] = cy * b.w + (s.xp - b.x0); s.o[2] = cy * b.w + (s.xm - b.x0);
    s.o[3] = (s.yp - b.y0) * b.w + cx; s.o[4] = (s.ym - b.y0) * b.w + cx;
  }
}

// Streams the windows of planes q[0 .. d) through a double buffer in LDS and calls
// consume(cc, window, plane, extra, live) for each.  Two channels are in flight per thread: while channel c is consumed
// from LDS, channel c+1 waits in registers (loaded one step earlier) and channel c+2 is being loaded.  extra = pre(cc) is
// loaded together with the window of channel cc (values of another plane that the consumer needs).  Every load and
// every LDS store of the loop is unconditional -- elements past the window's end re-read its first element, channels
// past the last one re-read the last one -- so that the compiler can wait for exactly the loads a step needs instead of
// for all loads in flight; `live` is false for the surplus step of an odd channel count (the same for the whole block):
// the consumer must neither store nor accumulate then.
// PER: elements per thread, at least window size / 256 (window_pass below picks it per block: windows of smooth flows hold
// 900 to 1100 elements where the capacity is 2304, and nine loads per thread and channel for four took half the time again).
template <int PX, int PER, typename Pre, typename Consume>
__device__ __forceinline__ void window_pass_of(const float* __restrict__ q, int d, size_t HW, int W, const Box& box,
                                            float (*win)[TileCfg<PX>::ELEMS], Pre pre, Consume consume) {
  constexpr int kPer = PER;
  const int count = box.w * box.h;
  // window elements of this thread: e = threadIdx.x + 256 k, row e / w, column e % w (exact in float for these sizes)
  unsigned goff[kPer];
  const float inv_w = 1.0f / (float)max(box.w, 1);
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int e = threadIdx.x + 256 * k;
    const int r = (int)(((float)e + 0.5f) * inv_w);
    goff[k] = e < count ? (unsigned)(r * W + (e - r * box.w)) : 0u;
  }
  const float* corner = q + (size_t)box.y0 * W + box.x0;
  auto fetch = [&](int c, float (&r)[kPer]) {
    const float* src = corner + (size_t)c * HW;
#pragma unroll
    for (int k = 0; k < kPer; k++) r[k] = src[goff[k]];
  };
  auto stash = [&](const float (&r)[kPer], float* buf) {
#pragma unroll
    for (int k = 0; k < kPer; k++) buf[threadIdx.x + 256 * k] = r[k];
  };
  const int last = d - 1;
  float ra[kPer], rb[kPer];
  fetch(0, ra);
  auto ea = pre(0);
  fetch(min(1, last), rb);
  auto eb = pre(min(1, last));
  stash(ra, win[0]);
  __syncthreads();
  for (int c0 = 0; c0 < d; c0 += 2) {
    {  // channel c0 is in win[0], c0 + 1 on its way into rb
      const auto e = ea;
      fetch(min(c0 + 2, last), ra);
      ea = pre(min(c0 + 2, last));
      consume(c0, win[0], q + (size_t)c0 * HW, e, true);
      stash(rb, win[1]);
      __syncthreads();
    }
    {  // channel c0 + 1 is in win[1], c0 + 2 on its way into ra
      const auto e = eb;
      const int c = min(c0 + 1, last);
      fetch(min(c0 + 3, last), rb);
      eb = pre(min(c0 + 3, last));
      consume(c, win[1], q + (size_t)c * HW, e, c0 + 1 < d);
      stash(ra, win[0]);
      __syncthreads();
    }
  }
}

template <int PX, typename Pre, typename Consume>
__device__ __forceinline__ void window_pass(const float* __restrict__ q, int d, size_t HW, int W, const Box& box,
                                            float (*win)[TileCfg<PX>::ELEMS], Pre pre, Consume consume) {
  static_assert(TileCfg<PX>::ELEMS == 9 * 256, "loads per thread: 4 to 9");
  const int count = __builtin_amdgcn_readfirstlane(box.w * box.h);
  if (count <= 4 * 256) window_pass_of<PX, 4>(q, d, HW, W, box, win, pre, consume);
  else if (count <= 6 * 256) window_pass_of<PX, 6>(q, d, HW, W, box, win, pre, consume);
  else window_pass_of<PX, 9>(q, d, HW, W, box, win, pre, consume);
}

// the five taps of every inside pixel of the lane, from the window or (far pixels) from the plane
template <int PX, typename Body>
__device__ __forceinline__ void each_pixel_taps(const TilePx (&px)[PX], const float* buf, const float* plane, Body body) {
#pragma unroll
  for (int i = 0; i < PX; i++) {
    if (px[i].inside) {
      float t[5];
      if (!px[i].far) {
#pragma unroll
        for (int k = 0; k < 5; k++) t[k] = buf[px[i].o[k]];
      } else {
#pragma unroll
        for (int k = 0; k < 5; k++) t[k] = plane[px[i].o[k]];
      }
      body(i, t);
    }
  }
}

// decode the block's tile (XCD-banded numbering); false: the block has no tile
__device__ __forceinline__ bool tile_of_block(int N, int tiles_x, int tiles_y, int& n, int& tx, int& ty) {
  const int per_xcd = gridDim.x >> 3;
  const int lb = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int tiles = tiles_x * tiles_y;
  if (lb >= N * tiles) return false;
  n = lb / tiles;
  const int r = lb - n * tiles;
  ty = r / tiles_x;
  tx = r - ty * tiles_x;
  return true;
}

// Pass A of the backward pass (fit, g0, coefficients, lists), the second map read twice.
__global__ __launch_bounds__(256) void quadfit_sources_tiles(const float* __restrict__ im0, const float* __restrict__ im1,
                                                             const float* __restrict__ flow, const float* __restrict__ gin,
                                                             float* __restrict__ res, QfWorkspace ws, int N, int d, int H, int W,
                                                             int fc, int tiles_x, int tiles_y) {
  constexpr int PX = kPxTile;
  constexpr int kPX = PX, kTH = TileCfg<PX>::TH;
  __shared__ float win[2][TileCfg<PX>::ELEMS];
  __shared__ int red[16];
  int n, tx, ty;
  if (!tile_of_block(N, tiles_x, tiles_y, n, tx, ty)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW;
  const float* a = im0 + (size_t)n * d * HW;
  const float* q = im1 + (size_t)n * d * HW;
  const float* fl = flow + (size_t)n * fc * HW;
  const int x = tx * kTW + lane;
  TilePx px[kPX];
  bool valid[kPX];
  int minx = INT_MAX, maxx = INT_MIN, miny = INT_MAX, maxy = INT_MIN;
#pragma unroll
  for (int i = 0; i < kPX; i++) {
    const int y = ty * kTH + wave * kPX + i;
    valid[i] = x < W && y < H;
    locate(px[i], fl, HW, H, W, x, y, valid[i], minx, maxx, miny, maxy);
  }
  const Box box = block_box(minx, maxx, miny, maxy, red, TileCfg<PX>::ELEMS);
#pragma unroll
  for (int i = 0; i < kPX; i++) place(px[i], box, W);

  float cost[kPX][5];
#pragma unroll
  for (int i = 0; i < kPX; i++)
#pragma unroll
    for (int k = 0; k < 5; k++) cost[i][k] = 0.f;
  struct FirstMap {
    float v[kPX];
  };
  auto first_map = [&](int cc) {  // the lane's pixels of the first feature map (offset 0 for a pixel outside the image)
    FirstMap m;
#pragma unroll
    for (int i = 0; i < kPX; i++) m.v[i] = a[(size_t)cc * HW + px[i].p];
    return m;
  };
  window_pass<PX>(q, d, HW, W, box, win, first_map, [&](int cc, const float* buf, const float* plane, const FirstMap& m, bool live) {
    each_pixel_taps<PX>(px, buf, plane, [&](int i, const float (&t)[5]) {  // QF.cu:63-71
      if (live) {
#pragma unroll
        for (int k = 0; k < 5; k++) cost[i][k] += m.v[i] * t[k];
      }
    });
  });

  Fit f[kPX];
#pragma unroll
  for (int i = 0; i < kPX; i++) {
    f[i].inside = px[i].inside;
    f[i].validX = f[i].validY = 0;
    f[i].c00 = f[i].ax = f[i].ay = f[i].bx = f[i].by = f[i].fx = f[i].fy = 0.f;
    if (px[i].inside) finish_fit(f[i], cost[i][0], cost[i][1], cost[i][3], cost[i][2], cost[i][4], px[i].ix, px[i].iy, H, W);
  }
  float* G0 = res + (size_t)n * d * HW;
  Factors k[kPX];
#pragma unroll
  for (int i = 0; i < kPX; i++) {
    k[i].any_valid = false;
    k[i].k00 = 0.;
    k[i].k0p = k[i].k0m = k[i].kp0 = k[i].km0 = k[i].dFds = 0.f;
    if (valid[i] && !px[i].inside)
      for (int cc = 0; cc < d; cc++) G0[(size_t)cc * HW + px[i].p] = 0.f;
    if (!px[i].inside) continue;
    k[i] = scatter_factors(f[i], gin, n, HW, px[i].p);
    const long long t = (long long)n * HW + px[i].p;
    store_source(ws, k[i], P, (long long)n * HW, t, (long long)px[i].iy * W + px[i].ix, px[i].p);
  }
  auto nothing = [](int) { return 0; };
  window_pass<PX>(q, d, HW, W, box, win, nothing, [&](int cc, const float* buf, const float* plane, int, bool live) {
    each_pixel_taps<PX>(px, buf, plane, [&](int i, const float (&t)[5]) {
      float g;
      if (k[i].any_valid)  // QF.cu:286-290
        g = 0.5 * (t[0] * k[i].k00 + t[1] * k[i].k0p + t[2] * k[i].k0m + t[3] * k[i].kp0 + t[4] * k[i].km0);
      else  // QF.cu:295
        g = t[0] * k[i].dFds;
      if (live) __builtin_nontemporal_store(g, &G0[(size_t)cc * HW + px[i].p]);
    });
  });
}

// Pass A of the backward pass with one read of the second feature map.  The gradient wrt the first map needs
// the finished fit (all channels) and then the five taps of every channel again.  Here a lane owns ONE pixel and
// keeps its taps of up to DMAX channels in registers (5 * DMAX floats) while the windows stream through LDS, so
// the second sweep over the channels is arithmetic and stores only.  Same sums in the same order as
// quadfit_sources_tiles (QF.cu:63-71 for the costs, QF.cu:279-297 for the gradient).
constexpr int kResidentChannels = 32;
constexpr int kResidentRows = 4;      // tile height: one row per wavefront
constexpr int kResidentElems = 1024;  // window capacity in floats (a 64 x 4 tile with +-3 pixels of spread needs ~800)
constexpr int kResidentDepth = 4;
constexpr int kResidentBand = 16;     // tile rows per band of the block order     // channels in flight per thread

template <int DMAX, bool FULL>  // FULL: exactly DMAX channels
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void quadfit_sources_resident(const float* __restrict__ im0, const float* __restrict__ im1,
                                                                const float* __restrict__ flow, const float* __restrict__ gin,
                                                                float* __restrict__ res, QfWorkspace ws, int N, int d, int H,
                                                                int W, int fc, int tiles_x, int tiles_y) {
  constexpr int kTH = kResidentRows, kElems = kResidentElems, kPer = (kElems + 255) / 256, D = kResidentDepth;
  __shared__ float win[2][kElems];
  __shared__ int red[16];
  int n, tx, ty;
  if (!tile_of_block(N, tiles_x, tiles_y, n, tx, ty)) return;
  {  // consecutive blocks walk DOWN a band of kResidentBand tile rows, then move one tile to the right: the blocks
     // in flight on one XCD cover a patch about as tall as wide, and the window rows that vertically adjacent
     // tiles share are read from memory once
    const int r = ty * tiles_x + tx;
    const int per_band = kResidentBand * tiles_x;
    const int band = r / per_band, rem = r - band * per_band;
    const int bh = min(kResidentBand, tiles_y - band * kResidentBand);
    tx = rem / bh;
    ty = band * kResidentBand + (rem - tx * bh);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW;
  const float* a = im0 + (size_t)n * d * HW;
  const float* q = im1 + (size_t)n * d * HW;
  const float* fl = flow + (size_t)n * fc * HW;
  const int x = tx * kTW + lane, y = ty * kTH + wave;
  const bool valid = x < W && y < H;
  TilePx px;
  int minx = INT_MAX, maxx = INT_MIN, miny = INT_MAX, maxy = INT_MIN;
  locate(px, fl, HW, H, W, x, y, valid, minx, maxx, miny, maxy);
  const Box box = block_box(minx, maxx, miny, maxy, red, kElems);
  place(px, box, W);

  // window elements of this thread: e = threadIdx.x + 256 k, row e / w, column e % w (exact in float for these sizes).
  // Elements past the window's end re-read its first element: every load and LDS access of the channel loop is
  // unconditional, so the loads of D channels stay in flight (no branch between a load and its use).
  const int count = box.w * box.h;
  unsigned goff[kPer];
  const float inv_w = 1.0f / (float)max(box.w, 1);
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int e = threadIdx.x + 256 * k;
    const int r = (int)(((float)e + 0.5f) * inv_w);
    goff[k] = e < count ? (unsigned)(r * W + (e - r * box.w)) : 0u;
  }
  const bool near = px.inside && !px.far;
  unsigned lo[5];  // LDS offsets of the taps (0 for a pixel that does not read the window)
#pragma unroll
  for (int k = 0; k < 5; k++) lo[k] = near ? px.o[k] : 0u;
  const float* corner = q + (size_t)box.y0 * W + box.x0;
  // D channels in flight per thread: window elements in regs, the pixel's value of the first map in av
  float regs[D][kPer], av[D];
  auto fetch = [&](int c, float (&r)[kPer], float& first) {
    const float* src = corner + (size_t)c * HW;
#pragma unroll
    for (int k = 0; k < kPer; k++) r[k] = src[goff[k]];
    first = a[(size_t)c * HW + px.p];
  };
  auto stash = [&](const float (&r)[kPer], float* buf) {
#pragma unroll
    for (int k = 0; k < kPer; k++) buf[threadIdx.x + 256 * k] = r[k];
  };

  float tap[DMAX][5];
  float cost[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
  // No load sits behind a condition that the compiler cannot resolve (it would have to wait for every load in flight
  // at each join): past the last channel the loads re-read the last channel and the stores rewrite the idle buffer.
#pragma unroll
  for (int j = 0; j < D; j++) fetch(FULL ? j : min(j, d - 1), regs[j], av[j]);
  stash(regs[0], win[0]);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < DMAX; c++) {
    if (FULL || c < d) {  // the same for the whole block
      const float a_cur = av[c % D];
      if (!FULL || c + D < DMAX)  // this set of registers went to LDS one channel ago
        fetch(FULL ? c + D : min(c + D, d - 1), regs[c % D], av[c % D]);
#pragma unroll
      for (int k = 0; k < 5; k++) tap[c][k] = win[c & 1][lo[k]];
#pragma unroll
      for (int k = 0; k < 5; k++) cost[k] += a_cur * tap[c][k];  // QF.cu:63-71
      if (!FULL || c + 1 < DMAX) stash(regs[(c + 1) % D], win[(c + 1) & 1]);
      __syncthreads();
    }
  }
  if (px.inside && px.far) {  // taps outside the window's capacity: the same sums from memory
    const int xm = max(px.ix - 1, 0), ym = max(px.iy - 1, 0), xp = min(px.ix + 1, W - 1), yp = min(px.iy + 1, H - 1);
    const unsigned fo[5] = {(unsigned)px.iy * W + px.ix, (unsigned)px.iy * W + xp, (unsigned)px.iy * W + xm,
                            (unsigned)yp * W + px.ix, (unsigned)ym * W + px.ix};  // taps 00, 0p, 0m, p0, m0
#pragma unroll
    for (int k = 0; k < 5; k++) cost[k] = 0.f;
#pragma unroll
    for (int c = 0; c < DMAX; c++) {
      if (c < d) {
        const float a_cur = a[(size_t)c * HW + px.p];
#pragma unroll
        for (int k = 0; k < 5; k++) tap[c][k] = q[(size_t)c * HW + fo[k]];
#pragma unroll
        for (int k = 0; k < 5; k++) cost[k] += a_cur * tap[c][k];
      }
    }
  }

  float* G0 = res + (size_t)n * d * HW;
  if (!px.inside) {
    if (valid)
      for (int cc = 0; cc < d; cc++) G0[(size_t)cc * HW + px.p] = 0.f;
    return;
  }
  Fit f;
  f.inside = true;
  f.validX = f.validY = 0;
  f.c00 = f.ax = f.ay = f.bx = f.by = f.fx = f.fy = 0.f;
  finish_fit(f, cost[0], cost[1], cost[3], cost[2], cost[4], px.ix, px.iy, H, W);
  const Factors kf = scatter_factors(f, gin, n, HW, px.p);
  const long long t = (long long)n * HW + px.p;
  store_source(ws, kf, P, (long long)n * HW, t, (long long)px.iy * W + px.ix, px.p);
#pragma unroll
  for (int c = 0; c < DMAX; c++) {
    if (c < d) {
      float g;
      if (kf.any_valid)  // QF.cu:286-290
        g = 0.5 * (tap[c][0] * kf.k00 + tap[c][1] * kf.k0p + tap[c][2] * kf.k0m + tap[c][3] * kf.kp0 + tap[c][4] * kf.km0);
      else  // QF.cu:295
        g = tap[c][0] * kf.dFds;
      __builtin_nontemporal_store(g, &G0[(size_t)c * HW + px.p]);  // (the caller reads it, later: kept out of the caches, it leaves them to the windows)
    }
  }
}

// The forward pass, and pass A of the backward pass when the forward pass has left its five costs per pixel, with everything
// the channel loop reads coming from memory straight into LDS (global_load_lds): the window of the second map and, forward, the
// tile's own pixels of the first.  No load of the loop has a register as its target, so nothing but the ring's own count is
// waited for, and one barrier per two channels is all the synchronisation.  With the costs at hand pass A streams the second map
// once and keeps no taps: resident in registers they allow two wavefronts per SIMD and every map is read twice.
// A pixel whose taps leave the window's capacity is worked out from memory behind the loop.
// Bound by memory.  4 x 32 x 384 x 1248, us: forward 153 -> 121 (590 MB at 4.9 TB/s), with the costs stored 129; pass A 268 -> 158;
// 2 x 64 x 192 x 624 forward + backward 222 -> 131, 2 x 48 x 448 x 1280 660 -> 413.  With 4 pixels of noise on the flow (a fifth of
// the pixels outside the window) 1230 -> 1015, with 12 (nearly all) as before.
constexpr int kRingElems = 9216;   // floats of LDS for the ring: four blocks per CU
constexpr int kFarThreads = 128;

// Reads of LDS issued together and waited for once, as one block the compiler does not look into: before an LDS read that it
// sees, it waits for the loads into LDS that may alias it, and with the buffers of a ring it takes that to be all of them -- the
// whole prefetch queue.  The caller has waited for the buffer's own loads.
constexpr int kPairs = 12;
__device__ __forceinline__ void lds_read12(const unsigned (&a)[kPairs], float (&v)[kPairs]) {  // (byte addresses)
  asm volatile(
      "ds_read_b32 %0, %12\n\t"
      "ds_read_b32 %1, %13\n\t"
      "ds_read_b32 %2, %14\n\t"
      "ds_read_b32 %3, %15\n\t"
      "ds_read_b32 %4, %16\n\t"
      "ds_read_b32 %5, %17\n\t"
      "ds_read_b32 %6, %18\n\t"
      "ds_read_b32 %7, %19\n\t"
      "ds_read_b32 %8, %20\n\t"
      "ds_read_b32 %9, %21\n\t"
      "ds_read_b32 %10, %22\n\t"
      "ds_read_b32 %11, %23\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
        "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]), "v"(a[8]), "v"(a[9]),
        "v"(a[10]), "v"(a[11])
      : "memory");
}
// the same from two channels' windows, STRIDE x 64 floats apart: each read fetches an element of both
typedef float float2v __attribute__((ext_vector_type(2)));
template <int STRIDE>
__device__ __forceinline__ void lds_read12(const unsigned (&a)[12], float2v (&v)[12]) {  // (byte addresses)
  static_assert(STRIDE < 256, "the offset is eight bits wide");
  asm volatile(
      "ds_read2st64_b32 %0, %12 offset1:%24\n\t"
      "ds_read2st64_b32 %1, %13 offset1:%24\n\t"
      "ds_read2st64_b32 %2, %14 offset1:%24\n\t"
      "ds_read2st64_b32 %3, %15 offset1:%24\n\t"
      "ds_read2st64_b32 %4, %16 offset1:%24\n\t"
      "ds_read2st64_b32 %5, %17 offset1:%24\n\t"
      "ds_read2st64_b32 %6, %18 offset1:%24\n\t"
      "ds_read2st64_b32 %7, %19 offset1:%24\n\t"
      "ds_read2st64_b32 %8, %20 offset1:%24\n\t"
      "ds_read2st64_b32 %9, %21 offset1:%24\n\t"
      "ds_read2st64_b32 %10, %22 offset1:%24\n\t"
      "ds_read2st64_b32 %11, %23 offset1:%24\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
        "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]), "v"(a[8]), "v"(a[9]),
        "v"(a[10]), "v"(a[11]), "n"(STRIDE)
      : "memory");
}
template <int STRIDE>
__device__ __forceinline__ void lds_read10(const unsigned (&a)[10], float2v (&v)[10]) {  // (byte addresses)
  static_assert(STRIDE < 256, "the offset is eight bits wide");
  asm volatile(
      "ds_read2st64_b32 %0, %10 offset1:%20\n\t"
      "ds_read2st64_b32 %1, %11 offset1:%20\n\t"
      "ds_read2st64_b32 %2, %12 offset1:%20\n\t"
      "ds_read2st64_b32 %3, %13 offset1:%20\n\t"
      "ds_read2st64_b32 %4, %14 offset1:%20\n\t"
      "ds_read2st64_b32 %5, %15 offset1:%20\n\t"
      "ds_read2st64_b32 %6, %16 offset1:%20\n\t"
      "ds_read2st64_b32 %7, %17 offset1:%20\n\t"
      "ds_read2st64_b32 %8, %18 offset1:%20\n\t"
      "ds_read2st64_b32 %9, %19 offset1:%20\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7]),
        "=&v"(v[8]), "=&v"(v[9])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]), "v"(a[8]), "v"(a[9]), "n"(STRIDE)
      : "memory");
}

// Streams the windows of planes q[0 .. d) (and, FIRST, the tile's pixels of planes a[0 .. d)) through STAGES buffers of CH
// channels each: while one is consumed, STAGES - 1 more are on their way.  Loads return in order: when at most the loads of
// STAGES - 2 buffers are outstanding, the one at hand has landed (a wavefront's stores in between make the wait longer, never
// shorter).  A buffer is refilled one barrier after its consumption.  consume(c, two, buffer's byte address, own pixels' offset in
// floats, distance of the channels / 64): channel c and, CH = 2 and `two`, c + 1 (else the second is the last channel once more).
// Two channels at a time halve the reads and the barriers; with the first map in the ring as well they leave it too few buffers
// (forward 4 x 32 x 384 x 1248 121 / 126 us; pass A 160 / 158, gather pass 168 / 160).
template <int PX, int PER, int STAGES, int CH, bool FIRST, typename Consume>
__device__ __forceinline__ void ring_pass_of(const float* __restrict__ q, const float* __restrict__ a, const unsigned (&pix)[PX], int d,
                                             size_t HW, int W, const Box& box, float* ring, Consume consume) {
  typedef const __attribute__((address_space(1))) void* GlobalPtr;
  typedef __attribute__((address_space(3))) void* LdsPtr;
  constexpr int kLoads = PER + (FIRST ? PX : 0), kChannel = 256 * kLoads, kStage = CH * kChannel;
  static_assert(kStage * STAGES <= kRingElems && STAGES >= 2 && (STAGES - 2) * CH * kLoads < 63, "the ring's space; the counter's range");
  const int count = box.w * box.h;
  unsigned goff[PER];
  const float inv_w = 1.0f / (float)max(box.w, 1);
#pragma unroll
  for (int k = 0; k < PER; k++) {  // (row e / w, column e % w, exact in float for these sizes; past the window: its first element)
    const int e = threadIdx.x + 256 * k;
    const int r = (int)(((float)e + 0.5f) * inv_w);
    goff[k] = e < count ? (unsigned)(r * W + (e - r * box.w)) : 0u;
  }
  const float* corner = q + (size_t)box.y0 * W + box.x0;
  const int wave_first = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & ~63u));
  auto fetch = [&](int group, float* buf) {
#pragma unroll
    for (int u = 0; u < CH; u++) {
      const int c = min(CH * group + u, d - 1);
      const float* src = corner + (size_t)c * HW;
      float* to = buf + u * kChannel + wave_first;
#pragma unroll
      for (int k = 0; k < PER; k++) __builtin_amdgcn_global_load_lds((GlobalPtr)(src + goff[k]), (LdsPtr)(to + 256 * k), 4, 0, 0);
      if (FIRST) {
        const float* own = a + (size_t)c * HW;
#pragma unroll
        for (int i = 0; i < PX; i++)
          __builtin_amdgcn_global_load_lds((GlobalPtr)(own + pix[i]), (LdsPtr)(to + 256 * (PER + i)), 4, 0, 0);
      }
    }
  };
  // (what the wavefront has in flight already is not the ring's: the count starts from nothing)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int groups = (d + CH - 1) / CH;
#pragma unroll
  for (int c = 0; c < STAGES - 1; c++)
    if (c < groups) fetch(c, ring + c * kStage);
  int at = 0, refill = STAGES - 1;
  for (int c = 0; c < groups; c++) {
    if (c + STAGES - 2 < groups) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((STAGES - 2) * CH * kLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    if (c + STAGES - 1 < groups) fetch(c + STAGES - 1, ring + refill * kStage);
    consume(CH * c, CH * c + 1 < d, (unsigned)(size_t)(const __attribute__((address_space(3))) float*)(ring + at * kStage), 256u * PER,
            std::integral_constant<int, kChannel / 64>{});
    at = at + 1 == STAGES ? 0 : at + 1;
    refill = refill + 1 == STAGES ? 0 : refill + 1;
  }
}
template <int PX, bool FIRST, typename Consume>
__device__ __forceinline__ void ring_pass(const float* __restrict__ q, const float* __restrict__ a, const unsigned (&pix)[PX], int d,
                                          size_t HW, int W, const Box& box, float* ring, Consume consume) {
  static_assert(PX == 2 && TileCfg<PX>::ELEMS == 9 * 256, "loads per thread: 4 to 9");
  const int count = __builtin_amdgcn_readfirstlane(box.w * box.h);
  constexpr int CH = FIRST ? 1 : 2;
  if (count <= 4 * 256) ring_pass_of<PX, 4, FIRST ? 5 : 4, CH, FIRST>(q, a, pix, d, HW, W, box, ring, consume);
  else if (count <= 6 * 256) ring_pass_of<PX, 6, FIRST ? 4 : 3, CH, FIRST>(q, a, pix, d, HW, W, box, ring, consume);
  else ring_pass_of<PX, 9, FIRST ? 3 : 2, CH, FIRST>(q, a, pix, d, HW, W, box, ring, consume);
}

// MODE 0: the forward pass (costs: its five sums per pixel, a plane of N * H * W each, or null).  MODE 1: pass A from the costs.
template <int MODE>
__global__ __launch_bounds__(256) void quadfit_ring_tiles(const float* __restrict__ im0, const float* __restrict__ im1,
                                                          const float* __restrict__ flow, const float* __restrict__ gin,
                                                          float* __restrict__ costs, float* __restrict__ res, QfWorkspace ws, int N,
                                                          int d, int H, int W, int fc, int tiles_x, int tiles_y) {
  constexpr int PX = kPxTile, kTH = TileCfg<PX>::TH;
  __shared__ __align__(16) float ring[kRingElems];
  __shared__ int red[16];
  int n, tx, ty;
  if (!tile_of_block(N, tiles_x, tiles_y, n, tx, ty)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW, base = (long long)n * HW;
  const float* a = im0 + (size_t)n * d * HW;
  const float* q = im1 + (size_t)n * d * HW;
  const float* fl = flow + (size_t)n * fc * HW;
  const int x = tx * kTW + lane;
  TilePx px[PX];
  bool valid[PX];
  unsigned pix[PX];
  int minx = INT_MAX, maxx = INT_MIN, miny = INT_MAX, maxy = INT_MIN;
#pragma unroll
  for (int i = 0; i < PX; i++) {
    const int y = ty * kTH + wave * PX + i;
    valid[i] = x < W && y < H;
    locate(px[i], fl, HW, H, W, x, y, valid[i], minx, maxx, miny, maxy);
    pix[i] = px[i].p;
  }
  Factors k[PX];
  auto factors = [&](int i, const float (&c)[5]) {  // finished fit of pixel i
    Fit f;
    f.inside = px[i].inside;
    f.validX = f.validY = 0;
    f.c00 = f.ax = f.ay = f.bx = f.by = f.fx = f.fy = 0.f;
    if (px[i].inside) finish_fit(f, c[0], c[1], c[3], c[2], c[4], px[i].ix, px[i].iy, H, W);
    return f;
  };
  if (MODE == 1) {
#pragma unroll
    for (int i = 0; i < PX; i++) {
      k[i] = Factors{};
      if (!px[i].inside) continue;
      const long long t = base + pix[i];
      float c[5];
#pragma unroll
      for (int j = 0; j < 5; j++) c[j] = costs[j * P + t];
      k[i] = scatter_factors(factors(i, c), gin, n, HW, pix[i]);
      store_source(ws, k[i], P, base, t, (long long)px[i].iy * W + px[i].ix, pix[i]);
    }
  }
  const Box box = block_box(minx, maxx, miny, maxy, red, TileCfg<PX>::ELEMS);
  unsigned lo[PX][5];
  bool far[PX], any_far = false;
#pragma unroll
  for (int i = 0; i < PX; i++) {
    place(px[i], box, W);
    far[i] = px[i].far;
    any_far = any_far || far[i];
#pragma unroll
    for (int j = 0; j < 5; j++) lo[i][j] = px[i].inside && !far[i] ? 4u * px[i].o[j] : 0u;
  }
  // where the window holds few pixels of the tile it is not worth its loads: all of them from memory then
  const bool windowless = __syncthreads_count(any_far) > kFarThreads;
  any_far = __ballot(any_far) != 0;
  // taps from memory, both pixels of the lane together; use(cc, first map, taps) per channel.  Few pixels: four channels in flight;
  // a whole tile of scattered taps: one, the lines of a channel's taps then stay in the cache until they have been used
  // (4 x 32 x 384 x 1248, 12 pixels of noise on the flow: 630 us with one, 655 with two, 766 with four; 4 pixels: 211, 214, 205).
  auto from_memory_of = [&](auto ahead, auto use) {
    constexpr int kFarAhead = decltype(ahead)::value;
    unsigned o[PX][5];
#pragma unroll
    for (int i = 0; i < PX; i++) {
      far[i] = far[i] || (windowless && px[i].inside);
      const int ix = far[i] ? px[i].ix : 0, iy = far[i] ? px[i].iy : 0;  // (other pixels read the plane's first corner)
      o[i][0] = (unsigned)iy * W + ix;
      o[i][1] = (unsigned)iy * W + min(ix + 1, W - 1);
      o[i][2] = (unsigned)iy * W + max(ix - 1, 0);
      o[i][3] = (unsigned)min(iy + 1, H - 1) * W + ix;
      o[i][4] = (unsigned)max(iy - 1, 0) * W + ix;
    }
    for (int c0 = 0; c0 < d; c0 += kFarAhead) {
      float v[kFarAhead][PX], t[kFarAhead][PX][5];
#pragma unroll
      for (int u = 0; u < kFarAhead; u++) {
        const size_t plane = (size_t)min(c0 + u, d - 1) * HW;
#pragma unroll
        for (int i = 0; i < PX; i++) {
          if (MODE == 0) v[u][i] = a[plane + pix[i]];
#pragma unroll
          for (int j = 0; j < 5; j++) t[u][i][j] = q[plane + o[i][j]];
        }
      }
#pragma unroll
      for (int u = 0; u < kFarAhead; u++)
        if (c0 + u < d) use(c0 + u, v[u], t[u]);
    }
  };
  auto from_memory = [&](auto use) {
    if (windowless) from_memory_of(std::integral_constant<int, 1>{}, use);
    else if (any_far) from_memory_of(std::integral_constant<int, 4>{}, use);
  };
  if (MODE == 0) {
    float cost[PX][5];
#pragma unroll
    for (int i = 0; i < PX; i++)
#pragma unroll
      for (int j = 0; j < 5; j++) cost[i][j] = 0.f;
    if (!windowless)
      ring_pass<PX, true>(q, a, pix, d, HW, W, box, ring, [&](int, bool, unsigned buf, unsigned own, auto) {
        unsigned addr[kPairs];
        float v[kPairs];
#pragma unroll
        for (int i = 0; i < PX; i++) {
#pragma unroll
          for (int j = 0; j < 5; j++) addr[5 * i + j] = buf + lo[i][j];
          addr[10 + i] = buf + 4u * (own + 256u * i + threadIdx.x);
        }
        lds_read12(addr, v);
#pragma unroll
        for (int i = 0; i < PX; i++)
#pragma unroll
          for (int j = 0; j < 5; j++) cost[i][j] += v[10 + i] * v[5 * i + j];  // QF.cu:63-71
      });
    if (any_far || windowless) {
      float sum[PX][5];
#pragma unroll
      for (int i = 0; i < PX; i++)
#pragma unroll
        for (int j = 0; j < 5; j++) sum[i][j] = 0.f;
      from_memory([&](int, const float (&v)[PX], const float (&t)[PX][5]) {
#pragma unroll
        for (int i = 0; i < PX; i++)
#pragma unroll
          for (int j = 0; j < 5; j++) sum[i][j] += v[i] * t[i][j];
      });
#pragma unroll
      for (int i = 0; i < PX; i++)
#pragma unroll
        for (int j = 0; j < 5; j++) cost[i][j] = far[i] ? sum[i][j] : cost[i][j];
    }
#pragma unroll
    for (int i = 0; i < PX; i++) {
      if (!valid[i]) continue;
      const Fit f = factors(i, cost[i]);
      float* o = res + (size_t)n * 3 * HW + pix[i];
      float score = 0.f;
      if (f.inside)  // QF.cu:136
        score = f.ax * f.fx * f.fx + f.bx * f.fx + f.c00 + f.ay * f.fy * f.fy + f.by * f.fy;
      o[0] = f.fx;
      o[HW] = f.fy;
      o[2 * HW] = score;
      if (costs) {
#pragma unroll
        for (int j = 0; j < 5; j++) __builtin_nontemporal_store(cost[i][j], &costs[j * P + base + pix[i]]);
      }
    }
    return;
  }
  float* G0 = res + (size_t)n * d * HW;
  auto gradient = [&](int i, const float* t) -> float {
    if (!px[i].inside) return 0.f;
    if (k[i].any_valid)  // QF.cu:286-290
      return 0.5 * (t[0] * k[i].k00 + t[1] * k[i].k0p + t[2] * k[i].k0m + t[3] * k[i].kp0 + t[4] * k[i].km0);
    return t[0] * k[i].dFds;  // QF.cu:295
  };
  if (!windowless)
    ring_pass<PX, false>(q, nullptr, pix, d, HW, W, box, ring, [&](int cc, bool two, unsigned buf, unsigned, auto stride) {
      unsigned addr[10];
      float2v v[10];
#pragma unroll
      for (int i = 0; i < PX; i++)
#pragma unroll
        for (int j = 0; j < 5; j++) addr[5 * i + j] = buf + lo[i][j];
      lds_read10<decltype(stride)::value>(addr, v);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        if (u == 1 && !two) break;
#pragma unroll
        for (int i = 0; i < PX; i++) {
          const float t[5] = {v[5 * i][u], v[5 * i + 1][u], v[5 * i + 2][u], v[5 * i + 3][u], v[5 * i + 4][u]};
          const float g = gradient(i, t);
          if (valid[i] && !far[i]) __builtin_nontemporal_store(g, &G0[(size_t)(cc + u) * HW + pix[i]]);
        }
      }
    });
  from_memory([&](int cc, const float (&)[PX], const float (&t)[PX][5]) {
#pragma unroll
    for (int i = 0; i < PX; i++) {
      const float g = gradient(i, t[i]);
      if (far[i] || (windowless && valid[i])) __builtin_nontemporal_store(g, &G0[(size_t)cc * HW + pix[i]]);
    }
  });
}

// The same two passes for images with too few tiles to fill the chip.  On 64 x 96 x 312 the tiled kernels are 60 blocks
// that walk 64 channels one barrier at a time (48 us forward, 98 us pass A).  Here a block owns 64 pixels of a row and its
// four wavefronts share the CHANNELS: a wavefront reads the taps of eight of 32 channels straight from memory -- 48 loads in
// flight per lane -- and leaves the five products of each in LDS; then the products are summed over the channels in the
// reference's order (QF.cu:63-71: the sum is a chain, the products are not), one tap per wavefront.  NC > 0: d <= 32 NC
// channels, whose taps the backward pass keeps in registers for the gradient wrt the first map; NC = 0: any d, read again.
constexpr int kSplitChunk = 32, kSplitPer = kSplitChunk / 4;

template <int MODE, int NC>
__global__ __launch_bounds__(256) void quadfit_split(const float* __restrict__ im0, const float* __restrict__ im1,
                                                     const float* __restrict__ flow, const float* __restrict__ gin,
                                                     float* __restrict__ res, QfWorkspace ws, int N, int d, int H, int W,
                                                     int fc, int tiles_x, int tiles_y) {
  __shared__ float prod[kSplitChunk][5][64];
  __shared__ float sums[5][64];
  int n, tx, y;
  if (!tile_of_block(N, tiles_x, tiles_y, n, tx, y)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t HW = (size_t)H * W;
  const float* a = im0 + (size_t)n * d * HW;
  const float* q = im1 + (size_t)n * d * HW;
  const int x = tx * 64 + lane;
  const bool valid = x < W;
  TilePx px;
  int unused0 = 0, unused1 = 0, unused2 = 0, unused3 = 0;
  locate(px, flow + (size_t)n * fc * HW, HW, H, W, x, y, valid, unused0, unused1, unused2, unused3);
  const unsigned row = (unsigned)px.iy * W;  // (a pixel that is not inside reads the plane's first value; its sums are not used)
  const unsigned o[5] = {row + px.ix, row + px.xp, row + px.xm, (unsigned)px.yp * W + px.ix, (unsigned)px.ym * W + px.ix};
  float tap[NC > 0 ? NC * kSplitPer : kSplitPer][5];
  float cost[2] = {0.f, 0.f};  // this wavefront's tap; wavefront 0 also sums tap 4
  auto chunk = [&](int c0, float (*t)[5]) {
    float v[kSplitPer];
#pragma unroll
    for (int j = 0; j < kSplitPer; j++) {
      const size_t plane = (size_t)min(c0 + wave * kSplitPer + j, d - 1) * HW;
      v[j] = a[plane + px.p];
#pragma unroll
      for (int k = 0; k < 5; k++) t[j][k] = q[plane + o[k]];
    }
#pragma unroll
    for (int j = 0; j < kSplitPer; j++)
#pragma unroll
      for (int k = 0; k < 5; k++) prod[wave * kSplitPer + j][k][lane] = v[j] * t[j][k];
    __syncthreads();
    const int nc = min(kSplitChunk, d - c0);
    for (int c = 0; c < nc; c++) cost[0] += prod[c][wave][lane];
    if (wave == 0)
      for (int c = 0; c < nc; c++) cost[1] += prod[c][4][lane];
  };
  if (NC > 0) {
#pragma unroll
    for (int b = 0; b < NC; b++) {
      if (b * kSplitChunk < d) {
        if (b > 0) __syncthreads();
        chunk(b * kSplitChunk, tap + b * kSplitPer);
      }
    }
  } else {
    for (int c0 = 0; c0 < d; c0 += kSplitChunk) {
      if (c0 > 0) __syncthreads();
      chunk(c0, tap);
    }
  }
  sums[wave][lane] = cost[0];
  if (wave == 0) sums[4][lane] = cost[1];
  __syncthreads();
  Fit f;
  f.inside = px.inside;
  f.validX = f.validY = 0;
  f.c00 = f.ax = f.ay = f.bx = f.by = f.fx = f.fy = 0.f;
  if (px.inside) finish_fit(f, sums[0][lane], sums[1][lane], sums[3][lane], sums[2][lane], sums[4][lane], px.ix, px.iy, H, W);
  if (MODE == 0) {
    if (wave != 0 || !valid) return;
    float* out = res + (size_t)n * 3 * HW + px.p;
    float score = 0.f;
    if (f.inside)  // QF.cu:136
      score = f.ax * f.fx * f.fx + f.bx * f.fx + f.c00 + f.ay * f.fy * f.fy + f.by * f.fy;
    out[0] = f.fx;
    out[HW] = f.fy;
    out[2 * HW] = score;
    return;
  }
  if (!valid) return;
  Factors kf{};
  if (px.inside) kf = scatter_factors(f, gin, n, HW, px.p);
  if (wave == 0 && px.inside) {
    const long long P = (long long)N * HW, t = (long long)n * HW + px.p;
    store_source(ws, kf, P, (long long)n * HW, t, o[0], px.p);
  }
  float* G0 = res + (size_t)n * d * HW;
  auto gradient = [&](int c0, const float (*t)[5]) {
#pragma unroll
    for (int j = 0; j < kSplitPer; j++) {
      const int c = c0 + wave * kSplitPer + j;
      if (c < d) {
        float g = 0.f;
        if (px.inside) {
          if (kf.any_valid)  // QF.cu:286-290
            g = 0.5 * (t[j][0] * kf.k00 + t[j][1] * kf.k0p + t[j][2] * kf.k0m + t[j][3] * kf.kp0 + t[j][4] * kf.km0);
          else  // QF.cu:295
            g = t[j][0] * kf.dFds;
        }
        G0[(size_t)c * HW + px.p] = g;
      }
    }
  };
  if (NC > 0) {
#pragma unroll
    for (int b = 0; b < NC; b++) gradient(b * kSplitChunk, tap + b * kSplitPer);
  } else {
    for (int c0 = 0; c0 < d; c0 += kSplitChunk) {
#pragma unroll
      for (int j = 0; j < kSplitPer; j++) {
        const size_t plane = (size_t)min(c0 + wave * kSplitPer + j, d - 1) * HW;
#pragma unroll
        for (int k = 0; k < 5; k++) tap[j][k] = q[plane + o[k]];
      }
      gradient(c0, tap);
    }
  }
}

// Pass B of the backward pass on tiles of target pixels: the (source, coefficient) pairs of every pixel are
// collected once; per channel the window of the FIRST feature map that covers the tile's sources is
// staged in LDS and the pairs are summed from it.
constexpr int kPxGather = 2;

template <int PX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void quadfit_gather_tiles(const float* __restrict__ im0, float* __restrict__ g1, QfWorkspace ws,
                                                            int N, int d_all, int per_group, int H, int W, int tiles_x, int tiles_y) {
  // blockIdx.y: this block's group of per_group channels (launches that would leave the chip short of blocks are split by
  // channel; every group collects the tile's pairs for itself)
  const int d_lo = (int)blockIdx.y * per_group, d = min(per_group, d_all - d_lo);
  constexpr int kTH = TileCfg<PX>::TH;
  __shared__ __align__(16) float ring[kRingElems];
  __shared__ int red[16];
  int n, tx, ty;
  if (!tile_of_block(N, tiles_x, tiles_y, n, tx, ty)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t HW = (size_t)H * W;
  const long long P = (long long)N * HW, base = (long long)n * HW;
  const float* a = im0 + ((size_t)n * d_all + d_lo) * HW;
  float* G1 = g1 + ((size_t)n * d_all + d_lo) * HW;
  const int x = tx * kTW + lane;
  const float inv_w = 1.0f / (float)W;
  bool valid[PX];
  unsigned pix[PX];
  int np[PX];
  unsigned off[PX][kPairs];  // packed (y << 16 | x) of the source, then its offset in the window
  float cf[PX][kPairs];
  int minx = INT_MAX, maxx = INT_MIN, miny = INT_MAX, maxy = INT_MIN;
  // (position whose sources reach a pixel, tap they reach it with), as an offset in the plane; a neighbour outside the
  // image has no list.  Three reads stand behind every pair -- list length, list, coefficient.  They are issued
  // unconditionally and in batches (an absent list reads the pixel's own, an unused entry coefficient 0 of the sample):
  // lengths and lists of all pixels of the lane together, then the coefficients of one pixel at a time -- three round
  // trips to memory; behind `if (cnt > 0)` / `if (s < cnt)` each read waits for the one before it, some fifty in a row.
  static_assert(kRingElems >= 4 * 2 * 64 * kPairs, "the ring holds the pairs of 64 pixels per wavefront");
  float2* const front = reinterpret_cast<float2*>(ring) + 64 * kPairs * wave + lane;
  int cnt[PX][5];
  int4 sl[PX][5];
#pragma unroll
  for (int i = 0; i < PX; i++) {
    const int y = ty * kTH + wave * PX + i;
    valid[i] = x < W && y < H;
    pix[i] = valid[i] ? (unsigned)y * W + x : 0u;
    np[i] = 0;
    const bool has[5] = {valid[i], valid[i] && x > 0, valid[i] && x < W - 1, valid[i] && y > 0, valid[i] && y < H - 1};
    const int step[5] = {0, -1, 1, -W, W};
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const long long ctr = base + (long long)pix[i] + (has[k] ? step[k] : 0);
      cnt[i][k] = ws.count[ctr];
      sl[i][k] = *reinterpret_cast<const int4*>(ws.slots + ctr * kSlots);
    }
  }
#pragma unroll
  for (int i = 0; i < PX; i++) {
    const int y = ty * kTH + wave * PX + i;
    const bool has[5] = {valid[i], valid[i] && x > 0, valid[i] && x < W - 1, valid[i] && y > 0, valid[i] && y < H - 1};
    float cv[5][kSlots];
    unsigned spv[5][kSlots];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      cnt[i][k] = has[k] ? min(cnt[i][k], kSlots) : 0;
      const int sv[4] = {sl[i][k].x, sl[i][k].y, sl[i][k].z, sl[i][k].w};
#pragma unroll
      for (int s = 0; s < kSlots; s++) {
        spv[k][s] = s < cnt[i][k] ? (unsigned)sv[s] : 0u;  // source pixel, offset in its plane
        cv[k][s] = ws.coef[(long long)k * P + base + spv[k][s]];
      }
    }
    // (the values are pinned here, all of them: left alone, the optimizer moves each read back behind the branch that
    // uses it)
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
      for (int s = 0; s < kSlots; s++) asm volatile("" : "+v"(cv[k][s]));
    // The pairs that exist, moved to the front through the wavefront's own LDS (the windows' space, still unused): a
    // write at a running index per entry.  (As selects between registers this took twelve compares and moves for each of
    // the twenty entries: a third of the launch.)
#pragma unroll
    for (int k = 0; k < 5; k++) {
#pragma unroll
      for (int s = 0; s < kSlots; s++) {
        if (s < cnt[i][k]) {
          if (np[i] < kPairs) front[np[i] * 64] = make_float2(__uint_as_float(spv[k][s]), cv[k][s]);
          np[i]++;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kPairs; j++) {
      const float2 e = front[j * 64];
      const bool used = j < np[i];
      const unsigned sp = used ? __float_as_uint(e.x) : 0u;  // (below 2^24: the float quotient is off by one at most)
      int sy = (int)((float)sp * inv_w), sx = (int)sp - sy * W;
      if (sx < 0) { sy--; sx += W; }
      if (sx >= W) { sy++; sx -= W; }
      off[i][j] = ((unsigned)sy << 16) | (unsigned)sx;
      cf[i][j] = used ? e.y : 0.f;
      if (used) {
        minx = min(minx, sx); maxx = max(maxx, sx);
        miny = min(miny, sy); maxy = max(maxy, sy);
      }
    }
  }
  const Box box = block_box(minx, maxx, miny, maxy, red, TileCfg<PX>::ELEMS);
  // A pixel with more pairs than registers, or with a source outside the window, is left to pass C.  (It used to walk its
  // lists here, three dependent reads per entry and channel: eighteen such pixels in 479232 made the launch 290 us instead
  // of 200 on 4 x 32 x 384 x 1248, and 581 us of 64 x 96 x 312, where one pixel in sixty-five is one.)
  bool slow[PX];
  unsigned need = 0;
#pragma unroll
  for (int i = 0; i < PX; i++) {
    slow[i] = np[i] > kPairs;
#pragma unroll
    for (int j = 0; j < kPairs; j++) {
      const int sx = off[i][j] & 0xffff, sy = off[i][j] >> 16;
      const bool used = j < np[i];
      if (used && !(sx - box.x0 < box.w && sy - box.y0 < box.h)) slow[i] = true;
      off[i][j] = used ? 4u * (unsigned)((sy - box.y0) * box.w + (sx - box.x0)) : 0u;
    }
#pragma unroll
    for (int j = 0; j < kPairs; j++) {
      if (slow[i]) {
        off[i][j] = 0u;
        cf[i][j] = 0.f;
      }
      if (__ballot(!slow[i] && j < np[i]) != 0) need |= 1u << j;  // pairs nobody in the wavefront has are skipped by a uniform branch
    }
    if (blockIdx.y == 0) {
      const bool listed = valid[i] && slow[i];
      const unsigned long long all = __ballot(listed);
      if (all) {
        int at = 0;
        if (lane == __builtin_ctzll(all)) at = atomicAdd(ws.slow_count, __popcll(all));
        at = __builtin_amdgcn_readlane(at, __builtin_ctzll(all));
        if (listed) ws.slow[at + __popcll(all & ((1ull << lane) - 1))] = (int)(base + pix[i]);
      }
    }
  }
  const unsigned none[PX] = {};
  ring_pass<PX, false>(a, nullptr, none, d, HW, W, box, ring, [&](int cc, bool two, unsigned buf, unsigned, auto stride) {
    // all window reads of a pixel are issued before the first product: a read inside the branch that skips an unused pair
    // is waited for on the spot, one LDS round trip after the other (an unused pair reads element 0, a broadcast)
#pragma unroll
    for (int i = 0; i < PX; i++) {
      unsigned addr[kPairs];
      float2v v[kPairs];
#pragma unroll
      for (int j = 0; j < kPairs; j++) addr[j] = buf + off[i][j];
      lds_read12<decltype(stride)::value>(addr, v);
      float acc[2] = {0.f, 0.f};
#pragma unroll
      for (int j = 0; j < kPairs; j++)
        if (need & (1u << j)) {
          acc[0] = __builtin_fmaf(v[j][0], cf[i][j], acc[0]);
          acc[1] = __builtin_fmaf(v[j][1], cf[i][j], acc[1]);
        }
      if (valid[i]) {
        __builtin_nontemporal_store(slow[i] ? 0.f : acc[0], &G1[(size_t)cc * HW + pix[i]]);
        if (two) __builtin_nontemporal_store(slow[i] ? 0.f : acc[1], &G1[(size_t)(cc + 1) * HW + pix[i]]);
      }
    }
  });
}

// Workgroup barrier that orders LDS traffic only: global loads issued before it stay in flight.
__device__ __forceinline__ void lds_only_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

#include "quadfit_image_kernels.h"

// ---------------------------------------------------------------------------------------------
// median
// ---------------------------------------------------------------------------------------------
constexpr int kBins = 32;  // bins per staged chunk
constexpr int kPitch = kBins + 1;

// 64 pixels x nb bins between HBM and the wavefront's LDS tile; lane -> (pixel 2i + lane/32, bin lane%32)
__device__ __forceinline__ void stage_in(const float* __restrict__ vol, float (*tile)[kPitch], long long p0, long long P,
                                         int D, int c0, int nb, int lane) {
  const int b = lane & 31, half = lane >> 5;
#pragma unroll 8
  for (int i = 0; i < 32; i++) {
    const int px = 2 * i + half;
    const long long qpx = p0 + px;
    float v = 0.f;
    if (qpx < P && b < nb) v = vol[qpx * D + c0 + b];
    tile[px][b] = v;
  }
}
__device__ __forceinline__ void stage_out(float* __restrict__ gvol, float (*tile)[kPitch], long long p0, long long P, int D,
                                          int c0, int nb, int lane) {
  const int b = lane & 31, half = lane >> 5;
#pragma unroll 8
  for (int i = 0; i < 32; i++) {
    const int px = 2 * i + half;
    const long long qpx = p0 + px;
    if (qpx < P && b < nb) gvol[qpx * D + c0 + b] = tile[px][b];
  }
}

struct Crossing {
  bool found;
  int c;
  float score, pmid, alpha;
};
// the walk of MM.cu:26-43 == MM.cu:59-75 over one staged chunk
__device__ __forceinline__ void walk(Crossing& s, const float* row, int c0, int nb) {
  if (s.found) return;
  for (int j = 0; j < nb; j++) {
    const float cScore = row[j];
    if (s.score < 0.5 && s.score + cScore >= 0.5) {
      s.alpha = (1. - 2. * s.score - cScore) / (2. * cScore);  // MM.cu:34
      s.pmid = cScore;
      s.c = c0 + j;
      s.found = true;
      return;
    }
    s.score = s.score + cScore;
  }
}

// MM.cu:17-44.  P = n*h*w pixels; out (n,2,h,w).
__global__ __launch_bounds__(256) void median_forward_kernel(const float* __restrict__ vol, float* __restrict__ out,
                                                             long long P, long long HW, int D) {
  __shared__ float tiles[4][64][kPitch];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long p0 = ((long long)blockIdx.x * 4 + wave) * 64;
  const long long p = p0 + lane;
  Crossing s{false, 0, 0.f, 1.f, 0.f};
  for (int c0 = 0; c0 < D; c0 += kBins) {
    const int nb = min(kBins, D - c0);
    stage_in(vol, tiles[wave], p0, P, D, c0, nb, lane);
    __syncthreads();
    walk(s, tiles[wave][lane], c0, nb);
    if (__syncthreads_and(s.found || p >= P)) break;
  }
  if (p < P) {
    const long long n = p / HW, q = p - n * HW;
    float med = 0.f, mass = 0.f;
    if (s.found) {
      med = (float)s.c - 0.f + s.alpha;  // MM.cu:35
      mass = s.pmid;
    }
    out[n * 2 * HW + q] = med;
    out[n * 2 * HW + HW + q] = mass;
  }
}

// MM.cu:46-93 for the 64 pixels from p0 on.  Pass 1 finds each pixel's crossing, pass 2 writes every bin's gradient.  (All
// wavefronts of the block, each with a tile and 64 pixels of its own.)
__device__ __forceinline__ void backward_from_bins(const float* __restrict__ vol, float* __restrict__ gvol, float (*tile)[kPitch],
                                                   long long p0, long long P, int D, int lane, float g0v, float g1v) {
  const long long p = p0 + lane;
  Crossing s{false, 0, 0.f, 1.f, 0.f};
  for (int c0 = 0; c0 < D; c0 += kBins) {
    const int nb = min(kBins, D - c0);
    stage_in(vol, tile, p0, P, D, c0, nb, lane);
    __syncthreads();
    walk(s, tile[lane], c0, nb);
    if (__syncthreads_and(s.found || p >= P)) break;
  }
  const float cross = g0v * s.alpha / (-s.pmid) + g1v;  // MM.cu:69
  const float neg = -g0v / (2. * s.pmid);               // MM.cu:85
  const float pos = +g0v / (2. * s.pmid);               // MM.cu:88
  float score = 0.f;
  for (int c0 = 0; c0 < D; c0 += kBins) {
    const int nb = min(kBins, D - c0);
    __syncthreads();
    stage_in(vol, tile, p0, P, D, c0, nb, lane);
    __syncthreads();
    float* row = tile[lane];
    for (int j = 0; j < nb; j++) {  // MM.cu:77-92; the crossing bin keeps the value of MM.cu:69
      const float cScore = row[j];
      float g = (s.found && c0 + j == s.c) ? cross : 0.f;
      if (score + cScore < 0.5) g = neg;
      else if (score >= 0.5) g = pos;
      row[j] = g;
      score = score + cScore;
    }
    __syncthreads();
    stage_out(gvol, tile, p0, P, D, c0, nb, lane);
  }
}

__global__ __launch_bounds__(256) void median_backward_kernel(const float* __restrict__ vol, const float* __restrict__ gin,
                                                              float* __restrict__ gvol, long long P, long long HW, int D) {
  __shared__ float tiles[4][64][kPitch];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long p0 = ((long long)blockIdx.x * 4 + wave) * 64;
  const long long p = p0 + lane;
  float g0v = 0.f, g1v = 0.f;
  if (p < P) {
    const long long n = p / HW, q = p - n * HW;
    g0v = gin[n * 2 * HW + q];
    g1v = gin[n * 2 * HW + HW + q];
  }
  backward_from_bins(vol, gvol, tiles[wave], p0, P, D, lane, g0v, g1v);
}

// ---------------------------------------------------------------------------------------------
// Median, whole histograms in LDS (up to 255 bins): the histograms of 64 consecutive pixels are one
// contiguous run of 64*D floats, staged with 16-byte loads into rows of odd pitch; each lane walks its
// row; the backward pass writes the gradients over the row and the run goes back out the same way.
// HBM sees the histogram once per pass.
// ---------------------------------------------------------------------------------------------
constexpr int kMaxRowBins = 255;
constexpr int kWalkAhead = 8;  // LDS reads in flight in the forward walk

// In: kBatch loads per lane are issued before the first of them is stored to LDS (a loop that stores each value right
// after its load waits for memory once per element: 9 round trips per wavefront at 33 bins where one or two suffice).
template <int VEC, bool OUT>
__device__ __forceinline__ void stage_rows(const float* __restrict__ src, float* __restrict__ dst, float* tile, int total,
                                           int D, int Dp, int lane) {
  constexpr int kStep = 64 * VEC;
  constexpr int kBatch = OUT ? 1 : 8;
  if (VEC == 4 && Dp == D) {  // odd bin counts need no padding: the tile is a plain copy of the run, 16 bytes per lane and step
    const int full = total & ~3;
    if (OUT) {
      for (int i = lane * 4; i < full; i += kStep) *reinterpret_cast<float4*>(dst + i) = *reinterpret_cast<const float4*>(tile + i);
      for (int i = full + lane; i < total; i += 64) dst[i] = tile[i];
    } else {
      for (int i = lane * 4; i < full; i += kStep * 8) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = *reinterpret_cast<const float4*>(src + (i + u * kStep < full ? i + u * kStep : 0));
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (i + u * kStep < full) *reinterpret_cast<float4*>(tile + i + u * kStep) = v[u];
      }
      for (int i = full + lane; i < total; i += 64) tile[i] = src[i];
    }
    return;
  }
  const int qs = kStep / D, rs = kStep - qs * D;
  int i = lane * VEC;
  int px = i / D, b = i - px * D;
  for (; i < total; i += kStep * kBatch) {
    float4 v4[kBatch];
    float v1[kBatch];
    if (!OUT) {  // unconditional loads (an index past the end re-reads the wavefront's first elements)
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const int iu = i + u * kStep;
        if (VEC == 4) v4[u] = *reinterpret_cast<const float4*>(src + (iu + 3 < total ? iu : 0));
        else v1[u] = src[iu < total ? iu : 0];
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
      const int iu = i + u * kStep;
      if (iu < total) {
        if (VEC == 4 && iu + 3 < total) {
          float* e[4];
          int pe = px, be = b;
#pragma unroll
          for (int k = 0; k < 4; k++) {
            e[k] = tile + pe * Dp + be;
            if (++be >= D) { be = 0; pe++; }
          }
          if (OUT) {
            float4 v;
            v.x = *e[0]; v.y = *e[1]; v.z = *e[2]; v.w = *e[3];
            *reinterpret_cast<float4*>(dst + iu) = v;
          } else {
            *e[0] = v4[u].x; *e[1] = v4[u].y; *e[2] = v4[u].z; *e[3] = v4[u].w;
          }
        } else {  // the run's last, partial vector (or VEC == 1)
          int pe = px, be = b;
          for (int k = 0; k < VEC && iu + k < total; k++) {
            if (OUT) dst[iu + k] = tile[pe * Dp + be];
            else tile[pe * Dp + be] = VEC == 4 ? src[iu + k] : v1[u];
            if (++be >= D) { be = 0; pe++; }
          }
        }
      }
      b += rs;
      px += qs;
      if (b >= D) { b -= D; px++; }
    }
  }
}

// The walk of MM.cu:26-43 == MM.cu:59-75 over a whole histogram, without the early exit.  The crossing bin's interpolation (a
// double division) is formed once, after the walk: inside the loop it would run in every iteration in which ANY lane of the
// wavefront crosses.  The comparisons against 0.5 are the reference's (a float promoted to double compares as the float does);
// in front of the crossing the running sum is below one half or a NaN, so the bin that brings it there is the crossing.
struct Walked {
  bool found;
  bool regular;  // every sum from the crossing on is at least one half (no crossing: no sum is a NaN)
  int cidx;
  float before, pmid;  // sum in front of the crossing bin, its mass
};
// What the walk does with one bin
template <bool CHECK>
__device__ __forceinline__ void walk_bin(Walked& s, float& run, float mass, int c) {
  const float sum = run + mass;
  const bool half = sum >= 0.5f, hit = half && !s.found;
  s.pmid = hit ? mass : s.pmid;
  s.cidx = hit ? c : s.cidx;
  s.before = hit ? run : s.before;
  if (CHECK) s.regular = s.regular && (half || !s.found);
  s.found = s.found || half;
  run = sum;
}
template <bool CHECK>
__device__ __forceinline__ Walked walk_histogram(const float* row, int D) {
  Walked s{false, true, 0, 0.f, 1.f};
  float run = 0.f;
#pragma unroll 4
  for (int c = 0; c < D; c++) walk_bin<CHECK>(s, run, row[c], c);
  if (CHECK) s.regular = s.regular && (s.found || run == run);
  return s;
}
__device__ __forceinline__ float crossing_offset(float before, float pmid) {
  return (1. - 2. * before - pmid) / (2. * pmid);  // MM.cu:34
}
// What the backward pass takes from the forward pass, one plane each: the crossing's offset, its mass, and its bin -- num_disp
// where there is none, -1 where the running sum falls below one half again (or becomes a NaN) and the bins alone decide.
__device__ __forceinline__ void save_crossing(float* __restrict__ saved, long long P, long long p, const Walked& s, float alpha, int D) {
  saved[p] = alpha;
  saved[P + p] = s.pmid;
  saved[2 * P + p] = !s.regular ? -1.f : (float)(s.found ? s.cidx : D);
}

template <int VEC, bool BACKWARD, bool SAVE>
__global__ __launch_bounds__(64) void median_rows_kernel(const float* __restrict__ vol, const float* __restrict__ gin,
                                                         float* __restrict__ res, float* __restrict__ saved, long long P,
                                                         long long HW, int D, int Dp, long long first_tile) {
  extern __shared__ __align__(16) float tile[];  // 64 rows of pitch Dp
  const int lane = threadIdx.x;
  const long long p0 = (first_tile + blockIdx.x) * 64;
  const int npx = (int)min((long long)64, P - p0);
  const int total = npx * D;
  stage_rows<VEC, false>(vol + p0 * D, nullptr, tile, total, D, Dp, lane);
  __syncthreads();
  float* row = tile + lane * Dp;
  Walked s{false, true, 0, 0.f, 1.f};
  if (lane < npx) s = walk_histogram<SAVE>(row, D);
  const float alpha = s.found ? crossing_offset(s.before, s.pmid) : 0.f;
  const long long p = p0 + lane;
  const long long n = p / HW, q = p - n * HW;
  if (!BACKWARD) {
    if (lane < npx) {
      res[n * 2 * HW + q] = s.found ? (float)s.cidx - 0.f + alpha : 0.f;  // MM.cu:35
      res[n * 2 * HW + HW + q] = s.found ? s.pmid : 0.f;
      if (SAVE) save_crossing(saved, P, p, s, alpha, D);
    }
    return;
  }
  if (lane < npx) {
    const float g0v = gin[n * 2 * HW + q], g1v = gin[n * 2 * HW + HW + q];
    const float cross = g0v * alpha / (-s.pmid) + g1v;  // MM.cu:69
    const float neg = -g0v / (2. * s.pmid);             // MM.cu:85
    const float pos = +g0v / (2. * s.pmid);             // MM.cu:88
    float score = 0.f;
#pragma unroll 4
    for (int c = 0; c < D; c++) {  // MM.cu:77-92; the crossing bin keeps the value of MM.cu:69
      const float cScore = row[c];
      const float sum = score + cScore;
      float g = (s.found && c == s.cidx) ? cross : 0.f;
      g = (sum < 0.5f) ? neg : ((score >= 0.5f) ? pos : g);
      row[c] = g;
      score = sum;
    }
  }
  __syncthreads();
  stage_rows<VEC, true>(nullptr, res + p0 * D, tile, total, D, Dp, lane);
}

// The forward pass with the run of 64 histograms going from memory straight into LDS (global_load_lds, 16 bytes a lane): all
// loads of a tile are in flight at once, where staging through registers had eight a lane and then waited.  The run stands in
// LDS as in memory and a lane reads RD bins of its row at a time: one where the bin count is odd, two where it is twice an odd
// number, four where it is a multiple of four.  In the last case rows whose pitch would put neighbours into the same banks
// have their 16-byte pieces rotated, row by row, on the way in (the loads pick the piece, LDS takes them in lane order).
// Bound by memory; behind it the walk, where long rows leave room for few wavefronts in LDS (100 bins: six a CU).  us, staged
// through registers / so: 4 x 384 x 1248 x 33 51.9 / 44.3 (6.1 TB/s), x 16 25.9 / 23.0, x 22 33.9 / 31.1; 384 x 1248 x 65 49.5 /
// 26.3, x 64 32.2 / 24.9; 2 x 384 x 1248 x 128 187 / 120; 2 x 187 x 621 x 64 19.6 / 15.6; 100 x 140 x 33 7.7 / 4.4.  Without the
// non-temporal hint 47.1 at 33 bins; four reads ahead instead of eight 123 at 128 bins.
template <int RD, bool SAVE>
__global__ __launch_bounds__(64) void median_forward_run_kernel(const float* __restrict__ vol, float* __restrict__ res,
                                                                float* __restrict__ saved, long long P, long long HW, int D) {
  extern __shared__ __align__(16) float tile[];  // 64 rows of D floats
  typedef const __attribute__((address_space(1))) void* GlobalPtr;
  typedef __attribute__((address_space(3))) void* LdsPtr;
  typedef float vec __attribute__((ext_vector_type(RD)));
  constexpr int kReadOnce = 2;  // the instruction's non-temporal bit
  const int lane = threadIdx.x;
  const long long p0 = (long long)blockIdx.x * 64, p = p0 + lane;
  const int npx = (int)min((long long)64, P - p0);
  const int total = npx * D, pieces = total >> 2;  // (at least one: npx * D >= 4)
  const float* const src = vol + p0 * D;
  // rotation of a row, RD == 4: a row is D4 pieces long; banks repeat every 16 pieces, so of each 16 / g rows, g the common
  // factors of 16 and D4, the pieces j already lie in different banks, and the next 16 / g rows are turned by one more piece
  const int D4 = D >> 2, shift = RD == 4 ? max(0, 4 - (__ffs(D4) - 1)) : 0, turns = RD == 4 ? min(16, D4 & -D4) - 1 : 0;
  auto rotation = [&](int px) { return (px >> shift) & turns; };
  if (RD == 4) {
    const int qs = 64 / D4, rs = 64 - qs * D4;
    int px = lane / D4, slot = lane - px * D4;
    for (int i = 0; i < total; i += 256) {  // (lane l writes piece i / 4 + l)
      int j = slot - rotation(px);
      j += j < 0 ? D4 : 0;
      const int piece = px < npx ? px * D4 + j : 0;
      __builtin_amdgcn_global_load_lds((GlobalPtr)(src + 4 * piece), (LdsPtr)(tile + i), 16, 0, kReadOnce);
      slot += rs;
      px += qs;
      if (slot >= D4) { slot -= D4; px++; }
    }
  } else {
    // (a load writes 16 bytes for every lane that takes part: in the last round only those with a piece, the run's end is the tile's)
    const int whole = pieces & ~63;
    for (int j = 0; j < whole; j += 64)
      __builtin_amdgcn_global_load_lds((GlobalPtr)(src + 4 * (j + lane)), (LdsPtr)(tile + 4 * j), 16, 0, kReadOnce);
    if (whole + lane < pieces)
      __builtin_amdgcn_global_load_lds((GlobalPtr)(src + 4 * (whole + lane)), (LdsPtr)(tile + 4 * whole), 16, 0, kReadOnce);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (RD != 4 && lane < (total & 3)) tile[4 * pieces + lane] = src[4 * pieces + lane];
  __syncthreads();
  Walked s{false, true, 0, 0.f, 1.f};
  float run = 0.f;
  if (lane < npx) {
    const vec* const row = reinterpret_cast<const vec*>(tile) + lane * (D / RD);
    const int per = D / RD, r = RD == 4 ? rotation(lane) : 0;
    for (int j0 = 0; j0 < per; j0 += kWalkAhead) {
      vec v[kWalkAhead];
#pragma unroll
      for (int u = 0; u < kWalkAhead; u++) {
        int slot = min(j0 + u, per - 1) + r;
        if (RD == 4) slot -= slot >= per ? per : 0;
        v[u] = row[slot];
      }
#pragma unroll
      for (int u = 0; u < kWalkAhead; u++)
        if (j0 + u < per) {
#pragma unroll
          for (int k = 0; k < RD; k++) walk_bin<SAVE>(s, run, v[u][k], (j0 + u) * RD + k);
        }
      if (!SAVE && __ballot(!s.found) == 0) break;
    }
    if (SAVE) s.regular = s.regular && (s.found || run == run);
    const float alpha = s.found ? crossing_offset(s.before, s.pmid) : 0.f;
    const long long n = p / HW, q = p - n * HW;
    res[n * 2 * HW + q] = s.found ? (float)s.cidx - 0.f + alpha : 0.f;  // MM.cu:35
    res[n * 2 * HW + HW + q] = s.found ? s.pmid : 0.f;
    if (SAVE) save_crossing(saved, P, p, s, alpha, D);
  }
}

// The backward pass over FULL tiles of 64 pixels for odd bin counts up to 4 * NV - 1 (no padding: the tile in LDS is a plain
// copy of the run), as a loop: a wavefront keeps the next tile's run in flight (NV 16-byte loads per lane, held in registers)
// while it walks the current one.  With one tile per wavefront only a quarter of the resident wavefronts have loads in
// flight at any time (the rest walk, store or are being launched), and the pass runs at half the rate memory allows.
template <int NV>
__global__ __launch_bounds__(64) void median_backward_stream_kernel(const float* __restrict__ vol, const float* __restrict__ gin,
                                                                    float* __restrict__ res, long long tiles, long long HW, int D) {
  extern __shared__ __align__(16) float tile[];  // 64 rows of D floats
  const int lane = threadIdx.x;
  const int per = 16 * D;  // 16-byte elements of a tile
  typedef float vec4 __attribute__((ext_vector_type(4)));  // (an array of HIP's float4 structs ends up in scratch memory)
  vec4* tile4 = reinterpret_cast<vec4*>(tile);
  vec4 v[NV];
  float gn0 = 0.f, gn1 = 0.f;
  // every load unconditional: an element past the run re-reads the lane's first one, and so does every element of the
  // surplus fetch behind a wavefront's last tile (live = false)
  auto fetch = [&](long long t, bool live) {
    const vec4* src = reinterpret_cast<const vec4*>(vol) + t * per;
    const int last = live ? per : 0;
#pragma unroll
    for (int u = 0; u < NV; u++) v[u] = __builtin_nontemporal_load(src + (lane + 64 * u < last ? lane + 64 * u : lane));  // read once
    const long long p = t * 64 + lane, n = p / HW, q = p - n * HW;
    gn0 = gin[n * 2 * HW + q];
    gn1 = gin[n * 2 * HW + HW + q];
  };
  long long t = blockIdx.x;
  if (t >= tiles) return;
  fetch(t, true);
  const float* row = tile + lane * D;
  for (; t < tiles; t += gridDim.x) {
#pragma unroll
    for (int u = 0; u < NV; u++)
      if (lane + 64 * u < per) tile4[lane + 64 * u] = v[u];
    const float g0v = gn0, g1v = gn1;
    const long long tn = t + gridDim.x;
    fetch(tn < tiles ? tn : t, tn < tiles);
    lds_only_barrier();  // (a full barrier would also wait for the loads just issued)
    const Walked s = walk_histogram<false>(row, D);
    const float alpha = s.found ? crossing_offset(s.before, s.pmid) : 0.f;
    const float cross = g0v * alpha / (-s.pmid) + g1v;  // MM.cu:69
    const float neg = -g0v / (2. * s.pmid);             // MM.cu:85
    const float pos = +g0v / (2. * s.pmid);             // MM.cu:88
    float* wrow = tile + lane * D;
    float score = 0.f;
#pragma unroll 4
    for (int c = 0; c < D; c++) {  // MM.cu:77-92; the crossing bin keeps the value of MM.cu:69
      const float cScore = wrow[c];
      const float sum = score + cScore;
      float g = (s.found && c == s.cidx) ? cross : 0.f;
      g = (sum < 0.5f) ? neg : ((score >= 0.5f) ? pos : g);
      wrow[c] = g;
      score = sum;
    }
    lds_only_barrier();
    vec4* dst = reinterpret_cast<vec4*>(res) + t * per;
#pragma unroll
    for (int u = 0; u < NV; u++)
      if (lane + 64 * u < per) dst[lane + 64 * u] = tile4[lane + 64 * u];  // (plain stores: the non-temporal hint costs this pass 7%)
    lds_only_barrier();  // the next tile overwrites the rows
  }
}

// Gradient of a histogram from the crossing that the forward pass saved (save_crossing): bins in front of it, the crossing
// bin, bins behind it -- the volume is not read again, the pass writes it and little else.  One wavefront per 64 pixels, whose
// gradients are one contiguous run; the three values of a pixel are handed out through LDS and every lane stores 16 bytes at a
// time.  A run with a pixel whose bins alone decide goes through the reference's two walks.
// Bound by the stores: 4 x 384 x 1248 x 33 42.6 us, 291 MB at 6.8 TB/s (from the volume: 88 us; plain stores instead of
// non-temporal ones: 61.7), 2 x 187 x 621 x 64 13.1 us.
template <int VEC>
__global__ __launch_bounds__(64) void median_backward_saved_kernel(const float* __restrict__ vol, const float* __restrict__ gin,
                                                                   const float* __restrict__ saved, float* __restrict__ gvol,
                                                                   long long P, long long HW, int D, int gin_planes) {
  __shared__ float tile[64][kPitch];
  __shared__ float4 bins[64];  // value in front of the crossing, at it, its bin
  typedef float vec4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x;
  const long long p0 = (long long)blockIdx.x * 64, p = p0 + lane;
  const int npx = (int)min((long long)64, P - p0);
  float g0v = 0.f, g1v = 0.f, alpha = 0.f, pmid = 1.f, at = 0.f;
  if (lane < npx) {
    const long long n = p / HW, q = p - n * HW;
    g0v = gin[n * gin_planes * HW + q];
    if (gin_planes == 2) g1v = gin[n * 2 * HW + HW + q];
    alpha = saved[p];
    pmid = saved[P + p];
    at = saved[2 * P + p];
  }
  if (__ballot(at < 0.f) != 0) {
    backward_from_bins(vol, gvol, tile, p0, P, D, lane, g0v, g1v);
    return;
  }
  const float cross = g0v * alpha / (-pmid) + g1v;  // MM.cu:69
  const float neg = -g0v / (2. * pmid);             // MM.cu:85 (and MM.cu:88 with its sign turned)
  bins[lane] = make_float4(neg, cross, at, 0.f);
  __syncthreads();
  const int total = npx * D;
  float* dst = gvol + p0 * D;
  constexpr int kStep = 64 * VEC;
  const int qs = kStep / D, rs = kStep - qs * D;
  int i = lane * VEC, px = i / D, b = i - px * D;
  auto value = [&](const float4& v, int bin) {
    const float f = (float)bin;
    return f < v.z ? v.x : (f == v.z ? v.y : -v.x);
  };
  for (; i < total; i += kStep) {
    const float4 v0 = bins[px];
    if (VEC == 4) {  // (four bins of one pixel, or the last of one and the first of the next: at least four bins each)
      const float4 v1 = bins[min(px + 1, 63)];
      vec4 g;
#pragma unroll
      for (int k = 0; k < 4; k++) g[k] = b + k < D ? value(v0, b + k) : value(v1, b + k - D);
      if (i + 3 < total) {
        __builtin_nontemporal_store(g, reinterpret_cast<vec4*>(dst + i));
      } else {
        for (int k = 0; k < 4 && i + k < total; k++) dst[i + k] = g[k];
      }
    } else {
      dst[i] = value(v0, b);
    }
    b += rs;
    px += qs;
    if (b >= D) { b -= D; px++; }
  }
}

template <bool BACKWARD, bool SAVE>
void launch_median_rows(const float* vol, const float* gin, float* res, float* saved, long long P, long long HW, int D, bool aligned,
                        hipStream_t stream) {
  const int Dp = D | 1;
  constexpr int kStreamNV = 10;
  if (!BACKWARD && aligned && D >= 4 && !inpaint::knobs().median_tile_per_wave) {
    const dim3 grid((unsigned)((P + 63) / 64)), block(64);
    const size_t lds = (size_t)64 * D * sizeof(float);
    if (D % 4 == 0) hipLaunchKernelGGL((median_forward_run_kernel<4, SAVE>), grid, block, lds, stream, vol, res, saved, P, HW, D);
    else if (D % 2 == 0) hipLaunchKernelGGL((median_forward_run_kernel<2, SAVE>), grid, block, lds, stream, vol, res, saved, P, HW, D);
    else hipLaunchKernelGGL((median_forward_run_kernel<1, SAVE>), grid, block, lds, stream, vol, res, saved, P, HW, D);
    return;
  }
  if (BACKWARD && aligned && (D & 1) && D >= 5 && D < 4 * kStreamNV && P >= 64 && !inpaint::knobs().median_tile_per_wave) {
    // full tiles in the streaming loop, the last partial tile (if any) below
    const long long tiles = P / 64;
    const long long waves = std::min<long long>(tiles, 16ll * inpaint::compute_unit_count());
    hipLaunchKernelGGL((median_backward_stream_kernel<kStreamNV>), dim3((unsigned)waves), dim3(64), (size_t)64 * D * sizeof(float),
                       stream, vol, gin, res, tiles, HW, D);
    if (P % 64 == 0) return;
    // (the kernel below takes its pixels from P and blockIdx: give it the last tile only)
    hipLaunchKernelGGL((median_rows_kernel<4, BACKWARD, SAVE>), dim3(1), dim3(64), (size_t)64 * Dp * sizeof(float), stream, vol, gin, res,
                       saved, P, HW, D, Dp, tiles);
    return;
  }
  const dim3 grid((unsigned)((P + 63) / 64)), block(64);
  const size_t lds = (size_t)64 * Dp * sizeof(float);
  if (aligned && D >= 4)
    hipLaunchKernelGGL((median_rows_kernel<4, BACKWARD, SAVE>), grid, block, lds, stream, vol, gin, res, saved, P, HW, D, Dp, 0ll);
  else
    hipLaunchKernelGGL((median_rows_kernel<1, BACKWARD, SAVE>), grid, block, lds, stream, vol, gin, res, saved, P, HW, D, Dp, 0ll);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

namespace {

// Whether the per-pixel passes of the quadratic fit take the split kernels: too few tiles (64 x 8 pixels) to fill the chip.  The
// split kernels work through whole chunks of 32 channels, so with fewer channels they pay up to fewer tiles only.  Measured, us,
// split / ring, forward pass: 4 channels 40 tiles 7.4 / 8.9, 128 10.7 / 8.9; 8 channels 60 tiles 7.2 / 9.8, 91 9.5 / 10.0, 128
// 11.0 / 10.3; 16 channels 128 tiles 11.0 / 11.5, 195 17.0 / 11.0; 24 channels 128 tiles 10.9 / 13.8, 195 16.9 / 14.0; 32 channels
// 128 tiles 10.8 / 16.5, 195 17.8 / 17.3, 248 19.2 / 17.7; 64 channels 60 tiles 11.7 / 28.4, 195 31.5 / 28.8; 96 channels 128 tiles
// 27.8 / 41.1, 195 45.9 / 40.1.  Backward pass (split / the faster of the others): 32 channels 128 tiles 51 / 50, 195 61 / 55; 64
// channels 128 tiles 64 / 78, 195 82 / 83; 96 channels 195 tiles 147 / 115.
bool quadfit_few_tiles(long long tiles, int ic) {
  if (inpaint::knobs().quadfit_split >= 0) return inpaint::knobs().quadfit_split == 1;
  return tiles <= (long long)inpaint::compute_unit_count() * std::min(ic, 24) / kSplitChunk;
}

// Channels per block of the gather pass: all of them where the tiles fill the chip (four blocks resident per CU), else so
// few that about that many blocks result, at least the four that the ring of windows holds.
int gather_channels_per_block(long long tiles, int ic) {
  const long long groups = std::max<long long>(1, 4ll * inpaint::compute_unit_count() / tiles);
  return std::max<int>(4, (int)((ic + groups - 1) / groups + 3) / 4 * 4);
}

template <int MODE>
void launch_quadfit_split(const float* im0, const float* im1, const float* flow, const float* gin, float* res, const QfWorkspace& ws,
                          int n, int ic, int ih, int iw, int fc, hipStream_t st) {
  const int tx = (iw + 63) / 64;
  const dim3 grid((unsigned)(((long long)n * tx * ih + 7) / 8 * 8)), block(256);
  if (ic <= kSplitChunk)
    hipLaunchKernelGGL((quadfit_split<MODE, 1>), grid, block, 0, st, im0, im1, flow, gin, res, ws, n, ic, ih, iw, fc, tx, ih);
  else if (ic <= 2 * kSplitChunk)
    hipLaunchKernelGGL((quadfit_split<MODE, 2>), grid, block, 0, st, im0, im1, flow, gin, res, ws, n, ic, ih, iw, fc, tx, ih);
  else
    hipLaunchKernelGGL((quadfit_split<MODE, 0>), grid, block, 0, st, im0, im1, flow, gin, res, ws, n, ic, ih, iw, fc, tx, ih);
}

}  // namespace

extern "C" {

const char* flowaux_last_error(void) { return inpaint::error_buffer(); }

int flowaux_profile(int enable) {
  g_timer.enabled = enable != 0;
  g_timed_pass = enable == 2 ? 2 : 1;
  g_timer.reset();
  return 0;
}

int flowaux_profile_read(double* total_ms, int* launches) { return g_timer.read(total_ms, launches); }

static int forward_of(const char* name, const float* im0, const float* im1, const float* flow, float* out, float* costs, int n, int ic,
                      int ih, int iw, int flow_channels, void* stream) {
  if (!im0 || !im1 || !flow || !out) return fail(INPAINT_ERR_ARG, "%s: null pointer", name);
  if (n < 1 || ic < 1 || ih < 1 || iw < 1) return fail(INPAINT_ERR_ARG, "%s: bad shape %dx%dx%dx%d", name, n, ic, ih, iw);
  if (flow_channels < 2) return fail(INPAINT_ERR_ARG, "%s: the flow needs at least 2 channels, got %d", name, flow_channels);
  if ((long long)ih * iw >= (1ll << 31)) return fail(INPAINT_ERR_ARG, "%s: image too large", name);
  const long long P = (long long)n * ih * iw;
  const int tiles_x = (iw + kTW - 1) / kTW, tiles_y = (ih + TileCfg<kPxTile>::TH - 1) / TileCfg<kPxTile>::TH;
  const long long tiles = (long long)n * tiles_x * tiles_y;
  if (tiles >= (1ll << 31) - 8) return fail(INPAINT_ERR_ARG, "%s: too many tiles", name);
  if (!costs && inpaint::knobs().quadfit_px_path)
    hipLaunchKernelGGL(quadfit_forward_kernel, banded_grid(P), dim3(256), 0, (hipStream_t)stream, im0, im1, flow, out, n,
                       ic, ih, iw, flow_channels);
  else if (!costs && quadfit_few_tiles(tiles, ic))
    launch_quadfit_split<0>(im0, im1, flow, nullptr, out, QfWorkspace{}, n, ic, ih, iw, flow_channels, (hipStream_t)stream);
  else
    hipLaunchKernelGGL((quadfit_ring_tiles<0>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, (hipStream_t)stream, im0, im1,
                       flow, nullptr, costs, out, QfWorkspace{}, n, ic, ih, iw, flow_channels, tiles_x, tiles_y);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int quadfit_forward(const float* im0, const float* im1, const float* flow, float* out, int n, int ic, int ih, int iw,
                    int flow_channels, void* stream) {
  return forward_of("quadfit_forward", im0, im1, flow, out, nullptr, n, ic, ih, iw, flow_channels, stream);
}

int quadfit_forward_saving(const float* im0, const float* im1, const float* flow, float* out, float* costs, int n, int ic, int ih,
                           int iw, int flow_channels, void* stream) {
  if (!costs) return fail(INPAINT_ERR_ARG, "quadfit_forward_saving: null pointer");
  return forward_of("quadfit_forward_saving", im0, im1, flow, out, costs, n, ic, ih, iw, flow_channels, stream);
}

// Not where the split kernels run, whose backward pass keeps all taps in registers and is bound by latency, and up to 32 channels
// not before every CU has a tile: the resident pass A has twice as many (forward + backward, us, with / without the costs: 32
// channels 195 tiles 80 / 72, 250 81 / 73, 300 84 / 85, 480 89 / 92, 960 124 / 140; 64 channels 195 tiles 112 / 178).
int quadfit_saving_pays(int n, int ic, int ih, int iw) {
  if (n < 1 || ic < 1 || ih < 1 || iw < 1 || inpaint::knobs().quadfit_px_path || inpaint::knobs().quadfit_reread) return 0;
  const long long tiles = (long long)n * ((iw + kTW - 1) / kTW) * ((ih + TileCfg<kPxTile>::TH - 1) / TileCfg<kPxTile>::TH);
  return !quadfit_few_tiles(tiles, ic) && (ic > kResidentChannels || tiles > inpaint::compute_unit_count());
}

long long quadfit_backward_workspace_bytes(int n, int ih, int iw) {
  if (n < 1 || ih < 1 || iw < 1) return 0;
  return qf_workspace_bytes((long long)n * ih * iw);
}

static int backward_of(const char* name, const float* im0, const float* im1, const float* flow, const float* gin, const float* costs,
                       float* g0, float* g1, int n, int ic, int ih, int iw, int flow_channels, void* workspace, long long workspace_bytes,
                       void* stream) {
  if (!im0 || !im1 || !flow || !gin || !g0 || !g1) return fail(INPAINT_ERR_ARG, "%s: null pointer", name);
  if (n < 1 || ic < 1 || ih < 1 || iw < 1) return fail(INPAINT_ERR_ARG, "%s: bad shape %dx%dx%dx%d", name, n, ic, ih, iw);
  if (flow_channels < 2) return fail(INPAINT_ERR_ARG, "%s: the flow needs at least 2 channels, got %d", name, flow_channels);
  if ((long long)ih * iw >= (1ll << 31)) return fail(INPAINT_ERR_ARG, "%s: image too large", name);
  const long long P = (long long)n * ih * iw, total = P * ic;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid = banded_grid(P), block(256);
  if (!workspace) {  // no workspace: scatter with float atomics
    hipLaunchKernelGGL(inpaint::fill_zero_f32, dim3(inpaint::grid_stride(total)), dim3(256), 0, st, g1, total);
    hipLaunchKernelGGL(quadfit_backward_kernel, grid, block, 0, st, im0, im1, flow, gin, g0, g1, n, ic, ih, iw, flow_channels);
    INPAINT_HIP(hipGetLastError());
    return 0;
  }
  if (workspace_bytes < qf_workspace_bytes(P))
    return fail(INPAINT_ERR_ARG, "%s: workspace of %lld bytes, %lld needed", name, workspace_bytes, qf_workspace_bytes(P));
  if (((uintptr_t)workspace & 15) != 0) return fail(INPAINT_ERR_ARG, "%s: workspace must be 16-byte aligned", name);
  if (P >= (1ll << 31)) return fail(INPAINT_ERR_ARG, "%s: too many pixels for the inverse map", name);
  const QfWorkspace ws = qf_carve(workspace, P);
  // the counters start at zero (a fill kernel, so that the call can be captured into a graph)
  hipLaunchKernelGGL(inpaint::fill_zero_f32, dim3(inpaint::grid_stride(P + 64)), dim3(256), 0, st,
                     reinterpret_cast<float*>(ws.count), P + 64);
  const int tiles_x = (iw + kTW - 1) / kTW, tiles_y = (ih + TileCfg<kPxTile>::TH - 1) / TileCfg<kPxTile>::TH;
  const long long tiles = (long long)n * tiles_x * tiles_y;
  const bool px_path = !costs && inpaint::knobs().quadfit_px_path;
  if (px_path)
    hipLaunchKernelGGL(quadfit_backward_sources, grid, block, 0, st, im0, im1, flow, gin, g0, ws, n, ic, ih, iw, flow_channels);
  else {
    if (g_timed_pass == 1) g_timer.begin(st);
    if (costs) {
      hipLaunchKernelGGL((quadfit_ring_tiles<1>), dim3((unsigned)((tiles + 7) / 8 * 8)), block, 0, st, im0, im1, flow, gin,
                         const_cast<float*>(costs), g0, ws, n, ic, ih, iw, flow_channels, tiles_x, tiles_y);
    } else if (quadfit_few_tiles(tiles, ic) && !inpaint::knobs().quadfit_reread) {
      launch_quadfit_split<1>(im0, im1, flow, gin, g0, ws, n, ic, ih, iw, flow_channels, st);
    } else if (ic <= kResidentChannels && !inpaint::knobs().quadfit_reread) {
      const int ry = (ih + kResidentRows - 1) / kResidentRows;
      const long long rt = (long long)n * tiles_x * ry;
      const dim3 rgrid((unsigned)((rt + 7) / 8 * 8));
      if (ic == kResidentChannels)
        hipLaunchKernelGGL((quadfit_sources_resident<kResidentChannels, true>), rgrid, block, 0, st, im0, im1, flow, gin, g0, ws, n,
                           ic, ih, iw, flow_channels, tiles_x, ry);
      else
        hipLaunchKernelGGL((quadfit_sources_resident<kResidentChannels, false>), rgrid, block, 0, st, im0, im1, flow, gin, g0, ws, n,
                           ic, ih, iw, flow_channels, tiles_x, ry);
    } else {
      hipLaunchKernelGGL(quadfit_sources_tiles, dim3((unsigned)((tiles + 7) / 8 * 8)), block, 0, st, im0, im1, flow, gin, g0,
                         ws, n, ic, ih, iw, flow_channels, tiles_x, tiles_y);
    }
    if (g_timed_pass == 1) g_timer.end(st, 1);
  }
  if (px_path || ih > 65535 || iw > 65535 || (long long)ih * iw >= (1ll << 24)) {
    hipLaunchKernelGGL(quadfit_backward_gather, grid, block, 0, st, im0, g1, ws, n, ic, ih, iw);
  } else {
    const int gy = (ih + TileCfg<kPxGather>::TH - 1) / TileCfg<kPxGather>::TH;
    const long long gt = (long long)n * tiles_x * gy;
    if (g_timed_pass == 2) g_timer.begin(st);
    const int per = gather_channels_per_block(gt, ic);
    hipLaunchKernelGGL((quadfit_gather_tiles<kPxGather>), dim3((unsigned)((gt + 7) / 8 * 8), (unsigned)((ic + per - 1) / per)), block, 0,
                       st, im0, g1, ws, n, ic, per, ih, iw, tiles_x, gy);
    if (g_timed_pass == 2) g_timer.end(st, 1);
  }
  hipLaunchKernelGGL(quadfit_backward_overflow, dim3((unsigned)std::min<long long>((P + 127) / 128, 512)), block, 0, st, im0, flow, g1, ws, n, ic, ih, iw, flow_channels);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int quadfit_backward(const float* im0, const float* im1, const float* flow, const float* gin, float* g0, float* g1, int n,
                     int ic, int ih, int iw, int flow_channels, void* workspace, long long workspace_bytes, void* stream) {
  return backward_of("quadfit_backward", im0, im1, flow, gin, nullptr, g0, g1, n, ic, ih, iw, flow_channels, workspace, workspace_bytes,
                     stream);
}

int quadfit_backward_saved(const float* im0, const float* im1, const float* flow, const float* gin, const float* costs, float* g0,
                           float* g1, int n, int ic, int ih, int iw, int flow_channels, void* workspace, long long workspace_bytes,
                           void* stream) {
  if (!costs || !workspace) return fail(INPAINT_ERR_ARG, "quadfit_backward_saved: null pointer");
  return backward_of("quadfit_backward_saved", im0, im1, flow, gin, costs, g0, g1, n, ic, ih, iw, flow_channels, workspace,
                     workspace_bytes, stream);
}

static int image_args(const char* name, bool pointers, int ic, int ih, int iw, long long flow_pixel_stride, long long flow_channel_stride) {
  if (!pointers) return fail(INPAINT_ERR_ARG, "%s: null pointer", name);
  if (ic < 1 || ih < 1 || iw < 1) return fail(INPAINT_ERR_ARG, "%s: bad shape %dx%dx%d", name, ih, iw, ic);
  // (offsets into a map are 32 bits wide; a pixel has four threads, and a launch fewer than 2^32 of them)
  if ((long long)ih * iw * ic >= (1ll << 31) || (long long)ih * iw > (1ll << 30) - 1024) return fail(INPAINT_ERR_ARG, "%s: image too large", name);
  if (flow_pixel_stride < 1 || flow_channel_stride < 1) return fail(INPAINT_ERR_ARG, "%s: bad strides of the flow", name);
  return 0;
}
static dim3 image_grid(long long P) { return dim3((unsigned)(((P + quadfit_image::kPixels - 1) / quadfit_image::kPixels + 7) / 8 * 8)); }

int quadfit_image_forward(const float* im0, const float* im1, const float* flow, float* out, float* costs, int ic, int ih, int iw,
                          long long flow_pixel_stride, long long flow_channel_stride, void* stream) {
  if (const int rc = image_args("quadfit_image_forward", im0 && im1 && flow && out, ic, ih, iw, flow_pixel_stride, flow_channel_stride))
    return rc;
  const quadfit_image::FlowStrides fs{flow_pixel_stride, flow_channel_stride};
  const dim3 grid = image_grid((long long)ih * iw), block(256);
  if (ic % 4 == 0 && aligned16(im0) && aligned16(im1))
    hipLaunchKernelGGL((quadfit_image::forward<4>), grid, block, 0, (hipStream_t)stream, im0, im1, flow, fs, out, costs, ic, ih, iw);
  else
    hipLaunchKernelGGL((quadfit_image::forward<1>), grid, block, 0, (hipStream_t)stream, im0, im1, flow, fs, out, costs, ic, ih, iw);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int quadfit_image_backward(const float* im0, const float* im1, const float* flow, const float* gin, const float* costs, float* g0,
                           float* g1, int ic, int ih, int iw, long long flow_pixel_stride, long long flow_channel_stride,
                           void* workspace, long long workspace_bytes, void* stream) {
  if (const int rc = image_args("quadfit_image_backward", im0 && im1 && flow && gin && costs && g0 && g1 && workspace, ic, ih, iw,
                                flow_pixel_stride, flow_channel_stride))
    return rc;
  const long long P = (long long)ih * iw;
  if (workspace_bytes < qf_workspace_bytes(P))
    return fail(INPAINT_ERR_ARG, "quadfit_image_backward: workspace of %lld bytes, %lld needed", workspace_bytes, qf_workspace_bytes(P));
  if (((uintptr_t)workspace & 15) != 0) return fail(INPAINT_ERR_ARG, "quadfit_image_backward: workspace must be 16-byte aligned");
  const QfWorkspace ws = qf_carve(workspace, P);
  const quadfit_image::FlowStrides fs{flow_pixel_stride, flow_channel_stride};
  const dim3 grid = image_grid(P), block(256);
  hipStream_t st = (hipStream_t)stream;
  // the counters start at zero (a fill kernel, so that the call can be captured into a graph)
  hipLaunchKernelGGL(inpaint::fill_zero_f32, dim3(inpaint::grid_stride(P + 64)), dim3(256), 0, st, reinterpret_cast<float*>(ws.count),
                     P + 64);
  const bool wide = ic % 4 == 0 && aligned16(im0) && aligned16(im1) && aligned16(g0) && aligned16(g1);
  if (wide) {
    hipLaunchKernelGGL((quadfit_image::sources<4>), grid, block, 0, st, im1, flow, fs, gin, costs, g0, ws, ic, ih, iw);
    hipLaunchKernelGGL((quadfit_image::gather<4>), grid, block, 0, st, im0, g1, ws, ic, ih, iw);
  } else {
    hipLaunchKernelGGL((quadfit_image::sources<1>), grid, block, 0, st, im1, flow, fs, gin, costs, g0, ws, ic, ih, iw);
    hipLaunchKernelGGL((quadfit_image::gather<1>), grid, block, 0, st, im0, g1, ws, ic, ih, iw);
  }
  hipLaunchKernelGGL(quadfit_image::overflow, dim3((unsigned)std::min<long long>((P + 127) / 128, 512)), block, 0, st, im0, flow, fs, g1,
                     ws, ic, ih, iw);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int medimax_forward(const float* vol, float* out, int n, int ih, int iw, int num_disp, void* stream) {
  if (!vol || !out) return fail(INPAINT_ERR_ARG, "medimax_forward: null pointer");
  if (n < 1 || ih < 1 || iw < 1 || num_disp < 1)
    return fail(INPAINT_ERR_ARG, "medimax_forward: bad shape %dx%dx%dx%d", n, ih, iw, num_disp);
  const long long HW = (long long)ih * iw, P = n * HW;
  if (num_disp <= kMaxRowBins)
    launch_median_rows<false, false>(vol, nullptr, out, nullptr, P, HW, num_disp, aligned16(vol), (hipStream_t)stream);
  else
    hipLaunchKernelGGL(median_forward_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, (hipStream_t)stream, vol, out, P,
                     HW, num_disp);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int medimax_backward(const float* vol, const float* gin, float* gvol, int n, int ih, int iw, int num_disp, void* stream) {
  if (!vol || !gin || !gvol) return fail(INPAINT_ERR_ARG, "medimax_backward: null pointer");
  if (n < 1 || ih < 1 || iw < 1 || num_disp < 1)
    return fail(INPAINT_ERR_ARG, "medimax_backward: bad shape %dx%dx%dx%d", n, ih, iw, num_disp);
  const long long HW = (long long)ih * iw, P = n * HW;
  if (num_disp <= kMaxRowBins) {
    g_timer.begin((hipStream_t)stream);
    launch_median_rows<true, false>(vol, gin, gvol, nullptr, P, HW, num_disp, aligned16(vol) && aligned16(gvol), (hipStream_t)stream);
    g_timer.end((hipStream_t)stream, 1);
  } else
    hipLaunchKernelGGL(median_backward_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, (hipStream_t)stream, vol, gin,
                     gvol, P, HW, num_disp);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int medimax_forward_saving(const float* vol, float* out, float* saved, int n, int ih, int iw, int num_disp, void* stream) {
  if (!vol || !out || !saved) return fail(INPAINT_ERR_ARG, "medimax_forward_saving: null pointer");
  if (n < 1 || ih < 1 || iw < 1 || num_disp < 1 || num_disp > kMaxRowBins)
    return fail(INPAINT_ERR_ARG, "medimax_forward_saving: bad shape %dx%dx%dx%d", n, ih, iw, num_disp);
  const long long HW = (long long)ih * iw;
  launch_median_rows<false, true>(vol, nullptr, out, saved, n * HW, HW, num_disp, aligned16(vol), (hipStream_t)stream);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

int medimax_backward_saved(const float* vol, const float* gin, int gin_planes, const float* saved, float* gvol, int n, int ih, int iw,
                           int num_disp, void* stream) {
  if (!vol || !gin || !saved || !gvol) return fail(INPAINT_ERR_ARG, "medimax_backward_saved: null pointer");
  if (gin_planes != 1 && gin_planes != 2) return fail(INPAINT_ERR_ARG, "medimax_backward_saved: one or two planes of gradient, not %d", gin_planes);
  if (n < 1 || ih < 1 || iw < 1 || num_disp < 1 || num_disp > kMaxRowBins)
    return fail(INPAINT_ERR_ARG, "medimax_backward_saved: bad shape %dx%dx%dx%d", n, ih, iw, num_disp);
  const long long HW = (long long)ih * iw, P = n * HW;
  const dim3 grid((unsigned)((P + 63) / 64)), block(64);
  g_timer.begin((hipStream_t)stream);
  if (aligned16(gvol) && num_disp >= 4)
    hipLaunchKernelGGL((median_backward_saved_kernel<4>), grid, block, 0, (hipStream_t)stream, vol, gin, saved, gvol, P, HW, num_disp,
                       gin_planes);
  else
    hipLaunchKernelGGL((median_backward_saved_kernel<1>), grid, block, 0, (hipStream_t)stream, vol, gin, saved, gvol, P, HW, num_disp,
                       gin_planes);
  g_timer.end((hipStream_t)stream, 1);
  INPAINT_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
