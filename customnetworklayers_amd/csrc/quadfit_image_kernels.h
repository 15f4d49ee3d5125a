// Quadratic fit of one image whose feature maps have their channels innermost (H x W x C), as the module takes them.
//
// With the channels of a pixel side by side a tap is one contiguous run: lanes are channels (four each, 16-byte loads), the five
// taps of a pixel are five runs, and the list of sources of a target pixel is the same for all the lanes that work on it.  No
// windows, no pixel that leaves one, and none of the copies between layouts that the kernels on planes need.  Only the sums that
// decide the fit run over the channels in order: their products change hands in LDS and a lane sums one tap of one pixel.
//
// A block owns 64 consecutive pixels.  Same arithmetic, operation by operation, as the kernels on planes.
// Bound by latency on small images (64 x 96 x 312: forward 7 us, backward 10 + 8 + 5), by memory on large ones.  Module, forward +
// backward, us, kernels on planes with their copies / these: 64 x 96 x 312 232 / 127 and 32 x 200 x 640 334 / 130 (host time), 32 x 448 x
// 1280 1296 / 134, 64 x 448 x 1280 2443 / 266; with 12 pixels of noise on the flow 4679 / 335; forward alone 1150 / 76.  The forward
// pass works through whole chunks of 32 channels: with fewer than eight it loses on large images, which are not sent here
// (image_pays in QuadFit_cuda_ext.py).
#pragma once

namespace quadfit_image {

constexpr int kPixels = 64;                     // pixels per block
constexpr int kChunk = 32, kPitch = kChunk + 4; // channels per round of products, floats between pixels in LDS (an odd number of 16-byte pieces)

// first of the block's pixels, blocks numbered so that every XCD works through one band of the image; >= P: none
__device__ __forceinline__ int first_pixel() {
  const int per_xcd = gridDim.x >> 3;
  return ((blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3)) * kPixels;
}

struct FlowStrides {
  long long pixel, channel;  // floats between pixels (row after row), between the channels of one
};
__device__ __forceinline__ void locate_pixel(TilePx& s, const float* __restrict__ flow, FlowStrides fs, int H, int W, int p, bool valid) {
  int a = 0, b = 0, c = 0, d = 0;
  const int q = valid ? p : 0, y = q / W, x = q - y * W;
  locate_at(s, flow[q * fs.pixel], flow[q * fs.pixel + fs.channel], H, W, x, y, valid, a, b, c, d);
}
// offsets of the five taps in floats (a pixel that is not inside reads the image's first; its sums are not used)
__device__ __forceinline__ void tap_offsets(const TilePx& s, int W, int C, unsigned (&o)[5]) {
  const unsigned row = (unsigned)s.iy * W;
  o[0] = (row + s.ix) * C;
  o[1] = (row + s.xp) * C;
  o[2] = (row + s.xm) * C;
  o[3] = ((unsigned)s.yp * W + s.ix) * C;
  o[4] = ((unsigned)s.ym * W + s.ix) * C;
}

template <int VEC>
struct Vec {
  typedef float type __attribute__((ext_vector_type(VEC)));
};

// Forward pass; costs: the five sums per pixel (planes of H * W), or null.
template <int VEC>
__global__ __launch_bounds__(256) void forward(const float* __restrict__ im0, const float* __restrict__ im1,
                                               const float* __restrict__ flow, FlowStrides fs, float* __restrict__ out,
                                               float* __restrict__ costs, int C, int H, int W) {
  typedef typename Vec<VEC>::type vec;
  constexpr int kPieces = kChunk / VEC, kItems = kPixels * kPieces / 256;
  __shared__ __align__(16) float prod[5][kPixels][kPitch];
  __shared__ unsigned off[5][kPixels];
  __shared__ float sums[5][kPixels];
  const int P = H * W, p0 = first_pixel();
  if (p0 >= P) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  TilePx px{};
  if (wave == 0) {
    locate_pixel(px, flow, fs, H, W, p0 + lane, p0 + lane < P);
    unsigned o[5];
    tap_offsets(px, W, C, o);
#pragma unroll
    for (int k = 0; k < 5; k++) off[k][lane] = o[k];
  }
  __syncthreads();
  // item i of a thread: piece `piece` of pixel pix[i]
  const int piece = threadIdx.x % kPieces;
  unsigned at[kItems][6];
#pragma unroll
  for (int i = 0; i < kItems; i++) {
    const int pix = threadIdx.x / kPieces + i * (256 / kPieces);
#pragma unroll
    for (int k = 0; k < 5; k++) at[i][k] = off[k][pix];
    at[i][5] = (unsigned)min(p0 + pix, P - 1) * C;
  }
  vec v[kItems][6];
  auto load = [&](int c0) {  // (past the last channel: the last piece again)
    const unsigned c = (unsigned)min(c0 + piece * VEC, C - VEC);
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      v[i][5] = *reinterpret_cast<const vec*>(im0 + at[i][5] + c);
#pragma unroll
      for (int k = 0; k < 5; k++) v[i][k] = *reinterpret_cast<const vec*>(im1 + at[i][k] + c);
    }
  };
  load(0);
  float cost[2] = {0.f, 0.f};  // this wavefront's tap; wavefront 0 also sums tap 4
  for (int c0 = 0; c0 < C; c0 += kChunk) {
#pragma unroll
    for (int i = 0; i < kItems; i++) {
      const int pix = threadIdx.x / kPieces + i * (256 / kPieces);
#pragma unroll
      for (int k = 0; k < 5; k++) *reinterpret_cast<vec*>(&prod[k][pix][piece * VEC]) = v[i][5] * v[i][k];
    }
    if (c0 + kChunk < C) load(c0 + kChunk);
    lds_only_barrier();
    const int nc = min(kChunk, C - c0);
    auto sum = [&](const float* row, float& acc) {  // QF.cu:63-71
      if (nc == kChunk) {
#pragma unroll
        for (int c = 0; c < kChunk; c += 4) {
          const float4 t = *reinterpret_cast<const float4*>(row + c);
          acc += t.x;
          acc += t.y;
          acc += t.z;
          acc += t.w;
        }
      } else {
        for (int c = 0; c < nc; c++) acc += row[c];
      }
    };
    sum(prod[wave][lane], cost[0]);
    if (wave == 0) sum(prod[4][lane], cost[1]);
    lds_only_barrier();
  }
  sums[wave][lane] = cost[0];
  if (wave == 0) sums[4][lane] = cost[1];
  __syncthreads();
  const int p = p0 + lane;
  if (wave != 0 || p >= P) return;
  Fit f;
  f.inside = px.inside;
  f.validX = f.validY = 0;
  f.c00 = f.ax = f.ay = f.bx = f.by = f.fx = f.fy = 0.f;
  if (px.inside) finish_fit(f, sums[0][lane], sums[1][lane], sums[3][lane], sums[2][lane], sums[4][lane], px.ix, px.iy, H, W);
  float score = 0.f;
  if (f.inside)  // QF.cu:136
    score = f.ax * f.fx * f.fx + f.bx * f.fx + f.c00 + f.ay * f.fy * f.fy + f.by * f.fy;
  out[3 * (size_t)p] = f.fx;
  out[3 * (size_t)p + 1] = f.fy;
  out[3 * (size_t)p + 2] = score;
  if (costs) {
#pragma unroll
    for (int k = 0; k < 5; k++) costs[(size_t)k * P + p] = sums[k][lane];
  }
}

// Backward pass, per source pixel: fit from the costs, scatter coefficients and list entry, gradient wrt the first map.
template <int VEC>
__global__ __launch_bounds__(256) void sources(const float* __restrict__ im1, const float* __restrict__ flow, FlowStrides fs,
                                               const float* __restrict__ gin, const float* __restrict__ costs, float* __restrict__ g0,
                                               QfWorkspace ws, int C, int H, int W) {
  typedef typename Vec<VEC>::type vec;
  __shared__ unsigned off[5][kPixels];
  __shared__ double k00[kPixels];
  __shared__ __align__(16) float4 kr[kPixels];  // 0p, 0m, p0, m0
  __shared__ float2 other[kPixels];             // dFds, state: 0 outside, 1 only the centre, 2 fitted
  const int P = H * W, p0 = first_pixel();
  if (p0 >= P) return;
  if (threadIdx.x < kPixels) {
    const int p = p0 + threadIdx.x;
    TilePx px;
    locate_pixel(px, flow, fs, H, W, p, p < P);
    unsigned o[5];
    tap_offsets(px, W, C, o);
#pragma unroll
    for (int k = 0; k < 5; k++) off[k][threadIdx.x] = o[k];
    Factors k{};
    if (px.inside) {
      Fit f;
      f.inside = true;
      f.validX = f.validY = 0;
      f.c00 = f.ax = f.ay = f.bx = f.by = f.fx = f.fy = 0.f;
      float c[5];
#pragma unroll
      for (int j = 0; j < 5; j++) c[j] = costs[(size_t)j * P + p];
      finish_fit(f, c[0], c[1], c[3], c[2], c[4], px.ix, px.iy, H, W);
      k = scatter_factors(f, gin[3 * (size_t)p], gin[3 * (size_t)p + 1], gin[3 * (size_t)p + 2]);
      store_source(ws, k, P, 0, p, (long long)px.iy * W + px.ix, p);
    }
    k00[threadIdx.x] = k.k00;
    kr[threadIdx.x] = make_float4(k.k0p, k.k0m, k.kp0, k.km0);
    other[threadIdx.x] = make_float2(k.dFds, !px.inside ? 0.f : (k.any_valid ? 2.f : 1.f));
  }
  __syncthreads();
  const int pieces = C / VEC, total = min(kPixels, P - p0) * pieces;
  const int dp = 256 / pieces, dq = 256 - dp * pieces;
  int pix = threadIdx.x / pieces, piece = threadIdx.x - pix * pieces;
  for (int i = threadIdx.x; i < total; i += 256) {
    const unsigned c = (unsigned)piece * VEC;
    vec t[5], g;
#pragma unroll
    for (int k = 0; k < 5; k++) t[k] = *reinterpret_cast<const vec*>(im1 + off[k][pix] + c);
    const double a = k00[pix];
    const float4 r = kr[pix];
    const float2 s = other[pix];
#pragma unroll
    for (int e = 0; e < VEC; e++) {
      const float fitted = 0.5 * (t[0][e] * a + t[1][e] * r.x + t[2][e] * r.y + t[3][e] * r.z + t[4][e] * r.w);  // QF.cu:286-290
      const float centre = t[0][e] * s.x;                                                                        // QF.cu:295
      g[e] = s.y == 2.f ? fitted : (s.y == 1.f ? centre : 0.f);
    }
    __builtin_nontemporal_store(g, reinterpret_cast<vec*>(g0 + (size_t)(p0 + pix) * C + c));
    piece += dq;
    pix += dp;
    if (piece >= pieces) { piece -= pieces; pix++; }
  }
}

// Backward pass, per target pixel: the sources listed at it and at its four neighbours (see the inverse map of the kernels on
// planes), summed for all channels.
template <int VEC>
__global__ __launch_bounds__(256) void gather(const float* __restrict__ im0, float* __restrict__ g1, QfWorkspace ws, int C, int H, int W) {
  typedef typename Vec<VEC>::type vec;
  constexpr int kEntries = 5 * kSlots, kAhead = 4;
  static_assert(kSlots == 4, "a list is read as one int4");
  __shared__ int counts[5][kPixels];
  __shared__ float2 entries[kPixels][kEntries + 1];  // (offset of the source in floats, coefficient)
  const int P = H * W, p0 = first_pixel();
  if (p0 >= P) return;
  int cnt[2] = {0, 0};
  unsigned src[2][kSlots];
  float cf[2][kSlots];
#pragma unroll
  for (int r = 0; r < 2; r++) {  // (pixel, list): 320 of them
    const int i = threadIdx.x + 256 * r;
    if (i >= 5 * kPixels) break;
    const int pix = i & (kPixels - 1), k = i / kPixels, p = p0 + pix;
    const int y = p / W, x = p - y * W;
    const bool has = p < P && (k == 0 || (k == 1 && x > 0) || (k == 2 && x < W - 1) || (k == 3 && y > 0) || (k == 4 && y < H - 1));
    const int ctr = has ? p + (k == 1 ? -1 : (k == 2 ? 1 : (k == 3 ? -W : (k == 4 ? W : 0)))) : 0;
    const int n = ws.count[ctr];
    const int4 e = *reinterpret_cast<const int4*>(ws.slots + (size_t)ctr * kSlots);
    cnt[r] = has ? min(n, kSlots) : 0;
    const int s[kSlots] = {e.x, e.y, e.z, e.w};
#pragma unroll
    for (int j = 0; j < kSlots; j++) {
      const unsigned from = j < cnt[r] ? (unsigned)s[j] : 0u;
      cf[r][j] = ws.coef[(size_t)k * P + from];
      src[r][j] = from * C;
    }
    counts[k][pix] = cnt[r];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int i = threadIdx.x + 256 * r;
    if (i >= 5 * kPixels) break;
    const int pix = i & (kPixels - 1), k = i / kPixels;
    int at = 0;
    for (int j = 0; j < k; j++) at += counts[j][pix];
#pragma unroll
    for (int j = 0; j < kSlots; j++)
      if (j < cnt[r]) entries[pix][at + j] = make_float2(__uint_as_float(src[r][j]), cf[r][j]);
  }
  __syncthreads();
  const int pieces = C / VEC, total = min(kPixels, P - p0) * pieces;
  const int dp = 256 / pieces, dq = 256 - dp * pieces;
  int pix = threadIdx.x / pieces, piece = threadIdx.x - pix * pieces;
  for (int i = threadIdx.x; i < total; i += 256) {
    const unsigned c = (unsigned)piece * VEC;
    const int n = counts[0][pix] + counts[1][pix] + counts[2][pix] + counts[3][pix] + counts[4][pix];
    vec acc = 0.f;
    for (int j0 = 0; j0 < n; j0 += kAhead) {
      float2 e[kAhead];
      vec v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; u++) e[u] = entries[pix][min(j0 + u, n - 1)];
#pragma unroll
      for (int u = 0; u < kAhead; u++) v[u] = *reinterpret_cast<const vec*>(im0 + __float_as_uint(e[u].x) + c);
#pragma unroll
      for (int u = 0; u < kAhead; u++)
#pragma unroll
        for (int w = 0; w < VEC; w++) acc[w] = j0 + u < n ? __builtin_fmaf(v[u][w], e[u].y, acc[w]) : acc[w];
    }
    __builtin_nontemporal_store(acc, reinterpret_cast<vec*>(g1 + (size_t)(p0 + pix) * C + c));
    piece += dq;
    pix += dp;
    if (piece >= pieces) { piece -= pieces; pix++; }
  }
}

// After the gather, with float atomics: the sources whose list was full.  One lane per (source, channel).
__global__ __launch_bounds__(256) void overflow(const float* __restrict__ im0, const float* __restrict__ flow, FlowStrides fs,
                                                float* __restrict__ g1, QfWorkspace ws, int C, int H, int W) {
  const int P = H * W;
  const long long total = (long long)*ws.ovf_count * C;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
    const int e = (int)(i / C), c = (int)(i - (long long)e * C), p = ws.ovf[e];
    TilePx px;
    locate_pixel(px, flow, fs, H, W, p, true);  // (the pixel is inside)
    unsigned o[5];
    tap_offsets(px, W, C, o);
    const float v = im0[(size_t)p * C + c];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const float cf = ws.coef[(size_t)k * P + p];
      if (cf != 0.f) unsafeAtomicAdd(g1 + o[k] + c, v * cf);
    }
  }
}

}  // namespace quadfit_image
