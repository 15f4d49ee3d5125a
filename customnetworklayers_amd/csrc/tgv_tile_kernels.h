// Register-tile kernel of the TGV layer's forward pass: several iterations per launch on a two-dimensional tile.
//
// The scheme of the TV layer's tiles: a workgroup holds a tile of 64 columns x WAVES * R rows of one channel in registers, R
// rows per wavefront, one pixel per lane and row, and does K iterations; K pixels on every side are computed for the tile's
// own use.  The first and the last row of a wavefront meet their neighbours in LDS (double-buffered, one LDS-only barrier per
// iteration); the triangle above a wavefront's first row is evaluated again rather than handed over.  What falls outside the
// tile reaches one pixel further in with every iteration and never an output pixel.
//
// Same arithmetic, operation by operation, as the strip kernels (and the oracle): same bits.
#pragma once

#include "tgv_strip_kernels.h"

namespace tgvtile {

using inpaint::div_by;
using inpaint::rcp_refined;
using tgvstrip::kHuberQuiet;
using tgvstrip::wave_any;
using tgvstrip::kD0;
using tvstrip::from_left_lane;
using tvstrip::from_right_lane;
using tvstrip::ldg;
using tvstrip::lds_barrier;
using tvstrip::stg;

// Huber weight min(1, rsqrt(A) * 0.2f), as tgvstrip::huber_w_full, without its care for A = 0: the root is a NaN there (0 times
// infinity), and the minimum of 1 and a NaN is 1, which is the weight.
__device__ __forceinline__ float huber_w_any(float A) {
  const float y = __builtin_amdgcn_rsqf(A);
  const float s = A * y;
  const float e = __builtin_fmaf(-s, s, A);
  return fminf(1.f, inpaint::exact_rcp(__builtin_fmaf(e, 0.5f * y, s)) * kD0);
}

constexpr int kMaxFwdSteps = 12;  // iterations one launch can hold

struct FwdStep {
  float *x05, *y, *x;  // where this iteration leaves its pre-prox state and its iterate (null: nowhere)
  float t;             // extrapolation factor
};
struct FwdSteps {
  FwdStep step[kMaxFwdSteps];
};

// Rows of the halo that neither a later iteration nor the output needs are skipped (a row more at either end with every iteration):
// 1 to 5% of a pass (4 x 2 x 384 x 1248 2508 -> 2484 us, 1 x 2 x 375 x 1241 at inference 589 -> 577, 2 x 2 x 224 x 512 199 -> 191); the
// wavefronts in the middle of a tile have none, and set its pace.
// Bound by instruction issue: about 80 vector instructions per pixel and iteration where the Huber terms of a row are quiet,
// 120 where none is, on two to five wavefronts per SIMD (the strips issue as many, but wait for memory every second
// iteration and read 19 planes for it).  Taller tiles waste less on the halo; 5 rows per wavefront are what fits 128 registers.
// 50 iterations of 1 x 2 x 375 x 1241: 440 us in strips, 299 in tiles of 40 rows, 7 iterations per launch; 4 x 2 x 384 x 1248:
// 1407 -> 986 in such tiles, with every x05 state kept 1538 -> 1297 (80 rows, 8 per launch); 30 iterations of 1 x 1 x 61 x 97:
// 90 -> 59 (12 rows, 5 per launch).
//
// xin, yin: the iterate, or, with `ring`, the x05 states of the two iterations before (as in tgv_forward_strip2).  keep_x,
// keep_y (optional): a copy of the input iterate.
constexpr int fwd_waves(int R) { return R >= 5 ? 4 : 5; }  // wavefronts per SIMD: 128 and 96 registers

template <int R, int WAVES, bool X05>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(fwd_waves(R), fwd_waves(R)))) void tgv_forward_tile(
    const float* __restrict__ wx, const float* __restrict__ wy, const float* __restrict__ bx, const float* __restrict__ by,
    const float* __restrict__ cf, const float* __restrict__ b, const float* __restrict__ xin, const float* __restrict__ yin,
    FwdSteps steps, int K, int ring, float tP, float* __restrict__ keep_x, float* __restrict__ keep_y, int N, int C, int H,
    int W, int tiles_x, int tiles_y) {
  __shared__ float edge[2][WAVES][2][3][64];  // [parity][wavefront][its first row, its last row][u, v1, v2]
  constexpr int TR = R * WAVES;
  const int per_xcd = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int ch = tile % C;  // (the channels of a tile are neighbours in the grid: they share c and the weights in the XCD's L2)
  int rest = tile / C;
  const int tx = rest % tiles_x;
  rest /= tiles_x;
  const int ty = rest % tiles_y, n = rest / tiles_y;
  if (n >= N) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = tx * (64 - 2 * K) - K + lane;
  const int h0 = ty * (TR - 2 * K) - K + wave * R;  // image row of this wavefront's first row
  const bool col_ok = w >= 0 && w < W;
  const bool rmask = col_ok && w < W - 1;  // the pixel has a right neighbour
  const bool store_lane = lane >= K && lane < 64 - K && w < W;
  const unsigned W4 = 4u * (unsigned)W;
  const unsigned wc = col_ok ? 4u * w : 0u;
  const size_t HW = (size_t)H * W, CHW = HW * C;
  const size_t p = (size_t)n * HW, q = ((size_t)n * 3 * C + ch) * HW;  // variable v of the channel starts v * CHW further
  const float *const b_p = b + ((size_t)n * C + ch) * HW;

  float y[3][R], x[3][R], bb[R], c[R], rc[R], wxs[R], wys[R], bxs[R], bys[R];
  float wxu, wyu, bxu, byu;  // weights of the row above
  auto prox = [&](float yt, float cv, float rc1, float bv) {  // TGV.cu:1740-1744
    float x_loc = div_by(cv * bv + yt, 1.f + cv, rc1);
    const float lo = yt - cv, hi = yt + cv;
    if (lo > 1.f + bv) x_loc = lo;
    if (hi < bv - 1.f) x_loc = hi;
    return x_loc;
  };
  {
    const int h = h0 - 1;
    const unsigned off = (unsigned)min(max(h, 0), H - 1) * W4 + wc;
    wxu = ldg(wx + p, off);
    wyu = ldg(wy + p, off);
    bxu = ldg(bx + p, off);
    byu = ldg(by + p, off);
    const bool ok = col_ok && h >= 0 && h < H;
    wxu = (ok && rmask) ? wxu : 0.f;
    wyu = (ok && h < H - 1) ? wyu : 0.f;
    bxu = ok ? bxu : 0.f;
    byu = ok ? byu : 0.f;
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    const unsigned off = (unsigned)min(max(h0 + i, 0), H - 1) * W4 + wc;
#pragma unroll
    for (int v = 0; v < 3; v++) {
      y[v][i] = ldg(yin + q + v * CHW, off);
      x[v][i] = ldg(xin + q + v * CHW, off);
    }
    bb[i] = ldg(b_p, off);
    c[i] = ldg(cf + p, off);
    wxs[i] = ldg(wx + p, off);
    wys[i] = ldg(wy + p, off);
    bxs[i] = ldg(bx + p, off);
    bys[i] = ldg(by + p, off);
  }
  unsigned rows = 0;  // bit i: row i is an output row of the tile inside the image
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int h = h0 + i, r = wave * R + i;
    const bool ok = col_ok && h >= 0 && h < H;
    if (r >= K && r < TR - K && h < H) rows |= 1u << i;
    // a pixel outside the image: y = x = b = c = 0 and no weight stays y = x = 0 through every iteration
    const inpaint::LaneMask inside(ok);
    c[i] = inside(c[i]);
    bb[i] = inside(bb[i]);
    rc[i] = rcp_refined(1.f + c[i]);
    wxs[i] = (ok && rmask) ? wxs[i] : 0.f;
    wys[i] = (ok && h < H - 1) ? wys[i] : 0.f;
    bxs[i] = inside(bxs[i]);
    bys[i] = inside(bys[i]);
#pragma unroll
    for (int v = 0; v < 3; v++) {
      y[v][i] = inside(y[v][i]);
      x[v][i] = inside(x[v][i]);
    }
    if (ring) {  // y holds x05[k-1], x holds x05[k-2]
      const float xj = prox(y[0][i], c[i], rc[i], bb[i]);
      const float xm = prox(x[0][i], c[i], rc[i], bb[i]);
      x[0][i] = xj;
      y[0][i] = xj + tP * (xj - xm);  // TGV.cu:1773
#pragma unroll
      for (int v = 1; v < 3; v++) {
        const float xv = y[v][i], xmv = x[v][i];
        x[v][i] = xv;
        y[v][i] = xv + tP * (xv - xmv);  // TGV.cu:1686-1690
      }
    }
  }
  auto store_rows = [&](float* dst, const float (&v)[R]) {
    if (store_lane) {
#pragma unroll
      for (int i = 0; i < R; i++)
        if ((rows >> i) & 1) stg(dst + (size_t)(h0 + i) * W, tgvstrip::offset_here(wc), v[i]);
    }
  };
  auto store_state = [&](float* dst, const float (&s)[3][R]) {
#pragma unroll
    for (int v = 0; v < 3; v++) store_rows(dst + q + v * CHW, s[v]);
  };
  if (keep_x) store_state(keep_x, x);
  if (keep_y) store_state(keep_y, y);
  struct Tri {  // the six products of one triangle (TGV.cu:1669-1684)
    float Fa, Fb, G1y, G1x, G2y, G2x;
  };
  // Iterations of a tile.  INNER: every pixel of the tile has its right and its lower neighbour in the image.
  auto iterate = [&](auto inner) {
    constexpr bool INNER = decltype(inner)::value;
    auto triangle = [&](float yc, float y1c, float y2c, float yd, float y1d, float y2d, float wxv, float wyv, float bxv, float byv,
                        bool has_lower) {
      const bool r = INNER || rmask, d = INNER || has_lower;
      // all differences ahead of the branches: the shifts then ride on the subtractions (and outside the selects: a shift
      // reads its neighbour's register, whatever that lane selects)
      float dr = yc - from_right_lane(yc), d1r = y1c - from_right_lane(y1c), d2r = y2c - from_right_lane(y2c);
      asm volatile("" : "+v"(dr), "+v"(d1r), "+v"(d2r));  // (here: behind a branch each shift is two instructions more)
      float z1 = r ? dr + y1c : 0.f, z2 = d ? (yc - yd) + y2c : 0.f;
      float u11 = r ? d1r : 0.f, u12 = d ? y1c - y1d : 0.f;
      float u21 = r ? d2r : 0.f, u22 = d ? y2c - y2d : 0.f;
      const float A = z2 * z2 * wyv + z1 * z1 * wxv;
      const float B1 = bxv * (u12 * u12 + u11 * u11), B2 = byv * (u22 * u22 + u21 * u21);
      // (a weight of 1, where all lanes are quiet, needs no product)
      if (wave_any(A > kHuberQuiet)) {
        const float hw = huber_w_any(A);
        z1 *= hw;
        z2 *= hw;
      }
      if (wave_any(fmaxf(B1, B2) > kHuberQuiet)) {
        const float h1 = huber_w_any(B1), h2 = huber_w_any(B2);
        u11 *= h1;
        u12 *= h1;
        u21 *= h2;
        u22 *= h2;
      }
      return Tri{wyv * z2, wxv * z1, bxv * u12, bxv * u11, byv * u22, byv * u21};
    };
    for (int it = 0; it < K; it++) {
      const FwdStep st = steps.step[it];
      const int par = it & 1;
#pragma unroll
      for (int v = 0; v < 3; v++) {
        edge[par][wave][0][v][lane] = y[v][0];
        edge[par][wave][1][v][lane] = y[v][R - 1];
      }
      lds_barrier();
      float yu[3], yb[3];  // (the tile's outermost rows have no neighbour: what they read instead only reaches rows that are not output)
#pragma unroll
      for (int v = 0; v < 3; v++) {
        yu[v] = edge[par][max(wave - 1, 0)][1][v][lane];
        yb[v] = edge[par][min(wave + 1, WAVES - 1)][0][v][lane];
      }
      // rows of this wavefront that a later iteration or the output still needs
      const int lo = max(it + 1 - wave * R, 0), hi = min(TR - 2 - it - wave * R, R - 1);
      Tri above{};
      if (lo == 0) above = triangle(yu[0], yu[1], yu[2], y[0][0], y[1][0], y[2][0], wxu, wyu, bxu, byu, h0 - 1 >= 0 && h0 - 1 < H - 1);
      float xh[R];
#pragma unroll
      for (int i = 0; i < R; i++) {
        if (i + 1 < lo || i > hi) continue;
        const int j = i + 1 < R ? i + 1 : i;
        const Tri t = triangle(y[0][i], y[1][i], y[2][i], i + 1 < R ? y[0][j] : yb[0], i + 1 < R ? y[1][j] : yb[1],
                               i + 1 < R ? y[2][j] : yb[2], wxs[i], wys[i], bxs[i], bys[i], h0 + i >= 0 && h0 + i < H - 1);
        if (i < lo) {
          above = t;
          continue;
        }
        float yt = y[0][i], y1n = y[1][i], y2n = y[2][i];
        yt -= -above.Fa;               // TGV.cu:1637
        y1n -= -above.G1y;             // TGV.cu:1638
        y2n -= -above.G2y;             // TGV.cu:1639
        yt -= -from_left_lane(t.Fb);   // TGV.cu:1665
        y1n -= -from_left_lane(t.G1x); // TGV.cu:1666
        y2n -= -from_left_lane(t.G2x); // TGV.cu:1667
        yt -= t.Fa;                    // TGV.cu:1678
        y1n -= t.G1y;                  // TGV.cu:1679
        y2n -= t.G2y + t.Fa;           // TGV.cu:1680
        yt -= t.Fb;                    // TGV.cu:1682
        y1n -= t.G1x + t.Fb;           // TGV.cu:1683
        y2n -= t.G2x;                  // TGV.cu:1684
        above = t;
        float x_loc = prox(yt, c[i], rc[i], bb[i]);
        y[0][i] = x_loc + st.t * (x_loc - x[0][i]);  // TGV.cu:1772
        y[1][i] = y1n + st.t * (y1n - x[1][i]);      // TGV.cu:1686-1687
        y[2][i] = y2n + st.t * (y2n - x[2][i]);
        // computed here: left to itself the compiler sinks every row's update to the end of the iteration, with all that
        // goes into it kept in registers until then (253 registers with R = 8, where 168 do)
        asm volatile("" : "+v"(y[0][i]), "+v"(y[1][i]), "+v"(y[2][i]), "+v"(x_loc), "+v"(y1n), "+v"(y2n));
        x[0][i] = x_loc;
        x[1][i] = y1n;
        x[2][i] = y2n;
        if (X05) xh[i] = yt;
      }
      if (X05 && st.x05) {
        store_rows(st.x05 + q, xh);
        store_rows(st.x05 + q + CHW, x[1]);
        store_rows(st.x05 + q + 2 * CHW, x[2]);
      }
      if (st.y) store_state(st.y, y);
      if (st.x) store_state(st.x, x);
    }
  };
  const int tw0 = tx * (64 - 2 * K) - K, th0 = ty * (TR - 2 * K) - K;
  if (tw0 >= 0 && tw0 + 64 < W && th0 >= 0 && th0 + TR < H) iterate(std::true_type{});
  else iterate(std::false_type{});
}

}  // namespace tgvtile
