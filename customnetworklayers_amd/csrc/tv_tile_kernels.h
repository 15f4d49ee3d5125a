// Register-tile kernels of the TV layer: several iterations per launch on a two-dimensional tile, for problems that do not
// fill the chip.
//
// A launch of the strip kernels does two iterations and, on a small image, lasts as long as one wavefront needs to walk its
// rows one after the other, plus about 4 us for starting a grid and waiting for its first loads.  Here a workgroup of four
// wavefronts holds a tile of 64 columns x 4 R rows in registers, R rows per wavefront, one pixel per lane and row: all rows
// of an iteration are independent work for the wavefront's one instruction stream, nothing is loaded between iterations but
// the x05 rows of the reverse sweep, and a launch does K iterations, so a pass has 2 / K of the launches.  The price is the
// halo: K pixels on every side are computed for the tile's own use.  Rows of neighbouring wavefronts meet in LDS (first and
// last row of each, double-buffered, one LDS-only barrier per iteration); the triangle above a wavefront's first row is
// evaluated again rather than handed over, which would cost a second barrier.  What falls outside the tile reaches one pixel
// further in with every iteration and never an output pixel.
//
// Same arithmetic, operation by operation, as the strip kernels (and the oracle): same bits.
#pragma once

#include "exact_math.h"
#include "tv_strip_kernels.h"

namespace tvtile {

using inpaint::div_by;
using inpaint::rcp_refined;
using tvstrip::Rebuild;
using tvstrip::from_left_lane;
using tvstrip::from_right_lane;
using tvstrip::kL;
using tvstrip::ldg;
using tvstrip::lds_barrier;
using tvstrip::prox_adjoint;
using tvstrip::rebuild_of;
using tvstrip::regime_threshold;
using tvstrip::stg;

constexpr int kMaxFwdSteps = 12;  // forward iterations one launch can hold

struct FwdStep {
  float *x05, *y, *x;  // where this iteration leaves its pre-prox value and its iterate (null: nowhere)
  float t;             // extrapolation factor
};
struct FwdSteps {
  FwdStep step[kMaxFwdSteps];
};

// Forward iterations (TV.cu:1194-1319, 1321-1455), one channel per workgroup (forward channels never couple; the two
// channels of a tile are neighbours in the grid and share c and the weights in the XCD's L2).  xin, yin: the iterate, or,
// with `ring`, the x05 rows of the two iterations before (as in tv_forward_strip2).  keep_x, keep_y (optional): a copy of
// the input iterate.  48 vector instructions per pixel and iteration; bound by launch and load latency (about 4 us) and
// instruction issue on one or two wavefronts per SIMD.  1 x 2 x 64 x 128, 20 iterations: 41 us in ten strip launches, 23 us
// in three launches of 6 to 7 iterations with R = 4; 48 iterations of 1 x 2 x 187 x 621: 130 -> 82 us (R = 8, 6 per launch).
template <int R, int WAVES, bool X05>
__global__ __launch_bounds__(64 * WAVES) void tv_forward_tile(
    const float* __restrict__ wx, const float* __restrict__ wy, const float* __restrict__ cf,
    const float* __restrict__ b, const float* __restrict__ xin, const float* __restrict__ yin, FwdSteps steps, int K,
    int ring, float tP, float* __restrict__ keep_x, float* __restrict__ keep_y, int N, int C, int H, int W, int tiles_x,
    int tiles_y) {
  __shared__ float edge[2][WAVES][2][64];  // [parity][wavefront][its first row, its last row]
  constexpr int TR = R * WAVES;
  const int per_xcd = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int ch = tile % C;
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
  const bool wx_ok = col_ok && w < W - 1;
  const bool store_lane = lane >= K && lane < 64 - K && w < W;
  const unsigned W4 = 4u * (unsigned)W;
  const unsigned wc = col_ok ? 4u * w : 0u;
  const size_t HW = (size_t)H * W;
  const size_t q = ((size_t)n * C + ch) * HW;
  const float *const wx_p = wx + (size_t)n * HW, *const wy_p = wy + (size_t)n * HW, *const cf_p = cf + (size_t)n * HW;
  const float *const b_p = b + q, *const x_p = xin + q, *const y_p = yin + q;

  float y[R], x[R], bb[R], c[R], rc[R], wxs[R], wys[R], wxu, wyu;
  auto prox = [&](float yt, float cv, float rc1, float bv) {  // TV.cu:1286-1292
    float x_loc = div_by(cv * bv + yt, 1.f + cv, rc1);
    const float lo = yt - cv, hi = yt + cv;
    if (lo > 1.f + bv) x_loc = lo;
    if (hi < bv - 1.f) x_loc = hi;
    return x_loc;
  };
  {
    const int h = h0 - 1;
    const unsigned off = (unsigned)min(max(h, 0), H - 1) * W4 + wc;
    wxu = ldg(wx_p, off);
    wyu = ldg(wy_p, off);
    const bool rok = h >= 0 && h < H;
    wxu = (rok && wx_ok) ? kL * wxu : 0.f;
    wyu = (rok && col_ok && h < H - 1) ? kL * wyu : 0.f;
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    const unsigned off = (unsigned)min(max(h0 + i, 0), H - 1) * W4 + wc;
    y[i] = ldg(y_p, off);
    x[i] = ldg(x_p, off);
    bb[i] = ldg(b_p, off);
    c[i] = ldg(cf_p, off);
    wxs[i] = ldg(wx_p, off);
    wys[i] = ldg(wy_p, off);
  }
  unsigned rows = 0;  // bit i: row i is an output row of the tile inside the image
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int h = h0 + i, r = wave * R + i;
    const bool ok = col_ok && h >= 0 && h < H;
    if (r >= K && r < TR - K && h < H) rows |= 1u << i;
    // a pixel outside the image: y = x = b = c = 0 and no weight stays y = 0 through every iteration
    const inpaint::LaneMask inside(ok);
    c[i] = inside(c[i]);
    bb[i] = inside(bb[i]);
    rc[i] = rcp_refined(1.f + c[i]);
    y[i] = inside(y[i]);
    x[i] = inside(x[i]);
    wxs[i] = (ok && wx_ok) ? kL * wxs[i] : 0.f;
    wys[i] = (ok && h < H - 1) ? kL * wys[i] : 0.f;
    if (ring) {  // y holds x05[k-1], x holds x05[k-2]
      const float xj = prox(y[i], c[i], rc[i], bb[i]);
      const float xm = prox(x[i], c[i], rc[i], bb[i]);
      x[i] = xj;
      y[i] = xj + tP * (xj - xm);  // TV.cu:1315
    }
  }
  const unsigned roff0 = (unsigned)max(h0, 0) * W4 + wc;  // (stored rows have h >= 0; a tile row above the image is never stored)
  const unsigned row_base = (unsigned)(h0 < 0 ? -h0 : 0);
  auto row_off = [&](int i) { return roff0 + ((unsigned)i - row_base) * W4; };
  auto store_rows = [&](float* dst, const float (&v)[R]) {
    if (store_lane) {
#pragma unroll
      for (int i = 0; i < R; i++)
        if ((rows >> i) & 1) stg(dst, row_off(i), v[i]);
    }
  };
  if (keep_x) store_rows(keep_x + q, x);
  if (keep_y) store_rows(keep_y + q, y);
  // one triangle (owner value yc, lower neighbour yd): the two products of TV.cu:1268-1274
  auto triangle = [&](float yc, float yd, float wxv, float wyv, float& e1, float& e2) {
    const float d1 = yc - yd;
    const float d2 = yc - from_right_lane(yc);
    const inpaint::HuberForward hub = inpaint::huber_forward(d1 * d1 * wyv + d2 * d2 * wxv);
    e1 = d1 * div_by(wyv, hub.m, hub.rm);
    e2 = d2 * div_by(wxv, hub.m, hub.rm);
  };

  for (int it = 0; it < K; it++) {
    const FwdStep st = steps.step[it];
    const int p = it & 1;
    edge[p][wave][0][lane] = y[0];
    edge[p][wave][1][lane] = y[R - 1];
    lds_barrier();
    const float yu = edge[p][max(wave - 1, 0)][1][lane];          // (the tile's outermost rows have no neighbour: what they
    const float yb = edge[p][min(wave + 1, WAVES - 1)][0][lane];  // read instead only reaches rows that are not output)
    float e1_above, e2_above;
    triangle(yu, y[0], wxu, wyu, e1_above, e2_above);
    float xh[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
      float e1, e2;
      triangle(y[i], i + 1 < R ? y[i + 1 < R ? i + 1 : i] : yb, wxs[i], wys[i], e1, e2);
      float yt = y[i];
      yt -= -e1_above;            // TV.cu:1258
      yt -= -from_left_lane(e2);  // TV.cu:1265
      yt -= e1;                   // TV.cu:1272
      yt -= e2;                   // TV.cu:1273
      e1_above = e1;
      const float x_loc = prox(yt, c[i], rc[i], bb[i]);
      y[i] = x_loc + st.t * (x_loc - x[i]);
      x[i] = x_loc;
      xh[i] = yt;
    }
    if (X05 && st.x05) store_rows(st.x05 + q, xh);
    if (st.y) store_rows(st.y + q, y);
    if (st.x) store_rows(st.x + q, x);
  }
}


constexpr int kMaxAdjSteps = 12;  // reverse-sweep steps one launch can hold

struct AdjStep {
  const float* xb;       // x05 row of the iteration before (with seg >= 0: the checkpoint the segment starts from)
  const float* xa_next;  // with seg >= 0: the x05 row the next step starts at (null after the last step)
  int seg;               // >= 0: this step is the first iteration of that segment, whose sums it leaves as a record
  float t;               // extrapolation factor of the step's iteration
};
struct AdjSteps {
  AdjStep step[kMaxAdjSteps];
};
struct AdjTileArgs {
  const float *wx, *wy, *cf, *b;
  const float *xa, *x_last;                      // x05 row of the first step; FIRST: the last x05 row
  const float *g05_in, *gx_in;                   // (FIRST: g05_in is the upstream gradient, gx_in is not read)
  const float *gc_in, *gwx_in, *gwy_in, *gb_in;  // accumulators (null: zero)
  float *g05_out, *gx_out, *gc_out, *gwx_out, *gwy_out, *gb_out;  // null: not wanted
  float *gx_final;                               // the completed g_x of the launch's last step (null: not wanted)
  float *seg_gc, *seg_gwx, *seg_gwy, *seg_gb;    // record of segment 0; segment s follows s planes (fields) further
  int N, H, W, tiles_x, tiles_y, K;
};

// Steps of the reverse sweep (TV.cu:586-859, 862-1126 with the y rebuild, as tv_adjoint_strip).  CL = 2: both channels of a
// tile of 32 columns in the two halves of each wavefront -- the three accumulators they share are kept on both halves, and
// v_permlane32_swap hands every lane both channels' terms, which it adds in channel order.  The accumulators stay in
// registers over the launch; a step that is a segment's first iteration stores them as the segment's record and clears
// them, so launches need not follow the segments.  FIRST (x_last given): the sweep's first step (TV.cu:222-287) on the way
// in.  The x05 row of the next step is loaded while this one computes.  About 150 vector instructions per pixel, channel
// and step, 20 more for the extra triangle of a wavefront; bound by their issue on one wavefront per SIMD (1.5 us per step)
// and by the launch (4.4 us).  1 x 2 x 64 x 128, 20 iterations: backward pass 86 us in strips, 66 us in three launches.
template <int CL, int R, int WAVES, bool TRUE_ADJ>
__global__ __launch_bounds__(64 * WAVES) void tv_adjoint_tile(AdjTileArgs a, AdjSteps steps) {
  static_assert(CL == 1 || CL == 2, "one channel, or two in the two halves of a wavefront");
  constexpr int L = 64 / CL;  // columns of the tile
  constexpr int TR = R * WAVES;
  constexpr float kGX = TRUE_ADJ ? 1.f : tvstrip::kLocalGXMult, kGC = TRUE_ADJ ? 1.f : tvstrip::kLocalGCMult;
  __shared__ float edge[2][WAVES][4][64];  // [parity][wavefront][y, g of its first row, y, g of its last row]
  const int K = a.K, H = a.H, W = a.W;
  const int per_xcd = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const int tx = tile % a.tiles_x;
  const int rest = tile / a.tiles_x;
  const int ty = rest % a.tiles_y, n = rest / a.tiles_y;
  if (n >= a.N) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & (L - 1), ch = lane / L;
  const int w = tx * (L - 2 * K) - K + col;
  const int h0 = ty * (TR - 2 * K) - K + wave * R;
  const bool col_ok = w >= 0 && w < W;
  const bool wx_ok = col_ok && w < W - 1;
  const bool store_lane = col >= K && col < L - K && w < W;
  const unsigned W4 = 4u * (unsigned)W;
  const size_t HW = (size_t)H * W;
  const unsigned wc = col_ok ? 4u * w : 0u;             // column offset in a plane
  const unsigned wf = wc + (unsigned)ch * 4u * (unsigned)HW;  // the same in a field: this lane's channel
  const size_t poff = (size_t)n * HW, foff = poff * CL;

  float c[R], rc[R], bb[R], wxs[R], wys[R], wxu, wyu;
  float thr[R];  // the prox regime test of TV.cu:806, 1154 is |b - x05| <= thr (regime_threshold)
  float g[R], gx[R], gc[R], gwx[R], gwy[R], gb[R], xa[R], xb[R];
  unsigned rows = 0;
  {
    const int h = h0 - 1;
    const unsigned row = (unsigned)min(max(h, 0), H - 1) * W4;
    wxu = ldg(a.wx + poff, row + wc);
    wyu = ldg(a.wy + poff, row + wc);
    const bool rok = h >= 0 && h < H;
    wxu = (rok && wx_ok) ? kL * wxu : 0.f;
    wyu = (rok && col_ok && h < H - 1) ? kL * wyu : 0.f;
  }
  const unsigned base = (unsigned)max(h0, 0) * W4;  // (as in the forward kernel: stored rows lie inside the image)
  const unsigned row_base = (unsigned)(h0 < 0 ? -h0 : 0);
  auto row_off = [&](int i) { return base + ((unsigned)i - row_base) * W4; };
  auto clamp_off = [&](int i) { return (unsigned)min(max(h0 + i, 0), H - 1) * W4; };
  auto load_rows = [&](float (&v)[R], const float* p, unsigned lane_off) {
#pragma unroll
    for (int i = 0; i < R; i++) v[i] = ldg(p, clamp_off(i) + lane_off);
  };
  auto store_rows = [&](float* p, unsigned lane_off, const float (&v)[R]) {
    if (store_lane) {
#pragma unroll
      for (int i = 0; i < R; i++)
        if ((rows >> i) & 1) stg(p, row_off(i) + lane_off, v[i]);
    }
  };
  const bool first = a.x_last != nullptr;
  load_rows(c, a.cf + poff, wc);
  load_rows(wxs, a.wx + poff, wc);
  load_rows(wys, a.wy + poff, wc);
  load_rows(bb, a.b + foff, wf);
  load_rows(xa, a.xa + foff, wf);
  load_rows(xb, steps.step[0].xb + foff, wf);
  load_rows(g, a.g05_in + foff, wf);
#pragma unroll
  for (int i = 0; i < R; i++) gx[i] = gc[i] = gwx[i] = gwy[i] = gb[i] = 0.f;
  if (!first) load_rows(gx, a.gx_in + foff, wf);
  if (a.gc_in) {
    load_rows(gc, a.gc_in + poff, wc);
    load_rows(gwx, a.gwx_in + poff, wc);
    load_rows(gwy, a.gwy_in + poff, wc);
    load_rows(gb, a.gb_in + foff, wf);
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int h = h0 + i, r = wave * R + i;
    const bool ok = col_ok && h >= 0 && h < H;
    if (r >= K && r < TR - K && h < H) rows |= 1u << i;
    const inpaint::LaneMask inside(ok);
    c[i] = inside(c[i]);
    rc[i] = rcp_refined(1.f + c[i]);
    thr[i] = regime_threshold(c[i]);
    bb[i] = inside(bb[i]);
    g[i] = inside(g[i]);
    gx[i] = inside(gx[i]);
    wxs[i] = (ok && wx_ok) ? kL * wxs[i] : 0.f;
    wys[i] = (ok && h < H - 1) ? kL * wys[i] : 0.f;
  }
  auto inside_rows = [&](float (&v)[R]) {
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int h = h0 + i;
      v[i] = (col_ok && h >= 0 && h < H) ? v[i] : 0.f;
    }
  };
  // two channels: the terms of channel 0 and of channel 1, on the lanes of both
  auto both = [&](float v, float& v0, float& v1) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v0 = __uint_as_float(s[0]);
    v1 = __uint_as_float(s[1]);
  };
  auto add_shared = [&](float& acc, float v) {  // acc += v, channel 0's term before channel 1's
    if (CL == 1) {
      acc += v;
    } else {
      float v0, v1;
      both(v, v0, v1);
      acc += v0;
      acc += v1;
    }
  };
  auto sub_shared = [&](float& acc, float v) {
    if (CL == 1) {
      acc = acc - v;
    } else {
      float v0, v1;
      both(v, v0, v1);
      acc = acc - v0;
      acc = acc - v1;
    }
  };
  inside_rows(xa);
  if (first) {
    // the sweep's first step (TV.cu:240-255): the upstream gradient through the prox at the last x05 row
    float xl[R];
    load_rows(xl, a.x_last + foff, wf);
    inside_rows(xl);
#pragma unroll
    for (int i = 0; i < R; i++) {
      const float opc = 1.f + c[i], df = g[i], bv = bb[i];
      const float rc2 = rcp_refined(opc * opc);
      const float diff = bv - xl[i];
      const bool quad = (thr[i] >= fabsf(diff));
      const float gc_q = df * (div_by(bv, opc, rc[i]) - div_by(c[i] * bv + xl[i], opc * opc, rc2)) * kGC;
      const float gb_q = div_by(df * c[i], opc, rc[i]) * 1.0f;
      g[i] = quad ? div_by(df, opc, rc[i]) : df;
      add_shared(gc[i], quad ? gc_q : (diff < 0 ? -df : df) * kGC);
      gb[i] = quad ? gb[i] + gb_q : 0.f;  // (TV.cu:254 writes zero outside the quadratic regime)
    }
  }

  Rebuild ra[R];  // of xa
  auto rebuild_rows = [&]() {
#pragma unroll
    for (int i = 0; i < R; i++)
      ra[i] = TRUE_ADJ ? Rebuild{tvstrip::prox_huber1(xa[i], c[i], rc[i], bb[i]), 0.f} : rebuild_of(xa[i], bb[i], c[i], rc[i]);
  };
  rebuild_rows();
  for (int it = 0; it < K; it++) {
    const AdjStep st = steps.step[it];
    const float t = st.t;
    float xn[R], xan[R];
    if (it + 1 < K) load_rows(xn, steps.step[it + 1].xb + foff, wf);
    if (st.seg >= 0 && st.xa_next) load_rows(xan, st.xa_next + foff, wf);
    inside_rows(xb);
    auto body = [&](auto end) {
      constexpr bool END = decltype(end)::value;
      float y[R];
#pragma unroll
      for (int i = 0; i < R; i++) {
        if (TRUE_ADJ) {  // (the forward pass's own y: ra.q is prox(xa))
          const float pb = END ? xb[i] : tvstrip::prox_huber1(xb[i], c[i], rc[i], bb[i]);
          y[i] = ra[i].q + t * (ra[i].q - pb);
          ra[i].q = pb;
        } else if (END) {
          y[i] = xb[i];
        } else {
          const Rebuild r = rebuild_of(xb[i], bb[i], c[i], rc[i]);
          const float y_q = ra[i].q + t * (ra[i].q - r.q), y_l = ra[i].l + t * (ra[i].l - r.l);
          y[i] = thr[i] >= fabsf(bb[i] - xa[i]) ? y_q : y_l;
          ra[i] = r;
        }
      }
      const int p = it & 1;
      edge[p][wave][0][lane] = y[0];
      edge[p][wave][1][lane] = g[0];
      edge[p][wave][2][lane] = y[R - 1];
      edge[p][wave][3][lane] = g[R - 1];
      lds_barrier();
      const int up = max(wave - 1, 0), dn = min(wave + 1, WAVES - 1);  // (the outermost rows: see the forward kernel)
      const float yu = edge[p][up][2][lane], gu = edge[p][up][3][lane];
      const float yb = edge[p][dn][0][lane], gbelow = edge[p][dn][1][lane];
      float df_i[R];
      float d_1, d_3, d_4;  // terms handed down to the next row
#pragma unroll
      for (int i = -1; i < R; i++) {
        // everything the triangle of row i contributes (see tv_adjoint_strip; the factor tp of O3, O4 with its sign turned)
        const float yk = i < 0 ? yu : y[i < 0 ? 0 : i], gk = i < 0 ? gu : g[i < 0 ? 0 : i];
        const float yd = i + 1 < R ? y[i + 1 < R ? i + 1 : 0] : yb, gd = i + 1 < R ? g[i + 1 < R ? i + 1 : 0] : gbelow;
        const float wxv = i < 0 ? wxu : wxs[i < 0 ? 0 : i], wyv = i < 0 ? wyu : wys[i < 0 ? 0 : i];
        const float yrt = from_right_lane(yk), grt = from_right_lane(gk);
        const float d1 = yk - yd, d2 = yk - yrt;
        const float a1 = d1 * d1 * wyv, a2 = d2 * d2 * wxv;
        const inpaint::HuberAdjoint hub = inpaint::huber_adjoint(a2 + a1);
        const bool act = hub.active;
        const float nom = hub.nom, dd = hub.twice, denom = 0.5f * dd;
        const float gpd = gk - gd, gpr = gk - grt;
        const float O1 = gpd * (wyv * nom), O2 = gpr * (wxv * nom);
        const float P1 = gpd * wyv * d1, P2 = gpr * wxv * d2;
        const float tu = dd * d1 * wyv;
        const float n3 = P1 * tu, n4 = P2 * tu;
        if (i >= 0) {
          const float tp = dd * (d1 * wyv + d2 * wxv);
          const float tl = dd * d2 * wxv;
          const float O3 = -(P1 * tp), O4 = -(P2 * tp);
          const float l1 = from_left_lane(O2), l3 = from_left_lane(P2 * tl), l4 = from_left_lane(P1 * tl);
          float ux, uy;
          if (!END || TRUE_ADJ) {  // TV.cu:749-769
            ux = kGX * d2 * (gpr * (nom - a2 * denom) - gpd * d2 * d1 * denom * wyv);
            uy = kGX * d1 * (gpd * (nom - a1 * denom) - gpr * d1 * d2 * denom * wxv);
          } else {  // TV.cu:1019-1037
            const float ux_a = kGX * (gpr * d2 * (nom - a2 * denom) - gpd * d2 * d2 * d1 * denom * wyv);
            const float uy_a = kGX * (gpd * d1 * (nom - a1 * denom) - gpr * d1 * d1 * d2 * denom * wxv);
            ux = act ? ux_a : kGX * d2 * gpr;
            uy = act ? uy_a : kGX * d1 * gpd;
          }
          // (no weight gradient in the last column and row)
          sub_shared(gwx[i], w < W - 1 ? ux : 0.f);
          sub_shared(gwy[i], h0 + i < H - 1 ? uy : 0.f);
          float tt = gk;
          tt -= -d_1;  // TV.cu:668 / 684
          tt -= d_3;   // TV.cu:675
          tt -= d_4;   // TV.cu:677
          tt -= -l1;   // TV.cu:701 / 718
          tt -= l3;    // TV.cu:707
          tt -= l4;    // TV.cu:710
          tt -= O1;    // TV.cu:732 / 763
          tt -= O2;    // TV.cu:733 / 764
          tt -= O3;    // TV.cu:741
          tt -= O4;    // TV.cu:743
          // momentum adjoint, TV.cu:796-801
          float df = (float)__builtin_fma(1. + (double)t, (double)tt, (double)gx[i]);  // (see tv_adjoint_strip)
          df = fmaxf(-tvstrip::kClipLocalGrad, fminf(df, tvstrip::kClipLocalGrad));
          gx[i] = -t * tt;
          const float rc2 = rcp_refined((1.f + c[i]) * (1.f + c[i]));
          float gc_add, gb_add;
          prox_adjoint<TRUE_ADJ>(df, bb[i], xa[i], c[i], rc[i], rc2, thr[i], g[i], gc_add, gb_add);
          add_shared(gc[i], gc_add);
          gb[i] += gb_add;
          df_i[i] = df;
        }
        d_1 = O1;
        d_3 = n3;
        d_4 = n4;
      }
      if (END && a.gx_final && it == K - 1) store_rows(a.gx_final + foff, wf, df_i);
      if (END) {  // the segment's sums into its record (TV.cu:178-218)
        const size_t so = (size_t)st.seg * a.N * HW;
        if (ch == 0) {
          store_rows(a.seg_gc + so + poff, wc, gc);
          store_rows(a.seg_gwx + so + poff, wc, gwx);
          store_rows(a.seg_gwy + so + poff, wc, gwy);
        }
        store_rows(a.seg_gb + so * CL + foff, wf, gb);
#pragma unroll
        for (int i = 0; i < R; i++) {
          gc[i] = gwx[i] = gwy[i] = gb[i] = 0.f;
          xa[i] = xan[i];
        }
        inside_rows(xa);
        rebuild_rows();
      } else {
#pragma unroll
        for (int i = 0; i < R; i++) xa[i] = xb[i];
      }
    };
    if (st.seg >= 0) body(std::true_type{});
    else body(std::false_type{});
#pragma unroll
    for (int i = 0; i < R; i++) xb[i] = xn[i];
  }
  if (a.g05_out) {
    store_rows(a.g05_out + foff, wf, g);
    store_rows(a.gx_out + foff, wf, gx);
  }
  if (a.gc_out) {
    if (ch == 0) {
      store_rows(a.gc_out + poff, wc, gc);
      store_rows(a.gwx_out + poff, wc, gwx);
      store_rows(a.gwy_out + poff, wc, gwy);
    }
    store_rows(a.gb_out + foff, wf, gb);
  }
}

}  // namespace tvtile
