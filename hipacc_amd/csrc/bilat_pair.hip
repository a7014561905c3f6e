// bilat_pair.hip -- bilateral filter on float images, each pixel pair's
// weight evaluated once (hh_bilat_pair.hpp).
//
// Per pair of pixels: difference, exponent, exponential (two issue slots) and
// the four sums of the pair; the tile kernel (bilateral.hip) spends 7 slots on
// each of the pair's two taps.  The sums are of d = X(q) - X(p), so that
// Y(p) = X(p) + SUM s d / SUM s: their rounding scales with the local contrast
// instead of the pixel's value (13x13 over 4096^2 pixels in [0, 1]: 3e-8 off
// the 64-bit result in the 2-norm, the tile kernel 2.8e-7).
//
// RAW forms d from the pixels themselves (halved, so that the difference of
// any two finite pixels is finite) and the exponent in two instructions, 9
// slots a pair: the weights and the norm are as exact as the tile kernel's.
// Without RAW the pixels are scaled by sqrt(c log2 e) first and the exponent
// is one FMA, 8 slots.  Rounding the scaled pixel moves a weight by its last
// place times the pixel's size over sigma; the sums of s d hide that below the
// last place of Y, but the norm, which the backward reads, would show it
// (pixels 1000 .. 1001 at sigma 0.1: norm 5e-4 off, Y 7e-8).  No value of one
// pixel enters another's sums in either form except through s.
//
// Tile kernel and here, us: 4096^2 13x13 527 and 411, 7x7 175 and 119;
// 16 x 1024^2 7x7 173 and 125, RAW 137.  VALU issue bound.
#include <cmath>

#include "hh_bilat_pair.hpp"

namespace hh {

typedef float pair_f4 __attribute__((ext_vector_type(4), aligned(4)));

template <int R, bool RAW>
__global__ __launch_bounds__(256, R <= 4 ? 4 : 3) void bilat_pair_kernel(const BilatArgs a, const PairGeom pg) {
  constexpr int V = 4, K = 2 * R + 1, HL = (R + V - 1) / V, NW = V + 2 * R;
  __shared__ __align__(16) float4 part[3][R][2][64];   // first R rows of waves 1..3: den, num
  const Geom& g = a.g;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const PairLane pl = pair_lane<HL>(pg, lane, 3 * pg.n + pg.n0);
  const float* in = static_cast<const float*>(g.in) + (long long)pl.b * g.in_plane;
  const int yw = pl.y0 + (wave == 0 ? 0 : pg.n0 + (wave - 1) * pg.n);   // first row of the segment
  const int nrow = wave == 0 ? pg.n0 : pg.n;
  const LaneCols<V> cols = lane_cols<V>(g, g.in_ox + pl.x);
  bool raw = true;   // the lane's 4 pixels are adjacent in memory
#pragma unroll
  for (int e = 0; e < V; ++e) raw = raw && !cols.cst[e] && cols.x[e] == cols.x[0] + e;

  const int lead = wave == 0 ? R : 0;      // rows walked above the segment
  const int ys = yw - lead;                // first row walked
  const int steps = nrow + lead;
  // rows ys .. ys + steps + R + 1 are loaded
  int lx, hx, ly, hy;
  raw_region(g, lx, hx, ly, hy);
  const bool walk = __all(raw && g.in_oy + ys >= ly && g.in_oy + ys + steps + R + 2 <= hy);
  const float* next = in + (long long)(g.in_oy + ys) * g.in_stride + cols.x[0];

  // Pixels of row y (iteration space), boundary handling applied; called for
  // consecutive rows from ys on.
  auto load_row = [&](int y, float (&v)[V]) {
    if (walk) {
      const pair_f4 q = *reinterpret_cast<const pair_f4*>(next);
      next += g.in_stride;
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = q[e];
      return;
    }
    bool rc;
    const int yy = row_src(g, g.in_oy + y, rc);
    const float* row = in + (long long)yy * g.in_stride;
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = row[cols.x[e]];
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = rc || cols.cst[e] ? g.const_f : v[e];
  };

  const float k2 = (float)(-4.0 * a.scale * a.scale);   // RAW: of halved differences
  const float sc = RAW ? 0.5f : (float)a.scale;
  // (as the sum of two floats: a factor's own rounding would move every pixel)
  const double inv = 1.0 / (double)sc;
  const float isc = (float)inv, iscl = (float)(inv - (double)isc);
  const float s0 = __builtin_amdgcn_exp2f(a.lsp[R * K + R]);
  // Scaled pixels are held within a limit: a finite pixel must not become
  // infinite (0 * inf would spread NaN where the weight is 0).  Pixels beyond
  // it differ by far more than sigma from every other value, so their own
  // output is the pixel (`limited`, uniform over the wave: some are).
  constexpr float kLimit = 1e38f;
  bool limited = false;
  auto hold = [&](const float (&v)[V], float (&x)[V]) {
#pragma unroll
    for (int e = 0; e < V; ++e) x[e] = v[e] * sc;
    if constexpr (!RAW) {
      static_assert(V == 4, "pixels per lane");
      const float m = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(x[0]), __builtin_fabsf(x[1])),
                                      __builtin_fmaxf(__builtin_fabsf(x[2]), __builtin_fabsf(x[3])));
      if (__any(m >= kLimit)) {
        limited = true;
#pragma unroll
        for (int e = 0; e < V; ++e)   // (infinities and NaN stay)
          x[e] = __builtin_fabsf(v[e]) <= 3.402823466e38f
                     ? __builtin_amdgcn_fmed3f(x[e], -kLimit, kLimit) : v[e];
      }
    }
  };
  // x, den, num: pixels of row y as held and their sums (without the centre tap)
  auto finish = [&](int y, const float (&x)[V], const float (&den)[V], const float (&num)[V]) {
    if (!pl.store || y >= g.is_h) return;
    float r[V], n[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
      n[e] = den[e] + s0;
      // with a centre weight the sum is no denormal and the reciprocal's last
      // bit only scales the correction SUM s d / SUM s
      const float q = s0 > 1e-30f ? num[e] * __builtin_amdgcn_rcpf(n[e]) : num[e] / n[e];
      const float xq = x[e] + q;
      r[e] = RAW ? xq * isc : __builtin_fmaf(xq, isc, xq * iscl);
    }
    float* dst = static_cast<float*>(g.out) + (long long)pl.b * g.out_plane +
                 (long long)(g.out_oy + y) * g.out_stride + g.out_ox + pl.x;
    float* nrm = a.norm ? a.norm + (long long)pl.b * a.norm_plane +
                              (long long)y * a.norm_stride + pl.x
                        : nullptr;
    if (pl.x + V <= g.is_w) {
      pair_f4 q = {r[0], r[1], r[2], r[3]};
      __builtin_nontemporal_store(q, reinterpret_cast<pair_f4*>(dst));
      if (nrm) {
        pair_f4 m = {n[0], n[1], n[2], n[3]};
        __builtin_nontemporal_store(m, reinterpret_cast<pair_f4*>(nrm));
      }
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e)
        if (pl.x + e < g.is_w) {
          dst[e] = r[e];
          if (nrm) nrm[e] = n[e];
        }
    }
  };

  float xr[R + 1][V], nx[V];               // rows y .. y + R as held; row y + R + 1 as loaded
  float den[R + 1][V], num[R + 1][V];      // sums of rows y .. y + R
  {
    float v[R + 1][V];
#pragma unroll
    for (int k = 0; k <= R; ++k) load_row(ys + k, v[k]);
    load_row(ys + R + 1, nx);
#pragma unroll
    for (int k = 0; k <= R; ++k) {
      hold(v[k], xr[k]);
#pragma unroll
      for (int e = 0; e < V; ++e) den[k][e] = num[k][e] = 0.0f;
    }
  }
#pragma unroll 1
  for (int r = 0; r < steps; ++r) {
    const int y = ys + r;
    if (!__any(y < g.is_h)) break;         // the rest of the band is below the image
    float nn[V];
    load_row(y + R + 2, nn);
#pragma unroll
    for (int dy = 0; dy <= R; ++dy) {
      if (r + dy < lead) continue;         // pairs of rows above the segment
      // The window of row y + dy slides over the offsets: its element m is
      // first used at dx = m - R - 3 and its sums are complete after
      // dx = m - R, when they go to the lane that owns the column.
      float win[NW], wd[NW], wn[NW];
      auto column = [](int m, int& d, int& e) {
        const int rel = m - R;
        d = rel >= 0 ? rel / V : -((-rel + V - 1) / V);
        e = rel - d * V;
      };
      const int first = dy == 0 ? 1 : -R;
#pragma unroll
      for (int dx = first; dx <= R; ++dx) {
        const float l = a.lsp[(R + dy) * K + R + dx];
#pragma unroll
        for (int m = dx == first ? dx + R : dx + R + V - 1; m < dx + R + V; ++m) {
          int d, e;
          column(m, d, e);
          win[m] = lane_shift(xr[dy][e], d);
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const int m = e + dx + R;
          const float d = win[m] - xr[0][e];
          const float s = __builtin_amdgcn_exp2f(RAW ? __builtin_fmaf(d * d, k2, l)
                                                     : __builtin_fmaf(-d, d, l));
          den[0][e] += s;
          num[0][e] = __builtin_fmaf(s, d, num[0][e]);
          if (dx == first || e == V - 1) {
            wd[m] = s;
            wn[m] = -s * d;
          } else {
            wd[m] += s;
            wn[m] = __builtin_fmaf(-s, d, wn[m]);
          }
        }
        // (one offset later: a DPP read right after the write would wait)
#pragma unroll
        for (int m = dx == first ? NW : dx + R - 1; m < (dx == R ? NW : dx + R); ++m) {
          int d, e;
          column(m, d, e);
          den[dy][e] += lane_shift(wd[m], -d);
          num[dy][e] += lane_shift(wn[m], -d);
          asm volatile("" : "+v"(den[dy][e]), "+v"(num[dy][e]));
        }
        // the sums are pinned per offset: left alone, the compiler sinks
        // their additions past the row and keeps hundreds of weights live
        // (9x9: 119 registers against more than 256)
#pragma unroll
        for (int e = 0; e < V; ++e) asm volatile("" : "+v"(den[0][e]), "+v"(num[0][e]));
      }
    }
    const int rs = r - lead;               // row of the segment
    if (rs >= 0) {
      if (wave > 0 && rs < R) {
        part[wave - 1][rs][0][lane] = make_float4(den[0][0], den[0][1], den[0][2], den[0][3]);
        part[wave - 1][rs][1][lane] = make_float4(num[0][0], num[0][1], num[0][2], num[0][3]);
      } else {
        finish(y, xr[0], den[0], num[0]);
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int e = 0; e < V; ++e) {
        xr[k][e] = xr[k + 1][e];
        den[k][e] = den[k + 1][e];
        num[k][e] = num[k + 1][e];
      }
    hold(nx, xr[R]);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      nx[e] = nn[e];
      den[R][e] = num[R][e] = 0.0f;
    }
  }
  __syncthreads();
  if (wave < 3) {
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const float4 pd = part[wave][k][0][lane], pn = part[wave][k][1][lane];
      const float d[V] = {den[k][0] + pd.x, den[k][1] + pd.y, den[k][2] + pd.z, den[k][3] + pd.w};
      const float m[V] = {num[k][0] + pn.x, num[k][1] + pn.y, num[k][2] + pn.z, num[k][3] + pn.w};
      finish(yw + nrow + k, xr[k], d, m);
    }
  }
  if (!RAW && limited && pl.store) {
    // outputs this wave wrote of pixels beyond the limit, except NaN ones (an
    // infinity or a NaN in the window)
    const int y1 = min(yw + nrow + (wave < 3 ? R : 0), g.is_h);
    for (int y = yw + (wave == 0 ? 0 : R); y < y1; ++y) {
      bool rc;
      const int yy = row_src(g, g.in_oy + y, rc);
      for (int e = 0; e < V && pl.x + e < g.is_w; ++e) {
        const LaneCols<1> col = lane_cols<1>(g, g.in_ox + pl.x + e);
        const float v = rc || col.cst[0] ? g.const_f : in[(long long)yy * g.in_stride + col.x[0]];
        if (!(__builtin_fabsf(v * sc) >= kLimit)) continue;
        float* dst = static_cast<float*>(g.out) + (long long)pl.b * g.out_plane +
                     (long long)(g.out_oy + y) * g.out_stride + g.out_ox + pl.x + e;
        const float old = *dst;
        if (old == old) *dst = v;
      }
    }
  }
}

int dispatch_bilat_pair(const BilatArgs& a, hipStream_t s) {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 256;
    return n;
  }();
  const Geom& g = a.g;
  if (g.in_dtype != HIPACC_F32 || g.out_dtype != HIPACC_F32 || g.cvt == HIPACC_CVT_ROUND)
    return HIPACC_ERR_UNSUPPORTED;
  // the exponent's factor stays far from the ends of the float range
  if (!(a.scale > 1e-15 && a.scale < 1e15)) return HIPACC_ERR_UNSUPPORTED;
  const int kk = a.ksize * a.ksize, r = a.ksize / 2;
  // The centre's weight must be the table's largest: Y is formed from the
  // centre pixel, so its last place is part of the error even where the pixel
  // has little part in Y (no weight at all in a table with a hole there).
  for (int t = 0; t < kk; ++t)
    if (!(a.lsp[t] == a.lsp[kk - 1 - t] && a.lsp[t] <= a.lsp[kk / 2])) return HIPACC_ERR_UNSUPPORTED;
  if (r < 2 || r > 7) return HIPACC_ERR_UNSUPPORTED;
  // Issue slots of a SIMD, both ways: a tile block is one wave per SIMD of 4
  // pixels x 7 slots a tap, a row of this kernel 4 pixels x 8.9 slots a pair
  // (both plus staging).  One block per CU waits for each row's loads and for
  // the pairs' chains, which more blocks hide: 250 slots a row.  The long
  // segments lose where the image does not fill the device a few times over
  // (us, tile and pair): 5x5 at 1920x1080 16.0 and 18.0, at 4 x 1024^2 29.6
  // and 31.7, at 1500^2 17.4 and 16.2; 7x7 at 1001x751 12.9 and 14.7, at
  // 1920x1080 24.7 and 25.5, at 1500^2 28.8 and 23.6; 13x13 at 1024^2 38 and
  // 43, at 1920x1080 69 and 66, at 2048^2 137 and 116.  RAW costs the pair
  // kernel up to a tenth of that and moves no line between the two sizes.
  const double tile = (double)ceil_div(ceil_div(g.is_w, 64) * ceil_div(g.is_h, 16) * g.batch, cus) *
                      (28.0 * kk + 300.0);
  const double row = 17.8 * kk + 180.0, first = 500.0, alone = 250.0;
  // (the shortest segments, before the search for the best ones)
  if (tile < (kPairRows + 1.0) * row + first) return HIPACC_ERR_UNSUPPORTED;
  const PairGeom pg = pair_geom(g.is_w, g.is_h, g.batch, r, cus);
  if (pg.blocks == 0) return HIPACC_ERR_UNSUPPORTED;
  const int rounds = ceil_div(pg.blocks, cus);
  if (tile < rounds * (pg.n + 1.0) * (row + (rounds == 1 ? alone : 0.0)) + first)
    return HIPACC_ERR_UNSUPPORTED;
  // Scaled pixels only where no norm is asked for, and where scaling neither
  // takes small pixels below the float range nor large ones to its limit.
  const bool raw = a.norm || !(a.scale > 1e-3 && a.scale < 1e9);
#define HH_BP(R)                                                                             \
  case R:                                                                                    \
    if (raw)                                                                                 \
      hipLaunchKernelGGL((bilat_pair_kernel<R, true>), dim3(pg.blocks), dim3(256), 0, s, a, pg);  \
    else                                                                                     \
      hipLaunchKernelGGL((bilat_pair_kernel<R, false>), dim3(pg.blocks), dim3(256), 0, s, a, pg); \
    break;
  switch (r) {
    HH_BP(2) HH_BP(3) HH_BP(4) HH_BP(5) HH_BP(6) HH_BP(7)
    default: return HIPACC_ERR_UNSUPPORTED;
  }
#undef HH_BP
  return hip_status(hipGetLastError(), "bilat_pair_kernel launch");
}

}  // namespace hh
