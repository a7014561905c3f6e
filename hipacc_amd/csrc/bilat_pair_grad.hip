// bilat_pair_grad.hip -- backward of the bilateral filter (grad_bilat.hip)
// with each pixel pair evaluated once, in the lane layout of
// hh_bilat_pair.hpp.
//
// With D = X(q) - X(p), a = dY / norm, z = X - Y and b = 2c a z, the pair's
// weight s serves the centre terms of both pixels (S2 = SUM s D^2 and, for
// dL/dc, S3 = SUM s D^3 towards the neighbour, and the pixel's own b with
// SUM s D) and the neighbour term of each (through the other's a and b):
//   N(q) += a(p) s [1 - 2c D^2] - [b(p) + b(q)] s D
//   N(p) += a(q) s [1 - 2c D^2] + [b(q) + b(p)] s D
//   dX(t) = N(t) + a(t) s(centre) + 2c a(t) S2(t)
//   dL/dc = -SUM_t [a(t) S3(t) + a(t) z(t) S2(t)]
// (SUM s D is also (Y - X) norm, which would save the addition of the two b,
// but -2c z^2 dY in its place squares the rounding of Y: an image of 1e6, flat
// over the window, with Y one last place off would get 0.4 dY for 0.)
// Differences are those of the pixels themselves (halved, so that the
// difference of any two finite pixels is finite), and every product starts
// with s: a weight of 0 leaves out a neighbour however far its value is.
//
// 18 issue slots a pair against 13 a tap in the tile kernel: 7x7 at
// 16 x 1024^2 367 us there, 276 here (CONSTANT, without a halo ring), VALU
// issue bound.
#include <cmath>

#include "hh_bilat_pair.hpp"
#include "hh_grad.hpp"

namespace hh {

typedef float pair_f4 __attribute__((ext_vector_type(4), aligned(4)));

template <int R>
__global__ __launch_bounds__(256, 2) void bilat_pair_grad_kernel(const BilatGradArgs a,
                                                                 const PairGeom pg) {
  constexpr int V = 4, K = 2 * R + 1, HL = (R + V - 1) / V, NW = V + 2 * R;
  __shared__ __align__(16) float4 part[3][R][3][64];  // first R rows of waves 1..3: N, S2, S3
  __shared__ double red[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const PairLane pl = pair_lane<HL>(pg, lane, 3 * pg.n + pg.n0);
  const float* X = a.x + (long long)pl.b * a.x_plane;
  const float* Y = a.y + (long long)pl.b * a.y_plane;
  const float* Dn = a.d + (long long)pl.b * a.d_plane;
  const float* Gy = a.gy + (long long)pl.b * a.gy_plane;
  const int yw = pl.y0 + (wave == 0 ? 0 : pg.n0 + (wave - 1) * pg.n);
  const int nrow = wave == 0 ? pg.n0 : pg.n;
  const int lead = wave == 0 ? R : 0;
  const int ys = yw - lead, steps = nrow + lead;
  const bool cmode = a.boundary == HIPACC_BOUNDARY_CONSTANT;
  const bool inside = pl.x >= 0 && pl.x + V <= a.w;
  // rows ys .. ys + steps + R + 1 are loaded
  const bool walk = __all(inside && ys >= 0 && ys + steps + R + 2 <= a.h);
  int xi[V];         // column each pixel of X reads; of the others, clamped
  int ci[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    ci[e] = min(max(pl.x + e, 0), a.w - 1);
    xi[e] = cmode ? ci[e] : bh_map(a.boundary, pl.x + e, 0, a.w, a.w);
  }

  struct Row {
    float x[V], y[V], d[V], g[V];
  };
  // Row y of the four images: X through its boundary handling, dY 0 outside
  // the image (no output there) and Y, norm any finite value.
  auto load_row = [&](int y, Row& r) {
    if (walk) {
      const pair_f4 qx = *reinterpret_cast<const pair_f4*>(X + (long long)y * a.x_stride + pl.x);
      const pair_f4 qy = *reinterpret_cast<const pair_f4*>(Y + (long long)y * a.y_stride + pl.x);
      const pair_f4 qd = *reinterpret_cast<const pair_f4*>(Dn + (long long)y * a.d_stride + pl.x);
      const pair_f4 qg = *reinterpret_cast<const pair_f4*>(Gy + (long long)y * a.gy_stride + pl.x);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        r.x[e] = qx[e];
        r.y[e] = qy[e];
        r.d[e] = qd[e];
        r.g[e] = qg[e];
      }
      return;
    }
    const int yc = min(max(y, 0), a.h - 1);
    const int yx = cmode ? yc : bh_map(a.boundary, y, 0, a.h, a.h);
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const bool in = y >= 0 && y < a.h && pl.x + e >= 0 && pl.x + e < a.w;
      const float x = X[(long long)yx * a.x_stride + xi[e]];
      r.x[e] = cmode && !in ? a.cval : x;
      r.y[e] = Y[(long long)yc * a.y_stride + ci[e]];
      const float d = Dn[(long long)yc * a.d_stride + ci[e]];
      r.d[e] = in ? d : 1.0f;
      const float g = Gy[(long long)yc * a.gy_stride + ci[e]];
      r.g[e] = in ? g : 0.0f;
    }
  };

  // of halved differences h: s = 2^(l + k2 h^2), 2c D^2 = c8 h^2, b D = (4c a z) h
  const float k2 = (float)(-4.0 * a.scale * a.scale), c8 = 8.0f * a.c, c4 = 4.0f * a.c;
  const float s0 = a.sp[R * K + R];
  float xr[R + 1][V], ar[R + 1][V], br[R + 1][V];      // rows y .. y + R
  float nn[R + 1][V], s2[R + 1][V], s3[R + 1][V];      // their sums
  // a loaded row becomes row k of the window; N starts with the term of the
  // pixel alone (own; the first R rows of waves 1..3 start with it in the
  // wave above)
  auto enter = [&](const Row& r, int k, bool own) {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const float av = r.g[e] / r.d[e];
      xr[k][e] = 0.5f * r.x[e];
      ar[k][e] = av;
      br[k][e] = c4 * (av * (r.x[e] - r.y[e]));
      nn[k][e] = own ? av * s0 : 0.0f;
      s2[k][e] = 0.0f;
      s3[k][e] = 0.0f;
    }
  };
  const double rc = 1.0 / (double)a.c;
  double dc = 0.0;   // the two terms cancel largely, and the pixels' sums too
  auto finish = [&](int y, const float (&av)[V], const float (&bv)[V], const float (&n)[V],
                    const float (&t2)[V], const float (&t3)[V]) {
    if (!pl.store || y >= a.h) return;
    float v[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
      v[e] = __builtin_fmaf(c8 * av[e], t2[e], n[e]);
      // a and b are 0 for the columns beside the image; D^3 = 8 h^3, and
      // a z D^2 = b h^2 / c in the halved differences' b
      dc += 8.0 * ((double)av[e] * (double)t3[e]) + rc * ((double)bv[e] * (double)t2[e]);
    }
    float* dst = a.gx + (long long)pl.b * a.gx_plane + (long long)y * a.gx_stride + pl.x;
    if (pl.x + V <= a.w) {
      const pair_f4 q = {v[0], v[1], v[2], v[3]};
      *reinterpret_cast<pair_f4*>(dst) = q;
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e)
        if (pl.x + e < a.w) dst[e] = v[e];
    }
  };

  Row nx;                                  // row y + R + 1 as loaded
  {
    Row r[R + 1];
#pragma unroll
    for (int k = 0; k <= R; ++k) load_row(ys + k, r[k]);
    load_row(ys + R + 1, nx);
#pragma unroll
    for (int k = 0; k <= R; ++k) enter(r[k], k, wave == 0 || k == R);
  }
#pragma unroll 1
  for (int r = 0; r < steps; ++r) {
    const int y = ys + r;
    if (!__any(y < a.h)) break;            // the rest of the band is below the image
    Row nr;
    load_row(y + R + 2, nr);
#pragma unroll
    for (int dy = 0; dy <= R; ++dy) {
      if (r + dy < lead) continue;         // pairs of rows above the segment
      // the window slides as in bilat_pair_kernel
      float wx[NW], wa[NW], wb[NW], on[NW], o2[NW], o3[NW];
      auto column = [](int m, int& d, int& e) {
        const int rel = m - R;
        d = rel >= 0 ? rel / V : -((-rel + V - 1) / V);
        e = rel - d * V;
      };
      const int first = dy == 0 ? 1 : -R;
#pragma unroll K
      for (int dx = first; dx <= R; ++dx) {
        const float l = a.lsp[(R + dy) * K + R + dx];
#pragma unroll
        for (int m = dx == first ? dx + R : dx + R + V - 1; m < dx + R + V; ++m) {
          int d, e;
          column(m, d, e);
          wx[m] = lane_shift(xr[dy][e], d);
          wa[m] = lane_shift(ar[dy][e], d);
          wb[m] = lane_shift(br[dy][e], d);
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const int m = e + dx + R;
          const float d = wx[m] - xr[0][e];
          const float s = __builtin_amdgcn_exp2f(__builtin_fmaf(d * d, k2, l));
          const float sd = s * d, t2 = sd * d;
          const float sp = __builtin_fmaf(-c8, t2, s), bs = wb[m] + br[0][e];
          nn[0][e] = __builtin_fmaf(wa[m], sp, nn[0][e]);
          nn[0][e] = __builtin_fmaf(bs, sd, nn[0][e]);
          s2[0][e] += t2;
          s3[0][e] = __builtin_fmaf(t2, d, s3[0][e]);
          if (dx == first || e == V - 1) {
            on[m] = ar[0][e] * sp;
            o2[m] = t2;
            o3[m] = -t2 * d;
          } else {
            on[m] = __builtin_fmaf(ar[0][e], sp, on[m]);
            o2[m] += t2;
            o3[m] = __builtin_fmaf(-t2, d, o3[m]);
          }
          on[m] = __builtin_fmaf(-bs, sd, on[m]);
        }
        // one offset later: a DPP read right after the write would wait
#pragma unroll
        for (int m = dx == first ? NW : dx + R - 1; m < (dx == R ? NW : dx + R); ++m) {
          int d, e;
          column(m, d, e);
          nn[dy][e] += lane_shift(on[m], -d);
          s2[dy][e] += lane_shift(o2[m], -d);
          s3[dy][e] += lane_shift(o3[m], -d);
          asm volatile("" : "+v"(nn[dy][e]), "+v"(s2[dy][e]), "+v"(s3[dy][e]));
        }
#pragma unroll
        for (int e = 0; e < V; ++e)        // pinned per offset as in bilat_pair_kernel
          asm volatile("" : "+v"(nn[0][e]), "+v"(s2[0][e]), "+v"(s3[0][e]));
      }
    }
    const int rs = r - lead;
    if (rs >= 0) {
      if (wave > 0 && rs < R) {
        part[wave - 1][rs][0][lane] = make_float4(nn[0][0], nn[0][1], nn[0][2], nn[0][3]);
        part[wave - 1][rs][1][lane] = make_float4(s2[0][0], s2[0][1], s2[0][2], s2[0][3]);
        part[wave - 1][rs][2][lane] = make_float4(s3[0][0], s3[0][1], s3[0][2], s3[0][3]);
      } else {
        finish(y, ar[0], br[0], nn[0], s2[0], s3[0]);
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int e = 0; e < V; ++e) {
        xr[k][e] = xr[k + 1][e];
        ar[k][e] = ar[k + 1][e];
        br[k][e] = br[k + 1][e];
        nn[k][e] = nn[k + 1][e];
        s2[k][e] = s2[k + 1][e];
        s3[k][e] = s3[k + 1][e];
      }
    enter(nx, R, true);
    nx = nr;
  }
  __syncthreads();
  if (wave < 3) {
    // rows of the next wave's segment: its sums plus this wave's share
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int y = yw + nrow + k;
      const float4 pn = part[wave][k][0][lane], p2 = part[wave][k][1][lane],
                   p3 = part[wave][k][2][lane];
      const float n[V] = {nn[k][0] + pn.x, nn[k][1] + pn.y, nn[k][2] + pn.z, nn[k][3] + pn.w};
      const float t2[V] = {s2[k][0] + p2.x, s2[k][1] + p2.y, s2[k][2] + p2.z, s2[k][3] + p2.w};
      const float t3[V] = {s3[k][0] + p3.x, s3[k][1] + p3.y, s3[k][2] + p3.z, s3[k][3] + p3.w};
      finish(y, ar[k], br[k], n, t2, t3);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) dc += __shfl_xor(dc, off, 64);
  if (lane == 0) red[wave] = dc;
  __syncthreads();
  if (threadIdx.x == 0)
    a.partials[blockIdx.x] = (float)(-(((red[0] + red[1]) + red[2]) + red[3]));
}

int dispatch_bilat_pair_grad(const BilatGradArgs& a, int* nblocks, hipStream_t s) {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 256;
    return n;
  }();
  const int r = a.ksize / 2, kk = a.ksize * a.ksize;
  if (!a.gx || !a.sym || r < 2 || r > 4) return HIPACC_ERR_UNSUPPORTED;
  if (!(a.scale > 1e-15 && a.scale < 1e15)) return HIPACC_ERR_UNSUPPORTED;   // as forward
  // Issue slots of a SIMD, both ways, as in dispatch_bilat_pair; a single round
  // of blocks, two waves a SIMD at most, waits for 600 slots a row (us, tile
  // and pair): 5x5 at 419x2622 22.4 and 23.8, at 2 x 384x3552 39.6 and 44.2, at
  // 1500^2 37.4 and 36.3; 7x7 at 1001x751 25.5 and 28.2, at 1920x1080 56.5 and
  // 49.6, at 2048^2 98 and 82; 9x9 at 1024^2 40.6 and 43.0, at 365x3458 48.9
  // and 49.5, at 1500^2 79.5 and 74.4.
  const double tile = (double)ceil_div(a.ntiles, cus) * (54.0 * kk + 900.0);
  const double row = 33.0 * kk + 300.0, first = 1500.0, alone = 600.0;
  if (tile < (kPairRows + 1.0) * row + first) return HIPACC_ERR_UNSUPPORTED;
  const PairGeom pg = pair_geom(a.w, a.h, a.batch, r, cus, kGradBlocks);
  if (pg.blocks == 0) return HIPACC_ERR_UNSUPPORTED;
  const int rounds = ceil_div(pg.blocks, cus);
  if (tile < rounds * (pg.n + 1.0) * (row + (rounds == 1 ? alone : 0.0)) + first)
    return HIPACC_ERR_UNSUPPORTED;
  switch (r) {
    case 2: hipLaunchKernelGGL((bilat_pair_grad_kernel<2>), dim3(pg.blocks), dim3(256), 0, s, a, pg); break;
    case 3: hipLaunchKernelGGL((bilat_pair_grad_kernel<3>), dim3(pg.blocks), dim3(256), 0, s, a, pg); break;
    default: hipLaunchKernelGGL((bilat_pair_grad_kernel<4>), dim3(pg.blocks), dim3(256), 0, s, a, pg); break;
  }
  *nblocks = pg.blocks;
  return hip_status(hipGetLastError(), "bilat_pair_grad_kernel launch");
}

}  // namespace hh
