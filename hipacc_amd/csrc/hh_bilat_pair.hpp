// hh_bilat_pair.hpp -- lane layout shared by the bilateral kernels that
// evaluate each pixel pair once (bilat_pair.hip).
//
// The weight of a pair of pixels (p, q) is the same seen from either end when
// the spatial table is point-symmetric, and it costs most of a tap (the
// difference, the exponent, one exponential).  So a lane walks its pixels p
// down the rows and, for the half plane of offsets below and to the right of
// p, adds each weight to the sums of both p and q = p + o.  The rows q lies in
// are up to R below: their sums are kept in registers (R + 1 rows) and leave
// when p reaches them.  q may belong to a neighbour lane: the sums a lane
// makes for the 4 + 2 R columns around its 4 pixels are formed locally and
// the outer ones handed over through DPP wave shifts once per row pair.
//
// Lanes are laid out over "bands" of rows: a band of an image is a row of
// G = ceil(w / 4) pixel groups with HL = ceil(R / 4) halo groups at either
// end, and the bands of all images follow each other in one sequence of
// groups that waves cut into pieces of 64 - 2 HL (plus HL lanes of overlap at
// either side).  Narrow images therefore fill whole waves: at 1024 columns
// 4 % of the lanes are halo, where one strip per wave would idle 20 %.
//
// The 4 waves of a block take consecutive row segments of the same groups.
// A wave's sums for the R rows after its segment would have to be made again
// by the next wave (R extra rows of pairs per segment); instead the next wave
// leaves the sums of its first R rows in LDS and, after the barrier, the
// upper wave adds its share and finishes those rows.  Only the first wave of
// a block walks R rows above its segment.
#pragma once

#include "hh_stream.hpp"

namespace hh {

struct PairGeom {
  int groups;       // 4-pixel groups of an image row
  int lb;           // groups of a band with its halo
  int n, n0;        // rows of a wave's segment; of a block's first wave
  int bands;        // per image
  int total;        // groups of all bands of all images
  int blocks;
};

constexpr int kPairRows = 4;   // of a segment, at least

// Rows of a wave: the first wave's segment is shorter by the time of the rows
// it walks above it (half of their pairs).  n minimises the blocks a CU gets x
// the rows of a wave, with 1.5 rows for a segment's start and end.
static inline PairGeom pair_geom(int w, int h, int batch, int r, int cus, int most = 1 << 30) {
  PairGeom best{};
  const int hl = (r + 3) / 4, s = 64 - 2 * hl;
  double bt = 0.0;
  for (int n = r > kPairRows ? r : kPairRows; n <= 512; n += n < 128 ? 1 : 16) {
    PairGeom p;
    p.groups = ceil_div(w, 4);
    p.lb = p.groups + 2 * hl;
    p.n = n;
    p.n0 = n - (r + 2) / 2 > 1 ? n - (r + 2) / 2 : 1;
    const int rows = 3 * n + p.n0;
    p.bands = ceil_div(h, rows);
    const long long total = (long long)p.bands * batch * p.lb;
    if (total >= (1ll << 30)) continue;
    p.total = (int)total;
    p.blocks = ceil_div(p.total, s);
    if (p.blocks > most) continue;
    const int rounds = ceil_div(p.blocks, cus);
    // one or two waves per SIMD wait for their rows, the edge waves most
    const double t = (double)rounds * (n + 1.5) * (rounds == 1 ? 1.25 : rounds == 2 ? 1.08 : 1.0);
    if (bt == 0.0 || t < bt) {
      bt = t;
      best = p;
    }
    if (rows >= h) break;
  }
  return best;
}

// Lane's place: image, first row of its band, first column of its group
// (iteration space; may lie outside the image), whether it stores.
struct PairLane {
  int b, y0, x;
  bool store;
};
template <int HL>
__device__ __forceinline__ PairLane pair_lane(const PairGeom& pg, int lane, int rows) {
  PairLane l;
  const int u = (int)blockIdx.x * (64 - 2 * HL) + lane - HL;
  const int uc = min(max(u, 0), pg.total - 1);
  const int band = uc / pg.lb;
  const int i = uc - band * pg.lb - HL;
  l.b = band / pg.bands;
  l.y0 = (band - l.b * pg.bands) * rows;
  l.x = i * 4;
  l.store = lane >= HL && lane < 64 - HL && u < pg.total && i >= 0 && i < pg.groups;
  return l;
}

}  // namespace hh
