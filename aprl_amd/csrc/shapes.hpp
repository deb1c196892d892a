// Source-shape machinery shared by the FP64 and FP32-split particle paths:
// cell-tile node boxes, the chord crossing cuts, the taps of one chord
// segment before the shape's fixed convolution, and that convolution on the
// way into (gathers) and out of (deposit) a tile's box in LDS.
//
// Every function is a template on the real type R: double with coordinates
// from the grid's origin, or float (FP32-split) with coordinates taken
// relative to the particle's own start cell. The weights are the
// reference's (longitudinal_shape.h), summed in another order.
#pragma once

#include "fixedsum.hpp"
#include "tilecounts.hpp"

#include "particles.hpp"

namespace aprl_gpu {

enum : int { kShapeQuintic = 0, kShapeBinomial3X = 2 };

// Extended node box of a cell tile per shape: every tap of a chord that
// starts in the tile and moves less than one cell per axis lies inside.
// (X0, Y0, Z0) is the box origin below the tile origin; RZ is how many
// neighbour tiles the box reaches along z (one along x and y).
template <int SHAPE>
struct Box;
template <>
struct Box<kShapeBinomial3X> {
  // binomialXZSegment taps: x [i-1, i+2], y [j, j+1], z [k-1, k+2]
  static constexpr int X0 = 2, Y0 = 1, Z0 = 2;
  static constexpr int NX = kTileX + 5, NY = kTileY + 3, NZ = kTileZ + 5;
  static constexpr int RZ = 1;
  // a chord puts at most 1 + 1/12 of its current on one raw node (its
  // segments' linear weights sum to at most 1, their curvature terms to
  // width^2 / 12), and the smoothing averages
  static constexpr double kWeightBound = 1.125;
};
template <>
struct Box<kShapeQuintic> {
  // quintic Gauss-point taps: x [i, i+1], y [j, j+1], z [k-5, k+6]
  static constexpr int X0 = 1, Y0 = 1, Z0 = 6;
  static constexpr int NX = kTileX + 3, NY = kTileY + 3, NZ = kTileZ + 13;
  static constexpr int RZ = 2;
  // a chord's raw weights sum to at most 1; the compensation's absolute
  // values to about 3.01
  static constexpr double kWeightBound = 3.125;
};
template <int SHAPE>
constexpr int boxNodes() {
  return Box<SHAPE>::NX * Box<SHAPE>::NY * Box<SHAPE>::NZ;
}

// The source shapes are a plain spline convolved with fixed weights:
// binomial3-x is the linear shape smoothed by (1, 2, 1)/4 in x and z, the
// compensated quintic the degree-5 / degree-4 B-spline in z convolved with
// seven compensation weights. A chord's taps are therefore few before that
// convolution ("raw" taps: 12 instead of 64 per segment, 44 instead of 92
// per Gauss point), and the convolution is the same for every particle: it
// is applied once per tile box. Raw node box of a tile: X0, Y0, Z0 below the
// tile origin; HX and HZ are the convolution's reach, Box the raw box
// widened by it.
template <int SHAPE>
struct RawBox;
template <>
struct RawBox<kShapeBinomial3X> {
  // linear taps x [i, i+1], y [j, j+1], z [k, k+1]
  static constexpr int X0 = 1, Y0 = 1, Z0 = 1, HX = 1, HZ = 1;
  static constexpr int NX = kTileX + 3, NY = kTileY + 3, NZ = kTileZ + 3;
};
template <>
struct RawBox<kShapeQuintic> {
  // taps x [i, i+1], y [j, j+1], z [k-2, k+3]
  static constexpr int X0 = 1, Y0 = 1, Z0 = 3, HX = 0, HZ = 3;
  static constexpr int NX = kTileX + 3, NY = kTileY + 3, NZ = kTileZ + 7;
};
template <int SHAPE>
constexpr int rawNodes() {
  using B = Box<SHAPE>;
  using W = RawBox<SHAPE>;
  static_assert(B::X0 == W::X0 + W::HX && B::Y0 == W::Y0 && B::Z0 == W::Z0 + W::HZ, "raw box origin");
  static_assert(B::NX == W::NX + 2 * W::HX && B::NY == W::NY && B::NZ == W::NZ + 2 * W::HZ, "raw box extent");
  return W::NX * W::NY * W::NZ;
}

template <int SHAPE>
struct TileBox {
  int x0, y0, z0;
  // raw box: whether it contains the raw nodes [i, i + wx) x [j, j + wy) x
  // [k, k + wz) (unsigned differences: a wild index fails), and the index
  // of one
  __device__ bool rawHolds(int i, int j, int k, int wx, int wy, int wz) const {
    using W = RawBox<SHAPE>;
    return static_cast<unsigned>(i - (x0 + W::HX)) <= static_cast<unsigned>(W::NX - wx) &&
           static_cast<unsigned>(j - y0) <= static_cast<unsigned>(W::NY - wy) &&
           static_cast<unsigned>(k - (z0 + W::HZ)) <= static_cast<unsigned>(W::NZ - wz);
  }
  __device__ int rawIndex(int i, int j, int k) const {
    using W = RawBox<SHAPE>;
    return ((k - (z0 + W::HZ)) * W::NY + (j - y0)) * W::NX + (i - (x0 + W::HX));
  }
};
template <int SHAPE>
__device__ __forceinline__ TileBox<SHAPE> tileBox(int tile, int ntx, int nty) {
  const int tx = tile % ntx, ty = (tile / ntx) % nty, tz = tile / (ntx * nty);
  return TileBox<SHAPE>{tx * kTileX - Box<SHAPE>::X0, ty * kTileY - Box<SHAPE>::Y0, tz * kTileZ - Box<SHAPE>::Z0};
}

// Crossing cuts of longitudinal_shape::weights (longitudinal_shape.h:100-103):
// chord start x and displacement v in lattice units; the face crossings as
// chord fractions, with 0 and 1, in ascending order.
constexpr int kMaxCuts = 10;
template <class R>
__device__ int orbitCuts(const R x[3], const R v[3], R cuts[kMaxCuts], unsigned& err) {
  int count = 2;
  cuts[0] = R(0.);
  cuts[1] = R(1.);
  for (int a = 0; a < 3; ++a) {
    if (v[a] != R(0.)) {
      const R lo = fmin(x[a], x[a] + v[a]), hi = fmax(x[a], x[a] + v[a]);
      for (long long j = static_cast<long long>(floor(lo)) + 1; j < hi; ++j) {
        if (count == kMaxCuts) { err |= kErrCrossings; return count; }
        cuts[count++] = (static_cast<R>(j) - x[a]) / v[a];
      }
    }
  }
  for (int s = 1; s < count; ++s) {  // insertion sort, same order as std::sort
    const R key = cuts[s];
    int t = s - 1;
    while (t >= 0 && cuts[t] > key) { cuts[t + 1] = cuts[t]; --t; }
    cuts[t + 1] = key;
  }
  return count;
}

// Compensation weight q of the quintic (longitudinal_shape.h:25-55): the
// seven-point correction of the degree-5 spline's three lowest moments.
__device__ __forceinline__ constexpr double quinticCompensation(int q) {
  const double p = 5., a = p / 6., b = 3 * p / 40. + p * (p - 1) / 72.,
               d = 5 * p / 112. + p * (p - 1) / 80. + p * (p - 1) * (p - 2) / 1296.;
  const int m = q < 3 ? q : 6 - q;
  return m == 0 ? -d / 64.
                : (m == 1 ? b / 16. + 3 * d / 32.
                          : (m == 2 ? -a / 4. - b / 4. - 15 * d / 64. : 1 + a / 2. + 3 * b / 8. + 5 * d / 16.));
}

// The quintic's weights along z on one segment: for t = g + hz s, s in
// [-1, 1], the averages over s of the degree-5 (degree-4) spline's six (five)
// pieces, of s times them and (degree 4) of s^2 times them, all times
// DEGREE!. The pieces are polynomials in t measured from the cell's middle,
// and a piece and its mirror image differ in the sign of t's odd powers: the
// averages of the powers are formed once and every two mirrored pieces from
// one even and one odd sum.
struct SplineMoments {
  double a[6], b[6], c[5];  // averages of t^j, s t^j, s^2 t^j
};
__device__ __forceinline__ SplineMoments splineMoments(double g, double hz) {
#pragma clang fp contract(fast)
  const double g2 = g * g, z2 = hz * hz, z4 = z2 * z2;
  SplineMoments m;
  m.a[1] = g;
  m.a[2] = g2 + z2 * (1. / 3.);
  m.a[3] = g * (g2 + z2);
  m.a[4] = g2 * (g2 + 2. * z2) + z4 * .2;
  m.a[5] = g * (g2 * (g2 + (10. / 3.) * z2) + z4);
  m.b[1] = hz * (1. / 3.);
  m.b[2] = (2. / 3.) * hz * g;
  m.b[3] = hz * (g2 + .2 * z2);
  m.b[4] = hz * g * ((4. / 3.) * g2 + .8 * z2);
  m.b[5] = hz * (g2 * ((5. / 3.) * g2 + 2. * z2) + z4 * (1. / 7.));
  m.c[1] = g * (1. / 3.);
  m.c[2] = g2 * (1. / 3.) + z2 * .2;
  m.c[3] = g * (g2 * (1. / 3.) + .6 * z2);
  m.c[4] = g2 * (g2 * (1. / 3.) + 1.2 * z2) + z4 * (1. / 7.);
  return m;
}

// The raw taps of one chord segment [first, last] (see RawBox): corner(i, j,
// k) reports the segment's lowest raw node, then tap(d, oi, oj, ok, w) each
// tap's component, offset from that node and weight. The integrals of
// longitudinal_shape.h:61-117 before the shape's convolution. corner returns whether
// the wave's taps all lie inside; they then go to tapInside, else to tap.
// The quintic's integrands are polynomials of degree 6 along a segment, which
// lies in one cell: the weights come from the moments of the z spline
// (splineMoments) instead of its values at four quadrature points, 330
// instead of 700 instructions a segment. They are formed in FP64 from
// positions relative to the cell in both forms: one midpoint stands for four
// points, whose roundings would average out. Against quadruple precision
// the rms error is 1.6e-17 instead of 8e-16 (FP64, 32 cells from the grid's
// origin) and 1.5e-17 instead of 1.5e-8 (FP32-split).
template <int SHAPE, class R, class Corner, class TapInside, class Tap>
__device__ __forceinline__ void rawSegment(int nx, int ny, const int org[3], const R x[3], const R v[3], R first, R last,
                                           Corner corner, TapInside tapInside, Tap tapAny) {
#pragma clang fp contract(fast)
  const R width = last - first;
  const R mid = (first + last) * R(0.5);
  const R px = x[0] + mid * v[0], py = x[1] + mid * v[1], pz = x[2] + mid * v[2];
  int li = static_cast<int>(floor(px)), lj = static_cast<int>(floor(py));
  const int lk = static_cast<int>(floor(pz));
  int i = li + org[0], j = lj + org[1];
  if (i == nx) { --i; --li; }
  if (j == ny) { --j; --lj; }
  const R cx = static_cast<R>(li), cy = static_cast<R>(lj), cz = static_cast<R>(lk);
  if constexpr (SHAPE == kShapeBinomial3X) {
    const int k = lk + org[2];
    const R wx[2] = {R(1.) - (px - cx), px - cx}, wy[2] = {R(1.) - (py - cy), py - cy},
            wz[2] = {R(1.) - (pz - cz), pz - cz};
    const R sign[2] = {R(-1.), R(1.)};
    const R curvature = width * width * R(1. / 12.);
    const R xy = curvature * v[0] * v[1];
    const R xz = curvature * v[0] * v[2];
    const R yz = curvature * v[1] * v[2];
    auto taps = [&](auto tap) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          tap(0, 0, a, b, width * (wy[a] * wz[b] + yz * sign[a] * sign[b]));
          tap(1, a, 0, b, width * (wx[a] * wz[b] + xz * sign[a] * sign[b]));
          tap(2, a, b, 0, width * (wx[a] * wy[b] + xy * sign[a] * sign[b]));
        }
    };
    if (corner(i, j, k)) taps(tapInside);
    else taps(tapAny);
  } else {
    const bool inside = corner(i, j, lk + org[2] - 2);
    double at[3], half[3];
    const R cell[3] = {cx, cy, cz};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double vd = static_cast<double>(v[d]);
      at[d] = (static_cast<double>(x[d]) - static_cast<double>(cell[d])) +
              .5 * (static_cast<double>(first) + static_cast<double>(last)) * vd;
      half[d] = .5 * (static_cast<double>(last) - static_cast<double>(first)) * vd;
    }
    const double wide = static_cast<double>(last) - static_cast<double>(first);
    const double fx = at[0], gx = 1. - at[0], hx = half[0];
    auto taps = [&](auto tap) {
      const SplineMoments m = splineMoments(at[2] - .5, half[2]);
      {
        // pieces 3 + h (and mirrored 2 - h) of 120 times the degree-5 spline
        constexpr double c[3][6] = {{52.5625, 48.125, -27.5, -35., 5., 10.},
                                    {7.40625, 23.4375, 26.25, 7.5, -7.5, -5.},
                                    {.03125, .3125, 1.25, 2.5, 2.5, 1.}};
        const double scale = wide * (1. / 120.);
        const double x0 = scale * gx, x1 = scale * fx, xh = scale * hx;
        const double y0 = scale * (1. - at[1]), y1 = scale * at[1], yh = scale * half[1];
#pragma unroll
        for (int h = 0; h < 3; ++h) {
          const double even = c[h][0] + (c[h][2] * m.a[2] + c[h][4] * m.a[4]);
          const double odd = c[h][1] * m.a[1] + (c[h][3] * m.a[3] + c[h][5] * m.a[5]);
          const double oddS = c[h][1] * m.b[1] + (c[h][3] * m.b[3] + c[h][5] * m.b[5]);
          const double evenS = c[h][2] * m.b[2] + c[h][4] * m.b[4];
#pragma unroll
          for (int mirror = 0; mirror < 2; ++mirror) {
            const int q = mirror ? 2 - h : 3 + h;
            const double n0 = mirror ? even - odd : even + odd, n1 = mirror ? evenS - oddS : evenS + oddS;
            tap(0, 0, 0, q, n0 * y0 - n1 * yh);
            tap(0, 0, 1, q, n0 * y1 + n1 * yh);
            tap(1, 0, 0, q, n0 * x0 - n1 * xh);
            tap(1, 1, 0, q, n0 * x1 + n1 * xh);
          }
        }
      }
      {
        // pieces 2 + h (and mirrored 2 - h) of 24 times the degree-4 spline
        constexpr double c[3][5] = {{14.375, 0., -15., 0., 6.}, {4.75, 11., 6., -4., -4.}, {.0625, .5, 1.5, 2., 1.}};
        const double scale = wide * (1. / 24.);
        const double y0 = scale * (1. - at[1]), y1 = scale * at[1], yh = scale * half[1];
#pragma unroll
        for (int h = 0; h < 3; ++h) {
          const double even = c[h][0] + (c[h][2] * m.a[2] + c[h][4] * m.a[4]);
          const double evenS = c[h][2] * m.b[2] + c[h][4] * m.b[4];
          const double evenSS = c[h][0] * (1. / 3.) + (c[h][2] * m.c[2] + c[h][4] * m.c[4]);
          const double odd = c[h][1] * m.a[1] + c[h][3] * m.a[3];
          const double oddS = c[h][1] * m.b[1] + c[h][3] * m.b[3];
          const double oddSS = c[h][1] * m.c[1] + c[h][3] * m.c[3];
#pragma unroll
          for (int mirror = 0; mirror < (h ? 2 : 1); ++mirror) {
            const int q = mirror ? 2 - h : 2 + h;
            const double n0 = h == 0 ? even : (mirror ? even - odd : even + odd);
            const double n1 = h == 0 ? evenS : (mirror ? evenS - oddS : evenS + oddS);
            const double n2 = h == 0 ? evenSS : (mirror ? evenSS - oddSS : evenSS + oddSS);
            const double u0 = n0 * gx - n1 * hx, u1 = n0 * fx + n1 * hx;
            const double s0 = n1 * gx - n2 * hx, s1 = n1 * fx + n2 * hx;
            tap(2, 0, 0, q, u0 * y0 - s0 * yh);
            tap(2, 1, 0, q, u1 * y0 - s1 * yh);
            tap(2, 0, 1, q, u0 * y1 + s0 * yh);
            tap(2, 1, 1, q, u1 * y1 + s1 * yh);
          }
        }
      }
    };
    if (inside) taps(tapInside);
    else taps(tapAny);
  }
}

// One raw tap of a deposit whose segment touches nodes outside the tile's
// raw box or the component's y (quintic: and x) range: the reference's
// errors (longitudinal_shape.h:181-185), nothing for a tap that reaches no
// node of the component, else its index in the raw box (-1: none).
template <int SHAPE>
__device__ __forceinline__ int rawDepositIndex(const TileBox<SHAPE>& box, const int n[3], int i, int j, int k,
                                               unsigned& err) {
  using W = RawBox<SHAPE>;
  if (i < -W::HX || i >= n[0] + W::HX) {
    if (W::HX == 0) err |= kErrCurrentX;
    return -1;
  }
  if (j < 0 || j >= n[1]) {
    err |= kErrCurrentY;
    return -1;
  }
  if (k < -W::HZ || k >= n[2] + W::HZ) return -1;
  if (!box.rawHolds(i, j, k, 1, 1, 1)) {
    err |= kErrTileHalo;
    return -1;
  }
  return box.rawIndex(i, j, k);
}

// Which taps of component d (extents n) of a segment with lowest raw node
// (i, j, k) are added: bit tapBit(oi, oj, ok) each, all of them when the
// segment lies inside the tile's raw box and the components' x and y ranges.
__device__ __forceinline__ constexpr unsigned tapBit(int oi, int oj, int ok) {
  return 1u << ((ok * 2 + oj) * 2 + oi);
}
template <int SHAPE>
__device__ __forceinline__ bool rawDepositInside(const TileBox<SHAPE>& box, int nx, int ny, int i, int j, int k) {
  return box.rawHolds(i, j, k, 2, 2, SHAPE == kShapeQuintic ? 6 : 2) && j >= 0 && j < ny &&
         (RawBox<SHAPE>::HX > 0 || (i >= 0 && i < nx));
}
template <int SHAPE>
__device__ __forceinline__ unsigned rawDepositMask(const TileBox<SHAPE>& box, const int n[3], int d, int i, int j,
                                                   int k, unsigned& err) {
  const int wx = d == 0 ? 1 : 2, wy = d == 1 ? 1 : 2;
  const int wz = SHAPE == kShapeQuintic ? (d == 2 ? 5 : 6) : (d == 2 ? 1 : 2);
  unsigned mask = 0;
#pragma unroll 1
  for (int t = 0; t < 4 * wz; ++t) {
    const int oi = t & 1, oj = (t >> 1) & 1, ok = t >> 2;
    if (oi < wx && oj < wy && rawDepositIndex<SHAPE>(box, n, i + oi, j + oj, k + ok, err) >= 0) mask |= 1u << t;
  }
  return mask;
}

// The raw box of a tile of several chunks (TileBoxes).
template <int SHAPE>
__device__ __forceinline__ long long* rawBoxOf(const TileBoxes& T, int firstChunk, int slot) {
  return T.raw + static_cast<size_t>(T.byChunk ? firstChunk - slot : slot) * 3 * rawNodes<SHAPE>();
}

// The owner side's table of the covering tiles of tile (tx, ty, tz): threads
// 0..9(2RZ+1)-1 fill, per neighbour offset (oz + RZ, oy + 1, ox + 1), the
// box (its occupied slot; -1: unoccupied) and the exponent from the tile
// scan. The caller synchronizes before reading it.
template <int SHAPE>
__device__ __forceinline__ void coveringTiles(const unsigned long long* tileScan, const int* tileShift, int tx,
                                              int ty, int tz, int ntx, int nty, int ntz, int* nbBox, int* nbShift) {
  constexpr int RZ = Box<SHAPE>::RZ, NB = 9 * (2 * RZ + 1);
  if (threadIdx.x >= NB) return;
  const int nb = static_cast<int>(threadIdx.x);
  const int x = tx + nb % 3 - 1, y = ty + (nb / 3) % 3 - 1, z = tz + nb / 9 - RZ;
  int box = -1, sh = 0;
  if (x >= 0 && x < ntx && y >= 0 && y < nty && z >= 0 && z < ntz) {
    const int s = (z * nty + y) * ntx + x;
    const unsigned long long sc = tileScan[s];
    if (chunkField(tileScan[s + 1]) > chunkField(sc)) {
      box = occupiedField(sc);
      sh = tileShift[s];
    }
  }
  nbBox[nb] = box;
  nbShift[nb] = sh;
}

// Owner-side sums of lattice node (i, j, k) of tile (tx, ty, tz), the
// components' three values together (their addresses differ by a constant,
// and three loads are in flight per covering tile): over the neighbour tiles
// whose extended box covers the node, in ascending (z, y, x) tile order, the
// tiles' sums converted with that tile's exponent. has: whether the component
// owns the node.
template <int SHAPE>
__device__ __forceinline__ void ownedNodeSums(const long long* boxes, const int* nbBox, const int* nbShift, int tx, int ty,
                                              int tz, int i, int j, int k, const bool has[3], double sum[3]) {
  using B = Box<SHAPE>;
  constexpr int N = boxNodes<SHAPE>(), RZ = B::RZ;
  // tile t' covers node i when t'*T - X0 <= i < t'*T - X0 + NX
  auto lowTile = [](int v, int t0, int n, int tile) {
    const int a = v + t0 - n + tile;  // floor((v + t0 - n) / tile) + 1 for v + t0 - n >= -tile
    return a >= 0 ? a / tile : -((-a + tile - 1) / tile);
  };
  const int xLo = max(tx - 1, lowTile(i, B::X0, B::NX, kTileX)), xHi = min(tx + 1, (i + B::X0) / kTileX);
  const int yLo = max(ty - 1, lowTile(j, B::Y0, B::NY, kTileY)), yHi = min(ty + 1, (j + B::Y0) / kTileY);
  const int zLo = max(tz - RZ, lowTile(k, B::Z0, B::NZ, kTileZ)), zHi = min(tz + RZ, (k + B::Z0) / kTileZ);
  sum[0] = sum[1] = sum[2] = 0.0;
  for (int z = zLo; z <= zHi; ++z)
    for (int y = yLo; y <= yHi; ++y)
      for (int x = xLo; x <= xHi; ++x) {
        const int nb = ((z - tz + RZ) * 3 + (y - ty + 1)) * 3 + (x - tx + 1);
        const int box = nbBox[nb];
        if (box < 0) continue;
        const int li = i - (x * kTileX - B::X0), lj = j - (y * kTileY - B::Y0), lk = k - (z * kTileZ - B::Z0);
        const long long* const at = boxes + static_cast<size_t>(box) * 3 * N + (lk * B::NY + lj) * B::NX + li;
        long long v[3] = {0, 0, 0};
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (has[d]) v[d] = at[d * N];
#pragma unroll
        for (int d = 0; d < 3; ++d) sum[d] += ldexp(static_cast<double>(v[d]), -nbShift[nb]);
      }
}

// The node loop of the owner reduction of one tile: node(i, j, k, has, sum)
// for every lattice node some component owns (the last tile of an axis also
// owns the closing node). ne: the components' extents.
template <int SHAPE, class Node>
__device__ __forceinline__ void reduceOwnedTile(const int ne[3][3], int tile, const unsigned long long* tileScan,
                                                const int* tileShift, const long long* boxes, int ntx, int nty, int ntz,
                                                Node node) {
  constexpr int NB = 9 * (2 * Box<SHAPE>::RZ + 1);
  const int tx = tile % ntx, ty = (tile / ntx) % nty, tz = tile / (ntx * nty);
  __shared__ int nbBox[NB], nbShift[NB];
  coveringTiles<SHAPE>(tileScan, tileShift, tx, ty, tz, ntx, nty, ntz, nbBox, nbShift);
  __syncthreads();
  const int nx = ne[0][0], ny = ne[1][1], nz = ne[2][2];  // cells
  const int i0 = tx * kTileX, wx = (tx == ntx - 1 ? nx + 1 : i0 + kTileX) - i0;
  const int j0 = ty * kTileY, wy = (ty == nty - 1 ? ny + 1 : j0 + kTileY) - j0;
  const int k0 = tz * kTileZ, wz = (tz == ntz - 1 ? nz + 1 : k0 + kTileZ) - k0;
  for (int t = threadIdx.x; t < wx * wy * wz; t += blockDim.x) {
    const int i = i0 + t % wx, j = j0 + (t / wx) % wy, k = k0 + t / (wx * wy);
    const bool has[3] = {i < nx, j < ny, k < nz};
    double sum[3];
    ownedNodeSums<SHAPE>(boxes, nbBox, nbShift, tx, ty, tz, i, j, k, has, sum);
    node(i, j, k, has, sum);
  }
}

// A tile's box from its raw box (3 components each): the shape's convolution,
// one thread per (x, y) column of the box, each node's exact sum rounded once
// to the fixed-point unit. Binomial3-x (weights 1, 2, 1 twice, then a division
// by 16) keeps its sums as 16 h + l; the quintic sums whole numbers in FP64, a
// raw sum's high and low words apart (quinticQuotient). Nodes outside a
// component (of nx x ny x nz cells) are not written; none of them is read.
template <int SHAPE>
__device__ __forceinline__ void convolveRawBox(const long long* raw, const TileBox<SHAPE>& box, int nx, int ny, int nz,
                                               long long* slot) {
  using B = Box<SHAPE>;
  using W = RawBox<SHAPE>;
  constexpr int N = boxNodes<SHAPE>(), NR = rawNodes<SHAPE>(), P = B::NX * B::NY, PR = W::NX * W::NY;
  for (int t = threadIdx.x; t < 3 * P; t += blockDim.x) {
    const int d = t / P, r = t - d * P, ly = r / B::NX, lx = r - ly * B::NX;
    const int n0 = nx + (d != 0), n1 = ny + (d != 1), n2 = nz + (d != 2);
    const int i = box.x0 + lx, j = box.y0 + ly;
    if (i < 0 || i >= n0 || j < 0 || j >= n1) continue;
    long long* const out = slot + d * N + ly * B::NX + lx;
    const long long* const in = raw + d * NR + ly * W::NX;
    auto put = [&](int lk, long long val) {
      const int k = box.z0 + lk;
      if (k >= 0 && k < n2) out[lk * P] = val;
    };
    if constexpr (SHAPE == kShapeBinomial3X) {
      long long h0 = 0, h1 = 0;  // the two planes before, summed in x
      int l0 = 0, l1 = 0;
#pragma unroll
      for (int lk = 0; lk < B::NZ; ++lk) {
        long long h2 = 0;
        int l2 = 0;
        if (lk < W::NZ) {
          const long long* p = in + lk * PR;
          const long long a = lx >= 2 ? p[lx - 2] : 0, b = lx >= 1 && lx <= W::NX ? p[lx - 1] : 0,
                          c = lx < W::NX ? p[lx] : 0;
          h2 = (a >> 4) + 2 * (b >> 4) + (c >> 4);
          l2 = static_cast<int>(a & 15) + 2 * static_cast<int>(b & 15) + static_cast<int>(c & 15);
        }
        put(lk, h0 + 2 * h1 + h2 + ((l0 + 2 * l1 + l2 + 8) >> 4));
        h0 = h1;
        h1 = h2;
        l0 = l1;
        l1 = l2;
      }
    } else {
      double high[W::NZ], low[W::NZ];
#pragma unroll
      for (int m = 0; m < W::NZ; ++m) {
        const long long v = in[m * PR + lx];
        high[m] = static_cast<double>(static_cast<int>(v >> 32));
        low[m] = static_cast<double>(static_cast<unsigned>(v));
      }
#pragma unroll
      for (int lk = 0; lk < B::NZ; ++lk) {
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int q = 0; q < 7; ++q)
          if (lk - q >= 0 && lk - q < W::NZ) {
            a = fma(kQuinticNum[q], high[lk - q], a);
            b = fma(kQuinticNum[q], low[lk - q], b);
          }
        put(lk, quinticQuotient(a, b));
      }
    }
  }
}

// The deposit side's write-out of one chunk's LDS raw box acc (3
// components). A tile of one chunk writes its box; chunks of a larger tile
// add their nonzero raw sums to the tile's raw box with integer atomics,
// whose sums do not depend on their order or on how the tile's entries fall
// into chunks, for foldTile to write the box from.
template <int SHAPE>
__device__ __forceinline__ void flushRawBox(const unsigned long long* acc, const TileBox<SHAPE>& box, int nx, int ny,
                                            int nz, const TileBoxes& T, const unsigned long long* tileScan, int tile) {
  const unsigned long long sc = tileScan[tile];
  if (chunkField(tileScan[tile + 1]) - chunkField(sc) == 1) {
    convolveRawBox<SHAPE>(reinterpret_cast<const long long*>(acc), box, nx, ny, nz,
                          T.boxes + static_cast<size_t>(occupiedField(sc)) * 3 * boxNodes<SHAPE>());
    return;
  }
  unsigned long long* const raw = reinterpret_cast<unsigned long long*>(rawBoxOf<SHAPE>(T, chunkField(sc), occupiedField(sc)));
  for (int t = threadIdx.x; t < 3 * rawNodes<SHAPE>(); t += blockDim.x) {
    const unsigned long long val = acc[t];
    if (val) atomicAdd(raw + t, val);
  }
}

// A thread takes one column of a box (429 or 363).
constexpr int kFoldThreads = 512;
// The box of a tile of several chunks (its first chunk, its occupied slot)
// from its raw box, which is cleared for the next deposit.
template <int SHAPE>
__device__ __forceinline__ void foldTile(int firstChunk, int slot, const TileBox<SHAPE>& box, int nx, int ny, int nz,
                                         const TileBoxes& T) {
  constexpr int N = 3 * rawNodes<SHAPE>(), kPer = (N + kFoldThreads - 1) / kFoldThreads;
  __shared__ long long sums[N];
  long long* const raw = rawBoxOf<SHAPE>(T, firstChunk, slot);
  long long v[kPer];  // every load ahead of the first store
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int t = static_cast<int>(threadIdx.x) + r * kFoldThreads;
    v[r] = t < N ? raw[t] : 0;
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int t = static_cast<int>(threadIdx.x) + r * kFoldThreads;
    if (t < N) {
      sums[t] = v[r];
      raw[t] = 0;
    }
  }
  __syncthreads();
  convolveRawBox<SHAPE>(sums, box, nx, ny, nz, T.boxes + static_cast<size_t>(slot) * 3 * boxNodes<SHAPE>());
}

// The value one lane below (kRowBelow) or above (kRowAbove) in a row of 16
// lanes; 0 past the row's ends.
constexpr int kRowBelow = 0x111, kRowAbove = 0x101;  // DPP row_shr:1, row_shl:1
template <int CTRL>
__device__ __forceinline__ float rowMove(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double rowMove(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// The gather side's staging: field values of the tile box with the shape's
// convolution applied, on the raw nodes a chord's raw taps read (out, 3
// components of rawNodes). GA is the form's gather arguments, R its real
// type; kChunk threads call it. Binomial3-x: a row of 16 lanes takes a (y,
// component) row of the box, each lane one x column's nine z values, summed
// in z in registers and in x from the neighbour lanes. `electric` selects
// E_cand + E_old, zero outside the components (such nodes carry no field),
// or B, with indices clamped to the component (the open sample of
// NativeHalo::openMagneticValue).
template <bool ELECTRIC, class GA, class R>
__device__ __forceinline__ void stageBinomial(const GA& G, const TileBox<kShapeBinomial3X>& box, R* out) {
#pragma clang fp contract(fast)
  using B = Box<kShapeBinomial3X>;
  using W = RawBox<kShapeBinomial3X>;
  constexpr int kRows = 3 * B::NY, kPer = (kRows * 16 + kChunk - 1) / kChunk, NR = rawNodes<kShapeBinomial3X>();
  static_assert(B::NX <= 16 && kChunk % 16 == 0, "one row of 16 lanes holds a box row");
  const int lx = static_cast<int>(threadIdx.x) & 15;
  R f[kPer][B::NZ];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int row = static_cast<int>(threadIdx.x >> 4) + r * (kChunk / 16);
    const int d = row / B::NY, ly = row - d * B::NY;
    const int (*n)[3] = ELECTRIC ? G.ne : G.nb;
    const int n0 = d == 0 ? n[0][0] : (d == 1 ? n[1][0] : n[2][0]);
    const int n1 = d == 0 ? n[0][1] : (d == 1 ? n[1][1] : n[2][1]);
    const int n2 = d == 0 ? n[0][2] : (d == 1 ? n[1][2] : n[2][2]);
    const R* src;
    if constexpr (ELECTRIC) src = d == 0 ? G.esum[0] : (d == 1 ? G.esum[1] : G.esum[2]);
    else src = d == 0 ? G.b[0] : (d == 1 ? G.b[1] : G.b[2]);
    int i = box.x0 + lx, j = box.y0 + ly;
    bool in = lx < B::NX && d < 3;
    if (ELECTRIC) {
      in = in && i >= 0 && i < n0 && j >= 0 && j < n1;
    } else {
      i = min(max(i, 0), n0 - 1);
      j = min(max(j, 0), n1 - 1);
    }
    const size_t plane = static_cast<size_t>(n0) * n1;
    const R* at = src + static_cast<size_t>(j) * n0 + i;
#pragma unroll
    for (int q = 0; q < B::NZ; ++q) {
      const int k = box.z0 + q;
      f[r][q] = R(0);
      if (ELECTRIC) {
        if (in && k >= 0 && k < n2) f[r][q] = at[k * plane];
      } else if (in) {
        f[r][q] = at[min(max(k, 0), n2 - 1) * plane];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const int row = static_cast<int>(threadIdx.x >> 4) + r * (kChunk / 16);
    const int d = row / B::NY, ly = row - d * B::NY;
    const bool mine = d < 3 && lx >= 1 && lx <= W::NX;
#pragma unroll
    for (int q = 0; q < W::NZ; ++q) {
      const R z = R(0.25) * (f[r][q] + f[r][q + 2]) + R(0.5) * f[r][q + 1];
      const R v = R(0.25) * (rowMove<kRowBelow>(z) + rowMove<kRowAbove>(z)) + R(0.5) * z;
      if (mine) out[d * NR + (q * W::NY + ly) * W::NX + lx - 1] = v;
    }
  }
}

// B nodes of a tile for the quintic's trilinear sample (source_coupling.cpp:
// 83-86; source_coupling_math.h:122-138): [-1, 9] in x and y, [-1, 5] in z
// around the tile, with the indices clamped to the components' extents.
constexpr int kBNX = kTileX + 3, kBNY = kTileY + 3, kBNZ = kTileZ + 3, kBNodes = kBNX * kBNY * kBNZ;
template <class GA, class R>
__device__ __forceinline__ void stageB(const GA& G, const TileBox<kShapeQuintic>& box, R* out) {
  auto clamp = [](int v, int n) { return v < 0 ? 0 : (v > n - 1 ? n - 1 : v); };
  const int z0 = box.z0 + Box<kShapeQuintic>::Z0 - 1;
  for (int t = threadIdx.x; t < kBNodes; t += kChunk) {
    const int lx = t % kBNX, ly = (t / kBNX) % kBNY, lz = t / (kBNX * kBNY);
#pragma unroll
    for (int axis = 0; axis < 3; ++axis) {
      const int* n = G.nb[axis];
      const int i = clamp(box.x0 + lx, n[0]), j = clamp(box.y0 + ly, n[1]), k = clamp(z0 + lz, n[2]);
      out[axis * kBNodes + t] = G.b[axis][(static_cast<size_t>(k) * n[1] + j) * n[0] + i];
    }
  }
}
// The trilinear sample at mid (cells from org's node), from memory or from
// the staged nodes: a chord's middle lies less than half a cell from the tile
// it starts in, so its nodes are staged; nodes that are not (a chord longer
// than a cell, an error of the E gather) are read from memory all the same.
// Staging replaces 24 scattered loads a lane and pays where a chunk holds
// several entries a lane: gathers 350 -> 316 us with 4e6 entries, but 19.4 ->
// 20.0 us with 1e5 (FP64 30 -> 31 us), whose chunks hold one.
template <bool STAGED, class GA, class R>
__device__ __forceinline__ void sampleQuinticB(const GA& G, const TileBox<kShapeQuintic>& box, const R* bs,
                                               const int org[3], const R mid[3], R res[3]) {
  const int o[3] = {box.x0, box.y0, box.z0 + Box<kShapeQuintic>::Z0 - 1}, extent[3] = {kBNX, kBNY, kBNZ};
  int cell[2][3];
  R fraction[2][3];
  bool staged = STAGED;
  for (int half = 0; half < 2; ++half)
    for (int d = 0; d < 3; ++d) {
      const R x = mid[d] - R(.5) * half, fl = floor(x);
      cell[half][d] = static_cast<int>(fl) + org[d];
      fraction[half][d] = x - fl;
      staged = staged && static_cast<unsigned>(cell[half][d] - o[d]) <= static_cast<unsigned>(extent[d] - 2);
    }
  auto sample = [&](auto node) {
#pragma unroll
    for (int axis = 0; axis < 3; ++axis) {
      const int hx = axis == 0 ? 0 : 1, hy = axis == 1 ? 0 : 1, hz = axis == 2 ? 0 : 1;
      R sum = R(0);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const R xw = i ? fraction[hx][0] : R(1) - fraction[hx][0];
            const R yw = j ? fraction[hy][1] : R(1) - fraction[hy][1];
            const R zw = k ? fraction[hz][2] : R(1) - fraction[hz][2];
            sum += xw * yw * zw * node(axis, cell[hx][0] + i, cell[hy][1] + j, cell[hz][2] + k);
          }
      res[axis] = sum;
    }
  };
  if (staged) {
    sample([&](int axis, int i, int j, int k) {
      return bs[axis * kBNodes + ((k - o[2]) * kBNY + (j - o[1])) * kBNX + (i - o[0])];
    });
  } else {
    auto clamp = [](int v, int n) { return v < 0 ? 0 : (v > n - 1 ? n - 1 : v); };
    sample([&](int axis, int i, int j, int k) {
      const int* n = G.nb[axis];
      return G.b[axis][(static_cast<size_t>(clamp(k, n[2])) * n[1] + clamp(j, n[1])) * n[0] + clamp(i, n[0])];
    });
  }
}

// Quintic: a lane per (x, y, component) column, its 17 z values convolved
// with the compensation in FP64 into the 11 raw planes (E_cand + E_old).
template <class GA, class R>
__device__ __forceinline__ void stageQuintic(const GA& G, const TileBox<kShapeQuintic>& box, R* out) {
#pragma clang fp contract(fast)
  using B = Box<kShapeQuintic>;
  using W = RawBox<kShapeQuintic>;
  constexpr int P = B::NX * B::NY, NR = rawNodes<kShapeQuintic>();
  for (int t = threadIdx.x; t < 3 * P; t += kChunk) {
    const int d = t / P, r = t - d * P, ly = r / B::NX, lx = r - ly * B::NX;
    const int n0 = d == 0 ? G.ne[0][0] : (d == 1 ? G.ne[1][0] : G.ne[2][0]);
    const int n1 = d == 0 ? G.ne[0][1] : (d == 1 ? G.ne[1][1] : G.ne[2][1]);
    const int n2 = d == 0 ? G.ne[0][2] : (d == 1 ? G.ne[1][2] : G.ne[2][2]);
    const R* src = d == 0 ? G.esum[0] : (d == 1 ? G.esum[1] : G.esum[2]);
    const int i = box.x0 + lx, j = box.y0 + ly;
    const bool in = i >= 0 && i < n0 && j >= 0 && j < n1;
    const size_t plane = static_cast<size_t>(n0) * n1;
    const R* at = src + static_cast<size_t>(j) * n0 + i;
    R f[B::NZ];
#pragma unroll
    for (int q = 0; q < B::NZ; ++q) {
      const int k = box.z0 + q;
      f[q] = R(0);
      if (in && k >= 0 && k < n2) f[q] = at[k * plane];
    }
#pragma unroll
    for (int q = 0; q < W::NZ; ++q) {
      double sum = 0.0;
#pragma unroll
      for (int c = 0; c < 7; ++c) sum += quinticCompensation(c) * static_cast<double>(f[q + c]);
      out[d * NR + q * P + r] = static_cast<R>(sum);
    }
  }
}

// A chunk's residual statistics in a fixed order: every thread of the
// workgroup (kChunk) enters its particle's values (zeros without one); the
// chunk's max force and defect / scale / call sums go to out[0..3]. Rows of
// 16 lanes are summed in registers, then the rows one after the other. sh
// holds kChunk / 4 doubles.
template <int CTRL>
__device__ __forceinline__ double lanePermute(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ void chunkStats(double* sh, double force, double defect, double scale, double calls,
                                           double* out) {
  auto step = [&](auto permute) {
    force = fmax(force, permute(force));
    defect += permute(defect);
    scale += permute(scale);
    calls += permute(calls);
  };
  step([](double v) { return lanePermute<0xB1>(v); });   // quad_perm [1, 0, 3, 2]
  step([](double v) { return lanePermute<0x4E>(v); });   // quad_perm [2, 3, 0, 1]
  step([](double v) { return lanePermute<0x141>(v); });  // row_half_mirror
  step([](double v) { return lanePermute<0x140>(v); });  // row_mirror
  constexpr int kRows = kChunk / 16;
  const int row = static_cast<int>(threadIdx.x >> 4);
  if ((threadIdx.x & 15u) == 0u) {
    sh[row] = force;
    sh[kRows + row] = defect;
    sh[2 * kRows + row] = scale;
    sh[3 * kRows + row] = calls;
  }
  __syncthreads();
  if (threadIdx.x < 4u) {
    const double* v = sh + threadIdx.x * kRows;
    double acc = v[0];
    for (int r = 1; r < kRows; ++r) acc = threadIdx.x == 0u ? fmax(acc, v[r]) : acc + v[r];
    out[threadIdx.x] = acc;
  }
}

// Orbit average of the staged field over the chord x + t v (0 <= t <= 1, in
// cells, inside the grid) with the deposit's weights: res[d] = sum of weight
// times raw node. A chord that leaves the tile's raw box is an error.
template <int SHAPE, class R>
__device__ __forceinline__ void gatherRaw(int nx, int ny, const R* es, const TileBox<SHAPE>& box, const int org[3],
                                          const R x[3], const R v[3], R res[3], unsigned& err) {
#pragma clang fp contract(fast)
  using W = RawBox<SHAPE>;
  constexpr int NR = rawNodes<SHAPE>();
  res[0] = res[1] = res[2] = R(0);
  R cuts[kMaxCuts];
  const int count = orbitCuts(x, v, cuts, err);
  int base = 0;
  auto corner = [&](int i, int j, int k) {
    const bool holds = box.rawHolds(i, j, k, 2, 2, SHAPE == kShapeQuintic ? 6 : 2);
    if (!holds) err |= kErrTileHalo;
    base = holds ? box.rawIndex(i, j, k) : 0;
    return true;
  };
  auto tap = [&](int d, int oi, int oj, int ok, auto w) {
    res[d] += static_cast<R>(w) * es[d * NR + base + (ok * W::NY + oj) * W::NX + oi];
  };
#pragma unroll 1
  for (int s = 1; s < count; ++s)
    if (cuts[s] - cuts[s - 1] > R(0))
      rawSegment<SHAPE, R>(nx, ny, org, x, v, cuts[s - 1], cuts[s], corner, tap, tap);
}

// binomialXZMagneticSample (source_coupling_math.h:142-167) at mid (cells
// from org's node): the trilinear sample of the staged, smoothed B.
template <class R>
__device__ __forceinline__ void sampleBinomial(const R* bs, const TileBox<kShapeBinomial3X>& box, const int org[3],
                                               const R mid[3], R res[3], unsigned& err) {
#pragma clang fp contract(fast)
  using W = RawBox<kShapeBinomial3X>;
  constexpr int NR = rawNodes<kShapeBinomial3X>();
#pragma unroll
  for (int comp = 0; comp < 3; ++comp) {
    int cell[3];
    R f[3];
    for (int d = 0; d < 3; ++d) {
      const R pos = mid[d] - (comp == d ? R(0) : R(0.5)), fl = floor(pos);
      cell[d] = static_cast<int>(fl) + org[d];
      f[d] = pos - fl;
    }
    const bool holds = box.rawHolds(cell[0], cell[1], cell[2], 2, 2, 2);
    if (!holds) err |= kErrTileHalo;
    const R* at = bs + comp * NR + (holds ? box.rawIndex(cell[0], cell[1], cell[2]) : 0);
    R plane[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const R* p = at + k * W::NX * W::NY;
      plane[k] = (R(1) - f[1]) * ((R(1) - f[0]) * p[0] + f[0] * p[1]) +
                 f[1] * ((R(1) - f[0]) * p[W::NX] + f[0] * p[W::NX + 1]);
    }
    res[comp] = (R(1) - f[2]) * plane[0] + f[2] * plane[1];
  }
}

}  // namespace aprl_gpu
