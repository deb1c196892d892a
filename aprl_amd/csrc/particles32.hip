// gfx950 particle kernels of the conservative-source step in the FP32-split
// form: fields, currents, gathered fields and momenta in FP32; positions as
// an absolute int32 lattice cell plus an FP32 in-cell offset.
//
// The step is the FP64 form's (tile sort, orbit gathers from LDS-staged
// tile boxes, Lapenta-Markidis push, fixed-point tile deposition, owner
// reduction) with these differences:
//  * chord cuts, binomial3-x weights and gathers run in FP32 on coordinates
//    taken relative to the particle's start cell, so the in-cell offset keeps
//    its 24 bits whatever the absolute position; the quintic's weights are
//    formed in FP64 from those coordinates (rawSegment);
//  * the push converts its inputs to FP64 and reuses the FP64 orbit push
//    (prescribed magnets, Newton root, boundary checks) on absolute box
//    coordinates, then stores the end point as cell + FP32 offset again;
//  * the Picard loop runs a fixed number of trials (at least the two the
//    reference requires with active particles, simulation_source_coupling.cpp:
//    50): its convergence tolerances (force < 1e-13) lie below FP32
//    resolution, and a fixed count keeps the host out of the step.

#include <algorithm>
#include <cmath>
#include <limits>

#include "diagnostics.hpp"
#include "particle_device.hpp"
#include "shapes.hpp"

namespace aprl_gpu {

// ---------------------------------------------------------------------------
// Kernel argument blocks.

struct GArgs32 {
  float* esum[3];         // E_cand + E_old of the trial
  const float* esum0[3];  // E* + E_old, E* the zero-current preview
  const float* b[3];      // B^(n+1/2)
  int ne[3][3], nb[3][3];
  int nx, ny, nz;
  int oc[3];       // absolute lattice cell of the grid origin
  float ch[3];     // c dt / h per axis (ballistic guess, cells per unit u/gamma)
  float negS;      // (-1*dt)/eps0
};

struct PArgs32 {
  const int* cell[3];
  const float* off[3];
  const float* u[3];
  const float* q;
  const float* m;
  float* fin[6];
  float* fout[6];
  int* cell1[3];
  float* off1[3];
  float* chord[3];  // trial chord x1 - x0 in cells, rounded once from FP64
  float* u1[3];
  float* gridAbs;
  const int* state;  // entry states (kStateActive / kStateCarrier for live entries)
  int* evt;          // boundary event code of the trial
  float* cut[3];     // t1, t2, carrier-part deposit weight
  float* wend;       // carrier end weight
  const float* w;    // weight slot (a carrier's current weight)
  const float* beta; // held speed of held entries
  const unsigned long long* tileBound;  // per tile: largest entry current bound
  float kq[3];  // h_a / (dx dy dz dt): current density per unit charge and cell of motion
  double h[3];
  int n;
};

// ---------------------------------------------------------------------------
// Chord of one particle relative to its start cell.

struct Chord32 {
  int org[3];        // grid index of the start cell
  float x[3], v[3];  // start offset and displacement, in cells
};

__device__ __forceinline__ Chord32 chordOf(const GArgs32& G, int c0x, int c0y, int c0z, const float off0[3],
                                           const float v[3]) {
  Chord32 r;
  r.org[0] = c0x - G.oc[0];
  r.org[1] = c0y - G.oc[1];
  r.org[2] = c0z - G.oc[2];
  for (int a = 0; a < 3; ++a) {
    r.x[a] = off0[a];
    r.v[a] = v[a];
  }
  return r;
}

// clipOpenOrbit (source_coupling_math.h:235-250) in start-cell coordinates:
// the grid spans [-org, n - org) per axis. On success the chord is replaced
// by its clipped part and the kept fraction is returned in kept.
__device__ bool clipChord(const GArgs32& G, Chord32& c, float& kept, unsigned& err) {
  float first = 0.f, last = 1.f;
  const int size[3] = {G.nx, G.ny, G.nz};
  // a chord that lies in the grid needs none of the divisions
  bool inside = true;
  for (int a = 0; a < 3; ++a) {
    const float lo = static_cast<float>(-c.org[a]), hi = static_cast<float>(size[a] - c.org[a]), e = c.x[a] + c.v[a];
    inside = inside && c.x[a] >= lo && c.x[a] <= hi && e >= lo && e <= hi;
  }
  kept = 1.f;
  if (inside) return true;
  bool valid = true;
  for (int a = 0; a < 3; ++a) {
    const float x = c.x[a], d = c.v[a];
    if (!isfinite(x) || !isfinite(d)) { err |= kErrNonfinite; return false; }
    const float lo = static_cast<float>(-c.org[a]) - x, hi = static_cast<float>(size[a] - c.org[a]) - x;
    if (d == 0.f) {
      if (lo > 0.f || hi < 0.f) valid = false;
      continue;
    }
    const float tlo = lo / d, thi = hi / d;
    if (d > 0.f) { first = fmaxf(first, tlo); last = fminf(last, thi); }
    else { last = fminf(last, tlo); first = fmaxf(first, thi); }
  }
  if (!valid || !(last >= first)) return false;
  for (int a = 0; a < 3; ++a) {
    const float d = c.v[a];
    if (first != 0.f) c.x[a] += first * d;
    c.v[a] = (last - first) * d;
  }
  kept = last - first;
  return true;
}

// ---------------------------------------------------------------------------
// Sort.

__device__ __forceinline__ int clampIndex32(int v, int n) { return v < 0 ? 0 : (v > n - 1 ? n - 1 : v); }

__global__ void kTileKeys32(const int* cx, const int* cy, const int* cz, const float* oz, int* state, int n,
                            GArgs32 G, int ntx, int nty, unsigned* key, TileRangeArgs R, SortArgs K, DigitCounts D,
                            double hz) {
  __shared__ unsigned blockActive;
  __shared__ unsigned digits[256];
  if (threadIdx.x == 0) blockActive = 0u;
  __syncthreads();
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  clearTileRanges(R, p);
  if (p == 0) *K.removed = 0u;
  bool active = false;
  unsigned tile = 0u;
  if (p < n) {
    const double z = (static_cast<double>(cz[p]) + static_cast<double>(oz[p])) * hz;
    if (!liveEntry(K, state, p, z)) {
      tile = static_cast<unsigned>(R.ntiles);
    } else {
      const int x = clampIndex32(cx[p] - G.oc[0], G.nx);
      const int y = clampIndex32(cy[p] - G.oc[1], G.ny);
      const int zc = clampIndex32(cz[p] - G.oc[2], G.nz);
      tile = (static_cast<unsigned>(zc / kTileZ) * nty + y / kTileY) * ntx + x / kTileX;
      active = state[p] == kStateActive;
    }
    key[p] = tile;
  }
  countFirstDigit(D, digits, p < n, tile);
  // live active entries of the workgroup, summed by kTileCounts
  const unsigned long long act = __ballot(active);
  if (act && static_cast<int>(__lane_id()) == __ffsll(static_cast<long long>(act)) - 1)
    atomicAdd(&blockActive, static_cast<unsigned>(__popcll(act)));
  __syncthreads();
  if (threadIdx.x == 0) K.blockActive[blockIdx.x] = blockActive;
}

struct PermuteArgs32 {
  const int* cellSrc[3];
  int* cellDst[3];
  const float* src[9];
  float* dst[9];
  const uint64_t* idSrc;
  uint64_t* idDst;
  const int* stateSrc;
  int* stateDst;
  const float* betaSrc;
  float* betaDst;
};

// State scatter into sorted order, and the tile ranges of the sorted keys.
// blockIdx.y splits the gathered arrays over four times as many waves
// (y = 0: cells and offsets, tile ranges and bounds; 1: momenta; 2: q, m,
// w; 3: ids, states, held speeds).
__global__ void kPermute32(PermuteArgs32 A, const unsigned* perm, int n, TileBoundsArgs T) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  const int part = static_cast<int>(blockIdx.y);
  unsigned tile = ~0u;
  double bound = 0.0;
  if (p < n) {
    const unsigned from = perm[p];
    if (part < 3) {
#pragma unroll
      for (int a = 0; a < 3; ++a) A.dst[3 * part + a][p] = A.src[3 * part + a][from];
    } else {
      A.idDst[p] = A.idSrc[from];
      A.stateDst[p] = A.stateSrc[from];
      A.betaDst[p] = A.betaSrc[from];
    }
    if (part == 0) {
#pragma unroll
      for (int a = 0; a < 3; ++a) A.cellDst[a][p] = A.cellSrc[a][from];
      tileBoundsAt(T, p);
      const unsigned k = T.key[p];
      if (k < static_cast<unsigned>(T.ntiles)) {
        tile = k;
        bound = entryCurrentBound(static_cast<double>(A.src[6][from]), A.stateSrc[from], T.perCharge);
      }
    }
  }
  if (part == 0) raiseTileBound(T.bound, tile, bound);
}

// ---------------------------------------------------------------------------
// Gathers, push, deposit, reduction.

__device__ __forceinline__ void chordAt(const PArgs32& P, int p, bool guess, const GArgs32& G, int c0[3],
                                        float off0[3], float v[3]) {
  for (int d = 0; d < 3; ++d) {
    c0[d] = P.cell[d][p];
    off0[d] = P.off[d][p];
  }
  if (guess) {
    // ballistic end point x0 + c dt u0 / gamma0 (source_coupling.cpp:133-147)
    const float ux = P.u[0][p], uy = P.u[1][p], uz = P.u[2][p];
    const float ig = rsqrtf(1.f + ux * ux + uy * uy + uz * uz);
    v[0] = G.ch[0] * ux * ig;
    v[1] = G.ch[1] * uy * ig;
    v[2] = G.ch[2] * uz * ig;
  } else {
    // the push's displacement rounded once: keeps its relative precision
    // where x1 - x0 is far below the offsets' resolution (transverse motion)
    for (int d = 0; d < 3; ++d) v[d] = P.chord[d][p];
  }
}

// Chunked orbit gathers, one lane per particle, as the FP64 form's: MODE 0 at
// (x0, ballistic guess) against the zero-current preview into fin; MODE 1 the
// residual gather at (x0, x1) into fout, with the chunk's force max and
// defect / scale / call sums when chunkOut is given.
template <int MODE, int SHAPE, bool LOOP>
__global__ void __launch_bounds__(kChunk) kGatherChunks32(PArgs32 P, GArgs32 G, StepArgs S, const int4* chunks,
                                                          int ntx, int nty, double dt, double* chunkOut,
                                                          unsigned* errOut) {
  constexpr int N = 3 * rawNodes<SHAPE>();
  __shared__ float es[N];
  __shared__ float bs[SHAPE == kShapeBinomial3X ? N : (LOOP ? 3 * kBNodes : 1)];
  __shared__ double stats[MODE == 1 ? kChunk / 4 : 1];
  const int cb = xcdContiguous(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
  const int4 ch = chunks[cb];
  const TileBox<SHAPE> box = tileBox<SHAPE>(ch.x, ntx, nty);
  // this lane's first particle is loaded ahead of the staging (lanes past the
  // chunk's end read its first entry and ignore it)
  int p, stored, c0[3];
  float off0[3], v[3];
  auto load = [&](int first) {
    p = first + static_cast<int>(threadIdx.x);
    const int pv = p < ch.z ? p : ch.y;
    stored = P.state[pv];
    chordAt(P, pv, MODE == 0, G, c0, off0, v);
  };
  load(ch.y);
  if constexpr (SHAPE == kShapeBinomial3X) {
    stageBinomial<true>(G, box, es);
    stageBinomial<false>(G, box, bs);
  } else {
    stageQuintic(G, box, es);
    if constexpr (LOOP) stageB(G, box, bs);
  }
  __syncthreads();
  unsigned err = 0;
  double force = 0., defect = 0., scale = 0., calls = 0.;
  auto particle = [&]() {
    // carriers move without fields and take no part in the residual; a held
    // entry takes part from its release point with the rest of the step
    const int st = p < ch.z ? stored : kStateRemoved;
    bool live = st == kStateActive;
    double dtp = dt;
    if (st == kStateHeld) {
      double x0[3], uh[3];
      for (int d = 0; d < 3; ++d) {
        x0[d] = (static_cast<double>(c0[d]) + static_cast<double>(off0[d])) * P.h[d];
        uh[d] = P.u[d][p];
      }
      const HeldMove h = heldMove(S, x0, uh, static_cast<double>(P.beta[p]));
      if (h.release && h.remaining > 0.0) {
        live = true;
        dtp = h.remaining;
        for (int d = 0; d < 3; ++d) {
          // held leg to the release point, in cells; the rest of the chord
          const float dk = static_cast<float>((h.x1[d] - x0[d]) / P.h[d]);
          off0[d] += dk;
          if (MODE == 0) v[d] *= static_cast<float>(dtp / dt);
          else v[d] -= dk;
        }
      }
    }
    if (live) {
      float g[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, mid[3], kept;
      Chord32 c = chordOf(G, c0[0], c0[1], c0[2], off0, v);
      if (clipChord(G, c, kept, err)) {
        gatherRaw<SHAPE, float>(G.nx, G.ny, es, box, c.org, c.x, c.v, g, err);
        for (int d = 0; d < 3; ++d) {
          g[d] *= 0.5f * kept;
          mid[d] = c.x[d] + 0.5f * c.v[d];
        }
        if constexpr (SHAPE == kShapeBinomial3X) sampleBinomial(bs, box, c.org, mid, g + 3, err);
        else sampleQuinticB<LOOP>(G, box, bs, c.org, mid, g + 3);
      } else {
        err |= kErrOrbitOutside | (SHAPE == kShapeBinomial3X ? kErrMagneticOutside : kErrMagneticNoDomain);
      }
      float* const* dst = MODE == 0 ? P.fin : P.fout;
      for (int d = 0; d < 6; ++d) dst[d][p] = g[d];
      if (MODE == 1 && chunkOut) {
        // localResidual (source_coupling.cpp:105-159)
        double de[3], db[3];
        for (int d = 0; d < 3; ++d) {
          de[d] = static_cast<double>(g[d]) - P.fin[d][p];
          db[d] = static_cast<double>(g[3 + d]) - P.fin[3 + d][p];
        }
        const double q = P.q[p], m = P.m[p];
        force = fmax(force, fabs(q / m) * dtp / kC *
                                (sqrt(de[0] * de[0] + de[1] * de[1] + de[2] * de[2]) +
                                 kC * sqrt(db[0] * db[0] + db[1] * db[1] + db[2] * db[2])));
        double w1 = 0., w2 = 0.;
        for (int d = 0; d < 3; ++d) {
          const double dx = static_cast<double>(v[d]) * P.h[d];
          w1 += q * de[d] * dx;
          w2 += q * g[d] * dx;
        }
        defect += fabs(w1);
        scale += static_cast<double>(P.gridAbs[p]) + fabs(w2);
        calls += 1.;
      }
    }
  };
  if constexpr (LOOP) {
#pragma unroll 1
    for (int first = ch.y; first < ch.z; first += kChunk) {
      if (first != ch.y) load(first);
      particle();
    }
  } else {
    particle();
  }
  if (MODE == 1 && chunkOut) chunkStats(stats, force, defect, scale, calls, chunkOut + 4 * cb);
  if (err) atomicOr(errOut, err);
}

// One entry of kPushSplit.
__device__ __forceinline__ void pushSplitEntry(const PArgs32& P, const StepArgs& S, double o0, double o1, double o2,
                                               int p, unsigned* errOut) {
  unsigned err = 0;
  const double o[3] = {o0, o1, o2};
  int c0[3];
  double x0[3], u0[3];
  for (int a = 0; a < 3; ++a) {
    c0[a] = P.cell[a][p];
    x0[a] = (static_cast<double>(c0[a]) + static_cast<double>(P.off[a][p])) * P.h[a];
    u0[a] = P.u[a][p];
  }
  double x[3], u[3], absGrid, t1, t2, wDeposit, wEnd, usedE[3], usedB[3];
  for (int a = 0; a < 3; ++a) {
    usedE[a] = P.fin[a][p];
    usedB[a] = P.fin[3 + a][p];
  }
  const int code = entryStep(S, o, P.state[p], x0, u0, P.q[p], P.m[p], static_cast<double>(P.w[p]),
                             static_cast<double>(P.beta[p]), usedE, usedB, x, u, absGrid, t1, t2, wDeposit, wEnd,
                             err);
  for (int a = 0; a < 3; ++a) {
    const double rel = static_cast<double>(P.off[a][p]) + (x[a] - x0[a]) / P.h[a];
    double fl = floor(rel);
    float off = static_cast<float>(rel - fl);
    if (off >= 1.f) {  // rel - fl rounded up to 1
      off = 0.f;
      fl += 1.;
    }
    int cell = c0[a];
    if (isfinite(fl) && fabs(fl) < 1e9) cell += static_cast<int>(fl);
    else err |= kErrNonfinite;
    P.cell1[a][p] = cell;
    P.off1[a][p] = off;
    P.chord[a][p] = static_cast<float>((x[a] - x0[a]) / P.h[a]);
    P.u1[a][p] = static_cast<float>(u[a]);
  }
  P.gridAbs[p] = static_cast<float>(absGrid);
  P.evt[p] = code;
  if (code) {
    P.cut[0][p] = static_cast<float>(t1);
    P.cut[1][p] = static_cast<float>(t2);
    P.cut[2][p] = static_cast<float>(wDeposit);
    P.wend[p] = static_cast<float>(wEnd);
    err |= kEvtAny;
  }
  if (err) atomicOr(errOut, err);
}

// One trial's push: FP32 state and fields widened to FP64, the FP64 orbit
// push on absolute box coordinates (origin o = the grid origin cell times
// h) or a carrier's straight move (position += dt u c / gamma), the
// segment's boundary events, and the end point split again into cell +
// FP32 offset.
__global__ void __launch_bounds__(128) kPushSplit(PArgs32 P, StepArgs S, double o0, double o1, double o2,
                                                  unsigned* errOut) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < P.n) pushSplitEntry(P, S, o0, o1, o2, p, errOut);
}

// Deterministic tile deposition (Current::deposit, longitudinal_shape.h:
// 175-187) of the FP32 chords into 64-bit fixed-point LDS tile boxes; the
// scheme is the FP64 form's: one exponent per tile from the tile's current
// bound, integer sums independent of order.
template <int SHAPE, bool LOOP>
__global__ void __launch_bounds__(kChunk) __attribute__((amdgpu_waves_per_eu(SHAPE == kShapeQuintic ? 2 : 3)))
kDepositSplit(PArgs32 P, GArgs32 G, StepArgs S, const int4* chunks, const int* tileBegin, const int* tileEnd,
              const unsigned long long* tileScan, int ntx, int nty, TileBoxes T, int* tileShift,
              unsigned* errOut) {
  using W = RawBox<SHAPE>;
  constexpr int N = rawNodes<SHAPE>();
  __shared__ unsigned long long acc[3 * N];
  const int4 ch = chunks[blockIdx.x];
  const int tile = ch.x;
  const TileBox<SHAPE> box = tileBox<SHAPE>(tile, ntx, nty);
  for (int t = threadIdx.x; t < 3 * N; t += blockDim.x) acc[t] = 0ull;
  // scale_a = q * dx_a / (dx dy dz dt), eb_deposition.cpp:41-51
  auto scaleOf = [&](int p, const float v[3], float s[3]) {
    const float q = P.q[p];
    for (int d = 0; d < 3; ++d) s[d] = q * P.kq[d] * v[d];
  };
  const unsigned long long tsc = tileScan[tile];
  const int shift = tileFixedShift(Box<SHAPE>::kWeightBound, P.tileBound[tile], tileEnd[tile] - tileBegin[tile]);
  if (threadIdx.x == 0 && static_cast<int>(blockIdx.x) == chunkField(tsc)) tileShift[tile] = shift;
  __syncthreads();
  unsigned err = 0;
  auto particle = [&](int p) {
    int c0[3];
    float off0[3], v[3], scale[3], part3[3];  // scales of the leg, and of the chord part (with its weight)
    chordAt(P, p, false, G, c0, off0, v);
    // A held entry released inside the step deposits its held leg to the
    // release point first, then the rest of the chord.
    float dk[3] = {0.f, 0.f, 0.f};
    int legs = 1;
    if (P.state[p] == kStateHeld) {
      double x0[3], uh[3];
      for (int d = 0; d < 3; ++d) {
        x0[d] = (static_cast<double>(c0[d]) + static_cast<double>(off0[d])) * P.h[d];
        uh[d] = P.u[d][p];
      }
      const HeldMove h = heldMove(S, x0, uh, static_cast<double>(P.beta[p]));
      if (h.release && h.kink) {
        legs = 2;
        for (int d = 0; d < 3; ++d) dk[d] = static_cast<float>((h.x1[d] - x0[d]) / P.h[d]);
      }
    }
    Chord32 c = chordOf(G, c0[0], c0[1], c0[2], off0, v);
    float cuts[kMaxCuts];
    int base = 0;
    unsigned mask[3] = {0, 0, 0};
    double fixed[3];  // part3 in the tile's fixed-point units
    auto corner = [&](int i, int j, int k) {
      base = box.rawIndex(i, j, k);
      const bool inside = rawDepositInside<SHAPE>(box, G.nx, G.ny, i, j, k);
#pragma unroll
      for (int d = 0; d < 3; ++d) fixed[d] = ldexp(static_cast<double>(part3[d]), shift);
      if (__all(inside)) return true;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        mask[d] = part3[d] == 0.f ? 0u : ~0u;
        if (mask[d] && !inside) mask[d] = rawDepositMask<SHAPE>(box, G.ne[d], d, i, j, k, err);
      }
      return false;
    };
    auto tapInside = [&](int d, int oi, int oj, int ok, auto w) {
      atomicAdd(&acc[d * N + base + (ok * W::NY + oj) * W::NX + oi], fixedPoint(fixed[d], static_cast<double>(w)));
    };
    auto tap = [&](int d, int oi, int oj, int ok, auto w) {
      if (mask[d] & tapBit(oi, oj, ok)) tapInside(d, oi, oj, ok, w);
    };
    // A boundary event splits the last leg: [0, t1] at unit weight (the
    // active part) and [t1, t2] at the carrier part's deposit weight.
    const int e = P.evt[p];
    const float t1 = e ? P.cut[0][p] : 1.f, t2 = e ? P.cut[1][p] : 1.f, wCarrier = e ? P.cut[2][p] : 0.f;
#pragma unroll 1
    for (int leg = 0; leg < legs; ++leg) {
      const bool last = leg + 1 == legs;
      if (legs == 2) {
        // leg 0: dk from the start; leg 1: the rest from the kink
        for (int d = 0; d < 3; ++d) {
          c.x[d] = off0[d] + (leg ? dk[d] : 0.f);
          c.v[d] = leg ? v[d] - dk[d] : dk[d];
        }
      }
      scaleOf(p, c.v, scale);
      const int count = orbitCuts(c.x, c.v, cuts, err);
      const float f1 = last ? t1 : 1.f, f2 = last ? t2 : 1.f, fw = last ? wCarrier : 0.f;
      for (int sgm = 1; sgm < count; ++sgm) {
        const float k0 = cuts[sgm - 1], k1 = cuts[sgm];
        if (k1 - k0 <= 0.f) continue;
        // without an event: one part [k0, k1] (t1 = t2 = 1)
#pragma unroll 1
        for (int part = 0; part < 2; ++part) {
          const float a = part ? fmaxf(k0, f1) : k0;
          const float b = part ? fminf(k1, f2) : fminf(k1, f1);
          if (!(b > a)) continue;
          for (int d = 0; d < 3; ++d) part3[d] = part ? scale[d] * fw : scale[d];
          rawSegment<SHAPE, float>(G.nx, G.ny, c.org, c.x, c.v, a, b, corner, tapInside, tap);
        }
      }
    }
  };
  const int p0 = ch.y + static_cast<int>(threadIdx.x);
  if constexpr (LOOP) {
#pragma unroll 1
    for (int p = p0; p < ch.z; p += kChunk) particle(p);
  } else {
    if (p0 < ch.z) particle(p0);
  }
  __syncthreads();
  flushRawBox<SHAPE>(acc, box, G.nx, G.ny, G.nz, T, tileScan, tile);
  if (err) atomicOr(errOut, err);
}

// Node-owner reduction of the tile boxes (sums in FP64): with J the FP32
// current, rounded once (only the last trial's is read), with ESUM the
// trial's E_cand + E_old (applyCurrentSource(-1) on the preview,
// source_coupling.cpp:84-89) for the next residual gather, from the
// zero-current sums.
template <int SHAPE, bool J, bool ESUM>
__global__ void __launch_bounds__(256) kReduceCurrentSplit(float* jx, float* jy, float* jz, GArgs32 G,
                                                           const int* active, const unsigned long long* tileScan,
                                                           const int* tileShift, const long long* boxes, int ntx,
                                                           int nty, int ntz) {
  const int tile = active[xcdContiguous(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x))];
  reduceOwnedTile<SHAPE>(
      G.ne, tile, tileScan, tileShift, boxes, ntx, nty, ntz,
      [&](int i, int j, int k, const bool has[3], const double sum[3]) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if (!has[d]) continue;
          const size_t idx = (static_cast<size_t>(k) * G.ne[d][1] + j) * G.ne[d][0] + i;
          const float jv = static_cast<float>(sum[d]);
          if (J) (d == 0 ? jx : (d == 1 ? jy : jz))[idx] = jv;
          if (ESUM) {
            const bool applied = d == 0 ? (j > 0 && j < G.ny && k != 0 && k != G.nz)
                                        : (d == 1 ? (i > 0 && i < G.nx && k != 0 && k != G.nz)
                                                  : (i > 0 && i < G.nx && j > 0 && j < G.ny));
            const float e = G.esum0[d][idx];
            G.esum[d][idx] = applied ? e + G.negS * jv : e;
          }
        }
      });
}

// ---------------------------------------------------------------------------
// Host side.

void reserveSplitParticles(SplitStore& P, std::size_t capacity) {
  if (capacity <= P.capacity) return;
  for (int a = 0; a < 3; ++a) {
    P.cell[a].resize(capacity);
    P.cellT[a].resize(capacity);
    P.endCell[a].resize(capacity);
    P.chord[a].resize(capacity);
  }
  for (int a = 0; a < 9; ++a) {
    P.s[a].resize(capacity);
    P.t[a].resize(capacity);
  }
  P.id.resize(capacity);
  P.idT.resize(capacity);
  P.state.resize(capacity);
  P.stateT.resize(capacity);
  P.beta.resize(capacity);
  P.betaT.resize(capacity);
  P.evt.resize(capacity);
  for (int a = 0; a < 3; ++a) P.cut[a].resize(capacity);
  P.wend.resize(capacity);
  if (!P.removed.size()) P.removed.resize(1);
  for (int a = 0; a < 6; ++a) {
    P.fields[0][a].resize(capacity);
    P.fields[1][a].resize(capacity);
    P.end[a].resize(capacity);
  }
  P.gridAbs.resize(capacity);
  P.key.resize(capacity);
  P.keySorted.resize(capacity);
  P.permSorted.resize(capacity);
  P.capacity = capacity;
  P.sortTempBytes = 0;
  reserveSortTemp(P.sortTemp, P.sortTempBytes, capacity);
}

namespace {
// Split absolute coordinate x (metres) on the lattice of spacing h.
inline void splitCoordinate(double x, double h, int& cell, float& off) {
  const double r = x / h;
  if (!std::isfinite(r) || std::fabs(r) >= 2.0e9)
    throw std::out_of_range("Particle position is outside the FP32-split lattice range");
  double fl = std::floor(r);
  float f = static_cast<float>(r - fl);
  if (f >= 1.0f) {
    f = 0.0f;
    fl += 1.0;
  }
  cell = static_cast<int>(fl);
  off = f;
}
}  // namespace

void uploadSplitParticles(SplitStore& P, const FieldState32& F, std::size_t n, const double* x3, const double* u3,
                          const double* q, const double* m, const double* w, const uint64_t* id) {
  reserveSplitParticles(P, n);
  const double h[3] = {F.g.dx, F.g.dy, F.g.dz};
  std::vector<int> cells(n);
  std::vector<float> col(n);
  for (int a = 0; a < 3; ++a) {
    for (std::size_t i = 0; i < n; ++i) splitCoordinate(x3[3 * i + a], h[a], cells[i], col[i]);
    hipCheck(hipMemcpy(P.cell[a].get(), cells.data(), n * sizeof(int), hipMemcpyHostToDevice), "hipMemcpy");
    hipCheck(hipMemcpy(P.s[a].get(), col.data(), n * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
    for (std::size_t i = 0; i < n; ++i) col[i] = static_cast<float>(u3[3 * i + a]);
    hipCheck(hipMemcpy(P.s[3 + a].get(), col.data(), n * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
  }
  const double* scalars[3] = {q, m, w};
  for (int a = 0; a < 3; ++a) {
    for (std::size_t i = 0; i < n; ++i) col[i] = static_cast<float>(scalars[a][i]);
    hipCheck(hipMemcpy(P.s[6 + a].get(), col.data(), n * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
  }
  hipCheck(hipMemcpy(P.id.get(), id, n * sizeof(uint64_t), hipMemcpyHostToDevice), "hipMemcpy");
  P.count = n;
  ++P.generation;
}

// Grows the store keeping the persistent state of its first `count`
// entries (cells, offsets, momenta, charges, ids, entry states, held
// speeds); the per-step arrays are rewritten by every step.
void growSplitParticles(SplitStore& P, std::size_t capacity) {
  if (capacity <= P.capacity) return;
  DeviceArray<int> cell[3], state;
  DeviceArray<float> s[9], beta;
  DeviceArray<uint64_t> id;
  for (int a = 0; a < 3; ++a) cell[a].swap(P.cell[a]);
  for (int a = 0; a < 9; ++a) s[a].swap(P.s[a]);
  id.swap(P.id);
  state.swap(P.state);
  beta.swap(P.beta);
  reserveSplitParticles(P, capacity);
  const std::size_t n = P.count;
  if (!n) return;
  for (int a = 0; a < 3; ++a)
    hipCheck(hipMemcpy(P.cell[a].get(), cell[a].get(), n * sizeof(int), hipMemcpyDeviceToDevice), "hipMemcpy");
  for (int a = 0; a < 9; ++a)
    hipCheck(hipMemcpy(P.s[a].get(), s[a].get(), n * sizeof(float), hipMemcpyDeviceToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.id.get(), id.get(), n * sizeof(uint64_t), hipMemcpyDeviceToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.state.get(), state.get(), n * sizeof(int), hipMemcpyDeviceToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.beta.get(), beta.get(), n * sizeof(float), hipMemcpyDeviceToDevice), "hipMemcpy");
}

void appendSplitParticles(SplitStore& P, const FieldState32& F, std::size_t k, const double* x3, const double* u3,
                          const double* q, const double* m, const double* w, const uint64_t* id, const int* state,
                          const double* beta) {
  if (!k) return;
  const std::size_t n = P.count;
  const double h[3] = {F.g.dx, F.g.dy, F.g.dz};
  std::vector<float> col(k);
  // convert before growing, so that a rejected position leaves the store as it was
  std::vector<int> allCells(3 * k);
  std::vector<float> offsets(3 * k);
  for (int a = 0; a < 3; ++a)
    for (std::size_t i = 0; i < k; ++i) splitCoordinate(x3[3 * i + a], h[a], allCells[a * k + i], offsets[a * k + i]);
  if (n + k > P.capacity) growSplitParticles(P, std::max(n + k, P.capacity + P.capacity / 4 + 1024));
  for (int a = 0; a < 3; ++a) {
    hipCheck(hipMemcpy(P.cell[a].get() + n, allCells.data() + a * k, k * sizeof(int), hipMemcpyHostToDevice),
             "hipMemcpy");
    hipCheck(hipMemcpy(P.s[a].get() + n, offsets.data() + a * k, k * sizeof(float), hipMemcpyHostToDevice),
             "hipMemcpy");
    for (std::size_t i = 0; i < k; ++i) col[i] = static_cast<float>(u3[3 * i + a]);
    hipCheck(hipMemcpy(P.s[3 + a].get() + n, col.data(), k * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
  }
  const double* scalars[4] = {q, m, w, beta};
  DeviceArray<float>* dst[4] = {&P.s[6], &P.s[7], &P.s[8], &P.beta};
  for (int a = 0; a < 4; ++a) {
    for (std::size_t i = 0; i < k; ++i) col[i] = static_cast<float>(scalars[a][i]);
    hipCheck(hipMemcpy(dst[a]->get() + n, col.data(), k * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
  }
  hipCheck(hipMemcpy(P.id.get() + n, id, k * sizeof(uint64_t), hipMemcpyHostToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.state.get() + n, state, k * sizeof(int), hipMemcpyHostToDevice), "hipMemcpy");
  P.count = n + k;
  ++P.generation;
}

void downloadSplitParticles(const SplitStore& P, const FieldState32& F, double* x3, double* u3, double* q, double* m,
                            double* w, uint64_t* id) {
  hipCheck(hipStreamSynchronize(F.stream), "hipStreamSynchronize");
  const std::size_t n = P.count;
  const double h[3] = {F.g.dx, F.g.dy, F.g.dz};
  std::vector<int> cells(n);
  std::vector<float> col(n);
  for (int a = 0; a < 3; ++a) {
    if (x3) {
      hipCheck(hipMemcpy(cells.data(), P.cell[a].get(), n * sizeof(int), hipMemcpyDeviceToHost), "hipMemcpy");
      hipCheck(hipMemcpy(col.data(), P.s[a].get(), n * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
      for (std::size_t i = 0; i < n; ++i)
        x3[3 * i + a] = (static_cast<double>(cells[i]) + static_cast<double>(col[i])) * h[a];
    }
    if (u3) {
      hipCheck(hipMemcpy(col.data(), P.s[3 + a].get(), n * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
      for (std::size_t i = 0; i < n; ++i) u3[3 * i + a] = col[i];
    }
  }
  double* scalars[3] = {q, m, w};
  for (int a = 0; a < 3; ++a)
    if (scalars[a]) {
      hipCheck(hipMemcpy(col.data(), P.s[6 + a].get(), n * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
      for (std::size_t i = 0; i < n; ++i) scalars[a][i] = col[i];
    }
  if (id) hipCheck(hipMemcpy(id, P.id.get(), n * sizeof(uint64_t), hipMemcpyDeviceToHost), "hipMemcpy");
}

namespace {

GArgs32 gatherArgs32(CouplingState& C, const FieldState32& F, const int oc[3]) {
  GArgs32 G{};
  for (int a = 0; a < 3; ++a) {
    G.esum[a] = C.esum32[a].get();
    G.esum0[a] = C.esum032[a].get();
    G.b[a] = F.base(3 + a);
    for (int d = 0; d < 3; ++d) {
      G.ne[a][d] = static_cast<int>(F.dims[a][d]);
      G.nb[a][d] = static_cast<int>(F.dims[3 + a][d]);
    }
    G.oc[a] = oc[a];
  }
  G.nx = static_cast<int>(F.g.nx);
  G.ny = static_cast<int>(F.g.ny);
  G.nz = static_cast<int>(F.g.nz);
  G.ch[0] = static_cast<float>(F.g.dt * kC / F.g.dx);
  G.ch[1] = static_cast<float>(F.g.dt * kC / F.g.dy);
  G.ch[2] = static_cast<float>(F.g.dt * kC / F.g.dz);
  G.negS = static_cast<float>(-1.0 * F.g.dt / kEps0);
  return G;
}

PArgs32 particleArgs32(SplitStore& P, const FieldState32& F) {
  PArgs32 A{};
  for (int a = 0; a < 3; ++a) {
    A.cell[a] = P.cell[a].get();
    A.off[a] = P.s[a].get();
    A.u[a] = P.s[3 + a].get();
    A.cell1[a] = P.endCell[a].get();
    A.off1[a] = P.end[a].get();
    A.chord[a] = P.chord[a].get();
    A.u1[a] = P.end[3 + a].get();
  }
  for (int a = 0; a < 6; ++a) {
    A.fin[a] = P.fields[0][a].get();
    A.fout[a] = P.fields[1][a].get();
  }
  A.q = P.s[6].get();
  A.m = P.s[7].get();
  A.w = P.s[8].get();
  A.beta = P.beta.get();
  A.gridAbs = P.gridAbs.get();
  A.state = P.state.get();
  A.evt = P.evt.get();
  for (int a = 0; a < 3; ++a) A.cut[a] = P.cut[a].get();
  A.wend = P.wend.get();
  const double h[3] = {F.g.dx, F.g.dy, F.g.dz};
  const double den = F.g.dx * F.g.dy * F.g.dz * F.g.dt;
  for (int a = 0; a < 3; ++a) {
    A.h[a] = h[a];
    A.kq[a] = static_cast<float>(h[a] / den);
  }
  A.n = static_cast<int>(P.count);
  return A;
}

// Entries per chunk: kChunk, and up to 8 times as many from 2^19 entries on,
// where a chunk's fixed cost (staging its tile's fields; clearing its tile's
// current and writing it out, for the quintic up to 3993 atomics unless the
// tile has one chunk) is then paid for several entries a lane. At least 1024
// full chunks remain, four for each CU.
// At 4e6 entries in 128x128x960 (quintic): deposit 658 -> 536 us (527 us with
// raw sums added), gathers 331 -> 316 us (with B staged, sampleQuinticB); at
// 6e5 in 64x64x512 565 -> 533 us a binomial3-x step, 733 -> 704 us a quintic
// one. The FP64 kernels keep one entry per lane: their loop takes 54 more
// registers and at 1e6 entries the step was 1% slower with it.
int chunkSize32(int n) {
  int size = kChunk;
  for (int m = n >> 18; m > 1 && size < 8 * kChunk; m >>= 1) size *= 2;
  return size;
}

void sortSplit(CouplingState& C, SplitStore& P, const GArgs32& G, const SortArgs& K, int ntx, int nty, int ntiles,
               const DigitCounts& D, unsigned seq, hipStream_t st) {
  FieldState32& F = *C.fields32;
  const int n = static_cast<int>(P.count);
  ScopedKernel sk(F.profiler, st, "sort");
  const unsigned blocks = ceilDiv(n, 256);
  kTileKeys32<<<blocks, 256, 0, st>>>(P.cell[0].get(), P.cell[1].get(), P.cell[2].get(), P.s[2].get(),
                                      P.state.get(), n, G, ntx, nty, P.key.get(),
                                      TileRangeArgs{C.tileBegin.get(), C.tileEnd.get(), ntiles, C.tileBound.get()}, K,
                                      D, F.g.dz);
  launchCheck("tile keys");
  tileSort(P.sortTemp.get(), P.sortTempBytes, P.key.get(), P.keySorted.get(), P.permSorted.get(),
           static_cast<unsigned>(n), tileKeyBits(ntiles), st);
  PermuteArgs32 A{};
  for (int a = 0; a < 3; ++a) {
    A.cellSrc[a] = P.cell[a].get();
    A.cellDst[a] = P.cellT[a].get();
  }
  for (int a = 0; a < 9; ++a) {
    A.src[a] = P.s[a].get();
    A.dst[a] = P.t[a].get();
  }
  A.idSrc = P.id.get();
  A.idDst = P.idT.get();
  A.stateSrc = P.state.get();
  A.stateDst = P.stateT.get();
  A.betaSrc = P.beta.get();
  A.betaDst = P.betaT.get();
  // |q kq_a v_a| with |v_a| < c dt / h_a cells, with a margin for the FP32 rounding
  const double h[3] = {F.g.dx, F.g.dy, F.g.dz};
  double perCharge = 0.0;
  for (int a = 0; a < 3; ++a)
    perCharge = std::max(perCharge, static_cast<double>(static_cast<float>(h[a] / (F.g.dx * F.g.dy * F.g.dz * F.g.dt))) *
                                        (kC * F.g.dt / h[a]));
  perCharge *= 1.0 + 1e-6;
  const TileBoundsArgs T{P.keySorted.get(), n, ntiles, C.tileBegin.get(), C.tileEnd.get(), C.tileBound.get(),
                         perCharge};
  kPermute32<<<dim3(blocks, 4), 256, 0, st>>>(A, P.permSorted.get(), n, T);
  launchCheck("permute");
  for (int a = 0; a < 3; ++a) P.cell[a].swap(P.cellT[a]);
  for (int a = 0; a < 9; ++a) P.s[a].swap(P.t[a]);
  P.id.swap(P.idT);
  P.state.swap(P.stateT);
  P.beta.swap(P.betaT);
  const int rz = C.shape == kShapeQuintic ? Box<kShapeQuintic>::RZ : Box<kShapeBinomial3X>::RZ;
  buildChunkLists(C, st, ntx, nty, ntiles, rz, n, chunkSize32(n), C.mailbox.device(), seq);
}

}  // namespace

struct SplitStepContext {
  bool pending = false, middleDone = false, verify = false;
  int n = 0, sortedEntries = 0, ntx = 0, nty = 0, ntz = 0, ntiles = 0;
  std::size_t chunkBound = 0;
  unsigned sortSeq = 0, postSeq = 0;  // mailbox sequence numbers of the sort phase and of the step's end
  unsigned trials = 2, nChunks = 0, occupied = 0, active = 0;
  GArgs32 G{};
  StepArgs S{};
  double o[3] = {0.0, 0.0, 0.0};
};

// Phase 1 of a split step: checks, J clear, sort and chunk lists (their
// totals copied back asynchronously), and the zero-current preview.
// The split positions live on the lattice x = cell * h; the grid origin
// must be one of its nodes: oc its lattice cell, o = oc * h.
static void splitOrigin(const FieldState32& F, const double origin[3], int oc[3], double o[3]) {
  const double h[3] = {F.g.dx, F.g.dy, F.g.dz};
  for (int a = 0; a < 3; ++a) {
    const double r = origin[a] / h[a];
    if (!std::isfinite(r) || std::fabs(r) >= 1.0e9 || std::fabs(r - std::nearbyint(r)) > 1e-6)
      throw std::invalid_argument("An FP32-split grid origin must lie on the cell lattice (origin = integer * spacing)");
    oc[a] = static_cast<int>(std::nearbyint(r));
    o[a] = static_cast<double>(oc[a]) * h[a];
  }
}

// The step's sort phase on stream ss: tile lists and readback words sized,
// error words cleared, then (with particles) the stable tile sort, the
// state permute and the chunk lists, whose totals are posted to the mailbox
// under the returned sequence number.
static unsigned sortPhaseSplit(CouplingState& C, SplitStore& P, const double origin[3], hipStream_t ss) {
  FieldState32& F = *C.fields32;
  int oc[3];
  double o[3];
  splitOrigin(F, origin, oc, o);
  const int n = static_cast<int>(P.count);
  const int ntx = static_cast<int>((F.g.nx + kTileX - 1) / kTileX);
  const int nty = static_cast<int>((F.g.ny + kTileY - 1) / kTileY);
  const int ntz = static_cast<int>((F.g.nz + kTileZ - 1) / kTileZ);
  const int ntiles = ntx * nty * ntz;
  reserveTileLists(C, ss, ntiles, n);
  reserveCouplingWords(C, ss);
  DigitCounts D{};
  if (n) {
    reserveSortTemp(P.sortTemp, P.sortTempBytes, P.count);
    D = tileSortCounts(P.sortTemp.get(), static_cast<unsigned>(n), tileKeyBits(ntiles));
  }
  clearStepWords(C, D, ss);
  if (!n) return 0;
  SortArgs K{};
  K.window = F.window ? 1 : 0;
  K.nz = static_cast<int>(F.g.nz);
  K.lowZ = o[2];
  K.upZ = std::fma(static_cast<double>(F.g.nz), F.g.dz, o[2]);
  K.dz = F.g.dz;
  K.words = C.error.get();
  K.removed = P.removed.get();
  reserveKeyBlocks(C, n);
  K.blockActive = C.keyActive.get();
  const unsigned seq = C.mailbox.next(0);
  sortSplit(C, P, gatherArgs32(C, F, oc), K, ntx, nty, ntiles, D, seq, ss);
  return seq;
}

void prepareStepSplit(CouplingState& C, SplitStore& P, const double origin[3]) {
  FieldState32& F = *C.fields32;
  if (C.prepared.valid) throw std::logic_error("A prepared coupling step is already pending");
  if (C.split && C.split->pending) throw std::logic_error("The previous FP32-split coupling step was not finished");
  hipStream_t ss = C.sortStream.get();
  // J of the last deposit is cleared through that step's active-tile list,
  // which this sort rewrites: clear it now, ahead of the sort (every step
  // starts from J = 0, and the step's own clear then finds nothing to do)
  if (F.footprint.valid && !F.currentZero) launchClearCurrent(F);
  hipCheck(hipEventRecord(C.prepareStart.get(), F.stream), "hipEventRecord");
  hipCheck(hipStreamWaitEvent(ss, C.prepareStart.get(), 0), "hipStreamWaitEvent");
  const unsigned seq = sortPhaseSplit(C, P, origin, ss);
  hipCheck(hipEventRecord(C.sortReady.get(), ss), "hipEventRecord");
  auto& R = C.prepared;
  R.valid = true;
  R.store = &P;
  R.generation = P.generation;
  R.count = P.count;
  for (int a = 0; a < 3; ++a) R.origin[a] = origin[a];
  R.seq = seq;
}

void splitStepBegin(CouplingState& C, SplitStore& P, const double origin[3], double time, unsigned substeps) {
  FieldState32& F = *C.fields32;
  if (!C.split) C.split = std::make_shared<SplitStepContext>();
  SplitStepContext& X = *C.split;
  if (X.pending) throw std::logic_error("The previous FP32-split coupling step was not finished");
  if (F.window && F.phase != 2) throw std::logic_error("Moving-window electric phase mismatch");
  if (F.window && !F.inletSet) throw std::logic_error("Moving-window inlet planes were not supplied");
  if (substeps == 0) throw std::invalid_argument("Particle substeps must be positive");
  int oc[3];
  double o[3];
  splitOrigin(F, origin, oc, o);
  const int n = static_cast<int>(P.count);
  hipStream_t st = F.stream;
  launchClearCurrent(F);
  for (int a = 0; a < 3; ++a)
    if (C.esum032[a].size() != F.compSize(a)) {
      C.esum032[a].resize(F.compSize(a));
      C.esum32[a].resize(F.compSize(a));
    }
  const GArgs32 G = gatherArgs32(C, F, oc);
  const int ntx = static_cast<int>((F.g.nx + kTileX - 1) / kTileX);
  const int nty = static_cast<int>((F.g.ny + kTileY - 1) / kTileY);
  const int ntz = static_cast<int>((F.g.nz + kTileZ - 1) / kTileZ);
  const int ntiles = ntx * nty * ntz;
  const std::size_t chunkBound = chunkListBound(ntiles, n);
  const unsigned trials = std::max(2u, C.splitTrials);
  if (preparedFor(C, &P, P.generation, P.count, origin)) {
    hipCheck(hipStreamWaitEvent(st, C.sortReady.get(), 0), "hipStreamWaitEvent");
    X.sortSeq = C.prepared.seq;
  } else {
    if (C.prepared.valid) hipCheck(hipStreamWaitEvent(st, C.sortReady.get(), 0), "hipStreamWaitEvent");
    X.sortSeq = sortPhaseSplit(C, P, origin, st);
  }
  C.prepared.valid = false;
  // E* + E^n on the nodes of active tiles only (their only readers)
  float* const sums[3] = {C.esum032[0].get(), C.esum032[1].get(), C.esum032[2].get()};
  if (n)
    launchElectricPreviewTiles(F, F.ptrs(), sums, F.window ? F.inletPlane[0] : nullptr,
                               F.window ? F.inletPlane[1] : nullptr, C.activeTiles.get(), C.tileScan.get() + ntiles,
                               TileGrid{ntx, nty, ntz, kTileX, kTileY, kTileZ});
  X.pending = true;
  X.middleDone = false;
  X.n = n;
  X.sortedEntries = n;
  X.ntx = ntx;
  X.nty = nty;
  X.ntz = ntz;
  X.ntiles = ntiles;
  X.chunkBound = chunkBound;
  X.trials = trials;
  X.G = G;
  for (int a = 0; a < 3; ++a) X.o[a] = o[a];
  X.S = stepArgsFor(C, F.g, F.hasCpml ? &F.cpml : nullptr, F.window, o, time, substeps);
}

// Phase 2: wait for the chunk totals, enqueue the Picard trials and the
// commit, and the one asynchronous readback of the step; the store's
// state arrays are swapped (stream order keeps later work consistent).
void splitStepMiddle(CouplingState& C, SplitStore& P) {
  FieldState32& F = *C.fields32;
  if (!C.split || !C.split->pending || C.split->middleDone) throw std::logic_error("FP32-split step phase mismatch");
  SplitStepContext& X = *C.split;
  int n = X.n;
  const int ntx = X.ntx, nty = X.nty, ntz = X.ntz, ntiles = X.ntiles;
  const std::size_t chunkBound = X.chunkBound;
  unsigned trials = X.trials;
  const GArgs32& G = X.G;
  const double* o = X.o;
  hipStream_t st = F.stream;
  (void)ntiles;
  unsigned nChunks = 0, nActive = 0, occupiedTiles = 0;
  if (n) {
    C.mailbox.wait(0, X.sortSeq, st);
    const unsigned* box = C.mailbox.host();
    nChunks = box[8];
    nActive = box[9];
    occupiedTiles = box[11];
    // finishMovingWindowStep's checks of the entries, applied to this origin
    raiseParticleErrors(box[10]);
    const int behind = static_cast<int>(box[12]);
    if (box[13]) cropCounters(C, st, n - behind, n, P.state.get(), P.s[6].get(), P.s[8].get(), true);
    n -= behind;  // removed and cropped entries now trail the live ones
    P.count = static_cast<std::size_t>(n);
    X.n = n;
    // with no active entry (held ones and carriers only) no particle makes a
    // coupling call, and the reference converges in one trial
    // (simulation_source_coupling.cpp:50)
    if (!box[14]) trials = 1;
    if (nChunks > chunkBound) throw std::logic_error("Chunk list exceeds its bound");
  } else {
    trials = 1;
  }
  const bool quintic = C.shape == kShapeQuintic;
  const int boxN = quintic ? boxNodes<kShapeQuintic>() : boxNodes<kShapeBinomial3X>();
  const int rawN = quintic ? rawNodes<kShapeQuintic>() : rawNodes<kShapeBinomial3X>();
  const TileBoxes boxes = reserveStepBuffers(C, 3 * static_cast<std::size_t>(boxN), 3 * static_cast<std::size_t>(rawN),
                                             nChunks, occupiedTiles, st);

  const StepArgs& S = X.S;
  PArgs32 A = particleArgs32(P, F);
  A.tileBound = C.tileBound.get();
  const bool verify = C.splitVerify;
  const bool loop = chunkSize32(X.sortedEntries) > kChunk;
  for (unsigned trial = 0; trial < trials; ++trial) {
    unsigned* errT = C.error.get() + kTrialWord + trial;
    const bool last = trial + 1 == trials;
    if (nChunks && trial == 0) {
      ScopedKernel sk(F.profiler, st, "gather");
      GArgs32 G0 = G;
      for (int a = 0; a < 3; ++a) G0.esum[a] = C.esum032[a].get();
#define APRL_GATHER32(M, SH, L) \
  kGatherChunks32<M, SH, L><<<nChunks, kChunk, 0, st>>>(A, M ? G : G0, S, C.chunks.get(), ntx, nty, F.g.dt, stats, errT)
      double* const stats = nullptr;
      if (quintic) {
        if (loop) APRL_GATHER32(0, kShapeQuintic, true);
        else APRL_GATHER32(0, kShapeQuintic, false);
      } else {
        if (loop) APRL_GATHER32(0, kShapeBinomial3X, true);
        else APRL_GATHER32(0, kShapeBinomial3X, false);
      }
      launchCheck("gather");
    }
    if (n) {
      ScopedKernel sk(F.profiler, st, "push");
      kPushSplit<<<ceilDiv(n, 128), 128, 0, st>>>(A, S, o[0], o[1], o[2], errT);
      launchCheck("push");
    }
    if (!nChunks) {
      referenceCurrentTrial(C, F, C.esum32[2].get(), C.esum032[2].get(), false, false, ntx, nty, ntz);
      continue;
    }
    {
      ScopedKernel sk(F.profiler, st, "deposit");
#define APRL_DEPOSIT32(SH, L)                                                                                    \
  kDepositSplit<SH, L><<<nChunks, kChunk, 0, st>>>(A, G, S, C.chunks.get(), C.tileBegin.get(), C.tileEnd.get(),  \
                                                   C.tileScan.get(), ntx, nty, boxes, C.tileShift.get(), errT)
      if (quintic) {
        if (loop) APRL_DEPOSIT32(kShapeQuintic, true);
        else APRL_DEPOSIT32(kShapeQuintic, false);
      } else {
        if (loop) APRL_DEPOSIT32(kShapeBinomial3X, true);
        else APRL_DEPOSIT32(kShapeBinomial3X, false);
      }
#undef APRL_DEPOSIT32
      launchCheck("deposit");
      foldTiles(C, boxes, F.g, nChunks, occupiedTiles, nullptr, st);
    }
    // the last trial's E_cand + E_old is read only by a verifying residual
    const bool esum = !last || verify;
    {
      ScopedKernel sk(F.profiler, st, "reduce_current");
      float* j[3] = {F.base(6), F.base(7), F.base(8)};
      const bool writeJ = last || C.refCurrent;
#define APRL_REDUCE32(SH, WJ, WE)                                                                                     \
  kReduceCurrentSplit<SH, WJ, WE><<<nActive, 256, 0, st>>>(j[0], j[1], j[2], G, C.activeTiles.get(), C.tileScan.get(), \
                                                           C.tileShift.get(), boxes.boxes, ntx, nty, ntz)
      if (quintic) {
        if (writeJ && esum) APRL_REDUCE32(kShapeQuintic, true, true);
        else if (writeJ) APRL_REDUCE32(kShapeQuintic, true, false);
        else APRL_REDUCE32(kShapeQuintic, false, true);
      } else {
        if (writeJ && esum) APRL_REDUCE32(kShapeBinomial3X, true, true);
        else if (writeJ) APRL_REDUCE32(kShapeBinomial3X, true, false);
        else APRL_REDUCE32(kShapeBinomial3X, false, true);
      }
#undef APRL_REDUCE32
      launchCheck("reduce current");
    }
    F.currentZero = false;
    F.footprint.valid = true;
    F.footprint.active = C.activeTiles.get();
    F.footprint.count = static_cast<int>(nActive);
    F.footprint.ntx = ntx;
    F.footprint.nty = nty;
    F.footprint.ntz = ntz;
    F.footprint.tx = kTileX;
    F.footprint.ty = kTileY;
    F.footprint.tz = kTileZ;
    // TransverseReferenceCurrent::apply after the trial's deposit
    referenceCurrentTrial(C, F, C.esum32[2].get(), C.esum032[2].get(), esum, true, ntx, nty, ntz);
    if (last && !verify) break;
    {
      ScopedKernel sk(F.profiler, st, "residual");
      double* stats = last ? C.reduceBlocks.get() : nullptr;
      const GArgs32& G0 = G;
      if (quintic) {
        if (loop) APRL_GATHER32(1, kShapeQuintic, true);
        else APRL_GATHER32(1, kShapeQuintic, false);
      } else {
        if (loop) APRL_GATHER32(1, kShapeBinomial3X, true);
        else APRL_GATHER32(1, kShapeBinomial3X, false);
      }
#undef APRL_GATHER32
      launchCheck("residual");
    }
    if (last) reduceChunkStats(st, C.reduceBlocks.get(), static_cast<int>(nChunks), C.reduceOut.get());
    for (int a = 0; a < 6; ++a) std::swap(A.fin[a], A.fout[a]);
  }
  // one readback per step: the trial error words (and the verifying
  // residual), final once the last trial has run; the step's end waits for
  // them only, so the commit below runs while the host enqueues the next step
  X.postSeq = C.mailbox.next(1);
  postTrialWords(C, st, trials, verify && nChunks, X.postSeq);
  // commitConservativeElectric with the last trial's current
  if (F.window) windowCommitElectric(F, F.ptrs());
  else launchElectric(F, F.ptrs(), F.inletPlane[0], F.inletPlane[1]);
  if (F.window) F.phase = 3;
  X.verify = verify;
  X.trials = trials;
  X.nChunks = nChunks;
  X.occupied = occupiedTiles;
  X.active = nActive;
  X.middleDone = true;
  for (int a = 0; a < 3; ++a) P.cell[a].swap(P.endCell[a]);
  for (int a = 0; a < 6; ++a) P.s[a].swap(P.end[a]);
  C.lastStep.valid = true;
  C.lastStep.store = &P;
  C.lastStep.generation = P.generation;
  for (int a = 0; a < 3; ++a) C.lastStep.origin[a] = o[a];
}

// Phase 3: wait for the step, raise the first device error in trial order,
// fill the report.
void splitStepEnd(CouplingState& C, SplitStore& P, aprl_step_report* report) {
  if (!C.split || !C.split->pending || !C.split->middleDone) throw std::logic_error("FP32-split step phase mismatch");
  SplitStepContext& X = *C.split;
  X.pending = false;
  const unsigned trials = X.trials;
  const bool verify = X.verify;
  const unsigned nChunks = X.nChunks;
  C.mailbox.wait(1, X.postSeq, C.fields32->stream);
  const unsigned* words = C.mailbox.host() + 16;
  const double* sums = C.mailbox.hostDoubles();
  for (unsigned t = 0; t < trials; ++t) raiseParticleErrors(words[t]);
  // Boundary events of the last trial: carriers, removals, counters. The
  // commit only touches entry states, weights and counters, which nothing
  // reads before the next step or query.
  if (X.n && (words[trials - 1] & kEvtAny))
    commitEvents(C, C.fields32->stream, X.n, P.evt.get(), P.state.get(), P.s[8].get(), P.s[6].get(), P.wend.get(),
                 P.removed.get(), C.error.get() + kTrialWord + (trials - 1), true);
  double force = 0., work = 0.;
  if (verify && nChunks) {
    force = sums[0];
    work = sums[3] == 0. ? 0. : (sums[2] > 0. ? sums[1] / sums[2] : sums[1]);
  }
  if (report) {
    report->iterations = trials;
    report->force = force;
    report->work = work;
    report->tiles = X.occupied;
    report->chunks = nChunks;
    report->active_tiles = X.active;
  }
}

void couplingStepSplit(CouplingState& C, SplitStore& P, const double origin[3], double time, unsigned substeps,
                       aprl_step_report* report) {
  splitStepBegin(C, P, origin, time, substeps);
  splitStepMiddle(C, P);
  splitStepEnd(C, P, report);
}

}  // namespace aprl_gpu
