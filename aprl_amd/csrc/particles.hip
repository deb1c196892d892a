// gfx950 particle kernels of the conservative-source step (FP64 form):
// tile sort, orbit gather + Lapenta-Markidis push with prescribed magnets,
// deterministic tile deposition of the binomial3-x or compensated-quintic
// current, residual gathers with fixed-order reductions, and the Picard
// orchestration.
//
// The push follows source_coupling_math.h / source_coupling.cpp in the
// reference's association order (contraction off), so with identical field
// inputs it is bitwise the reference's. The gathers' and the deposit's weights
// are longitudinal_shape.h's summed in another order, with contraction
// (shapes.hpp).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>

#include "blockscan.hpp"
#include "diagnostics.hpp"
#include "particle_device.hpp"
#include "shapes.hpp"
#include "tuner.hpp"

namespace aprl_gpu {

// ---------------------------------------------------------------------------
// Kernel argument blocks.

struct GArgs {
  double* esum[3];         // E_cand + E_old of the trial
  const double* esum0[3];  // E* + E_old, E* the zero-current preview
  const double* b[3];      // B^(n+1/2)
  int ne[3][3], nb[3][3];  // (nx, ny, nz) of E (= J) and B components
  int nx, ny, nz;          // cells
  double o[3], h[3];
  double negS;             // (-1*dt)/eps0, applyCurrentSource(-1)
  // the Picard stop word: a trial's kernels return at once when it is set
  // (null for work that always runs)
  const unsigned* stop;
};

struct PArgs {
  double* x[3];
  double* u[3];
  const double* q;
  const double* m;
  double* fin[6];   // fields the trial pushes with: Ex Ey Ez Bx By Bz
  double* fout[6];  // next fields of the residual gather
  double* x1[3];
  double* u1[3];
  double* gridAbs;
  const int* state;  // entry states (kStateActive / kStateCarrier for live entries)
  int* evt;          // boundary event code of the trial
  double* cut[3];    // t1, t2, carrier-part deposit weight
  double* wend;      // carrier end weight
  const double* w;   // weight slot (a carrier's current weight)
  const double* beta;  // held speed of held entries
  const unsigned long long* tileBound;  // per tile: largest entry current bound
  double scaleDen;   // dx*dy*dz*dt
  int n;
};

// ---------------------------------------------------------------------------
// Device math restated from the reference.

// clipOpenOrbit for one owner of the whole domain, source_coupling_math.h:235-250.
struct Clip { double b[3], e[3], first, last; bool valid; };
__device__ Clip clipOrbit(const GArgs& G, const double begin[3], const double end[3], unsigned& err) {
  Clip r;
  r.first = 0.;
  r.last = 1.;
  r.valid = true;
  const int size[3] = {G.nx, G.ny, G.nz};
  for (int a = 0; a < 3; ++a) {
    r.b[a] = begin[a];
    r.e[a] = end[a];
    const double x = (begin[a] - G.o[a]) / G.h[a], d = (end[a] - begin[a]) / G.h[a];
    if (!isfinite(x) || !isfinite(d)) { err |= kErrNonfinite; r.valid = false; return r; }
    if (d == 0.) {
      if (x < 0. || x > size[a]) r.valid = false;
      continue;
    }
    {
      const double t = -x / d;
      if (d > 0.) r.first = fmax(r.first, t);
      else r.last = fmin(r.last, t);
    }
    {
      const double t = (double(size[a]) - x) / d;
      if (d > 0.) r.last = fmin(r.last, t);
      else r.first = fmax(r.first, t);
    }
  }
  r.valid = r.valid && r.last >= r.first;
  if (r.valid)
    for (int a = 0; a < 3; ++a) {
      const double d = end[a] - begin[a];
      if (r.first != 0.) r.b[a] = begin[a] + r.first * d;
      if (r.last != 1.) r.e[a] = begin[a] + r.last * d;
    }
  return r;
}

// The chord begin -> end in cells from the grid's origin, clipped to the grid
// (clipOpenOrbit): start x, displacement v, kept fraction. A chord that lies
// in the grid needs none of the clip's divisions. x is the quotient that
// names the start's tile (kTileKeys): a product with 1 / h differs from it by
// a rounding, and a chord that starts on a tile's face and moves a whole cell
// would then leave its tile's box.
__device__ __forceinline__ bool chordInGrid(const GArgs& G, const double begin[3], const double end[3], double x[3],
                                            double v[3], double& kept, unsigned& err) {
  const int size[3] = {G.nx, G.ny, G.nz};
  bool inside = true;
  for (int a = 0; a < 3; ++a) {
    x[a] = (begin[a] - G.o[a]) / G.h[a];
    v[a] = (end[a] - begin[a]) / G.h[a];
    const double last = x[a] + v[a], n = size[a];
    inside = inside && x[a] >= 0. && x[a] <= n && last >= 0. && last <= n;
  }
  kept = 1.;
  if (inside) return true;
  const Clip path = clipOrbit(G, begin, end, err);
  for (int a = 0; a < 3; ++a) {
    x[a] = (path.b[a] - G.o[a]) / G.h[a];
    v[a] = (path.e[a] - path.b[a]) / G.h[a];
  }
  kept = path.last - path.first;
  return path.valid;
}

// ---------------------------------------------------------------------------
// Sort and chunk list.

__device__ __forceinline__ int clampCell(double lattice, int n) {
  const int c = static_cast<int>(floor(lattice));
  return c < 0 ? 0 : (c > n - 1 ? n - 1 : c);
}

__global__ void kTileKeys(const double* x, const double* y, const double* z, int* state, int n, GArgs G, int ntx,
                          int nty, unsigned* key, TileRangeArgs R, SortArgs K, DigitCounts D) {
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
    if (!liveEntry(K, state, p, z[p])) {
      tile = static_cast<unsigned>(R.ntiles);
    } else {
      const int cx = clampCell((x[p] - G.o[0]) / G.h[0], G.nx);
      const int cy = clampCell((y[p] - G.o[1]) / G.h[1], G.ny);
      const int cz = clampCell((z[p] - G.o[2]) / G.h[2], G.nz);
      tile = (static_cast<unsigned>(cz / kTileZ) * nty + cy / kTileY) * ntx + cx / kTileX;
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

struct PermuteArgs {
  const double* src[9];
  double* dst[9];
  const uint64_t* idSrc;
  uint64_t* idDst;
  const int* stateSrc;
  int* stateDst;
  const double* betaSrc;
  double* betaDst;
};

// State scatter into sorted order, and the tile ranges of the sorted keys.
// The gathered reads of a permute are latency-bound: blockIdx.y splits the
// arrays over four times as many waves (y = 0: positions, tile ranges and
// bounds; 1: momenta; 2: q, m, w; 3: ids, states, held speeds).
__global__ void kPermute(PermuteArgs A, const unsigned* perm, int n, TileBoundsArgs T) {
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
      tileBoundsAt(T, p);
      const unsigned k = T.key[p];
      if (k < static_cast<unsigned>(T.ntiles)) {
        tile = k;
        bound = entryCurrentBound(A.src[6][from], A.stateSrc[from], T.perCharge);
      }
    }
  }
  if (part == 0) raiseTileBound(T.bound, tile, bound);
}

// Per tile, packed (packTileCounts): chunk count, whether it is occupied,
// and whether any tile within one tile in x and y and rz tiles in z is
// occupied (its J nodes can then receive current); entry ntiles is 0 so
// that the exclusive scan ends with the totals. Per workgroup, the sum of
// its counts.
__device__ __forceinline__ unsigned long long tileCount(const int* begin, const int* end, int ntx, int nty, int ntz,
                                                        int rz, int chunk, int t) {
  if (t >= ntx * nty * ntz) return 0ull;
  const int tx = t % ntx, ty = (t / ntx) % nty, tz = t / (ntx * nty);
  unsigned touched = 0;
  for (int oz = -rz; oz <= rz; ++oz)
    for (int oy = -1; oy <= 1; ++oy)
      for (int ox = -1; ox <= 1; ++ox) {
        const int x = tx + ox, y = ty + oy, z = tz + oz;
        if (x < 0 || x >= ntx || y < 0 || y >= nty || z < 0 || z >= ntz) continue;
        const int s = (z * nty + y) * ntx + x;
        if (end[s] > begin[s]) touched = 1;
      }
  const unsigned chunks = static_cast<unsigned>((end[t] - begin[t] + chunk - 1) / chunk);
  return packTileCounts(chunks, chunks ? 1u : 0u, touched);
}
__global__ void __launch_bounds__(kScanThreads) kTileCounts(const int* begin, const int* end, int ntx, int nty,
                                                            int ntz, int rz, int chunk, unsigned long long* counts,
                                                            unsigned long long* sums, const unsigned* keyActive,
                                                            int keyBlocks, unsigned* activeEntries) {
  __shared__ unsigned long long ws[kScanWaves + 1];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned long long c = tileCount(begin, end, ntx, nty, ntz, rz, chunk, t);
  if (t <= ntx * nty * ntz) counts[t] = c;
  unsigned long long total;
  (void)blockExclusiveScan(c, ws, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
  // the live active entries: the key kernel's workgroups store their counts
  // and these fewer ones add them to the one word (an atomic of every key
  // workgroup on it took 12 ns each: the key kernel 184 -> 60 us with 4e6
  // entries, beside the magnetic sweep, 8.0 -> 4.9 us with 1e5)
  unsigned long long part = 0ull;
  for (int q = t; q < keyBlocks; q += static_cast<int>(gridDim.x) * kScanThreads) part += keyActive[q];
  (void)blockExclusiveScan(part, ws, total);
  if (threadIdx.x == 0 && total) atomicAdd(activeEntries, static_cast<unsigned>(total));
}

// Exclusive scan of the counts, the chunk list in tile order and the list of
// active tiles (tiles with an occupied neighbour). A workgroup sums the
// workgroup sums before it itself (integers: exact in any order), so that
// the scan takes no launch of its own: at 64x64x512 (33 workgroups) the
// lists take two launches instead of four on the chain of launches that
// the sort phase waits for; at the most tiles (8192 workgroups) a lane reads
// at most 32 sums.
// With a mailbox, the lane of entry ntiles also posts the scan total
// (chunks, active tiles, occupied tiles) and the sort-phase words to host
// memory (values at words 8..14, sequence number in flag word 0).
__global__ void __launch_bounds__(kScanThreads) kChunkList(const int* begin, const int* end,
                                                           const unsigned long long* counts,
                                                           const unsigned long long* sums, unsigned long long* scan,
                                                           int ntiles, int chunk, int4* chunks, int* active, unsigned* box,
                                                           unsigned seq, const unsigned* words) {
  __shared__ unsigned long long ws[kScanWaves + 1];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long part = 0ull, before, total;
  for (int q = static_cast<int>(threadIdx.x); q < static_cast<int>(blockIdx.x); q += kScanThreads) part += sums[q];
  const unsigned long long count = t < ntiles ? counts[t] : 0ull;
  (void)blockExclusiveScan(part, ws, before);
  const unsigned long long sc = before + blockExclusiveScan(count, ws, total);
  if (t <= ntiles) scan[t] = sc;
  if (box && t == ntiles) {
    volatile unsigned* v = box;
    v[8] = static_cast<unsigned>(chunkField(sc));
    v[9] = static_cast<unsigned>(activeField(sc));
    for (int w = 0; w < 5; ++w) v[10 + w] = words[w];
    v[11] = static_cast<unsigned>(occupiedField(sc));  // in place of word 1
    __threadfence_system();
    v[0] = seq;
  }
  if (t >= ntiles) return;
  if (activeField(count)) active[activeField(sc)] = t;
  const int e = end[t];
  int c = chunkField(sc), fold = chunkField(count) > 1 ? occupiedField(sc) + 1 : 0;
  for (int p = begin[t]; p < e; p += chunk, ++c, fold = 0) chunks[c] = make_int4(t, p, min(e, p + chunk), fold);
}

__global__ void kClearWords(unsigned* a, unsigned na, unsigned* b, unsigned nb) {
  const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < na) a[t] = 0u;
  for (unsigned q = t; q < nb; q += gridDim.x * blockDim.x) b[q] = 0u;
}

// ---------------------------------------------------------------------------
// Gathers, push, deposit, residual.

// One Picard trial's residual: the chunk partials reduced in a fixed tree
// to (max force, defect sum, scale sum, coupling calls) in out. With a
// Picard word (W.stop) thread 0 then takes the reference's convergence
// decision on the device (simulation_source_coupling.cpp:46-51): at least
// two trials when a particle made a coupling call, force < 1e-13 and
// work < 1e-8, the same double arithmetic as the host test; a trial whose
// error word holds a device error also stops the trials. Once the word is
// set, later trials skip the reduction. With a mailbox, thread 0 posts the
// sums (doubles at byte 2048), the stop word (word 15) and the trial words
// firstWord..W.trial (words 16..) to host memory, sequence number in flag
// word 1, whether or not the trial ran. Called by all 256 threads of one
// workgroup; sh holds 4 x 256 doubles.
struct PicardWords {
  unsigned* stop;
  unsigned trial;
  const unsigned* trialWords;  // error words of trials 0..kMaxTrials-1
  unsigned firstWord;
};

__device__ void residualTail(const double* blockIn, int blocks, double* out, unsigned* box, unsigned seq,
                             const PicardWords& W, double* sh) {
  double* sf = sh;
  double* sd = sh + 256;
  double* ss = sh + 512;
  double* sc = sh + 768;
  const bool skip = W.stop && *W.stop;
  if (!skip) {
    double f = 0., d = 0., s = 0., c = 0.;
    for (int b = threadIdx.x; b < blocks; b += 256) {
      f = fmax(f, blockIn[4 * b]);
      d += blockIn[4 * b + 1];
      s += blockIn[4 * b + 2];
      c += blockIn[4 * b + 3];
    }
    sf[threadIdx.x] = f; sd[threadIdx.x] = d; ss[threadIdx.x] = s; sc[threadIdx.x] = c;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if (threadIdx.x < w) {
        sf[threadIdx.x] = fmax(sf[threadIdx.x], sf[threadIdx.x + w]);
        sd[threadIdx.x] += sd[threadIdx.x + w];
        ss[threadIdx.x] += ss[threadIdx.x + w];
        sc[threadIdx.x] += sc[threadIdx.x + w];
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      out[0] = sf[0]; out[1] = sd[0]; out[2] = ss[0]; out[3] = sc[0];
      if (W.stop) {
        const double force = sf[0];
        const double work = sc[0] == 0. ? 0. : (ss[0] > 0. ? sd[0] / ss[0] : sd[0]);
        const unsigned iterations = W.trial + 1;
        if (W.trialWords[W.trial] & ~kEvtAny) *W.stop = iterations | kStopError;
        else if (iterations >= (sc[0] > 0. ? 2u : 1u) && force < 1e-13 && work < 1e-8) *W.stop = iterations;
      }
    }
  }
  if (threadIdx.x == 0 && box) {
    volatile double* vd = reinterpret_cast<volatile double*>(reinterpret_cast<unsigned char*>(box) + 2048);
    vd[0] = out[0]; vd[1] = out[1]; vd[2] = out[2]; vd[3] = out[3];
    volatile unsigned* v = box;
    v[15] = W.stop ? *W.stop : 0u;
    for (unsigned w = W.firstWord; w <= W.trial; ++w) v[16 + w - W.firstWord] = W.trialWords[w];
    __threadfence_system();
    v[1] = seq;
  }
}

// Chunked orbit gathers from LDS-staged tile fields, one lane per particle:
// the orbit average of 1/2 (E_cand + E_old) over the clipped chord with the
// exact adjoint weights of the deposit (source_coupling.cpp:74-82), and B at
// the chord's midpoint. MODE 0: the first trial's gather at (x0, ballistic
// guess) against the zero-current preview (source_coupling.cpp:133-147); it
// writes the fields the first push uses. MODE 1: the residual gather of
// localResidual (source_coupling.cpp:148-202) at (x0, x1): next fields, and
// the chunk's force max and defect / scale / call sums in a fixed order.
// The fields are staged with the shape's convolution applied (stageBinomial,
// stageQuintic), so a chord of two segments reads 24 (quintic: 88) values
// instead of 128 (736), and B 24 staged ones instead of 96 from memory.
// 64x64x512, 1e5 particles, trial-0 and residual gather before and now:
// quintic 99 and 123 -> 34 and 37 us, binomial3-x 28 and 34 -> 20 and 27 us;
// FP32-split quintic, 4e6 particles: 878 and 950 -> 352 and 355 us. What is
// left is the staging's and the particles' load latency; the quintic's spline
// moments took it from 34 and 37 to 27 and 30 us (FP64, 236 -> 147 registers),
// from 352 and 355 to 330 and 333 us (4e6 particles).
template <int MODE, int SHAPE>
__global__ void __launch_bounds__(kChunk) __attribute__((amdgpu_waves_per_eu(SHAPE == kShapeBinomial3X ? 3 : 2)))
kGatherChunks(PArgs P, GArgs G, StepArgs S, const int4* chunks, int ntx, int nty, double dt, double* chunkOut,
              unsigned* errOut) {
  if (G.stop && *G.stop) return;
  constexpr int N = 3 * rawNodes<SHAPE>();
  __shared__ double es[N];
  __shared__ double bs[SHAPE == kShapeBinomial3X ? N : 1];
  __shared__ double stats[MODE == 1 ? kChunk / 4 : 1];
  const int cb = xcdContiguous(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
  const int4 ch = chunks[cb];
  const TileBox<SHAPE> box = tileBox<SHAPE>(ch.x, ntx, nty);
  const int p = ch.y + static_cast<int>(threadIdx.x);
  // This lane's particle data is loaded before the tile is staged, so that
  // its latency overlaps the staging loads' (lanes past the chunk's end read
  // its first entry and ignore it).
  const int pv = p < ch.z ? p : ch.y;
  const int stored = P.state[pv];
  double a[3], uv[3];
  for (int d = 0; d < 3; ++d) {
    a[d] = P.x[d][pv];
    uv[d] = MODE == 0 ? P.u[d][pv] : P.x1[d][pv];  // u (first gather) or the trial end x1
  }
  if constexpr (SHAPE == kShapeBinomial3X) {
    stageBinomial<true>(G, box, es);
    stageBinomial<false>(G, box, bs);
  } else {
    stageQuintic(G, box, es);
  }
  __syncthreads();
  // carriers move without fields and take no part in the residual; a held
  // entry takes part from its release point with the rest of the step
  const int st = p < ch.z ? stored : kStateRemoved;
  bool live = st == kStateActive;
  double dtp = dt;
  unsigned err = 0;
  if (st == kStateHeld) {
    const double uh[3] = {P.u[0][p], P.u[1][p], P.u[2][p]};
    const HeldMove h = heldMove(S, a, uh, P.beta[p]);
    if (h.release && h.remaining > 0.0) {
      live = true;
      for (int d = 0; d < 3; ++d) a[d] = h.x1[d];
      dtp = h.remaining;
    }
  }
  double force = 0., defect = 0., scale = 0., calls = 0.;
  if (live) {
    double b[3];
    if (MODE == 0) {
      const double gamma = gammaFromU(uv[0], uv[1], uv[2]);
      const double s = dtp * kC / gamma;
      for (int d = 0; d < 3; ++d) {
        b[d] = a[d];
        b[d] += s * uv[d];
      }
    } else {
      for (int d = 0; d < 3; ++d) b[d] = uv[d];
    }
    double x[3], v[3], mid[3], kept, g[6] = {0., 0., 0., 0., 0., 0.};
    if (chordInGrid(G, a, b, x, v, kept, err)) {
      const int org[3] = {0, 0, 0};  // x is grid-relative
      gatherRaw<SHAPE, double>(G.nx, G.ny, es, box, org, x, v, g, err);
      for (int d = 0; d < 3; ++d) {
        g[d] *= .5 * kept;
        mid[d] = x[d] + .5 * v[d];
      }
      if constexpr (SHAPE == kShapeBinomial3X) sampleBinomial(bs, box, org, mid, g + 3, err);
      else sampleQuinticB<false>(G, box, bs, org, mid, g + 3);
    } else {
      err |= kErrOrbitOutside | (SHAPE == kShapeBinomial3X ? kErrMagneticOutside : kErrMagneticNoDomain);
    }
    double* const* dst = MODE == 0 ? P.fin : P.fout;
    for (int d = 0; d < 6; ++d) dst[d][p] = g[d];
    if (MODE == 1) {
      double de[3], db[3];
      for (int d = 0; d < 3; ++d) {
        de[d] = g[d] - P.fin[d][p];
        db[d] = g[3 + d] - P.fin[3 + d][p];
      }
      const double q = P.q[p], m = P.m[p];
      force = fabs(q / m) * dtp / kC * (sqrt(de[0] * de[0] + de[1] * de[1] + de[2] * de[2]) +
                                        kC * sqrt(db[0] * db[0] + db[1] * db[1] + db[2] * db[2]));
      double w1 = 0., w2 = 0.;
      for (int d = 0; d < 3; ++d) {
        w1 += q * de[d] * (b[d] - a[d]);
        w2 += q * g[d] * (b[d] - a[d]);
      }
      defect = fabs(w1);
      scale = P.gridAbs[p] + fabs(w2);
      calls = 1.;
    }
  }
  if (MODE == 1) chunkStats(stats, force, defect, scale, calls, chunkOut + 4 * cb);
  if (err) atomicOr(errOut, err);
}

// Push of source_coupling.cpp:133-147 for one trial with the gathered
// fields (the substeps with prescribed magnets), or the straight move of a
// CPML carrier (position += dt u c / gamma, simulation.cpp:4407-4413), then
// the segment's boundary events. (The tile current bounds the deposit's
// fixed-point exponents come from are set once per step by the sort.)
__global__ void __launch_bounds__(128) kPush(PArgs P, GArgs G, StepArgs S, unsigned* errOut) {
  if (G.stop && *G.stop) return;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P.n) return;
  unsigned err = 0;
  const double x0[3] = {P.x[0][p], P.x[1][p], P.x[2][p]};
  const double u0[3] = {P.u[0][p], P.u[1][p], P.u[2][p]};
  double x[3], u[3], absGrid, t1, t2, wDeposit, wEnd;
  const double usedE[3] = {P.fin[0][p], P.fin[1][p], P.fin[2][p]};
  const double usedB[3] = {P.fin[3][p], P.fin[4][p], P.fin[5][p]};
  const int code = entryStep(S, G.o, P.state[p], x0, u0, P.q[p], P.m[p], P.w[p], P.beta[p], usedE, usedB, x, u,
                             absGrid, t1, t2, wDeposit, wEnd, err);
  for (int a = 0; a < 3; ++a) {
    P.x1[a][p] = x[a];
    P.u1[a][p] = u[a];
  }
  P.gridAbs[p] = absGrid;
  P.evt[p] = code;
  if (code) {
    P.cut[0][p] = t1;
    P.cut[1][p] = t2;
    P.cut[2][p] = wDeposit;
    P.wend[p] = wEnd;
    err |= kEvtAny;
  }
  if (err) atomicOr(errOut, err);
}

// Deterministic tile deposition of Current::deposit (longitudinal_shape.h:
// 175-187): one workgroup per chunk, one lane per particle, every raw tap of
// the chord x0 -> x1 (RawBox) accumulated into an LDS copy of the tile's raw
// box in 64-bit fixed point; the write-out applies the shape's convolution
// (kFoldTiles for a tile of several chunks). The binary exponent comes from a bound on the whole tile's
// current (the shape's weight bound times the tile's particle count times
// the largest bound of one entry, set by the sort), so every chunk of a
// tile uses the same scale. Integer addition is associative, so a tile's raw
// sums are the same in any order of its entries and in any division into
// chunks; each raw tap is rounded once, to 2^-62 of the tile bound, and a
// node's convolved sum over the whole tile once more to that unit.
// Bound by the LDS atomics (64 lanes on random nodes conflict) and the
// per-particle arithmetic with two or three waves per SIMD to hide either
// (231 registers for the quintic): 24 or 88 raw taps for a chord of two
// segments instead of 128 or 736, added without a mask when the whole wave's
// taps lie inside the box (fixedPoint). 64x64x512, 1e5 particles, with the
// reference's taps, with raw taps of quadrature sums (two lanes a quintic
// particle), and with splineMoments: quintic 116, 60 and 36 us (FP32-split 78,
// 44 and 34 us), binomial3-x 28, 26 and 24.5 us (FP32-split 28, 19 and 17 us);
// the chunks of larger tiles add raw sums instead of convolved ones (3993
// nodes instead of 6171, 2541 instead of 3861) for 33 (30) and 22.5 (15.4)
// us, and kFoldTiles.
template <int SHAPE>
__global__ void __launch_bounds__(kChunk) __attribute__((amdgpu_waves_per_eu(SHAPE == kShapeQuintic ? 2 : 3)))
kDeposit(PArgs P, GArgs G, StepArgs S, const int4* chunks, const int* tileBegin, const int* tileEnd,
         const unsigned long long* tileScan, int ntx, int nty, TileBoxes T, int* tileShift, unsigned* errOut) {
  if (G.stop && *G.stop) return;
  using W = RawBox<SHAPE>;
  constexpr int N = rawNodes<SHAPE>();
  __shared__ unsigned long long acc[3 * N];
  const int4 ch = chunks[blockIdx.x];
  const int tile = ch.x;
  const TileBox<SHAPE> box = tileBox<SHAPE>(tile, ntx, nty);
  for (int t = threadIdx.x; t < 3 * N; t += blockDim.x) acc[t] = 0ull;
  const unsigned long long tsc = tileScan[tile];
  const int shift = tileFixedShift(Box<SHAPE>::kWeightBound, P.tileBound[tile], tileEnd[tile] - tileBegin[tile]);
  if (threadIdx.x == 0 && static_cast<int>(blockIdx.x) == chunkField(tsc)) tileShift[tile] = shift;
  __syncthreads();
  unsigned err = 0;
  const int p = ch.y + static_cast<int>(threadIdx.x);
  if (p < ch.z) {
    double scale[3], part3[3];  // of the leg, and of the chord part (with its weight)
    double x[3], v[3], cuts[kMaxCuts];
    const int org[3] = {0, 0, 0};  // x is grid-relative
    int base = 0;
    unsigned mask[3] = {0, 0, 0};
    double fixed[3];  // part3 in the tile's fixed-point units
    auto corner = [&](int i, int j, int k) {
      base = box.rawIndex(i, j, k);
      const bool inside = rawDepositInside<SHAPE>(box, G.nx, G.ny, i, j, k);
#pragma unroll
      for (int d = 0; d < 3; ++d) fixed[d] = ldexp(part3[d], shift);
      if (__all(inside)) return true;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        mask[d] = part3[d] == 0. ? 0u : ~0u;
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
    // active part) and [t1, t2] at the carrier part's deposit weight. A held
    // entry released inside the step deposits its held leg x0 -> kink first.
    const int e = P.evt[p];
    const double t1 = e ? P.cut[0][p] : 1.0, t2 = e ? P.cut[1][p] : 1.0, wCarrier = e ? P.cut[2][p] : 0.0;
    double xa[3], xb[3], xk[3];
    for (int d = 0; d < 3; ++d) {
      xa[d] = P.x[d][p];
      xb[d] = P.x1[d][p];
      xk[d] = xa[d];
    }
    int legs = 1;
    if (P.state[p] == kStateHeld) {
      const double uh[3] = {P.u[0][p], P.u[1][p], P.u[2][p]};
      const HeldMove h = heldMove(S, xa, uh, P.beta[p]);
      if (h.release && h.kink) {
        legs = 2;
        for (int d = 0; d < 3; ++d) xk[d] = h.x1[d];
      }
    }
    const double q = P.q[p];
#pragma unroll 1
    for (int leg = 0; leg < legs; ++leg) {
      const bool last = leg + 1 == legs;
      for (int d = 0; d < 3; ++d) {
        const double s0 = leg ? xk[d] : xa[d], s1 = last ? xb[d] : xk[d];
        // scale_a = q * (x1_a - x0_a) / (dx dy dz dt), eb_deposition.cpp:41-51
        scale[d] = q * (s1 - s0) / P.scaleDen;
        x[d] = (s0 - G.o[d]) / G.h[d];
        v[d] = (s1 - s0) / G.h[d];
      }
      const int count = orbitCuts(x, v, cuts, err);
      const double f1 = last ? t1 : 1.0, f2 = last ? t2 : 1.0, fw = last ? wCarrier : 0.0;
      for (int sgm = 1; sgm < count; ++sgm) {
        const double c0 = cuts[sgm - 1], c1 = cuts[sgm];
        if (c1 - c0 <= 0.) continue;
        // without an event: one part [c0, c1] (t1 = t2 = 1)
#pragma unroll 1
        for (int part = 0; part < 2; ++part) {
          const double a = part ? fmax(c0, f1) : c0;
          const double b = part ? fmin(c1, f2) : fmin(c1, f1);
          if (!(b > a)) continue;
          for (int d = 0; d < 3; ++d) part3[d] = part ? scale[d] * fw : scale[d];
          rawSegment<SHAPE, double>(G.nx, G.ny, org, x, v, a, b, corner, tapInside, tap);
        }
      }
    }
  }
  __syncthreads();
  flushRawBox<SHAPE>(acc, box, G.nx, G.ny, G.nz, T, tileScan, tile);
  if (err) atomicOr(errOut, err);
}

// After a deposit: the boxes of the tiles of several chunks from their raw
// boxes. One workgroup per chunk, of which the tiles' first ones work. Bound
// by the latency of its chain (chunk, raw box, LDS, store) in small grids:
// 5.7 us at 64x64x512 with 1e5 particles (quintic 8.3 us), 18 us at
// 128x128x960 with 1e6 (8.2 us with each column's loads between its stores).
// A chunk that convolves what it adds saves this launch, but rounds each of
// its sums, so that the current depends on the division into chunks; exact
// (quotient and remainder added apart) it took deposit and reduction from 36
// and 30 to 47 and 46 us (quintic, 1e5).
template <int SHAPE>
__global__ void __launch_bounds__(kFoldThreads) kFoldTiles(TileBoxes T, const int4* chunks, int nx, int ny, int nz,
                                                           const unsigned* stop) {
  const int chunk = static_cast<int>(blockIdx.x);
  const int4 ch = chunks[chunk];
  const unsigned stopped = stop ? *stop : 0u;
  if (stopped || !ch.w) return;
  foldTile<SHAPE>(chunk, ch.w - 1, tileBox<SHAPE>(ch.x, (nx + kTileX - 1) / kTileX, (ny + kTileY - 1) / kTileY), nx,
                  ny, nz, T);
}

void foldTiles(CouplingState& C, const TileBoxes& T, const aprl_grid_geometry& g, unsigned nChunks, unsigned occupied,
               const unsigned* stop, hipStream_t st) {
  if (nChunks == occupied) return;  // no tile of several chunks
  const int nx = static_cast<int>(g.nx), ny = static_cast<int>(g.ny), nz = static_cast<int>(g.nz);
  if (C.shape == kShapeQuintic)
    kFoldTiles<kShapeQuintic><<<nChunks, kFoldThreads, 0, st>>>(T, C.chunks.get(), nx, ny, nz, stop);
  else
    kFoldTiles<kShapeBinomial3X><<<nChunks, kFoldThreads, 0, st>>>(T, C.chunks.get(), nx, ny, nz, stop);
  launchCheck("fold tiles");
}

// Node-owner reduction into J, one workgroup per active cell tile (a tile
// with an occupied tile within its box reach): each owned node sums, over
// the covering occupied tiles in fixed (tz, ty, tx) order, the tile's exact
// integer total converted with the tile's exponent. It also writes E_cand +
// E_old of the trial (applyCurrentSource(-1) on the preview,
// source_coupling.cpp:84-89) for the next residual gather, from the
// zero-current sums E* + E_old. J itself is only read after the last trial:
// writeJ is off for a trial that cannot be it. Nodes of other tiles keep the
// zeros J held at the start of the step.
// Bound by the boxes' loads (about five boxes cover a node) and, in small
// grids, their latency: the three components' loads go together, no box is
// cleared (the next deposit overwrites it), and J is written once a step.
// At first, with the components one after the other and every box cleared,
// then with the boxes of larger tiles cleared, and now: 19.5, 11.6 and 11.6 us
// (1e4 particles in 32x32x256), 34.5, 21 and 18.5 us (1e5 in 64x64x512;
// quintic 51, 30 and 26 us), 213, 129 and 114 us (1e6 in 128x128x960);
// FP32-split quintic, 4e6 particles, 510 and 436, 245 and 227, 226 and 208 us.
template <int SHAPE>
__global__ void __launch_bounds__(256) kReduceCurrent(double* jx, double* jy, double* jz, GArgs G, const int* active,
                                                      const unsigned long long* tileScan, const int* tileShift,
                                                      const long long* boxes, int ntx, int nty, int ntz, int writeJ) {
  if (G.stop && *G.stop) return;
  const int tile = active[xcdContiguous(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x))];
  reduceOwnedTile<SHAPE>(
      G.ne, tile, tileScan, tileShift, boxes, ntx, nty, ntz,
      [&](int i, int j, int k, const bool has[3], const double sum[3]) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if (!has[d]) continue;
          const size_t idx = (static_cast<size_t>(k) * G.ne[d][1] + j) * G.ne[d][0] + i;
          if (writeJ) (d == 0 ? jx : (d == 1 ? jy : jz))[idx] = sum[d];
          const bool applied = d == 0 ? (j > 0 && j < G.ny && k != 0 && k != G.nz)
                                      : (d == 1 ? (i > 0 && i < G.nx && k != 0 && k != G.nz)
                                                : (i > 0 && i < G.nx && j > 0 && j < G.ny));
          const double e = G.esum0[d][idx];
          G.esum[d][idx] = applied ? e + G.negS * sum[d] : e;
        }
      });
}

__global__ void __launch_bounds__(256) kReduceBlocks(const double* blockIn, int blocks, double* out, unsigned* box,
                                                     unsigned seq, PicardWords W) {
  __shared__ double sh[4 * 256];
  residualTail(blockIn, blocks, out, box, seq, W, sh);
}

// ---------------------------------------------------------------------------
// Host orchestration.

static GArgs gatherArgs(const CouplingState& C, const FieldState& F, const double origin[3]) {
  GArgs G{};
  for (int a = 0; a < 3; ++a) {
    G.esum[a] = C.esum[a].get();
    G.esum0[a] = C.esum0[a].get();
    G.b[a] = F.base(3 + a);
    for (int d = 0; d < 3; ++d) {
      G.ne[a][d] = static_cast<int>(F.dims[a][d]);
      G.nb[a][d] = static_cast<int>(F.dims[3 + a][d]);
    }
    G.o[a] = origin[a];
  }
  G.nx = static_cast<int>(F.g.nx);
  G.ny = static_cast<int>(F.g.ny);
  G.nz = static_cast<int>(F.g.nz);
  G.h[0] = F.g.dx; G.h[1] = F.g.dy; G.h[2] = F.g.dz;
  G.negS = -1.0 * F.g.dt / kEps0;
  return G;
}

static PArgs particleArgs(ParticleStore& P) {
  PArgs A{};
  for (int a = 0; a < 3; ++a) {
    A.x[a] = P.s[a].get();
    A.u[a] = P.s[3 + a].get();
    A.x1[a] = P.end[a].get();
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
  A.n = static_cast<int>(P.count);
  return A;
}

void reserveParticles(ParticleStore& P, std::size_t capacity) {
  if (capacity <= P.capacity) return;
  for (int a = 0; a < 9; ++a) { P.s[a].resize(capacity); P.t[a].resize(capacity); }
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

// Grows the store to `capacity` entries keeping the persistent state of
// its first `count` entries (SoA, ids, entry states, held speeds); the
// per-step arrays are rewritten by every step.
void growParticles(ParticleStore& P, std::size_t capacity) {
  if (capacity <= P.capacity) return;
  DeviceArray<double> s[9], beta;
  DeviceArray<uint64_t> id;
  DeviceArray<int> state;
  for (int a = 0; a < 9; ++a) s[a].swap(P.s[a]);
  id.swap(P.id);
  state.swap(P.state);
  beta.swap(P.beta);
  reserveParticles(P, capacity);
  const std::size_t n = P.count;
  if (!n) return;
  for (int a = 0; a < 9; ++a)
    hipCheck(hipMemcpy(P.s[a].get(), s[a].get(), n * sizeof(double), hipMemcpyDeviceToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.id.get(), id.get(), n * sizeof(uint64_t), hipMemcpyDeviceToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.state.get(), state.get(), n * sizeof(int), hipMemcpyDeviceToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.beta.get(), beta.get(), n * sizeof(double), hipMemcpyDeviceToDevice), "hipMemcpy");
}

void appendParticles(ParticleStore& P, std::size_t k, const double* x3, const double* u3, const double* q,
                     const double* m, const double* w, const uint64_t* id, const int* state, const double* beta) {
  if (!k) return;
  const std::size_t n = P.count;
  if (n + k > P.capacity) growParticles(P, std::max(n + k, P.capacity + P.capacity / 4 + 1024));
  std::vector<double> col(k);
  for (int a = 0; a < 3; ++a) {
    for (std::size_t i = 0; i < k; ++i) col[i] = x3[3 * i + a];
    hipCheck(hipMemcpy(P.s[a].get() + n, col.data(), k * sizeof(double), hipMemcpyHostToDevice), "hipMemcpy");
    for (std::size_t i = 0; i < k; ++i) col[i] = u3[3 * i + a];
    hipCheck(hipMemcpy(P.s[3 + a].get() + n, col.data(), k * sizeof(double), hipMemcpyHostToDevice), "hipMemcpy");
  }
  const double* scalars[3] = {q, m, w};
  for (int a = 0; a < 3; ++a)
    hipCheck(hipMemcpy(P.s[6 + a].get() + n, scalars[a], k * sizeof(double), hipMemcpyHostToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.id.get() + n, id, k * sizeof(uint64_t), hipMemcpyHostToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.state.get() + n, state, k * sizeof(int), hipMemcpyHostToDevice), "hipMemcpy");
  hipCheck(hipMemcpy(P.beta.get() + n, beta, k * sizeof(double), hipMemcpyHostToDevice), "hipMemcpy");
  P.count = n + k;
  ++P.generation;
}

void raiseParticleErrors(unsigned e) {
  e &= ~kEvtAny;
  if (!e) return;
  if (e & kErrNonfinite) throw std::runtime_error("Nonfinite open coupling orbit");
  if (e & kErrBehindInlet) throw std::runtime_error("Active particle fell behind moving inlet");
  if (e & kErrCarrierBehind) throw std::runtime_error("Current carrier fell behind moving inlet");
  if (e & kErrRemapOutside)
    throw std::runtime_error("Moving-window remap particle crossed a non-adjacent slab or outer boundary");
  if (e & kErrUpstream)
    throw std::runtime_error("An active particle is upstream of the moving window; the inlet guard did not contain its release event");
  if (e & kErrStartInCpml) throw std::out_of_range("Active particle starts inside the non-physical CPML region");
  if (e & kErrStartOutside) throw std::out_of_range("Particle trajectory starts outside the global E/B domain");
  if (e & kErrBeyondExit) throw std::runtime_error("Active particle started beyond trusted moving-window exit");
  if (e & kErrCpmlLocate) throw std::runtime_error("Cannot locate the first particle entry into CPML");
  if (e & kErrExitLocate) throw std::runtime_error("Cannot locate the first particle-domain exit");
  if (e & kErrEndpointOutside) throw std::out_of_range("Particle trajectory endpoint is outside the E/B domain");
  if (e & kErrOrbitOutside) throw std::out_of_range("Quintic active orbit outside domain");
  if (e & kErrMagneticOutside) throw std::out_of_range("Notch magnetic orbit outside domain");
  if (e & kErrMagneticNoDomain) throw std::out_of_range("Active coupling magnetic orbit has no in-domain portion");
  if (e & kErrRootNonphysical) throw std::runtime_error("Nonphysical local mean-gamma root");
  if (e & kErrRootNoConverge) throw std::runtime_error("Local mean-gamma root did not converge");
  if (e & kErrCurrentY) throw std::out_of_range("Transverse current support outside y grid");
  if (e & kErrCurrentX) throw std::out_of_range("Transverse current support outside x grid");
  if (e & kErrCrossings) throw std::runtime_error("Orbit exceeds the device crossing budget");
  if (e & kErrTileHalo) throw std::runtime_error("Particle chord is longer than one cell per axis in one step");
  throw std::runtime_error("Unknown device error");
}

StepArgs stepArgsFor(const CouplingState& C, const aprl_grid_geometry& g, const aprl_cpml_parameters* cp,
                     bool window, const double origin[3], double time, unsigned substeps) {
  StepArgs S{};
  S.time = time;
  S.dt = g.dt;
  S.substeps = static_cast<int>(substeps);
  S.frame = C.frame;
  S.nMagnets = static_cast<int>(C.magnets.size());
  for (int n = 0; n < S.nMagnets; ++n) S.mag[n] = C.magnets[n];
  const double sp[3] = {g.dx, g.dy, g.dz};
  const std::size_t cells[3] = {g.nx, g.ny, g.nz};
  const double eps = std::numeric_limits<double>::epsilon();
  S.cpmlEnabled = 0;
  S.cpmlOrder = cp ? cp->polynomial_order : 0.0;
  for (int a = 0; a < 3; ++a) {
    const double lo = origin[a], hi = origin[a] + static_cast<double>(cells[a]) * sp[a];
    if (2 * C.cpmlCells[a] >= cells[a] && C.cpmlCells[a] > 0)
      throw std::invalid_argument("Particle CPML region must leave a physical interior");
    S.physLo[a] = lo + static_cast<double>(C.cpmlCells[a]) * sp[a];
    S.physHi[a] = hi - static_cast<double>(C.cpmlCells[a]) * sp[a];
    S.cpmlTol[a] = 64.0 * eps * std::max(1.0, std::max(std::abs(lo), std::abs(hi)));
    S.cpmlOuterLo[a] = lo;
    S.cpmlOuterHi[a] = hi;
    S.cpmlCells[a] = static_cast<int>(C.cpmlCells[a]);
    S.cpmlRate[a] = 0.0;
    S.cpmlThick[a] = static_cast<double>(C.cpmlCells[a]) * sp[a];
    if (C.cpmlCells[a]) {
      // EBCPMLParameters::maximumConductivityRate, eb_cpml.cpp:263-281
      S.cpmlEnabled = 1;
      const double order = cp ? cp->polynomial_order : 0.0, reflection = cp ? cp->target_reflection : 0.0;
      if (!(order > 0.0) || !(reflection > 0.0 && reflection < 1.0))
        throw std::invalid_argument("Cannot evaluate an invalid CPML conductivity profile");
      S.cpmlRate[a] = -(order + 1.0) * kC * std::log(reflection) / (2.0 * S.cpmlThick[a]);
    }
    S.outLo[a] = origin[a];
    S.outHi[a] = std::fma(static_cast<double>(cells[a]), sp[a], origin[a]);
    S.outTol[a] = 64.0 * eps * std::max(1.0, std::max(std::abs(S.outLo[a]), std::abs(S.outHi[a])));
    S.extent[a] = static_cast<double>(cells[a]) * sp[a];
    S.posTol[a] = 64.0 * eps * std::max(1.0, std::max(std::abs(origin[a]), S.extent[a]));
  }
  S.hasExit = C.hasExit ? 1 : 0;
  S.window = window ? 1 : 0;
  S.exitLabZ = C.exitLabZ;
  S.hasActivation = C.hasActivation ? 1 : 0;
  S.activationLabZ = C.activationLabZ;
  S.holdTransverse = C.holdTransverse ? 1 : 0;
  return S;
}

int tileKeyBits(int ntiles) {
  const unsigned v = static_cast<unsigned>(ntiles);  // keys 0..ntiles (ntiles: behind the live entries)
  int b = 1;
  while (b < 32 && (v >> b) != 0u) ++b;
  return b;
}

// Stable sort of the particle state by start tile (removed and cropped
// entries last), then the tile ranges and the chunk list (tile order,
// kChunk particles per chunk) in device memory.
static void sortAndChunk(CouplingState& C, ParticleStore& P, const GArgs& G, const SortArgs& K, int ntx, int nty,
                         int ntiles, const DigitCounts& D, unsigned seq, hipStream_t st) {
  FieldState& F = *C.fields;
  const int n = static_cast<int>(P.count);
  ScopedKernel sk(F.profiler, st, "sort");
  const unsigned blocks = ceilDiv(n, 256);
  kTileKeys<<<blocks, 256, 0, st>>>(
      P.s[0].get(), P.s[1].get(), P.s[2].get(), P.state.get(), n, G, ntx, nty, P.key.get(),
      TileRangeArgs{C.tileBegin.get(), C.tileEnd.get(), ntiles, C.tileBound.get()}, K, D);
  launchCheck("tile keys");
  tileSort(P.sortTemp.get(), P.sortTempBytes, P.key.get(), P.keySorted.get(), P.permSorted.get(),
           static_cast<unsigned>(n), tileKeyBits(ntiles), st);
  PermuteArgs A{};
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
  // |scale| = |q| |dx_a| / (dx dy dz dt) < |q| c dt / (dx dy dz dt), with a margin for rounding
  const double perCharge = kC * F.g.dt / (F.g.dx * F.g.dy * F.g.dz * F.g.dt) * (1.0 + 1e-9);
  const TileBoundsArgs T{P.keySorted.get(), n, ntiles, C.tileBegin.get(), C.tileEnd.get(), C.tileBound.get(),
                         perCharge};
  kPermute<<<dim3(blocks, 4), 256, 0, st>>>(A, P.permSorted.get(), n, T);
  launchCheck("permute");
  for (int a = 0; a < 9; ++a) P.s[a].swap(P.t[a]);
  P.id.swap(P.idT);
  P.state.swap(P.stateT);
  P.beta.swap(P.betaT);
  const int rz = C.shape == kShapeQuintic ? Box<kShapeQuintic>::RZ : Box<kShapeBinomial3X>::RZ;
  buildChunkLists(C, st, ntx, nty, ntiles, rz, n, kChunk, C.mailbox.device(), seq);
}

// From the tile ranges of the sorted keys (written by the permute): packed
// chunk, occupied and active counts, their scan, the chunk list and the
// active-tile list (all in tile order).
void buildChunkLists(CouplingState& C, hipStream_t st, int ntx, int nty, int ntiles, int rz, int n, int chunk, unsigned* box,
                     unsigned seq) {
  const int ntz = ntiles / (ntx * nty);
  const unsigned blocks = ceilDiv(ntiles + 1, kScanThreads);
  kTileCounts<<<blocks, kScanThreads, 0, st>>>(C.tileBegin.get(), C.tileEnd.get(), ntx, nty, ntz, rz, chunk,
                                                C.tileCounts.get(), C.tileSums.get(), C.keyActive.get(),
                                                static_cast<int>(ceilDiv(n, 256)), C.error.get() + 4);
  launchCheck("tile counts");
  kChunkList<<<blocks, kScanThreads, 0, st>>>(C.tileBegin.get(), C.tileEnd.get(), C.tileCounts.get(),
                                               C.tileSums.get(), C.tileScan.get(), ntiles, chunk, C.chunks.get(),
                                               C.activeTiles.get(), box, seq, C.error.get());
  launchCheck("chunk list");
}

// Tile arrays sized for ntiles and a chunk list for n particles.
void reserveTileLists(CouplingState& C, hipStream_t st, int ntiles, int n) {
  if (static_cast<unsigned long long>(ntiles) > kMaxTiles)
    throw std::invalid_argument("The grid has more than " + std::to_string(kMaxTiles) + " cell tiles of 8x8x4");
  if (C.tileBegin.size() != static_cast<std::size_t>(ntiles)) {
    C.tileBegin.resize(ntiles);
    C.tileEnd.resize(ntiles);
    C.tileShift.resize(ntiles);
    C.activeTiles.resize(ntiles);
    C.tileBound.resize(ntiles);
    hipCheck(hipMemsetAsync(C.tileBound.get(), 0, static_cast<std::size_t>(ntiles) * sizeof(unsigned long long), st),
             "hipMemsetAsync");
    C.tileCounts.resize(ntiles + 1);
    C.tileScan.resize(ntiles + 1);
    C.tileSums.resize(ceilDiv(ntiles + 1, kScanThreads));
    C.chunkCapacity = 0;
  }
  const std::size_t chunkBound = chunkListBound(ntiles, n);
  if (chunkBound > kMaxChunks)
    throw std::invalid_argument("More than " + std::to_string(kMaxChunks) + " particle chunks in one step");
  if (chunkBound > C.chunkCapacity) {
    // headroom: admissions raise the bound a little in many steps
    const std::size_t capacity = std::min<std::size_t>(chunkBound + chunkBound / 4 + 64, kMaxChunks);
    C.chunks.resize(capacity);
    C.chunkCapacity = capacity;
  }
}

// At most one partial chunk per occupied tile plus the full ones.
std::size_t chunkListBound(int ntiles, int n) {
  return (static_cast<std::size_t>(n) + kChunk - 1) / kChunk +
         std::min<std::size_t>(static_cast<std::size_t>(ntiles), static_cast<std::size_t>(n));
}

void reserveKeyBlocks(CouplingState& C, int n) {
  const std::size_t blocks = ceilDiv(n, 256);
  if (C.keyActive.size() < blocks) C.keyActive.resize(blocks + blocks / 2);
}

void clearStepWords(CouplingState& C, const DigitCounts& D, hipStream_t st) {
  const unsigned words = static_cast<unsigned>(D.words);
  kClearWords<<<std::max(1u, std::min(ceilDiv(words, 1024), 256u)), 256, 0, st>>>(C.error.get(), kErrorWords, D.table,
                                                                                  words);
  launchCheck("clear words");
}

void reserveSortTemp(DeviceArray<unsigned char>& temp, std::size_t& have, std::size_t n) {
  const std::size_t bytes = tileSortBytes(static_cast<unsigned>(n));
  if (bytes <= have) return;
  temp.resize(bytes);
  have = bytes;
}

// A kernel on the step's stream rather than asynchronous copies and an event:
// a copy of a few words took 4 us and a 13 us gap before the E commit behind
// it, two more held up the sort phase, and the waits went through the event.
// 64x64x512, 1e5 particles: 318 -> 309 us a step (quintic 380 -> 369 us), 32x32x256
// with 2e4: 234 -> 217 us.
__global__ void __launch_bounds__(kMaxTrials) kPostTrials(const unsigned* words, unsigned trials, const double* sums,
                                                          unsigned* box, unsigned seq) {
  volatile unsigned* v = box;
  volatile double* d = reinterpret_cast<double*>(reinterpret_cast<unsigned char*>(box) + 2048);
  if (threadIdx.x < trials) v[16 + threadIdx.x] = words[threadIdx.x];
  if (sums && threadIdx.x < 4u) d[threadIdx.x] = sums[threadIdx.x];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) v[1] = seq;
}

void postTrialWords(CouplingState& C, hipStream_t st, unsigned trials, bool residual, unsigned seq) {
  kPostTrials<<<1, kMaxTrials, 0, st>>>(C.error.get() + kTrialWord, trials, residual ? C.reduceOut.get() : nullptr,
                                        C.mailbox.device(), seq);
  launchCheck("post trials");
}

void reduceChunkStats(hipStream_t st, const double* in, int chunks, double* out) {
  kReduceBlocks<<<1, 256, 0, st>>>(in, chunks, out, nullptr, 0u, PicardWords{nullptr, 0u, nullptr, 0u});
  launchCheck("chunk stats");
}

TileBoxes reserveStepBuffers(CouplingState& C, std::size_t boxWords, std::size_t rawWords, unsigned nChunks,
                             unsigned occupied, hipStream_t st) {
  const std::size_t extra = nChunks - occupied;
  const std::size_t need = boxWords * occupied, raw = rawWords * std::min<std::size_t>(extra, occupied);
  // at least 16 MiB: of 8 to 10 MB, in a process that had freed memory before,
  // an allocation took 0.5 ms instead of 0.04 ms, a seventh of a small grid's
  // first steps
  if (need > C.boxes.size()) C.boxes.resize(std::max<std::size_t>(need + need / 2, 1u << 21));
  if (raw > C.rawBoxes.size()) {
    // at least 64 boxes, 1 to 2 MB: half of a few is soon used up
    const std::size_t n = std::max(raw + raw / 2, 64 * rawWords);
    C.rawBoxes.resize(n);
    hipCheck(hipMemsetAsync(C.rawBoxes.get(), 0, n * sizeof(long long), st), "hipMemsetAsync");
  }
  const std::size_t blocks = 4 * static_cast<std::size_t>(std::max(1u, nChunks));
  if (C.reduceBlocks.size() < blocks) C.reduceBlocks.resize(blocks + blocks / 2);
  return TileBoxes{C.boxes.get(), C.rawBoxes.get(), extra <= occupied ? 1 : 0};
}

void reserveCouplingWords(CouplingState& C, hipStream_t st) {
  if (C.error.size() < static_cast<std::size_t>(kErrorWords)) C.error.resize(kErrorWords);
  if (C.reduceOut.size() < 4) C.reduceOut.resize(4);

  if (!C.counterQ.size()) {
    C.counterQ.resize(kCounterSlots);
    C.counterN.resize(kCounterSlots);
    hipCheck(hipMemsetAsync(C.counterQ.get(), 0, kCounterSlots * sizeof(double), st), "hipMemsetAsync");
    hipCheck(hipMemsetAsync(C.counterN.get(), 0, kCounterSlots * sizeof(unsigned long long), st), "hipMemsetAsync");
  }
}

namespace {
// Block partials of the counters, added in block order to the cumulative
// counters; a null flag always adds, otherwise only when it carries kEvtAny.
__global__ void __launch_bounds__(64) kCounterTotals(const double* blockQ, const unsigned* blockN, int blocks,
                                                     const unsigned* flag, double* q, unsigned long long* count) {
  if (flag && !(*flag & kEvtAny)) return;
  const int t = static_cast<int>(threadIdx.x);
  if (t >= kCounterSlots) return;
  double acc = 0.0;
  unsigned long long cnt = 0;
  for (int b = 0; b < blocks; ++b) {
    acc += blockQ[b * kCounterSlots + t];
    cnt += blockN[b * kCounterSlots + t];
  }
  q[t] += acc;
  count[t] += cnt;
}

void reserveBlockCounters(CouplingState& C, int blocks) {
  const std::size_t need = static_cast<std::size_t>(std::max(blocks, 1)) * kCounterSlots;
  if (C.blockQ.size() < need) {
    C.blockQ.resize(need + need / 2);
    C.blockN.resize(need + need / 2);
  }
}
}  // namespace

void commitEvents(CouplingState& C, hipStream_t st, int n, const int* evt, int* state, void* w, const void* q,
                  void* wend, unsigned* removed, const unsigned* trialWord, bool fp32) {
  if (n <= 0) return;
  const int blocks = static_cast<int>(ceilDiv(n, kEventBlock));
  reserveBlockCounters(C, blocks);
  if (fp32)
    kCommitEvents<float><<<blocks, kEventBlock, 0, st>>>(n, evt, state, static_cast<float*>(w),
                                                          static_cast<const float*>(q), static_cast<float*>(wend),
                                                          removed, trialWord, C.blockQ.get(), C.blockN.get());
  else
    kCommitEvents<double><<<blocks, kEventBlock, 0, st>>>(n, evt, state, static_cast<double*>(w),
                                                           static_cast<const double*>(q), static_cast<double*>(wend),
                                                           removed, trialWord, C.blockQ.get(), C.blockN.get());
  kCounterTotals<<<1, 64, 0, st>>>(C.blockQ.get(), C.blockN.get(), blocks, trialWord, C.counterQ.get(),
                                   C.counterN.get());
  launchCheck("commit events");
}

void cropCounters(CouplingState& C, hipStream_t st, int lo, int n, const int* state, const void* q, const void* w,
                  bool fp32) {
  if (n <= lo) return;
  const int blocks = static_cast<int>(ceilDiv(n - lo, kEventBlock));
  reserveBlockCounters(C, blocks);
  if (fp32)
    kCropCounters<float><<<blocks, kEventBlock, 0, st>>>(lo, n, state, static_cast<const float*>(q),
                                                          static_cast<const float*>(w), C.blockQ.get(), C.blockN.get());
  else
    kCropCounters<double><<<blocks, kEventBlock, 0, st>>>(lo, n, state, static_cast<const double*>(q),
                                                           static_cast<const double*>(w), C.blockQ.get(),
                                                           C.blockN.get());
  kCounterTotals<<<1, 64, 0, st>>>(C.blockQ.get(), C.blockN.get(), blocks, nullptr, C.counterQ.get(),
                                   C.counterN.get());
  launchCheck("crop counters");
}

std::size_t liveEntries(std::size_t count, const DeviceArray<unsigned>& removed, hipStream_t st) {
  if (!count || !removed.size()) return count;
  unsigned r = 0;
  hipCheck(hipStreamSynchronize(st), "hipStreamSynchronize");
  hipCheck(hipMemcpy(&r, removed.get(), sizeof(unsigned), hipMemcpyDeviceToHost), "hipMemcpy");
  return count - std::min<std::size_t>(count, r);
}

// The step's sort phase on stream ss: tile lists and readback words
// sized, error words cleared, then (with particles) the stable tile sort,
// the state permute and the chunk lists, whose totals are posted to the
// mailbox under the returned sequence number.
static unsigned sortPhase(CouplingState& C, ParticleStore& P, const double origin[3], hipStream_t ss) {
  FieldState& F = *C.fields;
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
  K.lowZ = origin[2];
  K.upZ = std::fma(static_cast<double>(F.g.nz), F.g.dz, origin[2]);
  K.dz = F.g.dz;
  K.words = C.error.get();
  K.removed = P.removed.get();
  reserveKeyBlocks(C, n);
  K.blockActive = C.keyActive.get();
  const unsigned seq = C.mailbox.next(0);
  sortAndChunk(C, P, gatherArgs(C, F, origin), K, ntx, nty, ntiles, D, seq, ss);
  return seq;
}

bool preparedFor(const CouplingState& C, const void* store, std::uint64_t generation, std::size_t count,
                 const double origin[3]) {
  const auto& R = C.prepared;
  return R.valid && R.store == store && R.generation == generation && R.count == count && R.origin[0] == origin[0] &&
         R.origin[1] == origin[1] && R.origin[2] == origin[2];
}

// Starts the next step's sort phase on the coupling's sort stream after
// everything already enqueued on the grid's stream, so that it overlaps
// the field work enqueued after it (clear, window begin, magnetic update).
void prepareStep(CouplingState& C, ParticleStore& P, const double origin[3]) {
  FieldState& F = *C.fields;
  if (C.prepared.valid) throw std::logic_error("A prepared coupling step is already pending");
  hipStream_t ss = C.sortStream.get();
  // J of the last deposit is cleared through that step's active-tile list,
  // which this sort rewrites: clear it now, ahead of the sort (every step
  // starts from J = 0, and the step's own clear then finds nothing to do)
  if (F.footprint.valid && !F.currentZero) launchClearCurrent(F);
  hipCheck(hipEventRecord(C.prepareStart.get(), F.stream), "hipEventRecord");
  hipCheck(hipStreamWaitEvent(ss, C.prepareStart.get(), 0), "hipStreamWaitEvent");
  const unsigned seq = sortPhase(C, P, origin, ss);
  hipCheck(hipEventRecord(C.sortReady.get(), ss), "hipEventRecord");
  auto& R = C.prepared;
  R.valid = true;
  R.store = &P;
  R.generation = P.generation;
  R.count = P.count;
  for (int a = 0; a < 3; ++a) R.origin[a] = origin[a];
  R.seq = seq;
}

// Per-step state of a plain FP64 step between its two phases.
struct PlainStepContext {
  bool pending = false;
  int n = 0, ntx = 0, nty = 0, ntz = 0;
  unsigned nChunks = 0, nActive = 0, occupied = 0, activeEntries = 0;
  unsigned enqueued = 0;       // Picard trials enqueued so far
  unsigned checkedTrials = 0;  // trial words read back so far
  unsigned postSeq = 0;        // mailbox sequence of the last posted trial
  unsigned commitAfter = 0;    // trials ahead of the gated E commit (0: none enqueued)
  bool quintic = false;
  double origin[3] = {0.0, 0.0, 0.0};
  TileBoxes boxes{};
  PArgs A{};
  GArgs G{};
  StepArgs S{};
};

namespace {

// Enqueue Picard trials [first, last) of the step; the last one posts its
// residual, the stop word and the unchecked trial words to the mailbox.
// Every trial runs behind the device stop word: once a trial has converged
// (or failed), the kernels of the later ones return at once, so trials can
// be enqueued ahead of the convergence decision.
void enqueueTrials(CouplingState& C, PlainStepContext& X, unsigned first, unsigned last) {
  FieldState& F = *C.fields;
  hipStream_t st = F.stream;
  const int n = X.n, ntx = X.ntx, nty = X.nty, ntz = X.ntz;
  const unsigned nChunks = X.nChunks, nActive = X.nActive;
  const bool quintic = X.quintic;
  PArgs& A = X.A;
  const GArgs& G = X.G;
  const StepArgs& S = X.S;
  unsigned* const stop = C.error.get() + kStopWord;
  for (unsigned trial = first; trial < last; ++trial) {
    unsigned* errT = C.error.get() + kTrialWord + trial;
    if (nChunks && trial == 0) {
      // The first trial pushes against the preview with J cleared
      // (simulation_source_coupling.cpp:43).
      GArgs G0 = G;
      for (int a = 0; a < 3; ++a) G0.esum[a] = C.esum0[a].get();
      G0.stop = nullptr;
      ScopedKernel sk(F.profiler, st, "gather");
      if (quintic)
        kGatherChunks<0, kShapeQuintic><<<nChunks, kChunk, 0, st>>>(A, G0, S, C.chunks.get(), ntx, nty, F.g.dt,
                                                                         nullptr, errT);
      else
        kGatherChunks<0, kShapeBinomial3X><<<nChunks, kChunk, 0, st>>>(A, G0, S, C.chunks.get(), ntx, nty, F.g.dt,
                                                                            nullptr, errT);
      launchCheck("gather");
    }
    if (n) {
      ScopedKernel sk(F.profiler, st, "push");
      kPush<<<ceilDiv(n, 128), 128, 0, st>>>(A, G, S, errT);
      launchCheck("push");
    }
    if (nChunks) {
      {
        ScopedKernel sk(F.profiler, st, "deposit");
        if (quintic)
          kDeposit<kShapeQuintic><<<nChunks, kChunk, 0, st>>>(
              A, G, S, C.chunks.get(), C.tileBegin.get(), C.tileEnd.get(), C.tileScan.get(), ntx, nty,
              X.boxes, C.tileShift.get(), errT);
        else
          kDeposit<kShapeBinomial3X><<<nChunks, kChunk, 0, st>>>(
              A, G, S, C.chunks.get(), C.tileBegin.get(), C.tileEnd.get(), C.tileScan.get(), ntx, nty,
              X.boxes, C.tileShift.get(), errT);
        launchCheck("deposit");
        foldTiles(C, X.boxes, F.g, nChunks, X.occupied, stop, st);
      }
      {
        ScopedKernel sk(F.profiler, st, "reduce_current");
        // with active particles the first trial never converges
        const int writeJ = trial > 0 || !X.activeEntries || C.refCurrent;
        if (quintic)
          kReduceCurrent<kShapeQuintic><<<nActive, 256, 0, st>>>(F.base(6), F.base(7), F.base(8), G,
                                                                 C.activeTiles.get(), C.tileScan.get(),
                                                                 C.tileShift.get(), X.boxes.boxes, ntx, nty, ntz,
                                                                 writeJ);
        else
          kReduceCurrent<kShapeBinomial3X><<<nActive, 256, 0, st>>>(F.base(6), F.base(7), F.base(8), G,
                                                                    C.activeTiles.get(), C.tileScan.get(),
                                                                    C.tileShift.get(), X.boxes.boxes, ntx, nty,
                                                                    ntz, writeJ);
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
    }
    // TransverseReferenceCurrent::apply after the trial's deposit
    // (simulation_source_coupling.cpp:44)
    referenceCurrentTrial(C, F, C.esum[2].get(), C.esum0[2].get(), true, nChunks > 0, ntx, nty, ntz, stop);
    const bool post = trial + 1 == last;
    if (post) X.postSeq = C.mailbox.next(1);
    const PicardWords W{stop, trial, C.error.get() + kTrialWord, X.checkedTrials};
    unsigned* const box = post ? C.mailbox.device() : nullptr;
    const unsigned seq = post ? X.postSeq : 0u;
    if (nChunks) {
      ScopedKernel sk(F.profiler, st, "residual");
      if (quintic)
        kGatherChunks<1, kShapeQuintic><<<nChunks, kChunk, 0, st>>>(A, G, S, C.chunks.get(), ntx, nty, F.g.dt,
                                                                         C.reduceBlocks.get(), errT);
      else
        kGatherChunks<1, kShapeBinomial3X><<<nChunks, kChunk, 0, st>>>(A, G, S, C.chunks.get(), ntx, nty, F.g.dt,
                                                                            C.reduceBlocks.get(), errT);
    }
    // a separate launch: folding it into the gather's last workgroup needs
    // a device-scope fence in every workgroup (the XCDs' L2s write back),
    // which was measured to make the gather three times slower
    kReduceBlocks<<<1, 256, 0, st>>>(C.reduceBlocks.get(), static_cast<int>(nChunks), C.reduceOut.get(), box, seq, W);
    launchCheck("residual");
    // The next trial pushes with the fields this residual gathered.
    for (int a = 0; a < 6; ++a) std::swap(A.fin[a], A.fout[a]);
  }
  X.enqueued = last;
}

}  // namespace

void plainStepBegin(CouplingState& C, ParticleStore& P, const double origin[3], double time, unsigned substeps) {
  FieldState& F = *C.fields;
  if (!C.plain) C.plain = std::make_shared<PlainStepContext>();
  PlainStepContext& X = *C.plain;
  if (X.pending) throw std::logic_error("The previous coupling step was not finished");
  if (F.window && F.phase != 2) throw std::logic_error("Moving-window electric phase mismatch");
  if (F.window && !F.inletSet) throw std::logic_error("Moving-window inlet planes were not supplied");
  if (substeps == 0) throw std::invalid_argument("Particle substeps must be positive");
  int n = static_cast<int>(P.count);
  hipStream_t st = F.stream;
  // J is zero at the start of every step (simulation.cpp:518); the tile
  // reduction below rewrites only the neighbourhood of occupied tiles.
  launchClearCurrent(F);
  for (int a = 0; a < 3; ++a)
    if (C.esum0[a].size() != F.compSize(a)) {
      C.esum0[a].resize(F.compSize(a));
      C.esum[a].resize(F.compSize(a));
    }

  const int ntx = static_cast<int>((F.g.nx + kTileX - 1) / kTileX);
  const int nty = static_cast<int>((F.g.ny + kTileY - 1) / kTileY);
  const int ntz = static_cast<int>((F.g.nz + kTileZ - 1) / kTileZ);
  const int ntiles = ntx * nty * ntz;
  const std::size_t chunkBound = chunkListBound(ntiles, n);
  // Readbacks arrive in the mailbox: the scan total (chunks, active tiles)
  // and the sort-phase words at words 8..14 (flag 0); the posting trial's
  // residual sums (doubles), the stop word and the trial error words from
  // word 15 (flag 1).
  unsigned sortSeq = 0;
  if (preparedFor(C, &P, P.generation, P.count, origin)) {
    hipCheck(hipStreamWaitEvent(st, C.sortReady.get(), 0), "hipStreamWaitEvent");
    sortSeq = C.prepared.seq;
  } else {
    if (C.prepared.valid) hipCheck(hipStreamWaitEvent(st, C.sortReady.get(), 0), "hipStreamWaitEvent");
    sortSeq = sortPhase(C, P, origin, st);
  }
  C.prepared.valid = false;
  // Zero-current preview E* (MovingWindowFields::previewElectricBoundary),
  // kept as E* + E^n; it runs while the host waits for the chunk count. The
  // sums are read only on the nodes of active tiles (gathers stage the boxes
  // of occupied tiles; the reduction rewrites active tiles).
  double* const sums[3] = {C.esum0[0].get(), C.esum0[1].get(), C.esum0[2].get()};
  if (n)
    launchElectricPreviewTiles(F, F.ptrs(), sums, F.window ? F.inletPlane[0] : nullptr,
                               F.window ? F.inletPlane[1] : nullptr, C.activeTiles.get(), C.tileScan.get() + ntiles,
                               TileGrid{ntx, nty, ntz, kTileX, kTileY, kTileZ});
  unsigned nChunks = 0, nActive = 0, occupiedTiles = 0, activeEntries = 0;
  if (n) {
    C.mailbox.wait(0, sortSeq, st);
    const unsigned* box = C.mailbox.host();
    nChunks = box[8];
    nActive = box[9];
    occupiedTiles = box[11];
    // finishMovingWindowStep's checks of the entries, applied to this origin
    raiseParticleErrors(box[10]);
    activeEntries = box[14];
    const int behind = static_cast<int>(box[12]);
    if (box[13]) cropCounters(C, st, n - behind, n, P.state.get(), P.s[6].get(), P.s[8].get(), false);
    n -= behind;  // removed and cropped entries now trail the live ones
    P.count = static_cast<std::size_t>(n);
    if (nChunks > chunkBound) throw std::logic_error("Chunk list exceeds its bound");
  }
  const bool quintic = C.shape == kShapeQuintic;
  const int boxN = quintic ? boxNodes<kShapeQuintic>() : boxNodes<kShapeBinomial3X>();
  const int rawN = quintic ? rawNodes<kShapeQuintic>() : rawNodes<kShapeBinomial3X>();
  X.boxes = reserveStepBuffers(C, 3 * static_cast<std::size_t>(boxN), 3 * static_cast<std::size_t>(rawN), nChunks,
                               occupiedTiles, st);

  X.S = stepArgsFor(C, F.g, F.hasCpml ? &F.cpml : nullptr, F.window, origin, time, substeps);
  X.A = particleArgs(P);
  X.A.scaleDen = F.g.dx * F.g.dy * F.g.dz * F.g.dt;
  X.A.tileBound = C.tileBound.get();
  X.G = gatherArgs(C, F, origin);
  X.G.stop = C.error.get() + kStopWord;
  X.n = n;
  X.ntx = ntx;
  X.nty = nty;
  X.ntz = ntz;
  X.nChunks = nChunks;
  X.nActive = nActive;
  X.occupied = occupiedTiles;
  X.activeEntries = activeEntries;
  X.quintic = quintic;
  X.enqueued = 0;
  X.checkedTrials = 0;
  for (int a = 0; a < 3; ++a) X.origin[a] = origin[a];
  X.pending = true;
  // With active particles the convergence test needs at least two trials
  // (simulation_source_coupling.cpp:50); the first batch is the last
  // step's trial count.
  const unsigned batch = C.picardFixed ? C.picardFixed
                                       : std::min<unsigned>(kMaxTrials, std::max(C.picardBatch, activeEntries ? 2u : 1u));
  enqueueTrials(C, X, 0, batch);
  // commitConservativeElectric enqueued behind the batch, gated on the stop
  // word: it runs when a trial of the batch has converged, so the device
  // does not wait for the host to read the decision. (The energy ledger's
  // commit, several launches, stays after the decision, and so does the
  // commit while its workgroup size is being tuned: a skipped launch would
  // be a false sample.)
  X.commitAfter = 0;
  if (!(F.window && F.ledger.enabled) && autotuneSettled(shapeKey("electric", F.g, sizeof(double)))) {
    launchElectric(F, F.ptrs(), F.inletPlane[0], F.inletPlane[1], C.error.get() + kStopWord);
    X.commitAfter = X.enqueued;
  }
}

void plainStepFinish(CouplingState& C, ParticleStore& P, aprl_step_report* report) {
  if (!C.plain || !C.plain->pending) throw std::logic_error("Coupling step phase mismatch");
  PlainStepContext& X = *C.plain;
  X.pending = false;
  FieldState& F = *C.fields;
  hipStream_t st = F.stream;
  unsigned iterations = 0, lastWord = 0, stop = 0;
  double force = 0., work = 0.;
  for (;;) {
    C.mailbox.wait(1, X.postSeq, st);
    const unsigned* box = C.mailbox.host();
    const double* sums = C.mailbox.hostDoubles();
    stop = box[15];
    const unsigned ran = stop ? (stop & ~kStopError) : X.enqueued;
    // device errors in trial order, as the reference raises them
    for (unsigned t = X.checkedTrials; t < ran; ++t) raiseParticleErrors(box[16 + t - X.checkedTrials]);
    if (ran) lastWord = box[16 + ran - 1 - X.checkedTrials];
    X.checkedTrials = X.enqueued;
    iterations = ran;
    force = sums[0];
    work = sums[3] == 0. ? 0. : (sums[2] > 0. ? sums[1] / sums[2] : sums[1]);
    if (stop || X.enqueued == static_cast<unsigned>(kMaxTrials)) break;
    // not converged within the batch: one more trial at a time
    enqueueTrials(C, X, X.enqueued, X.enqueued + 1);
  }
  if (!stop) {
    std::string m = "Conservative source coupling failed: force=" + std::to_string(force) +
                    " work=" + std::to_string(work) + " iterations=" + std::to_string(iterations);
    throw std::runtime_error(m);
  }
  C.picardBatch = iterations;
  // commitConservativeElectric: E^n + curl B - dt/eps0 J, then the committed
  // CPML-E (history advance), PEC and inlet overwrite; done already by the
  // gated commit when the converged trial was ahead of it
  const bool gatedRan = X.commitAfter && iterations <= X.commitAfter && !(stop & kStopError);
  if (!gatedRan) {
    if (F.window) windowCommitElectric(F, F.ptrs());
    else launchElectric(F, F.ptrs(), F.inletPlane[0], F.inletPlane[1]);
  }
  if (F.window) F.phase = 3;
  // Boundary events of the converged trial: carriers, removals, counters.
  if (lastWord & kEvtAny)
    commitEvents(C, st, X.n, P.evt.get(), P.state.get(), P.s[8].get(), P.s[6].get(), P.wend.get(), P.removed.get(),
                 C.error.get() + kTrialWord + (iterations - 1), false);
  // The trial end state becomes the particle state; the start positions
  // stay in the end arrays for the step diagnostics.
  for (int a = 0; a < 6; ++a) P.s[a].swap(P.end[a]);
  C.lastStep.valid = true;
  C.lastStep.store = &P;
  C.lastStep.generation = P.generation;
  for (int a = 0; a < 3; ++a) C.lastStep.origin[a] = X.origin[a];
  if (report) {
    report->iterations = iterations;
    report->force = force;
    report->work = work;
    report->tiles = X.occupied;
    report->chunks = X.nChunks;
    report->active_tiles = X.nActive;
  }
}

void couplingStep(CouplingState& C, ParticleStore& P, const double origin[3], double time, unsigned substeps,
                  aprl_step_report* report) {
  plainStepBegin(C, P, origin, time, substeps);
  plainStepFinish(C, P, report);
}

}  // namespace aprl_gpu
