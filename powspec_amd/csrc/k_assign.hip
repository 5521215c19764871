// k_assign.hip -- NGP/CIC/TSC/PCS mass assignment with grid interlacing on
// gfx950, replacing the reference's per-particle `omp atomic` scatter
// (src/genr_mesh.c:50-412) and its zero/subtract/shift passes
// (src/genr_mesh.c:590-602, 793-858).
//
// Design:
//  1. count:   per particle, the FP64 cell coordinate decides the base cell of
//              the window on the plain grid (same operation order as the
//              reference, contraction off) and the half-cell-shifted grid's
//              offset from it; the union window is mapped to the 1..8 mesh
//              tiles it touches and each tile's counter, in an LDS window of
//              counters per workgroup, is incremented.
//  2. scan:    exclusive prefix sum of the tile counters.
//  3. fill:    each (particle, tile) pair is written as a 24-byte record of
//              cells relative to the tile.
//  4. deposit: one workgroup per tile and grid accumulates the tile's records
//              into an LDS copy of the tile (fixed-point integer LDS atomics)
//              and writes the tile to HBM once with coalesced row stores
//              (tiles of whole z rows: both grids, and their z transform).
//              Every mesh cell is written exactly once: no zeroing pass, no
//              global atomics.
// Surveys assign data and randoms into the same tiles with weights w and
// -alpha*w, which fuses the data-minus-random subtraction
// (src/genr_mesh.c:802-806, 841-845).
#include "psh_internal.h"
#include "fft_core.h"

#include <algorithm>
#include <type_traits>

namespace {

// A particle as one of its tiles sees it: cells relative to the tile's first
// (a window that begins in the neighbouring tile before it has negative
// ones), so the deposit needs neither the tile's place nor the periodic wrap.
constexpr int kRecBias = 8;   // added to the local cells, which start at -W
struct __align__(8) Rec {
  float f[3];      // window fraction on the plain grid, per axis
  float w;         // particle weight times the catalogue scale
  uint32_t bxy;    // biased local base cell x | y << 16 (plain grid)
  uint32_t bz;     // biased local base cell z | delta bits (shifted grid) << 16
};
static_assert(sizeof(Rec) == 24, "record layout");

using DevPart = PshDevPart;

constexpr int kFewParts = 8;   // part tables passed as kernel arguments

// Periodic wrap into [0, Ng).  Bases and window ends are at most a window
// (or a grid) away from [0, Ng), so one compare settles nearly every call;
// the remainder covers coordinates further out.
__device__ __forceinline__ int wrap(int c, int Ng) {
  if ((unsigned)c < (unsigned)Ng) return c;
  const int r = c % Ng;
  return r < 0 ? r + Ng : r;
}

// a / L correctly rounded, rL being 1 / L rounded: one Newton step brings
// a rL within an ulp, and the step after that rounds correctly (Markstein's
// theorem on quotients from a correctly rounded reciprocal).  Five FP64
// operations where the compiler's division takes about a dozen, several of
// them at a quarter of the rate.  Finite a and L away from overflow, as grid
// coordinates are; an infinite a gives NaN, and such a particle fails the box
// check (boxes) or leaves no valid box (surveys).
__host__ __device__ __forceinline__ double div_rn(double a, double L, double rL) {
  double q = a * rL;
  q = __builtin_fma(__builtin_fma(-q, L, a), rL, q);
  return __builtin_fma(__builtin_fma(-q, L, a), rL, q);
}

// Base cell (leftmost window cell, unwrapped) and window fraction of a grid
// coordinate x >= 0, following src/genr_mesh.c:57-66 (NGP), 94-104 (CIC),
// 152-172 (TSC), 256-263 (PCS).  The fraction is d = x - (int)x for CIC/PCS
// and the signed offset from the middle node for TSC.
template <int SCHEME>
__device__ __forceinline__ void axis_base(double x, int &b, double &d) {
  const int x0 = (int)x;
  d = x - x0;
  if (SCHEME == 0) {
    b = (d >= 0.5) ? x0 + 1 : x0;
  } else if (SCHEME == 1) {
    b = x0;
  } else if (SCHEME == 2) {
    b = (d < 0.5) ? x0 - 1 : x0;
    if (!(d < 0.5)) d -= 1;
  } else {
    b = x0 - 1;
  }
}

// Cells of a particle along one axis: plain-grid base wrapped into [0, Ng),
// window fraction, and the shifted grid's base minus the plain one (mod Ng),
// 0 or 1.  The shifted grid uses the reference's periodic shift
// (src/genr_mesh.c:595-600: x >= smin + L -> x - L) before the coordinate
// (x - smin) * Ng / L, which is the plain one plus 1/2 up to rounding: the
// offset follows from the plain fraction unless that lies within kShiftEps
// of a value where the offset changes; then (and where g.shift_exact says
// that the box corner's rounding may exceed kShiftEps cells) the shifted
// coordinate is formed as the reference forms it.
constexpr float kShiftEps = 1e-6f;

template <int SCHEME, bool IL>
__device__ __forceinline__ void axis_cells(double r, const PshAssignGeom &g, int a, int &b,
                                           float &f, int &delta) {
#pragma clang fp contract(off)
  const double Ngd = (double)g.Ng;
  int bu;
  double d;
  axis_base<SCHEME>(div_rn((r - g.bmin[a]) * Ngd, g.L[a], g.rL[a]), bu, d);
  b = wrap(bu, g.Ng);
  const float ff = (float)d;
  f = SCHEME == 0 ? 0.f : ff;
  delta = 0;
  if (IL) {
    // NGP: 1 below the half cell; CIC, PCS: 1 from the half cell on; TSC
    // (signed fraction): 1 for the fractions below the half cell, d >= 0
    bool sure;
    if (SCHEME == 0) {
      delta = ff < 0.5f;
      sure = fabsf(ff - 0.5f) > kShiftEps && ff > kShiftEps && ff < 1.f - kShiftEps;
    } else if (SCHEME == 2) {
      delta = ff >= 0.f;
      sure = fabsf(ff) > kShiftEps && fabsf(ff) < 0.5f - kShiftEps;
    } else {
      delta = ff >= 0.5f;
      sure = fabsf(ff - 0.5f) > kShiftEps;
    }
    if (g.shift_exact || !sure) {
      double p = r;
      if (p >= g.smin[a] + g.L[a]) p -= g.L[a];
      int bs;
      double ds;
      axis_base<SCHEME>(div_rn((p - g.smin[a]) * Ngd, g.L[a], g.rL[a]), bs, ds);
      delta = wrap(bs - bu, g.Ng);
    }
  }
}

__device__ __forceinline__ int find_part(const DevPart *parts, int nparts,
                                         size_t gi) {
  int lo = 0, hi = nparts - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (parts[mid].start <= gi) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// One particle as loaded: position and weight, its part's weight scale and
// destination mock.
struct Loaded {
  double r[4];
  float wscale;
  int mock;
};

// A part descriptor held in scalar registers (the part of a workgroup's
// first particle).
struct UPart {
  const double *xyzw;
  size_t start, n;
  float wscale;
  int mock;
};

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// The part containing particle `gi0`; every lane passes the same gi0.
__device__ __forceinline__ UPart uniform_part(const DevPart *parts, int nparts, size_t gi0) {
  const DevPart &P = parts[find_part(parts, nparts, gi0)];
  UPart u;
  u.xyzw = reinterpret_cast<const double *>(uniform64(reinterpret_cast<uint64_t>(P.xyzw)));
  u.start = uniform64(P.start);
  u.n = uniform64(P.n);
  u.wscale = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(P.wscale)));
  u.mock = __builtin_amdgcn_readfirstlane(P.mock);
  return u;
}

typedef __attribute__((address_space(1))) const double gdouble;

// Load particle gi (zeros when !live).  P0 is the part the caller expects gi
// to lie in (chunks rarely cross part boundaries), so the table search runs
// only for particles outside it; callers keep the next particle's loads in
// flight while they process the current one.
__device__ __forceinline__ Loaded load_particle(const DevPart *parts, int nparts, UPart P0,
                                                size_t gi, bool live) {
  Loaded L;
  L.r[0] = L.r[1] = L.r[2] = L.r[3] = 0.0;
  L.wscale = 0.f;
  L.mock = 0;
  if (!live) return L;
  const double *px = P0.xyzw;
  size_t ps = P0.start;
  float pw = P0.wscale;
  int pm = P0.mock;
  if (gi < P0.start || gi - P0.start >= P0.n) {
    const int q = find_part(parts, nparts, gi);
    px = parts[q].xyzw;
    ps = parts[q].start;
    pw = parts[q].wscale;
    pm = parts[q].mock;
  }
  L.wscale = pw;
  L.mock = pm;
  const gdouble *g = (const gdouble *)(px + 4 * (gi - ps));   // device memory
  L.r[0] = g[0];
  L.r[1] = g[1];
  L.r[2] = g[2];
  L.r[3] = g[3];
  return L;
}

// The tiles a particle's windows meet: the tile of its plain base, and per
// axis the offset of the tile of the union window's last cell (0: the same
// tile).  A window plus the shifted grid's cell meets at most two tiles per
// axis, so combination k (bit 0: z, 1: y, 2: x) is a tile of its own when
// its axes all have a second tile.
struct PartTiles {
  int t0;
  int off[3];   // x, y, z
  // the record as tile k sees it: a second tile along an axis lies the
  // tile's extent after the first
  __device__ __forceinline__ Rec record(Rec r, const PshAssignGeom &g, int k) const {
    if (k & 4) r.bxy -= (uint32_t)g.tile[0];
    if (k & 2) r.bxy -= (uint32_t)g.tile[1] << 16;
    if (k & 1) r.bz -= (uint32_t)g.tile[2];
    return r;
  }
  __device__ __forceinline__ bool has(int k) const {
    return (!(k & 4) || off[0]) && (!(k & 2) || off[1]) && (!(k & 1) || off[2]);
  }
  __device__ __forceinline__ uint32_t tile(int k) const {
    return (uint32_t)(t0 + ((k & 4) ? off[0] : 0) + ((k & 2) ? off[1] : 0) +
                      ((k & 1) ? off[2] : 0));
  }
};

// Tiles (mock-local indices) touched by a particle rr = (x, y, z, w) and its
// record as the first of them sees it.  Returns false (and sets flag bit 2) when the shifted grid's base
// is inconsistent.  With CHECK and g.check_box, a coordinate outside
// [bmin, bmin + L) (bmin = 0 for simulation boxes) sets flag bit 4: the box
// check of simulation catalogues (src/genr_mesh.c:517-533) folded into the
// count pass, which reads every particle anyway (NaN passes, as it passes
// the reference's min/max comparisons).
template <int SCHEME, bool IL, bool CHECK>
__device__ __forceinline__ bool particle_tiles(const PshAssignGeom &g, const double *rr,
                                               float wscale, PartTiles &pt, Rec &rec,
                                               int *flags) {
  constexpr int W = SCHEME + 1;
  if (CHECK && g.check_box) {
    bool bad = false;
#pragma unroll
    for (int a = 0; a < 3; a++) bad |= (rr[a] < g.bmin[a]) || (rr[a] >= g.bmin[a] + g.L[a]);
    if (bad) atomicOr(flags, 4);
  }
  int b[3], dl[3];
#pragma unroll
  for (int a = 0; a < 3; a++) axis_cells<SCHEME, IL>(rr[a], g, a, b[a], rec.f[a], dl[a]);
  if (IL && (dl[0] | dl[1] | dl[2]) > 1) {
    atomicOr(flags, 2);
    return false;
  }
  int t[3], o[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    t[a] = b[a] >> g.tile_shift[a];
    o[a] = (wrap(b[a] + W - 1 + dl[a], g.Ng) >> g.tile_shift[a]) - t[a];
  }
  pt.t0 = (t[0] * g.ntile[1] + t[1]) * g.ntile[2] + t[2];
  pt.off[0] = o[0] * g.ntile[1] * g.ntile[2];
  pt.off[1] = o[1] * g.ntile[2];
  pt.off[2] = o[2];
  rec.w = (float)rr[3] * wscale;
#pragma unroll
  for (int a = 0; a < 3; a++) b[a] = (b[a] & (g.tile[a] - 1)) + kRecBias;
  rec.bxy = (uint32_t)b[0] | ((uint32_t)b[1] << 16);
  rec.bz = (uint32_t)b[2] | ((uint32_t)(dl[0] | (dl[1] << 1) | (dl[2] << 2)) << 16);
  return true;
}

// Largest |weight| of a launch, for the fixed-point scale of the deposit
// (flags[1] holds the bits of a non-negative float).  The plain read skips
// the atomic where the maximum is already known: one address takes every
// wave's, and waves of equal weights would queue there.
__device__ __forceinline__ void publish_wmax(float wmax, int *flags) {
  for (int o = 32; o > 0; o >>= 1) wmax = fmaxf(wmax, __shfl_xor(wmax, o));
  unsigned *p = reinterpret_cast<unsigned *>(flags) + 1;
  const unsigned w = __float_as_uint(wmax);
  if (__lane_id() == 0 && w > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(p, w);
}

// Run-aggregated increment of global counters: lanes with `act` whose counter index `t`
// equals the previous lane's form a run (space-ordered catalogues put
// neighbouring particles into one tile, so a wave holds a few long runs);
// the run's first lane adds the run length with one atomic and every
// lane gets old + its rank in the run (RET), or nothing (count only).
// Shuffled catalogues make every lane its own run: one atomic per lane, as
// without aggregation.
template <bool RET>
__device__ __forceinline__ uint32_t run_increment(uint32_t *hist, uint32_t t, bool act) {
  const int lane = __lane_id();
  const uint32_t tp = __shfl_up(t, 1, 64);
  const bool actp = __shfl_up(act ? 1 : 0, 1, 64) != 0;
  const bool head = act && (lane == 0 || !actp || tp != t);
  const uint64_t heads = __ballot(head);
  const uint64_t bound = heads | ~__ballot(act);   // a run ends before these lanes
  uint32_t old = 0;
  if (head) {
    const uint64_t after = lane == 63 ? 0ull : bound & (~0ull << (lane + 1));
    const int next = after ? __ffsll((unsigned long long)after) - 1 : 64;
    const uint32_t len = (uint32_t)(next - lane);
    if (RET) old = atomicAdd(&hist[t], len);
    else atomicAdd(&hist[t], len);
  }
  if (!RET) return 0u;
  // first lane of this lane's run: the highest head at or below it
  const uint64_t below = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1ull));
  const int hl = below ? 63 - __clzll((long long)below) : lane;
  const uint32_t base = __shfl(old, hl, 64);
  return base + (uint32_t)(lane - hl);
}

// Bucketing.  Workgroup b takes particles [b chunk, (b+1) chunk) -- a split
// that depends on the total only, so captured graphs stay valid for any mock
// sizes -- and counts their (particle, tile) pairs in LDS, in a window of
// the tiles of its first particle's mock: all of them up to kWinTiles, else
// kWinTilesBig around the first particle's tile (a catalogue ordered by x
// stays inside; the x tile index is the slowest), or none of them for few
// particles (kWinParticles).  Pairs outside the window or of another mock are
// singles, counted and placed with global atomics.
//  count: each nonzero window counter is added to the tile's count with one
//         atomic, whose return value -- the place of the workgroup's range in
//         the bucket -- goes to whist;
//  scan:  starts = exclusive sums of counts + singles; the singles of a
//         bucket follow the ranges of the workgroups (cursors);
//  fill:  starts + whist is where the workgroup's range begins: slots are
//         handed out with LDS atomics.
// Without whist (no memory for it) every pair counts as a single in the
// count pass, and the fill pass counts its chunk again to reserve ranges.
// The deposit accumulates in integers, so the order of records within a
// bucket does not matter.
// Bound: the catalogue's bytes where its order keeps a tile's records
// together, the 128-byte lines of isolated 24-byte records where it does not.
// Measured on MI355X, count + fill: 2e7 space-ordered particles at N = 1024
// (PCS, interlaced, 131072 tiles) 1.86 -> 0.73 ms with the cells from
// multiplications and one coordinate per axis (the FP64 divisions and the
// second coordinate were most of 450 instructions per particle) and the
// window in place of a global atomic per run; 2e4 particles at N = 64
// 75 -> 12 us and 1e6 at N = 256 86 -> 41 us with chunks that fill the chip.
constexpr int kChunkMax = 16384;
constexpr int kWinTiles = 32768;      // 128 KB of LDS, one workgroup per CU
constexpr int kWinTilesBig = 16384;   // 64 KB, two
// ... and none of them for fewer particles than this, whose few workgroups of
// at least half a window would take longer than global atomics for every
// pair.  Count + scan + fill, global / window, interlaced: 2e4 random
// particles and 262144 tiles, CIC 0.04 / 0.20 ms, PCS 0.05 / 0.36; 131072
// tiles (N = 1024), CIC 0.04 / 0.14, 5e5 0.11 / 0.14, 1e6 0.18 / 0.17, in
// space order 2e5 0.07 / 0.08, 5e5 0.09 / 0.09, 4e6 0.44 / 0.26.
constexpr size_t kWinParticles = (size_t)1 << 19;
constexpr int kBucketThreads = 1024;

__host__ __device__ inline uint32_t window_tiles(uint32_t tpm, size_t ntotal) {
  if (tpm <= (uint32_t)kWinTiles) return tpm;
  return ntotal < kWinParticles ? 0u : (uint32_t)kWinTilesBig;
}

// Particles per workgroup: as many as leave two workgroups for each of the
// 256 CUs, between 256 and kChunkMax, and at least half of the window
// (whose clearing and flushing a chunk pays for).
inline size_t bucket_chunk(const PshAssignGeom &g, size_t ntotal) {
  const uint32_t win = window_tiles((uint32_t)g.ntile[0] * g.ntile[1] * g.ntile[2], ntotal);
  if (g.lean && win) return kChunkMax;   // few workgroups' ranges to keep
  size_t c = 256;
  while (c < (size_t)kChunkMax && (2 * c * 512 <= ntotal || c * 2 < win)) c *= 2;
  return c;
}

template <int SCHEME, bool IL, bool FILL>
__global__ void __launch_bounds__(kBucketThreads, 8)   // 8 waves per SIMD: two workgroups per CU
assign_bucket(PshAssignGeom g, const DevPart *__restrict__ parts, int nparts, size_t ntotal,
              uint32_t chunk, uint32_t *__restrict__ counts, uint32_t *__restrict__ cursors,
              const uint32_t *__restrict__ starts, Rec *__restrict__ recs, size_t rec_cap,
              int *__restrict__ flags, uint32_t *__restrict__ whist) {
  extern __shared__ uint32_t hist[];
  const uint32_t tpm = (uint32_t)g.ntile[0] * g.ntile[1] * g.ntile[2];
  const uint32_t win = window_tiles(tpm, ntotal);
  const uint32_t T = blockDim.x;
  const size_t c0 = (size_t)blockIdx.x * chunk;
  const size_t c1 = min(ntotal, c0 + (size_t)chunk);
  const UPart P0 = uniform_part(parts, nparts, c0);
  const int mock0 = P0.mock;
  uint32_t wbase = 0;
  if (win && win < tpm) {
    // a quarter of the window below the first particle's tile
    const Loaded L0 = load_particle(parts, nparts, P0, c0, true);
    PartTiles pt;
    Rec rec;
    int ign = 0;
    pt.t0 = 0;
    particle_tiles<SCHEME, false, false>(g, L0.r, 0.f, pt, rec, &ign);
    const uint32_t t = (uint32_t)__builtin_amdgcn_readfirstlane(pt.t0);
    wbase = min(t > win / 4 ? t - win / 4 : 0u, tpm - win);
  }
  const uint32_t mbase0 = (uint32_t)mock0 * tpm + wbase;
  uint32_t *wh = whist ? whist + (size_t)blockIdx.x * win : nullptr;
  const int iters = (int)((chunk + T - 1) / T);

  // one sweep over the chunk; the next particle's loads are in flight while
  // the current one is processed, and every lane of a wave runs the same
  // number of iterations (the run aggregation sees whole waves)
  auto sweep = [&](auto check, auto use) {
    size_t gi = c0 + threadIdx.x;
    bool cur_live = gi < c1;
    Loaded cur = load_particle(parts, nparts, P0, gi, cur_live);
#pragma unroll 1
    for (int it = 0; it < iters; it++) {
      const size_t gn = gi + T;
      const bool nxt_live = it + 1 < iters && gn < c1;
      const Loaded nxt = load_particle(parts, nparts, P0, gn, nxt_live);
      PartTiles pt;
      Rec rec;
      bool live = cur_live;
      pt.t0 = pt.off[0] = pt.off[1] = pt.off[2] = 0;
      if (live)
        live = particle_tiles<SCHEME, IL, decltype(check)::value>(g, cur.r, cur.wscale, pt, rec,
                                                                  flags);
      use(pt, rec, live, cur.mock);
      cur = nxt;
      cur_live = nxt_live;
      gi = gn;
    }
  };
  auto clear = [&]() {
    for (uint32_t i = threadIdx.x; i < win; i += T) hist[i] = 0;
    __syncthreads();
  };
  uint32_t ranges = 0;   // nonzero counters and singles
  // counts the pairs inside the window and, with `singles`, the others (the
  // k-th tiles of a wave's lanes together)
  auto count_pairs = [&](auto check, bool singles) {
    sweep(check, [&](const PartTiles &pt, const Rec &, bool live, int mock) {
      const bool mine = live && mock == mock0;
      bool out = false;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        if (!live || !pt.has(k)) continue;
        const uint32_t w = pt.tile(k) - wbase;
        if (mine && w < win) atomicAdd(&hist[w], 1u);
        else out = true;
      }
      if (!singles || !__ballot(out)) return;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const bool act = out && pt.has(k) && !(mine && pt.tile(k) - wbase < win);
        if (!__ballot(act)) continue;
        run_increment<false>(cursors, act ? (uint32_t)mock * tpm + pt.tile(k) : 0u, act);
        ranges += act;
      }
    });
    __syncthreads();
  };

  if (!FILL) {
    __shared__ uint32_t nrange;
    if (threadIdx.x == 0) nrange = 0;
    clear();
    count_pairs(std::true_type{}, true);
    for (uint32_t i = threadIdx.x; i < win; i += T) {
      const uint32_t v = hist[i];
      ranges += v != 0;
      if (wh) wh[i] = v ? atomicAdd(&counts[mbase0 + i], v) : 0u;
      else if (v) atomicAdd(&cursors[mbase0 + i], v);
    }
    // ranges of records that fill the buckets (record_group)
    for (int o = 32; o > 0; o >>= 1) ranges += __shfl_xor(ranges, o);
    if (__lane_id() == 0) atomicAdd(&nrange, ranges);
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(reinterpret_cast<uint32_t *>(flags) + 2, nrange);
    return;
  }
  if (wh) {
    for (uint32_t i = threadIdx.x; i < win; i += T) hist[i] = starts[mbase0 + i] + wh[i];
  } else if (win) {
    clear();
    count_pairs(std::false_type{}, false);
    for (uint32_t i = threadIdx.x; i < win; i += T)
      if (hist[i]) hist[i] = atomicAdd(&cursors[mbase0 + i], hist[i]);
  }
  __syncthreads();
  float wmax = 0.f;
  sweep(std::false_type{}, [&](const PartTiles &pt, const Rec &rec, bool live, int mock) {
    const bool mine = live && mock == mock0;
    if (live) wmax = fmaxf(wmax, fabsf(rec.w));
    uint32_t slot[8];
    bool out = false;
    // every slot is asked for before the first record is written
#pragma unroll
    for (int k = 0; k < 8; k++) {
      slot[k] = 0xffffffffu;
      if (!live || !pt.has(k)) continue;
      const uint32_t w = pt.tile(k) - wbase;
      if (mine && w < win) slot[k] = atomicAdd(&hist[w], 1u);
      else out = true;
    }
    if (__ballot(out)) {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const bool act = out && pt.has(k) && !(mine && pt.tile(k) - wbase < win);
        if (!__ballot(act)) continue;
        const uint32_t q =
            run_increment<true>(cursors, act ? (uint32_t)mock * tpm + pt.tile(k) : 0u, act);
        if (act) slot[k] = q;
      }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (!live || !pt.has(k)) continue;
      if (slot[k] < rec_cap) recs[slot[k]] = pt.record(rec, g, k);
      else atomicOr(flags, 1);
    }
  });
  publish_wmax(wmax, flags);
}

// ---- exclusive scan of uint32 counters -------------------------------------
// One workgroup up to kScanOne counters (a launch costs more than the scan),
// else three kernels.  TWO: the counters are in[i] + cursors[i], and cursors
// becomes out[i] + in[i].
constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanBlock = kScanThreads * kScanItems;
constexpr int kScanOneThreads = 1024;
constexpr size_t kScanOne = 32768;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v,
                                                         uint32_t *sh,
                                                         uint32_t &total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  uint32_t x = v;
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
      uint32_t t = sh[w];
      sh[w] = run;
      run += t;
    }
    sh[16] = run;
  }
  __syncthreads();
  total = sh[16];
  uint32_t res = x - v + sh[wid];
  __syncthreads();
  return res;
}

template <bool TWO>
__global__ void __launch_bounds__(kScanOneThreads)
scan_one(const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
         uint32_t *__restrict__ cursors, int n) {
  __shared__ uint32_t sh[17];
  uint32_t carry = 0;
  // a thread takes 16 consecutive counters with 16-byte accesses (word by
  // word, a wave's accesses touch 64 lines each: 31 us for 16384 counters)
  constexpr int K = 16;
  for (int base = 0; base < n; base += K * kScanOneThreads) {
    const int i0 = base + K * threadIdx.x;
    const bool whole = i0 + K <= n;
    uint32_t v[K], c[K], s = 0;
#pragma unroll
    for (int k = 0; k < K; k += 4) {
      uint4 a = make_uint4(0u, 0u, 0u, 0u), b = a;
      if (whole) {
        a = *reinterpret_cast<const uint4 *>(in + i0 + k);
        if (TWO) b = *reinterpret_cast<const uint4 *>(cursors + i0 + k);
      }
      v[k] = a.x, v[k + 1] = a.y, v[k + 2] = a.z, v[k + 3] = a.w;
      c[k] = b.x, c[k + 1] = b.y, c[k + 2] = b.z, c[k + 3] = b.w;
    }
    if (!whole) {
#pragma unroll
      for (int k = 0; k < K; k++) {
        if (i0 + k >= n) break;
        v[k] = in[i0 + k];
        if (TWO) c[k] = cursors[i0 + k];
      }
    }
#pragma unroll
    for (int k = 0; k < K; k++) s += v[k] + c[k];
    uint32_t tot;
    uint32_t ex = block_exclusive_scan(s, sh, tot) + carry;
#pragma unroll
    for (int k = 0; k < K; k++) {   // c: the exclusive sum; v: c + v
      const uint32_t t = v[k] + c[k];
      v[k] += ex;
      c[k] = ex;
      ex += t;
    }
#pragma unroll
    for (int k = 0; k < K; k += 4) {
      if (whole) {
        *reinterpret_cast<uint4 *>(out + i0 + k) = make_uint4(c[k], c[k + 1], c[k + 2], c[k + 3]);
        if (TWO)
          *reinterpret_cast<uint4 *>(cursors + i0 + k) =
              make_uint4(v[k], v[k + 1], v[k + 2], v[k + 3]);
      } else {
#pragma unroll
        for (int q = k; q < k + 4; q++) {
          if (i0 + q >= n) break;
          out[i0 + q] = c[q];
          if (TWO) cursors[i0 + q] = v[q];
        }
      }
    }
    carry += tot;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

template <bool TWO>
__global__ void __launch_bounds__(kScanThreads)
scan_local(const uint32_t *__restrict__ in, const uint32_t *__restrict__ in2,
           uint32_t *__restrict__ out, uint32_t *__restrict__ bsum, size_t n) {
  __shared__ uint32_t sh[17];
  size_t base = (size_t)blockIdx.x * kScanBlock + (size_t)threadIdx.x * kScanItems;
  uint32_t v[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    v[i] = (base + i < n) ? in[base + i] + (TWO ? in2[base + i] : 0u) : 0u;
    s += v[i];
  }
  uint32_t tot;
  uint32_t ex = block_exclusive_scan(s, sh, tot);
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    if (base + i < n) out[base + i] = ex;
    ex += v[i];
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(kScanThreads)
scan_sums(uint32_t *__restrict__ bsum, int nb) {
  __shared__ uint32_t sh[17];
  uint32_t carry = 0;
  for (int base = 0; base < nb; base += kScanThreads) {
    int i = base + threadIdx.x;
    uint32_t v = (i < nb) ? bsum[i] : 0u;
    uint32_t tot;
    uint32_t ex = block_exclusive_scan(v, sh, tot);
    if (i < nb) bsum[i] = ex + carry;
    carry += tot;
  }
  if (threadIdx.x == 0) bsum[nb] = carry;
}

template <bool TWO>
__global__ void __launch_bounds__(kScanThreads)
scan_add(const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
         uint32_t *__restrict__ cursors, const uint32_t *__restrict__ bsum, size_t n, int nb) {
  size_t base = (size_t)blockIdx.x * kScanBlock;
  uint32_t off = bsum[blockIdx.x];
  for (int i = threadIdx.x; i < kScanBlock; i += kScanThreads) {
    size_t k = base + i;
    if (k < n) {
      uint32_t v = out[k] + off;
      out[k] = v;
      if (TWO) cursors[k] = v + in[k];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = bsum[nb];
}

template <bool TWO>
hipError_t launch_scan(const uint32_t *in, uint32_t *out, uint32_t *cursors, uint32_t *tmp,
                       size_t n, hipStream_t s) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out) |
                         reinterpret_cast<uintptr_t>(cursors)) & 15) == 0;
  if (n <= kScanOne && aligned) {
    hipLaunchKernelGGL((scan_one<TWO>), dim3(1), dim3(kScanOneThreads), 0, s, in, out, cursors,
                       (int)n);
  } else {
    const int nsb = (int)((n + kScanBlock - 1) / kScanBlock);
    hipLaunchKernelGGL((scan_local<TWO>), dim3(nsb), dim3(kScanThreads), 0, s, in, cursors, out,
                       tmp, n);
    hipLaunchKernelGGL(scan_sums, dim3(1), dim3(kScanThreads), 0, s, tmp, nsb);
    hipLaunchKernelGGL((scan_add<TWO>), dim3(nsb), dim3(kScanThreads), 0, s, in, out, cursors,
                       tmp, n, nsb);
  }
  return hipGetLastError();
}

__global__ void fill_zero_u32(uint32_t *p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

// Start of an assignment in one launch: the tile counters and the flags
// cleared and, when they are few, the part table written from the arguments
// (a copy from host memory costs the caller a staging copy and another
// launch).
struct FewParts {
  int n;
  DevPart p[kFewParts];
};

__global__ void __launch_bounds__(256)
assign_begin(uint32_t *__restrict__ counts, uint32_t *__restrict__ cursors, size_t n,
             int *__restrict__ flags, DevPart *__restrict__ parts, FewParts few) {
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    counts[i] = 0u;
    cursors[i] = 0u;
  }
  if (blockIdx.x == 0) {
    if (threadIdx.x < 4) flags[threadIdx.x] = 0;
    if ((int)threadIdx.x < few.n) parts[threadIdx.x] = few.p[threadIdx.x];
  }
}

// ---- deposit: one workgroup per tile ------------------------------------------

// The products that are added to something are fused into the addition
// explicitly: left to the compiler, which fusions it makes depends on the code
// around the call, and so would the last bits of the weights.
__device__ __forceinline__ void window_weights(int scheme, float f, float *w) {
#pragma clang fp contract(off)
  switch (scheme) {
    case 0:
      w[0] = 1.f;
      break;
    case 1:
      w[0] = 1.f - f;
      w[1] = f;
      break;
    case 2: {
      const float a = 0.5f - f, h = 0.5f * a;
      w[0] = a * h;
      w[1] = __builtin_fmaf(-f, f, 0.75f);
      w[2] = __builtin_fmaf(-a, h, 1.f) - w[1];
      break;
    }
    default: {
      const float d2 = f * f;
      w[3] = f * d2;
      w[2] = __builtin_fmaf(__builtin_fmaf(-f, d2, __builtin_fmaf(f, f, f)), 3.f, 1.f);
      w[1] = __builtin_fmaf(3.f, w[3], __builtin_fmaf(-6.f, d2, 4.f));
      w[0] = __builtin_fmaf(-f, d2, (6.f - w[1]) - w[2]);
      break;
    }
  }
}

// Fixed-point LDS accumulators (value * 2^s as a signed integer; FP32 LDS
// atomics are an order of magnitude slower on gfx950).  Integer addition is
// associative, so a tile does not depend on the order of its records.
//  - 32-bit (ds_add_u32): the exponent leaves about 2^-30 * cells-per-tile
//    relative precision per contribution -- ample for boxes, whose fields
//    are sums of positive weights;
//  - 64-bit (ds_add_u64): each contribution keeps its FP32 precision; used
//    when weights of both signs meet (survey data minus alpha * randoms),
//    where large-scale modes are small differences of large sums.
template <bool WIDE>
struct Acc;
// add(p, a, b, half) accumulates a * b rounded to an integer, half being
// 0.5 with the sign of the product.  32-bit: one FMA and a truncating
// conversion, trunc(a b + half) = a b rounded half away from zero (the
// rounding of a b + half in FP32 can move a product of 2^23 or more by one
// unit, a relative 1.2e-7, the FP32 precision the tile carries anyway).
template <>
struct Acc<false> {
  using T = int;
  static constexpr int TOP = 30;
  __device__ static __forceinline__ void add(int *p, float a, float b, float half) {
    atomicAdd(p, (int)__builtin_fmaf(a, b, half));
  }
};
template <>
struct Acc<true> {
  using T = long long;
  static constexpr int TOP = 62;
  __device__ static __forceinline__ void add(long long *p, float a, float b, float) {
    atomicAdd(reinterpret_cast<unsigned long long *>(p),
              (unsigned long long)__float2ll_rn(a * b));
  }
};

// Window axes x and y: an axis a >= branch_axes is deposited without
// branches (a window cell outside the tile gets weight 0 and the address of
// a cell inside; adding the integer 0 there is exact), an axis
// below keeps a branch per plane or row, which skips whole planes or rows
// outside the tile.  Measured on MI355X: y without branches for CIC and TSC,
// with them for PCS (whose 4-cell rows make a skipped row worth more).
// Axis z: the tile's rows are padded by W cells on each side, so a window
// row is W consecutive cells from one base address (constant LDS offsets,
// no per-cell mask or address arithmetic); cells in the padding are
// dropped, their tile deposits them from its own record.  A record's tile
// meets the union of the plain and the shifted window, so the window's first
// cell lies in [-W, T[2]] and W cells of padding on each side hold every
// cell outside the tile.
// WRAP: some axis of the tile spans the grid, so that windows wrap around
// inside the tile; z then goes the branch-free way of x and y.
template <int SCHEME>
constexpr int branch_axes() { return SCHEME == 3 ? 2 : 1; }

// Accumulate one particle's window, whose first cell is l (local), into an
// LDS tile of fixed-point cells (rows of P2 >= T[2] + 2 W cells, the tile's
// first z cell at W).
template <int SCHEME, bool WIDE, bool WRAP>
__device__ __forceinline__ void deposit_one(typename Acc<WIDE>::T *lds, const int *T, int Ng,
                                            int P2, const int *l, const float *f, float w) {
  constexpr int W = SCHEME + 1;
  constexpr int kBranchAxes = branch_axes<SCHEME>();
  float wt[3][4];
#pragma unroll
  for (int a = 0; a < 3; a++) window_weights(SCHEME, f[a], wt[a]);
  // cell n of axis a, and whether it lies in the tile
  auto cell = [&](int a, int n, bool &in) -> int {
    int c = l[a] + n;
    if (WRAP && c >= Ng) c -= Ng;
    in = (unsigned)c < (unsigned)T[a];
    return c;
  };
  int zc[4];   // WRAP: the row's cells
  if (WRAP) {
#pragma unroll
    for (int n = 0; n < W; n++) {
      bool in;
      const int c = cell(2, n, in);
      zc[n] = in ? c : 0;
      if (!in) wt[2][n] = 0.f;
    }
  }
  if (SCHEME == 3) w *= (1.0f / 216.0f);
  const float half = __builtin_copysignf(0.5f, w);   // window weights are >= 0
  // row offsets: the products stay below 2^24 (a tile has at most 40960
  // cells), where the integer multiply-add runs at full rate
  const int z0 = WRAP ? W : l[2] + W;
  int ry[4];
  bool iny[4];
#pragma unroll
  for (int j = 0; j < W; j++) {
    const int c = cell(1, j, iny[j]);
    if (kBranchAxes <= 1 && !iny[j]) wt[1][j] = 0.f;
    ry[j] = __mul24(min(max(c, 0), T[1] - 1), P2) + z0;
  }
  const int PP = T[1] * P2;
#pragma unroll
  for (int i = 0; i < W; i++) {
    bool inx;
    const int c = cell(0, i, inx);
    if (!inx) continue;
    const float wx = wt[0][i] * w;
    const int rx = __mul24(c, PP);
#pragma unroll
    for (int j = 0; j < W; j++) {
      if (kBranchAxes > 1 && !iny[j]) continue;
      const float wxy = wx * wt[1][j];
      typename Acc<WIDE>::T *row = lds + rx + ry[j];
#pragma unroll
      for (int k = 0; k < W; k++)
        Acc<WIDE>::add(WRAP ? row + zc[k] : row + k, wxy, wt[2][k], half);
    }
  }
}

// Fixed-point exponent of a tile: a cell value is a sum of at most cnt
// contributions of magnitude <= max|w| (window weights are <= 1 and sum to 1
// per axis), so |value| * 2^s < 2^TOP, one bit below the accumulator's sign.
template <int TOP>
__device__ __forceinline__ int tile_exponent(const int *flags, uint32_t cnt) {
  const float maxw = __uint_as_float((unsigned)flags[1]);
  const double bound = (double)maxw * (double)cnt * (1.0 + 1e-7);
  if (!(bound > 0.0)) return TOP;
  // ceil(log2(bound)) exactly: bound = m 2^e with m in [0.5, 1)
  int e;
  const double m = frexp(bound, &e);
  const int s = TOP - (m == 0.5 ? e - 1 : e);
  return s < -100 ? -100 : (s > 100 ? 100 : s);
}

typedef float v4f_t __attribute__((ext_vector_type(4)));

// Four consecutive mesh cells; non-temporal when the meshes are much larger
// than the caches (a template parameter: under a runtime flag the compiler
// merges both stores into an ordinary one).
template <bool NT>
__device__ __forceinline__ void store4(float *p, float4 v) {
  const v4f_t x = {v.x, v.y, v.z, v.w};
  if constexpr (NT) __builtin_nontemporal_store(x, reinterpret_cast<v4f_t *>(p));
  else *reinterpret_cast<v4f_t *>(p) = x;
}

// Deposit with the z transform fused in (boxes): a tile holds TX x TY whole
// z rows per grid, C lines over both grids, transformed by 1024 threads
// like the z pass; the rows (N + 2W cells) take about 130 KB of LDS at
// every size.  From N = 512, C = 32768 / N lines of 32-bit cells (16 values
// per thread).  Smaller grids put many more records into a tile, and a
// 32-bit cell's fixed-point step grows with the tile's record count (at
// N = 128 the quantisation reached 1e-5 of P(k) in sparsely populated
// bins): they take 64-bit cells, C = 16384 / N lines, 8 values per thread.
template <int N, bool IL>
struct ZfCfg {
  static constexpr bool WIDE = N <= 256;
  static constexpr int C = (WIDE ? 16384 : 32768) / N;   // lines per tile, both grids
  static constexpr int R = IL ? C / 2 : C;               // rows per grid
  static constexpr int TX = R >= 128 ? 16 : (R >= 32 ? 8 : 4);
  static constexpr int TY = R / TX;
  static constexpr int T = 1024;
  static_assert(TX * TY == R && TY >= 4, "tile rows");
};

// Tile of a workgroup.
struct DepTile {
  int T[3], T0[3];
  int mock;
  uint32_t tile;
};

__device__ __forceinline__ DepTile dep_tile(const PshAssignGeom &g, uint32_t tile) {
  // tile index -> (mock, x, y, z) tile; tile counts need not be powers of
  // two (a grid of 3 * 2^k or 5 * 2^k cells has 3 or 5 times a power)
  DepTile d;
  const uint32_t nz = (uint32_t)g.ntile[2], ny = (uint32_t)g.ntile[1];
  const uint32_t tpm = (uint32_t)g.ntile[0] * ny * nz;
  d.tile = tile;
  d.mock = (int)(tile / tpm);
  const uint32_t tl = tile - (uint32_t)d.mock * tpm;
  const uint32_t tyz = tl / nz;
  const uint32_t tx = tyz / ny;
#pragma unroll
  for (int a = 0; a < 3; a++) d.T[a] = g.tile[a];
  d.T0[0] = (int)tx * d.T[0];
  d.T0[1] = (int)(tyz - tx * ny) * d.T[1];
  d.T0[2] = (int)(tl - tyz * nz) * d.T[2];
  return d;
}

template <class AT>
__device__ __forceinline__ void clear_cells(AT *lds, int cells) {
  uint4 *z4 = reinterpret_cast<uint4 *>(lds);   // cells: a multiple of 4
  const int n4 = (int)(sizeof(AT) * cells / 16);
  for (int i = threadIdx.x; i < n4; i += blockDim.x) z4[i] = make_uint4(0u, 0u, 0u, 0u);
}

// The records of a bucket over the workgroup's threads: visit(r) for each,
// the next one loading while the current one is deposited.
//  - At most one record per thread: on the fewest waves that hold them
//    (nw = ceil(cnt / 64)), since a VALU-bound wave issues as many
//    instructions for 20 live lanes as for 64 and the other waves go straight
//    to the barrier.  Lane l of wave w < nw takes record l * nw + w (a
//    bijection of [0, 64 nw)), so a wave's lanes hold records nw apart in
//    fill order rather than neighbours.
//  - More: groups of 2^gs neighbours in the
//    order q -> (q * S) mod ngroups with S ~ 0.618 ngroups and
//    gcd(S, ngroups) = 1 (a permutation): a wave's groups lie far apart in
//    fill order, i.e. far apart in a space-ordered catalogue, so
//    its lanes' windows rarely meet in one cell (record_group).
//  - More, with STRETCH (PCS, whose 64 cells leave no room for neighbours in a
//    wave, and TSC with both grids in a workgroup): a stretch of consecutive records
//    per thread, the stretches of a wave's lanes far apart; a line's records
//    are then read one after another by one lane.  (Random order: whole waves
//    of consecutive records, as above.)  Dense ordered catalogues, interlaced:
//    PCS, 3e7 particles at N = 256, pairs in the permuted order 2.27 ms, single
//    records in it 1.84, stretches 1.53; 8e6 at N = 128 0.77, 0.46, 0.48; TSC
//    in whole z rows, with their transform, 1e8 at N = 256 pairs 7.8 ms,
//    stretches 5.6.  In the default tiles TSC gains at N = 128 (3e7 particles
//    1.31 -> 1.20) and loses without interlacing (N = 256 0.59 -> 0.71); NGP
//    and CIC lose up to a factor of two.
template <bool STRETCH, class F>
__device__ __forceinline__ void for_records(const Rec *__restrict__ recs, uint32_t cnt, uint32_t gs,
                                            F visit) {
  const uint32_t t = threadIdx.x, B = blockDim.x;
  if (cnt <= B) {
    const uint32_t nw = (cnt + 63u) >> 6, w = t >> 6;
    const uint32_t j = (t & 63u) * nw + w;
    const bool live = w < nw && j < cnt;
    Rec r;
    if (live) r = recs[j];
    __syncthreads();   // the cells are cleared
    if (live) visit(r);
    return;
  }
  if constexpr (STRETCH) {
    // n records per thread, one more for the first `rest` threads (whole
    // waves); stretch l nw + w belongs to lane l of wave w
    const uint32_t q = cnt / B, rest = cnt - q * B, n = q + (t < rest);
    uint32_t i = t, step = B;
    if (gs == 0) {
      const uint32_t l = t & 63u, w = t >> 6, a = rest >> 6, b = rest & 63u;
      i = (l * (B >> 6) + w) * q + l * a + min(l, b) + min(w, a) + (w > a && l < b);
      step = 1;
    }
    Rec r = recs[i];   // n >= 1
    __syncthreads();   // the cells are cleared
    for (uint32_t k = 0; k < n; k++) {
      Rec next;
      if (k + 1 < n) next = recs[i += step];
      visit(r);
      r = next;
    }
    return;
  }
  const uint32_t ng = (cnt + (1u << gs) - 1) >> gs;
  uint32_t S = ((uint32_t)((float)ng * 0.618034f)) | 1u;
  if (S >= ng) S = 1u;
  for (;;) {
    uint32_t a = S, b = ng;
    while (b) {
      const uint32_t q = a % b;
      a = b;
      b = q;
    }
    if (a == 1u) break;
    S += 2u;
    if (S >= ng) {
      S = 1u;
      break;
    }
  }
  const uint32_t in = t & ((1u << gs) - 1u), step = B >> gs;
  uint32_t q = t >> gs;
  uint32_t x = (uint32_t)(((uint64_t)q * S) % ng);
  const uint32_t D = (uint32_t)(((uint64_t)step * S) % ng);
  auto index = [&]() -> uint32_t { return q < ng ? (x << gs) + in : cnt; };
  auto next = [&]() {
    q += step;
    x += D;
    if (x >= ng) x -= ng;
  };
  uint32_t i = index();
  Rec r;
  if (i < cnt) r = recs[i];
  __syncthreads();   // the cells are cleared
  const uint32_t iters = (ng + step - 1) / step;
  for (uint32_t it = 0; it < iters; it++) {
    next();
    const uint32_t in2 = index();
    Rec r2;
    if (in2 < cnt) r2 = recs[in2];
    if (i < cnt) visit(r);
    i = in2;
    r = r2;
  }
}

// log2 of the records a wave reads from consecutive places of a bucket:
// larger groups use more of the 128-byte lines they touch, smaller ones keep
// the windows of a space-ordered catalogue's neighbours apart.  Ordered:
// 1 with stretches (for_records), 2 records for TSC (N = 256, 32 mocks: 1.71, 1.69,
// 1.76 ms for 1, 2, 4), 4 for NGP and CIC (N = 512, 2e7 particles: 301, 269, 247 us).
// A bucket filled in ranges of a few records (fewer than 16 on average, from
// the count pass's number of ranges) is in random order, where neighbours are
// no closer than others: a whole wave's (survey, N = 512, 1e8 randoms:
// 2.12 ms with 4, 1.82 with 64).
template <int SCHEME, bool STRETCH>
__device__ __forceinline__ uint32_t record_group(const uint32_t *starts, uint32_t ntiles,
                                                 const int *flags) {
  const bool random = starts[ntiles] / 16 < (uint32_t)flags[2];
  return random ? 6u : STRETCH ? 0u : SCHEME >= 2 ? 1u : 2u;
}

// One record's window on the plain or the shifted grid of a tile.
template <int SCHEME, bool WIDE>
__device__ __forceinline__ void deposit_rec(typename Acc<WIDE>::T *lds, const DepTile &d,
                                            const PshAssignGeom &g, int P2, bool wrap,
                                            bool shifted, const Rec &r, float scale) {
  int l[3] = {(int)(r.bxy & 0xffffu) - kRecBias, (int)(r.bxy >> 16) - kRecBias,
              (int)(r.bz & 0xffffu) - kRecBias};
  float f[3] = {r.f[0], r.f[1], r.f[2]};
  if (shifted) {
    const uint32_t dl = r.bz >> 16;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const int s = (dl >> a) & 1;
      l[a] += s;
      f[a] = f[a] + 0.5f - (float)s;
    }
  }
  const float ws = r.w * scale;
  if (wrap) deposit_one<SCHEME, WIDE, true>(lds, d.T, g.Ng, P2, l, f, ws);
  else deposit_one<SCHEME, WIDE, false>(lds, d.T, g.Ng, P2, l, f, ws);
}

// Bucket of a tile.  Records past the buffer were never written (overflow
// flag set, the run is repeated with a larger buffer): never read beyond
// rec_cap.
struct DepBucket {
  uint32_t s0, cnt;
  float scale, inv;
};

template <int TOP>
__device__ __forceinline__ DepBucket dep_bucket(const uint32_t *starts, uint32_t tile,
                                                size_t rec_cap, const int *flags) {
  const uint32_t cap = rec_cap < 0xffffffffu ? (uint32_t)rec_cap : 0xffffffffu;
  const uint32_t s0 = min(starts[tile], cap), s1 = min(starts[tile + 1], cap);
  DepBucket k;
  k.s0 = s0;
  k.cnt = s1 > s0 ? s1 - s0 : 0u;
  const int sexp = tile_exponent<TOP>(flags, k.cnt);
  k.scale = ldexpf(1.f, sexp);
  k.inv = ldexpf(1.f, -sexp);
  return k;
}

// A grid's tile to its mesh: rows of T[2] floats along z, 4 cells per thread.
template <int SCHEME, bool NT, class AT>
__device__ __forceinline__ void write_tile(const AT *lds, const DepTile &d, const PshAssignGeom &g,
                                           int P2, int lead, float inv, float *out) {
  const int nrow = d.T[0] * d.T[1];
  const int q4s = g.tile_shift[2] - 2;   // T[2] = 4 * 2^q4s (T[2] >= 4)
  const int q4 = 1 << q4s;
  for (int i = threadIdx.x; i < nrow * q4; i += blockDim.x) {
    const int row = i >> q4s, q = i & (q4 - 1);
    const int lx = row >> g.tile_shift[1], ly = row & (d.T[1] - 1);
    const size_t gidx = ((size_t)(d.T0[0] + lx) * g.Ng + (d.T0[1] + ly)) * g.row_pitch +
                        d.T0[2] + 4 * q;
    const int li = row * P2 + SCHEME + 1 + 4 * q;
    AT c[4];
    if (((P2 | (lead + SCHEME + 1)) & 3) == 0) {   // 16-byte aligned rows
      const uint4 *p = reinterpret_cast<const uint4 *>(lds + li);
#pragma unroll
      for (int h = 0; h < (int)(sizeof(c) / 16); h++) reinterpret_cast<uint4 *>(c)[h] = p[h];
    } else {
#pragma unroll
      for (int h = 0; h < 4; h++) c[h] = lds[li + h];
    }
    const float4 v = make_float4((float)c[0] * inv, (float)c[1] * inv, (float)c[2] * inv,
                                 (float)c[3] * inv);
    store4<NT>(out + gidx, v);
  }
}

// Deposit of one grid (plain, or with INTLACE every second group of 8
// workgroups the shifted one) of one tile per workgroup.  Bound: the LDS
// atomics of the windows and the stores of the mesh; their phases alternate
// within a workgroup, so it is other workgroups of the CU that overlap them.
// One grid per workgroup halves the LDS tile: 4 workgroups of 512 threads per
// CU instead of 2 for 32-bit cells, 2 instead of 1 for the survey's 64-bit
// cells, for a second read of the records (the two grids of a tile follow
// one another on one XCD: workgroups are dealt to the XCDs in turn).
// Measured on MI355X (with the records' local cells, the next record in
// flight and 16-byte LDS reads): N = 1024 PCS, 2e7 particles 2.72 -> 2.34 ms,
// 8.6 GB of mesh at 3.7 TB/s; the survey's 64-bit CIC, N = 512, 1.5e8 records
// 2.81 -> 1.64 ms; N = 512 CIC, 2e7 particles 0.31 -> 0.25 ms.
// BOTH: both grids of the tile in one workgroup, for catalogues whose second
// read costs more than that (launch_deposit).
template <int SCHEME, bool INTLACE, bool WIDE, bool NT, bool BOTH = false>
__global__ void __launch_bounds__(1024)
assign_deposit(PshAssignGeom g, const uint32_t *__restrict__ starts,
               const Rec *__restrict__ recs, size_t rec_cap,
               float *__restrict__ meshA, float *__restrict__ meshB,
               size_t mstride, const int *__restrict__ flags, int P2, int lead, int cells,
               uint32_t ntiles, uint32_t b0) {
  using AT = typename Acc<WIDE>::T;
  extern __shared__ __align__(16) long long ldsraw[];
  AT *lds = reinterpret_cast<AT *>(ldsraw) + lead;
  const uint32_t b = blockIdx.x + b0;
  uint32_t tile = b;
  bool shifted = false;
  if (INTLACE && !BOTH) {
    // blocks 16 n + (0..7) and 16 n + 8 + (0..7): the grids of tiles 8 n + (0..7)
    if (ntiles & 7) {
      shifted = b & 1;
      tile = b >> 1;
    } else {
      shifted = (b >> 3) & 1;
      tile = (b >> 4) * 8 + (b & 7);
    }
  }
  const DepBucket k = dep_bucket<Acc<WIDE>::TOP>(starts, tile, rec_cap, flags);
  const DepTile d = dep_tile(g, tile);
  const bool wrap = d.T[0] == g.Ng || d.T[1] == g.Ng || d.T[2] == g.Ng;
  clear_cells(lds - lead, BOTH ? 2 * cells : cells);
  constexpr bool STRETCH = SCHEME == 3 || BOTH;
  for_records<STRETCH>(recs + k.s0, k.cnt, record_group<SCHEME, STRETCH>(starts, ntiles, flags),
                       [&](const Rec &r) {
    deposit_rec<SCHEME, WIDE>(lds, d, g, P2, wrap, shifted, r, k.scale);
    if (BOTH) deposit_rec<SCHEME, WIDE>(lds + cells, d, g, P2, wrap, true, r, k.scale);
  });
  __syncthreads();

  write_tile<SCHEME, NT>(lds, d, g, P2, lead, k.inv,
                         (shifted ? meshB : meshA) + (size_t)d.mock * mstride);
  if (BOTH)
    write_tile<SCHEME, NT>(lds + cells, d, g, P2, lead, k.inv, meshB + (size_t)d.mock * mstride);
}

// Deposit of both grids of a tile of whole z rows, transformed along z.
template <int SCHEME, bool INTLACE, bool WIDE, bool NT, int NZ>
__global__ void __launch_bounds__(1024)
assign_deposit_z(PshAssignGeom g, const uint32_t *__restrict__ starts,
                 const Rec *__restrict__ recs, size_t rec_cap,
                 float *__restrict__ meshA, float *__restrict__ meshB,
                 size_t mstride, const int *__restrict__ flags) {
  using AT = typename Acc<WIDE>::T;
  extern __shared__ __align__(16) long long ldsraw[];
  AT *ldsq = reinterpret_cast<AT *>(ldsraw);
  const DepBucket k = dep_bucket<Acc<WIDE>::TOP>(starts, blockIdx.x, rec_cap, flags);
  const DepTile d = dep_tile(g, blockIdx.x);
  const int P2 = psh_tile_pitch(d.T[2], SCHEME);
  const int gcells = (int)psh_tile_cells(d.T, SCHEME);   // per grid, padded
  const bool wrap = d.T[0] == g.Ng || d.T[1] == g.Ng || d.T[2] == g.Ng;
  AT *ldsA = ldsq;
  AT *ldsB = ldsq + gcells;
  const int *T0 = d.T0;
  const int mock = d.mock;
  const float inv = k.inv;
  clear_cells(ldsq, gcells * (INTLACE ? 2 : 1));
  constexpr bool STRETCH = SCHEME >= 2;
  for_records<STRETCH>(recs + k.s0, k.cnt, record_group<SCHEME, STRETCH>(starts, gridDim.x, flags),
                       [&](const Rec &r) {
    deposit_rec<SCHEME, WIDE>(ldsA, d, g, P2, wrap, false, r, k.scale);
    if (INTLACE) deposit_rec<SCHEME, WIDE>(ldsB, d, g, P2, wrap, true, r, k.scale);
  });
  __syncthreads();

  // The tile's rows, both grids, as NZ / 2-point complex lines (cells
  // 2n, 2n + 1 of a row), transformed like the z pass (z_r2c_kernel) and
  // split into the half-complex row X[0..NZ/2] (k_z <= kzlim stored):
  // X[k] = E + W^k O, X[M - k] = conj(E - W^k O).
  using namespace pshfft;
  using Z = ZfCfg<NZ, INTLACE>;
  constexpr int M = NZ / 2, C = Z::C, TT = Z::T, W = SCHEME + 1;
  using LZ = Lds<M, C, false>;
  constexpr int V = max_values<M, C, TT, false>();
  float2 v[V];
  pass_load<M, C, TT, 0, false>(v, [&](int c, int n) -> float2 {
    const AT *row = (c < Z::R ? ldsA + c * P2 : ldsB + (c - Z::R) * P2) + W;
    return make_float2((float)row[2 * n] * inv, (float)row[2 * n + 1] * inv);
  });
  __syncthreads();   // every cell read before the exchange tile overwrites them
  float *xl = reinterpret_cast<float *>(ldsq);
  Passes<M, C, TT, 0, false, false, 2>::run(v, xl, g.tw);
  constexpr int NP = M / 2 + 1;
  constexpr int NI = (C * NP + TT - 1) / TT;
  float rk[NI], rmk[NI];
  store_last<M, C, TT, false>(v, [&](int c, int n, float2 x) { xl[LZ::idx(c, n)] = x.x; });
  __syncthreads();
#pragma unroll
  for (int it = 0; it < NI; it++) {
    const int item = threadIdx.x + it * TT;
    const int c = item / NP, k = item - c * NP;
    if (item < C * NP) {
      rk[it] = xl[LZ::idx(c, k)];
      rmk[it] = xl[LZ::idx(c, mirror<M>(k))];
    }
  }
  __syncthreads();
  store_last<M, C, TT, false>(v, [&](int c, int n, float2 x) { xl[LZ::idx(c, n)] = x.y; });
  __syncthreads();
  float2 *cA = reinterpret_cast<float2 *>(meshA + (size_t)mock * mstride);
  float2 *cB = INTLACE ? reinterpret_cast<float2 *>(meshB + (size_t)mock * mstride) : nullptr;
  const int H = g.row_pitch / 2;
#pragma unroll
  for (int it = 0; it < NI; it++) {
    const int item = threadIdx.x + it * TT;
    const int c = item / NP, k = item - c * NP;
    if (item >= C * NP) continue;
    const float ik = xl[LZ::idx(c, k)];
    const float imk = xl[LZ::idx(c, mirror<M>(k))];
    const float2 E = make_float2(0.5f * (rk[it] + rmk[it]), 0.5f * (ik - imk));
    const float2 O = make_float2(0.5f * (ik + imk), -0.5f * (rk[it] - rmk[it]));
    const float2 WO = cmul(g.tw[k], O);
    const int grid = c / Z::R, row = c - grid * Z::R;
    const int lx = row / Z::TY, ly = row - lx * Z::TY;
    float2 *orow = (grid ? cB : cA) + ((size_t)(T0[0] + lx) * g.Ng + (T0[1] + ly)) * H;
    if (k <= g.kzlim) mesh_store<NT>(orow + k, cadd(E, WO));
    if (M - k != k && M - k <= g.kzlim) {
      const float2 d = csub(E, WO);
      mesh_store<NT>(orow + (M - k), make_float2(d.x, -d.y));
    }
  }
}

template <int SCHEME>
hipError_t launch_deposit(const PshAssignGeom &g, size_t ntiles, size_t ntotal,
                          const uint32_t *starts, const Rec *recs,
                          size_t rec_cap, float *meshA, float *meshB,
                          size_t mstride, const int *flags, hipStream_t s) {
  // one grid per workgroup, except where the z transform is fused in
  const size_t cell = g.wide ? sizeof(long long) : sizeof(int);
  size_t cells = psh_tile_cells(g.tile, SCHEME) * (g.intlace && g.zfuse ? 2 : 1);
  // rows whose cells start on 16 bytes: a pitch of whole quads and `lead`
  // cells before the first, where the LDS holds them (the write-out then
  // reads quads: word by word, a wave's lanes stride 16 bytes and meet
  // four-fold in the banks)
  constexpr int W = SCHEME + 1;
  int pitch = psh_tile_pitch(g.tile[2], SCHEME), lead = 0;
  const size_t quads = (size_t)g.tile[0] * g.tile[1] * ((pitch + 3) & ~3) + 4;
  if (!g.zfuse && cell * quads <= 160 * 1024) {
    pitch = (pitch + 3) & ~3;
    lead = (4 - W % 4) % 4;
    cells = quads;
  }
  size_t lds = cell * cells;
  // non-temporal mesh stores when the launch's meshes outgrow the 256 MB
  // Infinity Cache (every cell is written once and read by the next pass
  // only after the whole launch)
  const bool stream = sizeof(float) * (size_t)g.tile[0] * g.tile[1] * g.tile[2] * ntiles *
                          (g.intlace ? 2 : 1) >
                      ((size_t)256 << 20);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  auto raise = [&](const void *k) {
    if (lds > 64 * 1024)
      (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  };
  if (g.zfuse) {
    // the fused z transform writes half-complex rows, 8 B per stored mode
    auto go = [&](auto nz) {
      constexpr int NZ = decltype(nz)::value;
      constexpr bool WD = ZfCfg<NZ, true>::WIDE;
      const int tx = g.intlace ? ZfCfg<NZ, true>::TX : ZfCfg<NZ, false>::TX;
      const int ty = g.intlace ? ZfCfg<NZ, true>::TY : ZfCfg<NZ, false>::TY;
      if (g.tile[0] != tx || g.tile[1] != ty || g.tile[2] != NZ || (g.wide != 0) != WD)
        return hipErrorInvalidValue;
      auto k = stream ? (g.intlace ? assign_deposit_z<SCHEME, true, WD, true, NZ>
                                   : assign_deposit_z<SCHEME, false, WD, true, NZ>)
                      : (g.intlace ? assign_deposit_z<SCHEME, true, WD, false, NZ>
                                   : assign_deposit_z<SCHEME, false, WD, false, NZ>);
      raise((const void *)k);
      hipLaunchKernelGGL(k, dim3((unsigned)ntiles), dim3(1024), lds, s, g, starts, recs, rec_cap,
                         meshA, meshB, mstride, flags);
      return hipGetLastError();
    };
    switch (g.Ng) {
      case 128: return go(std::integral_constant<int, 128>{});
      case 256: return go(std::integral_constant<int, 256>{});
      case 512: return go(std::integral_constant<int, 512>{});
      case 1024: return go(std::integral_constant<int, 1024>{});
      default: return hipErrorInvalidValue;
    }
  }
  auto k = stream ? (g.wide ? (g.intlace ? assign_deposit<SCHEME, true, true, true>
                                         : assign_deposit<SCHEME, false, true, true>)
                            : (g.intlace ? assign_deposit<SCHEME, true, false, true>
                                         : assign_deposit<SCHEME, false, false, true>))
                  : (g.wide ? (g.intlace ? assign_deposit<SCHEME, true, true, false>
                                         : assign_deposit<SCHEME, false, true, false>)
                            : (g.intlace ? assign_deposit<SCHEME, true, false, false>
                                         : assign_deposit<SCHEME, false, false, false>));
  // TSC in a launch of many tiles with 0.3 particles per cell and more: records
  // read once for both grids (deposit, one / both: N = 512, 1e8 particles in
  // space order 3.25 / 2.57 ms, shuffled 2.26 / 2.39; N = 640 2.84 / 2.65,
  // 2.24 / 2.39).  Fewer tiles leave the chip idle (N = 64 1.06 / 1.57) or
  // keep more of the second read in the caches (N = 256, 8e6 shuffled
  // 0.19 / 0.21); the other schemes are faster with one grid, or equal.
  bool both = false;
  if constexpr (SCHEME == 2) {
    both = g.intlace && !g.wide && ntiles >= 8192 && 2 * lds <= 160 * 1024 &&
           10 * ntotal >= 3 * ntiles * g.tile[0] * g.tile[1] * g.tile[2];
    if (both) {
      k = stream ? assign_deposit<2, true, false, true, true>
                 : assign_deposit<2, true, false, false, true>;
      lds *= 2;
    }
  }
  raise((const void *)k);
  // one thread per 16 cells (per 8 of 64 bits, whose LDS admits half the
  // workgroups: survey, N = 512, 1.89 -> 1.64 ms), 256..1024.  Two waves for
  // tiles of less than 2048 cells when there are so many of them that starting
  // the waves takes the time, twice what fills the chip: interlaced, both
  // grids in a workgroup of 256 / 256 for each / 128 for each: N = 256 CIC,
  // 2e4 particles, 4x4x4 0.24 / 0.43 / 0.24 ms; N = 512 in 4x4x64
  // 0.20 / 0.29 / 0.19, PCS 2e6 0.38 / 0.41 / 0.27; few tiles with many
  // records each want the waves: N = 64 in 4x4x64 PCS 2e6 0.41 / 0.23 / 0.44.
  const size_t tcells = (size_t)g.tile[0] * g.tile[1] * g.tile[2];
  const size_t blocks = ntiles * (g.intlace && !both ? 2 : 1);
  const size_t per = g.wide ? 8 : 16;
  unsigned threads = tcells < 2048 && blocks >= 8192 ? 128 : 256;
  while (threads < 1024 && threads * per < tcells) threads *= 2;
  // one launch, unless its threads pass the 32 bits that a launch counts them
  // in (both grids of N = 1024 in 4x4x4 tiles: 2^32)
  const size_t most = (0xffffffffu / threads) & ~15u;   // whole rounds of the XCDs
  for (size_t b0 = 0; b0 < blocks; b0 += most)
    hipLaunchKernelGGL(k, dim3((unsigned)std::min(most, blocks - b0)), dim3(threads), lds, s, g,
                       starts, recs, rec_cap, meshA, meshB, mstride, flags, pitch, lead,
                       (int)cells, (uint32_t)ntiles, (uint32_t)b0);
  return hipGetLastError();
}

}  // namespace

size_t psh_assign_record_bytes() { return sizeof(Rec); }

bool psh_zfuse_wide(int Ng) { return Ng <= 256; }

bool psh_zfuse_tile(int Ng, int intlace, int tile[3]) {
  auto set = [&](auto nz) {
    constexpr int NZ = decltype(nz)::value;
    tile[0] = intlace ? ZfCfg<NZ, true>::TX : ZfCfg<NZ, false>::TX;
    tile[1] = intlace ? ZfCfg<NZ, true>::TY : ZfCfg<NZ, false>::TY;
    tile[2] = NZ;
    return true;
  };
  switch (Ng) {
    case 128: return set(std::integral_constant<int, 128>{});
    case 256: return set(std::integral_constant<int, 256>{});
    case 512: return set(std::integral_constant<int, 512>{});
    case 1024: return set(std::integral_constant<int, 1024>{});
    default: return false;
  }
}

size_t psh_assign_whist_words(const PshAssignGeom &g, size_t ntotal) {
  const uint32_t tpm = (uint32_t)g.ntile[0] * g.ntile[1] * g.ntile[2];
  if (ntotal == 0 || (g.lean && tpm > (uint32_t)kWinTiles)) return 0;
  const size_t chunk = bucket_chunk(g, ntotal);
  const size_t words = (ntotal + chunk - 1) / chunk * window_tiles(tpm, ntotal);
  return words <= ((size_t)1 << 30) ? words : 0;   // at most 4 GB
}

hipError_t psh_fill_zero_u32(uint32_t *p, size_t n, hipStream_t s) {
  unsigned blocks = (unsigned)((n + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(fill_zero_u32, dim3(blocks), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t psh_exclusive_scan_u32(const uint32_t *in, uint32_t *out, uint32_t *tmp, size_t n,
                                  hipStream_t s) {
  if (n == 0) return hipErrorInvalidValue;
  return launch_scan<false>(in, out, nullptr, tmp, n, s);
}

size_t psh_assign_scan_bytes(size_t ntiles) {
  size_t nsb = (ntiles + kScanBlock - 1) / kScanBlock;
  return (nsb + 1) * sizeof(uint32_t);
}

namespace {
template <int SCHEME, bool IL>
hipError_t launch_bucket(bool fill, const PshAssignGeom &g, const PshDevPart *parts, int nparts,
                         size_t ntotal, uint32_t *counts, uint32_t *cursors,
                         const uint32_t *starts, Rec *recs, size_t rec_cap, int *flags,
                         uint32_t *whist, hipStream_t s) {
  const uint32_t tpm = (uint32_t)g.ntile[0] * g.ntile[1] * g.ntile[2];
  const size_t lds = sizeof(uint32_t) * window_tiles(tpm, ntotal);
  const uint32_t chunk = (uint32_t)bucket_chunk(g, ntotal);
  // two particles per thread at least, for the loads in flight
  unsigned threads = kBucketThreads;
  while (threads > 256 && threads * 2 > chunk) threads /= 2;
  auto k = fill ? assign_bucket<SCHEME, IL, true> : assign_bucket<SCHEME, IL, false>;
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
  hipLaunchKernelGGL(k, dim3((unsigned)((ntotal + chunk - 1) / chunk)), dim3(threads), lds, s, g,
                     parts, nparts, ntotal, chunk, counts, cursors, starts, recs, rec_cap, flags,
                     whist);
  return hipGetLastError();
}
}  // namespace

hipError_t psh_assign_run(const PshAssignGeom &g, PshDevPart *d_parts, const PshDevPart *h_parts,
                          int nparts, size_t ntotal, int nmock, uint32_t *counts,
                          uint32_t *starts, uint32_t *cursors, void *records, size_t rec_cap,
                          float *meshA, float *meshB, size_t mstride, uint32_t *d_scan_tmp,
                          int *d_flags, hipStream_t s, hipEvent_t ev_deposit, uint32_t *whist) {
  if (nparts < 1) return hipErrorInvalidValue;
  const size_t ntiles = (size_t)g.ntile[0] * g.ntile[1] * g.ntile[2] * nmock;
  hipError_t e;
  FewParts few{};
  if (h_parts && nparts <= kFewParts) {
    few.n = nparts;
    for (int i = 0; i < nparts; i++) few.p[i] = h_parts[i];
  } else if (h_parts) {
    if ((e = hipMemcpyAsync(d_parts, h_parts, sizeof(PshDevPart) * nparts,
                            hipMemcpyHostToDevice, s)) != hipSuccess)
      return e;
  }
  const size_t zb = (ntiles + 255) / 256;
  hipLaunchKernelGGL(assign_begin, dim3((unsigned)(zb < 1024 ? zb : 1024)), dim3(256), 0, s,
                     counts, cursors, ntiles, d_flags, d_parts, few);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  Rec *recs = reinterpret_cast<Rec *>(records);
  auto bucket = [&](bool fill) -> hipError_t {
    if (ntotal == 0) return hipSuccess;
    auto go = [&](auto scheme) {
      constexpr int S = decltype(scheme)::value;
      return g.intlace ? launch_bucket<S, true>(fill, g, d_parts, nparts, ntotal, counts, cursors,
                                                starts, recs, rec_cap, d_flags, whist, s)
                       : launch_bucket<S, false>(fill, g, d_parts, nparts, ntotal, counts,
                                                 cursors, starts, recs, rec_cap, d_flags, whist,
                                                 s);
    };
    switch (g.scheme) {
      case 0: return go(std::integral_constant<int, 0>{});
      case 1: return go(std::integral_constant<int, 1>{});
      case 2: return go(std::integral_constant<int, 2>{});
      default: return go(std::integral_constant<int, 3>{});
    }
  };
  if ((e = bucket(false)) != hipSuccess) return e;
  if ((e = launch_scan<true>(counts, starts, cursors, d_scan_tmp, ntiles, s)) != hipSuccess)
    return e;
  if ((e = bucket(true)) != hipSuccess) return e;
  if (ev_deposit) (void)hipEventRecord(ev_deposit, s);
  switch (g.scheme) {
    case 0: return launch_deposit<0>(g, ntiles, ntotal, starts, recs, rec_cap, meshA, meshB, mstride, d_flags, s);
    case 1: return launch_deposit<1>(g, ntiles, ntotal, starts, recs, rec_cap, meshA, meshB, mstride, d_flags, s);
    case 2: return launch_deposit<2>(g, ntiles, ntotal, starts, recs, rec_cap, meshA, meshB, mstride, d_flags, s);
    default: return launch_deposit<3>(g, ntiles, ntotal, starts, recs, rec_cap, meshA, meshB, mstride, d_flags, s);
  }
}
