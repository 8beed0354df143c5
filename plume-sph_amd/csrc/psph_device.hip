// psph_device.hip -- the per-step SPH particle path on one MI355X (gfx950).
//
// Data layout: structure-of-arrays in HBM, one array per particle field, all
// in "cell order" (particles sorted by the linear index of a uniform cell
// grid whose edge covers the largest kernel support).  Every step:
//   1. cell keys -> radix sort (key, index) -> gather every field (neighbours
//      are then contiguous: cell rows along x are contiguous index ranges);
//   2. targets (bc 100/99) are compacted and cut into "chunks" of <= 32
//      consecutive targets of a cell and "groups" of 8;
//   3. pair passes: one 64-lane wavefront per group, 8 targets x 8 streams of
//      candidates.  Per step and group, every tile (64 consecutive particles)
//      that can hold a pair gets a 64-bit mask of the particles that can be
//      one; a pass stages each such tile in LDS and evaluates the masked
//      particles, re-testing its own exact kernel box.  The reference's list
//      membership rule is evaluated per pair (same bucket, or |dx| <= 4.25 h_i
//      per axis) where the kernel box can reach past it.
// No MFMA: there is no dense contraction.  Reductions are deterministic
// (min/max via integer atomics on positive doubles; sums via fixed-order
// block partials).

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <type_traits>
#include <cmath>
#include <cstring>
#include <vector>

#include "psph_internal.h"

using namespace psph;

// A failed HIP call also leaves the thread's last-error state set; it is
// cleared here so that the error is reported once, by the return code, and not
// again by the next unrelated check of another user of the runtime (torch).
#define HIP_TRY(expr)                                                                        \
  do {                                                                                       \
    hipError_t e_ = (expr);                                                                  \
    if (e_ != hipSuccess) {                                                                  \
      (void)hipGetLastError();                                                               \
      return fail(PSPH_EHIP, "%s: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    }                                                                                        \
  } while (0)

#define PSPH_TRY(expr)            \
  do {                            \
    int rc_ = (expr);             \
    if (rc_) return rc_;          \
  } while (0)

namespace {

constexpr int kWave = 64;
constexpr uint32_t kXcds = 8;      // MI355X: 8 XCDs, each with its own L2
constexpr uint32_t kDead = 0xffffffffu;

// ---------------------------------------------------------------------------
// device-side error word: [0] = PSPH_E* code (0 = none), [1] = particle index
// ---------------------------------------------------------------------------
__device__ inline void raise_err(int *err, int code, uint32_t idx) {
  if (atomicCAS(err, 0, code) == 0) err[1] = (int)idx;
}

// The words of a context that kernels leave for the host, read in one copy: a
// step reads them where it needs them and not after every stage.
enum Word {
  W_DT, W_HMAX,               // bits of the least h / c and the largest h
  W_PAIRS, W_DEAD, W_REAL,    // pairs of the RHS; particles removed; real particles left
  W_BCOND,                    // groups of wall ghosts to refresh
  W_CURSOR, W_CHUNKS,         // visits handed out, chunks of targets
  W_LIVE, W_LIVE_REAL,
  W_ERR,                      // error words, [0] code and [1] particle: of the stages without one of
  W_ERR_RHS, W_ERR_DENS, W_ERR_VSM,   // their own, and of the passes whose errors a step reads at its end
  W_VMAX,                     // bits of the largest speed
  W_OVER, W_ITERS,            // lists that found no room since the last check; iterations of the adaptive h done
  W_ITER_CURSOR,              // and the cursors of their lists
  W_ITER_LAST = W_ITER_CURSOR + 7,
  W_COUNT
};
// an earlier stage of this step failed (n error words from err): the stages
// after it do nothing, as if the step had ended there
__device__ inline bool halted(const int *err, int n) {
  int bad = 0;
  for (int q = 0; q < n; q++) bad |= err[2 * q];
  return bad != 0;
}

__device__ inline bool need_neigh(int bc) { return bc == 100 || bc == 99; }
__device__ inline bool is_real(int bc) { return bc == 100 || bc == 99; }
__device__ inline bool contr_dens(int pg, int bc) {
  return bc == 100 || bc == 99 || (pg >= 1 && bc == 1) || (pg >= 2 && bc == 0);
}
__device__ inline bool contr_vel(int bc) { return bc == 100 || bc == 99 || bc == 2; }

// The reference tests abs(s_k) > CUTOFF with s_k = dx_k / h rounded to
// nearest.  Exactly equivalent and division-free: with u = half an ulp of cut,
// fl(|dx| / h) > cut  <=>  |dx| / h > cut + u (ties go to cut, whose last
// mantissa bit is even for cut = 3)  <=>  |dx| - cut h > u h.  The FMA gives
// round(|dx| - cut h); that difference is a multiple of ~h 2^-53, so it cannot
// lie within half an ulp of u h without equalling it, and the comparison of
// the rounded value with the representable u h is exact.  Applied to
// max_k |dx_k| it decides the whole box.
struct CutTest {
  double cut, u;
  __device__ inline bool outside(double amax, double h) const { return fma(-cut, h, amax) > u * h; }
};

// Closed-form EOS (particle.cc:528-604).
struct EosConst { double ng0, cvs, cvg, cva, rg, ra; int lans; };
__device__ inline void eos_dev(const EosConst &k, double rho, double e, double xi, double &p,
                               double &c, double &T, double &gam, double *cp) {
  double na = 1 - xi, ng = k.ng0 * xi, ns = xi - ng;
  double Cvm = ns * k.cvs + ng * k.cvg + na * k.cva;
  double Rm = ng * k.rg + na * k.ra;
  double Rmg = Rm / (ng + na);
  gam = 1 + Rm / Cvm;
  double desmg = rho * (na + ng);
  p = Rmg * desmg * e / Cvm;
  c = sqrt(gam * p / desmg);
  T = e / Cvm;
  if (k.lans) *cp = Cvm;
}

// ---------------------------------------------------------------------------
// simple kernels
// ---------------------------------------------------------------------------
__global__ void k_fill_u64(unsigned long long *p, unsigned long long v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_i32(int *p, int v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__device__ inline double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ inline double wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// Block-wide min / max of one value per thread (blockDim = 256); the
// result is valid in thread 0.  One atomic per block keeps the global
// update off a single contended address.
template <bool MAX>
__device__ inline double block_ext(double v) {
  __shared__ double part[4];
  v = MAX ? wave_max(v) : wave_min(v);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < 4; w++) v = MAX ? fmax(v, part[w]) : fmin(v, part[w]);
  return v;
}

// dt candidate min h/c over need_neigh particles (timestep.cc:94-135) and max h
// over the live ones; grid-stride, 256 threads per block.
__global__ __launch_bounds__(256) void k_dt_min(uint32_t n, const int32_t *bc, const double *h, const double *c,
                                                unsigned long long *words) {
  double v = 1.0e300, hm = 0;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int b = bc[i];
    if (b < 0) continue;
    const double hi = h[i];
    hm = fmax(hm, hi);
    if (!need_neigh(b)) continue;
    const double ci = c[i];
    if (!(ci > 0)) raise_err((int *)(words + W_ERR), PSPH_EINVARIANT, i);
    else v = fmin(v, hi / ci);
  }
  v = block_ext<false>(v);
  hm = block_ext<true>(hm);
  if (threadIdx.x != 0) return;
  if (v < 1.0e300) atomicMin(words + W_DT, (unsigned long long)__double_as_longlong(v));
  if (hm > 0) atomicMax(words + W_HMAX, (unsigned long long)__double_as_longlong(hm));
}
__global__ void k_step_words(unsigned long long *w) {
  if (threadIdx.x) return;
  w[W_DT] = 0x7FF0000000000000ull;                 // +inf
  w[W_HMAX] = w[W_PAIRS] = w[W_REAL] = w[W_VMAX] = 0;
}

// max h over live particles (the cell edge must cover every pair support)
__global__ __launch_bounds__(256) void k_h_max(uint32_t n, const int32_t *bc, const double *h, unsigned long long *out) {
  double v = 0;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    if (bc[i] >= 0) v = fmax(v, h[i]);
  v = block_ext<true>(v);
  if (threadIdx.x == 0 && v > 0) atomicMax(out, (unsigned long long)__double_as_longlong(v));
}

// Cell grid of the neighbour search.  Particles are sorted by
// (cell, Morton code of their position inside the cell at fbits bits per
// axis), so every cell is a contiguous index range and every run of 64
// consecutive particles of a cell (a "tile") is a compact cluster.
struct GridDesc {
  double lo[3];
  double inv_e;      // 1 / cell edge; 0: one cell holds everything
  int nx, ny, nz;
  uint32_t ncells;
  int fbits;
};

__device__ inline int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }
// floor((v - lo) * inv_e) clamped to [0, n - 1] without overflowing the int conversion
__device__ inline int cell_of(double v, double lo, double inv_e, int n) {
  const double f = floor((v - lo) * inv_e);
  return (int)fmin(fmax(f, 0.0), (double)(n - 1));
}

__global__ void k_cellkey(uint32_t n, const double *x, const double *y, const double *z,
                          const int32_t *bc, GridDesc g, uint32_t *key, uint32_t *idx) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  idx[i] = i;
  const int sh = 3 * g.fbits;
  if (bc[i] < 0) { key[i] = g.ncells << sh; return; }   // removed: sorts past every cell
  const double p[3] = {x[i], y[i], z[i]};
  const int nn[3] = {g.nx, g.ny, g.nz};
  int cc[3];
  uint32_t m = 0;
  const double nf = (double)(1 << g.fbits);
  for (int d = 0; d < 3; d++) {
    const double f = (p[d] - g.lo[d]) * g.inv_e;
    cc[d] = (int)fmin(fmax(floor(f), 0.0), (double)(nn[d] - 1));
    const int u = (int)fmin(fmax(floor((f - cc[d]) * nf), 0.0), nf - 1);
    for (int b = 0; b < g.fbits; b++) m |= (uint32_t)((u >> b) & 1) << (3 * b + d);
  }
  key[i] = ((((uint32_t)cc[2] * g.ny + cc[1]) * g.nx + cc[0]) << sh) | m;
}

// dst[i] = src[perm[i]] for N8 arrays of 8 bytes an element and N4 of 4: the
// index is read once and a thread has all its loads in flight (a launch per
// array: 75 us of a step at 240k particles, 615 us at 6.8M; so 26 and 441).
constexpr int kMove8 = 11, kMove4 = 7;
struct Moves {
  const uint64_t *s8[kMove8];
  uint64_t *d8[kMove8];
  const uint32_t *s4[kMove4];
  uint32_t *d4[kMove4];
};
template <int N8, int N4>
__global__ void k_gather(uint32_t n, const uint32_t *perm, Moves mv) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t from = perm[i];
  uint64_t v8[N8 ? N8 : 1];
  uint32_t v4[N4 ? N4 : 1];
#pragma unroll
  for (int k = 0; k < N8; k++) v8[k] = mv.s8[k][from];
#pragma unroll
  for (int k = 0; k < N4; k++) v4[k] = mv.s4[k][from];
#pragma unroll
  for (int k = 0; k < N8; k++) mv.d8[k][i] = v8[k];
#pragma unroll
  for (int k = 0; k < N4; k++) mv.d4[k][i] = v4[k];
}

// Reference bucket (preprocessor cells of edge 8 h_air, preprocess.cc:88-133)
// as packed coordinates: x in bits 0-9, y in bits 11-20, z in bits 22-31 (at
// most 1023 buckets per axis; kDead outside the grid).  A list holds the own
// bucket's particles and, from the 26 adjacent buckets, those within the
// list box (neighs.cc:37-211).
constexpr int kRefbMaxPerAxis = 1023;
__device__ inline uint32_t refb_pack(uint32_t x, uint32_t y, uint32_t z) { return x | (y << 11) | (z << 22); }
// buckets at most one apart on every axis: per field 1024 + a - b + 1 (the
// guard bits 10 and 21 stop borrows between fields), (a - b + 1) mod 1024 for z
__device__ inline bool refb_adjacent(uint32_t a, uint32_t b) {
  const uint32_t d = ((a | 0x00200400u) - b) + 0x00400801u;
  return (a != kDead) & (b != kDead) & ((d & 0x7ffu) - 1024u <= 2u) & (((d >> 11) & 0x7ffu) - 1024u <= 2u) & ((d >> 22) <= 2u);
}

// copies of n8 arrays of 8 bytes an element and n4 of 4, n elements each
__global__ void k_copy(uint32_t n, int n8, int n4, Moves mv) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int k = 0; k < kMove8; k++)
    if (k < n8) mv.d8[k][i] = mv.s8[k][i];
#pragma unroll
  for (int k = 0; k < kMove4; k++)
    if (k < n4) mv.d4[k][i] = mv.s4[k][i];
}

// After the sort: cs[c] = first index whose cell (key >> sh) >= c, c in [0,
// ncells]; the smoothing length at list time; the reference bucket.  Empty cells
// that follow each other are filled by the whole wave (one lane alone took 11 us
// at 65k particles of 1.7k targets).
struct RefBuckets { double lo[3], del; int nb[3]; };
__global__ void k_sorted(uint32_t n, const uint32_t *key, int sh, uint32_t ncells, uint32_t *cs, const double *x,
                         const double *y, const double *z, const double *h, RefBuckets b, uint32_t *refb, double *h_list) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool here = i <= n;
  uint32_t prev = 0, cur = 0;
  if (here) {
    prev = (i == 0) ? 0u : min(key[i - 1] >> sh, ncells) + 1u;
    cur = (i == n) ? ncells + 1u : min(key[i] >> sh, ncells) + 1u;
  }
  const bool many = cur > prev + 4;
  if (!many)
    for (uint32_t c = prev; c < cur; c++) cs[c] = i;
  uint64_t left = __ballot(many);
  while (left) {
    const int l = __builtin_ctzll(left);
    left &= left - 1;
    const uint32_t a = __builtin_amdgcn_readlane(prev, l), e = __builtin_amdgcn_readlane(cur, l);
    const uint32_t at = __builtin_amdgcn_readlane(i, l);
    for (uint32_t c = a + threadIdx.x % kWave; c < e; c += kWave) cs[c] = at;
  }
  if (i >= n) return;
  const double fx = floor((x[i] - b.lo[0]) / b.del), fy = floor((y[i] - b.lo[1]) / b.del),
               fz = floor((z[i] - b.lo[2]) / b.del);
  uint32_t r = kDead;
  if (fx >= 0 && fx < b.nb[0] && fy >= 0 && fy < b.nb[1] && fz >= 0 && fz < b.nb[2])
    r = refb_pack((uint32_t)fx, (uint32_t)fy, (uint32_t)fz);
  refb[i] = r;
  h_list[i] = h[i];
}

// indices whose flag is set, in order (tpos: the flags' sums)
__global__ void k_targets(uint32_t n, const uint32_t *flags, const uint32_t *tpos, uint32_t *targets) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && flags[i]) targets[tpos[i]] = i;
}

// ---------------------------------------------------------------------------
// Pair-pass skeleton
// ---------------------------------------------------------------------------
// Cells and tiles a wavefront's chunk of particles must visit: the chunk's
// bounding box grown by `reach` (the largest per-axis pair distance any
// predicate of the pass can accept) selects a block of cells, and of their
// tiles only those whose box meets the grown box.  Every candidate within
// reach of a chunk particle lies in such a tile.
struct Traversal {
  const uint32_t *cs, *toff;
  const float4 *tbox;
  GridDesc g;
  double reach;
};

struct ChunkBox {
  int c0[3], c1[3];
  float lo[3], hi[3];
};

__device__ inline bool tile_meets(const ChunkBox &b, const float4 *tbox, uint32_t t) {
  const float4 lo = tbox[2 * t], hi = tbox[2 * t + 1];
  return !(lo.x > b.hi[0] || hi.x < b.lo[0] || lo.y > b.hi[1] || hi.y < b.lo[1] || lo.z > b.hi[2] || hi.z < b.lo[2]);
}

struct PairCommon {
  const double *x, *y, *z;     // positions of the predicates (cells, boxes, tests)
  const double *ax, *ay, *az;  // positions of the pair arithmetic (the same arrays
                               // except in a frozen replay, Tape::xrec)
  const uint32_t *refb;
  const double *h_list;
  const int32_t *bc;
  uint32_t *gflag;            // optional: marks boundary ghosts (bc 1, 2) met as neighbours
  Traversal tr;
  const uint32_t *targets;
  const uint32_t *cfirst, *ccount, *nchunks;
  int list_all;
  int list_adj;               // some list box may reach past the adjacent buckets
  double list_factor;
  double del;                 // reference bucket edge
  double ext_lo[3];           // origin of the reference buckets
  CutTest cut;
  int *err;
  const int *halt;            // error words of the stages before this pass
  int nhalt;
};

// The region a chunk's neighbour lists can reach (neighs.cc:37-211): per
// target its own reference bucket and, within the adjacent buckets, its list
// box; the chunk's box is their union, with a margin for the rounding of the
// bucket index (1e-9 of a bucket).  It is often much smaller than the
// traversal's reach, which has to bound the largest list box of all.
__device__ inline ChunkBox chunk_list_box(const PairCommon &pc, const double *p, double lf, uint32_t rb) {
  ChunkBox b;
  const int nn[3] = {pc.tr.g.nx, pc.tr.g.ny, pc.tr.g.nz};
  const uint32_t bk[3] = {rb & 1023u, (rb >> 11) & 1023u, rb >> 22};
  const double m = 1e-9 * pc.del;
  for (int d = 0; d < 3; d++) {
    double lo, hi;
    if (rb == kDead || pc.list_all) {
      lo = p[d] - pc.tr.reach;
      hi = p[d] + pc.tr.reach;
    } else {
      const double blo = pc.ext_lo[d] + bk[d] * pc.del, bhi = blo + pc.del;
      lo = fmin(fmax(p[d] - lf, blo - pc.del), blo) - m;
      hi = fmax(fmin(p[d] + lf, bhi + pc.del), bhi) + m;
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    b.lo[d] = __double2float_rd(lo);
    b.hi[d] = __double2float_ru(hi);
    if (pc.tr.g.inv_e > 0) {
      b.c0[d] = cell_of(lo, pc.tr.g.lo[d], pc.tr.g.inv_e, nn[d]);
      b.c1[d] = cell_of(hi, pc.tr.g.lo[d], pc.tr.g.inv_e, nn[d]);
    } else {
      b.c0[d] = b.c1[d] = 0;
    }
  }
  return b;
}

// A chunk: up to kChunk targets, consecutive in the order of the cell's targets, so
// they sit within ~2 particle spacings of each other and the union of their
// neighbourhoods is little more than one of them.
constexpr double kFar = 1.0e300;
constexpr int kChunk = kWave / 2;

// List materialisation (parity checks only): one wavefront per chunk, a target a
// lane.  The candidates accepted are exactly the reference's list
// (neighs.cc:37-211).  out null counts, else device indices are written from
// offset[i] on.
template <int D>
__global__ __launch_bounds__(kWave) void k_list(PairCommon pc, uint32_t *count, const uint32_t *offset, uint32_t *out) {
  __shared__ double sx[kWave], sy[kWave], sz[kWave];
  __shared__ uint32_t srefb[kWave];
  const uint32_t chunk = blockIdx.x;
  if (chunk >= *pc.nchunks) return;
  const uint32_t cf = pc.cfirst[chunk], cc = pc.ccount[chunk];
  const uint32_t lane = threadIdx.x;
  const bool active = lane < cc;
  const uint32_t i = pc.targets[cf + (active ? lane : 0)];
  const double xi[3] = {pc.x[i], pc.y[i], pc.z[i]};
  const uint32_t rb = pc.refb[i];
  const double lf = pc.list_factor * pc.h_list[i];
  const ChunkBox box = chunk_list_box(pc, xi, lf, rb);
  const GridDesc &g = pc.tr.g;
  uint32_t n = 0, o = active && out ? offset[i] : 0;
  for (int cz = box.c0[2]; cz <= box.c1[2]; cz++)
    for (int cy = box.c0[1]; cy <= box.c1[1]; cy++)
      for (int cx = box.c0[0]; cx <= box.c1[0]; cx++) {
        const uint32_t cell = ((uint32_t)cz * g.ny + cy) * g.nx + cx;
        const uint32_t je = pc.tr.cs[cell + 1];
        uint32_t tl = pc.tr.toff[cell];
        for (uint32_t base = pc.tr.cs[cell]; base < je; base += kWave, tl++) {
          if (!tile_meets(box, pc.tr.tbox, tl)) continue;
          const uint32_t js = min(base + lane, je - 1);
          sx[lane] = pc.x[js]; sy[lane] = pc.y[js]; sz[lane] = pc.z[js];
          srefb[lane] = pc.refb[js];
          __syncthreads();
          const uint32_t cnt = active ? min((uint32_t)kWave, je - base) : 0;
          for (uint32_t q = 0; q < cnt; q++) {
            double amax = fabs(xi[0] - sx[q]);
            if (D == 3) amax = fmax(amax, fmax(fabs(xi[1] - sy[q]), fabs(xi[2] - sz[q])));
            // same bucket or the 4.25 h_i box (neighs.cc:37-211)
            bool in = (amax <= lf) & ((pc.list_adj == 0) | refb_adjacent(srefb[q], rb));
            in |= (srefb[q] == rb) | (pc.list_all != 0);
            if (!in) continue;
            if (out) out[o + n] = base + q;
            n++;
          }
          __syncthreads();
        }
      }
  if (active && !out) count[i] = n;
}

// ---------------------------------------------------------------------------
// Group passes.  The RHS, density, filter and adaptive-h passes take their targets in
// groups of kGroup consecutive targets of a cell, one wavefront per group.  For
// every group and tile that can hold a pair of it, a 64-bit mask made once per
// step says which of the tile's particles can be a pair of one of the group's
// targets in any of the passes.  A pass stages the tile in LDS, queues the
// masked particles, and evaluates kStreams of them at a time against all
// kGroup targets: lane = target + kGroup * stream, so a lane keeps its target
// and its partial sums in registers and reads a particle's record from LDS, and
// each pair re-tests the pass's exact kernel box.
//
// Why 8 x 8: the larger the group, the fewer staged tiles a target costs, but
// the fewer of the queued particles are pairs of a given target.  On the
// lattice after an adaptation (3 h = 4.5 spacings) 55-62 % of the evaluated
// lanes are pairs with 8 targets, 65-69 % with 4, 46-54 % with 16; walking bit
// masks of 32 targets x 2 lanes, where a wave ran as long as its fullest lane,
// had 41 %.
// Measured and not kept: a record per lane held against 4 targets in turn, the
// records gathered from the caches (65-76 cycles of the return path per 16-byte
// load, which kept it busy 90 % of the density and filter passes) or from
// windows of tiles that 4 or 8 waves stage together (60 % of the wave time went
// into the windows' barriers); the next tile through registers while one is
// worked on (density and filter 7.5 -> 25 ms at 4M).
// Against the masks of 32 targets x 2 lanes, us per launch (RHS, density, filter,
// masks): 1M FP64 6808, 3168, 2589, 563 (before: 8257, 3894, 3049, 992); 4M
// FP32-exp 14990, 7235, 6838, 1939 (18057, 8047, 6634, 3843); 1.7k FP64 in 65k
// particles, where 54 waves of 32 targets left the chip idle, 112, 75, 68, 22
// (508, 299, 273, 151), and 32, 19, 17 with 8 waves a group.
// ---------------------------------------------------------------------------
constexpr int kGroup = 8;                      // targets of a group
constexpr int kStreams = kWave / kGroup;       // particles evaluated at a time
constexpr int kGroupsPerChunk = kChunk / kGroup;
constexpr int kMaxSplit = 8;                   // waves that share a group

// Positions (x, y) and (z, h / 2) of every particle; the lists made next start at visit 0.
struct Geom {
  const double2 *xy, *zh;
};

__global__ void k_geom(uint32_t n, const double *x, const double *y, const double *z, const double *h, double2 *xy,
                       double2 *zh, unsigned long long *cursor) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *cursor = 0;
  if (i >= n) return;
  xy[i] = make_double2(x[i], y[i]);
  zh[i] = make_double2(z[i], 0.5 * h[i]);
}

// m &= ~(1 << b) for a wave-uniform 64-bit mask in scalar registers: one
// s_bitset0_b64 (the and-not of a shifted one takes two scalar instructions)
__device__ inline void clear_bit_u(uint64_t &m, uint32_t b) {
  asm volatile("s_bitset0_b64 %0, %1" : "+s"(m) : "s"(b));
}

// v = value in lane `lane` only (value and lane wave-uniform): one
// v_writelane_b32, which ignores EXEC.  With the value in a scalar register
// the lane select goes through M0 (one scalar operand per VALU instruction).
// M0 is written by a scalar move, so the lane select has no VALU-write
// hazard; the asm touches registers only (M0 declared clobbered).  lane < 64.
__device__ inline void set_lane(uint32_t &v, uint32_t value, uint32_t lane) {
  asm volatile("s_mov_b32 m0, %2\n\tv_writelane_b32 %0, %1, m0" : "+v"(v) : "s"(value), "s"(lane) : "m0");
}

__device__ inline uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// v of lane ^ (the lanes of a row of 16), by DPP moves
template <int CTRL>
__device__ inline double row_move(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
// v_permlane32_swap exchanges a's upper half with b's lower, v_permlane16_swap
// a's odd rows with b's even ones: the sum of the two results then holds a's
// partial sums on one half (the even rows) and b's on the other.
template <int ROWS>
__device__ inline double swap_add(double a, double b) {
  const uint64_t x = (uint64_t)__double_as_longlong(a), y = (uint64_t)__double_as_longlong(b);
  auto lo = ROWS == 2 ? __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)y, false, false)
                      : __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
  auto hi = ROWS == 2 ? __builtin_amdgcn_permlane32_swap((uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false)
                      : __builtin_amdgcn_permlane16_swap((uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
  return __longlong_as_double((long long)((uint64_t)hi[0] << 32 | lo[0])) +
         __longlong_as_double((long long)((uint64_t)hi[1] << 32 | lo[1]));
}
// The order of a cell's targets in which the group passes take them kGroup at a
// time: runs of up to kRun consecutive targets are halved along the longest side
// of their box, the halves likewise, down to groups, so that a group's box is
// small.  In the Morton order of the cells alone 8 consecutive targets of a
// lattice share 55 % of their grown boxes (of a disordered set 52 %), so halved
// 61 % (59 %): so many fewer pair blocks have lanes without a pair.
// One wavefront per run, two targets a lane; a target's place is the number of
// its segment's smaller keys, each key a coordinate's upper bits above the place
// it had (no two are equal).  Bound by that count: a chain of LDS reads where
// cells are few (the whole of k_cell_fill 18 us at 1.7k targets), 140 us at 4M.
// us per launch without and with it (RHS, density, filter): 1M FP64 7124, 3159,
// 2593 / 6270, 2710, 2240; 4M FP32-exp 15203, 8077, 7212 / 13390, 7080, 6300.
constexpr int kRun = 2 * kWave;
// the order of floats as an order of integers, and back; a NaN goes last
__device__ inline uint32_t order_key(float f, uint32_t place) {
  const uint32_t u = __float_as_uint(f == f ? f : INFINITY);
  return ((u ^ (uint32_t)((int32_t)u >> 31 | (int32_t)0x80000000)) & ~(uint32_t)(kRun - 1)) | place;
}
__device__ inline float order_value(uint32_t k) {
  k &= ~(uint32_t)(kRun - 1);
  return __uint_as_float(k ^ ((int32_t)k < 0 ? 0x80000000u : 0xffffffffu));
}

// what this wave wrote to LDS is there for its other lanes
__device__ inline void wave_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// the n places' segments of 2 HALF: each becomes its lower and its upper half
template <int HALF>
__device__ inline void halve_segments(uint32_t lane, uint32_t n, uint32_t (&key)[3][kRun], uint32_t *id) {
  if (n <= HALF) return;                            // (uniform) one segment, no longer than its half
  constexpr int kAcross = 2 * HALF < kWave ? 2 * HALF : kWave;
  uint32_t own[2][3], to[2], who[2], lo[2][3], up[2][3];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const uint32_t p = lane + q * kWave;
    who[q] = id[p];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      own[q][d] = key[d][p];                        // (all ones past the last place)
      lo[q][d] = own[q][d];
      up[q][d] = p < n ? own[q][d] : 0u;
    }
  }
#pragma unroll
  for (int d = 0; d < 3; d++) {
    if (HALF == kWave) {
      lo[0][d] = lo[1][d] = min(lo[0][d], lo[1][d]);
      up[0][d] = up[1][d] = max(up[0][d], up[1][d]);
    }
#pragma unroll
    for (int o = 1; o < kAcross; o <<= 1)
#pragma unroll
      for (int q = 0; q < (HALF == kWave ? 1 : 2); q++) {
        lo[q][d] = min(lo[q][d], (uint32_t)__shfl_xor((int)lo[q][d], o));
        up[q][d] = max(up[q][d], (uint32_t)__shfl_xor((int)up[q][d], o));
      }
    if (HALF == kWave) { lo[1][d] = lo[0][d]; up[1][d] = up[0][d]; }
  }
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const uint32_t p = lane + q * kWave, s0 = p & ~(2u * HALF - 1u);
    const float ex = order_value(up[q][0]) - order_value(lo[q][0]);
    const float ey = order_value(up[q][1]) - order_value(lo[q][1]);
    const float ez = order_value(up[q][2]) - order_value(lo[q][2]);
    const int axis = ex >= ey && ex >= ez ? 0 : ey >= ez ? 1 : 2;
    const uint32_t mine = axis == 0 ? own[q][0] : axis == 1 ? own[q][1] : own[q][2];
    const uint4 *keys = (const uint4 *)&key[axis][s0];
    uint32_t below = 0;
#pragma unroll 8
    for (int j = 0; j < HALF / 2; j++) {
      const uint4 k = keys[j];
      below += k.x < mine ? 1u : 0u;
      below += k.y < mine ? 1u : 0u;
      below += k.z < mine ? 1u : 0u;
      below += k.w < mine ? 1u : 0u;
    }
    // a segment no longer than its half stays as it is
    to[q] = min(s0 + 2 * HALF, n) <= s0 + HALF ? p : s0 + below;
  }
  wave_sync();
#pragma unroll
  for (int q = 0; q < 2; q++)
    if (lane + q * kWave < n) {
      id[to[q]] = who[q];
#pragma unroll
      for (int d = 0; d < 3; d++) key[d][to[q]] = (own[q][d] & ~(uint32_t)(kRun - 1)) | to[q];
    }
  wave_sync();
}

struct OrderLds {
  uint32_t key[3][kRun], id[kRun];
};
// one run: t[0..n), n <= kRun
__device__ inline void order_run(uint32_t lane, uint32_t n, const double *x, const double *y, const double *z,
                                 uint32_t *t, OrderLds &o) {
  static_assert(kRun == 2 * kWave && kGroup == 8, "halves of 64 to 8 places");
  const uint32_t first = t[0];
  const double org[3] = {x[first], y[first], z[first]};
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const uint32_t p = lane + q * kWave, i = t[min(p, n - 1)];
    const double at[3] = {x[i], y[i], z[i]};
    o.id[p] = i;
#pragma unroll
    for (int d = 0; d < 3; d++) o.key[d][p] = p < n ? order_key((float)(at[d] - org[d]), p) : ~0u;
  }
  wave_sync();
  halve_segments<64>(lane, n, o.key, o.id);
  halve_segments<32>(lane, n, o.key, o.id);
  halve_segments<16>(lane, n, o.key, o.id);
  halve_segments<8>(lane, n, o.key, o.id);
  for (uint32_t p = lane; p < n; p += kWave) t[p] = o.id[p];
  wave_sync();
}

// What a cell holds, and the sums of it over the cells before: tiles (64
// consecutive particles each), targets, chunks of kChunk consecutive targets.
struct CellSum { uint32_t tiles, targets, chunks; };
struct CellAdd {
  __host__ __device__ CellSum operator()(const CellSum &a, const CellSum &b) const {
    return CellSum{a.tiles + b.tiles, a.targets + b.targets, a.chunks + b.chunks};
  }
};
struct IsTarget {
  const int32_t *bc;
  __device__ bool operator()(uint32_t i) const { return need_neigh(bc[i]); }
};

// The particles of part p, one wavefront's: the cell p, or, where one cell holds
// everything, its kRun particles from p kRun on (a workgroup of 1024 for the whole
// cell took 80 us at 6.9k particles, 15 us so).  Tiles, chunks and runs start anew
// in each part, which is on their bounds where it is kRun particles.
__device__ inline void part_range(uint32_t p, uint32_t parts, bool one_cell, const uint32_t *cs, uint32_t &lo, uint32_t &hi) {
  if (one_cell) {
    lo = min(p * (uint32_t)kRun, cs[1]);
    hi = min(lo + (uint32_t)kRun, cs[1]);
  } else {
    lo = cs[p];
    hi = p < parts ? cs[p + 1] : lo;
  }
}

// (One part more, empty, for the scan.)
template <class T>
__global__ __launch_bounds__(kWave) void k_cell_counts(uint32_t parts, bool one_cell, const uint32_t *cs, T is, CellSum *out) {
  uint32_t lo, hi;
  part_range(blockIdx.x, parts, one_cell, cs, lo, hi);
  if (blockIdx.x == parts) hi = lo;
  uint32_t cnt = 0;
  for (uint32_t i = lo + threadIdx.x; i < hi; i += kWave) cnt += is(i) ? 1u : 0u;
  for (int o = kWave / 2; o > 0; o >>= 1) cnt += (uint32_t)__shfl_xor((int)cnt, o);
  if (threadIdx.x == 0) out[blockIdx.x] = CellSum{(hi - lo + kWave - 1) / kWave, cnt, (cnt + kChunk - 1) / kChunk};
}

// The part's tiles with their boxes, rounded outwards to float: [lo, hi] per tile,
// and in the w components the bits of its first particle and its particle count
// (toff null: not these); its targets, in the order of the passes; its chunks.
// (Counts, scans and lists in kernels of their own over particles, tiles and cells:
// 15 launches of a search; so 5.)
template <class T>
__global__ __launch_bounds__(kWave) void k_cell_fill(uint32_t parts, bool one_cell, const uint32_t *cs, T is,
                                                     const CellSum *sums, uint32_t *toff, float4 *tbox, const double *x,
                                                     const double *y, const double *z, uint32_t *targets,
                                                     uint32_t *cfirst, uint32_t *ccount, uint32_t *nchunks) {
  __shared__ __align__(16) OrderLds order;
  const uint32_t part = blockIdx.x, lane = threadIdx.x;
  uint32_t lo, hi;
  part_range(part, parts, one_cell, cs, lo, hi);
  const CellSum at = sums[part], to = sums[part + 1];
  if (lane == 0) {
    if (toff && (!one_cell || part == 0)) toff[part] = at.tiles;
    if (part == parts - 1) {
      if (toff) toff[one_cell ? 1u : parts] = to.tiles;
      *nchunks = to.chunks;
    }
  }
  for (uint32_t t = at.tiles; toff && t < to.tiles; t++) {
    const uint32_t base = lo + kWave * (t - at.tiles), end = min(hi, base + kWave);
    const uint32_t j = base + lane < end ? base + lane : base;
    const double px = x[j], py = y[j], pz = z[j];
    const double ax = wave_min(px), ay = wave_min(py), az = wave_min(pz);
    const double bx = wave_max(px), by = wave_max(py), bz = wave_max(pz);
    if (lane == 0) {
      tbox[2 * t] = make_float4(__double2float_rd(ax), __double2float_rd(ay), __double2float_rd(az), __uint_as_float(base));
      tbox[2 * t + 1] = make_float4(__double2float_ru(bx), __double2float_ru(by), __double2float_ru(bz),
                                    __uint_as_float(end - base));
    }
  }
  const uint32_t nt = to.targets - at.targets;
  if (!nt) return;
  for (uint32_t q = lane; q < to.chunks - at.chunks; q += kWave) {
    cfirst[at.chunks + q] = at.targets + q * kChunk;
    ccount[at.chunks + q] = min((uint32_t)kChunk, nt - q * kChunk);
  }
  uint32_t next = at.targets;
  for (uint32_t i0 = lo; i0 < hi; i0 += kWave) {
    const bool mine = i0 + lane < hi && is(i0 + lane);
    const uint64_t m = __ballot(mine);
    if (mine) targets[next + lanes_below(m)] = i0 + lane;
    next += (uint32_t)__popcll(m);
  }
  __threadfence_block();
  __syncthreads();                                 // the part's targets are there
  for (uint32_t t0 = 0; t0 < nt; t0 += kRun)
    if (nt - t0 > (uint32_t)kGroup) order_run(lane, min((uint32_t)kRun, nt - t0), x, y, z, targets + at.targets + t0, order);
}

// The tiles a group visits, with a 64-bit mask of the particles that can be a
// pair of one of its targets in any of the passes.
struct GroupLists {
  uint4 *visit;             // x, y: first particle and count of the tile; z, w: the mask
  uint32_t *off, *num;      // per group: first visit, visits
  uint32_t *fast;           // per group: list membership and in_support cannot fail for a masked
                            // particle inside a pass's kernel box
  unsigned long long *cursor;   // visits handed out
  uint32_t cap;             // visits that visit holds
};

struct GroupCommon {
  Geom g;
  GroupLists gl;
  double cutx;               // cut with a relative margin of 1e-12
  double cutj;               // of a particle's h / 2: cutx, or 2 cutx for lists of both roles
  double h_max;
  int both;                  // lists of the adjoint: kernel boxes of the larger h of a pair
  // lists for an iteration of the adaptive h: the kernel's h over h (0: lists
  // for the three passes) and the targets that have converged
  double c_smooth;
  const uint32_t *done;
  // optional: set where the visits found no room, by lists whose cursor the host
  // does not read before the pass; the pass then does nothing, else counts itself
  unsigned long long *over;
};

// The group of this workgroup, its target for this lane (lane % kGroup; past
// the last target the lanes repeat it) and the number of its targets; 0 for none.
__device__ inline uint32_t my_group(const PairCommon &pc, uint32_t &gid, uint32_t &i) {
  const uint32_t ngr = *pc.nchunks * kGroupsPerChunk;
  const uint32_t per = (ngr + kXcds - 1) / kXcds;
  const uint32_t local = blockIdx.x / kXcds;
  if (local >= per) return 0;
  gid = (blockIdx.x % kXcds) * per + local;
  if (gid >= ngr) return 0;
  const uint32_t chunk = gid / kGroupsPerChunk, t0 = gid % kGroupsPerChunk * kGroup;
  const uint32_t cc = pc.ccount[chunk];
  if (t0 >= cc) return 0;
  const uint32_t nt = min((uint32_t)kGroup, cc - t0);
  i = pc.targets[pc.cfirst[chunk] + t0 + min(threadIdx.x % kGroup, nt - 1u)];
  return nt;
}

__device__ inline double group_min(double v) {
  for (int o = 1; o < kGroup; o <<= 1) v = fmin(v, __shfl_xor(v, o));
  return v;
}
__device__ inline double group_max(double v) {
  for (int o = 1; o < kGroup; o <<= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}

// |x_k - c_k| - b_k <= max(chh + cutj h_j / 2, ch) holds on every axis for each
// particle j that is a pair of one of the group's targets in any of the passes
// (b with room for the rounding of c and of the differences).
struct GroupBox {
  double c[3], b[3];
  double chh, ch;            // cutx h / 2 (both roles: 0) and cutx h of the group's largest h
  float lo[3], up[3];        // the grown box
};

// One wavefront per share of a chunk: kGroupsPerChunk / nsplit groups.  The
// tiles whose box meets a group's grown box are counted to find room for the
// visits, then their particles are read, once for all the wave's groups, and
// tested.  A wave that finds no room only counts: the host grows the array and
// calls again.  A whole chunk per wave reads a tile once for four groups (at 4M
// the reads of one group per wave ran at 8 TB/s of L2: 6.1 ms against 3.8); a
// small set of particles has too few chunks to fill the chip and takes a group
// per wave.
template <int D>
__global__ __launch_bounds__(kWave) void k_group_lists(PairCommon pc, GroupCommon gc, const double *h, double cutoff2,
                                                       uint32_t nsplit) {
  __shared__ GroupBox gb[kGroupsPerChunk];
  __shared__ uint32_t rowpre[kWave], rowtile[kWave];
  const uint32_t units = *pc.nchunks * nsplit;
  const uint32_t per = (units + kXcds - 1) / kXcds;
  const uint32_t local = blockIdx.x / kXcds;
  if (local >= per) return;
  const uint32_t unit = (blockIdx.x % kXcds) * per + local;
  if (unit >= units) return;
  const uint32_t chunk = unit / nsplit, share = kGroupsPerChunk / nsplit, g0 = unit % nsplit * share;
  const uint32_t cc = pc.ccount[chunk];
  if (g0 * kGroup >= cc) return;
  const uint32_t ng = min(share, (cc - g0 * kGroup + kGroup - 1) / kGroup);
  const int lane = threadIdx.x;
  // kGroup lanes own a group's targets; past the last target they repeat it
  const uint32_t i = pc.targets[pc.cfirst[chunk] + min(g0 * kGroup + min((uint32_t)lane, ng * kGroup - 1u), cc - 1u)];
  const GridDesc &g = pc.tr.g;
  const int nn[3] = {g.nx, g.ny, g.nz};
  int c0[3] = {0, 0, 0}, c1[3] = {0, 0, 0};
  bool fast;
  {
    const double xi[3] = {pc.x[i], pc.y[i], pc.z[i]};
    const double hi = h[i];
    const double lf = pc.list_factor * pc.h_list[i], supp = cutoff2 * hi;
    // fast: the widest kernel box of the passes lies inside the list box and the
    // in_support box of every target and is narrower than a bucket, so that list
    // membership and in_support cannot fail for a particle inside it
    GroupBox B;
    double widest;
    bool in = true;                  // the target takes part
    if (gc.c_smooth > 0) {
      // the kernel box of c_smooth h_i, and of the list no particle beyond its
      // box and the target's bucket
      const double hs = hi * gc.c_smooth;
      const double box = gc.cutx * hs;
      fast = box <= cutoff2 * hs && (pc.list_all != 0 || (box <= lf && box * (1 + 1e-12) < pc.del));
      in = gc.done[i] == 0;
      const double w = pc.list_all ? box : fmin(box, fmax(lf, pc.del * (1 + 1e-9)));
      B.chh = -HUGE_VAL;
      B.ch = group_max(in ? w : 0.0);
      widest = B.ch * (1 + 1e-9);
    } else if (gc.both) {
      // |x_k - x_j| <= cutx max(h_i, h_j)
      fast = false;
      B.ch = gc.cutx * group_max(hi);
      B.chh = 0;
      widest = fmax(B.ch, gc.cutx * gc.h_max) * (1 + 1e-9);
    } else {
      widest = gc.cutx * fmax(0.5 * hi + 0.5 * gc.h_max, hi);
      fast = widest <= supp && (pc.list_all != 0 || (widest <= lf && widest * (1 + 1e-12) < pc.del));
      const double hg = group_max(hi);
      widest = gc.cutx * fmax(0.5 * hg + 0.5 * gc.h_max, hg) * (1 + 1e-9);
      B.chh = gc.cutx * (0.5 * hg);
      B.ch = gc.cutx * hg;
    }
    for (int d = 0; d < 3; d++) {
      const double lo = group_min(in ? xi[d] : kFar), up = group_max(in ? xi[d] : -kFar);
      B.c[d] = 0.5 * lo + 0.5 * up;
      B.b[d] = fmax(up - B.c[d], B.c[d] - lo);
      B.b[d] += 2e-15 * (fabs(B.c[d]) + B.b[d]);
      B.lo[d] = D == 3 || d == 0 ? __double2float_rd(lo - widest) : -INFINITY;
      B.up[d] = D == 3 || d == 0 ? __double2float_ru(up + widest) : INFINITY;
      if (g.inv_e > 0) {
        // the cells any of the groups reaches
        c0[d] = __builtin_amdgcn_readfirstlane(cell_of(wave_min((double)B.lo[d]), g.lo[d], g.inv_e, nn[d]));
        c1[d] = __builtin_amdgcn_readfirstlane(cell_of(wave_max((double)B.up[d]), g.lo[d], g.inv_e, nn[d]));
      }
    }
    if (lane % kGroup == 0 && (uint32_t)lane / kGroup < ng) gb[lane / kGroup] = B;
    if (!__any(in)) c1[0] = c0[0] - 1, c1[1] = c0[1] - 1;
  }
  const uint64_t fb = __ballot(fast);
  const int rows_y = c1[1] - c0[1] + 1, nrow = rows_y * (c1[2] - c0[2] + 1);
  uint32_t off[kGroupsPerChunk] = {}, num[kGroupsPerChunk] = {};
  for (int write = 0; write < 2; write++) {
    for (int rb = 0; rb < nrow; rb += kWave) {
      // the tiles of a row of cells are consecutive: first tile of each row, and
      // how many tiles the rows before it hold
      uint32_t first = 0, len = 0;
      if (rb + lane < nrow) {
        const int cy = c0[1] + (rb + lane) % rows_y, cz = c0[2] + (rb + lane) / rows_y;
        const uint32_t cell = ((uint32_t)cz * g.ny + cy) * g.nx;
        first = pc.tr.toff[cell + c0[0]];
        len = pc.tr.toff[cell + c1[0] + 1] - first;
      }
      uint32_t upto = len;
      for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t v = __shfl_up(upto, o);
        if (lane >= o) upto += v;
      }
      __syncthreads();
      rowpre[lane] = upto - len;
      rowtile[lane] = first;
      __syncthreads();
      const uint32_t total = __builtin_amdgcn_readlane(upto, kWave - 1);
      for (uint32_t kb = 0; kb < total; kb += kWave) {
        // the lanes test a tile each
        const uint32_t k = kb + lane;
        uint32_t meets = 0;
        float4 tlo = make_float4(0.f, 0.f, 0.f, 0.f), thi = tlo;
        if (k < total) {
          uint32_t ra = 0;                          // the last row that starts at or before k
          for (uint32_t o = kWave / 2; o > 0; o >>= 1)
            if (rowpre[ra + o] <= k) ra += o;
          const uint32_t t = rowtile[ra] + (k - rowpre[ra]);
          tlo = pc.tr.tbox[2 * t];
          thi = pc.tr.tbox[2 * t + 1];
          for (uint32_t q = 0; q < ng; q++) {
            const GroupBox &B = gb[q];
            const bool out = tlo.x > B.up[0] || thi.x < B.lo[0] || tlo.y > B.up[1] || thi.y < B.lo[1] ||
                             tlo.z > B.up[2] || thi.z < B.lo[2];
            meets |= out ? 0u : 1u << q;
          }
        }
        if (!write) {
#pragma unroll
          for (uint32_t q = 0; q < kGroupsPerChunk; q++) num[q] += (uint32_t)__popcll(__ballot((meets >> q) & 1u));
          continue;
        }
        uint64_t tm = __ballot(meets != 0);
        uint32_t mlo[kGroupsPerChunk] = {}, mhi[kGroupsPerChunk] = {};   // this lane's tile's masks
        while (tm) {
          const uint32_t l = (uint32_t)__builtin_ctzll(tm);
          clear_bit_u(tm, l);
          const uint32_t base = __builtin_amdgcn_readlane(__float_as_uint(tlo.w), l);
          const uint32_t cnt = __builtin_amdgcn_readlane(__float_as_uint(thi.w), l);
          const uint32_t gm = __builtin_amdgcn_readlane(meets, l);
          const uint32_t j = base + min((uint32_t)lane, cnt - 1u);
          const double2 xy = gc.g.xy[j], zh = gc.g.zh[j];
          const double chh = gc.cutj * zh.y;
          const uint64_t valid = cnt < kWave ? (1ull << cnt) - 1 : ~0ull;
#pragma unroll
          for (uint32_t q = 0; q < kGroupsPerChunk; q++) {
            if (!((gm >> q) & 1u)) continue;
            const GroupBox &B = gb[q];
            double d = fabs(xy.x - B.c[0]) - B.b[0];
            if (D == 3) d = fmax(d, fmax(fabs(xy.y - B.c[1]) - B.b[1], fabs(zh.x - B.c[2]) - B.b[2]));
            const uint64_t in = (__ballot(d - chh <= B.chh) | __ballot(d <= B.ch)) & valid;
            set_lane(mlo[q], (uint32_t)in, l);
            set_lane(mhi[q], (uint32_t)(in >> 32), l);
          }
        }
#pragma unroll
        for (uint32_t q = 0; q < kGroupsPerChunk; q++) {
          const uint64_t has = __ballot((mlo[q] | mhi[q]) != 0);
          if (mlo[q] | mhi[q])
            gc.gl.visit[(size_t)off[q] + num[q] + lanes_below(has)] =
                make_uint4(__float_as_uint(tlo.w), __float_as_uint(thi.w), mlo[q], mhi[q]);
          num[q] += (uint32_t)__popcll(has);
        }
      }
    }
    if (!write) {
      uint32_t room = 0;
      unsigned long long first = 0;
      for (uint32_t q = 0; q < kGroupsPerChunk; q++) room += num[q];
      if (lane == 0) first = atomicAdd(gc.gl.cursor, (unsigned long long)room);
      uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)first);
      if (__builtin_amdgcn_readfirstlane((uint32_t)(first >> 32)) || (unsigned long long)at + room > gc.gl.cap) {
        if (gc.over && lane == 0) atomicOr(gc.over, 1ull);
        return;
      }
      for (uint32_t q = 0; q < kGroupsPerChunk; q++) {
        off[q] = at;
        at += num[q];
        num[q] = 0;
      }
    }
  }
#pragma unroll
  for (uint32_t q = 0; q < kGroupsPerChunk; q++) {
    const uint32_t gid = chunk * kGroupsPerChunk + g0 + q;
    if (lane == 0 && q < ng) {
      gc.gl.off[gid] = off[q];
      gc.gl.num[gid] = num[q];
      gc.gl.fast[gid] = ((fb >> (q * kGroup)) & 0xffu) == 0xffu ? 1u : 0u;
    }
  }
}

// 64 lanes' 16 (4) bytes from memory to consecutive LDS places
template <int BYTES>
__device__ inline void load_to_lds(const void *from, void *to) {
  auto *g = (const __attribute__((address_space(1))) uint32_t *)from;
  auto *l = (__attribute__((address_space(3))) uint32_t *)to;
  if constexpr (BYTES == 16) __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0);
  else __builtin_amdgcn_global_load_lds(g, l, 4, 0, 0);
}

// A tile's particles: positions, then the pass's record arrays (NA16 of 16
// bytes a particle, NA4 of 4).  Place kWave is out of every kernel's reach.
template <class P>
struct TileLds {
  double2 xy[kWave + 1], zh[kWave + 1];
  float4 a16[P::NA16][kWave + 1];
  float a4[P::NA4 ? P::NA4 : 1][P::NA4 ? kWave + 4 : 4];   // (whole 16 bytes)
  __device__ const double2 *d2(int k) const { return (const double2 *)a16[k]; }
  __device__ const float4 *f4(int k) const { return a16[k]; }
  __device__ const float *f1(int k) const { return a4[k]; }
};

// one wave's LDS; the tile's place takes the wave's sums at the end
template <class P>
struct GroupLds {
  union {
    TileLds<P> st;
    struct { double sum[P::NACC][kGroup]; uint64_t bad; uint32_t npairs; } tot;
  };
  uint8_t queue[2 * kWave];                        // places in the tile
};

template <class T>
using const_ptr = const __attribute__((address_space(4))) T *;   // read by scalar loads where uniform

// v plus its value kGroup, 2 kGroup, ... lanes on: the sum over the streams, on
// every lane (order fixed)
__device__ inline double stream_sum(double v) {
  static_assert(kGroup == 8, "lane = target + 8 stream");
  v += row_move<0x128>(v);                        // row_ror 8
  v = swap_add<1>(v, v);
  return swap_add<2>(v, v);
}

// A pair pass over groups.  Each pass supplies: Tgt (the lane's target), Rec
// (one particle) and load() of it from a staged tile, pack(), which writes the
// arrays the tiles are loaded from, hker() (h of the kernel-box test),
// pair_d(), which adds to the target's NACC partial sums, and finish() for the
// lane that holds a target's totals.
//
// Bound by VALU issue.  Whatever is left in the queue after a tile stays in the
// registers of its streams (nl of them) while the next tile is staged.
//
// The waves of a workgroup (blockDim.x / 64) share a group: each takes its visits
// in turn, in LDS of its own, and the first adds up their sums.
//
// FROZEN (a frozen replay): the predicates read g's and pc.x (the recorded
// run's positions) and the pair arithmetic pc.ax; otherwise both are pc.x.
template <int D, class P, bool FROZEN>
__global__ __launch_bounds__(kMaxSplit * kWave, P::kWaves) void k_group_pass(PairCommon pc, GroupCommon gc,
                                                                             typename P::Args a) {
  extern __shared__ char lds[];                    // a GroupLds<P> per wave
  uint32_t gid, i;
  const uint32_t nt = my_group(pc, gid, i);
  if (!nt || halted(pc.halt, pc.nhalt)) return;
  if (gc.over) {
    if (gc.over[0]) return;
    if (gid == 0 && threadIdx.x == 0) atomicAdd(gc.over + (W_ITERS - W_OVER), 1ull);
  }
  const int lane = threadIdx.x % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), split = blockDim.x / kWave;
  GroupLds<P> &own_lds = ((GroupLds<P> *)lds)[wave];
  TileLds<P> &st = own_lds.st;
  uint8_t *const queue = own_lds.queue;
  const uint32_t stream = (uint32_t)lane / kGroup, slot = (uint32_t)lane % kGroup;
  typename P::Own own;
  typename P::Tgt T;
  P::load_target(a, i, T, own);
  // a lane without a target of its own meets nothing
  const double xi[3] = {slot < nt && P::wants(T) ? pc.x[i] : -kFar, pc.y[i], pc.z[i]};
  double xa[3] = {0, 0, 0};
  if constexpr (FROZEN) { xa[0] = pc.ax[i]; xa[1] = pc.ay[i]; xa[2] = pc.az[i]; }
  if (lane == 0) {
    st.xy[kWave] = make_double2(kFar, kFar);
    st.zh[kWave] = make_double2(kFar, 0.0);
  }
  // what membership takes of the target: kept where every pair is tested
  uint32_t ri = 0;
  double lf = 0, supp = 0;
  if constexpr (P::kRefb) {
    ri = pc.refb[i];
    lf = pc.list_factor * pc.h_list[i];
    supp = P::support(a, i);
  }
  double acc[P::NACC];
#pragma unroll
  for (int k = 0; k < P::NACC; k++) acc[k] = 0;
  uint32_t npairs = 0;                             // of all targets (wave-uniform)
  uint64_t bad = 0;                                // lanes that met an invalid neighbour (wave-uniform)
  const bool slow = FROZEN || __builtin_amdgcn_readfirstlane(gc.gl.fast[gid]) == 0 || pc.gflag != nullptr;
  const uint32_t nv = __builtin_amdgcn_readfirstlane(gc.gl.num[gid]);
  const_ptr<uint32_t> vis = (const_ptr<uint32_t>)(uintptr_t)(gc.gl.visit + __builtin_amdgcn_readfirstlane(gc.gl.off[gid]));
  uint32_t ahead[4] = {0, 0, 0, 0};                // the next visit
  if (wave < nv)
    for (int k = 0; k < 4; k++) ahead[k] = vis[(size_t)wave * 4 + k];
  double2 xy, zh;
  uint32_t j = 0;
  typename P::Rec r;
  uint32_t nl = 0;                                 // streams that hold their particle in registers
  for (uint32_t v = wave;; v += split) {
    uint32_t base = 0;
    uint64_t m = 0;
    const uint32_t held = nl;
    if (v < nv) {
      base = ahead[0];
      const uint32_t cnt = ahead[1];
      m = (uint64_t)ahead[3] << 32 | ahead[2];
      const_ptr<uint32_t> e = vis + (size_t)min(v + split, nv - 1) * 4;
      for (int k = 0; k < 4; k++) ahead[k] = e[k];
      const uint32_t from = base + min((uint32_t)lane, cnt - 1u);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the last tile has been read
      load_to_lds<16>(gc.g.xy + from, st.xy);
      load_to_lds<16>(gc.g.zh + from, st.zh);
#pragma unroll
      for (int k = 0; k < P::NA16; k++) load_to_lds<16>(a.pk.f4(k) + from, st.a16[k]);
#pragma unroll
      for (int k = 0; k < P::NA4; k++) load_to_lds<4>(a.pk.f1(P::NA16 + k) + from, st.a4[k]);
      if ((m >> lane) & 1) queue[held + lanes_below(m)] = (uint8_t)lane;
    } else {
      if (!held) break;
      // the last block's other streams take the place out of reach
      m = 0xffu >> held;
      if ((uint32_t)lane < kStreams - held) queue[held + lane] = (uint8_t)kWave;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // tile and queue are there
    // the streams below nl hold theirs
    auto load = [&](const uint8_t *at) {
      const uint32_t p = at[stream];
      xy = st.xy[p];
      zh = st.zh[p];
      P::load(st, p, r);
      if (slow) j = base + p;
    };
    const uint8_t *qp = queue;
    uint32_t left = held + (uint32_t)__popcll(m);
    for (; left >= kStreams; left -= kStreams, qp += kStreams) {
      if (stream >= nl) load(qp);
      nl = 0;
      double dx[3];
      dx[0] = xi[0] - xy.x;
      double amax = fabs(dx[0]);
      if (D == 3) {
        dx[1] = xi[1] - xy.y; dx[2] = xi[2] - zh.x;
        amax = fmax(amax, fmax(fabs(dx[1]), fabs(dx[2])));
      }
      const double hk = P::hker(T, zh.y);
      uint64_t in = __ballot(!pc.cut.outside(amax, hk));
      if (slow) {
        const bool mine = (in >> lane) & 1;
        // list membership (neighs.cc:37-211: same bucket or 4.25 h_i box) and in_support
        uint32_t rj;
        if constexpr (P::kRefb) {
          rj = r.refb;
        } else {
          rj = mine ? pc.refb[j] : 0u;
          ri = pc.refb[i];
          lf = pc.list_factor * pc.h_list[i];
          supp = P::support(a, i);
        }
        bool member = amax <= lf;
        if (pc.list_adj != 0) member &= refb_adjacent(rj, ri);
        member |= (rj == ri) | (pc.list_all != 0);
        bool ok = mine & member & (amax <= supp);
        if (pc.gflag) {
          // recorded step: the boundary ghosts (bc 1, 2) met as neighbours
          const int bj = ok ? pc.bc[j] : 0;
          ok &= P::counts_ghost(a, bj);
          if (ok && (bj == 1 || bj == 2)) pc.gflag[j] = 1u;
        }
        if constexpr (FROZEN) {
          const uint32_t ja = ok ? j : i;
          dx[0] = xa[0] - pc.ax[ja];
          if (D == 3) { dx[1] = xa[1] - pc.ay[ja]; dx[2] = xa[2] - pc.az[ja]; }
        }
        in = __ballot(ok);
      }
      if constexpr (P::kCountPairs) {
        npairs += (uint32_t)__popcll(in);
        bad |= in & __ballot(!P::valid(r));
      }
      if (__builtin_amdgcn_inverse_ballot_w64(in)) P::template pair_d<D>(a, T, r, hk, dx, amax, acc);
    }
    if (v >= nv) break;
    if (stream >= nl && stream < left) load(qp);
    nl = left;
  }
  double sum[P::NACC];
#pragma unroll
  for (int k = 0; k < P::NACC; k++) sum[k] = stream_sum(acc[k]);
  for (int o = 32; o >= kGroup; o >>= 1) bad |= bad >> o;
  if (split > 1) {
    // the waves' sums, added in their order
    if (lane < kGroup)
      for (int k = 0; k < P::NACC; k++) own_lds.tot.sum[k][lane] = sum[k];
    if (lane == 0) { own_lds.tot.bad = bad; own_lds.tot.npairs = npairs; }
    __syncthreads();
    if (wave != 0) return;
    for (uint32_t w = 1; w < split; w++) {
      const GroupLds<P> &o = ((GroupLds<P> *)lds)[w];
      for (int k = 0; k < P::NACC; k++) sum[k] += o.tot.sum[k][lane % kGroup];
      bad |= o.tot.bad;
      npairs += o.tot.npairs;
    }
  }
  if ((uint32_t)lane < nt) P::finish(a, own, sum, ((bad >> lane) & 1u) != 0, i, pc.err);
  // pairs of the group's targets, without the targets themselves
  if constexpr (P::kCountPairs)
    if (lane == 0 && npairs > nt) atomicAdd(a.pairs, (unsigned long long)(npairs - nt));
}

constexpr double kInvSqrtPi = 0.564189583547756;   // sph_lib.cc:207

// The pair arithmetic type R is double (FP64 form) or float (FP32-pair form):
// the pair predicate is FP64 in both, so both forms visit exactly the same
// pairs; accumulators, integration and the EOS stay FP64.
// ---------------------------------------------------------------------------
// 1 / x in FP64 for normal x and 1 / x: the hardware estimate and two Newton
// steps whose last rounds once (within a rounding of the quotient).  5
// instructions; the IEEE division takes 10 and the scaling that the quotients
// here, far from the ends of the range, do not need.
__device__ inline double rcp_newton(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}
template <class R> __device__ inline R rrcp(R x);
template <> __device__ inline double rrcp<double>(double x) { return rcp_newton(x); }
template <> __device__ inline float rrcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }
template <class R> __device__ inline R rfma(R a, R b, R c);
template <> __device__ inline double rfma<double>(double a, double b, double c) { return fma(a, b, c); }
template <> __device__ inline float rfma<float>(float a, float b, float c) { return fmaf(a, b, c); }
// |x| as the source modifier of the consuming instruction (x < 0 ? -x : x
// would cost a compare and a select)
template <class R> __device__ inline R rabs(R x);
template <> __device__ inline double rabs<double>(double x) { return __builtin_fabs(x); }
template <> __device__ inline float rabs<float>(float x) { return __builtin_fabsf(x); }

// exp(-e) in FP64 for e >= 0 without a table (Cody and Waite's reduction: e = -k
// ln 2 - r with k an integer, |r| <= ln 2 / 2, ln 2 in two parts; then 1 + r +
// r^2 q(r) with q the degree-9 polynomial through the Chebyshev nodes of the
// interval, computed for this file in 60-digit arithmetic: truncation 1.7e-17).
// Measured over 0 <= e <= 27.5: 1.0 ulp at most, 0.30 ulp rms (a table of
// exp(-k/8) and a series of degree 10: 1.9 and 0.47; the C library's: 0.51 and 0.29).  16 VALU instructions
// and no LDS.
__device__ inline double exp_neg(double e) {
  const double magic = 6755399441055744.0;               // 1.5 * 2^52: kd's low word is k
  const double kd = fma(e, -1.4426950408889634, magic), k = kd - magic;
  double r = fma(k, -0.6931471805598903, -e);
  r = fma(k, -5.497923018708371e-14, r);
  double p = 2.510038549551032e-08;
  p = fma(p, r, 2.7620088445409746e-07); p = fma(p, r, 2.7557268459997064e-06);
  p = fma(p, r, 2.4801521295954376e-05); p = fma(p, r, 0.00019841269863053618);
  p = fma(p, r, 0.0013888888917213717); p = fma(p, r, 0.008333333333330062);
  p = fma(p, r, 0.04166666666662413); p = fma(p, r, 0.16666666666666669);
  p = fma(p, r, 0.5); p = fma(p, r, 1.0); p = fma(p, r, 1.0);
  return __builtin_amdgcn_ldexp(p, (int)(uint32_t)__double_as_longlong(kd));
}

// exp(-e), e >= 0, in the pair arithmetic's type
template <class R> __device__ inline R rexp_neg(R e);
template <> __device__ inline double rexp_neg<double>(double e) { return exp_neg(e); }
template <> __device__ inline float rexp_neg<float>(float e) { return __expf(-e); }

// The exponential of the FP32-pair forms' FP64 weights.  FX false
// (PSPH_FP32_PAIR): exp_neg, FP64 throughout.  FX true (PSPH_FP32_EXP):
// the FP32 hardware exponential 2^-tf of the argument t = e log2(e), formed
// in FP64 and rounded once to tf: a relative error of the instruction's own
// (about one FP32 ulp) plus t 2^-24 ln 2 from the rounding of t (largest at
// the kernel box's corner, where the weight is e^-27 of the centre's), while
// h, 1/h and the norm stay FP64.  Taking the rounding of t back out (times
// 1 - (t - tf) ln 2) halves the form's difference to FP64 over the bench's
// steps and costs 4 % of the step: not kept.
constexpr double kLog2e = 1.4426950408889634;
// 2^-t of the FX form (t >= 0 in FP64)
__device__ inline double exp2_neg_fx(double t) { return (double)__builtin_amdgcn_exp2f(-(float)t); }
template <bool FX> __device__ inline double exp_neg_w(double e) {
  if constexpr (!FX) return exp_neg(e);
  else return exp2_neg_fx(e * kLog2e);
}

// The particle records that a pass reads, in arrays of 16-byte pieces (the last
// may be narrower): neighbouring lanes take neighbouring pieces.
struct Packs {
  void *p[5];
  __device__ double2 *d2(int k) const { return (double2 *)p[k]; }
  __device__ float4 *f4(int k) const { return (float4 *)p[k]; }
  __device__ float *f1(int k) const { return (float *)p[k]; }
};

template <class R> __device__ inline R pow16(R x) {
  x *= x; x *= x; x *= x;
  return x * x;
}

// ---------------------------------------------------------------------------
// RHS pass: mom_engr_update, USE_GSPH==0 (mom_engr_update.cc:30-439)
// ---------------------------------------------------------------------------
struct RhsArgs {
  const double *h, *m, *rho, *p, *c, *T, *cp, *vx, *vy, *vz, *svx, *svy, *svz, *e, *xi;
  const int32_t *bc;
  double *o_vx, *o_vy, *o_vz, *o_e, *o_p, *o_c, *o_T, *o_gam, *o_cp;
  double dt, g, cutoff, cutoff2, alpha, beta, ata, eps_half, prandtl, heat_scale;
  // per-pair constants, folded on the host: 2 beta; 20 eps / Pr (the heat
  // term's 10 eps / Pr, doubled because the energy sum holds 2 de/dt)
  double beta2, kheat;
  int lans, dim;
  EosConst eos;
  unsigned long long *pairs;
  Packs pk;
};

// Pair terms, written with the halves folded: c2 = c_i + c_j = 2 c_ab,
// rs = rho_i + rho_j = 2 rho_ab, cp2 = 2 cp_ab.  Pi = (beta mu - alpha c_ab)
// mu / rho_ab = (2 beta mu - alpha c2) mu / rs with mu = h v.r / den (one
// reciprocal of den rs gives both 1/den and 1/rs); the heat term's cp_ab /
// c_ab = cp2 / c2.  The energy sum holds 2 de/dt (finish takes half).
//
// The FP32-pair form keeps the pressure term m_j (p_j/rho_j^2 + p_i/rho_i^2)
// grad W in FP64: in air near hydrostatic balance its pair terms cancel to
// about 1 % of their size, and FP32 rounding there is what the velocities
// feel.  The kernel value is FP64 (exp_neg, or the FP32 instruction in FX);
// viscosity, heat conduction and the energy work terms stay FP32.
// -2 pi^(-D/2): grad W = G dx with G = -2 W / h^2 = kGradNorm h^-(D+2) exp(-r^2/h^2)
template <int D> constexpr double kGradNorm = -2.0 * kInvSqrtPi * kInvSqrtPi * kInvSqrtPi;
template <> constexpr double kGradNorm<1> = -2.0 * kInvSqrtPi;

template <class R, bool MIXED = std::is_same<R, float>::value, bool FX = false>
struct RhsPass {
  using Args = RhsArgs;
  static constexpr bool kMixed = MIXED;
  static constexpr bool kCountPairs = true;
  static constexpr int NACC = 4;               // 0-2: the velocity sums, 3: the energy sum (2 de/dt)
  struct Own { bool bad; };
  struct Tgt {
    double hh, pv64;
    R rhoi, Vi, pvsqi, ci, Ti, cpi, vel[3];
  };
  // a neighbour; m64, mpv64 (m p / rho^2) and mV (m / rho) only in the mixed
  // form, PV2 (p / rho^2) only in the others
  struct Rec {
    double m64, mpv64;
    R m, V, rho, c, T, cp, vx, vy, vz, PV2, mV;
  };
  // waves per SIMD: 96 VGPRs hold the FP32-exp and FP32-pure forms, 128 the others
  static constexpr int kWaves = std::is_same<R, double>::value || (MIXED && !FX) ? 4 : 5;
  __device__ static void load_target(const Args &a, uint32_t i, Tgt &t, Own &o) {
    t.hh = 0.5 * a.h[i];
    const double rho = a.rho[i];
    o.bad = !(rho > 0);
    const double Vi = 1.0 / rho;
    t.pv64 = a.p[i] * Vi * Vi;
    t.rhoi = (R)rho; t.Vi = (R)Vi; t.pvsqi = (R)t.pv64;
    t.ci = (R)a.c[i]; t.Ti = (R)a.T[i]; t.cpi = (R)a.cp[i];
    if (a.lans) { t.vel[0] = (R)a.svx[i]; t.vel[1] = (R)a.svy[i]; t.vel[2] = (R)a.svz[i]; }
    else { t.vel[0] = (R)a.vx[i]; t.vel[1] = (R)a.vy[i]; t.vel[2] = (R)a.vz[i]; }
  }
  __device__ static void pack(const Args &a, uint32_t j) {
    const double rj = a.rho[j];
    const double V = 1.0 / rj;
    const double pv = a.p[j] * V * V;
    const double mj = a.m[j];
    const double *ux = a.lans ? a.svx : a.vx, *uy = a.lans ? a.svy : a.vy, *uz = a.lans ? a.svz : a.vz;
    const R c = (R)a.c[j], T = (R)a.T[j], cp = (R)a.cp[j], vx = (R)ux[j], vy = (R)uy[j], vz = (R)uz[j];
    if constexpr (kMixed) {
      a.pk.d2(0)[j] = make_double2(mj, mj * pv);
      a.pk.f4(1)[j] = make_float4((R)V, (R)rj, c, T);
      a.pk.f4(2)[j] = make_float4(cp, vx, vy, vz);
      a.pk.f1(3)[j] = (float)(mj * V);
    } else if constexpr (std::is_same<R, float>::value) {
      a.pk.f4(0)[j] = make_float4((R)mj, (R)V, (R)rj, c);
      a.pk.f4(1)[j] = make_float4(T, cp, (R)pv, vx);
      a.pk.f1(2)[j] = vy;
      a.pk.f1(3)[j] = vz;
    } else {
      a.pk.d2(0)[j] = make_double2(mj, V);
      a.pk.d2(1)[j] = make_double2(rj, c);
      a.pk.d2(2)[j] = make_double2(T, cp);
      a.pk.d2(3)[j] = make_double2(pv, vx);
      a.pk.d2(4)[j] = make_double2(vy, vz);
    }
  }
  static constexpr int NA16 = kMixed ? 3 : std::is_same<R, float>::value ? 2 : 5;
  static constexpr int NA4 = kMixed ? 1 : std::is_same<R, float>::value ? 2 : 0;
  template <class L>
  __device__ static void load(const L &a, uint32_t j, Rec &r) {
    if constexpr (kMixed) {
      const double2 u = a.d2(0)[j];
      const float4 v = a.f4(1)[j], w = a.f4(2)[j];
      r.m64 = u.x; r.mpv64 = u.y; r.m = (R)u.x;
      r.V = v.x; r.rho = v.y; r.c = v.z; r.T = v.w;
      r.cp = w.x; r.vx = w.y; r.vy = w.z; r.vz = w.w;
      r.mV = a.f1(0)[j];
    } else if constexpr (std::is_same<R, float>::value) {
      const float4 u = a.f4(0)[j], v = a.f4(1)[j];
      r.m = u.x; r.V = u.y; r.rho = u.z; r.c = u.w;
      r.T = v.x; r.cp = v.y; r.PV2 = v.z; r.vx = v.w; r.vy = a.f1(0)[j]; r.vz = a.f1(1)[j];
    } else {
      const double2 p0 = a.d2(0)[j], p1 = a.d2(1)[j], p2 = a.d2(2)[j], p3 = a.d2(3)[j], p4 = a.d2(4)[j];
      r.m = p0.x; r.V = p0.y; r.rho = p1.x; r.c = p1.y; r.T = p2.x; r.cp = p2.y;
      r.PV2 = p3.x; r.vx = p3.y; r.vy = p4.x; r.vz = p4.y;
    }
  }
  // h_ij = (h_i + h_j)/2 (ME_UPDATE_SML 2).  The reference skips j == i; here
  // the target meets itself once, with dx = 0 and v_ij = 0, and every term it
  // adds is an exact zero (f dx, f v.r, no viscosity for v.r = 0, no heat for
  // |v_ij . dx| = 0), so no test is spent on it; the pair count leaves it out.
  __device__ static double hker(const Tgt &t, double hhj) { return t.hh + hhj; }
  __device__ static bool counts_ghost(const Args &, int) { return true; }
  __device__ static double support(const Args &a, uint32_t i) { return a.cutoff2 * a.h[i]; }
  __device__ static bool wants(const Tgt &) { return true; }
  static constexpr bool kRefb = false;
  __device__ static bool valid(const Rec &r) { return r.rho > R(0); }        // assert(uvecj[0] > 0)
  template <int D>
  __device__ static void pair_d(const Args &a, const Tgt &t, const Rec &s, double hijd, const double *dxd, double,
                                double *acc) {
    if constexpr (kMixed) pair_mixed<D>(a, t, s, hijd, dxd, acc);
    else pair_plain<D>(a, t, s, hijd, dxd, acc);
  }
  template <int D>
  __device__ static void pair_plain(const Args &a, const Tgt &t, const Rec &s, double hijd, const double *dxd, double *acc) {
    const R rhoj = s.rho;
    const R h = (R)hijd;
    const R ih = rrcp<R>(h);
    R dx[3], dist_sq = 0, expt = 0;
#pragma unroll
    for (int k = 0; k < D; k++) {
      dx[k] = (R)dxd[k];
      const R sk = dx[k] * ih;
      dist_sq += dx[k] * dx[k];
      expt += sk * sk;
    }
    const R ih2 = ih * ih;
    const R ihD = (D == 3) ? ih2 * ih : ih;
    // G = -2 W / h^2: grad W = G dx
    const R G = (R(kGradNorm<D>) * ih2) * (ihD * rexp_neg<R>(expt));
    const R Vj = s.V;
    R vij[3];
    vij[0] = t.vel[0] - s.vx;
    if (D == 3) { vij[1] = t.vel[1] - s.vy; vij[2] = t.vel[2] - s.vz; }
    const R c2 = t.ci + s.c;
    // (fused explicitly: the heat term needs the products v_k dx_k rounded, and
    // the compiler would sum those)
    R vrab = 0;
#pragma unroll
    for (int k = 0; k < D; k++) vrab = rfma<R>(dx[k], vij[k], vrab);
    const R dotvv = D == 3 ? rfma<R>(vij[2], vij[2], rfma<R>(vij[0], vij[0], vij[1] * vij[1])) : vij[0] * vij[0];
    // art_vis (sph_lib.cc:402-424): Pi = (beta mu - alpha c) mu / rho_ab for
    // approaching pairs, mu = h v.r / (r^2 + ata h^2)
    R vis;
    {
      const R rs = t.rhoi + rhoj;
      const R den = dist_sq + R(a.ata) * h * h;
      const R r = rrcp<R>(den * rs);
      const R miu = h * vrab * (rs * r);
      vis = (R(a.beta2) * miu - R(a.alpha) * c2) * miu * (den * r);
      vis = vrab < R(0) ? vis : R(0);
    }
    if (a.lans) vis -= R(a.eps_half) * dotvv * Vj;        // SPH_epsilon_mom
    const R mpv = s.m * (s.PV2 + t.pvsqi + vis);
    R heat = 0;
    if (a.lans && D == 3) {
      // k_ij F_ij of SPH_epsilon_heat_conductivity (6-arg, sph_lib.cc:1399-1439)
      // and compute_F (sph_lib.cc:257-281): 10 eps cp r^2 |v|^2 / (Pr sum|v_k dx_k|)
      // / (h c) * (dW.dx / r^2); the r^2 factors cancel: dW.dx = G r^2.
      R dotvr = 0;
#pragma unroll
      for (int k = 0; k < D; k++) dotvr += rabs<R>(vij[k] * dx[k]);
      const R wr = G * dist_sq;
      const R cp2 = s.cp + t.cpi;
      const R kF = R(a.kheat) * cp2 * dotvv * wr * rrcp<R>(dotvr * h * c2);
      heat = s.m * Vj * t.Vi * (t.Ti - s.T) * kF;
      heat = ((dotvr != R(0)) & (wr != R(0))) ? heat : R(0);
    }
    R de = 0;
    const R Gm = mpv * G;
#pragma unroll
    for (int k = 0; k < D; k++) {
      const R f = Gm * dx[k];
      acc[k] -= (double)f;
      de = rfma<R>(f, vij[k], de);
    }
    acc[3] += (double)(de + heat);
  }
  template <int D>
  __device__ static void pair_mixed(const Args &a, const Tgt &t, const Rec &s, double hijd, const double *dxd, double *acc) {
    const double hd = hijd;
    const float h = (float)hd;
    const float ih = rrcp<float>(h);
    const double ih64 = (double)ih * fma(-hd, (double)ih, 2.0);     // one Newton step: ~1e-14
    const double ih2 = ih64 * ih64;
    const double ihD = (D == 3) ? ih2 * ih64 : ih64;
    double r2 = 0;
    float dx[3];
#pragma unroll
    for (int k = 0; k < D; k++) { r2 = fma(dxd[k], dxd[k], r2); dx[k] = (float)dxd[k]; }
    // G = -2 W / h^2: grad W = G dx
    const double G64 = (kGradNorm<D> * ih2) * (ihD * exp_neg_w<FX>(r2 * ih2));
    const float G = (float)G64, dist_sq = (float)r2;
    const float Vj = s.V, rhoj = s.rho;
    float vij[3];
    vij[0] = t.vel[0] - s.vx;
    if (D == 3) { vij[1] = t.vel[1] - s.vy; vij[2] = t.vel[2] - s.vz; }
    const float c2 = t.ci + s.c;
    float vrab = 0;
#pragma unroll
    for (int k = 0; k < D; k++) vrab = fmaf(dx[k], vij[k], vrab);
    const float dotvv = D == 3 ? fmaf(vij[2], vij[2], fmaf(vij[0], vij[0], vij[1] * vij[1])) : vij[0] * vij[0];
    float vis;
    {
      const float rs = t.rhoi + rhoj;
      const float den = dist_sq + (float)a.ata * h * h;
      const float r = rrcp<float>(den * rs);
      const float miu = h * vrab * (rs * r);
      vis = ((float)a.beta2 * miu - (float)a.alpha * c2) * miu * (den * r);
      vis = vrab < 0.f ? vis : 0.f;
    }
    if (a.lans) vis -= (float)a.eps_half * dotvv * Vj;
    // pressure part in FP64, viscous part in FP32; f = (M_p + M_v) G dx
    const double f = fma(s.m64, t.pv64, s.mpv64) * G64 + (double)(s.m * vis * G);
#pragma unroll
    for (int k = 0; k < D; k++) acc[k] = fma(-f, dxd[k], acc[k]);
    float heat = 0;
    if (a.lans && D == 3) {
      float dotvr = 0;
#pragma unroll
      for (int k = 0; k < D; k++) dotvr += rabs<float>(vij[k] * dx[k]);
      const float wr = G * dist_sq;
      const float cp2 = s.cp + t.cpi;
      const float kF = (float)a.kheat * cp2 * dotvv * wr * rrcp<float>(dotvr * h * c2);
      heat = s.mV * t.Vi * (t.Ti - s.T) * kF;
      heat = ((dotvr != 0.f) & (wr != 0.f)) ? heat : 0.f;
    }
    acc[3] += fma(f, (double)vrab, (double)heat);
  }
  __device__ static bool finish(const Args &a, const Own &o, const double *sum, bool bad, uint32_t i, int *err) {
    if (o.bad || bad) { raise_err(err, PSPH_EINVARIANT, i); return false; }
    const double gz = -a.g, dt = a.dt;
    // v += dt rhs_v; gravity on the last axis; e += dt (rhs_e + v_last g)
    // (mom_engr_update.cc:372-388); the velocity in the energy term is the
    // FP64 one of the target; sum[3] holds 2 rhs_e
    const double vl = a.dim == 3 ? (a.lans ? a.svz[i] : a.vz[i]) : (a.lans ? a.svx[i] : a.vx[i]);
    double nv0 = a.vx[i] + dt * (sum[0]);
    double nv1 = a.vy[i] + dt * (sum[1]);
    double nv2 = a.vz[i] + dt * (sum[2]);
    if (a.dim == 3) nv2 += dt * gz; else nv0 += dt * gz;
    const double ne = a.e[i] + dt * (0.5 * sum[3] + vl * gz);
    a.o_vx[i] = nv0; a.o_vy[i] = nv1; a.o_vz[i] = nv2;
    a.o_e[i] = ne;
    double p, c, T, gam, cp = a.cp[i];
    eos_dev(a.eos, a.rho[i], ne, a.xi[i], p, c, T, gam, &cp);
    a.o_p[i] = p; a.o_c[i] = c; a.o_T[i] = T; a.o_gam[i] = gam; a.o_cp[i] = cp;
    return true;
  }
};

// ---------------------------------------------------------------------------
// Density pass: smooth_density (density_massfrac.cc:25-359)
// ---------------------------------------------------------------------------
struct DensArgs {
  const double *h, *m, *rho, *e;
  const int32_t *bc, *phase;
  double *o_rho, *o_e, *xi, *p, *c, *T, *gam, *cp;
  int32_t *inv;
  double cutoff, cutoff2, e_ratio, msfrc_thresh;
  int pghost, energy_smooth;
  EosConst eos;
  CutTest cut;
  double *o_wn;            // optional: energy-smoothing normalisation (adjoint recompute)
  int e_sq16;              // e_ratio^2 == 16: exp(-16 x) = exp(-x)^16 by four squarings
  double e_norm;           // the energy-smoothing kernel's norm times h^D: (e_ratio / sqrt(pi))^D
  Packs pk;
};

// pi^(-D/2): W = kNorm h^-D exp(-s^2)
template <int D> constexpr double kNorm = kInvSqrtPi * kInvSqrtPi * kInvSqrtPi;
template <> constexpr double kNorm<1> = kInvSqrtPi;

// mr = m / rho of the candidate (the energy-smoothing weight's factor).  m is
// staged twice, as m1 (phase 1, else 0) and m2 (phase 2, else 0), so that a
// pair adds to both sums without selecting between them; a candidate that
// does not contribute (contr_dens false or another phase) stages zero masses
// and mr = 0, so its terms are exact zeros and no pair tests for it.
// The FP32-pair form evaluates the density and energy-smoothing weights in
// FP64: the pressure gradient of the next step amplifies
// relative errors of rho and e by its cancellation.
template <class R, bool MIXED = std::is_same<R, float>::value, bool FX = false>
struct DensPass {
  using Args = DensArgs;
  static constexpr bool kMixed = MIXED;
  static constexpr bool kCountPairs = false;
  static constexpr int NACC = 4;               // r1, r2, wn, en
  struct Own {};
  struct Tgt { double hh; };
  using W = typename std::conditional<kMixed, double, R>::type;   // the mixed form reads FP64 copies only
  struct Rec { W m1, m2, mr, e; };
  static constexpr int kWaves = 4;             // per SIMD: at most 128 VGPRs
  __device__ static void load_target(const Args &a, uint32_t i, Tgt &t, Own &) { t.hh = 0.5 * a.h[i]; }
  __device__ static void pack(const Args &a, uint32_t j) {
    const int ph = a.phase[j];
    const int ok = (contr_dens(a.pghost, a.bc[j]) && (ph == 1 || ph == 2)) ? ph : 0;
    const double mj = a.m[j];
    const double m1 = ok == 1 ? mj : 0.0, m2 = ok == 2 ? mj : 0.0;
    const double mr = ok ? mj / a.rho[j] : 0.0, e = ok ? a.e[j] : 0.0;
    if constexpr (std::is_same<W, float>::value) {
      a.pk.f4(0)[j] = make_float4((W)m1, (W)m2, (W)mr, (W)e);
    } else {
      a.pk.d2(0)[j] = make_double2(m1, m2);
      a.pk.d2(1)[j] = make_double2(mr, e);
    }
  }
  static constexpr int NA16 = std::is_same<W, float>::value ? 1 : 2, NA4 = 0;
  template <class L>
  __device__ static void load(const L &a, uint32_t j, Rec &r) {
    if constexpr (std::is_same<W, float>::value) {
      const float4 u = a.f4(0)[j];
      r = Rec{u.x, u.y, u.z, u.w};
    } else {
      const double2 u = a.d2(0)[j], v = a.d2(1)[j];
      r = Rec{u.x, u.y, v.x, v.y};
    }
  }
  // kernel at h_ij (DENSITY_UPDATE_SML 11); contr_dens and the phase are in
  // the packed masses.  The energy-smoothing kernel (support 0.75 h_ij) lies
  // inside that box.
  __device__ static double hker(const Tgt &t, double hhj) { return t.hh + hhj; }
  __device__ static bool counts_ghost(const Args &, int) { return true; }
  __device__ static double support(const Args &a, uint32_t i) { return a.cutoff2 * a.h[i]; }
  __device__ static bool wants(const Tgt &) { return true; }
  static constexpr bool kRefb = false;
  __device__ static bool valid(const Rec &) { return true; }
  template <int D>
  __device__ static void pair_d(const Args &a, const Tgt &t, const Rec &s, double hijd, const double *ds, double amax,
                                double *acc) {
    if constexpr (kMixed && FX) {
      // The FP32-exp form: the weights in FP32 (reciprocal of h_ij, s^2, the
      // exponential, the norm), the sums in FP64.  Over the 4M bench window
      // this moves rho by 2e-8 rel L1 against FP64 (3e-9 with FP64 weights
      // and the FP32 exponential) and the velocities not measurably (3.9e-7
      // against 3.6e-7), for 10 % of the pass.
      const float ih = rrcp<float>((float)hijd);
      float r2 = 0;
#pragma unroll
      for (int k = 0; k < D; k++) { const float d = (float)ds[k]; r2 = fmaf(d, d, r2); }
      const float ih2 = ih * ih;
      const float ex = __builtin_amdgcn_exp2f(-(r2 * (ih2 * (float)kLog2e)));
      const float ihD = (D == 3) ? ih2 * ih : ih;
      const double wk = (double)(((float)kNorm<D> * ihD) * ex);
      acc[0] = fma(wk, s.m1, acc[0]);
      acc[1] = fma(wk, s.m2, acc[1]);
      if (a.energy_smooth && !a.cut.outside(a.e_ratio * amax, hijd)) {
        const float ee = a.e_sq16 ? pow16(ex) : __builtin_amdgcn_exp2f(-(float)(a.e_ratio * a.e_ratio) * (r2 * (ih2 * (float)kLog2e)));
        const double vr = (double)(((float)a.e_norm * ihD) * ee) * s.mr;
        acc[2] += vr;
        acc[3] += vr * s.e;
      }
    } else if constexpr (kMixed) {
      const float ih32 = rrcp<float>((float)hijd);
      const double ih = (double)ih32 * fma(-hijd, (double)ih32, 2.0);
      double r2 = 0;
#pragma unroll
      for (int k = 0; k < D; k++) r2 = fma(ds[k], ds[k], r2);
      const double ih2 = ih * ih;
      const double expt = r2 * ih2;
      const double ihD = (D == 3) ? ih2 * ih : ih;
      const double ex = exp_neg_w<FX>(expt);
      // one of m1, m2 is 0: that sum gains an exact zero
      const double wk = (kNorm<D> * ihD) * ex;
      acc[0] = fma(wk, s.m1, acc[0]);
      acc[1] = fma(wk, s.m2, acc[1]);
      if (a.energy_smooth && !a.cut.outside(a.e_ratio * amax, hijd)) {
        const double ee = a.e_sq16 ? pow16(ex) : exp_neg_w<FX>(a.e_ratio * a.e_ratio * expt);
        const double vr = (a.e_norm * ihD) * (ee * s.mr);
        acc[2] += vr;
        acc[3] += vr * s.e;
      }
    } else {
    const R hij = (R)hijd;
    const R ih = rrcp<R>(hij);
    R expt = 0;
#pragma unroll
    for (int k = 0; k < D; k++) {
      R sk = (R)ds[k] * ih;
      expt += sk * sk;
    }
    const R ihD = (D == 3) ? ih * ih * ih : ih;
    const R ex = rexp_neg<R>(expt);
    const R wk = (R(kNorm<D>) * ihD) * ex;
    acc[0] += (double)(wk * s.m1);
    acc[1] += (double)(wk * s.m2);
    if (a.energy_smooth) {
      // weight(4 ds / h_ij, h_ij / 4) m_j / rho_j (HAVE_ENERGY_SMOOTH 1); exact FP64 box test
      if (!a.cut.outside(a.e_ratio * amax, hijd)) {
        const R e2 = R(a.e_ratio * a.e_ratio);
        const R vr = (R(a.e_norm) * ihD) * ((a.e_sq16 ? pow16(ex) : rexp_neg<R>(e2 * expt)) * s.mr);
        acc[2] += (double)vr;
        acc[3] += (double)(vr * s.e);
      }
    }
    }
  }
  __device__ static bool finish(const Args &a, const Own &, const double *sum, bool, uint32_t i, int *err) {
    double density = 0.0;
    density += sum[0];
    density += sum[1];
    const double xi = sum[1] / density;
    double e = a.e[i];
    if (a.energy_smooth) {
      if (!(sum[2] > 0)) { raise_err(err, PSPH_EINVARIANT, i); return false; }
      e = sum[3] / sum[2];
      if (a.o_wn) a.o_wn[i] = sum[2];
    }
    if (!(density > 0) || !(xi <= 1)) { raise_err(err, PSPH_EINVARIANT, i); return false; }
    a.o_rho[i] = density;
    a.o_e[i] = e;
    a.xi[i] = xi;
    if (xi >= a.msfrc_thresh && a.inv[i] != 2) a.inv[i] = 2;
    double p, c, T, gam, cp = a.cp[i];
    eos_dev(a.eos, density, e, xi, p, c, T, gam, &cp);
    a.p[i] = p; a.c[i] = c; a.T[i] = T; a.gam[i] = gam; a.cp[i] = cp;
    return true;
  }
};

// ---------------------------------------------------------------------------
// LANS velocity filter: smooth_velocity (smooth_velocity.cc:25-165)
// ---------------------------------------------------------------------------
struct VsmArgs {
  const double *h, *m, *rho, *vx, *vy, *vz;
  const int32_t *bc;
  double *svx, *svy, *svz;
  double cutoff, cutoff2;
  double *o_wn;            // optional: the filter's normalisation sum (adjoint recompute)
  Packs pk;
};

// The FP32-pair form evaluates the filter weights in FP64
// (kernel argument, exponential, m_j / rho_j): sv moves the particles, and
// FP32 weights (relative error ~3e-7, dominated by the rounding of s^2 and of
// h) made the velocity filter the largest source of FP32-vs-FP64 difference,
// ~15x the RHS's FP32 terms.
//
// A neighbour that is not contr_vel packs m / rho = 0, so its terms are exact
// zeros and no pair tests for it (in a recorded step the boundary-ghost marks
// do).
template <class R, bool FX = false>
struct VsmPass {
  using Args = VsmArgs;
  static constexpr bool kMixed = std::is_same<R, float>::value;
  static constexpr bool kCountPairs = false;
  static constexpr int NACC = 4;               // 0-2: the velocity differences, 3: the weights
  struct Own {};
  struct Tgt { double hi, ih2, v64[3]; double ih; };
  struct Rec { double mr, v[3]; };
  static constexpr int kWaves = 4;             // per SIMD: at most 128 VGPRs
  __device__ static void load_target(const Args &a, uint32_t i, Tgt &t, Own &) {
    t.hi = a.h[i];
    t.ih = 1.0 / t.hi;
    t.ih2 = FX ? t.ih * t.ih * kLog2e : t.ih * t.ih;    // the FX form's exponential takes s^2 log2(e)
    t.v64[0] = a.vx[i]; t.v64[1] = a.vy ? a.vy[i] : 0; t.v64[2] = a.vz ? a.vz[i] : 0;
  }
  __device__ static void pack(const Args &a, uint32_t j) {
    a.pk.d2(0)[j] = make_double2(contr_vel(a.bc[j]) ? a.m[j] / a.rho[j] : 0.0, a.vx[j]);
    a.pk.d2(1)[j] = make_double2(a.vy ? a.vy[j] : 0.0, a.vz ? a.vz[j] : 0.0);
  }
  static constexpr int NA16 = 2, NA4 = 0;
  template <class L>
  __device__ static void load(const L &a, uint32_t j, Rec &r) {
    const double2 u = a.d2(0)[j], v = a.d2(1)[j];
    r = Rec{u.x, {u.y, v.x, v.y}};
  }
  __device__ static double hker(const Tgt &t, double) { return t.hi; }
  __device__ static bool counts_ghost(const Args &, int b) { return contr_vel(b); }
  __device__ static double support(const Args &a, uint32_t i) { return a.cutoff2 * a.h[i]; }
  __device__ static bool wants(const Tgt &) { return true; }
  static constexpr bool kRefb = false;
  __device__ static bool valid(const Rec &) { return true; }
  template <int D>
  __device__ static void pair_d(const Args &, const Tgt &t, const Rec &s, double, const double *ds, double, double *acc) {
    if constexpr (kMixed) {
      double r2 = 0;
#pragma unroll
      for (int k = 0; k < D; k++) r2 = fma(ds[k], ds[k], r2);
      // the weight without the kernel's norm, which cancels in dv / wn
      double ew;
      if constexpr (FX) ew = exp2_neg_fx(r2 * t.ih2);
      else ew = exp_neg(r2 * t.ih2);
      const double w = ew * s.mr;
#pragma unroll
      for (int k = 0; k < D; k++) acc[k] = fma(w, s.v[k] - t.v64[k], acc[k]);
      acc[3] += w;
    } else {
      R expt = 0;
#pragma unroll
      for (int k = 0; k < D; k++) {
        R sk = (R)ds[k] * t.ih;
        expt += sk * sk;
      }
      const R mvw = rexp_neg<R>(expt) * s.mr;           // the norm cancels in dv / wn
#pragma unroll
      for (int k = 0; k < D; k++) acc[k] += mvw * (s.v[k] - t.v64[k]);
      acc[3] += mvw;
    }
  }
  __device__ static bool finish(const Args &a, const Own &, const double *sum, bool, uint32_t i, int *err) {
    if (!(sum[3] > 0)) { raise_err(err, PSPH_EINVARIANT, i); return false; }
    const double iw = 1.0 / sum[3];
    if (a.o_wn) {                                    // the normalisation sum with the kernel's norm
      const double nk = kInvSqrtPi * (1.0 / a.h[i]);
      a.o_wn[i] = sum[3] * (a.vy ? nk * nk * nk : nk);
    }
    a.svx[i] = a.vx[i] + sum[0] * iw;
    if (a.svy) { a.svy[i] = a.vy[i] + sum[1] * iw; a.svz[i] = a.vz[i] + sum[2] * iw; }
    return true;
  }
};

// ---------------------------------------------------------------------------
// Adaptive smoothing length: adaptive_sml (neighs.cc:479-693).  One launch
// per iteration of the reference's loop; h is updated in place (no pass reads
// another particle's h) and done[] marks particles whose |dh/h| < thresh.
// ---------------------------------------------------------------------------
struct AdaptArgs {
  const double *m;
  const int32_t *bc;
  const uint32_t *refb;
  double *h;
  uint32_t *done;
  double cutoff, cutoff2, c_smooth, eta, ratio, thresh;
  int pghost, dim;
  Packs pk;
};

// The exponential is FP64 (exp_neg), or in the FX form (PSPH_FP32_EXP) the FP32
// exponential of the FP64 argument: its rounding is independent from pair to
// pair, so rho* and h move by ~1e-9 relative over a particle's ~2000 list pairs.
// A candidate that does not contribute (contr_dens false) has a zero mass.  The
// kernel box (4.5 h) reaches past the list box (4.25 h of list time), so list
// membership is tested for every pair: the record carries the bucket.  Each
// iteration has visits of its own, for the boxes of the h it starts from and the
// targets that have not converged.  Bound by VALU issue.  60k targets, an
// iteration (visits in brackets): 2264 us with a bit mask of 32 targets x 2
// lanes, 577 (170) with groups.
template <class R, bool FX = false>
struct AdaptPass {
  using Args = AdaptArgs;
  static constexpr bool kCountPairs = false;
  static constexpr int NACC = 1;
  struct Own { double hcur; };
  struct Tgt { double Hs, iHs; bool done; };
  struct Rec { R m; uint32_t refb; };
  static constexpr int kWaves = 6;             // per SIMD: at most 80 VGPRs
  static constexpr bool kRefb = true;
  __device__ static void load_target(const Args &a, uint32_t i, Tgt &t, Own &o) {
    o.hcur = a.h[i];
    t.Hs = o.hcur * a.c_smooth;
    t.iHs = 1.0 / t.Hs;
    t.done = a.done[i] != 0;
  }
  __device__ static void pack(const Args &a, uint32_t j) {
    a.pk.d2(0)[j] = make_double2(contr_dens(a.pghost, a.bc[j]) ? a.m[j] : 0.0,
                                 __longlong_as_double((long long)a.refb[j]));
  }
  static constexpr int NA16 = 1, NA4 = 0;
  template <class L>
  __device__ static void load(const L &a, uint32_t j, Rec &r) {
    const double2 u = a.d2(0)[j];
    r = Rec{u.x, (uint32_t)__double_as_longlong(u.y)};
  }
  __device__ static double hker(const Tgt &t, double) { return t.Hs; }
  __device__ static double support(const Args &a, uint32_t i) { return a.cutoff2 * (a.h[i] * a.c_smooth); }
  __device__ static bool wants(const Tgt &t) { return !t.done; }
  __device__ static bool counts_ghost(const Args &a, int b) { return contr_dens(a.pghost, b); }
  __device__ static bool valid(const Rec &) { return true; }
  template <int D>
  __device__ static void pair_d(const Args &, const Tgt &t, const Rec &s, double, const double *dx, double, double *acc) {
    R expt = 0;
#pragma unroll
    for (int k = 0; k < D; k++) {
      const R sk = (R)dx[k] * t.iHs;
      expt += sk * sk;
    }
    acc[0] += exp_neg_w<FX>(expt) * s.m;
  }
  __device__ static bool finish(const Args &a, const Own &o, const double *sum, bool, uint32_t i, int *) {
    if (a.done[i] != 0) return true;
    const double nk = kInvSqrtPi * (1.0 / (o.hcur * a.c_smooth));
    const double rho_star = sum[0] * (a.dim == 3 ? nk * nk * nk : nk);
    const double m = a.m[i];
    const double Hnew = a.dim == 3 ? a.eta * cbrt(m / rho_star) : a.eta * (m / rho_star);
    a.h[i] = a.ratio * Hnew;
    if (fabs((Hnew - o.hcur) / o.hcur) < a.thresh) a.done[i] = 1u;
    return true;
  }
};

// ---------------------------------------------------------------------------
// Wall-ghost refresh: apply_bcond (bcond.cc:24-249) with the mirror images of
// search_bnd_images (bnd_image.cc:33-254) for a flat ground at z = zg.  Each
// wall ghost of the bucket layer that straddles the ground (bucket type
// MIXED) takes the state at its image (x, y, 2 zg - z): Shepard sums over the
// real and pressure-ghost particles j of the image's bucket and its 26
// neighbours, m_j W(s, h_j) with s = (image - x_j) / h_j inside the in_support
// box CUTOFF2 h_j, of rho, v / rho and e / rho over sum m_j W / rho_j; the
// mass fraction sums the neighbour buckets only (bcond.cc:140-146); the
// velocity is reflected in the ground plane and the EOS re-evaluated.
// Candidates come from the cell grid of the step's neighbour search, with the
// reach widened by the largest displacement since (positions have moved, the
// grid has not).  Only bc 2 entries are written and only bc 100/99/1 entries
// read, so ghosts are independent.
// ---------------------------------------------------------------------------
struct BcondArgs {
  const double *x, *y, *z, *h, *m;
  double *rho, *vx, *vy, *vz, *e, *xi, *p, *c, *T, *gam, *cp;
  const int32_t *bc;
  const uint32_t *cs, *toff;
  const float4 *tbox;        // tile boxes of the step's grid (positions at grid time)
  GridDesc g;
  double reach, zg, del, cutoff2;
  double ext_lo[3];
  int nb[3], bzg;
  CutTest cut;
  EosConst eos;
  double *wrec;              // recording for the adjoint: Shepard normaliser of each refreshed ghost
  uint32_t wrec_n;
  const double *px, *py, *pz;   // positions the support tests read (x, y, z except in a frozen replay)
};

// unit normal of the mirror plane, from a ghost towards its image
__device__ inline void mirror_normal(const double *coord, const double *refc, double *nrm) {
  double d = 0;
  for (int k = 0; k < 3; k++) { nrm[k] = refc[k] - coord[k]; d += nrm[k] * nrm[k]; }
  if (!(d > 0)) { nrm[0] = nrm[1] = 0; nrm[2] = 1; d = 1; }
  const double sd = sqrt(d);
  for (int k = 0; k < 3; k++) nrm[k] /= sd;
}

__device__ inline bool bucket_of(const BcondArgs &a, const double *p, int *b) {
  bool ok = true;
  for (int k = 0; k < 3; k++) {
    const double f = floor((p[k] - a.ext_lo[k]) / a.del);
    ok = ok && f >= 0 && f < a.nb[k];
    b[k] = ok ? (int)f : 0;
  }
  return ok;
}

// Particle::contr_image (particle.h:562-565)
__device__ inline bool contr_image(int bc) { return bc == 100 || bc == 99 || bc == 1; }

// the image of wall ghost i and its bucket, if it has one
__device__ inline bool ghost_image(const BcondArgs &a, uint32_t i, double *coord, double *refc, int *bi) {
  if (a.bc[i] != 2) return false;
  coord[0] = a.x[i]; coord[1] = a.y[i]; coord[2] = a.z[i];
  int bg[3];
  if (!bucket_of(a, coord, bg) || bg[2] != a.bzg) return false;
  refc[0] = coord[0]; refc[1] = coord[1]; refc[2] = 2 * a.zg - coord[2];
  return bucket_of(a, refc, bi);
}

// Every tile of the cell box c0..c1 for which near() (a lane per tile; a mask of
// the wave's items that the tile may concern) is not 0, by one wave, `part` of
// `parts` that share them in turn.  take(todo, count) gets up to 2 kWave of them:
// first particle, particle count, mask.
struct TileScratch {
  uint32_t rowpre[kWave], rowtile[kWave];
  uint32_t todo[2 * kWave][3];
};
template <class Near, class Take>
__device__ __forceinline__ void tiles_in_reach(const uint32_t *toff, const float4 *tbox, const GridDesc &g,
                                               const int *c0, const int *c1, TileScratch &sc, uint32_t part,
                                               uint32_t parts, Near near, Take take) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t ry = (uint32_t)(c1[1] - c0[1] + 1), rows = ry * (uint32_t)(c1[2] - c0[2] + 1);
  uint32_t nt = 0, seen = 0;
  for (uint32_t rb = 0; rb < rows; rb += kWave) {
    // the lanes take a row of cells each: its first tile, tiles up to it
    const uint32_t r = rb + lane;
    uint32_t first = 0, len = 0;
    if (r < rows) {
      const uint32_t row = ((uint32_t)(c0[2] + (int)(r / ry)) * g.ny + (uint32_t)(c0[1] + (int)(r % ry))) * g.nx;
      first = toff[row + c0[0]];
      len = toff[row + c1[0] + 1] - first;
    }
    uint32_t upto = len;
    for (uint32_t o = 1; o < kWave; o <<= 1) {
      const uint32_t v = (uint32_t)__shfl_up((int)upto, o);
      if (lane >= o) upto += v;
    }
    sc.rowpre[lane] = upto - len;
    sc.rowtile[lane] = first;
    const uint32_t ntiles = __builtin_amdgcn_readlane(upto, kWave - 1);
    const bool last = rb + kWave >= rows;         // its first turn takes what is left, also without tiles
    for (uint32_t kb = 0; kb < ntiles || (last && kb == 0); kb += kWave) {
      const uint32_t k = kb + lane;
      uint32_t m = 0, base = 0, cnt = 0;
      if (k < ntiles) {
        uint32_t ra = 0;                          // the last row that starts at or before k
        for (uint32_t o = kWave / 2; o > 0; o >>= 1)
          if (sc.rowpre[ra + o] <= k) ra += o;
        const uint32_t t = sc.rowtile[ra] + (k - sc.rowpre[ra]);
        const float4 tlo = tbox[2 * t], thi = tbox[2 * t + 1];
        base = __float_as_uint(tlo.w);
        cnt = __float_as_uint(thi.w);
        m = near(tlo, thi);
      }
      const uint64_t all = __ballot(m != 0);
      const bool mine = m != 0 && (seen + lanes_below(all)) % parts == part;
      seen += (uint32_t)__popcll(all);
      const uint64_t mt = __ballot(mine);
      if (mine) {
        uint32_t *e = sc.todo[nt + lanes_below(mt)];
        e[0] = base; e[1] = cnt; e[2] = m;
      }
      nt += (uint32_t)__popcll(mt);
      if (nt > kWave || (last && kb + kWave >= ntiles)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        take(sc.todo, nt);
        nt = 0;
      }
    }
  }
}

// of the tiles in todo (count of them), those that hold a particle for which
// of(j) is true, moved to the front; four tiles' loads at a time
template <class Of>
__device__ __forceinline__ uint32_t tiles_holding(uint32_t (*todo)[3], uint32_t count, Of of) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  uint32_t kept = 0;
  for (uint32_t t = 0; t < count; t += 4) {
    uint32_t e[4][3];
    bool has[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const uint32_t *p = todo[min(t + u, count - 1)];
      for (int d = 0; d < 3; d++) e[u][d] = __builtin_amdgcn_readfirstlane(p[d]);
      has[u] = of(e[u][0] + min(lane, e[u][1] - 1u));
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (t + u >= count || !__any(has[u])) continue;
      if (lane < 3) todo[kept][lane] = lane == 0 ? e[u][0] : lane == 1 ? e[u][1] : e[u][2];
      kept++;
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  return kept;
}

// the largest per-axis distance of r from a tile's box
__device__ inline double box_distance(const float4 &lo, const float4 &hi, const double *r) {
  return fmax(fmax(fmax((double)lo.x - r[0], r[0] - (double)hi.x), fmax((double)lo.y - r[1], r[1] - (double)hi.y)),
              fmax((double)lo.z - r[2], r[2] - (double)hi.z));
}

// Wall-ghost refresh.  A workgroup takes kBcondGroup consecutive particles that
// hold an imaged ghost (in cell order, so their images are compact); its waves
// share the tiles within reach.  A wave tests the tiles, a lane each, drops
// those without a contributor, then takes the others in turn: a particle a
// lane, whose weight and fields stay in registers while the images pass by, and
// whose successor's loads are under way meanwhile.  Each lane adds its
// particle's share to every ghost's sums; they are summed over lanes and waves
// at the end, in a fixed order.
//
// Bound by VALU issue (57 % of the time at 228k particles), then by the chain of
// loads row, tile, particle.  A lane per ghost that walked its own hits ran as
// long as the fullest lane and left the chip to one wave per 32 particles, most
// of them without a ghost: us per refresh 600 -> 118 at 228k particles (30k
// real), 962 -> 396 at 1M, 1440 -> 888 at 4M.  8 ghosts by 2 waves of 2 per
// SIMD; 4 ghosts by 2 waves of 3 per SIMD take 127, 435, 984, by 4 waves 132,
// 498, 1149: a group's own work (images, rows, tile tests) is done by each wave.
constexpr int kBcondGroup = 8;                 // consecutive particles: 7 sums each in registers
constexpr int kBcondWaves = 2;
constexpr unsigned kBcondGrid = 1024;          // workgroups: 4 per CU, all resident

// the groups with an imaged ghost, in any order (a group's result does not
// depend on its place)
__global__ void k_bcond_list(uint32_t n, BcondArgs a, uint32_t *list, unsigned long long *count) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  double coord[3], refc[3];
  int bi[3];
  const uint64_t act = __ballot(i < n && ghost_image(a, i, coord, refc, bi));
  const bool first = lane % kBcondGroup == 0 && ((act >> lane) & ((1u << kBcondGroup) - 1));
  const uint64_t has = __ballot(first);
  if (!has) return;
  uint32_t at = 0;
  if (lane == 0) at = (uint32_t)atomicAdd(count, (unsigned long long)__popcll(has));
  at = __builtin_amdgcn_readfirstlane(at);
  if (first) list[at + lanes_below(has)] = i / kBcondGroup;
}

// the four values' sums over the wave: row r of 16 lanes gets value r's, in
// every lane
__device__ inline double wave_sum4(double v0, double v1, double v2, double v3) {
  double v = swap_add<1>(swap_add<2>(v0, v2), swap_add<2>(v1, v3));
  v += row_move<0x128>(v);                        // row_ror 8, 4, 2, 1
  v += row_move<0x124>(v);
  v += row_move<0x122>(v);
  v += row_move<0x121>(v);
  return v;
}

// a candidate as it lies in memory
template <bool FROZEN>
struct BcondRaw {
  double x, y, z, h, m, rho, vx, vy, vz, e, xi, px, py, pz;
  int bc;
  __device__ void read(const BcondArgs &a, const uint32_t *tile, int lane) {
    const uint32_t j = __builtin_amdgcn_readfirstlane(tile[0]) +
                       min((uint32_t)lane, __builtin_amdgcn_readfirstlane(tile[1]) - 1u);
    bc = a.bc[j];
    x = a.x[j]; y = a.y[j]; z = a.z[j];
    if constexpr (FROZEN) { px = a.px[j]; py = a.py[j]; pz = a.pz[j]; }
    h = a.h[j]; m = a.m[j]; rho = a.rho[j];
    vx = a.vx[j]; vy = a.vy[j]; vz = a.vz[j];
    e = a.e[j]; xi = a.xi[j];
  }
};

// FROZEN: a frozen replay, where the support tests read px, py, pz
template <bool FROZEN>
__global__ __launch_bounds__(kBcondWaves * kWave, 2) void k_bcond(uint32_t n, BcondArgs a, const uint32_t *list,
                                                                const unsigned long long *count) {
  constexpr int NS = 7;                           // rho, v, e, normaliser, xi
  __shared__ double part[2][kBcondWaves][NS][kBcondGroup];
  struct Image { double r[3]; int b[3]; };
  // a wave's own: the images are read back where used, not kept in registers
  __shared__ Image image[kBcondWaves][kBcondGroup];
  __shared__ TileScratch scratch[kBcondWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t total = __builtin_amdgcn_readfirstlane((uint32_t)*count);
  // an XCD's workgroups share a stretch of the list
  const uint32_t per = (total + kXcds - 1) / kXcds, xcd = blockIdx.x % kXcds;
  const uint32_t end = min(total, (xcd + 1) * per);
  uint32_t turn = 0;
  for (uint32_t k = xcd * per + blockIdx.x / kXcds; k < end; k += gridDim.x / kXcds, turn++) {
    const uint32_t i = __builtin_amdgcn_readfirstlane(list[k]) * kBcondGroup + (uint32_t)lane;
    double at[3], refc[3] = {0, 0, 0};
    int bi[3] = {0, 0, 0};
    const bool act = lane < kBcondGroup && i < n && ghost_image(a, i, at, refc, bi);
    Image *img = image[wave];
    const uint32_t acts = (uint32_t)__ballot(act);
    if (lane < kBcondGroup)
      for (int d = 0; d < 3; d++) { img[lane].r[d] = refc[d]; img[lane].b[d] = bi[d]; }
    double lo[3], hi[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      lo[d] = act ? refc[d] : HUGE_VAL;
      hi[d] = act ? refc[d] : -HUGE_VAL;
      for (int o = 1; o < kBcondGroup; o <<= 1) {
        lo[d] = fmin(lo[d], __shfl_xor(lo[d], o));
        hi[d] = fmax(hi[d], __shfl_xor(hi[d], o));
      }
    }
    int c0[3], c1[3];
    const int nn[3] = {a.g.nx, a.g.ny, a.g.nz};
    for (int d = 0; d < 3; d++) {
      c0[d] = c1[d] = 0;
      if (a.g.inv_e > 0) {
        c0[d] = __builtin_amdgcn_readfirstlane(cell_of(lo[d] - a.reach, a.g.lo[d], a.g.inv_e, nn[d]));
        c1[d] = __builtin_amdgcn_readfirstlane(cell_of(hi[d] + a.reach, a.g.lo[d], a.g.inv_e, nn[d]));
      }
    }
    double s[NS][kBcondGroup];
#pragma unroll
    for (int q = 0; q < NS; q++)
      for (int g = 0; g < kBcondGroup; g++) s[q][g] = 0;
    tiles_in_reach(a.toff, a.tbox, a.g, c0, c1, scratch[wave], wave, kBcondWaves, [&](const float4 &tlo, const float4 &thi) {
      // A tile's particles have moved by at most the displacement that the
      // reach includes: its box at grid time within reach of an image is
      // necessary for any of them to be within the kernel box now.
      uint32_t near = 0;
#pragma unroll
      for (int g = 0; g < kBcondGroup; g++) near |= box_distance(tlo, thi, img[g].r) <= a.reach ? 1u << g : 0u;
      return near & acts;
    }, [&](uint32_t (*todo)[3], uint32_t nt) {
      // without the tiles that hold no contributor (wall ghosts only)
      const uint32_t kept = tiles_holding(todo, nt, [&](uint32_t j) { return contr_image(a.bc[j]); });
      BcondRaw<FROZEN> nx;
      if (kept) nx.read(a, todo[0], lane);
      for (uint32_t t = 0; t < kept; t++) {
        const BcondRaw<FROZEN> c = nx;
        const uint32_t gm = __builtin_amdgcn_readfirstlane(todo[t][2]);
        const uint32_t n_in = __builtin_amdgcn_readfirstlane(todo[t][1]);
        if (t + 1 < kept) nx.read(a, todo[t + 1], lane);
        double q[3] = {c.x, c.y, c.z};
        if constexpr (FROZEN) { q[0] = c.px; q[1] = c.py; q[2] = c.pz; }
        int bj[3];
        const bool ok = (uint32_t)lane < n_in && contr_image(c.bc) && bucket_of(a, q, bj);
        const double ih = rcp_newton(c.h), ih2 = ih * ih, nk = kInvSqrtPi * ih;
        const double mk = c.m * (nk * nk * nk), mr = mk * rcp_newton(c.rho);
#pragma unroll
        for (int g = 0; g < kBcondGroup; g++) {
          if (!((gm >> g) & 1)) continue;
          asm volatile("" ::: "memory");
          const double r0 = img[g].r[0], r1 = img[g].r[1], r2 = img[g].r[2];
          const int d0 = bj[0] - img[g].b[0], d1 = bj[1] - img[g].b[1], d2 = bj[2] - img[g].b[2];
          const double amax = fmax(fabs(r0 - q[0]), fmax(fabs(r1 - q[1]), fabs(r2 - q[2])));
          const bool nb = max(abs(d0), max(abs(d1), abs(d2))) <= 1;
          // in_support; W = 0 outside the kernel box
          if (ok & nb & (amax <= a.cutoff2 * c.h) & !a.cut.outside(amax, c.h)) {
            const double dx = r0 - c.x, dy = r1 - c.y, dz = r2 - c.z;
            const double ex = exp_neg((dx * dx + dy * dy + dz * dz) * ih2);
            const double w = mr * ex;
            s[0][g] = fma(mk, ex, s[0][g]);
            s[1][g] = fma(w, c.vx, s[1][g]);
            s[2][g] = fma(w, c.vy, s[2][g]);
            s[3][g] = fma(w, c.vz, s[3][g]);
            s[4][g] = fma(w, c.e, s[4][g]);
            s[5][g] += w;
            s[6][g] = fma(w, (d0 | d1 | d2) != 0 ? c.xi : 0.0, s[6][g]);   // not from the image's own bucket
          }
        }
      }
    });
    double (*pt)[NS][kBcondGroup] = part[turn & 1];
#pragma unroll
    for (int q = 0; q < NS; q++)
#pragma unroll
      for (int g = 0; g < kBcondGroup; g += 4) {
        const double v = wave_sum4(s[q][g], s[q][g + 1], s[q][g + 2], s[q][g + 3]);
        if (lane % 16 == 0) pt[wave][q][g + lane / 16] = v;
      }
    __syncthreads();
    // a wave in turn finishes; the others go on with the next group, and its
    // sums' places are written again only past the next barrier
    if (wave != turn % kBcondWaves || lane >= kBcondGroup || !((acts >> lane) & 1)) continue;
    asm volatile("" ::: "memory");
    const double coord[3] = {a.x[i], a.y[i], a.z[i]}, *mirror = img[lane].r;
    double u[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) {
      u[q] = 0;
      for (int w = 0; w < kBcondWaves; w++) u[q] += pt[w][q][lane];
    }
    const double wnorm = u[5];
    if (a.wrec && i < a.wrec_n) a.wrec[i] = wnorm;
    double nrm[3];
    mirror_normal(coord, mirror, nrm);
    if (wnorm > 0) {
      u[0] /= wnorm; u[1] /= wnorm; u[2] /= wnorm; u[3] /= wnorm; u[4] /= wnorm;
      u[6] /= wnorm;
    } else {
      u[0] = 1; u[1] = u[2] = u[3] = u[4] = 0; u[6] = 0;
    }
    const double vdotn = u[1] * nrm[0] + u[2] * nrm[1] + u[3] * nrm[2];
    a.rho[i] = u[0];
    a.vx[i] = u[1] - 2 * vdotn * nrm[0];
    a.vy[i] = u[2] - 2 * vdotn * nrm[1];
    a.vz[i] = u[3] - 2 * vdotn * nrm[2];
    a.e[i] = u[4];
    a.xi[i] = u[6];
    double p, c, T, gam, cp = a.cp[i];
    eos_dev(a.eos, u[0], u[4], u[6], p, c, T, gam, &cp);
    a.p[i] = p; a.c[i] = c; a.T[i] = T; a.gam[i] = gam; a.cp[i] = cp;
  }
}

// ---------------------------------------------------------------------------
// Position update + escape (update_pos.cc:34-168, bucket.cc:435-452)
// ---------------------------------------------------------------------------
// Schedule of a recorded run: tmode 1 records, by particle id, the tape step
// at which an erupt ghost turns real and a real particle escapes; tmode 2
// replays those events instead of testing positions.
struct PosTape {
  int mode;
  int32_t k;
  const uint32_t *pid;
  int32_t *tr_step, *esc_step;
};

// Then, of what is left: the real particles (bc 100/99), and the largest per-axis
// speed of the particles that move (reals with the filtered velocity under LANS,
// erupt ghosts with v).  Grid-stride, an atomic a block each.
__global__ __launch_bounds__(256) void k_update_pos(
    uint32_t n, int dim, int lans, int erupting, double dt, double *x, double *y, double *z, const double *vx,
    const double *vy, const double *vz, const double *svx, const double *svy, const double *svz, int32_t *bc, double *h,
    int32_t *inv, double ground, double h_new, double lo0, double lo1, double lo2, double hi0, double hi1, double hi2,
    unsigned long long *words, PosTape tp) {
  __shared__ unsigned int part[256 / kWave];
  if (halted((const int *)(words + W_ERR), 4)) return;
  unsigned int reals = 0;
  double vmax = 0;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    int b = bc[i];
    const bool was_real = is_real(b);
    if (!was_real && b != 0) continue;
    const double v[3] = {vx[i], vy[i], vz[i]};
    double u[3] = {v[0], v[1], v[2]};              // of a real particle
    if (lans && (was_real || erupting)) { u[0] = svx[i]; u[1] = svy[i]; u[2] = svz[i]; }
    if (was_real) {
      x[i] = x[i] + dt * u[0];
      if (dim == 3) { y[i] = y[i] + dt * u[1]; z[i] = z[i] + dt * u[2]; }
    } else if (erupting) {
      x[i] = x[i] + dt * v[0];
      if (dim == 3) {
        y[i] = y[i] + dt * v[1];
        z[i] = z[i] + dt * v[2];
        const bool turn = tp.mode == 2 ? tp.tr_step[tp.pid[i]] == tp.k : z[i] >= ground;
        if (turn) {
          b = 100; bc[i] = 100; h[i] = h_new; inv[i] = 2;
          if (tp.mode == 1) tp.tr_step[tp.pid[i]] = tp.k;
        }
      }
    }
    if (dim == 3 && is_real(b)) {
      const double TINY = 1.0E-08;
      bool esc = (x[i] - lo0) < -TINY || (y[i] - lo1) < -TINY || (z[i] - lo2) < -TINY ||
                 (x[i] - hi0) > TINY || (y[i] - hi1) > TINY || (z[i] - hi2) > TINY;
      if (tp.mode == 2) esc = tp.esc_step[tp.pid[i]] == tp.k;
      if (esc) {
        b = -1; bc[i] = -1; atomicAdd(words + W_DEAD, 1ull);
        if (tp.mode == 1) tp.esc_step[tp.pid[i]] = tp.k;
      }
    }
    reals += is_real(b) ? 1u : 0u;
    if (is_real(b)) vmax = fmax(vmax, fmax(fabs(u[0]), fmax(fabs(u[1]), fabs(u[2]))));
    else if (b == 0) vmax = fmax(vmax, fmax(fabs(v[0]), fmax(fabs(v[1]), fabs(v[2]))));
  }
  vmax = block_ext<true>(vmax);
  for (int o = kWave / 2; o > 0; o >>= 1) reals += (unsigned int)__shfl_xor((int)reals, o);
  if ((threadIdx.x & (kWave - 1)) == 0) part[threadIdx.x / kWave] = reals;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long sum = 0;
    for (int w = 0; w < 256 / kWave; w++) sum += part[w];
    if (sum) atomicAdd(words + W_REAL, sum);
    if (vmax > 0) atomicMax(words + W_VMAX, (unsigned long long)__double_as_longlong(vmax));
  }
}

// live particles and, of them, the real ones: grid-stride, an atomic a block each
__global__ __launch_bounds__(256) void k_count_live(uint32_t n, const int32_t *bc, unsigned long long *out) {
  __shared__ unsigned int part[2][256 / kWave];
  unsigned int cnt[2] = {0, 0};
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int b = bc[i];
    cnt[0] += b >= 0 ? 1u : 0u;
    cnt[1] += is_real(b) ? 1u : 0u;
  }
  for (int q = 0; q < 2; q++) {
    for (int o = kWave / 2; o > 0; o >>= 1) cnt[q] += (unsigned int)__shfl_xor((int)cnt[q], o);
    if ((threadIdx.x & (kWave - 1)) == 0) part[q][threadIdx.x / kWave] = cnt[q];
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    unsigned long long sum = 0;
    for (int w = 0; w < 256 / kWave; w++) sum += part[threadIdx.x][w];
    if (sum) atomicAdd(out + threadIdx.x, sum);
  }
}

// THashTable order (thashtab.cc:209-262) by three stable sorts, the last key
// first: key2; key0 and key1; the slot, with the removed particles past every
// slot.  The keys of the particles in the order that perm has so far:
__global__ void k_read_key01(uint32_t n, const uint32_t *perm, const uint32_t *k0, const uint32_t *k1, uint64_t *key) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = perm[i];
  key[i] = (uint64_t)k0[j] << 32 | k1[j];
}
// the slot as table_slot has it (psph_host.cpp): quotient, product and sum of the
// parts each rounded as there
__global__ void k_read_slot(uint32_t n, const uint32_t *perm, const uint32_t *k0, const uint32_t *k1, const int32_t *bc,
                            int table_size, int dim, uint64_t *key) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = perm[i];
  uint32_t slot = k0[j];                             // 1D: the hash is key0
  if (dim != 1) {
    const double umax = 4294967295.0;
    const int s2 = table_size / 10, s1 = table_size - s2;
    const int i1 = (int)((double)k0[j] / umax * s1), i2 = (int)((double)k1[j] / umax * s2);
    slot = (uint32_t)(i1 + i2) ^ 0x80000000u;        // (the sum of the sizes is an int)
  }
  key[i] = (bc[j] < 0 ? (uint64_t)1 << 32 : 0) | slot;
}

__global__ void k_iota_u32(uint32_t *p, uint32_t first, uint32_t n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = first + i;
}
// tab[id] = h (record) or h = tab[id] (replay) for the particles present
__global__ void k_h_by_id(uint32_t n, const uint32_t *pid, double *h, double *tab, int replay) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (replay) h[i] = tab[pid[i]];
  else tab[pid[i]] = h[i];
}

// positions of a step by particle id (rec: x block, y block, z block of nrec)
__global__ void k_pos_to_rec(uint32_t n, const uint32_t *pid, const double *x, const double *y, const double *z,
                             double *rec, uint32_t nrec) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t id = pid[i];
  if (id >= nrec) return;
  rec[id] = x[i]; rec[(size_t)nrec + id] = y[i]; rec[2 * (size_t)nrec + id] = z[i];
}
// and back, into the current order; a live particle without a record is an
// error (the replay no longer follows the recorded run)
__global__ void k_pos_from_rec(uint32_t n, const uint32_t *pid, const int32_t *bc, const double *rec,
                               uint32_t nrec, const double *x, const double *y, const double *z, double *px,
                               double *py, double *pz, int *err) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t id = pid[i];
  if (bc[i] < 0 || id >= nrec) {
    if (bc[i] >= 0) raise_err(err, PSPH_EINVARIANT, i);
    px[i] = x[i]; py[i] = y[i]; pz[i] = z[i];
    return;
  }
  px[i] = rec[id]; py[i] = rec[(size_t)nrec + id]; pz[i] = rec[2 * (size_t)nrec + id];
}

// fixed-order block partial sums (deterministic)
constexpr int kRedBlocks = 512;
__global__ void k_conservation(uint32_t n, const int32_t *bc, const double *m, const double *e,
                               const double *vx, const double *vy, const double *vz,
                               const double *xi, const double *z, double *part) {
  __shared__ double sh[8][256];
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    int b = bc[i];
    if (!(b == 100 || b == 99)) continue;
    double mi = m[i], v0 = vx[i], v1 = vy ? vy[i] : 0, v2 = vz ? vz[i] : 0;
    acc[0] += mi;
    acc[1] += mi * e[i];
    acc[2] += 0.5 * mi * (v0 * v0 + v1 * v1 + v2 * v2);
    acc[3] += mi * v0; acc[4] += mi * v1; acc[5] += mi * v2;
    acc[6] += mi * xi[i];
    acc[7] += mi * xi[i] * (z ? z[i] : 0);
  }
  for (int k = 0; k < 8; k++) sh[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int k = 0; k < 8; k++) sh[k][threadIdx.x] += sh[k][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 0; k < 8; k++) part[blockIdx.x * 8 + k] = sh[k][0];
}

inline unsigned blocks(size_t n, unsigned b = 256) { return (unsigned)((n + b - 1) / b); }
// grid of a grid-stride reduction: enough blocks to fill the chip, no more, and
// 8 elements a thread where they are few (the blocks' atomics on one word take
// their turns: the least h / c of 227k particles 24 us with one element, 12 so)
inline unsigned red_blocks(size_t n) { return std::min(blocks(n, 8 * 256), 2048u); }

}  // namespace

// ===========================================================================
// Context
// ===========================================================================
#define PSPH_DFIELDS(F) F(x) F(y) F(z) F(vx) F(vy) F(vz) F(svx) F(svy) F(svz) F(rho) F(e) F(m) \
  F(h) F(p) F(c) F(T) F(gam) F(cp) F(xi)
#define PSPH_UFIELDS(F) F(k0) F(k1) F(k2)
#define PSPH_IFIELDS(F) F(bc) F(phase) F(inv)

struct DevFields {
#define D_(a) double *a = nullptr;
#define U_(a) uint32_t *a = nullptr;
#define I_(a) int32_t *a = nullptr;
  PSPH_DFIELDS(D_) PSPH_UFIELDS(U_) PSPH_IFIELDS(I_)
#undef D_
#undef U_
#undef I_
};

// Frozen schedule of a recorded run (the adjoint and its finite-difference
// checks differentiate the step map with these discrete choices held fixed).
struct Tape {
  int mode = 0;                             // 0 off, 1 record, 2 replay
  int64_t k = 0;                            // steps taken since the start of the tape
  double t0 = 0;
  int64_t step0 = 0;
  size_t n0 = 0;
  std::vector<double> dt;                   // per step, after TimeProps::incrtime
  std::vector<int> hslot;                   // per step: adapted-h table, or -1
  std::vector<double *> htab;               // smoothing lengths after adaptation, by particle id
  std::vector<std::vector<int32_t>> inlet;  // per step: (q, n) per vent column
  int32_t *tr_step = nullptr, *esc_step = nullptr;   // by id, -1 = never
  size_t id_cap = 0;
  // Positions at each step's neighbour search, by particle id (x block, y
  // block, z block of xrec_n[k] entries).  A replay with `frozen` set builds
  // its cell order, tiles, visit lists and every pair predicate (kernel
  // boxes, list membership, support) from these, and only the pair
  // arithmetic from its own positions: the pair set and the summation order
  // are the recorded run's, so a finite difference through the replay sees
  // no kernel-box face crossings, as the adjoint does not.
  std::vector<double *> xrec;
  std::vector<uint32_t> xrec_n;
  // with cfg.wall_bc, the same at each step's wall-ghost refresh (after
  // update_pos): a frozen replay's refresh takes its contributor sets from them
  std::vector<double *> xrecb;
  std::vector<uint32_t> xrecb_n;
  bool frozen = false;
};

// What the reverse sweep needs of one step, in that step's cell order.
enum RecField {
  RF_X, RF_Y, RF_Z, RF_H, RF_M, RF_RHO, RF_P, RF_C, RF_T, RF_CP, RF_SVX, RF_SVY, RF_SVZ,
  RF_VX, RF_VY, RF_VZ, RF_E, RF_HLIST,                  // state after sort and h update
  RF_V1X, RF_V1Y, RF_V1Z, RF_E1,                         // after the RHS update
  RF_RHO2, RF_E2, RF_XI2, RF_WNE,                        // after the density pass
  RF_SV2X, RF_SV2Y, RF_SV2Z, RF_WNV,                     // after the velocity filter
  // wall-ghost refresh (only with cfg.wall_bc): positions after update_pos,
  // the refreshed ghost fields and each ghost's Shepard normaliser
  RF_XN, RF_YN, RF_ZN, RF_BRHO, RF_BVX, RF_BVY, RF_BVZ, RF_BE, RF_BXI, RF_BW,
  RF_N
};
constexpr int RF_NBASE = RF_XN;                          // fields recorded in every step
struct StepRec {
  size_t n = 0, cap = 0;
  double *d[RF_N] = {};
  uint32_t *pid = nullptr, *refb = nullptr, *ckey = nullptr;
  uint32_t *gflag = nullptr;                  // boundary ghosts met as neighbours in this step
  int32_t *bc = nullptr, *phase = nullptr;
  int32_t *bcn = nullptr;                     // bc after update_pos (wall-ghost refresh only)
  uint32_t *cs = nullptr, *toff = nullptr;   // cell starts and first tile of each cell
  float4 *tbox = nullptr;                     // tile boxes
  size_t cs_cap = 0, tile_cap = 0;
  GridDesc grid{};
  double reach = 0;
  double hmax = 0;                            // bounds h at list time
  double dt = 0, time = 0;
  int erupting = 0;
  uint32_t inj_lo = 0, inj_hi = 0;          // ids of the particles this step injected
  std::vector<double> inj_vel;              // their column exit velocity
};
struct Adjoint;

struct psph_ctx {
  psph_config cfg{};
  hipStream_t stream = nullptr;
  size_t cap = 0, n = 0;
  DevFields f;
  double *dsp[10] = {};        // spare double arrays (gather / double buffers)
  uint32_t *usp = nullptr;     // spare u32 array
  int32_t *isp = nullptr;      // spare i32 array
  double *h_list = nullptr;
  uint32_t *refb = nullptr, *key_a = nullptr, *key_b = nullptr, *idx_a = nullptr, *idx_b = nullptr;
  uint32_t *targets = nullptr;
  uint32_t *cfirst = nullptr, *ccount = nullptr;
  uint32_t *cs = nullptr, *toff = nullptr, *nchunks = nullptr;
  CellSum *cell_has = nullptr, *cell_at = nullptr;   // per cell: its contents, and of the cells before
  float4 *tbox = nullptr;
  size_t cs_cap = 0, tile_cap = 0, chunk_cap = 0;
  void *cub = nullptr;
  size_t cub_bytes = 0;
  unsigned long long *words = nullptr;   // on the device (Word)
  unsigned long long *seen = nullptr;    // their last copy, in pinned memory; then 2 words of lists' cursors
  char *up_h = nullptr, *up_d = nullptr; // particles on their way to the device (upload)
  bool up_busy = false;
  bool loaded_removed = false;           // removed particles (bc < 0) among those loaded
  double *d_part = nullptr;
  // grid of the last neighbour search
  bool grid_valid = false;
  GridDesc grid{};
  double reach_main = 0;       // per-axis reach of the RHS / density / filter predicates
  // the group passes' lists and positions (made once per step) and particle records
  bool lists_valid = false;
  uint4 *gvisit = nullptr;
  uint32_t *goff = nullptr, *gnum = nullptr, *gfast = nullptr;
  uint32_t ngroups = 0;              // of the lists last built
  unsigned long long *gcursor = nullptr;
  size_t gchunk_cap = 0;
  uint32_t gvisit_cap = 0;
  double2 *gxy = nullptr, *gzh = nullptr;
  void *pk[5] = {};
  double h_max = 0;
  // clock (TimeProps)
  double time = 0, next_output = 0;
  int64_t step = 0;
  int ioutput = 0;
  int64_t last_injected = 0, last_removed = 0, last_real = -1;
  unsigned long long last_pairs = 0;
  HostParticles inj;
  // persistent particle ids: load order, then injection order
  uint32_t *pid = nullptr, *pid_sp = nullptr;
  uint32_t next_pid = 0;
  // positions the pair predicates read in a frozen replay (Tape::xrec)
  double *px = nullptr, *py = nullptr, *pz = nullptr;
  // domain adaptation (psph_domain_init, psph_domain.inl)
  DomainBuckets dom;
  bool dom_ready = false;
  int dom_pending = 0;                 // scan_outside_layer's count of the last step
  std::vector<double> met_z, met_data;
  psph_meteo met{};
  uint32_t dom_seed = 0;
  double dom_jitter = 0;
  uint32_t *d_occ = nullptr;
  uint8_t *d_conv = nullptr, *d_sides = nullptr;
  int64_t last_domain = 0;
  Tape tape;
  StepRec *rec = nullptr;      // set: psph_step captures the step for the reverse sweep
  Adjoint *adj = nullptr;
  // per-stage HIP-event timing
  bool prof = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double prof_ms[PSPH_NSTAGES] = {};
  int64_t prof_n[PSPH_NSTAGES] = {};
};

// Brackets the main kernel(s) of a stage with events on the context stream.
struct StageTimer {
  psph_ctx *c;
  int id;
  StageTimer(psph_ctx *ctx, int stage) : c(ctx), id(stage) {
    if (c->prof) (void)hipEventRecord(c->ev0, c->stream);
  }
  void stop() {
    if (!c->prof || id < 0) return;
    (void)hipEventRecord(c->ev1, c->stream);
    (void)hipEventSynchronize(c->ev1);
    float ms = 0;
    if (hipEventElapsedTime(&ms, c->ev0, c->ev1) == hipSuccess) {
      c->prof_ms[id] += ms;
      c->prof_n[id] += 1;
    }
    id = -1;
  }
  ~StageTimer() { stop(); }
};

static int dmalloc(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes ? bytes : 8);
  if (e != hipSuccess) {
    (void)hipGetLastError();             // reported here, not again by the next check
    *p = nullptr;
    return fail(PSPH_ENOMEM, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
  }
  return 0;
}

// c->seen = the words, after everything queued so far
static int read_words(psph_ctx *c) {
  HIP_TRY(hipMemcpyAsync(c->seen, c->words, W_COUNT * 8, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  c->up_busy = false;
  return 0;
}
static double seen_double(const psph_ctx *c, Word w) {
  double v;
  std::memcpy(&v, &c->seen[w], 8);
  return v;
}
// the first error word that is set in c->seen; stage: what W_ERR stands for
static int seen_err(psph_ctx *c, const char *stage) {
  const char *names[] = {stage, "rhs", "density", "vsmooth"};
  for (int q = 0; q < 4; q++) {
    int he[2];
    std::memcpy(he, &c->seen[W_ERR + q], 8);
    if (!he[0]) continue;
    hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words + W_ERR, 0ull, 4);
    return fail(he[0], "%s: invariant violated at device particle %d (density<=0, mass fraction>1, "
                       "wnorm<=0 or sound speed<=0)", names[q], he[1]);
  }
  return 0;
}
static int check_err(psph_ctx *c, const char *stage) {
  PSPH_TRY(read_words(c));
  return seen_err(c, stage);
}

static int ensure_cub(psph_ctx *c, size_t bytes) {
  if (bytes <= c->cub_bytes) return 0;
  if (c->cub) hipFree(c->cub);
  c->cub = nullptr;
  PSPH_TRY(dmalloc(&c->cub, bytes));
  c->cub_bytes = bytes;
  return 0;
}

extern "C" int psph_create(const psph_config *cfg, size_t capacity, psph_ctx **out) {
  if (!cfg || !out) return fail(PSPH_EINVAL, "null argument");
  if (cfg->dim != 1 && cfg->dim != 3) return fail(PSPH_EINVAL, "dim must be 1 or 3");
  if (cfg->precision != PSPH_FP64 && cfg->precision != PSPH_FP32_PAIR && cfg->precision != PSPH_FP32_PURE &&
      cfg->precision != PSPH_FP32_EXP)
    return fail(PSPH_EINVAL, "unknown precision form %d", cfg->precision);
  if (cfg->kernel != PSPH_KERNEL_GAUSS_BOX)
    return fail(PSPH_EINVAL, "kernel %d: the reference's one kernel, the Gaussian box (PSPH_KERNEL_GAUSS_BOX), "
                             "is the only one", cfg->kernel);
  if (!(cfg->h_air > 0)) return fail(PSPH_EINVAL, "h_air must be > 0");
  {
    uint64_t bits;
    std::memcpy(&bits, &cfg->cutoff, 8);
    if (!(cfg->cutoff > 0) || (bits & 1u))
      return fail(PSPH_ENOTSUP, "cutoff %g: the exact kernel-box test needs a positive cut-off with an even "
                                "last significand bit", cfg->cutoff);
  }
  if (cfg->dim == 3 && !(cfg->bucket_edge > 0)) return fail(PSPH_EINVAL, "call psph_config_domain first");
  if (capacity < 64) capacity = 64;
  if (capacity > 0xffffff00u) return fail(PSPH_EINVAL, "capacity above 2^32 particles");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(PSPH_EHIP, "no HIP device");
  psph_ctx *c = new psph_ctx();
  c->cfg = *cfg;
  c->cap = capacity;
  int rc = 0;
  if (hipStreamCreate(&c->stream) != hipSuccess) { delete c; return fail(PSPH_EHIP, "hipStreamCreate"); }
#define A_(a) if (!rc) rc = dmalloc((void **)&c->f.a, capacity * sizeof(*c->f.a));
  PSPH_DFIELDS(A_) PSPH_UFIELDS(A_) PSPH_IFIELDS(A_)
#undef A_
  for (int k = 0; k < 10 && !rc; k++) rc = dmalloc((void **)&c->dsp[k], capacity * 8);
  if (!rc) rc = dmalloc((void **)&c->usp, capacity * 4);
  if (!rc) rc = dmalloc((void **)&c->isp, capacity * 4);
  if (!rc) rc = dmalloc((void **)&c->h_list, capacity * 8);
  if (!rc) rc = dmalloc((void **)&c->pid, capacity * 4);
  if (!rc) rc = dmalloc((void **)&c->pid_sp, capacity * 4);
  uint32_t **u32s[] = {&c->refb, &c->key_a, &c->key_b, &c->idx_a, &c->idx_b, &c->targets};
  for (auto pp : u32s)
    if (!rc) rc = dmalloc((void **)pp, capacity * 4);
  if (!rc) rc = dmalloc((void **)&c->words, W_COUNT * 8);
  if (!rc) { c->gcursor = c->words + W_CURSOR; c->nchunks = (uint32_t *)(c->words + W_CHUNKS); }
  if (!rc && hipHostMalloc((void **)&c->seen, (W_COUNT + 2) * 8, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    c->seen = nullptr;
    rc = fail(PSPH_ENOMEM, "hipHostMalloc");
  }
  if (!rc) rc = dmalloc((void **)&c->d_part, kRedBlocks * 8 * 8);
  if (rc) { psph_destroy(c); return rc; }
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words, 0ull, W_COUNT);
  c->next_output = cfg->t_output;
  *out = c;
  return 0;
}

static void adjoint_free(psph_ctx *c);
static void tape_clear(Tape &tp);

extern "C" int psph_destroy(psph_ctx *c) {
  if (!c) return 0;
  if (c->stream) hipStreamSynchronize(c->stream);
  adjoint_free(c);
  tape_clear(c->tape);
  if (c->tape.tr_step) hipFree(c->tape.tr_step);
  if (c->tape.esc_step) hipFree(c->tape.esc_step);
#define F_(a) if (c->f.a) hipFree(c->f.a);
  PSPH_DFIELDS(F_) PSPH_UFIELDS(F_) PSPH_IFIELDS(F_)
#undef F_
  for (auto p : c->dsp) if (p) hipFree(p);
  void *ptrs[] = {c->usp, c->isp, c->h_list, c->pid, c->pid_sp, c->refb, c->key_a, c->key_b, c->idx_a, c->idx_b,
                  c->targets, c->cfirst, c->ccount, c->cs, c->toff, c->cell_has, c->cell_at, c->tbox, c->cub, c->words, c->up_d, c->d_part,
                  c->gvisit, c->goff, c->gnum, c->gfast, c->gxy, c->gzh, c->px, c->py, c->pz,
                  c->d_occ, c->d_conv, c->d_sides};
  for (auto p : ptrs) if (p) hipFree(p);
  for (auto p : c->pk) if (p) hipFree(p);
  if (c->seen) hipHostFree(c->seen);
  if (c->up_h) hipHostFree(c->up_h);
  if (c->ev0) hipEventDestroy(c->ev0);
  if (c->ev1) hipEventDestroy(c->ev1);
  if (c->stream) hipStreamDestroy(c->stream);
  delete c;
  return 0;
}

// Up to kUpload particles go through pinned memory in one copy and a kernel that
// takes the fields apart, and nobody waits: the 25 copies of an inlet's few
// particles, each waited for, took about 0.2 ms of a step.
constexpr size_t kUpload = 4096;
constexpr size_t kUploadBytes = 19 * 8 + 6 * 4;      // of a particle
__global__ void k_append(uint32_t n, uint32_t at, const char *from, DevFields f) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *d = (const double *)from + i;
  const uint32_t *u = (const uint32_t *)(from + (size_t)n * 19 * 8) + i;
#define A_(a) f.a[at + i] = *d; d += n;
  PSPH_DFIELDS(A_)
#undef A_
#define A_(a) f.a[at + i] = *u; u += n;
  PSPH_UFIELDS(A_)
#undef A_
#define A_(a) f.a[at + i] = (int32_t)*u; u += n;
  PSPH_IFIELDS(A_)
#undef A_
}

static int upload_few(psph_ctx *c, const HostParticles &P, size_t at) {
  const size_t n = P.size();
  if (!c->up_h) {
    if (!c->up_d) PSPH_TRY(dmalloc((void **)&c->up_d, kUpload * kUploadBytes));
    if (hipHostMalloc((void **)&c->up_h, kUpload * kUploadBytes, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      c->up_h = nullptr;
      return fail(PSPH_ENOMEM, "hipHostMalloc");
    }
  }
  if (c->up_busy) HIP_TRY(hipStreamSynchronize(c->stream));   // the copy before has left the pinned memory
  char *to = c->up_h;
#define A_(a) std::memcpy(to, P.a.data(), n * sizeof(P.a[0])); to += n * sizeof(P.a[0]);
  PSPH_DFIELDS(A_) PSPH_UFIELDS(A_) PSPH_IFIELDS(A_)
#undef A_
  HIP_TRY(hipMemcpyAsync(c->up_d, c->up_h, n * kUploadBytes, hipMemcpyHostToDevice, c->stream));
  c->up_busy = true;
  hipLaunchKernelGGL(k_append, blocks(n), 256, 0, c->stream, (uint32_t)n, (uint32_t)at, c->up_d, c->f);
  HIP_TRY(hipGetLastError());
  return 0;
}

static int upload(psph_ctx *c, const HostParticles &P, size_t at) {
  size_t n = P.size();
  if (!n) return 0;
  if (n <= kUpload) return upload_few(c, P, at);
#define U_(a) HIP_TRY(hipMemcpyAsync(c->f.a + at, P.a.data(), n * sizeof(P.a[0]), hipMemcpyHostToDevice, c->stream));
  PSPH_DFIELDS(U_) PSPH_UFIELDS(U_)
  U_(bc) U_(phase)
#undef U_
  HIP_TRY(hipMemcpyAsync(c->f.inv + at, P.inv.data(), n * 4, hipMemcpyHostToDevice, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int psph_load(psph_ctx *c, const psph_soa *host, size_t n, double t0, int64_t step0) {
  if (!c || !host) return fail(PSPH_EINVAL, "null argument");
  if (n > c->cap) return fail(PSPH_ECAPACITY, "load: %zu particles exceed capacity %zu", n, c->cap);
  if (!host->x || !host->rho || !host->m || !host->h || !host->bc) return fail(PSPH_EINVAL, "load: x, rho, m, h and bc are required");
  HostParticles P;
  P.from_soa(host, n);
  c->loaded_removed = std::any_of(P.bc.begin(), P.bc.end(), [](int32_t b) { return b < 0; });
  PSPH_TRY(upload(c, P, 0));
  c->n = n;
  if (n) hipLaunchKernelGGL(k_iota_u32, blocks(n), 256, 0, c->stream, c->pid, 0u, (uint32_t)n);
  c->next_pid = (uint32_t)n;
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words + W_DEAD, 0ull, 1);
  c->time = t0;
  c->step = step0;
  c->ioutput = 0;
  c->next_output = c->cfg.t_output;
  while (c->next_output <= t0 && c->cfg.t_output > 0) { c->ioutput++; c->next_output = (c->ioutput + 1) * c->cfg.t_output; }
  c->grid_valid = false;
  return 0;
}

// Copies between device arrays of n elements, up to 18 in a launch (one each took
// 650 launches, and 2.4 ms of GPU time, of the gradients of 6 steps).
struct Copies {
  psph_ctx *c;
  size_t n;
  Moves mv{};
  int n8 = 0, n4 = 0;
  template <class T>
  int add(T *to, const T *from) {
    static_assert(sizeof(T) == 8 || sizeof(T) == 4, "elements of 8 or 4 bytes");
    if (sizeof(T) == 8) {
      if (n8 == kMove8) PSPH_TRY(flush());
      mv.s8[n8] = (const uint64_t *)from;
      mv.d8[n8++] = (uint64_t *)to;
    } else {
      if (n4 == kMove4) PSPH_TRY(flush());
      mv.s4[n4] = (const uint32_t *)from;
      mv.d4[n4++] = (uint32_t *)to;
    }
    return 0;
  }
  int flush() {
    if (n && (n8 || n4)) hipLaunchKernelGGL(k_copy, blocks(n), 256, 0, c->stream, (uint32_t)n, n8, n4, mv);
    n8 = n4 = 0;
    HIP_TRY(hipGetLastError());
    return 0;
  }
};

// live and real particles of bc[0..n)
static int count_live(psph_ctx *c, size_t n, const int32_t *bc, unsigned long long cnt[2]) {
  unsigned long long *out = c->words + W_LIVE;
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, out, 0ull, 2);
  if (n) hipLaunchKernelGGL(k_count_live, red_blocks(n), 256, 0, c->stream, (uint32_t)n, bc, out);
  HIP_TRY(hipGetLastError());
  PSPH_TRY(read_words(c));
  cnt[0] = c->seen[W_LIVE];
  cnt[1] = c->seen[W_LIVE_REAL];
  return 0;
}

extern "C" int psph_count(psph_ctx *c, size_t *n_total, size_t *n_real) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  unsigned long long cnt[2];
  PSPH_TRY(count_live(c, c->n, c->f.bc, cnt));
  if (n_total) *n_total = cnt[0];
  if (n_real) *n_real = cnt[1];
  return 0;
}

extern "C" int psph_device_view(psph_ctx *c, psph_soa *dev, size_t *n, void **stream) {
  if (!c || !dev) return fail(PSPH_EINVAL, "null argument");
  // finish pending work so that the caller may use the arrays on any stream
  HIP_TRY(hipStreamSynchronize(c->stream));
#define V_(a) dev->a = c->f.a;
  PSPH_DFIELDS(V_)
  V_(bc) V_(phase)
#undef V_
  dev->key0 = c->f.k0; dev->key1 = c->f.k1; dev->key2 = c->f.k2;
  dev->involved = c->f.inv;
  if (n) *n = c->n;
  if (stream) *stream = (void *)c->stream;
  return 0;
}

extern "C" int psph_get_config(psph_ctx *c, psph_config *cfg) {
  if (!c || !cfg) return fail(PSPH_EINVAL, "null argument");
  *cfg = c->cfg;
  return 0;
}

extern "C" int psph_time(psph_ctx *c, double *time, int64_t *step) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  if (time) *time = c->time;
  if (step) *step = c->step;
  return 0;
}

static int download(psph_ctx *c, HostParticles &P) {
  size_t n = c->n;
  P.resize(n);
  if (!n) return 0;
  HIP_TRY(hipStreamSynchronize(c->stream));
#define D_(a) HIP_TRY(hipMemcpy(P.a.data(), c->f.a, n * sizeof(P.a[0]), hipMemcpyDeviceToHost));
  PSPH_DFIELDS(D_) PSPH_UFIELDS(D_) PSPH_IFIELDS(D_)
#undef D_
  return 0;
}

// The n particles with these keys in THashTable order, removed ones last: their
// indices in c->idx_b.  On the host the order took 21 ms of a read of 98k
// particles (sort, and a permutation of every field), 15 ms of the gradients of 227k.
static int read_order(psph_ctx *c, uint32_t n, const uint32_t *k0, const uint32_t *k1, const uint32_t *k2,
                      const int32_t *bc) {
  if (!n) return 0;
  hipStream_t s = c->stream;
  uint64_t *a = (uint64_t *)c->dsp[0], *b = (uint64_t *)c->dsp[1];
  size_t b32 = 0, b64 = 0;
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, b32, k2, c->key_b, c->idx_a, c->idx_b, (int)n, 0, 32, s));
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, b64, a, b, c->idx_a, c->idx_b, (int)n, 0, 64, s));
  PSPH_TRY(ensure_cub(c, std::max(b32, b64)));
  hipLaunchKernelGGL(k_iota_u32, blocks(n), 256, 0, s, c->idx_a, 0u, n);
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(c->cub, b32, k2, c->key_b, c->idx_a, c->idx_b, (int)n, 0, 32, s));
  hipLaunchKernelGGL(k_read_key01, blocks(n), 256, 0, s, n, c->idx_b, k0, k1, a);
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(c->cub, b64, a, b, c->idx_b, c->idx_a, (int)n, 0, 64, s));
  hipLaunchKernelGGL(k_read_slot, blocks(n), 256, 0, s, n, c->idx_a, k0, k1, bc, c->cfg.p_table_size, c->cfg.dim, a);
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(c->cub, b64, a, b, c->idx_a, c->idx_b, (int)n, 0, 33, s));
  HIP_TRY(hipGetLastError());
  return 0;
}

extern "C" int psph_read(psph_ctx *c, psph_soa *host, size_t cap, size_t *n_out) {
  if (!c || !n_out) return fail(PSPH_EINVAL, "null argument");
  unsigned long long cnt[2];
  PSPH_TRY(count_live(c, c->n, c->f.bc, cnt));
  const size_t n = cnt[0];                    // removed particles are dropped
  *n_out = n;
  if (!host) return 0;
  if (n > cap) return fail(PSPH_ECAPACITY, "read: %zu particles, buffer holds %zu", n, cap);
  if (!n) return 0;
  PSPH_TRY(read_order(c, (uint32_t)c->n, c->f.k0, c->f.k1, c->f.k2, c->f.bc));
  // through the spare arrays, ten (nine) fields of 8 bytes and three of 4 at a time
  const double *src8[] = {
#define S_(a) c->f.a,
    PSPH_DFIELDS(S_)
#undef S_
  };
  double *dst8[] = {host->x, host->y, host->z, host->vx, host->vy, host->vz, host->svx, host->svy, host->svz, host->rho,
                    host->e, host->m, host->h, host->p, host->c, host->T, host->gam, host->cp, host->xi};
  const void *src4[] = {c->f.k0, c->f.k1, c->f.k2, c->f.bc, c->f.phase, c->f.inv};
  void *dst4[] = {host->key0, host->key1, host->key2, host->bc, host->phase, host->involved};
  void *spare4[] = {c->usp, c->isp, c->idx_a};
  for (int part = 0; part < 2; part++) {
    const int f0 = part * 10, nf = part ? 9 : 10;
    Moves mv{};
    for (int k = 0; k < nf; k++) { mv.s8[k] = (const uint64_t *)src8[f0 + k]; mv.d8[k] = (uint64_t *)c->dsp[k]; }
    for (int k = 0; k < 3; k++) { mv.s4[k] = (const uint32_t *)src4[part * 3 + k]; mv.d4[k] = (uint32_t *)spare4[k]; }
    if (part == 0) hipLaunchKernelGGL((k_gather<10, 3>), blocks(n), 256, 0, c->stream, (uint32_t)n, c->idx_b, mv);
    else hipLaunchKernelGGL((k_gather<9, 3>), blocks(n), 256, 0, c->stream, (uint32_t)n, c->idx_b, mv);
    HIP_TRY(hipGetLastError());
    for (int k = 0; k < nf; k++)
      if (dst8[f0 + k]) HIP_TRY(hipMemcpyAsync(dst8[f0 + k], c->dsp[k], n * 8, hipMemcpyDeviceToHost, c->stream));
    for (int k = 0; k < 3; k++)
      if (dst4[part * 3 + k]) HIP_TRY(hipMemcpyAsync(dst4[part * 3 + k], spare4[k], n * 4, hipMemcpyDeviceToHost, c->stream));
  }
  HIP_TRY(hipStreamSynchronize(c->stream));
  return 0;
}

// ---------------------------------------------------------------------------
// stages
// ---------------------------------------------------------------------------
extern "C" int psph_timestep(psph_ctx *c, double *dt_out) {
  if (!c || !dt_out) return fail(PSPH_EINVAL, "null argument");
  StageTimer tm(c, 0);
  hipLaunchKernelGGL(k_step_words, 1, 64, 0, c->stream, c->words);
  if (c->n) hipLaunchKernelGGL(k_dt_min, red_blocks(c->n), 256, 0, c->stream, (uint32_t)c->n, c->f.bc, c->f.h, c->f.c, c->words);
  tm.stop();
  PSPH_TRY(check_err(c, "timestep"));
  const double mn = seen_double(c, W_DT);
  double dt = 1.0E+10;                    // timestep.cc:99
  if (mn < dt) dt = mn;
  *dt_out = c->cfg.cfl * dt;
  return 0;
}

extern "C" int psph_advance_time(psph_ctx *c, double *dt) {   // TimeProps::incrtime
  if (!c || !dt) return fail(PSPH_EINVAL, "null argument");
  if ((c->time + (*dt)) > c->next_output) (*dt) = c->next_output - c->time;
  if ((c->time + (*dt)) > c->cfg.t_end) (*dt) = c->cfg.t_end - c->time;
  c->time += (*dt);
  c->step++;
  return 0;
}

// max h over the live particles (and the other words) in c->seen
static int reduce_hmax(psph_ctx *c) {
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words + W_HMAX, 0ull, 1);
  if (c->n) hipLaunchKernelGGL(k_h_max, red_blocks(c->n), 256, 0, c->stream, (uint32_t)c->n, c->f.bc, c->f.h, c->words + W_HMAX);
  return read_words(c);
}

// parts that the cells of n particles are filled in, and their chunks at most
static size_t cell_parts(size_t n, size_t ncells) { return ncells == 1 ? n / kRun + 1 : ncells; }
static size_t most_chunks(size_t n, size_t ncells) { return n / kChunk + cell_parts(n, ncells) + 1; }

// hmax: the largest h of the live particles
static int build_grid(psph_ctx *c, double hmax) {
  const psph_config &k = c->cfg;
  if (!(hmax > 0) || !std::isfinite(hmax)) hmax = k.h_air;
  c->h_max = hmax;
  c->reach_main = k.cutoff * hmax * (1 + 1e-9);
  GridDesc g{};
  if (k.list_all || k.dim == 1) {
    g.lo[0] = g.lo[1] = g.lo[2] = 0;
    g.inv_e = 0;
    g.nx = g.ny = g.nz = 1;
  } else {
    // cell edge: at least the reach of the RHS / density / velocity passes
    // (|dx_k| <= 3 (h_i + h_j) / 2 <= 3 h_max) and about 125 particles per
    // cell, so that a cell holds whole 64-particle chunks
    double vol = 1;
    for (int d = 0; d < 3; d++) vol *= k.ext_hi[d] - k.ext_lo[d];
    const double spacing = std::cbrt(vol / std::max<double>((double)c->n, 1.0));
    const double E = std::max(c->reach_main, 5.0 * spacing);
    int n3[3];
    for (int d = 0; d < 3; d++) {
      g.lo[d] = k.ext_lo[d] - E;
      n3[d] = (int)std::ceil((k.ext_hi[d] - k.ext_lo[d] + 2 * E) / E);
      if (n3[d] < 1) n3[d] = 1;
    }
    double ncell = (double)n3[0] * n3[1] * n3[2];
    if (ncell > 2.0e8) return fail(PSPH_ECAPACITY, "cell grid of %.3g cells (h_max %.4g) too large", ncell, hmax);
    g.inv_e = 1.0 / E;
    g.nx = n3[0]; g.ny = n3[1]; g.nz = n3[2];
  }
  g.ncells = (uint32_t)g.nx * g.ny * g.nz;
  int cbits = 0;
  while (cbits < 32 && ((uint64_t)1 << cbits) <= (uint64_t)g.ncells) cbits++;
  g.fbits = g.inv_e > 0 ? std::min(4, (32 - cbits) / 3) : 0;
  c->grid = g;
  size_t need = std::max((size_t)g.ncells, cell_parts(c->n, g.ncells)) + 1;
  if (need > c->cs_cap) {
    uint32_t **arrs[] = {&c->cs, &c->toff};
    for (auto pp : arrs) { if (*pp) hipFree(*pp); *pp = nullptr; }
    CellSum **sums[] = {&c->cell_has, &c->cell_at};
    for (auto pp : sums) { if (*pp) hipFree(*pp); *pp = nullptr; }
    c->cs_cap = 0;
    for (auto pp : arrs) PSPH_TRY(dmalloc((void **)pp, need * 4));
    for (auto pp : sums) PSPH_TRY(dmalloc((void **)pp, need * sizeof(CellSum)));
    c->cs_cap = need;
  }
  const size_t ub = c->n / kWave + (size_t)g.ncells + 1;
  const size_t cub_ = most_chunks(c->n, g.ncells);
  if (ub > c->tile_cap) {
    if (c->tbox) hipFree(c->tbox);
    c->tbox = nullptr;
    PSPH_TRY(dmalloc((void **)&c->tbox, ub * 2 * sizeof(float4)));
    c->tile_cap = ub;
  }
  if (cub_ > c->chunk_cap) {
    if (c->cfirst) hipFree(c->cfirst);
    if (c->ccount) hipFree(c->ccount);
    c->cfirst = c->ccount = nullptr;
    PSPH_TRY(dmalloc((void **)&c->cfirst, cub_ * 4));
    PSPH_TRY(dmalloc((void **)&c->ccount, cub_ * 4));
    c->chunk_cap = cub_;
  }
  return 0;
}

// exclusive scan of n + 1 values (the last input is 0) with hipcub
static int excl_scan(psph_ctx *c, const uint32_t *in, uint32_t *out, size_t n1) {
  size_t bytes = 0;
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n1, c->stream));
  PSPH_TRY(ensure_cub(c, bytes));
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(c->cub, bytes, in, out, (int)n1, c->stream));
  return 0;
}

// The contents of the cells that cs bounds: tiles (toff not null), targets (is)
// and their chunks.  has, at: cell_parts + 1 sums each.
template <class T>
static int fill_cells(psph_ctx *c, size_t n, uint32_t ncells, const uint32_t *cs, T is, CellSum *has, CellSum *at,
                      uint32_t *toff, float4 *tbox, const double *x, const double *y, const double *z, uint32_t *targets,
                      uint32_t *cfirst, uint32_t *ccount, uint32_t *nchunks) {
  const bool one = ncells == 1;
  const uint32_t parts = (uint32_t)cell_parts(n, ncells);
  hipLaunchKernelGGL((k_cell_counts<T>), parts + 1, kWave, 0, c->stream, parts, one, cs, is, has);
  size_t bytes = 0;
  HIP_TRY(hipcub::DeviceScan::ExclusiveScan(nullptr, bytes, has, at, CellAdd(), CellSum{0, 0, 0}, (int)parts + 1, c->stream));
  PSPH_TRY(ensure_cub(c, bytes));
  HIP_TRY(hipcub::DeviceScan::ExclusiveScan(c->cub, bytes, has, at, CellAdd(), CellSum{0, 0, 0}, (int)parts + 1, c->stream));
  hipLaunchKernelGGL((k_cell_fill<T>), parts, kWave, 0, c->stream, parts, one, cs, is, at, toff, tbox, x, y, z, targets,
                     cfirst, ccount, nchunks);
  HIP_TRY(hipGetLastError());
  return 0;
}

// seen: c->seen holds the largest h and the removed particles of this state
static int neighbors(psph_ctx *c, bool seen) {
  if (!seen) PSPH_TRY(reduce_hmax(c));
  const unsigned long long dead = c->seen[W_DEAD];
  PSPH_TRY(build_grid(c, seen_double(c, W_HMAX)));
  StageTimer tm(c, 1);
  const GridDesc &g = c->grid;
  uint32_t n = (uint32_t)c->n;
  hipStream_t s = c->stream;
  Tape &tp = c->tape;
  const bool frozen = tp.mode == 2 && tp.frozen;
  if (frozen) {
    if (tp.k >= (int64_t)tp.xrec.size()) return fail(PSPH_EINVAL, "replay: no recorded positions for step %lld", (long long)tp.k);
    if (!c->px) {
      PSPH_TRY(dmalloc((void **)&c->px, c->cap * 8));
      PSPH_TRY(dmalloc((void **)&c->py, c->cap * 8));
      PSPH_TRY(dmalloc((void **)&c->pz, c->cap * 8));
    }
    if (n) hipLaunchKernelGGL(k_pos_from_rec, blocks(n), 256, 0, s, n, c->pid, c->f.bc, tp.xrec[tp.k], tp.xrec_n[tp.k],
                              c->f.x, c->f.y, c->f.z, c->px, c->py, c->pz, (int *)(c->words + W_ERR));
  }
  if (n) {
    hipLaunchKernelGGL(k_cellkey, blocks(n), 256, 0, s, n, frozen ? c->px : c->f.x, frozen ? c->py : c->f.y,
                       frozen ? c->pz : c->f.z, c->f.bc, g, c->key_a, c->idx_a);
  }
  // One cell, and nothing to drop: every key is equal, and a stable sort and the
  // gather would leave all where it is (1D: 8 launches of 30 less).
  const bool in_order = g.ncells == 1 && g.fbits == 0 && !dead && !c->loaded_removed;
  if (n && !in_order) {
    int end_bit = 1;
    while (end_bit < 32 && ((uint64_t)1 << end_bit) <= ((uint64_t)g.ncells << (3 * g.fbits))) end_bit++;
    size_t bytes = 0;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, c->key_a, c->key_b, c->idx_a, c->idx_b, (int)n, 0, end_bit, s));
    PSPH_TRY(ensure_cub(c, bytes));
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(c->cub, bytes, c->key_a, c->key_b, c->idx_a, c->idx_b, (int)n, 0, end_bit, s));
    // gather every field into cell order; the places it goes to are the spare
    // arrays and those that this search fills only later
    double **f8[] = {
#define F_(a) &c->f.a,
      PSPH_DFIELDS(F_)
#undef F_
      &c->px, &c->py, &c->pz};
    double **to8[kMove8] = {&c->h_list};
    for (int k = 0; k < 10; k++) to8[k + 1] = &c->dsp[k];
    const int n8 = frozen ? 22 : 19;
    static_assert(sizeof f8 / sizeof f8[0] == 2 * kMove8, "two launches move every array");
    Moves mv;
    for (int k = 0; k < kMove8; k++) { mv.s8[k] = (const uint64_t *)*f8[k]; mv.d8[k] = (uint64_t *)*to8[k]; }
    uint32_t **to4[kMove4 - 1] = {&c->usp, &c->pid_sp, &c->idx_a, &c->refb, &c->targets, &c->key_a};
    int q4 = 0;
    auto move4 = [&](auto *&field, auto *&to) {
      mv.s4[q4] = (const uint32_t *)field;
      mv.d4[q4++] = (uint32_t *)to;
      auto *was = field;
      field = (decltype(was))to;
      to = (std::remove_reference_t<decltype(to)>)was;
    };
    move4(c->f.k0, *to4[0]); move4(c->f.k1, *to4[1]); move4(c->f.k2, *to4[2]);
    move4(c->pid, *to4[3]); move4(c->f.bc, *to4[4]); move4(c->f.phase, *to4[5]); move4(c->f.inv, c->isp);
    hipLaunchKernelGGL((k_gather<kMove8, kMove4>), blocks(n), 256, 0, s, n, c->idx_b, mv);
    for (int k = 0; k < kMove8; k++) std::swap(*f8[k], *to8[k]);
    for (int k = kMove8; k < n8; k++) {
      mv.s8[k - kMove8] = (const uint64_t *)*f8[k];
      mv.d8[k - kMove8] = (uint64_t *)*to8[k - kMove8];
    }
    if (frozen) hipLaunchKernelGGL((k_gather<kMove8, 0>), blocks(n), 256, 0, s, n, c->idx_b, mv);
    else hipLaunchKernelGGL((k_gather<19 - kMove8, 0>), blocks(n), 256, 0, s, n, c->idx_b, mv);
    for (int k = kMove8; k < n8; k++) std::swap(*f8[k], *to8[k - kMove8]);
    std::swap(c->key_a, c->key_b);   // key_a: sorted keys
  }
  // drop removed particles (their key == ncells sorts them to the tail)
  if (dead) {
    if (dead > n) return fail(PSPH_EINVARIANT, "removed-particle count %llu exceeds %u", dead, n);
    n -= (uint32_t)dead;
    c->n = n;
    hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, s, c->words + W_DEAD, 0ull, 1);
  }
  // the positions every predicate of this step reads
  const double *qx = frozen ? c->px : c->f.x, *qy = frozen ? c->py : c->f.y, *qz = frozen ? c->pz : c->f.z;
  if (tp.mode == 1 && (int64_t)tp.xrec.size() == tp.k) {
    double *rec = nullptr;
    const uint32_t nrec = std::max<uint32_t>(c->next_pid, 1);
    PSPH_TRY(dmalloc((void **)&rec, (size_t)nrec * 3 * 8));
    tp.xrec.push_back(rec);
    tp.xrec_n.push_back(nrec);
    if (n) hipLaunchKernelGGL(k_pos_to_rec, blocks(n), 256, 0, s, n, c->pid, c->f.x, c->f.y, c->f.z, rec, nrec);
  }
  // reference buckets (list membership) and h at list time
  int nb[3] = {1, 1, 1};
  double del = c->cfg.bucket_edge > 0 ? c->cfg.bucket_edge : 1.0;
  if (c->cfg.dim == 3)
    for (int d = 0; d < 3; d++) nb[d] = (int)std::llround((c->cfg.ext_hi[d] - c->cfg.ext_lo[d]) / del);
  for (int d = 0; d < 3; d++)
    if (nb[d] > kRefbMaxPerAxis)
      return fail(PSPH_ECAPACITY, "%d reference buckets on axis %d (at most %d)", nb[d], d, kRefbMaxPerAxis);
  const RefBuckets rb{{c->cfg.ext_lo[0], c->cfg.ext_lo[1], c->cfg.ext_lo[2]}, del, {nb[0], nb[1], nb[2]}};
  hipLaunchKernelGGL(k_sorted, blocks((size_t)n + 1), 256, 0, s, n, c->key_a, 3 * g.fbits, g.ncells, c->cs, qx, qy, qz,
                     c->f.h, rb, c->refb, c->h_list);
  // tiles, targets and their chunks (<= kChunk consecutive targets of one cell)
  PSPH_TRY(fill_cells(c, n, g.ncells, c->cs, IsTarget{c->f.bc}, c->cell_has, c->cell_at, c->toff, c->tbox, qx, qy, qz,
                      c->targets, c->cfirst, c->ccount, c->nchunks));
  HIP_TRY(hipGetLastError());
  tm.stop();
  c->grid_valid = true;
  c->lists_valid = false;
  return 0;
}

extern "C" int psph_neighbors(psph_ctx *c) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  return neighbors(c, false);
}

// half an ulp of the cut-off; the test above assumes its mantissa is even
static CutTest cut_test(double cut) {
  int e;
  std::frexp(cut, &e);                       // cut = f 2^e, f in [0.5, 1)
  return CutTest{cut, std::ldexp(1.0, e - 54)};
}

static Traversal traversal(psph_ctx *c, double reach) {
  return Traversal{c->cs, c->toff, c->tbox, c->grid, reach};
}

// a list box 4.25 h can reach past the adjacent buckets: the list test needs
// the bucket adjacency as well
static int list_adj(const psph_config &k, double hmax) {
  return (!k.list_all && k.dim == 3 && k.list_factor * hmax >= k.bucket_edge * (1 - 1e-12)) ? 1 : 0;
}

static PairCommon make_common(psph_ctx *c, double reach) {
  PairCommon pc;
  const bool frozen = c->tape.mode == 2 && c->tape.frozen;
  pc.x = frozen ? c->px : c->f.x; pc.y = frozen ? c->py : c->f.y; pc.z = frozen ? c->pz : c->f.z;
  pc.ax = c->f.x; pc.ay = c->f.y; pc.az = c->f.z;
  pc.refb = c->refb; pc.h_list = c->h_list;
  pc.bc = c->f.bc;
  pc.gflag = c->rec ? c->rec->gflag : nullptr;
  pc.tr = traversal(c, reach);
  pc.targets = c->targets;
  pc.cfirst = c->cfirst; pc.ccount = c->ccount; pc.nchunks = c->nchunks;
  pc.list_all = (c->cfg.list_all || c->cfg.dim == 1) ? 1 : 0;
  pc.list_factor = c->cfg.list_factor;
  pc.del = c->cfg.bucket_edge;
  for (int d = 0; d < 3; d++) pc.ext_lo[d] = c->cfg.ext_lo[d];
  // h_max bounds h at list time (it only grows with an adaptation)
  pc.list_adj = list_adj(c->cfg, c->h_max);
  pc.cut = cut_test(c->cfg.cutoff);
  pc.err = (int *)(c->words + W_ERR);
  pc.halt = pc.err;
  pc.nhalt = 0;
  return pc;
}

// workgroups for a pair pass: an upper bound on the chunks (each part of the
// cells may add a partial chunk), padded so that kXcds * ceil(nchunks /
// kXcds) exist
static unsigned chunk_grid(size_t n, size_t ncells) {
  size_t ub = most_chunks(n, ncells) + kXcds;
  return (unsigned)((ub + kXcds - 1) / kXcds * kXcds);
}

static void launch_list(psph_ctx *c, double reach, uint32_t *count, const uint32_t *offset, uint32_t *out) {
  const PairCommon pc = make_common(c, reach);
  const unsigned nb = chunk_grid(c->n, c->grid.ncells);
  if (c->cfg.dim == 3) hipLaunchKernelGGL(k_list<3>, nb, kWave, 0, c->stream, pc, count, offset, out);
  else hipLaunchKernelGGL(k_list<1>, nb, kWave, 0, c->stream, pc, count, offset, out);
}

// what the visits are made for: particles, cells, smoothing lengths and their
// bound, the visit cursor (the number of chunks follows it), and whether a pair
// counts for both of its particles
struct ListOf {
  size_t n, ncells;
  const double *h;
  double h_max;
  unsigned long long *cursor;
  bool both;
};

static GroupCommon group_common(psph_ctx *c) {
  GroupCommon gc{};
  gc.g = Geom{c->gxy, c->gzh};
  gc.gl = GroupLists{c->gvisit, c->goff, c->gnum, c->gfast, c->gcursor, c->gvisit_cap};
  gc.cutx = c->cfg.cutoff * (1.0 + 1e-12);     // a superset of the three passes' kernel boxes
  gc.cutj = gc.cutx;
  gc.h_max = c->h_max;
  return gc;
}

// memory of the group passes: positions, record arrays, per-group offsets
static int group_memory(psph_ctx *c, size_t chunks) {
  if (!c->gxy) PSPH_TRY(dmalloc((void **)&c->gxy, c->cap * sizeof(double2)));
  if (!c->gzh) PSPH_TRY(dmalloc((void **)&c->gzh, c->cap * sizeof(double2)));
  for (auto &p : c->pk)
    if (!p) PSPH_TRY(dmalloc(&p, c->cap * 16));
  if (chunks > c->gchunk_cap) {
    uint32_t **arrs[] = {&c->goff, &c->gnum, &c->gfast};
    for (auto pp : arrs) { if (*pp) hipFree(*pp); *pp = nullptr; }
    c->gchunk_cap = 0;
    for (auto pp : arrs) PSPH_TRY(dmalloc((void **)pp, chunks * kGroupsPerChunk * 4));
    c->gchunk_cap = chunks;
  }
  return 0;
}

static void launch_geom(psph_ctx *c, const PairCommon &pc) {
  hipLaunchKernelGGL(k_geom, blocks(c->n), 256, 0, c->stream, (uint32_t)c->n, pc.x, pc.y, pc.z, c->f.h, c->gxy, c->gzh,
                     c->gcursor);
}

// the groups' visits for the boxes that c_smooth and done say (GroupCommon): the
// kernel alone, its cursor at 0
static int launch_lists(psph_ctx *c, const PairCommon &pc, const ListOf &of, double c_smooth, const uint32_t *done,
                        unsigned long long *over) {
  // a group per wave up to a quarter of a million particles: at 77k 0.15 ms against
  // 0.20 with half a chunk; a chunk per wave beyond
  const uint32_t nsplit = of.n < (1u << 18) ? kGroupsPerChunk : 1;
  const unsigned G = chunk_grid(of.n, of.ncells) * nsplit;
  GroupCommon gc = group_common(c);
  gc.c_smooth = c_smooth;
  gc.done = done;
  gc.gl.cursor = of.cursor;
  gc.h_max = of.h_max;
  gc.both = of.both ? 1 : 0;
  if (of.both) gc.cutj = 2 * gc.cutx;
  gc.over = over;
  if (c->cfg.dim == 3)
    hipLaunchKernelGGL(k_group_lists<3>, G, kWave, 0, c->stream, pc, gc, of.h, c->cfg.cutoff2, nsplit);
  else
    hipLaunchKernelGGL(k_group_lists<1>, G, kWave, 0, c->stream, pc, gc, of.h, c->cfg.cutoff2, nsplit);
  HIP_TRY(hipGetLastError());
  return 0;
}

// the visits, in memory that holds them; cleared: the cursor is at 0
static int build_lists(psph_ctx *c, const PairCommon &pc, const ListOf &of, double c_smooth, const uint32_t *done,
                       bool cleared, uint32_t &ngroups) {
  for (;; cleared = false) {
    if (!cleared) hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, of.cursor, 0ull, 1);
    PSPH_TRY(launch_lists(c, pc, of, c_smooth, done, nullptr));
    unsigned long long *got = c->seen + W_COUNT;             // visits; chunks
    HIP_TRY(hipMemcpyAsync(got, of.cursor, 16, hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    c->up_busy = false;
    const unsigned long long total = got[0];
    ngroups = (uint32_t)got[1] * kGroupsPerChunk;
    if (total <= c->gvisit_cap) return 0;
    // the visits outgrew their memory: this call only counted
    constexpr unsigned long long kMost = 0xffffffffull;      // GroupLists::off
    if (total > kMost) return fail(PSPH_ENOMEM, "%llu tile visits exceed the maximum of %llu", total, kMost);
    if (c->gvisit) hipFree(c->gvisit);
    c->gvisit = nullptr;
    c->gvisit_cap = 0;
    const unsigned long long want = std::min(total + total / 8 + 1024, kMost);
    PSPH_TRY(dmalloc((void **)&c->gvisit, (size_t)want * sizeof(uint4)));
    c->gvisit_cap = (uint32_t)want;
  }
}

static ListOf own_lists(const psph_ctx *c) {
  return ListOf{c->n, c->grid.ncells, c->f.h, c->h_max, c->gcursor, false};
}

// Lists and positions of the group passes (positions, h and targets fixed since
// the last psph_neighbors / adaptation).
static int ensure_lists(psph_ctx *c) {
  if (c->lists_valid) return 0;
  StageTimer tm(c, 1);
  PSPH_TRY(group_memory(c, c->chunk_cap));
  const PairCommon pc = make_common(c, c->reach_main);
  launch_geom(c, pc);
  PSPH_TRY(build_lists(c, pc, own_lists(c), 0.0, nullptr, true, c->ngroups));
  c->lists_valid = true;
  return 0;
}

// A pass's outputs for its targets go to spare arrays; the other particles keep
// their values: the kernel that packs the pass's records copies those.
struct FieldCopy {
  const double *src[9];
  double *dst[9];
  int nf;
};
template <class P>
__global__ void k_pack(uint32_t n, typename P::Args a, const int32_t *bc, FieldCopy fc) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  P::pack(a, i);
  if (fc.nf && !need_neigh(bc[i]))
    for (int q = 0; q < fc.nf; q++) fc.dst[q][i] = fc.src[q][i];
}

// Waves per group.  A group alone is a chain of tile loads and pair blocks;
// where groups are fewer than the chip has room for (about 5000 waves), several
// waves share one.  RHS, density, filter, us, with 1 / 2 / 4 / 8 waves: 256
// groups (FP64) 119, 74, 68 / 74, 45, 40 / 43, 27, 24 / 32, 19, 17; 4308 groups
// (FP32-exp) 192, 105, 93 / 161, 95, 85 / 142, 87, 78 / 169, 108, 96; 10784
// groups 364, 210, 188 / 341, 194, 175 / 332, 196, 177 / 406, 259, 232; 20416
// groups (FP32-pair) 763, 500, 424 / 760, 490, 414 / 760, 485, 417 / 865, 594,
// 513; 400k targets (FP32-pure) 1522, 832, 1083 / 1522, 828, 1081 / 1568, 874,
// 1118.
static unsigned group_split(uint32_t ngroups) {
  return ngroups <= 1024 ? kMaxSplit : ngroups <= 16384 ? 4 : 1;
}

template <class P>
static void launch_pack(psph_ctx *c, typename P::Args &a, const FieldCopy &fc) {
  for (int k = 0; k < 5; k++) a.pk.p[k] = c->pk[k];
  hipLaunchKernelGGL((k_pack<P>), blocks(c->n), 256, 0, c->stream, (uint32_t)c->n, a, c->f.bc, fc);
}
template <int D, class P>
static void launch_group_kernel(psph_ctx *c, const PairCommon &pc, const GroupCommon &gc, const typename P::Args &a,
                                bool frozen) {
  const unsigned nb = (c->ngroups + kXcds - 1) / kXcds * kXcds;
  if (!nb) return;
  const unsigned split = group_split(c->ngroups);
  const size_t lds = split * sizeof(GroupLds<P>);
  if (frozen) hipLaunchKernelGGL((k_group_pass<D, P, true>), nb, split * kWave, lds, c->stream, pc, gc, a);
  else hipLaunchKernelGGL((k_group_pass<D, P, false>), nb, split * kWave, lds, c->stream, pc, gc, a);
}
template <int D, class P>
static void launch_group_pass(psph_ctx *c, const PairCommon &pc, const GroupCommon &gc, typename P::Args a,
                              const FieldCopy &fc) {
  launch_pack<P>(c, a, fc);
  launch_group_kernel<D, P>(c, pc, gc, a, c->tape.mode == 2 && c->tape.frozen);
}
// the RHS, density and filter passes; PM, PX, PP, PD: the pass in the FP32-pair,
// FP32-exp, FP32-pure and FP64 forms
// err: the pass's error word; the passes after the RHS do nothing if an earlier
// word is set
template <class PM, class PX, class PP, class PD>
static int launch_groups(psph_ctx *c, Word err, const typename PD::Args &a, const FieldCopy &fc) {
  PairCommon pc = make_common(c, c->reach_main);
  pc.err = (int *)(c->words + err);
  pc.nhalt = err == W_ERR_RHS ? 0 : err - W_ERR;
  const GroupCommon gc = group_common(c);
  const int form = c->cfg.precision;
  if (c->cfg.dim == 3) {
    if (form == PSPH_FP32_PAIR) launch_group_pass<3, PM>(c, pc, gc, a, fc);
    else if (form == PSPH_FP32_EXP) launch_group_pass<3, PX>(c, pc, gc, a, fc);
    else if (form == PSPH_FP32_PURE) launch_group_pass<3, PP>(c, pc, gc, a, fc);
    else launch_group_pass<3, PD>(c, pc, gc, a, fc);
  } else {
    if (form == PSPH_FP32_PAIR) launch_group_pass<1, PM>(c, pc, gc, a, fc);
    else if (form == PSPH_FP32_EXP) launch_group_pass<1, PX>(c, pc, gc, a, fc);
    else if (form == PSPH_FP32_PURE) launch_group_pass<1, PP>(c, pc, gc, a, fc);
    else launch_group_pass<1, PD>(c, pc, gc, a, fc);
  }
  return 0;
}

static EosConst eos_const(const psph_config &k) {
  return EosConst{k.ng0, k.cvs, k.cvg, k.cva, k.rg, k.ra, k.lans};
}

// the later passes of a step use the new h: widen the reach
static void set_reach(psph_ctx *c, double hmax) {
  c->lists_valid = false;                // h changed
  c->h_max = hmax;
  c->reach_main = c->cfg.cutoff * hmax * (1 + 1e-9);
}

extern "C" int psph_adapt_h(psph_ctx *c) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  if (!c->grid_valid) return fail(PSPH_EINVAL, "adapt_h: call psph_neighbors first");
  const psph_config &k = c->cfg;
  AdaptArgs a{};
  a.m = c->f.m; a.bc = c->f.bc; a.refb = c->refb; a.h = c->f.h; a.done = c->usp;
  a.cutoff = k.cutoff; a.cutoff2 = k.cutoff2; a.c_smooth = k.c_smooth; a.eta = k.eta;
  a.ratio = k.ratio_sml_dx; a.thresh = k.thresh; a.pghost = k.pghost_contrib; a.dim = k.dim;
  double hmax = c->h_max;
  if (c->n && k.num_loop > 0) {
    HIP_TRY(hipMemsetAsync(c->usp, 0, c->n * 4, c->stream));
    PSPH_TRY(group_memory(c, c->chunk_cap));
    const PairCommon pc = make_common(c, c->reach_main);
    launch_geom(c, pc);
    // FP64 arithmetic in every form (h enters every later pass, and a
    // relative error of h moves every kernel value by ~|s|^2 times as
    // much); the FX form takes its exponentials from the FP32 instruction
    const bool fx = k.precision == PSPH_FP32_EXP;
    if (fx) launch_pack<AdaptPass<double, true>>(c, a, FieldCopy{});
    else launch_pack<AdaptPass<double>>(c, a, FieldCopy{});
    const ListOf of = own_lists(c);
    auto pass = [&](unsigned long long *over) {
      GroupCommon gc = group_common(c);
      gc.over = over;
      if (k.dim == 3) {
        if (fx) launch_group_kernel<3, AdaptPass<double, true>>(c, pc, gc, a, false);
        else launch_group_kernel<3, AdaptPass<double>>(c, pc, gc, a, false);
      } else {
        if (fx) launch_group_kernel<1, AdaptPass<double, true>>(c, pc, gc, a, false);
        else launch_group_kernel<1, AdaptPass<double>>(c, pc, gc, a, false);
      }
    };
    // The first iteration's lists say how many groups there are and find their
    // memory.  The others are queued behind it and nobody waits: their boxes are
    // seldom larger, and where the memory does not hold them after all, that
    // iteration and those after it do nothing (GroupCommon::over) and are made
    // again from there.
    unsigned long long *over = c->words + W_OVER;
    for (int64_t it = 0; it < k.num_loop;) {
      {
        StageTimer tm(c, 2);
        PSPH_TRY(build_lists(c, pc, of, k.c_smooth, c->usp, it == 0, c->ngroups));
        pass(nullptr);
      }
      it++;
      if (it < k.num_loop) hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, over, 0ull, W_ITER_LAST + 1 - W_OVER);
      for (int64_t q = it; q < k.num_loop; q++) {
        StageTimer tm(c, 2);
        ListOf next = of;
        next.cursor = c->words + std::min<int64_t>(W_ITER_CURSOR + (q - it), W_ITER_LAST);
        if (W_ITER_CURSOR + (q - it) > W_ITER_LAST)
          hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, next.cursor, 0ull, 1);
        PSPH_TRY(launch_lists(c, pc, next, k.c_smooth, c->usp, over));
        pass(over);
      }
      HIP_TRY(hipGetLastError());
      PSPH_TRY(reduce_hmax(c));
      if (it >= k.num_loop || !c->ngroups || !c->seen[W_OVER]) break;
      it += (int64_t)c->seen[W_ITERS];
    }
    hmax = seen_double(c, W_HMAX);
    PSPH_TRY(seen_err(c, "adapt_h"));
  }
  set_reach(c, hmax);
  return 0;
}

// replays (or records) the smoothing lengths of an adaptation step by id
static int h_by_id(psph_ctx *c, double *tab, int replay) {
  if (c->n) hipLaunchKernelGGL(k_h_by_id, blocks(c->n), 256, 0, c->stream, (uint32_t)c->n, c->pid, c->f.h, tab, replay);
  HIP_TRY(hipGetLastError());
  if (!replay) return 0;
  PSPH_TRY(reduce_hmax(c));
  set_reach(c, seen_double(c, W_HMAX));
  return 0;
}

// The passes of a step; psph_step reads their errors at its end (seen_err).
static int rhs_pass(psph_ctx *c, double dt) {
  if (!c->grid_valid) return fail(PSPH_EINVAL, "rhs: call psph_neighbors first");
  const psph_config &k = c->cfg;
  uint32_t n = (uint32_t)c->n;
  // outputs go to spare arrays; non-targets keep their values
  double *ov[9] = {c->dsp[1], c->dsp[2], c->dsp[3], c->dsp[4], c->dsp[5], c->dsp[6], c->dsp[7], c->dsp[8], c->dsp[9]};
  double *src[9] = {c->f.vx, c->f.vy, c->f.vz, c->f.e, c->f.p, c->f.c, c->f.T, c->f.gam, c->f.cp};
  FieldCopy fc{};
  for (int q = 0; q < 9; q++) { fc.src[q] = src[q]; fc.dst[q] = ov[q]; }
  fc.nf = 9;
  RhsArgs a{};
  a.h = c->f.h; a.m = c->f.m; a.rho = c->f.rho; a.p = c->f.p; a.c = c->f.c; a.T = c->f.T; a.cp = c->f.cp;
  a.vx = c->f.vx; a.vy = c->f.vy; a.vz = c->f.vz; a.svx = c->f.svx; a.svy = c->f.svy; a.svz = c->f.svz;
  a.e = c->f.e; a.xi = c->f.xi; a.bc = c->f.bc;
  a.o_vx = ov[0]; a.o_vy = ov[1]; a.o_vz = ov[2];
  a.o_e = ov[3]; a.o_p = ov[4]; a.o_c = ov[5]; a.o_T = ov[6]; a.o_gam = ov[7]; a.o_cp = ov[8];
  a.dt = dt; a.g = k.g; a.cutoff = k.cutoff; a.cutoff2 = k.cutoff2; a.alpha = k.alpha; a.beta = k.beta;
  a.ata = k.ata; a.eps_half = k.eps_half; a.prandtl = k.prandtl; a.heat_scale = k.heat_scale;
  a.beta2 = 2.0 * k.beta; a.kheat = 20.0 * k.eps_half / k.prandtl;
  a.lans = k.lans; a.dim = k.dim; a.eos = eos_const(k); a.pairs = c->words + W_PAIRS;
  if (n) PSPH_TRY(ensure_lists(c));
  {
    StageTimer tm(c, 3);
    if (n) PSPH_TRY((launch_groups<RhsPass<float>, RhsPass<float, true, true>, RhsPass<float, false>, RhsPass<double>>(c, W_ERR_RHS, a, fc)));
  }
  HIP_TRY(hipGetLastError());
  std::swap(c->f.vx, c->dsp[1]); std::swap(c->f.vy, c->dsp[2]); std::swap(c->f.vz, c->dsp[3]);
  std::swap(c->f.e, c->dsp[4]); std::swap(c->f.p, c->dsp[5]); std::swap(c->f.c, c->dsp[6]);
  std::swap(c->f.T, c->dsp[7]); std::swap(c->f.gam, c->dsp[8]); std::swap(c->f.cp, c->dsp[9]);
  return 0;
}

extern "C" int psph_rhs(psph_ctx *c, double dt) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words + W_PAIRS, 0ull, 1);
  PSPH_TRY(rhs_pass(c, dt));
  PSPH_TRY(read_words(c));
  c->last_pairs = c->seen[W_PAIRS];
  return seen_err(c, "rhs");
}

static int density_pass(psph_ctx *c) {
  if (!c->grid_valid) return fail(PSPH_EINVAL, "density: call psph_neighbors first");
  const psph_config &k = c->cfg;
  uint32_t n = (uint32_t)c->n;
  FieldCopy fc{};
  fc.src[0] = c->f.rho; fc.dst[0] = c->dsp[1];
  fc.src[1] = c->f.e; fc.dst[1] = c->dsp[2];
  fc.nf = 2;
  DensArgs a{};
  a.h = c->f.h; a.m = c->f.m; a.rho = c->f.rho; a.e = c->f.e; a.bc = c->f.bc; a.phase = c->f.phase;
  a.o_rho = c->dsp[1]; a.o_e = c->dsp[2]; a.xi = c->f.xi; a.p = c->f.p; a.c = c->f.c; a.T = c->f.T;
  a.gam = c->f.gam; a.cp = c->f.cp; a.inv = c->f.inv;
  a.cutoff = k.cutoff; a.cutoff2 = k.cutoff2; a.e_ratio = k.e_smooth_ratio; a.msfrc_thresh = k.msfrc_thresh;
  a.pghost = k.pghost_contrib; a.energy_smooth = k.energy_smooth; a.eos = eos_const(k);
  a.cut = cut_test(k.cutoff);
  a.o_wn = c->rec ? c->rec->d[RF_WNE] : nullptr;
  a.e_sq16 = k.e_smooth_ratio * k.e_smooth_ratio == 16.0;
  {
    const double en = kInvSqrtPi * k.e_smooth_ratio;
    a.e_norm = k.dim == 3 ? en * en * en : en;
  }
  if (n) PSPH_TRY(ensure_lists(c));
  {
    StageTimer tm(c, 4);
    if (n) PSPH_TRY((launch_groups<DensPass<float>, DensPass<float, true, true>, DensPass<float, false>, DensPass<double>>(c, W_ERR_DENS, a, fc)));
  }
  HIP_TRY(hipGetLastError());
  std::swap(c->f.rho, c->dsp[1]);
  std::swap(c->f.e, c->dsp[2]);
  return 0;
}

extern "C" int psph_density(psph_ctx *c) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  PSPH_TRY(density_pass(c));
  return check_err(c, "density");
}

static int vsmooth_pass(psph_ctx *c) {
  if (!c->grid_valid) return fail(PSPH_EINVAL, "vsmooth: call psph_neighbors first");
  const psph_config &k = c->cfg;
  VsmArgs a{};
  a.h = c->f.h; a.m = c->f.m; a.rho = c->f.rho; a.vx = c->f.vx;
  a.vy = k.dim == 3 ? c->f.vy : nullptr; a.vz = k.dim == 3 ? c->f.vz : nullptr;
  a.bc = c->f.bc; a.svx = c->f.svx; a.svy = k.dim == 3 ? c->f.svy : nullptr; a.svz = k.dim == 3 ? c->f.svz : nullptr;
  a.cutoff = k.cutoff; a.cutoff2 = k.cutoff2;
  a.o_wn = c->rec ? c->rec->d[RF_WNV] : nullptr;
  if (c->n) PSPH_TRY(ensure_lists(c));
  {
    StageTimer tm(c, 5);
    if (c->n) PSPH_TRY((launch_groups<VsmPass<float>, VsmPass<float, true>, VsmPass<float>, VsmPass<double>>(c, W_ERR_VSM, a, FieldCopy{})));
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

extern "C" int psph_vsmooth(psph_ctx *c) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  PSPH_TRY(vsmooth_pass(c));
  return check_err(c, "vsmooth");
}

static int iferupt(const psph_ctx *c) {     // TimeProps::iferupt (properties.h:126-135)
  if (c->time < c->cfg.erupt_start) return 0;
  if (c->time > c->cfg.erupt_end) return 0;
  return 1;
}

// undo: the density pass was queued behind an RHS that may have failed
static int update_pos(psph_ctx *c, double dt, bool undo) {
  const psph_config &k = c->cfg;
  uint32_t n = (uint32_t)c->n;
  PosTape tp{c->tape.mode, (int32_t)c->tape.k, c->pid, c->tape.tr_step, c->tape.esc_step};
  if (tp.mode && (!tp.tr_step || c->next_pid > c->tape.id_cap)) return fail(PSPH_EINVAL, "update_pos: tape has no id table");
  StageTimer tm(c, 6);
  if (n)
    hipLaunchKernelGGL(k_update_pos, red_blocks(n), 256, 0, c->stream, n, k.dim, k.lans, iferupt(c), dt,
                       c->f.x, c->f.y, c->f.z, c->f.vx, c->f.vy, c->f.vz, c->f.svx, c->f.svy, c->f.svz,
                       c->f.bc, c->f.h, c->f.inv, k.dom_lo[2], k.ratio_sml_dx * k.h_air,
                       k.dom_lo[0], k.dom_lo[1], k.dom_lo[2], k.dom_hi[0], k.dom_hi[1], k.dom_hi[2],
                       c->words, tp);
  tm.stop();
  HIP_TRY(hipGetLastError());
  PSPH_TRY(read_words(c));
  if (undo) {
    c->last_pairs = c->seen[W_PAIRS];
    if ((uint32_t)c->seen[W_ERR] || (uint32_t)c->seen[W_ERR_RHS]) {
      // the density pass did nothing: its fields are where they were
      std::swap(c->f.rho, c->dsp[1]);
      std::swap(c->f.e, c->dsp[2]);
    }
    PSPH_TRY(seen_err(c, "rhs"));
  }
  c->last_removed = (int64_t)c->seen[W_DEAD];
  c->last_real = (int64_t)c->seen[W_REAL];
  c->grid_valid = false;
  return 0;
}

extern "C" int psph_update_pos(psph_ctx *c, double dt) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words + W_REAL, 0ull, 1);
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, c->words + W_VMAX, 0ull, 1);
  return update_pos(c, dt, false);
}

// id-indexed event tables of the tape, grown to hold `need` ids (new: -1)
static int tape_ids(psph_ctx *c, size_t need) {
  Tape &tp = c->tape;
  if (need <= tp.id_cap && tp.tr_step) return 0;
  size_t cap = std::max(need, std::max(2 * tp.id_cap, c->cap));
  int32_t *a = nullptr, *b = nullptr;
  PSPH_TRY(dmalloc((void **)&a, cap * 4));
  if (dmalloc((void **)&b, cap * 4)) { hipFree(a); return PSPH_ENOMEM; }
  hipLaunchKernelGGL(k_fill_i32, blocks(cap), 256, 0, c->stream, a, -1, (int)cap);
  hipLaunchKernelGGL(k_fill_i32, blocks(cap), 256, 0, c->stream, b, -1, (int)cap);
  if (tp.tr_step) {
    HIP_TRY(hipMemcpyAsync(a, tp.tr_step, tp.id_cap * 4, hipMemcpyDeviceToDevice, c->stream));
    HIP_TRY(hipMemcpyAsync(b, tp.esc_step, tp.id_cap * 4, hipMemcpyDeviceToDevice, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    hipFree(tp.tr_step);
    hipFree(tp.esc_step);
  }
  tp.tr_step = a;
  tp.esc_step = b;
  tp.id_cap = cap;
  return 0;
}

static void tape_clear(Tape &tp) {
  for (double *p : tp.htab) if (p) hipFree(p);
  tp.htab.clear();
  tp.dt.clear();
  tp.hslot.clear();
  tp.inlet.clear();
  for (double *p : tp.xrec) if (p) hipFree(p);
  tp.xrec.clear();
  tp.xrec_n.clear();
  for (double *p : tp.xrecb) if (p) hipFree(p);
  tp.xrecb.clear();
  tp.xrecb_n.clear();
  tp.frozen = false;
  tp.k = 0;
  tp.mode = 0;
}

// captures the step's intermediates into c->rec (defined with the adjoint)
static int rec_capture(psph_ctx *c, int stage, double dt);

extern "C" int psph_inject(psph_ctx *c, double dt, int64_t *added) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  if (added) *added = 0;
  c->last_injected = 0;
  Tape &tp = c->tape;
  std::vector<int32_t> *rec = nullptr;
  const std::vector<int32_t> *rep = nullptr;
  if (tp.mode == 1) { tp.inlet.emplace_back(); rec = &tp.inlet.back(); }
  if (tp.mode == 2) {
    if (tp.k >= (int64_t)tp.inlet.size()) return fail(PSPH_EINVAL, "inject: replay past the recorded run");
    rep = &tp.inlet[tp.k];
  }
  c->inj.resize(0);
  if (c->cfg.dim != 3 || !iferupt(c)) {
    if (rep && !rep->empty()) return fail(PSPH_EINVAL, "inject: recorded run erupted at this step");
    return 0;
  }
  PSPH_TRY(inject_host(c->cfg, c->time, dt, c->step, c->inj, rec, rep ? rep->data() : nullptr,
                       rep ? rep->size() : 0));
  size_t m = c->inj.size();
  if (c->n + m > c->cap)
    return fail(PSPH_ECAPACITY, "inject: %zu + %zu particles exceed capacity %zu", c->n, m, c->cap);
  if (tp.mode && c->next_pid + m > tp.id_cap) PSPH_TRY(tape_ids(c, c->next_pid + m));
  {
    StageTimer tm(c, 7);
    PSPH_TRY(upload(c, c->inj, c->n));
  }
  if (m) hipLaunchKernelGGL(k_iota_u32, blocks(m), 256, 0, c->stream, c->pid + c->n, c->next_pid, (uint32_t)m);
  c->next_pid += (uint32_t)m;
  c->n += m;
  c->last_injected = (int64_t)m;
  if (added) *added = (int64_t)m;
  c->grid_valid = false;
  return 0;
}

// wall-ghost refresh over the cell grid of the last neighbour search; disp:
// the largest per-axis displacement of any particle since that search
// ground on a bucket face: no MIXED bucket, nothing to refresh
static bool bcond_trivial(const psph_config &k) {
  const double fz = (k.dom_lo[2] - k.ext_lo[2]) / k.bucket_edge;
  return fz == std::floor(fz);
}

// wrec (optional, wrec_n entries): receives each refreshed ghost's Shepard
// normaliser, for the adjoint
// the bucket geometry, ground, support tests and EOS of the refresh
static BcondArgs bcond_geom(const psph_config &k) {
  BcondArgs a{};
  a.zg = k.dom_lo[2]; a.del = k.bucket_edge; a.cutoff2 = k.cutoff2;
  for (int d = 0; d < 3; d++) {
    a.ext_lo[d] = k.ext_lo[d];
    a.nb[d] = (int)std::llround((k.ext_hi[d] - k.ext_lo[d]) / k.bucket_edge);
  }
  a.bzg = (int)std::floor((k.dom_lo[2] - k.ext_lo[2]) / k.bucket_edge);
  a.cut = cut_test(k.cutoff);
  a.eos = eos_const(k);
  return a;
}

// qx, qy, qz (optional): the positions the support tests read
static int apply_bcond_grid(psph_ctx *c, double disp, double *wrec = nullptr, size_t wrec_n = 0,
                            const double *qx = nullptr, const double *qy = nullptr, const double *qz = nullptr) {
  const psph_config &k = c->cfg;
  if (k.dim != 3 || !c->n || bcond_trivial(k)) return 0;
  BcondArgs a = bcond_geom(k);
  a.wrec = wrec;
  a.wrec_n = (uint32_t)wrec_n;
  a.x = c->f.x; a.y = c->f.y; a.z = c->f.z; a.h = c->f.h; a.m = c->f.m;
  a.rho = c->f.rho; a.vx = c->f.vx; a.vy = c->f.vy; a.vz = c->f.vz; a.e = c->f.e; a.xi = c->f.xi;
  a.p = c->f.p; a.c = c->f.c; a.T = c->f.T; a.gam = c->f.gam; a.cp = c->f.cp;
  a.bc = c->f.bc; a.cs = c->cs; a.toff = c->toff; a.tbox = c->tbox; a.g = c->grid;
  a.px = qx ? qx : c->f.x; a.py = qx ? qy : c->f.y; a.pz = qx ? qz : c->f.z;
  const double hm = std::max(c->h_max, k.ratio_sml_dx * k.h_air);
  a.reach = k.cutoff * hm * (1 + 1e-9) + disp * (1 + 1e-9);
  const uint32_t n = (uint32_t)c->n;
  unsigned long long *count = c->words + W_BCOND;
  hipLaunchKernelGGL(k_fill_u64, 1, 64, 0, c->stream, count, 0ull, 1);
  hipLaunchKernelGGL(k_bcond_list, blocks(n), 256, 0, c->stream, n, a, c->usp, count);
  const unsigned grid = std::min(kBcondGrid, (n / kBcondGroup / kXcds + 1) * kXcds);
  if (qx) hipLaunchKernelGGL(k_bcond<true>, grid, kBcondWaves * kWave, 0, c->stream, n, a, c->usp, count);
  else hipLaunchKernelGGL(k_bcond<false>, grid, kBcondWaves * kWave, 0, c->stream, n, a, c->usp, count);
  HIP_TRY(hipGetLastError());
  return 0;
}

extern "C" int psph_apply_bcond(psph_ctx *c) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  if (!c->grid_valid) PSPH_TRY(psph_neighbors(c));
  return apply_bcond_grid(c, 0.0);
}

// domain adaptation (psph_domain.inl)
namespace {
int domain_adapt(psph_ctx *c);
int domain_scan_step(psph_ctx *c);
}  // namespace

extern "C" int psph_step(psph_ctx *c, psph_step_out *out) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  const psph_config &k = c->cfg;
  Tape &tp = c->tape;
  double dt;
  bool seen = false;                       // c->seen is of the state that the search will find
  if (k.adapt_domain && k.dim == 3 && !c->dom_ready)
    return fail(PSPH_EINVAL, "adapt_domain: call psph_domain_init after psph_load");
  if (tp.mode == 2) {
    if (tp.k >= (int64_t)tp.dt.size()) return fail(PSPH_EINVAL, "replay: past the end of the recorded run");
    dt = tp.dt[tp.k];
    c->time += dt;
    c->step++;
    hipLaunchKernelGGL(k_step_words, 1, 64, 0, c->stream, c->words);
  } else {
    PSPH_TRY(psph_timestep(c, &dt));
    seen = true;
    PSPH_TRY(psph_advance_time(c, &dt));
    if (tp.mode == 1) tp.dt.push_back(dt);
  }
  c->last_domain = 0;
  if (k.adapt_domain && k.dim == 3 && c->dom_pending) {
    // the region of real particles grows before this step's search
    // (main.cc:256-304); the wall ghosts are refreshed after it
    c->dom_pending = 0;
    seen = false;
    PSPH_TRY(domain_adapt(c));
    if (k.wall_bc && c->n) {
      PSPH_TRY(psph_neighbors(c));
      PSPH_TRY(apply_bcond_grid(c, 0.0));
    }
  }
  PSPH_TRY(neighbors(c, seen));
  if (tp.mode == 2) {
    const int slot = tp.hslot[tp.k];
    if (slot >= 0) PSPH_TRY(h_by_id(c, tp.htab[slot], 1));
  } else if (k.sml_update_int > 0 && c->step % k.sml_update_int == 0) {
    PSPH_TRY(psph_adapt_h(c));
    if (tp.mode == 1) {
      double *tab = nullptr;
      PSPH_TRY(dmalloc((void **)&tab, (size_t)c->next_pid * 8));
      tp.htab.push_back(tab);
      tp.hslot.push_back((int)tp.htab.size() - 1);
      PSPH_TRY(h_by_id(c, tab, 0));
    }
  } else if (tp.mode == 1) {
    tp.hslot.push_back(-1);
  }
  if (c->rec) PSPH_TRY(rec_capture(c, 0, dt));
  PSPH_TRY(rhs_pass(c, dt));
  if (c->rec) PSPH_TRY(rec_capture(c, 1, dt));
  PSPH_TRY(density_pass(c));
  if (c->rec) PSPH_TRY(rec_capture(c, 2, dt));
  if (k.lans) PSPH_TRY(vsmooth_pass(c));
  if (c->rec) PSPH_TRY(rec_capture(c, 3, dt));
  PSPH_TRY(update_pos(c, dt, true));
  int64_t added = 0;
  const uint32_t id0 = c->next_pid;
  PSPH_TRY(psph_inject(c, dt, &added));
  if (c->rec) {
    c->rec->inj_lo = id0;
    c->rec->inj_hi = c->next_pid;
    c->rec->inj_vel.assign(c->inj.vz.begin(), c->inj.vz.end());
  }
  if (k.adapt_domain && k.dim == 3) PSPH_TRY(domain_scan_step(c));   // main.cc:433-436
  if (k.wall_bc && k.dim == 3 && c->n) {
    // apply_bcond at the end of the step (main.cc:468): the grid is the one of
    // this step's neighbour search; particles have moved by at most dt vmax
    double vmax = seen_double(c, W_VMAX);
    for (size_t q = 0; q < (size_t)added; q++)
      vmax = std::max(vmax, std::max(std::fabs(c->inj.vx[q]), std::max(std::fabs(c->inj.vy[q]), std::fabs(c->inj.vz[q]))));
    double disp = std::fabs(dt) * vmax;
    const uint32_t nb = (uint32_t)c->n;
    if (tp.mode == 1 && (int64_t)tp.xrecb.size() == tp.k) {
      // positions at the refresh, by id, for a frozen replay
      double *rec = nullptr;
      const uint32_t nrec = std::max<uint32_t>(c->next_pid, 1);
      PSPH_TRY(dmalloc((void **)&rec, (size_t)nrec * 3 * 8));
      tp.xrecb.push_back(rec);
      tp.xrecb_n.push_back(nrec);
      hipLaunchKernelGGL(k_pos_to_rec, blocks(nb), 256, 0, c->stream, nb, c->pid, c->f.x, c->f.y, c->f.z, rec, nrec);
    }
    const bool frozen = tp.mode == 2 && tp.frozen;
    if (frozen) {
      // the contributor sets of the recorded run: support tests on its
      // positions, whose displacement since the search differs from this
      // run's by the perturbation (the reach takes 1% more)
      if (tp.k >= (int64_t)tp.xrecb.size() || !c->px)
        return fail(PSPH_EINVAL, "replay: no recorded refresh positions for step %lld", (long long)tp.k);
      hipLaunchKernelGGL(k_pos_from_rec, blocks(nb), 256, 0, c->stream, nb, c->pid, c->f.bc, tp.xrecb[tp.k],
                         tp.xrecb_n[tp.k], c->f.x, c->f.y, c->f.z, c->px, c->py, c->pz, (int *)(c->words + W_ERR));
      disp *= 1.01;
    }
    if (c->rec) PSPH_TRY(rec_capture(c, 4, dt));
    PSPH_TRY(apply_bcond_grid(c, disp, c->rec ? c->rec->d[RF_BW] : nullptr, c->rec ? c->rec->n : 0,
                              frozen ? c->px : nullptr, c->py, c->pz));
    if (c->rec) PSPH_TRY(rec_capture(c, 5, dt));
    if (frozen) PSPH_TRY(check_err(c, "replay refresh"));
  }
  if (tp.mode) tp.k++;
  // TimeProps::ifoutput (properties.h:104-120)
  bool output = false;
  if (c->time >= c->next_output || c->time == k.t_end) {
    c->ioutput++;
    c->next_output = ((c->ioutput + 1) * k.t_output) / 1.0;
    output = true;
  }
  if (out) {
    out->dt = dt; out->time = c->time; out->step = c->step;
    out->n_total = (int64_t)c->n - c->last_removed;
    out->n_real = c->last_real;            // the inlet adds erupt ghosts only
    out->n_injected = added; out->n_removed = c->last_removed;
    out->n_pairs = (int64_t)c->last_pairs;
    out->output = output;
    out->n_domain = c->last_domain;
  }
  return 0;
}

extern "C" int psph_run(psph_ctx *c, int64_t nsteps, psph_step_out *last) {
  for (int64_t s = 0; s < nsteps; s++) PSPH_TRY(psph_step(c, last));
  return 0;
}

extern "C" int psph_conservation(psph_ctx *c, double out[7]) {
  if (!c || !out) return fail(PSPH_EINVAL, "null argument");
  uint32_t n = (uint32_t)c->n;
  bool d3 = c->cfg.dim == 3;
  hipLaunchKernelGGL(k_conservation, kRedBlocks, 256, 0, c->stream, n, c->f.bc, c->f.m, c->f.e, c->f.vx,
                     d3 ? c->f.vy : nullptr, d3 ? c->f.vz : nullptr, c->f.xi, d3 ? c->f.z : nullptr, c->d_part);
  std::vector<double> part(kRedBlocks * 8);
  HIP_TRY(hipMemcpyAsync(part.data(), c->d_part, part.size() * 8, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  double acc[8] = {0};
  for (int b = 0; b < kRedBlocks; b++)
    for (int k = 0; k < 8; k++) acc[k] += part[b * 8 + k];
  for (int k = 0; k < 7; k++) out[k] = acc[k];
  return 0;
}

extern "C" int psph_diag_height(psph_ctx *c, double *H) {
  if (!c || !H) return fail(PSPH_EINVAL, "null argument");
  double cons[7];
  uint32_t n = (uint32_t)c->n;
  bool d3 = c->cfg.dim == 3;
  hipLaunchKernelGGL(k_conservation, kRedBlocks, 256, 0, c->stream, n, c->f.bc, c->f.m, c->f.e, c->f.vx,
                     d3 ? c->f.vy : nullptr, d3 ? c->f.vz : nullptr, c->f.xi, d3 ? c->f.z : nullptr, c->d_part);
  std::vector<double> part(kRedBlocks * 8);
  HIP_TRY(hipMemcpyAsync(part.data(), c->d_part, part.size() * 8, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  double num = 0, den = 0;
  for (int b = 0; b < kRedBlocks; b++) { den += part[b * 8 + 6]; num += part[b * 8 + 7]; }
  (void)cons;
  *H = den > 0 ? num / den : 0.0;
  return 0;
}

// Neighbour lists for parity checks, produced on the GPU by the membership rule
// of the physics passes, then mapped to read order and sorted (the reference's list order is bucket-insertion history;
// the set is what every pass consumes).
extern "C" int psph_get_neighbors(psph_ctx *c, int64_t *offsets, size_t n_cap, uint32_t *idx, size_t idx_cap) {
  if (!c || !offsets) return fail(PSPH_EINVAL, "null argument");
  if (!c->grid_valid) return fail(PSPH_EINVAL, "get_neighbors: call psph_neighbors first");
  const psph_config &k = c->cfg;
  uint32_t n = (uint32_t)c->n;
  // the list rule reaches the own bucket or the 4.25 h_i box (all pairs in 1D)
  const double r = (k.list_all || k.dim == 1) ? HUGE_VAL
                                              : std::max(k.list_factor * c->h_max, k.bucket_edge) * (1 + 1e-9);
  uint32_t *cnt = nullptr, *off = nullptr, *out = nullptr;
  PSPH_TRY(dmalloc((void **)&cnt, ((size_t)n + 1) * 4));
  PSPH_TRY(dmalloc((void **)&off, ((size_t)n + 1) * 4));
  HIP_TRY(hipMemsetAsync(cnt, 0, ((size_t)n + 1) * 4, c->stream));
  if (n) launch_list(c, r, cnt, nullptr, nullptr);
  size_t bytes = 0;
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, cnt, off, (int)n + 1, c->stream));
  PSPH_TRY(ensure_cub(c, bytes));
  HIP_TRY(hipcub::DeviceScan::ExclusiveSum(c->cub, bytes, cnt, off, (int)n + 1, c->stream));
  uint32_t total = 0;
  HIP_TRY(hipMemcpyAsync(&total, off + n, 4, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  PSPH_TRY(dmalloc((void **)&out, ((size_t)total + 1) * 4));
  if (n) launch_list(c, r, cnt, off, out);
  std::vector<uint32_t> hoff(n + 1), hout(total);
  HIP_TRY(hipMemcpyAsync(hoff.data(), off, ((size_t)n + 1) * 4, hipMemcpyDeviceToHost, c->stream));
  if (total) HIP_TRY(hipMemcpyAsync(hout.data(), out, (size_t)total * 4, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  hipFree(cnt); hipFree(off); hipFree(out);
  // device order -> read order
  HostParticles P;
  PSPH_TRY(download(c, P));
  auto perm = canonical_order(c->cfg, P.k0.data(), P.k1.data(), P.k2.data(), n);   // read pos -> dev idx
  std::vector<uint32_t> rank(n);
  for (uint32_t q = 0; q < n; q++) rank[perm[q]] = q;
  if ((size_t)n + 1 > n_cap) return fail(PSPH_ECAPACITY, "get_neighbors: offsets need %u entries", n + 1);
  size_t o = 0;
  std::vector<uint32_t> tmp;
  for (uint32_t q = 0; q < n; q++) {
    offsets[q] = (int64_t)o;
    uint32_t d = perm[q];
    uint32_t b = hoff[d], e = hoff[d + 1];
    if (P.bc[d] != 100 && P.bc[d] != 99) continue;
    tmp.assign(hout.begin() + b, hout.begin() + e);
    for (auto &v : tmp) v = rank[v];
    std::sort(tmp.begin(), tmp.end());
    if (idx) {
      if (o + tmp.size() > idx_cap) return fail(PSPH_ECAPACITY, "get_neighbors: idx buffer holds %zu", idx_cap);
      std::memcpy(idx + o, tmp.data(), tmp.size() * 4);
    }
    o += tmp.size();
  }
  offsets[n] = (int64_t)o;
  return 0;
}

extern "C" int psph_profile(psph_ctx *c, int enable) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  if (enable && !c->ev0) {
    HIP_TRY(hipEventCreate(&c->ev0));
    HIP_TRY(hipEventCreate(&c->ev1));
  }
  c->prof = enable != 0;
  for (int k = 0; k < PSPH_NSTAGES; k++) { c->prof_ms[k] = 0; c->prof_n[k] = 0; }
  return 0;
}

extern "C" int psph_profile_read(psph_ctx *c, double ms[PSPH_NSTAGES], int64_t launches[PSPH_NSTAGES]) {
  if (!c) return fail(PSPH_EINVAL, "null ctx");
  for (int k = 0; k < PSPH_NSTAGES; k++) {
    if (ms) ms[k] = c->prof_ms[k];
    if (launches) launches[k] = c->prof_n[k];
  }
  return 0;
}

#include "psph_adjoint.inl"
#include "psph_domain.inl"
#include "psph_noalloc.inl"
