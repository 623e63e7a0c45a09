// kernels_split.hpp -- two-pass D3Q19 two-component step with one lane per
// (site, component).
//
// The general two-pass schedule (kernels_twopass.hpp) gives a thread a whole
// site: both components' populations (76 doubles) live in its registers and
// every neighbour's solid flag is a separate mask load.  Here a wave holds one
// component of 64 consecutive sites (waves 2k and 2k+1 of a block: the two
// components of the same sites), which halves the registers per thread and
// makes every array base wave-uniform, so loads and stores address with a
// scalar base and a 32-bit offset.  The partner component's density and
// momentum pass through LDS.  The solid neighbourhood is the site's one
// 32-bit solid word; the new populations are written with streaming stores.
//
//   pass 1: pull the 19 streamed populations, density, psi -> S
//   pass 2: pull again, Shan-Chen force from psi in S, velocity shift,
//           BGK collision
//
// Large lattices take both passes in one launch (SplitPlan below), small ones
// in two.
//
// When a block's sites lie in one z-row (n_z a multiple of the block's
// sites), pass 2 stages the nine psi rows around the block in LDS with
// coalesced loads issued after the pulls, instead of gathering 19 scattered
// psi values per lane: 2.32 against 2.46 ms per FP64 collide at 256^3 (two
// launches, one array per population), with the same bits.
//
// Per-site arithmetic is the shared code of the other schedules (density,
// sc_force, total_density, weighted_velocity, collide_component), so all
// three give identical bits.
#pragma once

#include <type_traits>

#include "kernels_fused.hpp"
#include "kernels_shifted.hpp"
#include "split_order.hpp"

namespace dlbc {

constexpr int kSplitThreads = 256;  // FP64: 4 waves = 128 sites x 2 components
// Shifted storage: one lane per site holding both components (their
// populations sit side by side), 4 waves = 256 sites.
constexpr int kShiftThreads = 256;
constexpr int kShiftSites = 256;

// Grid of a split launch over `sites`: threads / 2 sites per block.  (A grid
// that gave each XCD one contiguous run of sites, an eighth of the lattice,
// measured slower: 3.76 against 3.43 ms per FP64 step of two launches at
// 256^3, with one array per population.)
inline int split_grid(int64_t sites, int threads = kSplitThreads) {
  return (int)((sites + threads / 2 - 1) / (threads / 2));
}

// The block of sites this workgroup takes.  Workgroup b runs on XCD b % 8.
// With g.order_chunk = K the XCDs take turns at K consecutive blocks: the
// j-th workgroup of XCD k takes block ((j / K) 8 + k) K + j % K.  Rows
// neighbouring in y then share an XCD and its L2, and in x too when a plane
// is a whole number of turns (8 K blocks).  Blocks from g.order_main on (the
// part of the grid short of a whole turn) keep site order.
__device__ inline int split_block(const Geo &g, int b) {
  const int K = g.order_chunk;
  if (K <= 0 || b >= g.order_main) return b;
  const int j = b >> 3;
  return ((j / K) * 8 + (b & 7)) * K + j % K;
}

// Whether the library picks an XCD block order for the two launches by itself
// (an eighth of an x-plane per turn) or keeps site order.  Site order: on the
// 256^3 channel (FP64, one array per population) chunks of 8 to 256 blocks cut the collide pass's L2 misses by a
// quarter (FETCH_SIZE 3.49 -> 2.60 GiB at K = 64) yet ran 2.53-2.74 ms
// against 2.46 ms in site order.
constexpr bool kSplitAutoChunk = false;

// order_main for chunk K over a grid of nb blocks: whole turns of 8 K blocks.
inline int split_order_main(int nb, int K) { return K > 0 ? nb / (8 * K) * (8 * K) : 0; }

// Whether every site of this lane's cache line is solid, for a wave of 64
// consecutive sites whose lines hold LINE sites each (lines aligned to the
// wave: the site stride is a multiple of 64).  Such lines are neither read nor
// written by a collide pass: a solid site keeps its populations.
template <int LINE>
__device__ inline bool line_all_solid(bool solid_site) {
  constexpr uint64_t kLineMask = LINE == 64 ? ~0ull : ((1ull << LINE) - 1ull);
  const uint64_t m = __ballot(solid_site);
  const int first = (threadIdx.x & 63) / LINE * LINE;
  return ((m >> first) & kLineMask) == kLineMask;
}

// Wave-uniform copy of an int: the compiler then keeps it in a scalar
// register, and pointers formed from it stay scalar (the wave index
// threadIdx.x >> 6 is uniform, but the compiler cannot tell).
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Site and component of this lane in wave w of block blk (the component is
// uniform per wave); false past the end of the lattice.
__device__ inline bool split_lane(const Geo &g, int blk, int w, int &s, int &f) {
  f = w & 1;
  s = uniform(blk * (kSplitThreads / 2) + (w >> 1) * 64) + (threadIdx.x & 63);
  return s < g.sites;
}

// ---- both passes in one launch -------------------------------------------------
// Every block of sites is visited by a psi workgroup and later by a collide
// workgroup, in the order of a table (split_order.hpp).  psi goes from one to
// the other through S (P), and then a flag for its block; a collide wave looks
// at the flags of the blocks that it reads before it reads them.  A wave that
// finds no flags for too long computes that psi itself (the same values): no
// wave waits for one that has not started.
//
// The hand-over has no release or acquire of the language: those are fences of
// whole caches at agent scope (buffer_wbl2, buffer_inv), and an acquire in every
// collide wave alone costs more than the launch saves (steps of FP64 128^3
// 1.95 times as long, 256^3 1.86, FP32 190x151x117 1.77, FP16 384^3 2.97; a
// release in every psi wave takes longer still).  It is made for gfx950 and rests
// on this:
//  - Out: psi and flags are stored at agent scope, which writes through the L2 of
//    the XCD to what all XCDs share, and such a store leaves vmcnt when it is
//    there.  Every psi wave waits for vmcnt 0, then the workgroup's barrier, then
//    one lane stores the flag.
//  - In: flags are loaded at agent scope, past the XCD's own caches.  psi is
//    loaded only after the flags were seen (a branch on their value, and a
//    barrier to the compiler), by ordinary loads; those are right as long as
//    neither L1 nor L2 of the reader holds an older copy of the line:
//     * a launch starts with both invalidated (S and P were written on other XCDs
//       by the launch before, like the populations, which rely on it, too);
//     * in the launch no line is read before its flag: a collide reads psi only
//       in split_needs, psi workgroups read none, and caches fetch only lines
//       that are asked for;
//     * a line belongs to one wave: 64 sites of one component are whole lines of
//       128 bytes, as blocks and the components' strides are whole multiples of 64
//       sites (asserted below, and in split_order_serves).  Its other bytes are
//       densities of solid sites, which no launch writes.
//  - A wave that computes psi itself stores the values that the others store, and
//    reads them after vmcnt 0 through its own XCD's L2, which they went through.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the hand-over of psi is made for the caches of gfx950"
#endif
static_assert(kSplitThreads / 2 % 64 == 0 && kShiftSites % 64 == 0 &&
                  64 * sizeof(double) % 128 == 0 && 64 * sizeof(float) % 128 == 0,
              "a wave writes whole lines of psi");

struct SplitPlan {
  const int32_t *order;  // what each turn of eight workgroups does
  uint8_t *flags;        // [2][nflag]: the psi of a block is written
  int nflag;             // flags of a set: the blocks rounded up to 8
  int set;               // the flags this launch sets; it clears the others
  int polls;             // looks at the flags before a wave computes the psi itself
};

// Flags of one set for nb blocks.
inline int split_flags(int nb) { return (nb + 7) / 8 * 8; }

// Nonzero in some lane while the psi that a collide of block blk of a lattice
// reads is not all flagged.  Lane group k takes the k-th interval of
// split_needs, a lane eight flags at a time.  blk0: the lattice's first flag.
__device__ inline uint64_t psi_missing(const SplitPlan &q, const Geo &g, int SB, int blk0, int blk) {
  const uint64_t *w = reinterpret_cast<const uint64_t *>(q.flags + (int64_t)q.set * q.nflag);
  const int lane = threadIdx.x & 63;
  int lo, hi;
  split_needs(g, SB, blk, lane >> 3, lo, hi);
  lo += blk0;
  hi += blk0;
  uint64_t miss = 0;
  if (lo <= hi)
    for (int k = (lo >> 3) + (lane & 7); k <= (hi >> 3); k += 8) {
      uint64_t need = 0x0101010101010101ull;
      if (k == (lo >> 3)) need &= ~0ull << (8 * (lo & 7));
      if (k == (hi >> 3)) need &= ~0ull >> (56 - 8 * (hi & 7));
      miss |= need & ~__hip_atomic_load(w + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  return miss;
}

// SplitPlan::polls: some tens of milliseconds, where a wave that the order
// serves waits a few microseconds.
constexpr int kPsiPolls = 1 << 14;

// Polls until psi_missing is zero in all lanes; false when that took too long.
__device__ inline bool psi_wait(const SplitPlan &q, const Geo &g, int SB, int blk0, int blk) {
  for (int t = 0; t < q.polls; ++t)
    if (__all(psi_missing(q, g, SB, blk0, blk) == 0)) return true;
  return false;
}

// A psi value that workgroups on other XCDs read during this launch.
template <bool SHARED, class T>
__device__ inline void psi_store(T *p, T v) {
  if constexpr (SHARED)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    *p = v;
}

// Flag a block once every wave of the workgroup has its psi out (and clear the
// flag for the next launch).
__device__ inline void psi_publish(const SplitPlan &q, int blk) {
  __syncthreads();
  if (threadIdx.x == 0) {
    __hip_atomic_store(q.flags + (int64_t)q.set * q.nflag + blk, (uint8_t)1, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q.flags + (int64_t)(q.set ^ 1) * q.nflag + blk, (uint8_t)0,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Element k of the array at `base` (wave-uniform).  OFF32 (every byte offset
// of the kernel below 2^32): the byte offset is formed in 32 bits, so the access
// takes the scalar base and a 32-bit lane offset instead of a 64-bit lane
// address (one address register and no 64-bit arithmetic per access).
template <bool OFF32, class T>
__device__ inline T *elem(T *base, int64_t k) {
  if constexpr (OFF32) {
    using Byte = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return reinterpret_cast<T *>(reinterpret_cast<Byte *>(base) +
                                 (uint32_t)((uint32_t)k * (uint32_t)sizeof(T)));
  } else {
    return base + k;
  }
}
template <bool OFF32, class T>
__device__ inline const T &at(const T *base, int64_t k) {
  return *elem<OFF32>(base, k);
}

// Index offsets from a site to its neighbours along each axis with the
// periodic wrap folded in (m: -1, p: +1), set up once per lane: a neighbour
// index is then the site plus up to three of them, instead of three wraps
// (compare and select each) and two 32-bit multiplies per neighbour.
struct NbrOffsets {
  int xm, xp, ym, yp, zm, zp;
};

__device__ inline NbrOffsets nbr_offsets(const Geo &g, int x, int y, int z) {
  const int plane = g.ny * g.nz;
  NbrOffsets o;
  o.xm = x == 0 ? (g.nx - 1) * plane : -plane;
  o.xp = x == g.nx - 1 ? -(g.nx - 1) * plane : plane;
  o.ym = y == 0 ? (g.ny - 1) * g.nz : -g.nz;
  o.yp = y == g.ny - 1 ? -(g.ny - 1) * g.nz : g.nz;
  o.zm = z == 0 ? g.nz - 1 : -1;
  o.zp = z == g.nz - 1 ? -(g.nz - 1) : 1;
  return o;
}

// Site s + (cx, cy, cz), each component in {-1, 0, 1} (the same index as
// site_of over the wrapped coordinates).
__device__ inline int nbr_site(int s, const NbrOffsets &o, int cx, int cy, int cz) {
  return s + (cx < 0 ? o.xm : (cx > 0 ? o.xp : 0)) + (cy < 0 ? o.ym : (cy > 0 ? o.yp : 0)) +
         (cz < 0 ? o.zm : (cz > 0 ? o.zp : 0));
}

// Whether the byte offsets of a component's populations (FP64), or of both
// components' (shifted storage, `elem` bytes a value), stay below 2^32.
inline bool split_off32(const Geo &g) { return 19 * 8 * g.sp < ((int64_t)1 << 32); }
inline bool shift_off32(const Geo &g, int elem) { return 38 * elem * g.sp < ((int64_t)1 << 32); }

// tile_elem<19> of a site; OFF32: in 32 bits, with a 24-bit product (site
// indices are below 2^30).
template <bool OFF32>
__device__ inline auto tile_off(int s) {
  if constexpr (OFF32)
    return (uint32_t)s + __umul24((uint32_t)s >> 6, 64u * 18u);
  else
    return tile_elem<19>(s);
}

// The 19 streamed populations of component f (array Af) at site s = (x, y, z)
// whose solid word is sw (pull with bounce-back, src/dlbc/lb/advection.d:61-89).
// Each load takes a wave-uniform base, population min(i, bounce(i)) of tile 0,
// and a lane offset.
template <bool SOLID, bool OFF32, class T>
__device__ inline T pull_one(const T *__restrict__ Af, const Geo &g, int i, int s,
                             const NbrOffsets &o, uint32_t sw) {
  using L = D3Q19;
  const int src = nbr_site(s, o, -L::c[i][0], -L::c[i][1], -L::c[i][2]);
  if (!SOLID) return at<OFF32>(Af + 64 * i, tile_off<OFF32>(src));
  const int b = L::bounce[i], mc = i < b ? i : b;
  const bool bb = (sw >> b) & 1u;
  return at<OFF32>(Af + 64 * mc, 64 * ((bb ? b : i) - mc) + tile_off<OFF32>(bb ? s : src));
}

template <bool SOLID, bool OFF32>
__device__ inline void split_pull(const double *__restrict__ Af, const Geo &g, int s,
                                  const NbrOffsets &o, uint32_t sw, double *n) {
#pragma unroll
  for (int i = 0; i < 19; ++i) n[i] = pull_one<SOLID, OFF32>(Af, g, i, s, o, sw);
}

// Coordinates of site s of this lane, where the wave's sites are consecutive
// from s - (lane): the wave's first site is decomposed once with
// wave-uniform (scalar) arithmetic and each lane adds its offset with at
// most one carry when n_z >= 64, instead of two 32-bit divisions per lane.
__device__ inline void lane_coords(int s, const Geo &g, int &x, int &y, int &z) {
  if (g.nz < 64) {
    coords(s, g, x, y, z);
    return;
  }
  const int lane = threadIdx.x & 63;
  int x0, y0, z0;
  coords(uniform(s - lane), g, x0, y0, z0);
  x = x0;
  y = y0;
  z = z0 + lane;
  if (z >= g.nz) {
    z -= g.nz;
    if (++y == g.ny) {
      y = 0;
      ++x;
    }
  }
}

// psi rows of a block of SB consecutive sites that lie in one z-row (n_z a
// multiple of SB), staged in LDS: the nine rows (x + dx, y + dy), dx, dy in
// {-1, 0, 1}, from z0 - 1 to z0 + SB (periodic), of both components.  Every
// neighbour psi (and the solid density in the same array) of the block is in
// them.  The rows are read with 16-byte loads (four FP32 or two FP64 values
// per lane, aligned: n_z, z0 and the component stride are multiples of 64),
// in units of one row and one 64-lane pass, dealt round-robin to the waves:
// a wave-uniform row base and consecutive z per lane, no wrap inside the
// block's span.  The 36 end values (z0 - 1 and z0 + SB of each row) take one
// pass of wave 0.  The loads go out first and the LDS stores follow, so that
// the loads overlap the population pulls issued before; the caller's barrier
// publishes the rows.
template <int SB, int THREADS, bool OFF32, class T>
__device__ inline void stage_psi_rows(const T *S, const Geo &g, int s0,
                                      T (*rows)[9][SB + 2]) {
  constexpr int VEC = 16 / (int)sizeof(T);  // values per 16-byte load
  typedef T Vec __attribute__((ext_vector_type(VEC)));
  constexpr int NW = THREADS / 64, NR = 18, PASS = SB / (64 * VEC);
  constexpr int NU = NR * PASS, UPW = (NU + NW - 1) / NW;  // units, per wave
  static_assert(SB % (64 * VEC) == 0, "staged rows take whole lane passes");
  int x0, y0, z0;
  coords(uniform(s0), g, x0, y0, z0);
  const int w = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // element offset of row pr: component pr / 9, row (dx, dy) = pr % 9 (the
  // wrap is arithmetic: a select among three coordinates became a lookup
  // table in scratch memory)
  auto pair_base = [&](int pr) {
    const int row = pr % 9;
    const int xx = wrap(x0 + row / 3 - 1, g.nx), yy = wrap(y0 + row % 3 - 1, g.ny);
    return (int64_t)(pr / 9) * g.sp + (int64_t)(xx * g.ny + yy) * g.nz;
  };
  Vec v[UPW];
#pragma unroll
  for (int q = 0; q < UPW; ++q) {
    const int u = w + q * NW, pr = (u < NU ? u : 0) / PASS, k = (u < NU ? u : 0) % PASS;
    const T *base = S + pair_base(pr) + z0;
    v[q] = u < NU ? *reinterpret_cast<const Vec *>(elem<OFF32>(base, VEC * (lane + 64 * k)))
                  : Vec(T(0));
  }
  // the two ends of every row's span: lane 2 pr + side of wave 0
  const bool edge = w == 0 && lane < 2 * NR;
  const int epr = lane >> 1, side = lane & 1;
  T ve = T(0);
  if (edge) {
    const int ze = side ? (z0 + SB == g.nz ? 0 : z0 + SB) : (z0 == 0 ? g.nz - 1 : z0 - 1);
    ve = at<OFF32>(S, pair_base(epr) + ze);
  }
#pragma unroll
  for (int q = 0; q < UPW; ++q) {
    const int u = w + q * NW;
    if (u < NU) {
      T *row = rows[u / PASS / 9][u / PASS % 9] + 1 + VEC * (lane + 64 * (u % PASS));
#pragma unroll
      for (int j = 0; j < VEC; ++j) row[j] = v[q][j];
    }
  }
  if (edge) rows[epr / 9][epr % 9][side ? SB + 1 : 0] = ve;
}

// The staged value of component ff at x + c_i for site k of the block (i < 0: x).
template <int SB, class T>
__device__ inline T staged_psi(const T (*rows)[9][SB + 2], int ff, int i, int k) {
  using L = D3Q19;
  if (i < 0) return rows[ff][4][k + 1];
  return rows[ff][(L::c[i][0] + 1) * 3 + L::c[i][1] + 1][k + 1 + L::c[i][2]];
}

// psi of wave w's sites and component of block blk.
template <bool SOLID, bool OFF32, bool SHARED>
__device__ inline void split_psi_wave(const double *__restrict__ A,
                                      const uint32_t *__restrict__ nbw, double *S, const Geo &g,
                                      int psi_form, int blk, int w) {
  int s, f;
  if (!split_lane(g, blk, w, s, f)) return;
  const uint32_t sw = SOLID ? nbw[s] : 0u;
  if (sw >> 31) return;  // solid: S keeps the site's density
  int x, y, z;
  lane_coords(s, g, x, y, z);
  double n[19];
  split_pull<SOLID, OFF32>(A + (int64_t)f * 19 * g.sp, g, s, nbr_offsets(g, x, y, z), sw, n);
  psi_store<SHARED>(elem<OFF32>(S + (int64_t)f * g.sp, s), psi_of(psi_form, density<D3Q19>(n)));
}

template <bool SOLID, bool OFF32>
__global__ void __launch_bounds__(kSplitThreads)
    k_split_psi(const double *__restrict__ A, const uint32_t *__restrict__ nbw,
                double *__restrict__ S, Geo g, int psi_form) {
  split_psi_wave<SOLID, OFF32, false>(A, nbw, S, g, psi_form, split_block(g, blockIdx.x),
                                      uniform(threadIdx.x >> 6));
}

// addShanChenForcePsi (src/dlbc/lb/force.d:238-309) for two components whose
// self-couplings gcc[f][f] are zero: the reference skips the f2 == f1 term,
// so only the other component contributes and every lane of a wave runs the
// same loop (sc_force with its lane-dependent skip runs both halves masked).
// Same operations in the same order as sc_force, hence the same bits.
template <class Psi, class Solid, class RhoSolid>
__device__ inline void sc_force_offdiag(int f1, double (&F)[3], const StepParams &p, Psi psi,
                                        Solid solid, RhoSolid rho_solid) {
  using L = D3Q19;
#pragma unroll
  for (int d = 0; d < 3; ++d) F[d] = 0.0;
  if (!p.sc) return;
  const double psi1 = psi(f1, -1);
  const int f2 = f1 ^ 1;
  const double cc = p.gcc[f1][f2];
  if (cc != 0.0) {
#pragma unroll
    for (int i = 1; i < L::q; ++i) {
      const double psi_n = psi(f2, i);  // read before the test, as in sc_force
      const double psi2 = solid(i) ? psi(f2, -1) : psi_n;
      const double pf = L::w[i] * psi1 * psi2 * cc;
#pragma unroll
      for (int d = 0; d < 3; ++d) F[d] -= pf * static_cast<double>(L::c[i][d]);
    }
  }
  const double wc = p.gwc[f1];
  if (wc != 0.0 && p.has_solid) {
#pragma unroll
    for (int i = 0; i < L::q; ++i) {
      if (solid(i)) {
        const double pf = L::w[i] * psi1 * rho_solid(f1, i) * wc;
#pragma unroll
        for (int d = 0; d < 3; ++d) F[d] -= pf * static_cast<double>(L::c[i][d]);
      }
    }
  }
}

// collide_component (distributeForce, body force, velocity shift, eqDist and
// BGK relaxation) for D3Q19 with every equilibrium value stored as soon as it
// is formed, instead of through a 19-value array: the same operations in the
// same order (lattice.hpp eq_dist, kernels_twopass.hpp collide_component), so
// the same bits, with fewer registers live at the stores.
template <class Out>
__device__ inline void collide_d3q19_streamed(int f, const double *n, double rho, double total,
                                              double (&F)[3], const double *wv,
                                              const StepParams &p, Out out) {
  using L = D3Q19;
#pragma unroll
  for (int d = 0; d < 3; ++d) F[d] += 0.0 * (rho / total);
  if (p.has_body) {
#pragma unroll
    for (int d = 0; d < 3; ++d) F[d] += p.body[f][d];
  }
  double dv[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    dv[d] = p.tau[f] * (p.gacc[d] + F[d] / rho);
    if (p.eq_form == kBDist2) dv[d] += wv[d];
  }
  const double omw = p.one_minus_omega[f], om = p.omega[f];
  auto relax = [&](int i, double eq) { out(i, n[i] * omw + om * eq); };
  if (p.eq_form != kBDist2) {  // eqdist.d:82-100
    double pv[3], v[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) pv[j] = 0.0;
#pragma unroll
    for (int i = 0; i < 19; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) pv[j] += n[i] * static_cast<double>(L::c[i][j]);
#pragma unroll
    for (int j = 0; j < 3; ++j) pv[j] /= rho;
#pragma unroll
    for (int j = 0; j < 3; ++j) v[j] = dv[j] + pv[j];
    double vdotv = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) vdotv += v[j] * v[j];
    constexpr double css = kCss;
    constexpr double css2 = 2.0 * css;
    constexpr double css2p2 = css2 * css;
    constexpr double css6p3 = 3.0 * css2p2 * css;
    constexpr double r_css = 1.0 / css, r_css2 = 1.0 / css2, r_css2p2 = 1.0 / css2p2,
                     r_css6p3 = 1.0 / css6p3;
    const double vv_css2 = div_const(vdotv, css2, r_css2);
    const bool third = p.eq_form == kThirdOrder;
#pragma unroll
    for (int i = 0; i < 19; ++i) {
      double vc = 0.0;
#pragma unroll
      for (int j = 0; j < 3; ++j) vc += v[j] * static_cast<double>(L::c[i][j]);
      double eq;
      if (!third)
        eq = rho * L::w[i] *
             (1.0 + div_const(vc, css, r_css) + div_const(vc * vc, css2p2, r_css2p2) - vv_css2);
      else
        eq = rho * L::w[i] *
             (1.0 + div_const(vc, css, r_css) + div_const(vc * vc, css2p2, r_css2p2) - vv_css2 +
              div_const(vc * vc * vc, css6p3, r_css6p3) - div_const(vdotv * vc, css2p2, r_css2p2));
      relax(i, eq);
    }
    return;
  }
  // BDist2, eqdist.d:102-184
  const double aN1 = 1.0 / 36.0, aN0 = 1.0 / 3.0;
  const double haN1 = 0.5 * aN1, aN1_6 = aN1 / 6.0;
  const double T = 1.0 / 3.0, holdit = 1.0 / T;
  const double tux = dv[0], tuy = dv[1], tuz = dv[2];
  const double tuxt = tux * holdit, tuyt = tuy * holdit, tuzt = tuz * holdit;
  const double uke = 0.5 * (tux * tuxt + tuy * tuyt + tuz * tuzt);
  const double cst = 1.0 - uke;
  const double const1 = aN1 * cst;
  auto pair = [&](double cdotu, int ip, int im, bool axis) {
    const double even = const1 + haN1 * cdotu * cdotu;
    const double odd = const1 * cdotu + aN1_6 * cdotu * cdotu * cdotu;
    if (axis) {
      relax(ip, 2.0 * (even + odd) * rho);
      relax(im, 2.0 * (even - odd) * rho);
    } else {
      relax(ip, (even + odd) * rho);
      relax(im, (even - odd) * rho);
    }
  };
  relax(0, aN0 * cst * rho);
  pair(tuxt, 1, 2, true);
  pair(tuyt, 3, 4, true);
  pair(tuzt, 5, 6, true);
  pair(tuxt + tuyt, 7, 14, false);
  pair(tuxt - tuyt, 13, 8, false);
  pair(tuxt + tuzt, 11, 18, false);
  pair(tuxt - tuzt, 12, 17, false);
  pair(tuyt + tuzt, 9, 16, false);
  pair(tuyt - tuzt, 15, 10, false);
}

// STAGED (n_z a multiple of the block's sites): the psi rows come from LDS.
// A template argument rather than a runtime test, so that the body holds one
// psi source: with both, every psi read sat behind a branch and a full wait.
// ONE: both passes in one launch (SplitPlan q); else the second pass alone.
template <bool SOLID, bool OFFDIAG, bool OFF32, bool STAGED, bool ONE>
__global__ void __launch_bounds__(kSplitThreads)
    k_split_collide(const double *__restrict__ A, double *__restrict__ B,
                    const uint32_t *__restrict__ nbw, double *S, Geo g, StepParams p,
                    SplitPlan q) {
  using L = D3Q19;
  constexpr int C = 2;
  constexpr int SB = kSplitThreads / 2;
  // density and first moment of both components of the block's sites
  __shared__ double xch[2][4][SB];
  // psi rows of the block when it lies in one z-row
  __shared__ double rows[STAGED ? 2 : 1][9][SB + 2];
  constexpr bool staged = STAGED;
  const int w = uniform(threadIdx.x >> 6);
  int blk;
  if constexpr (ONE) {
    const int32_t turn = q.order[blockIdx.x >> 3];
    if ((int)(blockIdx.x & 7) >= turn_count(turn)) return;
    blk = turn_first(turn) + (int)(blockIdx.x & 7) * turn_stride(turn);
    const bool is_psi = !turn_collide(turn);
    if (is_psi || !psi_wait(q, g, SB, 0, blk)) {
      // the wave's part of the block's psi, or (not waited for any longer) all
      // psi that this collide reads
      for (int i = 0; i < (is_psi ? 1 : 8); ++i) {
        int b = blk, b1 = blk;
        if (!is_psi) split_needs(g, SB, blk, i, b, b1);
        for (; b <= b1; ++b)
          for (int v = is_psi ? w : 0; v <= (is_psi ? w : kSplitThreads / 64 - 1); ++v)
            split_psi_wave<SOLID, OFF32, true>(A, nbw, S, g, p.psi_form, b, v);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (is_psi) {
        psi_publish(q, blk);
        return;
      }
    }
    asm volatile("" ::: "memory");  // psi is read from here on
  } else {
    blk = split_block(g, blockIdx.x);
  }
  int s, f;
  const bool inside = split_lane(g, blk, w, s, f);
  const int k = ((threadIdx.x >> 7) << 6) | (threadIdx.x & 63);  // site within the block
  const uint32_t sw = !inside ? (1u << 31) : (SOLID ? nbw[s] : 0u);
  NbrOffsets o{};
  double n[19];
  double rho = 0.0, mom[3] = {0.0, 0.0, 0.0};
  const bool bdist2 = p.eq_form == kBDist2;
  // A solid site's lane copies its own populations (the reference copies them
  // every step, advection.d:84-86): with every neighbour taken as solid, the
  // pull loads population bounce(i) of the site itself into n[i], in the same
  // load instructions as the fluid lanes' pulls, and the store below writes
  // n[bounce(i)] back to population i.  Whole cache lines are then written;
  // skipping the solid lanes left partially written lines, which cost 7 % of
  // the pass on the 256^3 channel.
  const bool solid_site = inside && (sw >> 31);
  const bool active = inside && !(SOLID && line_all_solid<16>(solid_site));
  if (active) {
    int x, y, z;
    lane_coords(s, g, x, y, z);
    o = nbr_offsets(g, x, y, z);
    split_pull<SOLID, OFF32>(A + (int64_t)f * 19 * g.sp, g, s, o, solid_site ? 0x7ffffu : sw,
                             n);
  }
  if (staged) stage_psi_rows<SB, kSplitThreads, OFF32>(S, g, blk * SB, rows);
  if (active) {
    rho = density<L>(n);
    if (bdist2) first_moment<L>(n, mom);
  }
  xch[f][0][k] = rho;
  if (bdist2) {
#pragma unroll
    for (int d = 0; d < 3; ++d) xch[f][1 + d][k] = mom[d];
  }
  __syncthreads();
  if (!active) return;
  // (a solid lane runs the arithmetic below on its own populations, whose
  // result it does not store: no divergent branch in a mixed wave)
  const double rho_partner = xch[f ^ 1][0][k];
  double mom_p[3];
  if (bdist2) {
#pragma unroll
    for (int d = 0; d < 3; ++d) mom_p[d] = xch[f ^ 1][1 + d][k];
  }
  auto nbr = [&](int i) { return nbr_site(s, o, L::c[i][0], L::c[i][1], L::c[i][2]); };
  double F[3];
  auto psi = [&](int ff, int i) {
    if (staged) return staged_psi<SB>(rows, ff, i, k);
    return at<OFF32>(S + ff * g.sp, i < 0 ? s : nbr(i));
  };
  auto solid = [&](int i) { return SOLID && ((sw >> i) & 1u); };
  auto rho_solid = [&](int ff, int i) {  // S holds the density at solid sites
    if (staged) return staged_psi<SB>(rows, ff, i, k);
    return at<OFF32>(S + ff * g.sp, nbr(i));
  };
  if constexpr (OFFDIAG)
    sc_force_offdiag(f, F, p, psi, solid, rho_solid);
  else
    sc_force<L, C>(f, F, p, psi, solid, rho_solid);
  const double total = total_density<C>([&](int ff) { return ff == f ? rho : rho_partner; });
  double wv[3];
  if (bdist2)
    weighted_velocity<L, C>([&](int ff, int d) { return ff == f ? mom[d] : mom_p[d]; }, total,
                            p, wv);
  double *__restrict__ Bf = B + (int64_t)f * 19 * g.sp;
  collide_d3q19_streamed(f, n, rho, total, F, wv, p, [&](int i, double v) {
    __builtin_nontemporal_store(solid_site ? n[L::bounce[i]] : v,
                                elem<OFF32>(Bf + 64 * i, tile_off<OFF32>(s)));
  });
}

// ---- shifted storage (FP32 / FP16 deviations, FP32 arithmetic) -------------
// The same two passes; psi goes through an FP32 array P (the values are FP32
// in every schedule) and the per-site arithmetic is shifted_collide_site, as
// in the tiled kernel, so a lattice gives the same bits under both schedules.
// S still gives the density at solid neighbours (wall force).

// Both components' streamed populations at site s (pull with bounce-back,
// src/dlbc/lb/advection.d:61-89): one 8-byte (FP32) or 4-byte (FP16) load
// per population and lane, from a wave-uniform base, population
// min(i, bounce(i)) of tile 0, at a lane offset.
template <class Store, bool SOLID, bool OFF32>
__device__ inline void ssplit_pull(const Store *__restrict__ A, const Geo &g, int s,
                                   const NbrOffsets &o, uint32_t sw, float (&n0)[19],
                                   float (&n1)[19]) {
  using L = D3Q19;
#pragma unroll
  for (int i = 0; i < 19; ++i) {
    const int src = nbr_site(s, o, -L::c[i][0], -L::c[i][1], -L::c[i][2]);
    const Store *p;
    if (!SOLID) {
      p = elem<OFF32>(A + 128 * i, 2 * tile_off<OFF32>(src));
    } else {
      const int b = L::bounce[i], mc = i < b ? i : b;
      const bool bb = (sw >> b) & 1u;
      p = elem<OFF32>(A + 128 * mc, 128 * ((bb ? b : i) - mc) + 2 * tile_off<OFF32>(bb ? s : src));
    }
    pair_load(p, n0[i], n1[i]);
  }
}

// The sites of block blk of a lattice (kShiftSites from blk * kShiftSites),
// one per lane of its waves w.
__device__ inline int shift_site(int blk, int w) {
  return uniform(blk * kShiftSites + 64 * w) + (threadIdx.x & 63);
}

// Pass 1 for the sites of wave w of block blk of a lattice: psi of both
// components into P.
template <class Store, bool SOLID, bool OFF32, bool SHARED = false>
__device__ inline void ssplit_psi_wave(const Store *__restrict__ A,
                                       const uint32_t *__restrict__ nbw, float *P, const Geo &g,
                                       const ShiftParams &p, int blk, int w) {
  const int s = shift_site(blk, w);
  if (s >= g.sites) return;
  const uint32_t sw = SOLID ? nbw[s] : 0u;
  if (sw >> 31) return;  // solid: psi is not read there
  int x, y, z;
  lane_coords(s, g, x, y, z);
  float n0[19], n1[19];
  ssplit_pull<Store, SOLID, OFF32>(A, g, s, nbr_offsets(g, x, y, z), sw, n0, n1);
  psi_store<SHARED>(elem<OFF32>(P, s), psi_f(p.psi_form, p.rho0[0] + shifted_drho(n0)));
  psi_store<SHARED>(elem<OFF32>(P + g.sp, s), psi_f(p.psi_form, p.rho0[1] + shifted_drho(n1)));
}

// The start of a workgroup of a one-launch step: its psi (then false: nothing is
// left to do), or the wait of a collide workgroup (true).  blk0: the lattice's
// first block in q.
template <class Store, bool SOLID, bool OFF32>
__device__ inline bool shift_one_launch(const Store *__restrict__ A,
                                        const uint32_t *__restrict__ nbw, float *P, const Geo &g,
                                        const ShiftParams &p, const SplitPlan &q, int blk0,
                                        int blk, bool collide) {
  const int w = uniform(threadIdx.x >> 6);
  if (!collide || !psi_wait(q, g, kShiftSites, blk0, blk)) {
    for (int i = 0; i < (collide ? 8 : 1); ++i) {
      int b = blk, b1 = blk;
      if (collide) split_needs(g, kShiftSites, blk, i, b, b1);
      for (; b <= b1; ++b)
        for (int v = collide ? 0 : w; v <= (collide ? kShiftThreads / 64 - 1 : w); ++v)
          ssplit_psi_wave<Store, SOLID, OFF32, true>(A, nbw, P, g, p, b, v);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!collide) {
      psi_publish(q, blk0 + blk);
      return false;
    }
  }
  asm volatile("" ::: "memory");  // psi is read from here on
  return true;
}

template <class Store, bool SOLID, bool OFF32>
__device__ inline void ssplit_psi_block(const Store *__restrict__ A,
                                        const uint32_t *__restrict__ nbw, float *P, const Geo &g,
                                        const ShiftParams &p, int blk) {
  ssplit_psi_wave<Store, SOLID, OFF32>(A, nbw, P, g, p, blk, uniform(threadIdx.x >> 6));
}

// Pass 2 for block blk of a lattice; rows: LDS for the block's psi rows when
// STAGED (n_z a multiple of kShiftSites).  STAGED is a template argument, not
// a runtime test: with both psi sources in one body the compiler merged the
// LDS and global reads into flat loads, each waiting for all memory traffic
// of the wave.  A lane collides component 0 (keeping the result in place of
// its populations) and then component 1, and stores each population of both
// components with one access.
template <class Store, bool SOLID, bool OFF32, bool STAGED = false>
__device__ inline void ssplit_collide_block(const Store *__restrict__ A, Store *__restrict__ B,
                                            const uint32_t *__restrict__ nbw, float *P,
                                            const Geo &g, const ShiftParams &p, int blk,
                                            float (*rows)[9][kShiftSites + 2]) {
  using L = D3Q19;
  constexpr int SB = kShiftSites;
  constexpr bool staged = STAGED;
  const int s = shift_site(blk, uniform(threadIdx.x >> 6));
  const int k = threadIdx.x;  // site within the block
  const uint32_t sw = s >= g.sites ? (1u << 31) : (SOLID ? nbw[s] : 0u);
  NbrOffsets o{};
  float n0[19], n1[19];
  // a solid site's lane copies its own populations, as in the FP64 pass: the
  // pull with every neighbour taken as solid loads population bounce(i) of the
  // site into n[i], and the store writes n[bounce(i)] back to population i
  const bool inside = s < g.sites, solid_site = inside && (sw >> 31);
  // a 128-byte line holds 16 (FP32) or 32 (FP16) sites' pairs
  const bool active =
      inside && !(SOLID && line_all_solid<128 / (2 * (int)sizeof(Store))>(solid_site));
  if (active) {
    int x, y, z;
    lane_coords(s, g, x, y, z);
    o = nbr_offsets(g, x, y, z);
    ssplit_pull<Store, SOLID, OFF32>(A, g, s, o, solid_site ? 0x7ffffu : sw, n0, n1);
  }
  if (staged) {
    stage_psi_rows<SB, kShiftThreads, OFF32>(P, g, blk * SB, rows);
    __syncthreads();
  }
  if (!active) return;
  const ShiftLane pl0 = shift_lane(p, 0), pl1 = shift_lane(p, 1);
  const float rho0 = pl0.rho0 + shifted_drho(n0), rho1 = pl1.rho0 + shifted_drho(n1);
  float j0[3], j1[3];
  shifted_moment(n0, j0);
  shifted_moment(n1, j1);
  auto nbr = [&](int i) { return nbr_site(s, o, L::c[i][0], L::c[i][1], L::c[i][2]); };
  auto psi = [&](int ff, int i) {
    if (staged) return staged_psi<SB>(rows, ff, i, k);
    return at<OFF32>(P + ff * g.sp, i < 0 ? s : nbr(i));
  };
  // both forces first (P holds the density at solid sites: wall force), so
  // the psi reads are consumed before the populations of a relaxation
  float F0[3], F1[3];
  shifted_force<SOLID>(0, sw, p, pl0, psi, [&](int i, bool) { return psi(0, i); }, F0);
  shifted_force<SOLID>(1, sw, p, pl1, psi, [&](int i, bool) { return psi(1, i); }, F1);
  shifted_relax(n0, rho0, rho1, j0, j1, F0, p, pl0,
                [&](int i, float v) { n0[i] = solid_site ? n0[i] : v; });
  shifted_relax(n1, rho1, rho0, j1, j0, F1, p, pl1, [&](int i, float v) {
    const int b = L::bounce[i];
    pair_store_nt<Store>(elem<OFF32>(B + 128 * i, 2 * tile_off<OFF32>(s)),
                         solid_site ? n0[b] : n0[i], solid_site ? n1[b] : v);
  });
}

template <class Store, bool SOLID, bool OFF32>
__global__ void __launch_bounds__(kShiftThreads)
    k_ssplit_psi(const Store *__restrict__ A, const uint32_t *__restrict__ nbw,
                 float *__restrict__ P, Geo g, ShiftParams p) {
  ssplit_psi_block<Store, SOLID, OFF32>(A, nbw, P, g, p, split_block(g, blockIdx.x));
}

// At most 128 VGPRs: four waves per SIMD.
template <class Store, bool SOLID, bool OFF32, bool STAGED, bool ONE>
__global__ void __launch_bounds__(kShiftThreads) __attribute__((amdgpu_waves_per_eu(4)))
    k_ssplit_collide(const Store *__restrict__ A, Store *__restrict__ B,
                     const uint32_t *__restrict__ nbw, float *P, Geo g, ShiftParams p,
                     SplitPlan q) {
  __shared__ float rows[STAGED ? 2 : 1][9][kShiftSites + 2];
  int blk;
  if constexpr (ONE) {
    const int32_t turn = q.order[blockIdx.x >> 3];
    if ((int)(blockIdx.x & 7) >= turn_count(turn)) return;
    blk = turn_first(turn) + (int)(blockIdx.x & 7) * turn_stride(turn);
    if (!shift_one_launch<Store, SOLID, OFF32>(A, nbw, P, g, p, q, 0, blk, turn_collide(turn)))
      return;
  } else {
    blk = split_block(g, blockIdx.x);
  }
  ssplit_collide_block<Store, SOLID, OFF32, STAGED>(A, B, nbw, P, g, p, blk, rows);
}

// Blocks of kShiftSites sites over a lattice.
inline int shift_grid(int64_t sites) { return (int)((sites + kShiftSites - 1) / kShiftSites); }

template <class Store, bool OFF32, bool STAGED, bool ONE>
inline void launch_ssplit_collide(const Store *a, Store *b, const uint32_t *nbw, float *P,
                                  const Geo &g, const ShiftParams &p, const SplitPlan &q, int nb,
                                  hipStream_t stream) {
  const dim3 grid(nb), block(kShiftThreads);
  if (p.has_solid)
    hipLaunchKernelGGL((k_ssplit_collide<Store, true, OFF32, STAGED, ONE>), grid, block, 0,
                       stream, a, b, nbw, P, g, p, q);
  else
    hipLaunchKernelGGL((k_ssplit_collide<Store, false, OFF32, STAGED, ONE>), grid, block, 0,
                       stream, a, b, nbw, P, g, p, q);
}

// pass 0: psi, 1: collide, 2: both in one launch of `norder` workgroups.
template <class Store, bool OFF32>
inline void launch_ssplit_impl(const Store *a, Store *b, const uint32_t *nbw, float *P,
                               const Geo &g, const ShiftParams &p, const SplitPlan &q, int norder,
                               hipStream_t stream, int pass) {
  const int nb = shift_grid(g.sites);
  const dim3 grid(nb), block(kShiftThreads);
  const bool staged = g.nz % kShiftSites == 0;
  if (pass == 0 && p.has_solid)
    hipLaunchKernelGGL((k_ssplit_psi<Store, true, OFF32>), grid, block, 0, stream, a, nbw, P, g,
                       p);
  else if (pass == 0)
    hipLaunchKernelGGL((k_ssplit_psi<Store, false, OFF32>), grid, block, 0, stream, a, nbw, P, g,
                       p);
  else if (pass == 2 && staged)
    launch_ssplit_collide<Store, OFF32, true, true>(a, b, nbw, P, g, p, q, norder, stream);
  else if (pass == 2)
    launch_ssplit_collide<Store, OFF32, false, true>(a, b, nbw, P, g, p, q, norder, stream);
  else if (staged)
    launch_ssplit_collide<Store, OFF32, true, false>(a, b, nbw, P, g, p, q, nb, stream);
  else
    launch_ssplit_collide<Store, OFF32, false, false>(a, b, nbw, P, g, p, q, nb, stream);
}

template <class Store>
inline void launch_ssplit_d3q19(const void *A, void *B, const uint32_t *nbw, float *P,
                                const Geo &g, const ShiftParams &p, const SplitPlan &q,
                                int norder, hipStream_t stream, int pass) {
  const Store *a = static_cast<const Store *>(A);
  Store *b = static_cast<Store *>(B);
  if (shift_off32(g, sizeof(Store)))
    launch_ssplit_impl<Store, true>(a, b, nbw, P, g, p, q, norder, stream, pass);
  else
    launch_ssplit_impl<Store, false>(a, b, nbw, P, g, p, q, norder, stream, pass);
}

template <bool OFF32, bool STAGED, bool ONE>
inline void launch_split_collide(const double *A, double *B, const uint32_t *nbw, double *S,
                                 const Geo &g, const StepParams &p, const SplitPlan &q, int nb,
                                 hipStream_t stream, bool solid, bool offdiag) {
  const dim3 grid(nb), block(kSplitThreads);
  if (solid && offdiag)
    hipLaunchKernelGGL((k_split_collide<true, true, OFF32, STAGED, ONE>), grid, block, 0, stream,
                       A, B, nbw, S, g, p, q);
  else if (solid)
    hipLaunchKernelGGL((k_split_collide<true, false, OFF32, STAGED, ONE>), grid, block, 0, stream,
                       A, B, nbw, S, g, p, q);
  else if (offdiag)
    hipLaunchKernelGGL((k_split_collide<false, true, OFF32, STAGED, ONE>), grid, block, 0, stream,
                       A, B, nbw, S, g, p, q);
  else
    hipLaunchKernelGGL((k_split_collide<false, false, OFF32, STAGED, ONE>), grid, block, 0, stream,
                       A, B, nbw, S, g, p, q);
}

// pass 0: psi, 1: collide, 2: both in one launch of `norder` workgroups.
template <bool OFF32>
inline void launch_split_impl(const double *A, double *B, const uint32_t *nbw, double *S,
                              const Geo &g, const StepParams &p, const SplitPlan &q, int norder,
                              hipStream_t stream, int pass) {
  const int nb = split_grid(g.sites);
  const dim3 grid(nb), block(kSplitThreads);
  const bool solid = p.has_solid != 0;
  if (pass == 0) {
    if (solid)
      hipLaunchKernelGGL((k_split_psi<true, OFF32>), grid, block, 0, stream, A, nbw, S, g,
                         p.psi_form);
    else
      hipLaunchKernelGGL((k_split_psi<false, OFF32>), grid, block, 0, stream, A, nbw, S, g,
                         p.psi_form);
    return;
  }
  const bool offdiag = p.gcc[0][0] == 0.0 && p.gcc[1][1] == 0.0;
  const bool staged = g.nz % (kSplitThreads / 2) == 0;
  if (pass == 2 && staged)
    launch_split_collide<OFF32, true, true>(A, B, nbw, S, g, p, q, norder, stream, solid, offdiag);
  else if (pass == 2)
    launch_split_collide<OFF32, false, true>(A, B, nbw, S, g, p, q, norder, stream, solid,
                                             offdiag);
  else if (staged)
    launch_split_collide<OFF32, true, false>(A, B, nbw, S, g, p, q, nb, stream, solid, offdiag);
  else
    launch_split_collide<OFF32, false, false>(A, B, nbw, S, g, p, q, nb, stream, solid, offdiag);
}

inline void launch_split_d3q19(const double *A, double *B, const uint32_t *nbw, double *S,
                               const Geo &g, const StepParams &p, const SplitPlan &q, int norder,
                               hipStream_t stream, int pass) {
  if (split_off32(g))
    launch_split_impl<true>(A, B, nbw, S, g, p, q, norder, stream, pass);
  else
    launch_split_impl<false>(A, B, nbw, S, g, p, q, norder, stream, pass);
}

}  // namespace dlbc
