// kernels_tile.hpp -- one Shan-Chen step of a D2Q9 lattice in one launch (FP64).
//
// A step of a two-dimensional lattice of up to some 10^5 sites is bound by
// latency: two launches (psi, then collide) of 4 to 8 us each, most of it
// waiting for memory and for the chain of one site's arithmetic.  Here a
// workgroup computes psi of a tile of 4 x 16 sites and of the 44 sites around
// it, and then collides the tile: one launch, at the price of the psi of the
// border, which its neighbours compute too.  One lane per site and component;
// the border has waves of its own, so that all loads go out at once, and a
// tile's populations stay in registers from their psi to their collision.
// Small tiles spread a small lattice over the chip: 8 x 8, 8 x 16, 12 x 16 and
// 16 x 16 sites took 4.7, 5.3, 5.7 and 6.2 us on 64^2 (4 x 16: 4.7), 13, 13.7,
// 12 and 14.6 us on 321 x 257 (4 x 16: 11.3).  us per step, two launches / one:
// 64^2 9.3 / 4.7, 192^2 12.5 / 9.9, 321 x 257 16.5 / 11.3; three components,
// 192^2 15.9 / 11.7.
//
// Per-site arithmetic is the shared code of the other schedules, so the bits
// are the same.
#pragma once

#include "kernels_split.hpp"

namespace dlbc {

constexpr int kTileX = 4, kTileY = 16;
constexpr int kTileSites = kTileX * kTileY;  // one wave of each component
constexpr int kTileEX = kTileX + 2, kTileEY = kTileY + 2, kTileCells = kTileEX * kTileEY;
constexpr int kTileRing = kTileCells - kTileSites;  // at most one wave, too
static_assert(kTileSites == 64 && kTileRing <= 64, "one wave each");

// Cell of the r-th ring position: the two end rows along x, then the two ends
// of the rows between.
__device__ inline void tile_ring(int r, int &ex, int &ey) {
  if (r < 2 * kTileEY) {
    ex = r < kTileEY ? 0 : kTileX + 1;
    ey = r < kTileEY ? r : r - kTileEY;
  } else {
    r -= 2 * kTileEY;
    ex = 1 + (r >> 1);
    ey = (r & 1) ? kTileY + 1 : 0;
  }
}

// Six waves per SIMD (two of some 82 VGPRs spilled; five waves: 12.4 us on
// 321 x 257 with 64-bit addresses and selects for solids in every pull, 11.3 as
// it stands).
template <int C, bool SOLID>
__global__ void __launch_bounds__(2 * C * 64) __attribute__((amdgpu_waves_per_eu(6)))
    k_tile_step(const double *__restrict__ A, double *__restrict__ B,
                const uint32_t *__restrict__ nbw, const double *__restrict__ S, Geo g,
                StepParams p, int tiles_y) {
  using L = D2Q9;
  constexpr int Q = L::q, D = L::d;
  __shared__ double psi[C][kTileCells];  // at solid sites: the density
  __shared__ double xch[C][1 + D][kTileSites];
  // waves 0 .. C-1: the components of the tile's sites, C .. 2C-1: of the ring
  const int w = uniform(threadIdx.x >> 6), k = threadIdx.x & 63;
  const bool own = w < C;
  const int f = own ? w : w - C;
  int ex, ey;  // the lane's cell
  if (own) {
    ex = k / kTileY + 1;
    ey = k % kTileY + 1;
  } else {
    tile_ring(k, ex, ey);
  }
  const int cell = ex * kTileEY + ey;
  int x = (int)(blockIdx.x / tiles_y) * kTileX + ex - 1;
  int y = (int)(blockIdx.x % tiles_y) * kTileY + ey - 1;
  // a tile may stand over the end of an axis: a cell past the lattice and its
  // border is not needed
  const bool needed = (own || k < kTileRing) && x <= g.nx && y <= g.ny;
  const bool inside = own && x < g.nx && y < g.ny;
  x = x < 0 ? x + g.nx : (x >= g.nx ? x - g.nx : x);
  y = y < 0 ? y + g.ny : (y >= g.ny ? y - g.ny : y);
  const int s = x * g.ny + y;
  auto place = [](int site) {  // tile_elem in 32 bits (see tile_step)
    return (uint32_t)site + __umul24((uint32_t)site >> 6, 64u * (Q - 1));
  };
  uint32_t sw = 1u << 31;
  double n[Q];
  double rho = 0.0, mom[D] = {};
  const bool bdist2 = p.eq_form == kBDist2;
  if (needed) {
    sw = SOLID ? nbw[s] : 0u;
    double v;
    if (sw >> 31) {
      v = S[f * g.sp + s];
    } else {
      const NbrOffsets o = nbr_offsets(g, x, y, 0);
      const double *__restrict__ Af = A + f * (Q * g.sp);
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int src = nbr_site(s, o, -L::c[i][0], -L::c[i][1], 0);
        const int b = L::bounce[i], lo = SOLID && b < i ? b : i;
        const bool bb = SOLID && ((sw >> b) & 1u);
        n[i] = at<true>(Af + 64 * lo, 64 * ((bb ? b : i) - lo) + place(bb ? s : src));
      }
      rho = density<L>(n);
      v = psi_of(p.psi_form, rho);
    }
    psi[f][cell] = v;
  }
  if (inside) {
    if (bdist2 && !(sw >> 31)) first_moment<L>(n, mom);
    xch[f][0][k] = rho;
#pragma unroll
    for (int d = 0; d < D; ++d) xch[f][1 + d][k] = mom[d];
  }
  __syncthreads();
  if (!inside || (sw >> 31)) return;  // solid populations stay as they are
  auto at_nbr = [&](int ff, int i) {
    return psi[ff][i < 0 ? cell : cell + L::c[i][0] * kTileEY + L::c[i][1]];
  };
  double F[D];
  sc_force<L, C>(
      f, F, p, at_nbr, [&](int i) { return SOLID && ((sw >> i) & 1u); }, at_nbr);
  const double total = total_density<C>([&](int ff) { return xch[ff][0][k]; });
  double wv[D];
  if (bdist2)
    weighted_velocity<L, C>([&](int ff, int d) { return xch[ff][1 + d][k]; }, total, p, wv);
  double *__restrict__ Bf = B + f * (Q * g.sp);
  collide_component<L>(f, n, rho, total, F, wv, p,
                       [&](int i, double v) { *elem<true>(Bf + 64 * i, place(s)) = v; });
}

template <int C>
inline void launch_tile_step(const double *A, double *B, const uint32_t *nbw, const double *S,
                             const Geo &g, const StepParams &p, hipStream_t stream) {
  const int tx = (g.nx + kTileX - 1) / kTileX, ty = (g.ny + kTileY - 1) / kTileY;
  const dim3 grid(tx * ty), block(2 * C * 64);
  if (p.has_solid)
    hipLaunchKernelGGL((k_tile_step<C, true>), grid, block, 0, stream, A, B, nbw, S, g, p, ty);
  else
    hipLaunchKernelGGL((k_tile_step<C, false>), grid, block, 0, stream, A, B, nbw, S, g, p, ty);
}

}  // namespace dlbc
