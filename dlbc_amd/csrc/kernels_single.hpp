// kernels_single.hpp -- one step of a single-component lattice without
// Shan-Chen force (FP64, any connectivity): streaming, bounce-back, body force
// and BGK collision in one launch.
//
// The step reads and writes each population once.  One lane per site: its
// neighbours' places come from six offsets set up once (nbr_offsets), the solid
// neighbourhood from one word, and every access takes a scalar base and a 32-bit
// lane offset.  (The general kernel, k_collide, wraps and multiplies every
// neighbour's coordinates and reads its mask byte.)  us per step, k_collide /
// here: D2Q9 64^2 4.6 / 3.4, 700^2 with plates 16.6 / 14.5; D3Q19 32^3 6.8 / 5.3,
// 70x45x98 with plates 23.3 / 18.8, 256^3 940 / 873 (5.8 TB/s, a plain copy 5.7),
// 256^3 with solid spheres 1307 / 858 (solid lanes write their lines whole).
//
// Per-site arithmetic is the shared code of the other schedules.
#pragma once

#include "kernels_split.hpp"

namespace dlbc {

// Threads of a workgroup: one wave, so that small lattices reach every CU.
constexpr int kSingleThreads = 64;

// Nontemporal stores where the two buffers exceed the memory-side cache by some
// (us per step, without / with): D3Q19 96^3 (257 MiB) 45.1 / 47.6, 100^3 (290 MiB)
// 53.9 / 53.8, 112^3 78 / 74, 256^3 906 / 873; D2Q9 1300^2 (232 MiB) 40.6 / 42.5,
// 1400^2 (269 MiB) 49.2 / 49.0, 1600^2 66 / 63; 70x45x98 18.8 / 21.0.
constexpr int64_t kSingleCached = 288ll << 20;

// Whether the kernel serves a lattice: neighbours one site away on every axis
// (not D1Q5), and 32-bit byte offsets.
inline bool single_supported(const Geo &g, int q) {
  return q != 5 && (int64_t)q * 8 * g.sp < (int64_t)1 << 32;
}

template <class L, bool SOLID, bool NT>
__global__ void __launch_bounds__(kSingleThreads)
    k_single(const double *__restrict__ A, double *__restrict__ B,
             const uint32_t *__restrict__ nbw, Geo g, StepParams p) {
  constexpr int Q = L::q, D = L::d;
  const int s = blockIdx.x * kSingleThreads + threadIdx.x;
  if (s >= g.sites) return;
  // a solid site's lane stores the site's own populations again, so that whole
  // cache lines are written; a line of solid sites only is left alone (as in
  // k_split_collide)
  uint32_t sw = SOLID ? nbw[s] : 0u;
  const bool solid_site = sw >> 31;
  if (SOLID && line_all_solid<16>(solid_site)) return;
  if (solid_site) sw = (1u << Q) - 1u;
  int x, y, z;
  lane_coords(s, g, x, y, z);
  const NbrOffsets o = nbr_offsets(g, x, y, z);
  auto place = [](int site) {  // tile_elem<Q> in 32 bits
    return (uint32_t)site + __umul24((uint32_t)site >> 6, 64u * (Q - 1));
  };
  double n[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const int src = nbr_site(s, o, -L::c[i][0], -L::c[i][1], -L::c[i][2]);
    const int b = L::bounce[i], lo = SOLID && b < i ? b : i;
    const bool bb = SOLID && ((sw >> b) & 1u);
    n[i] = at<true>(A + 64 * lo, 64 * ((bb ? b : i) - lo) + place(bb ? s : src));
  }
  const double rho = density<L>(n);
  double F[D], wv[D];
#pragma unroll
  for (int d = 0; d < D; ++d) F[d] = 0.0;
  const double total = total_density<1>([&](int) { return rho; });
  if (p.eq_form == kBDist2) {
    double mom[D];
    first_moment<L>(n, mom);
    weighted_velocity<L, 1>([&](int, int d) { return mom[d]; }, total, p, wv);
  }
  auto out = [&](int i, double v) {
    double *to = elem<true>(B + 64 * i, place(s));
    const double w = SOLID && solid_site ? n[L::bounce[i]] : v;
    if (NT)
      __builtin_nontemporal_store(w, to);
    else
      *to = w;
  };
  if constexpr (Q == 19)
    collide_d3q19_streamed(0, n, rho, total, F, wv, p, out);
  else
    collide_component<L>(0, n, rho, total, F, wv, p, out);
}

template <class L>
inline void launch_single(const double *A, double *B, const uint32_t *nbw, const Geo &g,
                          const StepParams &p, hipStream_t stream) {
  const dim3 grid((g.sites + kSingleThreads - 1) / kSingleThreads), block(kSingleThreads);
  const bool nt = 2 * 8 * L::q * g.sp > kSingleCached;
  if (p.has_solid && nt)
    hipLaunchKernelGGL((k_single<L, true, true>), grid, block, 0, stream, A, B, nbw, g, p);
  else if (p.has_solid)
    hipLaunchKernelGGL((k_single<L, true, false>), grid, block, 0, stream, A, B, nbw, g, p);
  else if (nt)
    hipLaunchKernelGGL((k_single<L, false, true>), grid, block, 0, stream, A, B, nbw, g, p);
  else
    hipLaunchKernelGGL((k_single<L, false, false>), grid, block, 0, stream, A, B, nbw, g, p);
}

// ---- several steps of a small D2Q9 lattice in one launch --------------------------
// A step of a lattice of some 10^4 sites takes 3 us, of which the launch and one
// trip to memory are nearly all.  A workgroup holds 24 x 24 sites in LDS, the
// T = (24 - TILE) / 2 sites around its TILE x TILE tile among them, and takes T
// steps: after step t the sites up to T - t from the tile are right, and in the
// end the tile, which it writes.  The border is computed by the neighbours too:
// 3.8 times the work at TILE = 8 (T = 8), 1.4 times at TILE = 16 (T = 4).  What
// bounds it then is the chain of a site's arithmetic and the two barriers of a
// step, 1.3 us: 64^2 went from 3.4 us a step (2.9 from a graph) to 1.85.
constexpr int kMultiR = 24;

template <int TILE>
constexpr int multi_steps() {
  return (kMultiR - TILE) / 2;
}

template <int TILE, bool SOLID>
__global__ void __launch_bounds__(kMultiR *kMultiR)
    k_single_multi(const double *__restrict__ A, double *__restrict__ B,
                   const uint32_t *__restrict__ nbw, Geo g, StepParams p, int tiles_y) {
  using L = D2Q9;
  constexpr int Q = L::q, D = L::d, T = multi_steps<TILE>(), R = kMultiR;
  __shared__ double pop[Q][R * R];
  const int t = threadIdx.x, rx = t / R, ry = t % R;
  // the lane's site: its cell's place on the periodic lattice
  const int tx = (int)(blockIdx.x / tiles_y) * TILE + rx - T;
  const int ty = (int)(blockIdx.x % tiles_y) * TILE + ry - T;
  int x = tx % g.nx, y = ty % g.ny;
  if (x < 0) x += g.nx;
  if (y < 0) y += g.ny;
  const int s = x * g.ny + y;
  const int64_t place = tile_elem<Q>(s);
  const uint32_t sw = SOLID ? nbw[s] : 0u;
  double n[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    n[i] = A[64 * i + place];
    pop[i][t] = n[i];
  }
  // cells from the border of the region
  const int edge = min(min(rx, R - 1 - rx), min(ry, R - 1 - ry));
#pragma unroll 1
  for (int step = 1; step <= T; ++step) {
    __syncthreads();
    // (a solid site keeps its populations)
    const bool live = edge >= step && !(sw >> 31);
    if (live) {
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const bool bb = SOLID && ((sw >> L::bounce[i]) & 1u);
        n[i] = bb ? pop[L::bounce[i]][t] : pop[i][t - L::c[i][0] * R - L::c[i][1]];
      }
    }
    __syncthreads();
    if (live) {
      const double rho = density<L>(n);
      double F[D], wv[D];
#pragma unroll
      for (int d = 0; d < D; ++d) F[d] = 0.0;
      const double total = total_density<1>([&](int) { return rho; });
      if (p.eq_form == kBDist2) {
        double mom[D];
        first_moment<L>(n, mom);
        weighted_velocity<L, 1>([&](int, int d) { return mom[d]; }, total, p, wv);
      }
      collide_component<L>(0, n, rho, total, F, wv, p, [&](int i, double v) { pop[i][t] = v; });
    }
  }
  // (every lane reads back what it wrote itself)
  const bool mine = edge >= T && tx >= 0 && ty >= 0 && tx < g.nx && ty < g.ny && !(sw >> 31);
  if (!mine) return;
#pragma unroll
  for (int i = 0; i < Q; ++i) B[64 * i + place] = pop[i][t];
}

template <int TILE>
inline void launch_single_multi(const double *A, double *B, const uint32_t *nbw, const Geo &g,
                                const StepParams &p, hipStream_t stream) {
  const int tx = (g.nx + TILE - 1) / TILE, ty = (g.ny + TILE - 1) / TILE;
  const dim3 grid(tx * ty), block(kMultiR * kMultiR);
  if (p.has_solid)
    hipLaunchKernelGGL((k_single_multi<TILE, true>), grid, block, 0, stream, A, B, nbw, g, p, ty);
  else
    hipLaunchKernelGGL((k_single_multi<TILE, false>), grid, block, 0, stream, A, B, nbw, g, p, ty);
}

}  // namespace dlbc
