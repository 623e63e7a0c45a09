// split_order.hpp -- the order of the workgroups of a one-launch Shan-Chen
// step (kernels_split.hpp), made on the host.
//
// Every block of SB consecutive sites is visited twice: by a psi workgroup and
// later by a collide workgroup, which reads the psi of its neighbour sites.
// The order keeps the two visits close, so that the second pull of the
// populations finds what the first one left in the memory-side cache (256 MB),
// and far enough apart that a collide workgroup does not wait: a psi workgroup
// is `kOrderAhead` blocks ahead of where the next collide workgroup needs it.
//
// A large plane is cut into strips of rows, and a strip is marched along x
// before the next one: the distance between the two visits is then about one
// plane of the strip, whatever the size of the lattice.  The psi strips lie a
// few rows ahead of the collide strips (the first also holds the last row, its
// periodic neighbour), so that every psi is computed once.
//
// The order is one of speed alone: a collide workgroup checks the blocks that
// it reads (split_needs) and could compute them itself.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "kernels_twopass.hpp"

namespace dlbc {

// Blocks of a strip's plane, and blocks that psi is ahead.
constexpr int kOrderStrip = 128, kOrderAhead = 768;

constexpr int32_t kOrderNone = -1;  // an empty place (turns of eight workgroups stay whole)

// The blocks whose psi a collide of block blk reads, as intervals [lo, hi] of
// blocks (empty where lo > hi): number k of eight.  Planes xa - 1 .. xb + 1
// around the block's (k >> 1), and of each the rows next to the block's (k even)
// and the rows it meets across the periodic end of y (k odd).  A block of more
// than two planes needs every block.
__host__ __device__ inline void split_needs(const Geo &g, int SB, int blk, int k, int &lo, int &hi) {
  const int plane = g.ny * g.nz, last = g.sites - 1;
  const int s0 = blk * SB, s1 = s0 + SB - 1 < last ? s0 + SB - 1 : last;
  const int xa = geo_div(s0, g.div_yz_m, g.div_yz_l), xb = geo_div(s1, g.div_yz_m, g.div_yz_l);
  lo = 0;
  hi = -1;
  if (xb > xa + 1) {
    if (k == 0) hi = last / SB;
    return;
  }
  const int dp = (k >> 1) - 1;  // planes xa - 1, xa, xa + 1 and, for two planes, xa + 2
  if (dp > xb - xa + 1) return;
  int x = xa + dp;
  x = x < 0 ? x + g.nx : (x >= g.nx ? x - g.nx : x);
  const int ya = geo_div(s0 - xa * plane, g.div_z_m, g.div_z_l);
  const int yb = geo_div(s1 - xb * plane, g.div_z_m, g.div_z_l);
  int r0, r1;  // rows
  if (xa == xb) {
    if (!(k & 1)) {
      r0 = ya > 0 ? ya - 1 : 0;
      r1 = yb < g.ny - 1 ? yb + 1 : yb;
    } else if (ya == 0 && yb < g.ny - 1) {
      r0 = r1 = g.ny - 1;
    } else if (yb == g.ny - 1 && ya > 0) {
      r0 = r1 = 0;
    } else {
      return;
    }
  } else if (!(k & 1)) {  // the end of plane xa
    r0 = ya > 0 ? ya - 1 : 0;
    r1 = g.ny - 1;
  } else {  // the start of plane xb
    r0 = 0;
    r1 = yb < g.ny - 1 ? yb + 1 : yb;
  }
  lo = (x * plane + r0 * g.nz) / SB;
  hi = (x * plane + r1 * g.nz + g.nz - 1) / SB;
}

// The places of a launch: 2 blk for the psi of block blk, 2 blk + 1 for its
// collide, kOrderNone for nothing.  Workgroup b runs on XCD b % 8; each turn of
// eight is of one kind, so that every XCD gets both in equal parts.  chunk > 0
// (a caller's choice): all psi first, and turns of `chunk` consecutive blocks for
// each XCD.
inline std::vector<int32_t> split_order(const Geo &g, int SB, int chunk,
                                        int strip = kOrderStrip, int ahead = kOrderAhead) {
  const int nb = (g.sites + SB - 1) / SB;
  const int64_t plane = (int64_t)g.ny * g.nz;
  std::vector<int32_t> psi, col, out;
  psi.reserve(nb);
  col.reserve(nb);
  // first block that starts at or after site s
  auto first = [&](int64_t s) {
    return (int)std::min<int64_t>(nb, (std::max<int64_t>(s, 0) + SB - 1) / SB);
  };
  const int64_t wrap0 = plane - g.nz - SB + 1;  // blocks from here hold a plane's last row
  if (chunk > 0) {
    const int main = nb / (8 * chunk) * (8 * chunk);
    for (int b = 0; b < nb; ++b) {
      const int j = b >> 3;
      psi.push_back(b >= main ? b : ((j / chunk) * 8 + (b & 7)) * chunk + j % chunk);
    }
    col = psi;
  } else {
    const int64_t pb = (plane + SB - 1) / SB;  // blocks of a plane
    int ns = (int)std::max<int64_t>(1, (pb + strip / 2) / strip);
    ns = std::min(ns, std::max(1, g.ny / 4));
    const int H = (g.ny + ns - 1) / ns;
    ns = (g.ny + H - 1) / H;
    const int e = (SB + g.nz - 1) / g.nz + 1;  // rows that psi strips lie ahead
    // the block that runs into the last plane, which the first collides read
    const int64_t s_last = (int64_t)(g.nx - 1) * plane;
    const int into = s_last % SB ? (int)(s_last / SB) : -1;
    const int64_t into_at = into >= 0 ? (int64_t)into * SB % plane : 0;
    for (int j = 0; j < ns; ++j) {
      const bool last = j == ns - 1, wraps = j == 0 && !last;
      const int y0 = j * H, y1 = last ? g.ny : (j + 1) * H;
      auto edge = [&](int y) { return std::min<int64_t>((int64_t)(y + e) * g.nz, wrap0); };
      const int64_t p0 = j == 0 ? 0 : edge(y0), p1 = j == 0 && last ? plane
                                                     : last         ? wrap0
                                                                    : edge(y1);
      if (into >= 0 && ((into_at >= p0 && into_at < p1) || (wraps && into_at >= wrap0)))
        psi.push_back(into);
      auto put = [&](int lo, int hi) {
        for (int b = lo; b < hi; ++b)
          if (b != into) psi.push_back(b);
      };
      for (int k = 0; k < g.nx; ++k) {
        const int64_t base = (k == 0 ? g.nx - 1 : k - 1) * plane;
        put(first(base + p0), first(base + p1));
        if (wraps) put(std::max(first(base + p1), first(base + wrap0)), first(base + plane));
      }
      for (int x = 0; x < g.nx; ++x) {
        const int64_t base = x * plane;
        for (int b = first(base + (int64_t)y0 * g.nz);
             b < first(base + (last ? plane : (int64_t)y1 * g.nz)); ++b)
          col.push_back(b);
      }
    }
  }
  // the psi places that a block's collide needs in front of it
  std::vector<int32_t> place(nb);
  for (int k = 0; k < nb; ++k) place[psi[k]] = k;
  auto need = [&](int blk) {
    if (chunk > 0) return nb;
    int n = 0;
    for (int k = 0; k < 8; ++k) {
      int lo, hi;
      split_needs(g, SB, blk, k, lo, hi);
      if (lo > hi) continue;
      if (k == 0 && hi == nb - 1 && lo == 0) return nb;
      // places rise with the block but for the blocks taken early: those of a
      // plane's end and the one that runs into the last plane
      const bool end = (int64_t)hi * SB % plane >= wrap0;
      for (int v = end ? lo : std::max(lo, hi - 1); v <= hi; ++v) n = std::max(n, place[v] + 1);
    }
    return n;
  };
  // psi in front of every collide place by `ahead`, in turns of eight
  size_t pp = 0, cp = 0;
  auto turn = [&](const std::vector<int32_t> &v, size_t &p, int kind) {
    for (int k = 0; k < 8; ++k, ++p) out.push_back(p < v.size() ? 2 * v[p] + kind : kOrderNone);
  };
  out.reserve(2 * (size_t)nb + 32);
  while (cp < col.size()) {
    int n = 0;
    for (size_t k = cp; k < std::min(cp + 8, col.size()); ++k) n = std::max(n, need(col[k]));
    while (pp < psi.size() && pp < (size_t)n + ahead) turn(psi, pp, 0);
    turn(col, cp, 1);
  }
  while (pp < psi.size()) turn(psi, pp, 0);
  return out;
}

// What is wrong with an order: blocks that are not visited once by each kind,
// neighbours outside split_needs, and psi that stands behind a collide that
// needs it.  0 for a good one.
inline int64_t split_order_faults(const Geo &g, int SB, const std::vector<int32_t> &o) {
  const int nb = (g.sites + SB - 1) / SB, plane = g.ny * g.nz;
  std::vector<int64_t> at[2];
  at[0].assign(nb, -1);
  at[1].assign(nb, -1);
  int64_t bad = o.size() % 8 != 0;
  for (size_t p = 0; p < o.size(); ++p) {
    if (o[p] == kOrderNone) continue;
    if (o[p] < 0 || o[p] >= 2 * nb || at[o[p] & 1][o[p] >> 1] != -1) {
      ++bad;
      continue;
    }
    at[o[p] & 1][o[p] >> 1] = (int64_t)p;
  }
  for (int b = 0; b < nb; ++b) {
    if (at[0][b] < 0 || at[1][b] < 0) {
      ++bad;
      continue;
    }
    int lo[8], hi[8];
    for (int k = 0; k < 8; ++k) {
      split_needs(g, SB, b, k, lo[k], hi[k]);
      if (lo[k] <= hi[k] && (lo[k] < 0 || hi[k] >= nb)) ++bad;
      for (int v = std::max(lo[k], 0); v <= std::min(hi[k], nb - 1); ++v)
        if (at[0][v] > at[1][b]) ++bad;
    }
    for (int s = b * SB; s < std::min(g.sites, (b + 1) * SB); ++s) {
      const int x = s / plane, y = s % plane / g.nz, z = s % g.nz;
      for (int i = 0; i < 19; ++i) {
        const int v = (((x + D3Q19::c[i][0] + g.nx) % g.nx * g.ny +
                        (y + D3Q19::c[i][1] + g.ny) % g.ny) * g.nz +
                       (z + D3Q19::c[i][2] + g.nz) % g.nz) / SB;
        bool in = false;
        for (int k = 0; k < 8; ++k) in |= v >= lo[k] && v <= hi[k];
        if (!in) ++bad;
      }
    }
  }
  return bad;
}

}  // namespace dlbc
