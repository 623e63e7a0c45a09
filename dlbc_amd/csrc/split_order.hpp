// split_order.hpp -- the order of the workgroups of a one-launch Shan-Chen
// step (kernels_split.hpp), made on the host.
//
// Every block of SB consecutive sites is visited twice: by a psi workgroup and
// later by a collide workgroup, which reads the psi of its neighbour sites.
// The order keeps the two visits close, so that the second pull of the
// populations finds what the first one left in the memory-side cache (256 MB),
// and far enough apart that a collide workgroup does not wait: psi is
// `kOrderAhead` blocks ahead of where the next collide workgroup needs it.
//
// A large plane is cut into strips of rows, and a strip is marched along x
// before the next one: the distance between the two visits is then about one
// plane of the strip, whatever the size of the lattice.  The psi strips lie a
// few rows ahead of the collide strips (the first also holds the last row, its
// periodic neighbour), so that every psi is computed once.
//
// The order is one of speed alone: a collide wave checks the flags of the
// blocks that it reads (split_needs) and can compute them itself.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "kernels_twopass.hpp"

namespace dlbc {

// Blocks of a strip's plane, blocks that psi is ahead, and turns of psi in a
// row.  FP64, 256^3 without solids, us per step.  Psi and collide turns one by
// one 2440, psi in rows of eight turns 2385 (one by one, workgroups that did
// nothing at all in the psi turns' place slowed the collide workgroups by a
// quarter).  With the spans below: strips of 128, 192 and 256 blocks 2254, 2285
// and 2254 (a whole plane, before them: 2610 against 2385); psi 896, 1024 and
// 1280 blocks ahead 2250, 2254 and 2265, at 128^3 in FP32 163, 151 and 148 (some
// 1280 workgroups are resident: closer, and collide workgroups wait).
// A FP16 block has half the bytes, and strips of twice the blocks lose less at
// their edges: 384^3 without solids 2405 us with 128, 2335 with 256, 2700 with 512.
constexpr int kOrderStrip = 128, kOrderStripF16 = 256, kOrderAhead = 1024, kOrderRow = 8;

// A turn: what eight consecutive workgroups do (workgroup b runs on XCD b % 8, so
// every XCD gets both kinds in equal parts).  Workgroup j < turn_count takes
// block turn_first + j * turn_stride, the others nothing.  Where 8 kOrderSpan
// consecutive blocks stand in a row, kOrderSpan turns give each XCD kOrderSpan
// of them, so that the psi rows that neighbouring blocks share are in its L2:
// FP64 256^3 2435 us with turns of consecutive blocks, 2285 with spans of 4,
// 2274 with 8, 2286 with 16; 190x151x117 with solids FP64 569, 536, 535 and 530,
// FP32 278, 264, 251 and 261.
constexpr int kOrderSpan = 8;
constexpr int32_t order_turn(int first, int count, bool spread, bool collide) {
  return first << 6 | count << 2 | (spread ? 2 : 0) | (collide ? 1 : 0);
}
__host__ __device__ inline int turn_first(int32_t t) { return t >> 6; }
__host__ __device__ inline int turn_count(int32_t t) { return t >> 2 & 15; }
__host__ __device__ inline int turn_stride(int32_t t) { return (t & 2) ? kOrderSpan : 1; }
__host__ __device__ inline bool turn_collide(int32_t t) { return t & 1; }

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

// Whether a lattice is served by this order: a collide wave looks at the flags of
// every block in split_needs, and the psi of all of them stands in front of it.
// Both are few where a block meets no more than two planes (planes of a block's
// sites or more; a block over more planes would wait for the whole lattice) and
// rows are not too long, of which a collide waits for nine whole ones.  us per
// step of large lattices, two launches / one: FP64 rows of 16, 64, 128, 192 and
// 512 blocks 316 / 279, 311 / 277, 304 / 292, 308 / 320 and 2936 / 3128; FP32 rows
// of 64, 128, 192 and 512 blocks 756 / 644, 749 / 666, 768 / 751 and 366 / 390, and
// of 192 in a smaller lattice 175 / 192; FP16 rows of 64 and 128 blocks 400 / 393
// and 399 / 409.  A lattice of no more than kOrderAll blocks (a member of a batch)
// has no more to wait for than such rows.  (Components of whole tiles of 64 sites:
// no line of psi holds sites of two waves.)
constexpr int kOrderAll = 256, kOrderRowMost = 128, kOrderRowMostF16 = 64;
inline bool split_order_serves(const Geo &g, int SB, int row_most = kOrderRowMost) {
  if (g.sp % 64 != 0) return false;
  return g.sites <= (int64_t)kOrderAll * SB ||
         ((int64_t)g.ny * g.nz >= SB && g.nz <= (int64_t)row_most * SB);
}

// The psi blocks and the collide blocks of a lattice in the order of their
// visits, numbered from blk0, appended to psi and col; need: for every collide
// the psi places it wants in front of it, counted in the whole of psi.
inline void split_order_lists(const Geo &g, int SB, int blk0, std::vector<int32_t> &psi,
                              std::vector<int32_t> &col, std::vector<int32_t> &need,
                              int strip = kOrderStrip) {
  const int nb = (g.sites + SB - 1) / SB;
  const int64_t plane = (int64_t)g.ny * g.nz;
  const size_t psi0 = psi.size(), col0 = col.size();
  // first block that starts at or after site s
  auto first = [&](int64_t s) {
    return (int)std::min<int64_t>(nb, (std::max<int64_t>(s, 0) + SB - 1) / SB);
  };
  const int64_t wrap0 = plane - g.nz - SB + 1;  // blocks from here hold a plane's last row
  const int64_t pb = (plane + SB - 1) / SB;     // blocks of a plane
  int ns = (int)std::max<int64_t>(1, (pb + strip / 2) / strip);
  ns = std::min(ns, std::max(1, g.ny / 4));
  const int H = (g.ny + ns - 1) / ns;  // rows of a strip
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
    // the psi strip's part of a plane; the first strip also takes the plane's end
    const int64_t p0 = j == 0 ? 0 : edge(y0);
    const int64_t p1 = !last ? edge(y1) : (j == 0 ? plane : wrap0);
    if (into >= 0 && ((into_at >= p0 && into_at < p1) || (wraps && into_at >= wrap0)))
      psi.push_back(blk0 + into);
    auto put = [&](int lo, int hi) {
      for (int b = lo; b < hi; ++b)
        if (b != into) psi.push_back(blk0 + b);
    };
    for (int k = 0; k < g.nx; ++k) {  // from the last plane, which plane 0 reads
      const int64_t base = (k == 0 ? g.nx - 1 : k - 1) * plane;
      put(first(base + p0), first(base + p1));
      if (wraps) put(std::max(first(base + p1), first(base + wrap0)), first(base + plane));
    }
    for (int x = 0; x < g.nx; ++x) {
      const int64_t base = x * plane;
      for (int b = first(base + (int64_t)y0 * g.nz);
           b < first(base + (last ? plane : (int64_t)y1 * g.nz)); ++b)
        col.push_back(blk0 + b);
    }
  }
  std::vector<int32_t> place(nb);
  for (int k = 0; k < nb; ++k) place[psi[psi0 + k] - blk0] = k;
  for (size_t c = col0; c < col.size(); ++c) {
    int n = 0;
    for (int k = 0; k < 8; ++k) {
      int lo, hi;
      split_needs(g, SB, col[c] - blk0, k, lo, hi);
      if (lo > hi) continue;
      // places rise with the block but for the blocks taken early: those of a
      // plane's end and the one that runs into the last plane
      const bool all = lo == 0 && hi == nb - 1, end = (int64_t)hi * SB % plane >= wrap0;
      if (all) n = nb;
      for (int v = all ? hi + 1 : (end ? lo : std::max(lo, hi - 1)); v <= hi; ++v)
        n = std::max(n, place[v] + 1);
    }
    need.push_back((int32_t)psi0 + n);
  }
}

// The turns of a launch over these lists: runs of consecutive blocks, psi in
// front of every collide by `ahead` blocks.  With several lattices (`starts`:
// their first blocks) no turn crosses from one to the next.
inline std::vector<int32_t> split_order_merge(const std::vector<int32_t> &psi,
                                              const std::vector<int32_t> &col,
                                              const std::vector<int32_t> &need,
                                              int ahead = kOrderAhead,
                                              const std::vector<int> &starts = {}) {
  std::vector<int32_t> out;
  out.reserve((psi.size() + col.size()) / 8 + (psi.size() + col.size()) / 64 + 32);
  // consecutive blocks from place p on, at most `most`
  auto run = [&](const std::vector<int32_t> &v, size_t p, int most) {
    const auto next = std::upper_bound(starts.begin(), starts.end(), v[p]);
    const int64_t end = next == starts.end() ? INT32_MAX : *next;
    int n = 1;
    while (n < most && p + n < v.size() && v[p + n] == v[p] + n && v[p] + n < end) ++n;
    return n;
  };
  // the turns of the next run of v, which is returned; need of a turn before it
  size_t pp = 0;
  auto put = [&](const std::vector<int32_t> &v, size_t p, bool collide, auto before) {
    constexpr int whole = 8 * kOrderSpan;
    if (kOrderSpan > 1 && run(v, p, whole) == whole) {
      for (int k = 0; k < kOrderSpan; ++k) {
        before(p, whole);
        out.push_back(order_turn(v[p] + k, 8, true, collide));
      }
      return whole;
    }
    const int n = run(v, p, 8);
    before(p, n);
    out.push_back(order_turn(v[p], n, false, collide));
    return n;
  };
  auto nothing = [](size_t, int) {};
  for (size_t cp = 0; cp < col.size();)
    cp += put(col, cp, true, [&](size_t p, int c) {
      int n = 0;
      for (int k = 0; k < c; ++k) n = std::max(n, need[p + k]);
      const bool due = pp < (size_t)n + ahead;
      while (due && pp < psi.size() && pp < (size_t)n + ahead + 8 * (kOrderRow - 1))
        pp += put(psi, pp, false, nothing);
    });
  while (pp < psi.size()) pp += put(psi, pp, false, nothing);
  return out;
}

// The order of one lattice.
inline std::vector<int32_t> split_order(const Geo &g, int SB, int strip = kOrderStrip,
                                        int ahead = kOrderAhead) {
  std::vector<int32_t> psi, col, need;
  split_order_lists(g, SB, 0, psi, col, need, strip);
  return split_order_merge(psi, col, need, ahead);
}

// What is wrong with an order: blocks that are not visited once by each kind,
// neighbours outside split_needs, and psi that stands behind a collide that
// needs it.  0 for a good one.
inline int64_t split_order_faults(const Geo &g, int SB, const std::vector<int32_t> &o) {
  const int nb = (g.sites + SB - 1) / SB, plane = g.ny * g.nz;
  std::vector<int64_t> at[2];
  at[0].assign(nb, -1);
  at[1].assign(nb, -1);
  int64_t bad = 0;
  for (size_t p = 0; p < o.size(); ++p)
    for (int j = 0; j < turn_count(o[p]); ++j) {
      const int b = turn_first(o[p]) + j * turn_stride(o[p]), k = turn_collide(o[p]) ? 1 : 0;
      if (b < 0 || b >= nb || turn_count(o[p]) > 8 || at[k][b] != -1) {
        ++bad;
        continue;
      }
      at[k][b] = (int64_t)p;
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
