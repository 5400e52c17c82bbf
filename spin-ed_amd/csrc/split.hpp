// split.hpp -- row gather of exchange bonds in a symmetry-free weight sector
// by halves of the state (combinatorial-rank bases: no permutation but the
// identity, with or without the spin flip).
//
// The representatives are the weight-w states in ascending order (with the
// flip, those with site n-1 down), so the states that share their high sites
// l .. n-1 form one contiguous group of rows, ordered by their low sites.
// For all rows of a group (high part hi, lows of weight k = w - |hi|):
//   * a bond inside the high part is active for every row or none, and its
//     targets are the same rows of another group: a coalesced read;
//   * a bond inside the low part stays in the group: its targets come from
//     the group's x in LDS, through a rank table of the low states;
//   * a bond across the cut leads to one other group, rank by table.
// A move into the top site of a flip sector leads to the complement, whose
// low states run backwards.  Nothing is searched and no entry is stored:
// against the gather cache (4 bytes and one scattered read per term) the
// matvec reads each group a few times in whole lines.
// The terms of a row are added in bond order with the fma of
// gather_row_real, so the sums are the same bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include "rowgather.hpp"

namespace spined {

constexpr int kSplitMaxLow = 13;   // rank table of 16 KB, groups of at most 1716 rows
constexpr int kSplitMaxHigh = 17;  // group table of at most 512 KB
constexpr int kSplitMaxBonds = 64;

struct SplitArgs {
  const uint32_t *__restrict__ goff;      // first row of each group, nhi + 1
  const uint16_t *__restrict__ lowstate;  // low states by weight, ascending
  const uint16_t *__restrict__ lowrank;   // rank of a low state in its weight
  const uint32_t *__restrict__ lowoff;    // start of each weight in lowstate
  uint32_t nhi;                           // groups (empty ones included)
  int32_t l, n, w;
  int32_t flip;                           // spin inversion in the group
  int32_t neg;                            // its sector is odd
};

// The bonds of a group, one per lane (lane j: bond j), so that every value
// of a bond is one v_readlane away: held in LDS instead, reading the bonds
// back took longer than the rows' own reads.
enum : uint32_t { kSplitLow = 0, kSplitSame = 1, kSplitBack = 2, kSplitCross = 3 };
struct SplitBonds {
  double c, da, dp;
  uint32_t base; // first row of the target group
  uint32_t info; // type | a << 2 | b << 8 (site, or bit of hi for a bond across) | complement << 14
  uint64_t on;   // bonds with off-diagonal terms in this group (uniform)
  uint64_t rest; // bonds beyond the leading low ones (uniform): split_diag
};

__device__ inline uint32_t lane_u32(uint32_t v, int j) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), j));
}
__device__ inline double lane_f64(double v, int j) {
  union {
    double d;
    int i[2];
  } u;
  u.d = v;
  u.i[0] = __builtin_amdgcn_readlane(u.i[0], j);
  u.i[1] = __builtin_amdgcn_readlane(u.i[1], j);
  return u.d;
}

// What a lane keeps of its bond from group to group.
struct SplitBond {
  double o, da, dp;
  uint32_t sites;
  bool have;
};
__device__ inline SplitBond split_bond(const BondArgs &bd, int lane) {
  SplitBond b{0.0, 0.0, 0.0, 0, lane < bd.nbonds};
  if (b.have) {
    b.sites = bd.sites[lane];
    b.o = bd.o[lane];
    b.da = bd.da[lane];
    b.dp = bd.dp[lane];
  }
  return b;
}

// Bonds of the group hi (by a whole wave).
__device__ inline SplitBonds split_bonds(const SplitArgs &s, const SplitBond &in, uint32_t hi) {
  SplitBonds r{in.o, in.da, in.dp, 0, 0, 0, 0};
  bool on = false, high = false;
  const bool have = in.have;
  if (have) {
    const uint32_t st = in.sites;
    const int s0 = static_cast<int>(st & 0xffu), s1 = static_cast<int>(st >> 8);
    const int a = s0 < s1 ? s0 : s1, b = s0 < s1 ? s1 : s0;
    const int l = s.l;
    on = r.c != 0.0 && a != b;
    high = b >= l;
    uint32_t to = hi, type = kSplitLow, ia = a, ib = b;
    if (a >= l) {
      type = kSplitSame;
      ib = ((hi >> (a - l)) ^ (hi >> (b - l))) & 1u; // active for all rows or none
      on = on && ib;
      ia = 0;
      to = hi ^ (1u << (a - l)) ^ (1u << (b - l));
    } else if (high) {
      type = kSplitCross;
      ib = (hi >> (b - l)) & 1u;
      to = hi ^ (1u << (b - l));
    }
    uint32_t comp = 0;
    if (s.flip && ((to >> (s.n - 1 - l)) & 1u)) {
      // into the top site: the complement is the representative
      to = ~to & ((1u << (s.n - l)) - 1u);
      if (type == kSplitSame) type = kSplitBack;
      comp = 1;
      if (s.neg) r.c = -r.c;
    }
    r.info = type | ia << 2 | ib << 8 | comp << 14;
    if (on) r.base = s.goff[to];
  }
  r.on = __ballot(on);
  const uint64_t all = __ballot(have);
  const uint64_t upper = __ballot(have && high);
  // from the first bond that is not inside the low part (also the end of
  // split_dlow's sums)
  r.rest = upper ? all & ~((1ull << __builtin_ctzll(upper)) - 1) : 0;
  return r;
}

// Diagonal partial sums of the low states over the leading low bonds:
// dlow[lowoff[k] + rank] (one thread per entry e of 2^l).
__device__ inline double split_dlow(const SplitArgs &s, const BondArgs &bd, uint32_t lo) {
  double d = 0.0;
  for (int t = 0; t < bd.nbonds; ++t) {
    const uint32_t st = bd.sites[t];
    const uint32_t s0 = st & 0xffu, s1 = st >> 8;
    if (static_cast<int>(s0 > s1 ? s0 : s1) >= s.l) break;
    d += (((lo >> s0) ^ (lo >> s1)) & 1u) ? bd.da[t] : bd.dp[t];
  }
  return d;
}

// Diagonals of R rows: d[q] holds the partial sum over the leading low bonds
// (split_dlow); the other bonds follow in order, as row_pass_a sums them.
template <int R>
__device__ inline void split_diag(const SplitBonds &sb, const uint32_t (&lo)[R], double (&d)[R]) {
  uint64_t m = sb.rest;
  while (m) {
    const int j = __builtin_ctzll(m);
    m &= m - 1;
    const uint32_t info = lane_u32(sb.info, j);
    const double da = lane_f64(sb.da, j), dp = lane_f64(sb.dp, j);
    const uint32_t type = info & 3u, a = (info >> 2) & 63u, b = (info >> 8) & 63u;
    if (type == kSplitSame || type == kSplitBack) {
      const double v = b ? da : dp;
#pragma unroll
      for (int q = 0; q < R; ++q) d[q] += v;
    } else {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t other = type == kSplitCross ? b : lo[q] >> b;
        d[q] += (((lo[q] >> a) ^ other) & 1u) ? da : dp;
      }
    }
  }
}

// Off-diagonal sums of R rows of one group (ranks r[q] < cnt, low states
// lo[q]) added to acc[q].  xs: the group's x; rank: the rank table (both in
// LDS).  Four bonds at a time: their reads are in flight together.
template <int R, class XT>
__device__ inline void split_rows(const SplitArgs &s, const SplitBonds &sb, const uint16_t *rank,
                                  const XT *xs, const XT *__restrict__ x, uint32_t cnt,
                                  const uint32_t (&r)[R], const uint32_t (&lo)[R],
                                  double (&acc)[R]) {
  constexpr int U = 4;
  const uint32_t lmask = (1u << s.l) - 1u;
  // the leading low bonds, without a branch on the kind of bond
  uint64_t lead = sb.on & ~sb.rest;
  while (lead) {
    XT v[U][R];
    bool act[U][R];
    double c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // past the last one, bond j stands in with no active row
      const bool have = lead != 0;
      const int j = have ? __builtin_ctzll(lead) : 0;
      lead &= lead - 1;
      c[u] = lane_f64(sb.c, j);
      const uint32_t info = lane_u32(sb.info, j);
      const uint32_t sa = (info >> 2) & 63u, sc = (info >> 8) & 63u;
      const uint32_t mask = have ? (1u << sa) | (1u << sc) : 0u;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        act[u][q] = have && (((lo[q] >> sa) ^ (lo[q] >> sc)) & 1u);
        v[u][q] = xs[rank[lo[q] ^ mask]];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double t = fma(c[u], static_cast<double>(v[u][q]), acc[q]);
        acc[q] = act[u][q] ? t : acc[q];
      }
  }
  uint64_t m = sb.on & sb.rest;
  while (m) {
    XT v[U][R];
    bool act[U][R];
    double c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      c[u] = 0.0;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        v[u][q] = XT(0);
        act[u][q] = false;
      }
      if (!m) continue;
      const int j = __builtin_ctzll(m);
      m &= m - 1;
      c[u] = lane_f64(sb.c, j);
      const uint32_t info = lane_u32(sb.info, j), base = lane_u32(sb.base, j);
      const uint32_t type = info & 3u, a = (info >> 2) & 63u, b = (info >> 8) & 63u;
      if (type == kSplitLow) {
        const uint32_t mask = (1u << a) | (1u << b);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          act[u][q] = ((lo[q] >> a) ^ (lo[q] >> b)) & 1u;
          v[u][q] = xs[rank[lo[q] ^ mask]];
        }
      } else if (type == kSplitCross) {
        const uint32_t flip = (1u << a) ^ ((info >> 14) & 1u ? lmask : 0u);
#pragma unroll
        for (int q = 0; q < R; ++q) {
          act[u][q] = ((lo[q] >> a) & 1u) != b;
          const uint32_t t = rank[lo[q] ^ flip];
          if (act[u][q]) v[u][q] = x[static_cast<uint64_t>(base) + t];
        }
      } else {
#pragma unroll
        for (int q = 0; q < R; ++q) {
          act[u][q] = true;
          const uint32_t t = type == kSplitSame ? r[q] : cnt - 1 - r[q];
          v[u][q] = x[static_cast<uint64_t>(base) + t];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double t = fma(c[u], static_cast<double>(v[u][q]), acc[q]);
        acc[q] = act[u][q] ? t : acc[q];
      }
  }
}

// R rows of the group hi by each of TB threads: rows r0, r0 + TB, ..., sums
// into y.
template <class XT, class YT, int R, int TB>
__device__ inline void split_group_rows(const SplitArgs &s, const SplitBonds &sb,
                                        const double *__restrict__ dlow, const uint16_t *rank,
                                        const XT *xs, const XT *__restrict__ x,
                                        YT *__restrict__ y, uint32_t g0, uint32_t cnt,
                                        uint32_t low0, uint32_t r0) {
  uint32_t r[R], lo[R];
  double acc[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    // a row past the end repeats the group's last
    r[q] = min(r0 + q * TB, cnt - 1);
    lo[q] = s.lowstate[low0 + r[q]];
    acc[q] = dlow[low0 + r[q]];
  }
  split_diag<R>(sb, lo, acc);
#pragma unroll
  for (int q = 0; q < R; ++q) acc[q] *= static_cast<double>(xs[r[q]]);
  split_rows<R>(s, sb, rank, xs, x, cnt, r, lo, acc);
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (r0 + q * TB < cnt) st_re(y, g0 + r[q], acc[q]);
}

// All rows of the group hi by a workgroup of TB threads, up to four rows per
// thread at once (they share the scalar work of a bond).
template <class XT, class YT, int TB>
__device__ inline void split_group(const SplitArgs &s, const SplitBonds &sb, uint32_t hi,
                                   const double *__restrict__ dlow, const uint16_t *rank,
                                   const XT *xs, const XT *__restrict__ x, YT *__restrict__ y,
                                   uint32_t g0, uint32_t cnt) {
  const uint32_t low0 = s.lowoff[s.w - __popc(hi)];
  for (uint32_t done = 0; done < cnt; done += 4 * TB) {
    const uint32_t left = cnt - done, r0 = done + threadIdx.x;
    if (left > 3 * TB)
      split_group_rows<XT, YT, 4, TB>(s, sb, dlow, rank, xs, x, y, g0, cnt, low0, r0);
    else if (left > 2 * TB)
      split_group_rows<XT, YT, 3, TB>(s, sb, dlow, rank, xs, x, y, g0, cnt, low0, r0);
    else if (left > TB)
      split_group_rows<XT, YT, 2, TB>(s, sb, dlow, rank, xs, x, y, g0, cnt, low0, r0);
    else
      split_group_rows<XT, YT, 1, TB>(s, sb, dlow, rank, xs, x, y, g0, cnt, low0, r0);
  }
}

} // namespace spined
