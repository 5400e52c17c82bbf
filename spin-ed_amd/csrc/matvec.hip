// matvec.hip -- matrix-free H*x row gather (ls_operator_matmat,
// src/SpinED/Internal.hs:377-378, :411-429).
//
// For representative r (row i) with |Stab r| = s_r:
//   y_i = D(r) x_i + sum_sigma conj(c_sigma) chi(h) sqrt(|Stab r'| / s_r) x_{idx(r')}
// where H|r> = sum_sigma c_sigma |sigma>, r' = h.sigma = min orbit(sigma),
// terms whose orbit has inconsistent phases (no symmetric state) or whose
// representative is not in the basis (another magnetisation sector) are
// dropped.  One lane owns one row and writes it once: no atomics.
//
// Per row, pass A walks the interaction tuples once: it accumulates the
// diagonal and marks the off-diagonal templates whose local state matches
// (a 64-bit word per 64 templates).  Pass B pops the marked templates in
// index order -- (tuple, a, b) order, the oracle's summation order -- and
// for each does orbit minimum, bucket + binary search and one fma gather.
// Lanes of a wave run pass B for max(#active) iterations; the orbit method
// (generic programs or ring run pruning) is a template parameter.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <vector>

#include "engine.hpp"
#include "rowgather.hpp"
#include "scan.hpp"

namespace spined {

namespace {

constexpr int kBlock = 256;

// ---- real rows -------------------------------------------------------------
// Row of slot i: identity, or the tile's schedule (rows of equal work side
// by side in a wave).
__device__ inline uint64_t scheduled_row(const uint16_t *__restrict__ sched, uint64_t i) {
  return sched ? (i & ~static_cast<uint64_t>(kScheduleTile - 1)) + sched[i] : i;
}

// One wave per workgroup: rows take unequal time, and a one-wave group frees
// its slot as soon as its own rows are done, which keeps more waves resident
// than four-wave groups that hold their slots until the slowest wave ends.
constexpr int kRowBlock = 64;

template <int METHOD, int NW, bool BONDS, class XT, class YT>
__global__ void __launch_bounds__(kRowBlock)
    matvec_real_kernel(OpArgs o, BondArgs bd, RatioArgs rt, GenericOrbitArgs ga,
                       RingOrbitArgs ra, IndexArgs ix, const uint32_t *__restrict__ stab,
                       uint64_t D, const XT *__restrict__ x, YT *__restrict__ y,
                       const uint16_t *__restrict__ sched) {
  // bond coefficients in LDS: a per-term global load would have to wait for
  // every gather issued before it (vector loads complete in order)
  __shared__ double so[BONDS ? 64 * NW : 1];
  if constexpr (BONDS) {
    for (int k = threadIdx.x; k < bd.nbonds; k += kRowBlock) so[k] = bd.o[k];
    __syncthreads();
  }
  const uint64_t lb = xcd_block(blockIdx.x, gridDim.x);
  const uint64_t slot = lb * kRowBlock + threadIdx.x;
  if (slot >= D) return;
  const uint64_t i = scheduled_row(sched, slot);
  st_re(y, i,
        gather_row_real<METHOD, NW, BONDS>(o, bd, rt, ga, ra, ix, stab, i, x, BONDS ? so : nullptr));
}

// matvec_real_kernel with L lanes per row (64 / L rows per wave): the same
// sums, the row's templates spread over its lanes (gather_row_real_lanes).
template <int METHOD, int NW, int L, class XT, class YT>
__global__ void __launch_bounds__(kRowBlock)
    matvec_real_lanes_kernel(OpArgs o, BondArgs bd, RatioArgs rt, GenericOrbitArgs ga,
                             RingOrbitArgs ra, IndexArgs ix, const uint32_t *__restrict__ stab,
                             uint64_t D, const XT *__restrict__ x, YT *__restrict__ y,
                             const uint16_t *__restrict__ sched) {
  __shared__ double so[64 * NW];
  for (int k = threadIdx.x; k < bd.nbonds; k += kRowBlock) so[k] = bd.o[k];
  __syncthreads();
  const uint64_t lb = xcd_block(blockIdx.x, gridDim.x);
  // a row's L lanes share the exit: the group's shuffles stay within it
  const uint64_t slot = lb * (kRowBlock / L) + threadIdx.x / L;
  if (slot >= D) return;
  const int sub = static_cast<int>(threadIdx.x % L);
  const uint64_t i = scheduled_row(sched, slot);
  const double v =
      gather_row_real_lanes<METHOD, NW, true, L>(o, bd, rt, ga, ra, ix, stab, i, x, so, sub);
  if (sub == 0) st_re(y, i, v);
}

// ---- gather cache -----------------------------------------------------------
// Active units (exchange bonds or templates) of a row, over any number of
// them.
template <bool BONDS>
__device__ inline uint32_t row_count(const OpArgs &o, const BondArgs &bd, uint64_t r) {
  uint32_t c = 0;
  if constexpr (BONDS) {
    for (int t = 0; t < bd.nbonds; ++t) {
      const uint32_t s = bd.sites[t];
      const uint32_t anti = static_cast<uint32_t>((r >> (s & 0xffu)) ^ (r >> (s >> 8))) & 1u;
      c += bd.o[t] != 0.0 ? anti : 0u;
    }
  } else {
    for (int t = 0; t < o.ntuples; ++t) {
      const uint32_t *rg = o.range + o.tuple_off[t] + t +
                           local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
      c += rg[1] - rg[0];
    }
  }
  return c;
}

// Diagonal of a row, summed in tuple order as the matrix-free kernels do.
template <bool BONDS>
__device__ inline double2 row_diag(const OpArgs &o, const BondArgs &bd, uint64_t r) {
  double re = 0.0, im = 0.0;
  if constexpr (BONDS) {
    for (int t = 0; t < bd.nbonds; ++t) {
      const uint32_t s = bd.sites[t];
      re += (((r >> (s & 0xffu)) ^ (r >> (s >> 8))) & 1u) ? bd.da[t] : bd.dp[t];
    }
  } else {
    for (int t = 0; t < o.ntuples; ++t) {
      const int a = local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
      re += o.diag_re[o.tuple_off[t] + a];
      im += o.diag_im[o.tuple_off[t] + a];
    }
  }
  return make_double2(re, im);
}

// Active units base .. base + 64 NW - 1 of a row, one bit each.
template <int NW, bool BONDS>
__device__ inline void row_active(const OpArgs &o, const BondArgs &bd, uint64_t r, int base,
                                  uint64_t (&act)[NW]) {
#pragma unroll
  for (int w = 0; w < NW; ++w) act[w] = 0;
  if constexpr (BONDS) {
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const int tb = base + 64 * w;
      const int te = bd.nbonds < tb + 64 ? bd.nbonds : tb + 64;
      for (int t = tb; t < te; ++t) {
        const uint32_t s = bd.sites[t];
        const uint64_t anti = ((r >> (s & 0xffu)) ^ (r >> (s >> 8))) & 1u;
        if (bd.o[t] != 0.0) act[w] |= anti << (t - tb);
      }
    }
  } else {
    const uint32_t lo = static_cast<uint32_t>(base), hi = lo + 64u * NW;
    for (int t = 0; t < o.ntuples; ++t) {
      const uint32_t *rg = o.range + o.tuple_off[t] + t +
                           local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
      const uint32_t b = rg[0] > lo ? rg[0] : lo, e = rg[1] < hi ? rg[1] : hi;
      if (b < e) mark_range<NW>(act, b - lo, e - lo);
    }
  }
}

// Where term t of a lane lies in its wave's entries: the wave's terms in
// groups of four per lane (one 16-byte load each), the last T mod 4 one by
// one (no padding beyond the wave's busiest row).
__device__ inline uint64_t term_pos(uint32_t t, uint32_t T, uint32_t lane) {
  const uint32_t full = T & ~3u;
  return t < full ? (static_cast<uint64_t>(t >> 2) * 256 + 4 * lane + (t & 3u))
                  : static_cast<uint64_t>(t) * 64 + lane;
}

// Terms of the busiest row of each wave (one wave = 64 slots).
template <bool BONDS>
__global__ void __launch_bounds__(kRowBlock)
    cache_count_kernel(OpArgs o, BondArgs bd, const uint64_t *__restrict__ reps, uint64_t D,
                       const uint16_t *__restrict__ sched, uint32_t *__restrict__ wave_terms) {
  const uint64_t slot = static_cast<uint64_t>(blockIdx.x) * kRowBlock + threadIdx.x;
  uint32_t c = 0;
  if (slot < D) c = row_count<BONDS>(o, bd, reps[scheduled_row(sched, slot)]);
  for (int off = 32; off > 0; off >>= 1) c = max(c, static_cast<uint32_t>(__shfl_xor(c, off, 64)));
  if (threadIdx.x == 0) wave_terms[blockIdx.x] = c;
}

// What the cached kernels read (GatherCache; engine.hpp has the layout).
struct CacheArgs {
  const uint64_t *__restrict__ woff;
  const uint32_t *__restrict__ entries;
  const uint16_t *__restrict__ aux;  // class of each term when it has no room in the entry
  const double *__restrict__ diag;   // per slot: one double, or two (re, im)
  const uint16_t *__restrict__ cnt;  // per slot
  const double *__restrict__ cls;    // nclass x (re, im)
  int32_t nclass;
  int32_t shift;                     // class = (entry >> shift) & cmask
  uint32_t imask, cmask;
};

// Entries of every term, in the order and with the orbits and lookups of
// gather_row_real; units beyond 64 NW in further rounds.  unit_cls: the
// coefficient class of each unit; phases: phase classes, 1 (all characters
// trivial), 2 (+-1) or L; CLS: more than one coefficient.  The outputs are arguments of their own: restrict
// does not hold inside a struct, and without it the group's programs are
// read by vector loads instead of scalar ones (2x the time on a 384-element
// group).
template <int METHOD, int NW, bool BONDS, bool CLS>
__global__ void __launch_bounds__(kRowBlock, 7)
    cache_fill_kernel(OpArgs o, BondArgs bd, GenericOrbitArgs ga, RingOrbitArgs ra, IndexArgs ix,
                      const uint32_t *__restrict__ stab, uint64_t D,
                      const uint16_t *__restrict__ sched, const uint64_t *__restrict__ woff,
                      const uint16_t *__restrict__ unit_cls, int32_t phases, int32_t shift,
                      int32_t complex_diag, uint32_t *__restrict__ entries,
                      uint16_t *__restrict__ aux, double *__restrict__ diag,
                      uint16_t *__restrict__ cnt) {
  ix = index_for_method<METHOD>(ix);
  const int units = BONDS ? bd.nbonds : o.ntemplates;
  __shared__ uint16_t s_cls[CLS ? 64 * NW : 1];
  if constexpr (CLS) {
    if (units <= 64 * NW)
      for (int j = threadIdx.x; j < units; j += kRowBlock) s_cls[j] = unit_cls[j];
    __syncthreads();
  }
  const uint64_t slot = static_cast<uint64_t>(blockIdx.x) * kRowBlock + threadIdx.x;
  if (slot >= D) return;
  const uint64_t i = scheduled_row(sched, slot);
  const uint64_t r = ix.reps[i];
  const double2 dg = row_diag<BONDS>(o, bd, r);
  if (complex_diag) {
    diag[2 * slot] = dg.x;
    diag[2 * slot + 1] = dg.y;
  } else {
    diag[slot] = dg.x;
  }
  const RowOrbit<METHOD, BONDS> rob(ra, bd, r);
  const int32_t si = static_cast<int32_t>(stab[i]);
  const uint64_t w0 = woff[blockIdx.x];
  const uint32_t T = static_cast<uint32_t>(woff[blockIdx.x + 1] - w0);
  uint32_t *out = entries + w0 * 64;
  // generic groups with trivial characters: the orbit minimum alone (no
  // phase can differ), |Stab| of the target from the basis' entry
  const bool min_only = METHOD == 0 && ga.trivial;
  uint32_t t = 0;
  uint4 group = make_uint4(0, 0, 0, 0);
  auto store = [&](int64_t k, const OrbitResult &orb, int j) __attribute__((always_inline)) {
    if (k < 0) return;
    const int32_t sk = min_only ? static_cast<int32_t>(stab[k]) : orb.count;
    // from LDS: a load here would wait for every load before it
    uint32_t cls = CLS ? (units <= 64 * NW ? s_cls[j] : unit_cls[j]) : 0u;
    if (phases == 2)
      cls = 2 * cls + (orb.phase != 0 ? 1u : 0u);
    else if (phases > 2)
      cls = cls * phases + orb.phase;
    if (aux) {
      aux[w0 * 64 + term_pos(t, T, threadIdx.x)] = static_cast<uint16_t>(cls);
      cls = 0;
    }
    // a class of 0 keeps the shift (up to 31) harmless
    const uint32_t ent =
        static_cast<uint32_t>(k) | (cls << shift) | (sk != si ? 1u << 31 : 0u);
    // groups of four leave as one 16-byte store: single entries (16 bytes
    // apart between lanes) made the fill of D = 2.3e8 25 ms longer
    const uint32_t q = t & 3u;
    if (t < (T & ~3u)) {
      group.x = q == 0 ? ent : group.x;
      group.y = q == 1 ? ent : group.y;
      group.z = q == 2 ? ent : group.z;
      group.w = q == 3 ? ent : group.w;
      if (q == 3u) reinterpret_cast<uint4 *>(out)[64ull * (t >> 2) + threadIdx.x] = group;
    } else {
      out[64ull * t + threadIdx.x] = ent;
    }
    ++t;
  };
  for (int base = 0; base < units; base += 64 * NW) {
    uint64_t act[NW];
    row_active<NW, BONDS>(o, bd, r, base, act);
    while (any_set<NW>(act)) {
      const int ja = base + pop_first<NW>(act);
      int jb = pop_first<NW>(act);
      jb = jb >= 0 ? base + jb : -1;
      OrbitResult oa{0, 0, 0, true}, ob{0, 0, 0, false};
      if (min_only) {
        oa.rep = orbit_min_generic(ga, r ^ (BONDS ? bd.flip[ja] : o.flip[ja]));
        if (jb >= 0) {
          ob.rep = orbit_min_generic(ga, r ^ (BONDS ? bd.flip[jb] : o.flip[jb]));
          ob.valid = true;
        }
      } else {
        oa = rob.orbit(o, bd, ga, ra, r, ja);
        if (jb >= 0) ob = rob.orbit(o, bd, ga, ra, r, jb);
      }
      int64_t ka, kb;
      find_index2(ix, oa.rep, oa.valid, ob.rep, ob.valid, ka, kb);
      store(ka, oa, ja);
      if (jb >= 0) store(kb, ob, jb);
    }
  }
  if (t < (T & ~3u) && (t & 3u))
    reinterpret_cast<uint4 *>(out)[64ull * (t >> 2) + threadIdx.x] = group;
  cnt[slot] = static_cast<uint16_t>(t);
}

// Vectors that a cached matvec works on: K row-interleaved real vectors, or
// one complex vector.  Same arithmetic as the matrix-free kernels.
template <class XT, class YT, int K> struct RealRows {
  using X = RowK<XT, K>;
  using Y = RowK<YT, K>;
  using C = double; // coefficient
  static constexpr int kGroups = K == 1 ? 2 : 1; // groups of four entries per step
  static __device__ C pick(double2 c) { return c.x; }
  double acc[K];
  __device__ void start(const double *diag, uint64_t slot, bool, const X &x) {
    const double d = diag[slot];
#pragma unroll
    for (int c = 0; c < K; ++c) acc[c] = d * static_cast<double>(x.v[c]);
  }
  __device__ void term(C k, double f, const X &x, bool use) {
    const double cf = k * f;
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const double t = fma(cf, static_cast<double>(x.v[c]), acc[c]);
      acc[c] = use ? t : acc[c];
    }
  }
  __device__ Y result() const {
    Y out;
#pragma unroll
    for (int c = 0; c < K; ++c) out.v[c] = static_cast<YT>(acc[c]);
    return out;
  }
};

template <class T> struct ComplexRows { // T = float2 or double2
  using X = T;
  using Y = T;
  using C = double2;
  static constexpr int kGroups = 2;
  static __device__ C pick(double2 c) { return c; }
  double re, im;
  __device__ void start(const double *diag, uint64_t slot, bool complex_diag, const X &x) {
    const double dr = complex_diag ? diag[2 * slot] : diag[slot];
    const double di = complex_diag ? diag[2 * slot + 1] : 0.0;
    const double xr = static_cast<double>(x.x), xi = static_cast<double>(x.y);
    re = fma(dr, xr, -(di * xi));
    im = fma(dr, xi, di * xr);
  }
  __device__ void term(C k, double f, const X &x, bool use) {
    const double kr = k.x * f, ki = k.y * f;
    const double xr = static_cast<double>(x.x), xi = static_cast<double>(x.y);
    const double tr = fma(-ki, xi, fma(kr, xr, re));
    const double ti = fma(ki, xr, fma(kr, xi, im));
    re = use ? tr : re;
    im = use ? ti : im;
  }
  __device__ Y result() const {
    Y out;
    st_c(&out, 0, make_double2(re, im));
    return out;
  }
};

// Matvec from the gather cache: the sums of the matrix-free kernels (same
// terms, coefficients and order) without orbits or index searches.
// CM: where a term's coefficient comes from -- 0: one class for all terms
// (a kernel argument), 1: up to kLdsClasses classes in LDS, 2: the table in
// memory (read before the gathers of its step: loads complete in order).
// Bound: the latency of the x gathers, and past the L2 the lines they fetch.
// One vector takes eight gathers per step (two groups of four entries; D =
// 6.3e7 ring, FP64: 5.30 ms with four, 5.13 with eight), wider records four
// (their registers would cost waves).  NT: entries read around the caches,
// for entry blocks that no cache keeps from one matvec to the next (1.2e9
// terms: 5.13 -> 4.99 ms; 2e7 terms, 87 MB: 65 -> 80 us, so not there).
// Against one load per entry, states and bonds read per row and the
// coefficient by bond, D = 28,968 takes 8.2 us (matrix-free: 72), D = 2.3e8
// 21.5 ms (24.2).
constexpr int kLdsClasses = 64;
constexpr uint64_t kCacheStreamBytes = uint64_t(128) << 20;

template <class R, int CM, bool NT>
__global__ void __launch_bounds__(kRowBlock)
    matvec_cached_kernel(CacheArgs c, RatioArgs rt, const uint32_t *__restrict__ stab, uint64_t D,
                         const typename R::X *__restrict__ x, typename R::Y *__restrict__ y,
                         const uint16_t *__restrict__ sched, int contiguous, int complex_diag,
                         double2 one) {
  using X = typename R::X;
  using C = typename R::C;
  __shared__ C scls[CM == 1 ? kLdsClasses : 1];
  if constexpr (CM == 1) {
    if (static_cast<int>(threadIdx.x) < c.nclass)
      scls[threadIdx.x] =
          R::pick(make_double2(c.cls[2 * threadIdx.x], c.cls[2 * threadIdx.x + 1]));
    __syncthreads();
  }
  const uint64_t lb = contiguous ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
  const uint64_t slot = lb * kRowBlock + threadIdx.x;
  const uint64_t w0 = c.woff[lb];
  const uint32_t T = static_cast<uint32_t>(c.woff[lb + 1] - w0);
  if (slot >= D) return;
  const uint32_t *in = c.entries + w0 * 64;
  const uint32_t lane = threadIdx.x;
  constexpr int Q = R::kGroups;
  const uint32_t nq = T >> 2;
  auto group = [&](uint32_t g) {
    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    const v4 *p = reinterpret_cast<const v4 *>(in) + 64ull * g + lane;
    const v4 none = {0, 0, 0, 0};
    if constexpr (NT) return g < nq ? __builtin_nontemporal_load(p) : none;
    return g < nq ? *p : none;
  };
  decltype(group(0)) e[Q];
#pragma unroll
  for (int z = 0; z < Q; ++z) e[z] = group(z);
  const uint64_t i = scheduled_row(sched, slot);
  const uint32_t n = c.cnt[slot];
  R row;
  row.start(c.diag, slot, complex_diag != 0, x[i]);
  auto coef = [&](uint32_t ent, uint64_t pos) {
    if constexpr (CM == 0) return R::pick(one);
    if constexpr (CM == 1) return scls[(ent >> c.shift) & c.cmask];
    uint32_t k = c.aux ? c.aux[w0 * 64 + pos] : ((ent >> c.shift) & c.cmask);
    k = min(k, static_cast<uint32_t>(c.nclass - 1)); // unwritten entries beyond a row's terms
    return R::pick(make_double2(c.cls[2 * k], c.cls[2 * k + 1]));
  };
  auto ratio = [&](uint32_t ent) {
    double f = 1.0;
    if (ent >> 31) {
      const uint32_t ck = stab[ent & c.imask], si = stab[i];
      f = rt.nd ? rt.ratio[rt.div_idx[ck] * rt.nd + rt.div_idx[si]]
                : sqrt(static_cast<double>(ck) / static_cast<double>(si));
    }
    return f;
  };
  const uint32_t n4 = min(n, nq << 2); // terms in groups
  for (uint32_t g = 0; g < nq; g += Q) {
    uint32_t ev[4 * Q];
    C cv[4 * Q];
    X xv[4 * Q];
#pragma unroll
    for (int q = 0; q < 4 * Q; ++q) {
      ev[q] = e[q / 4][q % 4];
      cv[q] = coef(ev[q], 256ull * min(g + q / 4, nq - 1) + 4 * lane + q % 4);
    }
    // lanes past their row's terms read x[i], which is at hand
#pragma unroll
    for (int q = 0; q < 4 * Q; ++q) xv[q] = x[4 * g + q < n4 ? ev[q] & c.imask : i];
    // after the gathers: loads return in order, and these come from HBM
#pragma unroll
    for (int z = 0; z < Q; ++z) e[z] = group(g + Q + z);
#pragma unroll
    for (int q = 0; q < 4 * Q; ++q) {
      const bool use = 4 * g + q < n4;
      row.term(cv[q], use ? ratio(ev[q]) : 1.0, xv[q], use);
    }
  }
  for (uint32_t t = nq << 2; t < T; ++t) {
    if (t >= n) break;
    const uint32_t ent = in[64ull * t + lane];
    row.term(coef(ent, 64ull * t + lane), ratio(ent), x[ent & c.imask], true);
  }
  y[i] = row.result();
}

// ---- split row gather (split.hpp) -------------------------------------------
__global__ void __launch_bounds__(kBlock)
    split_dlow_kernel(SplitArgs s, BondArgs bd, double *__restrict__ dlow) {
  const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
  if (e < (1u << s.l)) dlow[e] = split_dlow(s, bd, s.lowstate[e]);
}

// One workgroup per group of rows.  Bound: instruction issue (about 250
// vector instructions per row and wave) and the two LDS reads of each low
// bond, so a thread takes up to four rows at once, which share the scalar
// work of a bond.  D = 5.2e6 (26 sites): 85 us (FP64) and 86 us (FP32) with
// four rows, 150 and 148 with one; from the gather cache 145 and 117.
template <class XT, class YT>
__global__ void __launch_bounds__(kBlock)
    matvec_split_kernel(SplitArgs s, BondArgs bd, const double *__restrict__ dlow,
                        const XT *__restrict__ x, YT *__restrict__ y) {
  extern __shared__ char split_lds[];
  uint16_t *rank = reinterpret_cast<uint16_t *>(split_lds);
  XT *xs = reinterpret_cast<XT *>(split_lds + (sizeof(uint16_t) << s.l));
  const uint32_t hi = static_cast<uint32_t>(xcd_block(blockIdx.x, gridDim.x));
  const uint32_t g0 = s.goff[hi], cnt = s.goff[hi + 1] - g0;
  if (cnt == 0) return;
  const uint4 *rk = reinterpret_cast<const uint4 *>(s.lowrank);
  for (uint32_t t = threadIdx.x; t < (1u << s.l) / 8; t += kBlock)
    reinterpret_cast<uint4 *>(rank)[t] = rk[t];
  for (uint32_t t = threadIdx.x; t < cnt; t += kBlock) xs[t] = x[g0 + t];
  const SplitBonds sb =
      split_bonds(s, split_bond(bd, static_cast<int>(threadIdx.x & 63)), hi);
  __syncthreads();
  split_group<XT, YT, kBlock>(s, sb, hi, dlow, rank, xs, x, y, g0, cnt);
}

// Row-interleaved block of K real vectors (x[row * K + c]); per column the
// same sums as matvec_real_kernel.
template <int METHOD, int NW, bool BONDS, int K, class XT, class YT>
__global__ void __launch_bounds__(kBlock)
    matvec_block_kernel(OpArgs o, BondArgs bd, RatioArgs rt, GenericOrbitArgs ga,
                        RingOrbitArgs ra, IndexArgs ix, const uint32_t *__restrict__ stab,
                        uint64_t D, const XT *__restrict__ x, YT *__restrict__ y,
                        const uint16_t *__restrict__ sched) {
  const uint64_t lb = xcd_block(blockIdx.x, gridDim.x);
  const uint64_t slot = lb * kBlock + threadIdx.x;
  if (slot >= D) return;
  const uint64_t i = scheduled_row(sched, slot);
  double acc[K];
  gather_row_real_block<METHOD, NW, BONDS, K>(o, bd, rt, ga, ra, ix, stab, i, x, acc);
  RowK<YT, K> out;
#pragma unroll
  for (int c = 0; c < K; ++c) out.v[c] = static_cast<YT>(acc[c]);
  reinterpret_cast<RowK<YT, K> *>(y)[i] = out;
}

// Column-major block (column c at x + c * stride) <-> row-interleaved block
// (xr[row * K + c]); one thread per row.
template <class A, class B>
__global__ void __launch_bounds__(kBlock)
    cols_to_rows_kernel(const A *__restrict__ x, uint64_t stride, uint64_t D, int K,
                        B *__restrict__ xr) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= D) return;
  for (int c = 0; c < K; ++c) xr[i * K + c] = static_cast<B>(x[c * stride + i]);
}

template <class A, class B>
__global__ void __launch_bounds__(kBlock)
    rows_to_cols_kernel(const A *__restrict__ yr, uint64_t D, int K, B *__restrict__ y,
                        uint64_t stride) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= D) return;
  for (int c = 0; c < K; ++c) y[c * stride + i] = static_cast<B>(yr[i * K + c]);
}

// Row schedule of one tile (one workgroup per tile): the active units of
// each row, then a counting sort by count, stable in the row order.  Each of
// the 16 waves owns 256 consecutive rows: a first pass adds up its counts
// per bin, a scan over (bin, wave) gives its first slot of every bin, a
// second pass places 64 rows at a time (a row's rank among the lanes of its
// bin from ballots of the bin's bits).  One serial thread took 205 us for
// any basis.
constexpr int kSchedBins = 1024;
constexpr int kSchedBlock = 1024;

__device__ inline uint64_t same_bin_lanes(uint32_t bin, bool in) {
  uint64_t m = __ballot(in);
#pragma unroll
  for (int b = 0; b < 10; ++b) {
    const uint64_t v = __ballot((bin >> b) & 1u);
    m &= ((bin >> b) & 1u) ? v : ~v;
  }
  return m;
}

template <bool BONDS>
__global__ void __launch_bounds__(kSchedBlock)
    schedule_kernel(OpArgs o, BondArgs bd, const uint64_t *__restrict__ reps, uint64_t D,
                    uint16_t *__restrict__ sched) {
  constexpr int kWaves = kSchedBlock / 64, kPerWave = kScheduleTile / kWaves;
  __shared__ uint16_t count_of[kScheduleTile];
  __shared__ uint16_t first[kWaves][kSchedBins]; // at most kScheduleTile rows
  __shared__ uint32_t part[kSchedBlock];
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * kScheduleTile;
  const int rows = static_cast<int>(D - base < kScheduleTile ? D - base : kScheduleTile);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int t = threadIdx.x; t < kWaves * kSchedBins; t += kSchedBlock) first[t / kSchedBins][t % kSchedBins] = 0;
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1;
  for (int k0 = 0; k0 < kPerWave; k0 += 64) {
    const int k = wid * kPerWave + k0 + lane;
    const bool in = k < rows;
    uint32_t c = 0;
    if (in) c = min(row_count<BONDS>(o, bd, reps[base + k]), static_cast<uint32_t>(kSchedBins - 1));
    count_of[k] = static_cast<uint16_t>(c);
    const uint64_t m = same_bin_lanes(c, in);
    if (in && (m & below) == 0) first[wid][c] += static_cast<uint16_t>(__popcll(m));
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // exclusive scan over bins (each thread kSchedBins / kSchedBlock of them), the
  // waves of a bin in order
  constexpr int kPer = kSchedBins / kSchedBlock;
  uint32_t sum = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    for (int w = 0; w < kWaves; ++w) sum += first[w][threadIdx.x * kPer + q];
  part[threadIdx.x] = sum;
  __syncthreads();
  for (int off = 1; off < kSchedBlock; off <<= 1) {
    const uint32_t v = threadIdx.x >= static_cast<unsigned>(off) ? part[threadIdx.x - off] : 0;
    __syncthreads();
    part[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = part[threadIdx.x] - sum;
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t h = first[w][threadIdx.x * kPer + q];
      first[w][threadIdx.x * kPer + q] = static_cast<uint16_t>(run);
      run += h;
    }
  __syncthreads();
  for (int k0 = 0; k0 < kPerWave; k0 += 64) {
    const int k = wid * kPerWave + k0 + lane;
    const bool in = k < rows;
    const uint32_t c = count_of[k];
    const uint64_t m = same_bin_lanes(c, in);
    const uint32_t at = first[wid][c] + static_cast<uint32_t>(__popcll(m & below));
    // every lane has read its bin before the bin's first lane moves it on
    __builtin_amdgcn_wave_barrier();
    if (in) sched[base + at] = static_cast<uint16_t>(k);
    if (in && (m & below) == 0) first[wid][c] = static_cast<uint16_t>(at + __popcll(m));
    __builtin_amdgcn_wave_barrier();
  }
}

// Rows with more than 256 off-diagonal templates: per-tuple loop.
template <int METHOD, class XT, class YT>
__global__ void __launch_bounds__(kBlock)
    matvec_real_direct_kernel(OpArgs o, GenericOrbitArgs ga, RingOrbitArgs ra, IndexArgs ix,
                              const uint32_t *__restrict__ stab, uint64_t D,
                              const XT *__restrict__ x, YT *__restrict__ y) {
  ix = index_for_method<METHOD>(ix);
  const uint64_t lb = xcd_block(blockIdx.x, gridDim.x);
  const uint64_t i = lb * kBlock + threadIdx.x;
  if (i >= D) return;
  const uint64_t r = ix.reps[i];
  double diag = 0.0;
  for (int t = 0; t < o.ntuples; ++t) {
    const int a = local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
    diag += o.diag_re[o.tuple_off[t] + a];
  }
  double acc = diag * ld_re(x, i);
  const double sr = static_cast<double>(stab[i]);
  for (int t = 0; t < o.ntuples; ++t) {
    const uint32_t off = o.tuple_off[t];
    const int a = local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
    const uint32_t b = o.range[off + t + a], e = o.range[off + t + a + 1];
    for (uint32_t j = b; j < e; ++j) {
      const OrbitResult orb = do_orbit<METHOD>(ga, ra, r ^ o.flip[j]);
      if (!orb.valid) continue;
      const int64_t k = find_index(ix, orb.rep);
      if (k < 0) continue;
      double coef = o.coef_re[j] * sqrt(static_cast<double>(orb.count) / sr);
      if (orb.phase != 0) coef = -coef;
      acc = fma(coef, ld_re(x, static_cast<uint64_t>(k)), acc);
    }
  }
  st_re(y, i, acc);
}

// ---- complex rows ------------------------------------------------------------
template <int METHOD, class XT, class YT>
__global__ void __launch_bounds__(kBlock)
    matvec_complex_kernel(OpArgs o, GenericOrbitArgs ga, RingOrbitArgs ra, IndexArgs ix,
                          const uint32_t *__restrict__ stab, uint64_t D,
                          const XT *__restrict__ x, YT *__restrict__ y) {
  ix = index_for_method<METHOD>(ix);
  const uint64_t lb = xcd_block(blockIdx.x, gridDim.x);
  const uint64_t i = lb * kBlock + threadIdx.x;
  if (i >= D) return;
  const uint64_t r = ix.reps[i];
  double dre = 0.0, dim = 0.0;
  for (int t = 0; t < o.ntuples; ++t) {
    const int a = local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
    dre += o.diag_re[o.tuple_off[t] + a];
    dim += o.diag_im[o.tuple_off[t] + a];
  }
  const double2 xi = ld_c(x, i);
  double are = fma(dre, xi.x, -(dim * xi.y));
  double aim = fma(dre, xi.y, dim * xi.x);
  const double sr = static_cast<double>(stab[i]);
  for (int t = 0; t < o.ntuples; ++t) {
    const uint32_t off = o.tuple_off[t];
    const int a = local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
    const uint32_t b = o.range[off + t + a], e = o.range[off + t + a + 1];
    for (uint32_t j = b; j < e; ++j) {
      const OrbitResult orb = do_orbit<METHOD>(ga, ra, r ^ o.flip[j]);
      if (!orb.valid) continue;
      const int64_t k = find_index(ix, orb.rep);
      if (k < 0) continue;
      const double f = sqrt(static_cast<double>(orb.count) / sr);
      const double cre = o.phase_cos[orb.phase], cim = o.phase_sin[orb.phase];
      const double mre = o.coef_re[j], mim = o.coef_im[j];
      const double kre = fma(mre, cre, -(mim * cim)) * f;
      const double kim = fma(mre, cim, mim * cre) * f;
      const double2 xk = ld_c(x, static_cast<uint64_t>(k));
      are = fma(kre, xk.x, are);
      are = fma(-kim, xk.y, are);
      aim = fma(kre, xk.y, aim);
      aim = fma(kim, xk.x, aim);
    }
  }
  st_c(y, i, make_double2(are, aim));
}

// ---- counting (measurement) --------------------------------------------------
template <int METHOD>
__global__ void __launch_bounds__(kBlock)
    count_offdiag_kernel(OpArgs o, GenericOrbitArgs ga, RingOrbitArgs ra, IndexArgs ix,
                         uint64_t D, unsigned long long *__restrict__ partial) {
  ix = index_for_method<METHOD>(ix);
  __shared__ unsigned long long lds[kBlock / 64];
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
  unsigned long long c = 0;
  if (i < D) {
    const uint64_t r = ix.reps[i];
    for (int t = 0; t < o.ntuples; ++t) {
      const uint32_t off = o.tuple_off[t];
      const int a = local_state(o.tuple_sites[t], static_cast<int>(o.tuple_n[t]), r);
      const uint32_t b = o.range[off + t + a], e = o.range[off + t + a + 1];
      for (uint32_t j = b; j < e; ++j) {
        const OrbitResult orb = do_orbit<METHOD>(ga, ra, r ^ o.flip[j]);
        if (orb.valid && find_index(ix, orb.rep) >= 0) ++c;
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (int w = 0; w < kBlock / 64; ++w) s += lds[w];
    partial[blockIdx.x] = s;
  }
}

struct PhaseTable {
  DeviceBuffer<double> cos_t, sin_t;
  int L = 0;
};

// chi(phase) = exp(2 pi i phase / L), exact at quarter turns (same values
// as the oracle's phase_to_complex).
void phase_values(int64_t p, int64_t L, double &c, double &s) {
  p = ((p % L) + L) % L;
  if (p == 0) { c = 1.0; s = 0.0; }
  else if (2 * p == L) { c = -1.0; s = 0.0; }
  else if (4 * p == L) { c = 0.0; s = 1.0; }
  else if (4 * p == 3 * L) { c = 0.0; s = -1.0; }
  else {
    const double ang = 2.0 * M_PI * static_cast<double>(p) / static_cast<double>(L);
    c = std::cos(ang);
    s = std::sin(ang);
  }
}

OpArgs op_args(const Operator &op, const double *pc, const double *ps) {
  const auto &t = op.tables;
  OpArgs a{};
  a.tuple_sites = t.tuple_sites.ptr;
  a.tuple_n = t.tuple_n.ptr;
  a.tuple_off = t.tuple_off.ptr;
  a.range = t.range.ptr;
  a.diag_re = t.diag_re.ptr;
  a.diag_im = t.diag_im.ptr;
  a.flip = t.flip.ptr;
  a.coef_re = t.coef_re.ptr;
  a.coef_im = t.coef_im.ptr;
  a.phase_cos = pc;
  a.phase_sin = ps;
  a.ntuples = t.ntuples;
  a.ntemplates = t.ntemplates;
  return a;
}

unsigned grid_for(uint64_t n) { return static_cast<unsigned>((n + kBlock - 1) / kBlock); }

// Everything a launch needs, gathered once per call.
struct Ctx {
  OpArgs o;
  BondArgs bd;
  RatioArgs rt;
  GenericOrbitArgs ga;
  RingOrbitArgs ra;
  IndexArgs ix;
  const uint32_t *stab;
  uint64_t D;
  bool bonds;
  const uint16_t *sched;
  int lanes; // lanes per row of the exchange-bond matrix-free kernel (1, 2, 4)
};

template <int METHOD, int NW, bool BONDS, class XT, class YT>
void launch_real_nw(const Ctx &c, const XT *x, YT *y, hipStream_t s) {
  if constexpr (BONDS) {
    if (c.lanes == 2 || c.lanes == 4) {
      const uint64_t rows = kRowBlock / c.lanes;
      const unsigned g = static_cast<unsigned>((c.D + rows - 1) / rows);
      if (c.lanes == 2)
        matvec_real_lanes_kernel<METHOD, NW, 2, XT, YT><<<g, kRowBlock, 0, s>>>(
            c.o, c.bd, c.rt, c.ga, c.ra, c.ix, c.stab, c.D, x, y, c.sched);
      else
        matvec_real_lanes_kernel<METHOD, NW, 4, XT, YT><<<g, kRowBlock, 0, s>>>(
            c.o, c.bd, c.rt, c.ga, c.ra, c.ix, c.stab, c.D, x, y, c.sched);
      return;
    }
  }
  const unsigned g = static_cast<unsigned>((c.D + kRowBlock - 1) / kRowBlock);
  matvec_real_kernel<METHOD, NW, BONDS, XT, YT><<<g, kRowBlock, 0, s>>>(
      c.o, c.bd, c.rt, c.ga, c.ra, c.ix, c.stab, c.D, x, y, c.sched);
}

template <int METHOD, class XT, class YT>
void launch_real(const Ctx &c, const XT *x, YT *y, hipStream_t s) {
  const int units = c.bonds ? c.bd.nbonds : c.o.ntemplates;
  if (c.bonds && units <= 64)
    launch_real_nw<METHOD, 1, true>(c, x, y, s);
  else if (c.bonds && units <= 128)
    launch_real_nw<METHOD, 2, true>(c, x, y, s);
  else if (!c.bonds && units <= 64)
    launch_real_nw<METHOD, 1, false>(c, x, y, s);
  else if (!c.bonds && units <= 128)
    launch_real_nw<METHOD, 2, false>(c, x, y, s);
  else if (!c.bonds && units <= 256)
    launch_real_nw<METHOD, 4, false>(c, x, y, s);
  else
    matvec_real_direct_kernel<METHOD, XT, YT><<<grid_for(c.D), kBlock, 0, s>>>(
        c.o, c.ga, c.ra, c.ix, c.stab, c.D, x, y);
  SPINED_CHECK_LAUNCH();
}

template <int METHOD, class XT, class YT>
void launch_complex(const Ctx &c, const XT *x, YT *y, hipStream_t s) {
  matvec_complex_kernel<METHOD, XT, YT><<<grid_for(c.D), kBlock, 0, s>>>(c.o, c.ga, c.ra, c.ix,
                                                                        c.stab, c.D, x, y);
  SPINED_CHECK_LAUNCH();
}

template <int METHOD> void dispatch(const MatvecCall &m, const Ctx &c) {
  hipStream_t s = m.stream;
  using VT = VecType;
  if (m.xt == VT::F64 && m.yt == VT::F64)
    launch_real<METHOD>(c, static_cast<const double *>(m.x), static_cast<double *>(m.y), s);
  else if (m.xt == VT::F32 && m.yt == VT::F32)
    launch_real<METHOD>(c, static_cast<const float *>(m.x), static_cast<float *>(m.y), s);
  else if (m.xt == VT::F32 && m.yt == VT::F64)
    launch_real<METHOD>(c, static_cast<const float *>(m.x), static_cast<double *>(m.y), s);
  else if (m.xt == VT::C128 && m.yt == VT::C128)
    launch_complex<METHOD>(c, static_cast<const double2 *>(m.x), static_cast<double2 *>(m.y), s);
  else if (m.xt == VT::C64 && m.yt == VT::C64)
    launch_complex<METHOD>(c, static_cast<const float2 *>(m.x), static_cast<float2 *>(m.y), s);
  else
    throw Error(LS_INVALID_DATATYPE, "unsupported matvec type combination");
}

// Free memory that an automatically built gather cache leaves untouched.
constexpr uint64_t kCacheReserve = uint64_t(4) << 30;
// An automatic cache is built at the first matvec of a basis of kCacheMinRows
// rows, or when the matrix-free matvec takes about kCacheFirstWork orbit
// steps (some 300 us) -- the build, one pass over the orbits, then costs
// about what that matvec would.  Smaller operators build it at their second
// use (a single application is cheaper without), those of up to
// kCacheTinyRows rows never (the dense solver's unit vectors).
constexpr uint64_t kCacheMinRows = uint64_t(1) << 20;
constexpr uint64_t kCacheTinyRows = 64;
constexpr double kCacheFirstWork = 2e9;

int unit_count(const OperatorTables &t) {
  return t.bonds ? static_cast<int>(t.h_bond_sites.size()) : t.ntemplates;
}

// Whether an automatic cache of the operator is due at its `calls`-th use.
bool cache_due(const Operator &op, int calls) {
  const Basis &b = *op.basis;
  if (b.D >= kCacheMinRows) return true;
  if (b.D <= kCacheTinyRows) return false;
  const double orbit = op.orbit_method() == 1 ? 64.0 : 2.0 * b.tables.orbit_cost;
  return calls >= 2 ||
         static_cast<double>(b.D) * unit_count(op.tables) * orbit >= kCacheFirstWork;
}

// 16-bit class numbers
constexpr uint64_t kCacheMaxClasses = 65536;

// Coefficient classes: every distinct unit coefficient times every phase
// that an orbit can return, with the products of matvec_complex_kernel (and,
// for real characters, the sign flip of the real kernels).  False when there
// are too many.
bool cache_classes(const Operator &op, GatherCache &gc, hipStream_t s) {
  const auto &t = op.tables;
  const auto &bt = op.basis->tables;
  const int units = unit_count(t);
  std::vector<uint16_t> of_unit(std::max(units, 1), 0);
  std::vector<std::pair<double, double>> coefs;
  std::map<std::pair<uint64_t, uint64_t>, uint16_t> seen;
  for (int j = 0; j < units; ++j) {
    const double re = t.bonds ? t.h_bond_o[j] : t.h_coef_re[j];
    const double im = t.bonds ? 0.0 : t.h_coef_im[j];
    uint64_t a, b;
    std::memcpy(&a, &re, 8);
    std::memcpy(&b, &im, 8);
    const auto it = seen.emplace(std::make_pair(a, b), static_cast<uint16_t>(coefs.size()));
    if (it.second) coefs.push_back({re, im});
    if (coefs.size() > kCacheMaxClasses) return false;
    of_unit[j] = it.first->second;
  }
  if (coefs.empty()) coefs.push_back({0.0, 0.0});
  const int64_t np = bt.trivial_chars ? 1 : bt.real_chars ? 2 : bt.L;
  if (static_cast<uint64_t>(np) * coefs.size() > kCacheMaxClasses) return false;
  std::vector<double> cls;
  for (const auto &c : coefs)
    for (int64_t p = 0; p < np; ++p) {
      double cre = 1.0, cim = 0.0;
      if (np == 2)
        cre = p ? -1.0 : 1.0;
      else
        phase_values(p, np > 2 ? np : 1, cre, cim);
      if (t.is_real) {
        cls.push_back(p ? -c.first : c.first);
        cls.push_back(0.0);
      } else {
        cls.push_back(std::fma(c.first, cre, -(c.second * cim)));
        cls.push_back(std::fma(c.first, cim, c.second * cre));
      }
    }
  gc.phases = static_cast<int32_t>(np);
  gc.nclass = static_cast<int32_t>(cls.size() / 2);
  gc.one[0] = cls[0];
  gc.one[1] = cls[1];
  gc.cls.allocate(cls.size());
  SPINED_HIP(hipMemcpyAsync(gc.cls.ptr, cls.data(), 8 * cls.size(), hipMemcpyHostToDevice, s));
  gc.unit_cls.allocate(of_unit.size());
  SPINED_HIP(hipMemcpyAsync(gc.unit_cls.ptr, of_unit.data(), 2 * of_unit.size(),
                            hipMemcpyHostToDevice, s));
  SPINED_HIP(hipStreamSynchronize(s)); // the host vectors end here
  // entry: index bits, class bits, ratio bit
  int ib = 0, cb = 0;
  while ((1ull << ib) < op.basis->D) ++ib;
  while ((1ll << cb) < gc.nclass) ++cb;
  gc.in_entry = ib + cb <= 31;
  gc.shift = ib;
  gc.cmask = gc.in_entry ? static_cast<uint32_t>((1ull << cb) - 1) : 0u;
  gc.imask = static_cast<uint32_t>((1ull << ib) - 1);
  return true;
}

// Whether the row schedule serves the operator's gather cache alone: the
// matrix-free kernels of complex operators and of those of many templates take
// the rows in order.
bool schedule_of_cache(const Operator &op) {
  const auto &t = op.tables;
  return !t.is_real || unit_count(t) > (t.bonds ? 128 : 256);
}

void launch_schedule(const Operator &op, const Ctx &c, uint16_t *sched, hipStream_t s) {
  const Basis &b = *op.basis;
  const unsigned tiles = static_cast<unsigned>((b.D + kScheduleTile - 1) / kScheduleTile);
  if (c.bonds)
    schedule_kernel<true><<<tiles, kSchedBlock, 0, s>>>(c.o, c.bd, b.reps.ptr, b.D, sched);
  else
    schedule_kernel<false><<<tiles, kSchedBlock, 0, s>>>(c.o, c.bd, b.reps.ptr, b.D, sched);
  SPINED_CHECK_LAUNCH();
}

template <int METHOD, class F> void with_fill(const Ctx &c, F &&f) {
  const int units = c.bonds ? c.bd.nbonds : c.o.ntemplates;
  if (c.bonds && units <= 64)
    f(std::integral_constant<int, 1>{}, std::true_type{});
  else if (c.bonds)
    f(std::integral_constant<int, 2>{}, std::true_type{});
  else if (units <= 64)
    f(std::integral_constant<int, 1>{}, std::false_type{});
  else if (units <= 128)
    f(std::integral_constant<int, 2>{}, std::false_type{});
  else
    f(std::integral_constant<int, 4>{}, std::false_type{});
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  SPINED_HIP(hipStreamIsCapturing(s, &cap));
  return cap != hipStreamCaptureStatusNone;
}

// Builds the gather cache when it is requested (1), or when it is automatic
// (-1), due (see kCacheMinRows; repeated: more matvecs are known to follow)
// and fits in free memory with kCacheReserve to spare.  Caller holds gc.mu.
// True when the cache is ready.
template <int METHOD>
bool ensure_cache(const Operator &op, const Ctx &c, GatherCache &gc, hipStream_t s,
                  bool repeated = false, uint64_t reserve = kCacheReserve, uint64_t reusable = 0) {
  if (gc.built) return true;
  const Basis &b = *op.basis;
  const int units = unit_count(op.tables);
  if (gc.request == 0 || gc.unsuitable || b.D > (1ull << 31) || units > 65535) return false;
  // nothing is built under stream capture: its kernels would only run at a replay
  if (capturing(s)) {
    if (gc.request > 0) throw Error(LS_DEVICE_ERROR, "gather cache: not built under stream capture");
    return false;
  }
  struct Building {
    std::atomic<bool> &f;
    explicit Building(std::atomic<bool> &x) : f(x) { f.store(true); }
    ~Building() { f.store(false); }
  } building(gc.building);
  if (gc.request < 0 && !(repeated && b.D > kCacheTinyRows) && !cache_due(op, gc.calls.load()))
    return false;
  const uint64_t waves = (b.D + kRowBlock - 1) / kRowBlock;
  const unsigned g = static_cast<unsigned>(waves);
  if (!gc.counted) {
    const bool own_sched = !c.sched && schedule_of_cache(op) && op.schedule_request < 0 &&
                           b.D >= static_cast<uint64_t>(kScheduleTile);
    // where the reserve is spent no cache can fit: a matvec then needs no
    // device memory but its vectors, and its tables must not be refused
    if (gc.request < 0) {
      size_t free_b = 0, total_b = 0;
      SPINED_HIP(hipMemGetInfo(&free_b, &total_b));
      if (free_b < kCacheReserve + (own_sched ? b.D * sizeof(uint16_t) : 0)) return false;
    }
    if (!cache_classes(op, gc, s)) {
      gc.unsuitable = true; // also when asked for: as for more than 65,535 units
      return false;
    }
    gc.sched = c.sched;
    if (own_sched) {
      gc.own_sched.allocate(b.D);
      launch_schedule(op, c, gc.own_sched.ptr, s);
      gc.sched = gc.own_sched.ptr;
    }
    DeviceBuffer<uint32_t> wt(waves);
    if (c.bonds)
      cache_count_kernel<true><<<g, kRowBlock, 0, s>>>(c.o, c.bd, b.reps.ptr, b.D, gc.sched, wt.ptr);
    else
      cache_count_kernel<false><<<g, kRowBlock, 0, s>>>(c.o, c.bd, b.reps.ptr, b.D, gc.sched,
                                                        wt.ptr);
    SPINED_CHECK_LAUNCH();
    gc.woff.allocate(waves + 1);
    scan_counts(wt.ptr, waves, gc.woff.ptr, gc.woff.ptr + waves, s);
    uint64_t t = 0;
    SPINED_HIP(hipMemcpyAsync(&t, gc.woff.ptr + waves, 8, hipMemcpyDeviceToHost, s));
    SPINED_HIP(hipStreamSynchronize(s));
    gc.total = t * kRowBlock;
    gc.counted = true;
  }
  const uint64_t per_diag = op.tables.is_real ? 1 : 2;
  const uint64_t n_entries = std::max<uint64_t>(gc.total, 1);
  if (gc.request < 0) {
    size_t free_b = 0, total_b = 0;
    SPINED_HIP(hipMemGetInfo(&free_b, &total_b));
    const uint64_t blocks[3] = {n_entries * 4, gc.in_entry ? 0 : n_entries * 2, b.D * 8 * per_diag};
    uint64_t need = b.D * 2;
    for (uint64_t bytes : blocks) {
      need += bytes;
      if (bytes && pool_bytes(bytes) > 0) free_b += bytes; // a pooled block of this size
    }
    if (free_b < need + kCacheReserve || free_b + reusable < need + reserve) return false;
  }
  try {
    // pooled: a rebuild of the same operator's cache takes the blocks back
    // without a free and a fresh multi-GB mapping
    gc.entries.allocate_pooled(n_entries);
    if (!gc.in_entry) gc.aux.allocate_pooled(n_entries);
    gc.diag.allocate_pooled(b.D * per_diag);
    gc.cnt.allocate(b.D);
  } catch (const Error &) {
    gc.release_entries();
    if (gc.request > 0) throw;
    return false;
  }
  with_fill<METHOD>(c, [&](auto nw, auto bonds) {
    auto fill = [&](auto many) {
      cache_fill_kernel<METHOD, decltype(nw)::value, decltype(bonds)::value, decltype(many)::value>
          <<<g, kRowBlock, 0, s>>>(c.o, c.bd, c.ga, c.ra, c.ix, c.stab, c.D, gc.sched, gc.woff.ptr,
                                   gc.unit_cls.ptr, gc.phases, gc.shift,
                                   op.tables.is_real ? 0 : 1, gc.entries.ptr,
                                   gc.in_entry ? nullptr : gc.aux.ptr, gc.diag.ptr, gc.cnt.ptr);
    };
    if (gc.nclass > gc.phases)
      fill(std::true_type{});
    else
      fill(std::false_type{});
  });
  SPINED_CHECK_LAUNCH();
  gc.built = true;
  return true;
}

template <class R>
void launch_cached(const Operator &op, const Ctx &c, const GatherCache &gc, const void *x, void *y,
                   bool contiguous, hipStream_t s) {
  const unsigned g = static_cast<unsigned>((c.D + kRowBlock - 1) / kRowBlock);
  const CacheArgs ca{gc.woff.ptr, gc.entries.ptr, gc.in_entry ? nullptr : gc.aux.ptr, gc.diag.ptr,
                     gc.cnt.ptr,  gc.cls.ptr,     gc.nclass, gc.shift, gc.imask, gc.cmask};
  const auto *xp = static_cast<const typename R::X *>(x);
  auto *yp = static_cast<typename R::Y *>(y);
  const double2 one = make_double2(gc.one[0], gc.one[1]);
  const int cdiag = op.tables.is_real ? 0 : 1;
  const bool stream_entries = gc.total * 4 > kCacheStreamBytes;
  auto go = [&](auto cm) {
    if (stream_entries)
      matvec_cached_kernel<R, decltype(cm)::value, true><<<g, kRowBlock, 0, s>>>(
          ca, c.rt, c.stab, c.D, xp, yp, gc.sched, contiguous ? 1 : 0, cdiag, one);
    else
      matvec_cached_kernel<R, decltype(cm)::value, false><<<g, kRowBlock, 0, s>>>(
          ca, c.rt, c.stab, c.D, xp, yp, gc.sched, contiguous ? 1 : 0, cdiag, one);
  };
  if (gc.nclass == 1)
    go(std::integral_constant<int, 0>{});
  else if (gc.in_entry && gc.nclass <= kLdsClasses)
    go(std::integral_constant<int, 1>{});
  else
    go(std::integral_constant<int, 2>{});
  SPINED_CHECK_LAUNCH();
}

// Workgroup order of the cached kernels: each XCD a contiguous eighth of the
// rows (xcd_block), or the dispatch order (consecutive waves on different
// XCDs).  Neighbouring rows share gather targets, which an XCD's own L2 then
// serves (contiguous against dispatch order, one FP64 vector: D = 6.3e7 ring
// 4.99 and 5.26 ms, 8x4 torus, D = 9.4e6, 1.80 and 2.12, 5x7, D = 9.3e7, 15.7
// and 18.6, 32-site pyrochlore with four vectors 0.46 and 0.56, 6x6 square
// with its point group 4.44 and 4.42; without symmetries, D = 5.2e6, FP32, 123
// and 161 us).  For FP32 x of a ring the dispatch order is faster at D = 8.6e8
// (85 against 89 ms; 4.05 and 3.93 at 6.3e7).
bool contiguous_rows(const Operator &op, bool f32) {
  return !(op.basis->tables.ring_available && f32);
}

// Low sites of the split row gather for a basis, or -1 where it does not
// apply.  Rule: at least 2^20 rows and 256 rows per group.  26 sites at half
// filling (5.2e6 rows, 635 per group): 85 us against 145 from the gather
// cache, without its memory and its build; 24 sites (1.4e6 rows): 28 against
// 31; 22 sites (3.5e5): 11.5 against 11.5.  Away from half filling groups
// shrink: 28 sites, 7 up (72 per group): 210 us against 23.
constexpr uint64_t kSplitMinRows = uint64_t(1) << 20;
constexpr uint64_t kSplitMinGroup = 256;

int split_low(const Operator &op) {
  const Basis &b = *op.basis;
  const auto &t = op.tables;
  if (b.index_kind != 2 || b.rank_mode != 1 || !t.bonds || !t.is_real) return -1;
  if (static_cast<int>(t.h_bond_sites.size()) > kSplitMaxBonds || b.D < kSplitMinRows) return -1;
  const int l = b.n <= 26 ? 12 : kSplitMaxLow;
  const int nh = b.n - l - (b.tables.has_flip ? 1 : 0);
  if (nh < 1 || nh > kSplitMaxHigh || (b.D >> nh) < kSplitMinGroup) return -1;
  return l;
}

template <class XT, class YT>
void launch_split(const Operator &op, const Ctx &c, const XT *x, YT *y, hipStream_t s) {
  const Basis &b = *op.basis;
  const SplitPlan &p = b.split;
  const size_t lds = (sizeof(uint16_t) << p.l) + sizeof(XT) * p.largest;
  matvec_split_kernel<<<p.nhi, kBlock, lds, s>>>(b.split_args(p), c.bd, op.split_dlow.ptr, x, y);
  SPINED_CHECK_LAUNCH();
}

// Real matvec by the split row gather, unless a gather cache is asked for, the
// orbit kernels are (the cache turned off, other than by the autotuner), or
// several lanes per row.
bool try_split(const MatvecCall &m, const Ctx &c) {
  using VT = VecType;
  const Operator &op = *m.op;
  if (m.xt == VT::C64 || m.xt == VT::C128 || c.lanes != 1) return false;
  if (m.xt == VT::F64 && m.yt != VT::F64) return false;
  const int l = split_low(op);
  if (l < 0 || op.orbit_method() != 0) return false;
  {
    std::lock_guard<std::mutex> lk(op.cache->mu);
    const GatherCache &gc = *op.cache;
    if (gc.request > 0 || gc.built || (gc.request == 0 && !gc.tuning)) return false;
  }
  Basis &b = *op.basis;
  {
    std::lock_guard<std::mutex> lk(b.mu);
    // the tables are not built under stream capture either
    if ((b.split.l < 0 || !op.split_dlow.ptr) && capturing(m.stream)) return false;
    if (b.split.l < 0) {
      if (m.no_alloc) return false;
      build_split(b, b.split, l);
    }
    if (!op.split_dlow.ptr) {
      if (m.no_alloc) return false;
      // published once it is computed
      DeviceBuffer<double> d(size_t(1) << l);
      split_dlow_kernel<<<grid_for(uint64_t(1) << l), kBlock, 0, m.stream>>>(
          b.split_args(b.split), c.bd, d.ptr);
      SPINED_CHECK_LAUNCH();
      SPINED_HIP(hipStreamSynchronize(m.stream));
      op.split_dlow = std::move(d);
    }
  }
  if (m.xt == VT::F64)
    launch_split(op, c, static_cast<const double *>(m.x), static_cast<double *>(m.y), m.stream);
  else if (m.yt == VT::F32)
    launch_split(op, c, static_cast<const float *>(m.x), static_cast<float *>(m.y), m.stream);
  else
    launch_split(op, c, static_cast<const float *>(m.x), static_cast<double *>(m.y), m.stream);
  return true;
}

// Matvec from the gather cache when there is (or can be) one.
template <int METHOD> bool try_cached(const MatvecCall &m, const Ctx &c) {
  GatherCache &gc = *m.op->cache;
  std::lock_guard<std::mutex> lk(gc.mu);
  using VT = VecType;
  const bool known = (m.xt == m.yt) || (m.xt == VT::F32 && m.yt == VT::F64);
  if (!known) return false;
  if (m.no_alloc ? !gc.built : !ensure_cache<METHOD>(*m.op, c, gc, m.stream)) return false;
  if (!gc.recorded && capturing(m.stream)) gc.recorded = true;
  const bool order = contiguous_rows(*m.op, m.xt == VT::F32);
  if (m.xt == VT::F64)
    launch_cached<RealRows<double, double, 1>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else if (m.xt == VT::F32 && m.yt == VT::F32)
    launch_cached<RealRows<float, float, 1>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else if (m.xt == VT::F32)
    launch_cached<RealRows<float, double, 1>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else if (m.xt == VT::C128)
    launch_cached<ComplexRows<double2>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else
    launch_cached<ComplexRows<float2>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  return true;
}

template <int METHOD, int NW, bool BONDS, int K, class XT, class YT>
void launch_block_nw(const Ctx &c, const XT *x, YT *y, hipStream_t s) {
  matvec_block_kernel<METHOD, NW, BONDS, K, XT, YT><<<grid_for(c.D), kBlock, 0, s>>>(
      c.o, c.bd, c.rt, c.ga, c.ra, c.ix, c.stab, c.D, x, y, c.sched);
}

template <int METHOD, int K, class XT, class YT>
void launch_block_k(const Ctx &c, const XT *x, YT *y, hipStream_t s) {
  const int units = c.bonds ? c.bd.nbonds : c.o.ntemplates;
  if (c.bonds && units <= 64)
    launch_block_nw<METHOD, 1, true, K>(c, x, y, s);
  else if (c.bonds && units <= 128)
    launch_block_nw<METHOD, 2, true, K>(c, x, y, s);
  else if (!c.bonds && units <= 64)
    launch_block_nw<METHOD, 1, false, K>(c, x, y, s);
  else if (!c.bonds && units <= 128)
    launch_block_nw<METHOD, 2, false, K>(c, x, y, s);
  else if (!c.bonds && units <= 256)
    launch_block_nw<METHOD, 4, false, K>(c, x, y, s);
  else
    throw Error(LS_NOT_IMPLEMENTED, "block matvec with more than 256 off-diagonal templates");
  SPINED_CHECK_LAUNCH();
}

template <int METHOD, class XT, class YT>
void launch_block(const Ctx &c, int K, const XT *x, YT *y, hipStream_t s) {
  switch (K) {
  case 1: launch_real<METHOD>(c, x, y, s); break;
  case 2: launch_block_k<METHOD, 2>(c, x, y, s); break;
  case 4: launch_block_k<METHOD, 4>(c, x, y, s); break;
  case 8: launch_block_k<METHOD, 8>(c, x, y, s); break;
  default: throw Error(LS_INVALID_ARGUMENT, "block width must be 1, 2, 4 or 8");
  }
}

template <class XT, class YT>
void launch_cached_rows(const MatvecBlockCall &m, const Ctx &c, const GatherCache &gc) {
  const bool order = contiguous_rows(*m.op, false);
  if (m.K == 8)
    launch_cached<RealRows<XT, YT, 8>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else if (m.K == 4)
    launch_cached<RealRows<XT, YT, 4>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else if (m.K == 2)
    launch_cached<RealRows<XT, YT, 2>>(*m.op, c, gc, m.x, m.y, order, m.stream);
  else
    launch_cached<RealRows<XT, YT, 1>>(*m.op, c, gc, m.x, m.y, order, m.stream);
}

// Block matvec from the gather cache when there is (or can be) one.
template <int METHOD> bool try_cached_block(const MatvecBlockCall &m, const Ctx &c) {
  GatherCache &gc = *m.op->cache;
  std::lock_guard<std::mutex> lk(gc.mu);
  using VT = VecType;
  const bool f64 = m.xt == VT::F64 && m.yt == VT::F64;
  const bool f32 = m.xt == VT::F32 && (m.yt == VT::F32 || m.yt == VT::F64);
  if (!f64 && !f32) return false;
  if (!ensure_cache<METHOD>(*m.op, c, gc, m.stream)) return false;
  if (!gc.recorded && capturing(m.stream)) gc.recorded = true;
  if (f64)
    launch_cached_rows<double, double>(m, c, gc);
  else if (m.yt == VT::F32)
    launch_cached_rows<float, float>(m, c, gc);
  else
    launch_cached_rows<float, double>(m, c, gc);
  return true;
}

template <int METHOD> void dispatch_block(const MatvecBlockCall &m, const Ctx &c) {
  hipStream_t s = m.stream;
  using VT = VecType;
  if (m.xt == VT::F64 && m.yt == VT::F64)
    launch_block<METHOD>(c, m.K, static_cast<const double *>(m.x), static_cast<double *>(m.y), s);
  else if (m.xt == VT::F32 && m.yt == VT::F32)
    launch_block<METHOD>(c, m.K, static_cast<const float *>(m.x), static_cast<float *>(m.y), s);
  else if (m.xt == VT::F32 && m.yt == VT::F64)
    launch_block<METHOD>(c, m.K, static_cast<const float *>(m.x), static_cast<double *>(m.y), s);
  else
    throw Error(LS_INVALID_DATATYPE, "block matvec supports real float32/float64 vectors");
}

Ctx make_ctx(const Operator &op, const double *pc, const double *ps) {
  const Basis &b = *op.basis;
  const auto &t = op.tables;
  Ctx c{};
  c.o = op_args(op, pc, ps);
  c.bonds = t.bonds;
  c.bd = BondArgs{t.bond_sites.ptr, t.bond_dp.ptr, t.bond_da.ptr, t.bond_o.ptr, t.bond_flip.ptr,
                  static_cast<int32_t>(t.h_bond_sites.size()),
                  t.nn_ring && b.tables.ring_available ? t.bond_lo.ptr : nullptr,
                  t.nn_identity ? 1 : 0};
  c.rt = RatioArgs{b.tables.div_idx.ptr, b.tables.ratio.ptr, b.tables.nd};
  c.ga = b.tables.generic_args(true);
  c.ra = b.tables.ring_args(true);
  c.ix = b.index_args(t.keeps_weight);
  c.stab = b.stab.ptr;
  c.D = b.D;
  c.sched = op.schedule_built ? op.sched.ptr : nullptr;
  c.lanes = op.lanes_per_row;
  return c;
}

std::mutex g_phase_mu;

const PhaseTable &phase_table(const Basis &b, bool no_alloc = false) {
  // one table per (device, L); small and kept for the process lifetime
  static std::vector<std::pair<std::pair<int, int>, std::unique_ptr<PhaseTable>>> cache;
  std::lock_guard<std::mutex> lk(g_phase_mu);
  const int dev = current_device();
  for (auto &kv : cache)
    if (kv.first.first == dev && kv.first.second == b.tables.L) return *kv.second;
  if (no_alloc)
    throw Error(LS_INVALID_ARGUMENT, "complex phase table not on the device yet: apply the "
                                     "operator once (ls_operator_matmat) before a call that "
                                     "allocates nothing");
  auto t = std::make_unique<PhaseTable>();
  const int L = b.tables.L;
  if (L > (1 << 20)) throw Error(LS_NOT_IMPLEMENTED, "complex sectors with huge periodicity");
  std::vector<double> c(L), s(L);
  for (int p = 0; p < L; ++p) phase_values(p, L, c[p], s[p]);
  t->cos_t.allocate(L);
  t->sin_t.allocate(L);
  copy_in(t->cos_t.ptr, c.data(), 8 * L);
  copy_in(t->sin_t.ptr, s.data(), 8 * L);
  t->L = L;
  cache.emplace_back(std::make_pair(dev, L), std::move(t));
  return *cache.back().second;
}

} // namespace

void launch_matvec(const MatvecCall &m) {
  const Operator &op = *m.op;
  const Basis &b = *op.basis;
  if (m.size != b.D) throw Error(LS_DIMENSION_MISMATCH, "vector length differs from the basis dimension");
  if (b.D == 0) return;
  const bool cplx = m.xt == VecType::C64 || m.xt == VecType::C128;
  if (!cplx && !op.tables.is_real)
    throw Error(LS_INVALID_DATATYPE, "operator is complex; use a complex datatype");
  const double *pc = nullptr, *ps = nullptr;
  if (cplx) {
    const auto &pt = phase_table(b, m.no_alloc);
    pc = pt.cos_t.ptr;
    ps = pt.sin_t.ptr;
  }
  const Ctx c = make_ctx(op, pc, ps);
  if (try_split(m, c)) {
    op.last_path = 2;
    return;
  }
  const bool done = op.orbit_method() == 1 ? try_cached<1>(m, c) : try_cached<0>(m, c);
  op.last_path = done ? 1 : 0;
  if (done) return;
  if (op.orbit_method() == 1)
    dispatch<1>(m, c);
  else
    dispatch<0>(m, c);
}

namespace {
std::mutex g_ops_mu;
std::vector<Operator *> g_ops; // live operators (their gather caches can be reclaimed)
} // namespace

bool prepare_gather_cache(Operator &op, uint64_t reserve, uint64_t block_bytes) {
  if (op.basis->D == 0) return false;
  const Ctx c = make_ctx(op, nullptr, nullptr);
  GatherCache &gc = *op.cache;
  std::lock_guard<std::mutex> lk(gc.mu);
  // an automatic cache is not built where the split row gather serves
  if (gc.request < 0 && !gc.built && c.lanes == 1 && split_low(op) >= 0) return false;
  const uint64_t reusable = pool_bytes(block_bytes);
  return op.orbit_method() == 1 ? ensure_cache<1>(op, c, gc, stream(), true, reserve, reusable)
                                : ensure_cache<0>(op, c, gc, stream(), true, reserve, reusable);
}

void drop_gather_cache_if_built(Operator &op) {
  std::lock_guard<std::mutex> lk(op.cache->mu);
  if (op.cache->built && !op.cache->recorded) op.cache->release_entries();
}

Operator::Operator() {
  std::lock_guard<std::mutex> lk(g_ops_mu);
  g_ops.push_back(this);
}

Operator::~Operator() {
  std::lock_guard<std::mutex> lk(g_ops_mu);
  g_ops.erase(std::remove(g_ops.begin(), g_ops.end(), this), g_ops.end());
}

void drop_gather_cache(Operator &op) {
  std::lock_guard<std::mutex> lk(op.cache->mu);
  op.cache->drop();
}

// Caches in use (their lock held) or recorded in a graph are left alone.
void reclaim_gather_caches(int device) {
  std::lock_guard<std::mutex> lk(g_ops_mu);
  for (Operator *op : g_ops) {
    if (!op->basis || op->basis->device != device) continue;
    GatherCache &gc = *op->cache;
    if (gc.building.load() || !gc.mu.try_lock()) continue;
    if (gc.built && !gc.recorded) gc.release_entries();
    gc.mu.unlock();
  }
}

bool matvec_block_supported(const Operator &op) {
  const auto &t = op.tables;
  if (!t.is_real) return false;
  const int units = t.bonds ? static_cast<int>(t.h_bond_sites.size()) : t.ntemplates;
  return units <= (t.bonds ? 128 : 256);
}

void launch_matvec_block(const MatvecBlockCall &m) {
  const Operator &op = *m.op;
  const Basis &b = *op.basis;
  if (m.size != b.D) throw Error(LS_DIMENSION_MISMATCH, "vector length differs from the basis dimension");
  if (b.D == 0) return;
  if (!matvec_block_supported(op))
    throw Error(LS_NOT_IMPLEMENTED, "block matvec needs a real operator with <= 256 templates");
  const Ctx c = make_ctx(op, nullptr, nullptr);
  const bool done = op.orbit_method() == 1 ? try_cached_block<1>(m, c) : try_cached_block<0>(m, c);
  op.last_path = done ? 1 : 0;
  if (done) return;
  if (op.orbit_method() == 1)
    dispatch_block<1>(m, c);
  else
    dispatch_block<0>(m, c);
}

void launch_cols_to_rows(VecType t, const void *x, uint64_t stride, uint64_t D, int K, void *xr,
                         hipStream_t s) {
  if (D == 0 || K == 0) return;
  if (t == VecType::F64)
    cols_to_rows_kernel<<<grid_for(D), kBlock, 0, s>>>(static_cast<const double *>(x), stride, D,
                                                       K, static_cast<double *>(xr));
  else if (t == VecType::F32)
    cols_to_rows_kernel<<<grid_for(D), kBlock, 0, s>>>(static_cast<const float *>(x), stride, D,
                                                       K, static_cast<float *>(xr));
  else
    throw Error(LS_INVALID_DATATYPE, "real vectors expected");
  SPINED_CHECK_LAUNCH();
}

void launch_rows_to_cols(VecType t, const void *yr, uint64_t D, int K, void *y, uint64_t stride,
                         hipStream_t s) {
  if (D == 0 || K == 0) return;
  if (t == VecType::F64)
    rows_to_cols_kernel<<<grid_for(D), kBlock, 0, s>>>(static_cast<const double *>(yr), D, K,
                                                       static_cast<double *>(y), stride);
  else if (t == VecType::F32)
    rows_to_cols_kernel<<<grid_for(D), kBlock, 0, s>>>(static_cast<const float *>(yr), D, K,
                                                       static_cast<float *>(y), stride);
  else
    throw Error(LS_INVALID_DATATYPE, "real vectors expected");
  SPINED_CHECK_LAUNCH();
}

int block_chunk(uint64_t remaining) { return remaining >= 8 ? 8 : remaining >= 4 ? 4 : remaining >= 2 ? 2 : 1; }

void ensure_schedule(Operator &op) {
  std::lock_guard<std::mutex> lk(op.mu);
  const Basis &b = *op.basis;
  // automatic: bases of at least one tile
  const bool want = op.schedule_request == 1 ||
                    (op.schedule_request < 0 && b.D >= static_cast<uint64_t>(kScheduleTile));
  if (!want || b.D == 0) {
    if (op.schedule_built || op.sched.ptr) drop_gather_cache(op); // cache entries follow the slots
    op.schedule_built = false;
    op.sched.release();
    return;
  }
  if (op.schedule_built) return;
  // An automatic schedule that the cache alone would use comes with it (a first
  // complex matvec of 9,252 rows took 328 us with a schedule, 309 without).
  if (op.schedule_request < 0 && schedule_of_cache(op)) return;
  hipStream_t s = stream();
  drop_gather_cache(op);
  op.sched.allocate(b.D);
  launch_schedule(op, make_ctx(op, nullptr, nullptr), op.sched.ptr, s);
  SPINED_HIP(hipStreamSynchronize(s));
  op.schedule_built = true;
}

namespace {
// <x|y> = sum_r conj(x_r) y_r in FP64 (real types: im = 0).  One partial
// (re, im) per workgroup, then one workgroup sums them in a fixed order.
__device__ inline void load_pair(const float *v, uint64_t r, double &re, double &im) {
  re = v[r];
  im = 0.0;
}
__device__ inline void load_pair(const double *v, uint64_t r, double &re, double &im) {
  re = v[r];
  im = 0.0;
}
__device__ inline void load_pair(const float2 *v, uint64_t r, double &re, double &im) {
  const float2 t = v[r];
  re = t.x;
  im = t.y;
}
__device__ inline void load_pair(const double2 *v, uint64_t r, double &re, double &im) {
  const double2 t = v[r];
  re = t.x;
  im = t.y;
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    vdot_partial_kernel(const T *__restrict__ x, const T *__restrict__ y, uint64_t n,
                        double *__restrict__ partial) {
  __shared__ double lds[2][kBlock / 64];
  double re = 0.0, im = 0.0;
  for (uint64_t r = blockIdx.x * static_cast<uint64_t>(kBlock) + threadIdx.x; r < n;
       r += static_cast<uint64_t>(gridDim.x) * kBlock) {
    double xr, xi, yr, yi;
    load_pair(x, r, xr, xi);
    load_pair(y, r, yr, yi);
    re = fma(xr, yr, fma(xi, yi, re));
    im = fma(xr, yi, fma(-xi, yr, im));
  }
  for (int off = 32; off > 0; off >>= 1) {
    re += __shfl_down(re, off, 64);
    im += __shfl_down(im, off, 64);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    lds[0][wid] = re;
    lds[1][wid] = im;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
    for (int k = 0; k < kBlock / 64; ++k) t += lds[threadIdx.x][k];
    partial[2 * static_cast<uint64_t>(blockIdx.x) + threadIdx.x] = t;
  }
}

__global__ void __launch_bounds__(kBlock)
    vdot_reduce_kernel(const double *__restrict__ partial, unsigned nb, double *__restrict__ out) {
  __shared__ double lds[2][kBlock];
  double re = 0.0, im = 0.0;
  for (unsigned b = threadIdx.x; b < nb; b += kBlock) {
    re += partial[2 * b];
    im += partial[2 * b + 1];
  }
  lds[0][threadIdx.x] = re;
  lds[1][threadIdx.x] = im;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (threadIdx.x < static_cast<unsigned>(off)) {
      lds[0][threadIdx.x] += lds[0][threadIdx.x + off];
      lds[1][threadIdx.x] += lds[1][threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = lds[0][0];
    out[1] = lds[1][0];
  }
}
} // namespace

void launch_vdot(VecType t, const void *x, const void *y, uint64_t n, double *partial,
                 unsigned nb, double *out, hipStream_t s) {
  switch (t) {
  case VecType::F32:
    vdot_partial_kernel<<<nb, kBlock, 0, s>>>(static_cast<const float *>(x),
                                              static_cast<const float *>(y), n, partial);
    break;
  case VecType::F64:
    vdot_partial_kernel<<<nb, kBlock, 0, s>>>(static_cast<const double *>(x),
                                              static_cast<const double *>(y), n, partial);
    break;
  case VecType::C64:
    vdot_partial_kernel<<<nb, kBlock, 0, s>>>(static_cast<const float2 *>(x),
                                              static_cast<const float2 *>(y), n, partial);
    break;
  default:
    vdot_partial_kernel<<<nb, kBlock, 0, s>>>(static_cast<const double2 *>(x),
                                              static_cast<const double2 *>(y), n, partial);
  }
  SPINED_CHECK_LAUNCH();
  vdot_reduce_kernel<<<1, kBlock, 0, s>>>(partial, nb, out);
  SPINED_CHECK_LAUNCH();
}

unsigned vdot_blocks(uint64_t n) { return std::max(1u, std::min(grid_for(n), kVdotMaxBlocks)); }

uint64_t count_offdiag_device(const Operator &op) {
  const Basis &b = *op.basis;
  if (b.D == 0) return 0;
  hipStream_t s = stream();
  const OpArgs o = op_args(op, nullptr, nullptr);
  const auto ga = b.tables.generic_args(true);
  const auto ra = b.tables.ring_args(true);
  const IndexArgs ix = b.index_args(op.tables.keeps_weight);
  const unsigned g = grid_for(b.D);
  DeviceBuffer<unsigned long long> part(g);
  if (op.orbit_method() == 1)
    count_offdiag_kernel<1><<<g, kBlock, 0, s>>>(o, ga, ra, ix, b.D, part.ptr);
  else
    count_offdiag_kernel<0><<<g, kBlock, 0, s>>>(o, ga, ra, ix, b.D, part.ptr);
  SPINED_CHECK_LAUNCH();
  std::vector<unsigned long long> h(g);
  SPINED_HIP(hipMemcpyAsync(h.data(), part.ptr, 8ull * g, hipMemcpyDeviceToHost, s));
  SPINED_HIP(hipStreamSynchronize(s));
  uint64_t tot = 0;
  for (auto v : h) tot += v;
  return tot;
}

} // namespace spined
