// The whole Clenshaw filter of a spin chain in one launch, a column per team.
//
// A team (pf_team.h) owns one column of the block for all K steps.  The rows
// are taken in the reference order, cut into segments of equal high bits (the
// state's bits >= m): inside a segment the low bits run through all m-bit
// strings of one popcount class, so
//  * a bond with both sites in the high bits moves a whole segment onto another
//    one: flippable or not for all its rows at once, and its neighbour rows are
//    the same local indices of the target segment -- a uniform branch and a
//    coalesced load at a uniform offset;
//  * a bond with both sites in the low bits stays in the segment: the neighbour
//    is an LDS read at an offset from a small table of the popcount class (the
//    offset of a zero slot where the two spins are parallel);
//  * a bond across the cut (two, or six in the second form) is a masked load from one other
//    segment.
// Nothing is computed per bond and row: the rank arithmetic of the per-step
// kernels (ops.hip) is in the tables, which are per class, not per row.
//
// Resident form (T blocks hold the column): X and b3 of a lane's rows stay in
// registers and b2 in LDS for the whole filter; only the new vector is written
// (to the XCD's L2) and only the neighbour segments of other blocks are read
// back.  Streaming form (any team size): X, b3 and b2 come from memory every step
// and a wave stages its segment of b2 in LDS.
//
// What bounds it: at L=20 FP64 (54 groups of 128 rows per block) 57 % of the cycles
// are vector instructions (about 60 per 64 rows: two per low bond, the rest
// addresses), then the wait for the other blocks' segments and the barrier (0.9
// us with 32 blocks); the L2 serves 99 % of the reads.  Two rows per lane halve
// the uniform work and the loads (64-row groups: 7.7 us a step).  Measured on
// MI355X, us per step, per-step launches (autotuned) against this kernel:
//   L=14 FP64  1 column     4.8 -> 1.6      L=17 FP64  5 columns   5.3 -> 2.3
//   L=20 FP64  8 columns   15.8 -> 6.7      L=20 FP32  8 columns  10.6 -> 5.4
//   L=22 FP32 16 columns   57.0 -> 44.3     L=22 FP64 16 columns 124.5 -> 107 (streamed)
//   J1-J2 FP64 8 columns: L=18 8.6 -> 5.9, L=20 26.2 -> 14.2; FP32: L=20 15.4 -> 9.6,
//   L=21 28.5 -> 19.3

#include <algorithm>
#include <cstring>
#include <vector>

#include "pf_device.h"
#include "pf_internal.h"
#include "pf_team.h"

namespace pf {


// Waves of a block: 16 with 128 registers, or eight with 256 where the resident FP64
// forms spill otherwise (us a step, 16 and 8 waves: J1-J2 FP64 at L = 16 4.3 and
// 3.0, L = 18 8.6 and 5.9, L = 20 30.0 and 14.3; XXZ FP64 at L = 21 17.2 and 14.8; but
// XXZ FP64 at L = 20 6.8 and 8.4, J1-J2 FP32 at L = 20 9.6 and 12.7, and every
// streamed column slower with eight).
constexpr int team_waves(size_t elem, int NC, int R) {
  return elem == 8 && ((NC == 6 && R > 0) || (NC == 2 && R == 14)) ? 8 : 16;
}

// kGrp consecutive rows of one segment, two per lane.
constexpr uint32_t kGrp = 128;
struct TeamGrp {
  uint32_t i0;    // local index of the first row
  uint32_t tab;   // class table row of local index 0 (even)
  uint32_t seg0;  // row of local index 0
  uint32_t seg;   // segment ordinal
  uint32_t n;     // rows of the group (1..kGrp)
  uint32_t nh;    // entries of the high list
  uint32_t hoff;  // first entry
  uint32_t pos;   // position of local index 0 in a padded vector
};

// A vector in memory is padded: every segment starts at a multiple of kSegAlign
// elements and an element follows its last row, so that a lane's two rows are one
// aligned load (the second row of a group's last lane may be padding: its values
// are never used for a row).  In LDS a segment starts at a multiple of 4 elements
// and the element before it is zero.
constexpr uint32_t kSegAlign = 32;

// The resident form's record of a group, for one division into blocks (words):
//   0        local index of the first row | rows << 12 | local entries << 20 |
//            remote entries << 24
//   1        class table row of local index 0
//   2, 3, 4  row, LDS element and position of local index 0
//   5 ..     NC crossing bonds
//   then     kLocal segments of the block's own LDS, and RN remote segments (a
//            count's bits 2, 1, 0 and 3 say which of the places 0-3, 4-5, 6 and
//            7-14 are in use)
// A crossing bond is active << 31 | the low site's spin that flips << 30 |
// in the own block << 29 | target; a list entry is class << 31 | target: the
// LDS element or the position of the target's local index 0.
constexpr int kLocal = 7;
constexpr int rec_remote(int NC) { return NC == 6 ? 15 : 7; }
constexpr int kRecHead = 5;
constexpr int rec_words(int NC) { return kRecHead + NC + kLocal + rec_remote(NC); }

struct TeamArgs {
  const uint64_t* tab;    // [NQ][tab_rows]: four 16-bit entries each
  const TeamGrp* grp;     // all groups, by row
  const uint32_t* rec;    // resident form: records of the groups
  const uint32_t* hrow;   // high lists: class << 31 | position of the target segment
  const uint32_t* cross;  // [segment][NC]: as in the records, every target in memory
  double w[2];            // J/2 of the two classes of bonds
  uint32_t ccls;          // bit c: class of crossing bond c
  const int32_t* gblk;    // [T + 1]: groups of each block (resident form)
  const int32_t* ulist;   // segments by streaming unit
  const int32_t* uofs;    // [kTeamUnits + 1]
  const int32_t* sgrp;    // [nseg + 1]: first group of each segment
  int32_t ntab, T, order, polytype, ncols, expect, maxseg;
  uint32_t elems;         // padded length of a vector
  const double* diag;     // unscaled, in the team's row order
  const uint32_t* perm;   // the team's row -> reference row (null: the same)
  double scale, shift;
  const double* X;
  int64_t ldx;
  double* Y;
  int64_t ldy;
  char* work;          // slots of slot_bytes: two vectors (with has_x a third, X in T)
  int64_t slot_bytes;  // a multiple of 256
  int32_t nslots, has_x;
  uint32_t tab_lds, rows_lds;  // ends of the class tables and of the form's area in LDS
  TeamCtl* ctl;
  const double* coefs;
  // KPM moments: 1/norm of each column, and the dots [step][2][column][kTeamUnits]
  const double* colscale;
  double* dots;
};

// Rows of the class tables: 2^kTeamLow strings or a whole small sector, each
// class padded to an even count.  The words of a row lie this many rows apart:
// consecutive lanes read consecutive words (rows of 24 contiguous bytes took four
// times the LDS cycles), and the constant stride shares one address register.
constexpr uint32_t tab_rows(int NC) { return NC == 0 ? 2050u : 1048u; }
constexpr int kTeamUnits = 32;  // streaming work lists (dealt to the blocks of a team)

__device__ __forceinline__ TeamGrp cload_grp(const TeamGrp* p) {
  typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
  static_assert(sizeof(TeamGrp) == sizeof(u32x8));
  return __builtin_bit_cast(TeamGrp, cload(reinterpret_cast<const u32x8*>(p)));
}


__device__ __forceinline__ void team_ab(int type, int k, double& alpha, double& beta_k) {
  switch (type) {
    case PF_LEGENDRE: alpha = (2.0 * k + 1) / (k + 1); beta_k = -(double)k / (k + 1); break;
    case PF_HERMITE: alpha = 2.0; beta_k = -2.0 * k; break;
    default: alpha = 2.0; beta_k = -1.0; break;  // Chebyshev
  }
}

// The 16-bit class-table entries of a lane's two rows.
template <int NQ>
struct TeamTab {
  u32x4 q[NQ];
  __device__ __forceinline__ uint32_t at(int row, int e) const {
    return (q[e >> 2][2 * row + ((e >> 1) & 1)] >> (16 * (e & 1))) & 0xFFFFu;
  }
};
template <int NQ, int NC>
__device__ __forceinline__ TeamTab<NQ> tab_of(uint32_t at) {  // LDS byte offset of word 0
  TeamTab<NQ> t;
#pragma unroll
  for (int k = 0; k < NQ; ++k) t.q[k] = lread<u32x4>(at + 8u * tab_rows(NC) * k);
  return t;
}

template <typename T>
using pair_t = typename VT<T, 2>::t;

// Weighted sum over the bonds of up to two classes of couplings; UNI: one class,
// weighted once at the end.
template <typename T, bool UNI>
struct BondSum {
  T wa, wb;  // scaled J/2 of the classes (uniform)
  pair_t<T> s = (pair_t<T>)(T)0;
  __device__ __forceinline__ BondSum(T a, T b) : wa(a), wb(b) {}
  __device__ __forceinline__ void add(uint32_t second, pair_t<T> v) {  // uniform class
    if constexpr (UNI) s += v;
    else s += (second ? wb : wa) * v;
  }
  __device__ __forceinline__ void add(uint32_t second, int row, T v) {
    if constexpr (UNI) s[row] += v;
    else s[row] += (second ? wb : wa) * v;
  }
  __device__ __forceinline__ pair_t<T> value() const {
    if constexpr (UNI) return wa * s;
    else return s;
  }
};
// Low slots: of the first class, of the second.
constexpr int low_first(int NQ, int NC) { return NC == 0 ? 12 : 9; }
constexpr int low_second(int NQ, int NC) { return NQ == 3 ? 0 : NC == 0 ? 12 : 8; }

// All N values are loaded before any is used: without this the compiler sinks
// each LDS read to its addition and waits for every one of them.
template <typename V, int N>
__device__ __forceinline__ void keep(V (&v)[N]) {
  static_assert(N == 2 || N == 4 || N == 8 || N == 9 || N == 12);
  if constexpr (N == 2)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]));
  if constexpr (N == 4)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
  if constexpr (N == 8)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
  if constexpr (N == 9)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(v[8]));
  if constexpr (N == 12)
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]));
}
template <typename T, int N>
__device__ __forceinline__ T low_part(const uint32_t (&at)[N]) {
  T v[N];
#pragma unroll
  for (int e = 0; e < N; ++e) v[e] = lread<T>(at[e]);
  keep(v);
  T s = (N & 1) ? v[N - 1] : v[N - 2] + v[N - 1];
#pragma unroll
  for (int e = 0; e + 1 < N - 1; e += 2) s += v[e] + v[e + 1];
  return s;
}

// Bonds inside the low sites: LDS reads at the class table's offsets from the
// segment's zero slot `rows`.
template <typename T, int NQ, int NC, bool UNI>
__device__ __forceinline__ void low_sum(BondSum<T, UNI>& s, const TeamTab<NQ>& tab, uint32_t rows) {
  constexpr int N0 = low_first(NQ, NC), N1 = low_second(NQ, NC);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    uint32_t at[N0];
#pragma unroll
    for (int e = 0; e < N0; ++e) at[e] = rows + tab.at(r, e);
    s.add(0u, r, low_part<T>(at));
    if constexpr (N1 > 0) {
      uint32_t au[N1];
#pragma unroll
      for (int e = 0; e < N1; ++e) au[e] = rows + tab.at(r, N0 + e);
      s.add(1u, r, low_part<T>(au));
    }
  }
}

// Byte offset from the target's zero slot (the element before its local index 0)
// of a crossing bond e; t: the row's class-table entry, the flipped low state's
// offset | the low site's spin << 15.  `none` where the bond does not flip: 0
// reads the zero slot in LDS, an offset past the records reads zero from memory
// without an access.
__device__ __forceinline__ uint32_t cross_ofs(uint32_t t, uint32_t e, uint32_t none) {
  return ((e ^ (t << 15)) & 0x40000000u) == 0u ? t & 0x7FFFu : none;
}

// Streaming form: every bond that leaves the segment is a load from memory.
template <typename T, int NQ, int NC, bool UNI>
__device__ __forceinline__ void outer_sum(BondSum<T, UNI>& s, const TeamArgs& A, const TeamGrp& g,
                                          uint32_t vo, const TeamTab<NQ>& tab, uint32_t bytes,
                                          __amdgpu_buffer_rsrc_t b2) {
  constexpr uint32_t sz = sizeof(T);
  typedef pair_t<T> pt;
  T xc[NC][2];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const uint32_t e = cload(A.cross + (size_t)g.seg * NC + c);
    const uint32_t to = (e >> 31) ? ((e & 0x1FFFFFFFu) - 1u) * sz : bytes;
#pragma unroll
    for (int r = 0; r < 2; ++r)
      xc[c][r] = bload<T>(b2, cross_ofs(tab.at(r, 4 * NQ - 1 - c), e, bytes), to);
  }
  uint32_t h = 0;
  for (; h + 4 <= g.nh; h += 4) {  // uniform
    const u32x4 hr = cload(reinterpret_cast<const u32x4*>(A.hrow + g.hoff + h));
    pt y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = bload<pt>(b2, vo, (hr[k] & 0x7FFFFFFFu) * sz);
#pragma unroll
    for (int k = 0; k < 4; ++k) s.add(hr[k] >> 31, y[k]);
  }
  if (h < g.nh) {
    const u32x4 hr = cload(reinterpret_cast<const u32x4*>(A.hrow + g.hoff + h));
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (h + k < g.nh) s.add(hr[k] >> 31, bload<pt>(b2, vo, (hr[k] & 0x7FFFFFFFu) * sz));
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    s.add((A.ccls >> c) & 1u, 0, xc[c][0]);
    s.add((A.ccls >> c) & 1u, 1, xc[c][1]);
  }
}

// A lane's two rows of the caller's column (row + 1 only if `two`, else 0).
template <typename T>
__device__ __forceinline__ pair_t<T> x_pair(const TeamArgs& A, const double* X, int64_t row,
                                            bool two, double f = 1.0) {
  pair_t<T> v;
  v[0] = (T)(X[A.perm ? A.perm[row] : row] * f);
  v[1] = two ? (T)(X[A.perm ? A.perm[row + 1] : row + 1] * f) : (T)0;
  return v;
}
template <typename T>
__device__ __forceinline__ void y_pair(const TeamArgs& A, double* Y, int64_t row, bool two,
                                       pair_t<T> v) {
  Y[A.perm ? A.perm[row] : row] = (double)v[0];
  if (two) Y[A.perm ? A.perm[row + 1] : row + 1] = (double)v[1];
}
// Their diagonal elements, scaled.
template <typename T>
__device__ __forceinline__ pair_t<T> d_pair(const TeamArgs& A, int64_t row, bool two) {
  pair_t<T> v;
  v[0] = (T)((A.diag[row] - A.shift) * A.scale);
  v[1] = (T)(((two ? A.diag[row + 1] : 0.0) - A.shift) * A.scale);
  return v;
}

template <typename T>
struct TeamCoef {
  T cx, ch, cb;
};
// Factors of step k: out = cx X + ch H~ b2 + cb b3 (ch carries the scale of the
// off-diagonal sum separately).
// The KPM recurrence T_j = 2 H~ T_{j-1} - T_{j-2} (T_1 = H~ T_0) takes the same
// steps with no X term.
template <typename T, bool KPM>
__device__ __forceinline__ TeamCoef<T> team_coef(const TeamArgs& A, int j) {
  if constexpr (KPM) return {(T)0, j == 1 ? (T)1 : (T)2, j == 1 ? (T)0 : (T)-1};
  const int k = A.order - j;
  double alpha, beta, dummy;
  const double ck = cload(A.coefs + k);
  if (k >= 1) {
    team_ab(A.polytype, k, alpha, dummy);
    team_ab(A.polytype, k + 1, dummy, beta);
  } else {
    team_ab(A.polytype, 1, dummy, beta);
    alpha = A.polytype == PF_HERMITE ? 2.0 : 1.0;  // phi_1 (phi_0 = 1)
  }
  return {(T)ck, (T)alpha, (T)beta};
}

// KPM dots of one step.  FP64: <T_{j-1}, T_{j-1}> and <T_j, T_{j-1}>, from which
// mu_{2j-2} and mu_{2j-1} follow (2 T_m T_n = T_{m+n} + T_{m-n}): half the steps of
// the direct form.  FP32: <x, x> and <x, T_j>, because there the identity's
// rounding can exceed the direct form's.
struct TeamDots {
  double a = 0.0, b = 0.0;
  template <typename T>
  __device__ __forceinline__ void add(pair_t<T> x, pair_t<T> own, pair_t<T> o, bool ok, bool two) {
    if constexpr (sizeof(T) == 8) x = own;
    const double a0 = (double)x[0] * (double)x[0], b0 = (double)x[0] * (double)o[0];
    const double a1 = (double)x[1] * (double)x[1], b1 = (double)x[1] * (double)o[1];
    a += ok ? a0 : 0.0;
    b += ok ? b0 : 0.0;
    a += two ? a1 : 0.0;
    b += two ? b1 : 0.0;
  }
  // the wave's sums to LDS
  __device__ __forceinline__ void park(TeamShared& sh) {
    for (int o = 32; o > 0; o >>= 1) {
      a += __shfl_down(a, o, 64);
      b += __shfl_down(b, o, 64);
    }
    if ((threadIdx.x & 63u) == 0) {
      sh.red[2 * (threadIdx.x >> 6)] = a;
      sh.red[2 * (threadIdx.x >> 6) + 1] = b;
    }
  }
};
// The block's sums of step j (all waves parked): written by two threads of wave 1.
template <int W>
__device__ __forceinline__ void team_dots_out(const TeamArgs& A, const TeamShared& sh, int j,
                                              int col, uint32_t idx) {
  if (threadIdx.x >= 64u && threadIdx.x < 66u) {
    const uint32_t w = threadIdx.x - 64u;
    double t = 0.0;
    for (int i = 0; i < W; ++i) t += sh.red[2 * i + w];
    A.dots[((int64_t)(2 * (j - 1) + (int)w) * A.ncols + col) * kTeamUnits + idx] = t;
  }
}

// The streaming form of one column (any team size, any D).
template <typename T, int NQ, int NC, bool UNI, bool KPM, int W>
__device__ bool stream_column(const TeamArgs& A, TeamShared& sh, TeamPlace& me, int col,
                              char* slot) {
  constexpr uint32_t sz = sizeof(T);
  typedef pair_t<T> pt;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = uni(threadIdx.x >> 6);
  const uint32_t bytes = A.elems * sz;
  // a wave's copy of its segment: zero slot at element 3, rows from 4
  const uint32_t rows = A.tab_lds + (wave * (uint32_t)A.maxseg + 4u) * sz;
  const T wa = (T)(A.w[0] * A.scale), wb = (T)(A.w[1] * A.scale);
  const double* X = A.X + (int64_t)col * A.ldx;
  double* Y = A.Y + (int64_t)col * A.ldy;
  const __amdgpu_buffer_rsrc_t x32 = rsrc_of(slot + 2 * (int64_t)bytes, bytes);
  lwrite<T>(rows - sz, (T)0);
  const int steps = A.order;
  const double fx = KPM ? A.colscale[col] : 1.0;
  TeamDots dots;
  // the first vector (c_K X, or T_0 = x), then the steps 1 .. order
  for (int j = 0; j <= steps; ++j) {
    const bool first = j == 0;
    const TeamCoef<T> f = first && KPM ? TeamCoef<T>{(T)1, (T)0, (T)0} : team_coef<T, KPM>(A, j);
    const int par = j & 1;
    const __amdgpu_buffer_rsrc_t out = rsrc_of(slot + par * (int64_t)bytes, bytes);  // b3, then b1
    const __amdgpu_buffer_rsrc_t b2 = rsrc_of(slot + (1 - par) * (int64_t)bytes, bytes);
    const bool hasB3 = j >= 2;
    for (int u = (int)me.idx; u < kTeamUnits; u += (int)me.n) {
      const int s1 = cload(A.uofs + u + 1);
      int at = cload(A.uofs + u);
      // waves take the unit's segments one by one
      while (true) {
        uint32_t mine = 0;
        if (lane == 0) mine = atomicAdd(&sh.seg, 1u);
        const int si = at + (int)uni(mine);
        if (si >= s1) break;
        const int seg = cload(A.ulist + si);
        const int g0 = cload(A.sgrp + seg), g1 = cload(A.sgrp + seg + 1);
        if (!first)
          for (int gi = g0; gi < g1; ++gi) {
            const TeamGrp g = cload_grp(A.grp + gi);
            const uint32_t vo = (g.i0 + 2u * lane) * sz;
            if (2u * lane < g.n) lwrite<pt>(rows + vo, bload<pt>(b2, vo, g.pos * sz));
          }
        __builtin_amdgcn_wave_barrier();
        for (int gi = g0; gi < g1; ++gi) {
          const TeamGrp g = cload_grp(A.grp + gi);
          const uint32_t last = (g.n - 1u) / 2u, ln = lane < last ? lane : last;
          const bool ok = lane <= last, two = 2u * ln + 1u < g.n;
          const uint32_t i = g.i0 + 2u * ln, vo = i * sz;
          const int64_t row = (int64_t)g.seg0 + i;
          pt x;
          if (first || !A.has_x) x = x_pair<T>(A, X, row, two, fx);
          else x = bload<pt>(x32, vo, g.pos * sz);
          pt o = f.cx * x;
          if (first) {
            if (A.has_x && ok) bstore<pt>(x, x32, vo, g.pos * sz);
          } else {
            const pt b3 = hasB3 ? bload<pt>(out, vo, g.pos * sz) : (pt)(T)0;
            const pt d = d_pair<T>(A, row, two);
            const TeamTab<NQ> tab = tab_of<NQ, NC>((g.tab + i) * 8u);
            BondSum<T, UNI> bs(wa, wb);
            low_sum<T, NQ, NC, UNI>(bs, tab, rows - sz);
            outer_sum<T, NQ, NC, UNI>(bs, A, g, vo, tab, bytes, b2);
            const pt hs = bs.value();
            const pt own = lread<pt>(rows + vo);
            o += f.ch * (d * own + hs);
            o += f.cb * b3;
            if constexpr (KPM) dots.add<T>(x, own, o, ok, ok && two);
          }
          if (j < steps) {
            bstore<pt>(o, out, ok ? vo : bytes, g.pos * sz);
          } else if (!KPM && ok) {
            y_pair<T>(A, Y, row, two, o);
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
      if (u + (int)me.n < kTeamUnits) {  // more than one unit: restart the counter
        __syncthreads();
        if (threadIdx.x == 0) sh.seg = 0;
        __syncthreads();
      }
    }
    if (KPM && !first) {
      dots.park(sh);
      dots = TeamDots{};
    }
    if (j < steps && !team_step_end(A.ctl, sh, me, false, [&] {
          if (KPM && !first) team_dots_out<W>(A, sh, j, col, me.idx);
        }))
      return false;
  }
  if constexpr (KPM) {
    __syncthreads();
    team_dots_out<W>(A, sh, steps, col, me.idx);
  }
  return true;
}

// The record of a group as the step loop uses it, in LDS with every offset in
// bytes.  A wave reads it as one vector (a word per lane) one batch ahead and
// takes the words by readlane: no scalar-cache misses in the step loop.
enum { kRecI0, kRecCnt, kRecTab, kRecZero, kRecPos, kRecRow, kRecCls, kRecCross };
constexpr int lrec_words(int NC) { return kRecCross + NC + kLocal + rec_remote(NC); }
struct LRec {
  uint32_t v;  // lane l: word l
  __device__ __forceinline__ uint32_t operator[](int k) const {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, k);
  }
};
template <typename T, int NC>
__device__ __forceinline__ uint32_t lrec_word(const uint32_t* rec, int k, uint32_t base,
                                              uint32_t elems) {
  constexpr uint32_t sz = sizeof(T);
  const uint32_t* from = rec + kRecHead + NC;  // local, remote
  const uint32_t i0 = rec[0] & 0xFFFu;
  switch (k) {
    case kRecI0: return i0 * sz;
    case kRecCnt: return rec[0] >> 12;  // n | local << 8 | remote << 12
    case kRecTab: return (rec[1] + i0) * 8u;
    case kRecZero: return base + (rec[3] - 1u) * sz;
    case kRecPos: return rec[4] * sz;
    case kRecRow: return rec[2] + i0;
    case kRecCls: {
      uint32_t c = 0;
      for (int j = 0; j < kLocal + rec_remote(NC); ++j) c |= (from[j] >> 31) << j;
      return c;
    }
    default: break;
  }
  if (k < kRecCross + NC) {  // the target's zero slot, in LDS or memory
    const uint32_t e = rec[kRecHead + k - kRecCross], to = e & 0x1FFFFFFFu;
    if (!(e >> 31)) return elems * sz;  // no such bond: past the records
    return (e & 0xE0000000u) | (((e & 0x20000000u) ? base : 0u) + (to - 1u) * sz);
  }
  const uint32_t to = from[k - kRecCross - NC] & 0x7FFFFFFFu;
  return (k < kRecCross + NC + kLocal ? base : 0u) + to * sz;
}

// The resident form: block `idx` of the team's T holds groups gblk[idx] ..
// gblk[idx+1] (whole segments), wave w every 16th of them, at most R; their X,
// b3 and (while they fit) diagonal in registers, b2 in LDS with a zero slot
// before each segment.  Segments of the same block are read from LDS, the others
// from memory, all of a group's loads before its first sum.  LDS: class tables,
// records, rows, spare elements.
template <typename T, int NQ, int NC, bool UNI, bool KPM, int R>
__device__ __forceinline__ bool resident_column(const TeamArgs& A, TeamShared& sh, TeamPlace& me,
                                                int col, char* slot) {
  constexpr uint32_t sz = sizeof(T);
  typedef pair_t<T> pt;
  constexpr int W = team_waves(sizeof(T), NC, R);
  constexpr bool kDiagReg = R * W * sizeof(T) <= 56 * 16;
  constexpr int RN = rec_remote(NC);
  constexpr int LW = lrec_words(NC);
  const uint32_t lane = threadIdx.x & 63u;
  const int wave = (int)uni(threadIdx.x >> 6);
  const int idx = (int)uni(me.idx);
  const int ga = cload(A.gblk + idx), ge = cload(A.gblk + idx + 1);
  const uint32_t bytes = A.elems * sz;
  const T wa = (T)(A.w[0] * A.scale), wb = (T)(A.w[1] * A.scale);
  const double* X = A.X + (int64_t)col * A.ldx;
  double* Y = A.Y + (int64_t)col * A.ldy;
  const int mine = ge - ga - wave;  // groups r with 16 r < mine
  int left = mine;
  auto have = [&](int r) { return r * W < left; };  // uniform
  const uint32_t recs =
      A.tab_lds + ((uint32_t)wave * LW + (lane < (uint32_t)LW ? lane : LW - 1u)) * 4u;
  auto rec_at = [&](int r) { return LRec{lread<uint32_t>(recs + (uint32_t)(r * W * LW * 4))}; };
  // the lane (the last pair's for lanes past the end), and whether it is one
  auto last_of = [&](const LRec& c) { return ((c[kRecCnt] & 0xFFu) - 1u) >> 1; };
  const uint32_t spare = A.rows_lds - 4u * sz;  // takes the writes of lanes without a row
  pt x[R], p[R], d[kDiagReg ? R : 1];
  const T fk = KPM ? (T)1 : (T)cload(A.coefs + A.order);
  const double fx = KPM ? A.colscale[col] : 1.0;
  __amdgpu_buffer_rsrc_t out = rsrc_of(slot, bytes);
  __amdgpu_buffer_rsrc_t in = rsrc_of(slot + bytes, bytes);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    x[r] = p[r] = (pt)(T)0;
    if constexpr (kDiagReg) d[r] = (pt)(T)0;
    if (have(r)) {
      const LRec c = rec_at(r);
      const uint32_t last = last_of(c), ln = lane < last ? lane : last;
      const int64_t row = (int64_t)c[kRecRow] + 2u * ln;
      const bool two = 2u * ln + 1u < (c[kRecCnt] & 0xFFu);
      x[r] = x_pair<T>(A, X, row, two, fx);
      if constexpr (kDiagReg) d[r] = d_pair<T>(A, row, two);
      p[r] = fk * x[r];  // (the new vector; it moves to LDS behind the barrier)
      if constexpr (NC > 0)
        bstore<pt>(p[r], out, lane <= last ? c[kRecI0] + 2u * ln * sz : bytes, c[kRecPos]);
    }
  }
  TeamDots dots;
  for (int j = 1; j <= A.order; ++j) {
    const bool last_step = j == A.order;
    const TeamCoef<T> f = team_coef<T, KPM>(A, j);
    int zero;  // (opaque: the R conditions are not hoisted into saved masks)
    asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
    left = mine + zero;
    if (!team_step_end(A.ctl, sh, me, false, [&] {
          // p holds the new vector, LDS still the one before: exchange them
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (have(r)) {
              const LRec c = rec_at(r);
              const uint32_t at = lane <= last_of(c)
                                      ? c[kRecZero] + sz + c[kRecI0] + 2u * lane * sz : spare;
              const pt t = lread<pt>(at);
              lwrite<pt>(at, p[r]);
              p[r] = j == 1 ? (pt)(T)0 : t;  // (LDS is another column's then)
            }
          if (KPM && j > 1) team_dots_out<W>(A, sh, j - 1, col, me.idx);
        }))
      return false;
    const __amdgpu_buffer_rsrc_t t = in;
    in = out;
    out = t;
    LRec nx{};
    if (have(0)) nx = rec_at(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!have(r)) continue;
      const LRec c = nx;
      const uint32_t cnt = c[kRecCnt], rows = c[kRecZero];
      const uint32_t last = last_of(c), ln = lane < last ? lane : last;
      const uint32_t vo = c[kRecI0] + 2u * ln * sz;
      const uint32_t nr = cnt >> 12, nl = cnt >> 8;  // (single bits are tested)
      pt xr[RN];
      T xc[NC < 1 ? 1 : NC][2];
      pt dg;
      if constexpr (NC > 0) {
        auto load = [&](int s) { xr[s] = bload<pt>(in, vo, c[kRecCross + NC + kLocal + s]); };
        if constexpr (RN == 15)
          if (nr & 8u) {
#pragma unroll
            for (int s = 7; s < 15; ++s) load(s);
          }
        if (nr & 4u) {
#pragma unroll
          for (int s = 0; s < 4; ++s) load(s);
        }
        if (nr & 2u) {
          load(4);
          load(5);
        }
        if (nr & 1u) load(6);
      }
      if constexpr (!kDiagReg) dg = d_pair<T>(A, (int64_t)c[kRecRow] + 2u * ln, 2u * ln + 1u < (cnt & 0xFFu));
      else dg = d[r];
      const TeamTab<NQ> tab = tab_of<NQ, NC>(c[kRecTab] + 16u * ln);
      if (r + 1 < R && have(r + 1)) nx = rec_at(r + 1);
      if constexpr (NC > 0) {
#pragma unroll
        for (int x2 = 0; x2 < NC; ++x2) {
          const uint32_t e = c[kRecCross + x2], to = e & 0x1FFFFFFFu;
          const uint32_t t0 = tab.at(0, 4 * NQ - 1 - x2), t1 = tab.at(1, 4 * NQ - 1 - x2);
          if (e & 0x20000000u) {  // uniform: the target is in this block
            xc[x2][0] = lread<T>(to + cross_ofs(t0, e, 0u));
            xc[x2][1] = lread<T>(to + cross_ofs(t1, e, 0u));
          } else {
            xc[x2][0] = bload<T>(in, cross_ofs(t0, e, bytes), to);
            xc[x2][1] = bload<T>(in, cross_ofs(t1, e, bytes), to);
          }
        }
      }
      BondSum<T, UNI> bs(wa, wb);
      low_sum<T, NQ, NC, UNI>(bs, tab, rows);
      const pt own = lread<pt>(rows + sz + vo);
      if constexpr (NC > 0) {
        auto at = [&](int s) { return lread<pt>(c[kRecCross + NC + s] + vo); };
        auto add = [&](int s, pt v) { bs.add(UNI ? 0u : (c[kRecCls] >> s) & 1u, v); };
        if (nl & 4u) {
          pt v[4] = {at(0), at(1), at(2), at(3)};
          keep(v);
#pragma unroll
          for (int s = 0; s < 4; ++s) add(s, v[s]);
        }
        if (nl & 2u) {
          pt v[2] = {at(4), at(5)};
          keep(v);
          add(4, v[0]);
          add(5, v[1]);
        }
        if (nl & 1u) add(6, at(6));
        if constexpr (RN == 15)
          if (nr & 8u) {
#pragma unroll
            for (int s = 7; s < 15; ++s) add(kLocal + s, xr[s]);
          }
        if (nr & 4u) {
#pragma unroll
          for (int s = 0; s < 4; ++s) add(kLocal + s, xr[s]);
        }
        if (nr & 2u) {
          add(kLocal + 4, xr[4]);
          add(kLocal + 5, xr[5]);
        }
        if (nr & 1u) add(kLocal + 6, xr[6]);
#pragma unroll
        for (int x2 = 0; x2 < NC; ++x2) {
          bs.add((A.ccls >> x2) & 1u, 0, xc[x2][0]);
          bs.add((A.ccls >> x2) & 1u, 1, xc[x2][1]);
        }
      }
      const pt hs = bs.value();
      pt o = f.ch * (dg * own + hs);
      if constexpr (!KPM) o += f.cx * x[r];
      o += f.cb * p[r];
      p[r] = o;
      if constexpr (KPM)
        dots.add<T>(x[r], own, o, lane <= last, lane <= last && 2u * ln + 1u < (cnt & 0xFFu));
      if (!last_step) {
        if constexpr (NC > 0) bstore<pt>(o, out, lane <= last ? vo : bytes, c[kRecPos]);
      } else if (!KPM && lane <= last) {
        y_pair<T>(A, Y, (int64_t)c[kRecRow] + 2u * ln, 2u * ln + 1u < (cnt & 0xFFu), o);
      }
    }
    if constexpr (KPM) {
      dots.park(sh);
      dots = TeamDots{};
    }
  }
  if constexpr (KPM) {
    __syncthreads();
    team_dots_out<W>(A, sh, A.order, col, me.idx);
  }
  return true;
}

// R = 0: the streaming form only.  Dynamic LDS: class tables (at offset 0, so
// that offsets need no base), then the form's own area, then TeamShared.
template <typename T, int NQ, int NC, bool UNI, bool KPM, int R>
__global__ __launch_bounds__(64 * team_waves(sizeof(T), NC, R)) void
chain_team_kernel(const TeamArgs A) {
  constexpr int W = team_waves(sizeof(T), NC, R);
  TeamShared& sh = *reinterpret_cast<TeamShared*>(team_lds + A.rows_lds);
  // (team_enter in line: as a call, even inlined, the R = 4 form spills 34 registers
  // instead of 18 and a step at L = 20 takes 4 % longer)
  TeamPlace me{};
  if (threadIdx.x == 0) {
    sh.ok = team_join(A.ctl, (uint32_t)A.expect, (uint32_t)A.T, me);
    if (sh.ok) {
      sh.idx = me.idx;
      sh.n = me.n;
      sh.bar = (uint32_t)(me.bar - A.ctl->bar);
      if (me.idx == 0) {  // the team's work space
        sh.slot = team_add(&A.ctl->slots, 1u);
        if (me.n > 1) team_store(&me.bar->slot, sh.slot);
      }
    }
  }
  for (uint32_t t = threadIdx.x * 8u; t < A.tab_lds; t += W * 64u * 8u)
    lwrite<uint64_t>(t, A.tab[t / 8u]);
  __syncthreads();
  if (!uni(sh.ok)) return;
  // (every thread: wave 0 polls the barrier with all its lanes)
  me.idx = uni(sh.idx);
  me.n = uni(sh.n);
  me.bar = &A.ctl->bar[uni(sh.bar)];
  me.passed = 0;
  if constexpr (R > 0) {
    if (me.n == (uint32_t)A.T) {  // records; rows to zero (the zero slots stay)
      constexpr int LW = lrec_words(NC);
      const int ga = A.gblk[me.idx], ge = A.gblk[me.idx + 1];
      const uint32_t rows = A.tab_lds + (uint32_t)((ge - ga) * LW * 4 + 31) / 32u * 32u;
      const uint32_t* rec = A.rec + (int64_t)ga * rec_words(NC);
      // the block's first segment starts at element 4 of the rows
      const uint32_t base = ga < ge ? rows + (4u - rec[3]) * (uint32_t)sizeof(T) : 0u;
      for (int t = threadIdx.x; t < (ge - ga) * LW; t += W * 64)
        lwrite<uint32_t>(A.tab_lds + (uint32_t)t * 4u,
                         lrec_word<T, NC>(rec + (t / LW) * rec_words(NC), t % LW, base, A.elems));
      for (uint32_t t = rows + threadIdx.x * 4u; t < A.rows_lds; t += W * 64u * 4u)
        lwrite<uint32_t>(t, 0u);
    }
  }
  if (!team_step_end(A.ctl, sh, me, false, [] {})) return;
  if (threadIdx.x == 0 && me.n > 1) sh.slot = team_load(&me.bar->slot);
  __syncthreads();
  const uint32_t slot = uni(sh.slot);
  if (slot >= (uint32_t)A.nslots) return;  // (uniform over the team)
  char* work = A.work + (int64_t)slot * A.slot_bytes;
  while (true) {
    if (!team_next(A.ctl, sh, me)) return;
    const uint32_t col = uni(sh.job);
    if (col >= (uint32_t)A.ncols) return;
    bool ok;
    if constexpr (R > 0 && NC == 0) {
      ok = resident_column<T, NQ, NC, UNI, KPM, R>(A, sh, me, (int)col, work);
    } else if constexpr (R > 0) {
      ok = me.n == (uint32_t)A.T ? resident_column<T, NQ, NC, UNI, KPM, R>(A, sh, me, (int)col, work)
                                 : stream_column<T, NQ, NC, UNI, KPM, W>(A, sh, me, (int)col, work);
    } else {
      ok = stream_column<T, NQ, NC, UNI, KPM, W>(A, sh, me, (int)col, work);
    }
    if (!ok) return;
    if (threadIdx.x == 0 && me.idx == 0) (void)team_add(&A.ctl->done, 1u);
  }
}

// Control words to zero and the coefficients into device memory, by value: a
// launch captured in a graph carries its own coefficients.
constexpr int kCoefChunk = 448;
struct TeamCoefs {
  double c[kCoefChunk];
};
__global__ void team_begin_kernel(TeamCtl* ctl, double* dst, int at, int n, const TeamCoefs c) {
  if (ctl) {
    uint4* w = reinterpret_cast<uint4*>(ctl);
    for (uint32_t t = threadIdx.x; t < sizeof(TeamCtl) / 16; t += blockDim.x) w[t] = uint4{0, 0, 0, 0};
  }
  for (int t = threadIdx.x; t < n; t += blockDim.x) dst[at + t] = c.c[t];
}
// Every column done, or NaN everywhere.
__global__ void team_end_kernel(const TeamCtl* ctl, uint32_t jobs, double* Y, int64_t ldy,
                                int64_t D) {
  if (ctl->done == jobs && ctl->abort == 0) return;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < D;
       r += (int64_t)gridDim.x * blockDim.x)
    for (uint32_t c = 0; c < jobs; ++c) Y[r + (int64_t)c * ldy] = __builtin_nan("");
}

__global__ void team_permute_kernel(const uint32_t* __restrict__ perm,
                                    const double* __restrict__ src, int64_t D,
                                    double* __restrict__ dst) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < D) dst[r] = src[perm[r]];
}

// ------------------------------------------------------------- tables
// Device tables of one chain (built once with the operator) and the host-side
// figures the plan needs.
struct TeamTables {
  int NQ = 0, NC = 0, uni = 0, ntab = 0, nseg = 0, ngrp = 0, maxseg = 0;
  int64_t elems = 0;  // padded length of a vector
  double w[2] = {0.0, 0.0};
  uint32_t ccls = 0;
  void* dev = nullptr;  // one allocation
  // per element type (0: FP64, 1: FP32)
  const uint64_t* tab[2] = {};
  const TeamGrp* grp = nullptr;
  const uint32_t* hrow = nullptr;
  const uint32_t* cross = nullptr;
  const int32_t* ulist = nullptr;
  const int32_t* uofs = nullptr;
  const int32_t* sgrp = nullptr;
  const uint32_t* perm = nullptr;  // folded order: team row -> reference row
  const double* diag = nullptr;    // and the diagonal in that order
  // resident plans for T = 1 << lt blocks: group ranges, most groups and most
  // LDS elements of a block
  const int32_t* gblk[6] = {};
  const uint32_t* rec[6] = {};  // null: some group has too many neighbour segments
  int maxgrp[6] = {}, maxel[6] = {};
};

void team_destroy(TeamTables* t) {
  if (!t) return;
  if (t->dev) (void)hipFree(t->dev);
  delete t;
}

// Low bits of the cut: a whole small sector is one segment (one block, all
// neighbours in LDS); else 10, so that the class tables take 24 KB of LDS (48
// with second neighbours), the largest segment is 252 rows (88 % of the lanes
// of its groups hold a row) and half of the bonds of a 20-site chain are uniform.
constexpr int kTeamLow = 10;
constexpr int64_t kTeamTinyD = 2048;

// Null when the chain does not fit the team kernels (too many bonds across the
// cut or inside the low sites).
TeamTables* team_build(const ChainParams& ref, const uint32_t* C, const uint32_t* states,
                       const double* diag_dev) {
  if (ref.D < 2 || ref.nb < 1 || ref.D >= ((int64_t)1 << 24)) return nullptr;
  const int L = ref.L, Lup = ref.Lup;
  const bool tiny = ref.D <= kTeamTinyD;
  if (!tiny && L <= kTeamLow) return nullptr;
  const int m = tiny ? L : kTeamLow, hb = L - m;
  // The team's bits: the sites in order, or, when a bond joins the low sites to
  // far high ones (a ring), folded: bit 0 a site in the middle of the low arc,
  // then its neighbours on both sides in turn.  A ring's two cuts then lie at the
  // lowest high bits (segments next to each other: the same block) and at the two
  // highest low bits (a flip keeps long runs together).
  bool ring = false;
  for (int k = 0; k < ref.nb; ++k) ring = ring || (ref.lo[k] < m && ref.hi[k] > m + 3);
  ring = ring && !tiny;
  std::vector<int> bit_of(L), site_of(L);
  for (int p = 0; p < L; ++p) {
    const int c = m / 2 - 1;  // a middle site of the low arc 0 .. m-1
    const int site = !ring ? p : ((p & 1 ? c + (p + 1) / 2 : c - p / 2) + L) % L;
    site_of[p] = site;
    bit_of[site] = p;
  }
  ChainParams P = ref;
  for (int k = 0; k < P.nb; ++k) {
    const int x = bit_of[ref.lo[k]], y = bit_of[ref.hi[k]];
    P.lo[k] = (int8_t)std::min(x, y);
    P.hi[k] = (int8_t)std::max(x, y);
  }
  std::vector<int> low, cross, high;
  // at most two coupling values, a and b
  const double wv[2] = {P.bval[0], P.bval[P.nb - 1]};
  for (int k = 0; k < P.nb; ++k) {
    (P.hi[k] < m ? low : P.lo[k] >= m ? high : cross).push_back(k);
    if (P.bval[k] != wv[0] && P.bval[k] != wv[1]) return nullptr;
  }
  const int nl = (int)low.size(), nc = (int)cross.size();
  const bool one = wv[0] == wv[1];
  const bool uni = one && nc <= 2 && nl <= low_first(3, hb == 0 ? 0 : 2);
  const int NQ = uni ? 3 : 6, NC = hb == 0 ? 0 : uni ? 2 : 6;
  if (nc > NC) return nullptr;
  // low slots: the first class, then the second (either value may be the first;
  // a single value fills both)
  const int cap[2] = {low_first(NQ, NC), low_second(NQ, NC)};
  int first = 0;  // which value is class 0
  std::vector<int> slot(nl, -1);
  for (first = 0; first < 2; ++first) {
    int used[2] = {0, 0}, e = 0;
    for (; e < nl; ++e) {
      int c = one ? (used[0] < cap[0] ? 0 : 1) : (P.bval[low[e]] == wv[first] ? 0 : 1);
      if (used[c] >= cap[c]) break;
      slot[e] = (c ? cap[0] : 0) + used[c]++;
    }
    if (e == nl) break;
  }
  if (first == 2) return nullptr;
  auto cls = [&](int k) { return !one && P.bval[k] != wv[first] ? 1u : 0u; };
  TeamTables* T = new TeamTables();
  T->NQ = NQ;
  T->NC = NC;
  T->uni = uni;
  T->w[0] = wv[first];
  T->w[1] = wv[1 - first];
  for (int c = 0; c < nc; ++c) T->ccls |= cls(cross[c]) << c;

  // class tables: the m-bit strings of each popcount na, ascending
  auto count = [&](int na) { return (int64_t)C[m * kRankT + na]; };
  const int na0 = std::max(0, Lup - hb), na1 = std::min(m, Lup);
  std::vector<int> tbase(m + 1, 0);
  int ntab = 0;
  for (int na = na0; na <= na1; ++na) {
    tbase[na] = ntab;
    ntab += ((hb == 0 ? (int)P.D : (int)count(na)) + 1) & ~1;
  }
  T->ntab = ntab;
  std::vector<uint16_t> tab[2];
  const size_t trows = tab_rows(NC);
  for (auto& t : tab) t.assign(4 * NQ * trows, 0);
  std::vector<uint32_t> strings;  // of one class, when hb == 0 the basis itself
  for (int na = na0; na <= na1; ++na) {
    strings.clear();
    if (hb == 0) {
      strings.assign(states, states + P.D);
    } else {
      for (uint32_t a = 0; a < (1u << m); ++a)
        if (popc32(a) == na) strings.push_back(a);
    }
    for (size_t i = 0; i < strings.size(); ++i) {
      const uint32_t a = strings[i];
      auto put = [&](int e, int which, uint32_t v) {
        tab[which][((size_t)(e >> 2) * trows + tbase[na] + i) * 4 + (e & 3)] = (uint16_t)v;
      };
      for (int e = 0; e < nl; ++e) {
        const uint32_t mk = (1u << P.lo[low[e]]) | (1u << P.hi[low[e]]);
        if (popc32(a & mk) != 1) continue;  // parallel spins: the zero slot
        const uint32_t r = 1u + (uint32_t)full_rank(a ^ mk, C);
        put(slot[e], 0, r * 8u);
        put(slot[e], 1, r * 4u);
      }
      for (int c = 0; c < nc; ++c) {
        const uint32_t bit = 1u << P.lo[cross[c]];
        const uint32_t r = 1u + (uint32_t)full_rank(a ^ bit, C), up = (a & bit) ? 0x8000u : 0u;
        put(4 * NQ - 1 - c, 0, (r * 8u) | up);
        put(4 * NQ - 1 - c, 1, (r * 4u) | up);
      }
    }
  }

  // segments in row order, their groups and neighbour lists
  const uint32_t nB = 1u << hb;
  std::vector<int64_t> row0(nB, -1), pos(nB, 0), elem(nB, 0);
  int64_t rows = 0, at = kSegAlign, el = 4;
  for (uint32_t b = 0; b < nB; ++b) {
    const int na = Lup - popc32(b);
    if (na < 0 || na > m) continue;
    row0[b] = rows;
    pos[b] = at;
    const int64_t n = hb == 0 ? P.D : count(na);
    rows += n;
    at += (n + kSegAlign) / kSegAlign * kSegAlign;  // at least one element of padding
    elem[b] = el;
    el += (n + (n & 1) + 1 + 3) & ~(int64_t)3;  // the rows, an even count, and the next zero slot
    T->maxseg = std::max<int>(T->maxseg, (int)(el - elem[b]));
  }
  bool ok = rows == P.D && at < ((int64_t)1 << 28);
  T->elems = at;
  std::vector<TeamGrp> grp;
  std::vector<uint32_t> hrow, crs;
  std::vector<int32_t> sgrp;
  std::vector<int> ordinal(nB, -1);
  std::vector<uint32_t> segb;
  for (uint32_t b = 0; b < nB; ++b)
    if (row0[b] >= 0) {
      ordinal[b] = (int)segb.size();
      segb.push_back(b);
    }
  std::vector<std::vector<uint32_t>> hbit(segb.size());  // target b | class << 31
  for (uint32_t b = 0; ok && b < nB; ++b) {
    if (row0[b] < 0) continue;
    const int na = Lup - popc32(b);
    const int n = hb == 0 ? (int)P.D : (int)count(na);
    const uint32_t hoff = (uint32_t)hrow.size();
    for (const int k : high) {
      const uint32_t mk = (1u << (P.lo[k] - m)) | (1u << (P.hi[k] - m));
      if (popc32(b & mk) != 1) continue;
      hrow.push_back((uint32_t)pos[b ^ mk] | (cls(k) << 31));
      hbit[T->nseg].push_back((b ^ mk) | (cls(k) << 31));
    }
    const uint32_t nh = (uint32_t)hrow.size() - hoff;
    hrow.resize((hrow.size() + 3) & ~(size_t)3, 0u);  // lists are read four at a time
    for (int c = 0; c < NC; ++c) {
      uint32_t e = 0;
      if (c < nc) {
        const uint32_t bit = 1u << (P.hi[cross[c]] - m);
        if (row0[b ^ bit] >= 0)  // bit 30: the low site's spin that differs from the high one
          e = 0x80000000u | ((b & bit) ? 0u : 0x40000000u) | (uint32_t)pos[b ^ bit];
      }
      crs.push_back(e);
    }
    sgrp.push_back((int32_t)grp.size());
    for (int i0 = 0; i0 < n; i0 += kGrp)
      grp.push_back({(uint32_t)i0, (uint32_t)tbase[na], (uint32_t)row0[b], (uint32_t)T->nseg,
                     (uint32_t)std::min<int>(kGrp, n - i0), nh, hoff, (uint32_t)pos[b]});
    ++T->nseg;
  }
  if (!ok) {
    delete T;
    return nullptr;
  }
  // the team's rows in the reference order (checked: every row once)
  std::vector<uint32_t> perm;
  if (ring) {
    std::vector<uint32_t> lowst(1u << m), highst(nB);
    auto spread = [&](uint32_t v, int at) {
      uint32_t r = 0;
      for (; v; v &= v - 1u) r |= 1u << site_of[at + ctz32(v)];
      return r;
    };
    for (uint32_t a = 0; a < (1u << m); ++a) lowst[a] = spread(a, 0);
    for (uint32_t b = 0; b < nB; ++b) highst[b] = spread(b, m);
    std::vector<std::vector<uint32_t>> cls_low(m + 1);
    for (uint32_t a = 0; a < (1u << m); ++a) cls_low[popc32(a)].push_back(lowst[a]);
    perm.reserve(P.D);
    std::vector<char> seen(P.D, 0);
    for (const uint32_t b : segb)
      for (const uint32_t a : cls_low[Lup - popc32(b)]) {
        const uint64_t r = full_rank(highst[b] | a, C);
        ok = ok && r < (uint64_t)P.D && states[r] == (highst[b] | a) && !seen[r];
        if (!ok) break;
        seen[r] = 1;
        perm.push_back((uint32_t)r);
      }
    ok = ok && (int64_t)perm.size() == P.D;
    if (!ok) {
      delete T;
      return nullptr;
    }
  } else {
    for (size_t j = 0; ok && j < segb.size(); ++j) ok = (states[row0[segb[j]]] >> m) == segb[j];
    if (!ok) {
      delete T;
      return nullptr;
    }
  }
  hrow.resize(hrow.size() + 4, 0u);
  sgrp.push_back((int32_t)grp.size());
  T->ngrp = (int)grp.size();

  // resident plans: contiguous whole segments, about equal group counts
  std::vector<int32_t> gblk[6];
  std::vector<uint32_t> rec[6];
  const int RW = rec_words(NC), RN = rec_remote(NC);
  std::vector<int> owner(T->nseg);
  for (int lt = 0; lt < 6; ++lt) {
    const int n = 1 << lt;
    gblk[lt].assign(n + 1, T->ngrp);
    gblk[lt][0] = 0;
    int sg = 0, prev = 0;
    for (int j = 0; j < n; ++j) {
      const int s_first = sg;
      const double goal = (double)T->ngrp * (j + 1) / n;
      while (sg < T->nseg &&
             (j == n - 1 || sgrp[sg] + 0.5 * (sgrp[sg + 1] - sgrp[sg]) < goal))
        ++sg;
      for (int t = s_first; t < sg; ++t) owner[t] = j;
      gblk[lt][j + 1] = sgrp[sg];
      T->maxgrp[lt] = std::max(T->maxgrp[lt], sgrp[sg] - prev);
      if (sg > s_first) {
        const int64_t e1 = sg < T->nseg ? elem[segb[sg]] : el;
        T->maxel[lt] = std::max<int>(T->maxel[lt], (int)(e1 - elem[segb[s_first]]));
      }
      prev = sgrp[sg];
    }
    if (T->maxgrp[lt] > 13 * 16) continue;  // never resident
    // records; a target in the own block is given by its zero slot in LDS
    std::vector<uint32_t>& rc = rec[lt];
    rc.assign((size_t)T->ngrp * RW + 16, 0u);
    for (int sg2 = 0; sg2 < T->nseg && !rc.empty(); ++sg2) {
      uint32_t w[64] = {};
      auto element = [&](int t) { return (uint32_t)elem[segb[t]]; };
      std::vector<uint32_t> loc, rem;
      for (const uint32_t e : hbit[sg2]) {
        const uint32_t tb = e & 0x7FFFFFFFu;
        const int t = ordinal[tb];
        if (owner[t] == owner[sg2] && (int)loc.size() < kLocal)
          loc.push_back(element(t) | (e & 0x80000000u));
        else
          rem.push_back((uint32_t)pos[tb] | (e & 0x80000000u));
      }
      if ((int)rem.size() > RN) {
        rc.clear();
        break;
      }
      // 8, 4, 2, 1 entries at fixed places: one uniform test per size
      auto place = [&](const std::vector<uint32_t>& v, int at) {
        size_t j = 0;
        const size_t c = v.size();
        if (c & 8) for (int s = 7; s < 15; ++s) w[at + s] = v[j++];
        if (c & 4) for (int s = 0; s < 4; ++s) w[at + s] = v[j++];
        if (c & 2) for (int s = 4; s < 6; ++s) w[at + s] = v[j++];
        if (c & 1) w[at + 6] = v[j++];
      };
      place(loc, kRecHead + NC);
      place(rem, kRecHead + NC + kLocal);
      for (int c = 0; c < NC; ++c) {
        uint32_t e = crs[(size_t)sg2 * NC + c];
        if (e >> 31) {
          const int t = ordinal[segb[sg2] ^ (1u << (P.hi[cross[c]] - m))];
          if (owner[t] == owner[sg2]) e = (e & 0xC0000000u) | 0x20000000u | element(t);
        }
        w[kRecHead + c] = e;
      }
      for (int gi = sgrp[sg2]; gi < sgrp[sg2 + 1]; ++gi) {
        const TeamGrp& g = grp[gi];
        w[0] = g.i0 | (g.n << 12) | ((uint32_t)loc.size() << 20) | ((uint32_t)rem.size() << 24);
        w[1] = g.tab;
        w[2] = g.seg0;
        w[3] = element(sg2);
        w[4] = g.pos;
        std::copy(w, w + RW, rc.begin() + (size_t)gi * RW);
      }
    }
  }
  // streaming units: each segment, in row order, to the unit with the least
  // work so far, so that the units sweep the rows together
  std::vector<std::vector<int32_t>> units(kTeamUnits);
  std::vector<int64_t> load(kTeamUnits, 0);
  for (int sg = 0; sg < T->nseg; ++sg) {
    const int u = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    units[u].push_back(sg);
    load[u] += sgrp[sg + 1] - sgrp[sg];
  }
  std::vector<int32_t> ulist, uofs(1, 0);
  for (const auto& u : units) {
    ulist.insert(ulist.end(), u.begin(), u.end());
    uofs.push_back((int32_t)ulist.size());
  }

  // one upload
  std::vector<char> img;
  auto put = [&](const void* p, size_t n) {
    const size_t at = (img.size() + 255) & ~(size_t)255;
    img.resize(at + n);
    if (n) std::memcpy(img.data() + at, p, n);
    return at;
  };
  const size_t o_tab[2] = {put(tab[0].data(), tab[0].size() * 2),
                           put(tab[1].data(), tab[1].size() * 2)};
  const size_t o_grp = put(grp.data(), grp.size() * sizeof(TeamGrp));
  const size_t o_hrow = put(hrow.data(), hrow.size() * 4);
  const size_t o_crs = put(crs.data(), crs.size() * 4);
  const size_t o_ul = put(ulist.data(), ulist.size() * 4), o_uo = put(uofs.data(), uofs.size() * 4);
  const size_t o_sg = put(sgrp.data(), sgrp.size() * 4);
  const size_t o_pm = put(perm.data(), perm.size() * 4);
  size_t o_dg = 0;  // the permuted diagonal, after the image
  size_t o_gb[6];
  size_t o_rec[6];
  for (int lt = 0; lt < 6; ++lt) {
    o_gb[lt] = put(gblk[lt].data(), gblk[lt].size() * 4);
    o_rec[lt] = put(rec[lt].data(), rec[lt].size() * 4);
  }
  try {
    o_dg = (img.size() + 255) & ~(size_t)255;
    PF_HIP(hipMalloc(&T->dev, o_dg + (ring ? P.D * sizeof(double) : 0)));
    PF_HIP(hipMemcpy(T->dev, img.data(), img.size(), hipMemcpyHostToDevice));
    if (ring) {
      hipLaunchKernelGGL(team_permute_kernel, dim3((unsigned)((P.D + 255) / 256)), dim3(256), 0, 0,
                         (const uint32_t*)((char*)T->dev + o_pm), diag_dev, P.D,
                         (double*)((char*)T->dev + o_dg));
      PF_HIP(hipGetLastError());
    }
  } catch (...) {
    team_destroy(T);
    throw;
  }
  const char* base = (const char*)T->dev;
  for (int t = 0; t < 2; ++t) {
    T->tab[t] = (const uint64_t*)(base + o_tab[t]);
  }
  T->grp = (const TeamGrp*)(base + o_grp);
  T->hrow = (const uint32_t*)(base + o_hrow);
  T->cross = (const uint32_t*)(base + o_crs);
  T->ulist = (const int32_t*)(base + o_ul);
  T->uofs = (const int32_t*)(base + o_uo);
  T->sgrp = (const int32_t*)(base + o_sg);
  if (ring) {
    T->perm = (const uint32_t*)(base + o_pm);
    T->diag = (const double*)(base + o_dg);
  }
  for (int lt = 0; lt < 6; ++lt) {
    T->gblk[lt] = (const int32_t*)(base + o_gb[lt]);
    T->rec[lt] = rec[lt].empty() ? nullptr : (const uint32_t*)(base + o_rec[lt]);
  }
  return T;
}

// --------------------------------------------------------------- the plan
constexpr size_t kTeamLds = 160 * 1024 - sizeof(TeamShared);

static size_t team_table_bytes(const TeamTables* t) { return (size_t)8 * t->NQ * tab_rows(t->NC); }
// Dynamic LDS of the resident form: tables, records, rows with zero slots, and
// one spare element at the end.
static size_t team_resident_lds(const TeamTables* t, int lt, size_t sz) {
  return (team_table_bytes(t) + (size_t)t->maxgrp[lt] * lrec_words(t->NC) * 4 + 32 +
          ((size_t)t->maxel[lt] + 8) * sz + 31) & ~(size_t)31;
}
static size_t team_stream_lds(const TeamTables* t, size_t sz, int R) {
  return team_table_bytes(t) + ((size_t)team_waves(sz, t->NC, R) * t->maxseg + 8) * sz;
}

// Groups a wave holds in the resident form with 1 << lt blocks per column (the
// kernel instance: 1, 2, 4, 7, 8, 13, 14), or 0 when the column does not fit.
static int team_resident(const TeamTables* t, int dtype, int lt, bool kpm) {
  const size_t sz = dtype == PF_F64 ? 8 : 4;
  if (!t->rec[lt] || team_resident_lds(t, lt, sz) > kTeamLds) return 0;
  const bool f64 = dtype == PF_F64;
  for (const int r : {1, 2, 4, 7, 8, 13, 14}) {
    const bool made = r <= 4 || (f64 ? r == (t->NC == 6 ? 8 : kpm ? 7 : 14)
                                     : r == 7 || (r == 13 && t->NC == 2));
    if (made && t->maxgrp[lt] <= r * team_waves(sz, t->NC, r)) return r;
  }
  return 0;
}

// Time of one step on ncols columns with 1 << lt blocks per column, in us
// (fitted to measurements on MI355X: 16 128-row groups of a block are 1.0 to 3.8 us
// in the resident form, the rest is the barrier; a streamed row is 0.05 to 0.12
// ns).  Columns beyond 8 x 32 / T run in further rounds.
static double team_step_us(const TeamTables* t, int dtype, int ncols, int lt, bool kpm) {
  const int T = 1 << lt;
  const int rounds = (ncols + 8 * (32 / T) - 1) / (8 * (32 / T));
  const bool f64 = dtype == PF_F64;
  double us = T == 32 ? 2.0 : T == 16 ? 1.6 : T == 1 ? 1.1 : 1.4;
  if (const int R = team_resident(t, dtype, lt, kpm))
    us += (double)t->maxgrp[lt] / 16 *
          (t->NQ == 3 ? (f64 ? (R > 4 ? 1.9 : kpm ? 1.65 : 1.35) : 1.0) : (f64 ? 3.8 : 2.6));
  else
    us += (double)t->elems / T * (t->NQ == 3 ? (f64 ? 0.0021 : 0.0018) : (f64 ? 0.0042 : 0.0038));
  return rounds * us;
}
// The per-step kernels: launch-bound below 5 us, then at the rate of their
// algorithmic bytes (2.6 TB/s; half that when the blocks exceed the 256 MB
// Infinity Cache).
static double per_step_us(const pf_op* op, int dtype, int ncols) {
  const int64_t D = op->D;
  if (op->kind == kQsun) return qsun_per_step_us((double)D * ncols, dtype);
  const double mb = 4e-6 * (double)D * ncols * (dtype == PF_F64 ? 8 : 4);
  return std::max(5.0, mb / (mb > 512 ? 1.4 : 2.6));
}

int team_kpm_steps(int dtype, int N);

// Blocks per column of the fastest team form, and its time.
int team_best(const pf_op* op, int dtype, int ncols, double* us, bool kpm) {
  const TeamTables* t = op->team;
  int best = 0;
  *us = 1e300;
  if (op->kind == kQsun && qsun_team_ok(op))
    for (int lt = 0; lt < 6; ++lt) {
      if (!qsun_team_fits(op, dtype, lt)) continue;
      const int teams = 8 * (32 >> lt);
      const double x = (ncols + teams - 1) / teams * qsun_team_step_us(op, dtype, lt);
      if (x < *us) {
        *us = x;
        best = 1 << lt;
      }
    }
  if (!t) return best;
  for (int lt = 0; lt < 6; ++lt) {
    if ((t->NC == 0) != (lt == 0)) continue;
    const double x = team_step_us(t, dtype, ncols, lt, kpm);
    if (x < *us) {
      *us = x;
      best = 1 << lt;
    }
  }
  return best;
}

// Below this order the begin and end launches cost what the steps save.
constexpr int kTeamMinOrder = 8;

// Blocks per column for `order` steps on ncols columns, or 0.  `gain`: the steps
// that the per-step launches take for one of these.
static int team_choose(const pf_op* op, int dtype, int order, int ncols, int gain, bool kpm) {
  const TeamTables* t = op->team;
  const TuneCfg& f = op->force;
  const bool qsun = op->kind == kQsun && qsun_team_ok(op);
  if ((!t && !qsun) || order < 1 || f.team == 0) return 0;
  if (f.team > 0) return t && t->NC == 0 ? 1 : f.team;
  // forced launch knobs are those of the per-step kernels
  if (f.V || f.xcd >= 0 || f.nt >= 0 || f.pb >= 0 || f.wide >= 0 || f.occ >= 0 || f.part >= 0)
    return 0;
  if (order < kTeamMinOrder) return 0;
  // measured by the autotuner, else by the rule (by chunks of columns there)
  const auto it = op->tuned.find({dtype, ncols});
  const int tuned = it == op->tuned.end() ? -1 : it->second.team;
  if (tuned > 0 && !kpm) return tuned;  // (the moments have their own best size)
  if (tuned == 0 && gain == 1) return 0;
  double us;
  const int T = team_best(op, dtype, ncols, &us, kpm);
  return tuned > 0 || us < 0.95 * gain * per_step_us(op, dtype, ncols) ? T : 0;
}

int team_plan(const pf_op* op, int dtype, int polytype, int order, const double* X, int64_t ldx,
              const double* Y, int64_t ldy, int ncols) {
  if (polytype == PF_TAYLOR) return 0;
  // a column's result may replace that column of X, but no other
  const double* xe = X + (ncols - 1) * ldx + op->D;
  const double* ye = Y + (ncols - 1) * ldy + op->D;
  if (X < ye && Y < xe && !(X == Y && ldx == ldy)) return 0;
  return team_choose(op, dtype, order, ncols, 1, false);
}

// FP64 moments take half the steps here (TeamDots), so the team wins far above the
// sizes where the filter's does: 32 probes, N = 250, L = 20: 18.0 -> 3.6 ms (team of
// 16); 16 probes, L = 22: 9.1 -> 2.9 ms at N = 60 (streamed); FP32, the same steps:
// L = 20 8.0 -> 5.3 ms, L = 18 2.9 -> 1.5 ms (team of 8).
int team_kpm_plan(const pf_op* op, int dtype, int N, int ncols) {
  if (!op->team) return 0;
  return team_choose(op, dtype, team_kpm_steps(dtype, N), ncols, dtype == PF_F64 ? 2 : 1,
                     true);
}

static size_t team_align(size_t n) { return (n + 255) & ~(size_t)255; }
size_t team_ctl_bytes() { return team_align(sizeof(TeamCtl)); }

// Clears the control words and copies order + 1 coefficients.
void team_begin(void* ctl, double* cdev, const double* coeffs, int order, hipStream_t st) {
  for (int at = 0; at == 0 || at <= order; at += kCoefChunk) {
    TeamCoefs c;
    const int n = std::max(0, std::min(kCoefChunk, order + 1 - at));
    if (n) std::memcpy(c.c, coeffs + at, n * sizeof(double));
    hipLaunchKernelGGL(team_begin_kernel, dim3(1), dim3(1024), 0, st,
                       at ? nullptr : static_cast<TeamCtl*>(ctl), cdev, at, n, c);
    PF_HIP(hipGetLastError());
  }
}

size_t team_work_bytes(const pf_op* op, int dtype, int order, int ncols, int T) {
  if (op->kind == kQsun) return qsun_team_work_bytes(op, dtype, order, ncols, T);
  const size_t vec = (size_t)op->team->elems * (dtype == PF_F64 ? 8 : 4);
  return team_align(sizeof(TeamCtl)) + team_align((size_t)(order + 1) * 8) +
         std::min(ncols, 8 * (32 / T)) * 3 * vec;
}

template <typename T, int NQ, int NC, bool UNI, bool KPM, int R>
static void team_launch(const TeamArgs& A, int grid, size_t lds, hipStream_t st) {
  auto* k = chain_team_kernel<T, NQ, NC, UNI, KPM, R>;
  PF_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(64 * team_waves(sizeof(T), NC, R)), lds, st, A);
  PF_HIP(hipGetLastError());
}

template <typename T, int NQ, int NC, bool UNI, bool KPM>
static void team_launch_r(const TeamArgs& A, int R, int grid, size_t lds, hipStream_t st) {
  if (R == 1) return team_launch<T, NQ, NC, UNI, KPM, 1>(A, grid, lds, st);
  if (R == 2) return team_launch<T, NQ, NC, UNI, KPM, 2>(A, grid, lds, st);
  if constexpr (NC > 0) {
    if (R == 4) return team_launch<T, NQ, NC, UNI, KPM, 4>(A, grid, lds, st);
    if constexpr (sizeof(T) == 8) {
      // (the recurrence of the moments holds no X, so 16 waves spill less: 32 columns at
      // L = 20, blocks of 16 waves 3.71 ms, of eight 3.88)
      constexpr int RM = NC == 6 ? 8 : KPM ? 7 : 14;
      if (R == RM) return team_launch<T, NQ, NC, UNI, KPM, RM>(A, grid, lds, st);
    } else {
      if (R == 7) return team_launch<T, NQ, NC, UNI, KPM, 7>(A, grid, lds, st);
      if constexpr (NC == 2)
        if (R == 13) return team_launch<T, NQ, NC, UNI, KPM, 13>(A, grid, lds, st);
    }
    if (R == 0) return team_launch<T, NQ, NC, UNI, KPM, 0>(A, grid, lds, st);
  }
  throw Error{PF_ERR_UNSUPPORTED, "team filter: no kernel for this plan"};
}

template <typename T, bool KPM>
static void team_launch_t(const TeamTables* t, const TeamArgs& A, int R, int grid, size_t lds,
                          hipStream_t st) {
  if (t->NC == 0) {
    if (t->NQ == 3) team_launch_r<T, 3, 0, true, KPM>(A, R, grid, lds, st);
    else team_launch_r<T, 6, 0, false, KPM>(A, R, grid, lds, st);
  } else {
    if (t->NQ == 3) team_launch_r<T, 3, 2, true, KPM>(A, R, grid, lds, st);
    else team_launch_r<T, 6, 6, false, KPM>(A, R, grid, lds, st);
  }
}

// One launch over all columns: the filter (dots null) or the KPM recurrence of
// `order` steps.  work: control words, coefficients, the teams' vectors.
static void team_run(pf_op* op, int dtype, TeamArgs A, int T, void* work, size_t coef_bytes,
                     hipStream_t st) {
  const TeamTables* t = op->team;
  const int w = dtype == PF_F64 ? 0 : 1;
  const size_t sz = dtype == PF_F64 ? 8 : 4;
  const bool kpm = A.dots != nullptr;
  char* p = (char*)work;
  A.ctl = (TeamCtl*)p;
  p += team_align(sizeof(TeamCtl));
  A.coefs = (const double*)p;
  p += team_align(coef_bytes);
  int lt = 0;
  while ((1 << lt) < T) ++lt;
  const int R = team_resident(t, dtype, lt, kpm);
  const Affine af = op->affine(true);
  A.tab = t->tab[w];
  A.grp = t->grp;
  A.rec = t->rec[lt];
  A.hrow = t->hrow;
  A.cross = t->cross;
  A.w[0] = t->w[0];
  A.w[1] = t->w[1];
  A.ccls = t->ccls;
  A.gblk = t->gblk[lt];
  A.ulist = t->ulist;
  A.uofs = t->uofs;
  A.sgrp = t->sgrp;
  A.ntab = t->ntab;
  A.T = T;
  A.maxseg = t->maxseg;
  A.elems = (uint32_t)t->elems;
  A.tab_lds = (uint32_t)team_table_bytes(t);
  A.diag = t->diag ? t->diag : op->diag;
  A.perm = t->perm;
  A.scale = af.scale;
  A.shift = af.shift;
  A.work = p;
  // the streaming form keeps its own copy of X where the caller's is not FP64 in
  // the team's row order
  A.has_x = dtype != PF_F64 || t->perm || kpm;
  A.slot_bytes = (int64_t)(3 * (size_t)t->elems * sz);
  A.nslots = std::min(A.ncols, 8 * (32 / T));
  const int cus = std::max(1, op->h->prop.multiProcessorCount);
  const int nxcd = std::max(1, cus / 32);
  const int grid = std::max(T, cus / nxcd * nxcd);
  A.expect = grid / nxcd;
  size_t lds = R ? team_resident_lds(t, lt, sz) : team_table_bytes(t);
  if (t->NC > 0) lds = std::max(lds, team_stream_lds(t, sz, R));
  lds = (lds + 31) & ~(size_t)31;
  A.rows_lds = (uint32_t)lds;
  lds += sizeof(TeamShared);
  if (kpm) {
    if (dtype == PF_F64) team_launch_t<double, true>(t, A, R, grid, lds, st);
    else team_launch_t<float, true>(t, A, R, grid, lds, st);
  } else {
    if (dtype == PF_F64) team_launch_t<double, false>(t, A, R, grid, lds, st);
    else team_launch_t<float, false>(t, A, R, grid, lds, st);
  }
}

void team_filter(pf_op* op, int dtype, int polytype, const double* coeffs, int order,
                 const double* X, int64_t ldx, double* Y, int64_t ldy, int ncols, int T,
                 void* work, hipStream_t st) {
  if (op->kind == kQsun)
    return qsun_team_filter(op, dtype, polytype, coeffs, order, X, ldx, Y, ldy, ncols, T, work, st);
  TeamCtl* ctl = (TeamCtl*)work;
  double* cdev = (double*)((char*)work + team_ctl_bytes());
  team_begin(ctl, cdev, coeffs, order, st);
  TeamArgs A{};
  A.order = order;
  A.polytype = polytype;
  A.ncols = ncols;
  A.X = X;
  A.ldx = ldx;
  A.Y = Y;
  A.ldy = ldy;
  team_run(op, dtype, A, T, work, (size_t)(order + 1) * 8, st);
  hipLaunchKernelGGL(team_end_kernel, dim3(256), dim3(256), 0, st, ctl, (uint32_t)ncols, Y, ldy,
                     op->D);
  PF_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ KPM
__global__ void team_zero_kernel(double* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0.0;
}
// dots[step][which] summed over columns and blocks in a fixed order; NaN when a
// column was not finished
__global__ __launch_bounds__(256) void team_dots_kernel(const double* __restrict__ dots, int ncols,
                                                        const TeamCtl* ctl,
                                                        double* __restrict__ sums) {
  __shared__ double red[4];
  const double* p = dots + (int64_t)blockIdx.x * ncols * kTeamUnits;
  double t = 0.0;
  for (int i = threadIdx.x; i < ncols * kTeamUnits; i += 256) t += p[i];
  t = block_sum_256(t, red);
  if (threadIdx.x == 0)
    sums[blockIdx.x] = ctl->done == (uint32_t)ncols && ctl->abort == 0 ? t : __builtin_nan("");
}
// mu[n] += the moments of one chunk of columns from its dots
__global__ void team_moments_kernel(const double* __restrict__ sums, int f64, int N,
                                    double* __restrict__ mu) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  double v;
  if (f64) {  // sums[2j] = <T_j, T_j>, sums[2j+1] = <T_{j+1}, T_j>
    v = sums[n];
    if (n >= 2) v = 2.0 * v - sums[n & 1];
  } else {    // sums[2j+1] = <x, T_{j+1}>
    v = n == 0 ? sums[0] : sums[2 * n - 1];
  }
  mu[n] += v;
}

int team_kpm_steps(int dtype, int N) { return dtype == PF_F64 ? (N + 1) / 2 : N - 1; }

size_t team_kpm_bytes(const pf_op* op, int dtype, int N, int ncols, int T) {
  const size_t steps = team_kpm_steps(dtype, N);
  return team_work_bytes(op, dtype, 0, ncols, T) + team_align(2 * steps * ncols * kTeamUnits * 8) +
         team_align(2 * steps * 8);
}

void team_kpm(pf_op* op, int dtype, int N, const double* X, int64_t ldx, int ncols,
              const double* colscale, double* mu, int T, void* work, hipStream_t st) {
  const int steps = team_kpm_steps(dtype, N);
  TeamCtl* ctl = (TeamCtl*)work;
  double* dots = (double*)((char*)work + team_work_bytes(op, dtype, 0, ncols, T));
  const int64_t n = (int64_t)2 * steps * ncols * kTeamUnits;
  double* sums = (double*)((char*)dots + team_align(n * 8));
  team_begin(ctl, nullptr, nullptr, -1, st);
  hipLaunchKernelGGL(team_zero_kernel, dim3(512), dim3(256), 0, st, dots, n);
  PF_HIP(hipGetLastError());
  TeamArgs A{};
  A.order = steps;
  A.ncols = ncols;
  A.X = X;
  A.ldx = ldx;
  A.colscale = colscale;
  A.dots = dots;
  team_run(op, dtype, A, T, work, 8, st);
  hipLaunchKernelGGL(team_dots_kernel, dim3(2 * steps), dim3(256), 0, st, dots, ncols, ctl, sums);
  hipLaunchKernelGGL(team_moments_kernel, dim3((N + 255) / 256), dim3(256), 0, st, sums,
                     dtype == PF_F64, N, mu);
  PF_HIP(hipGetLastError());
}

}  // namespace pf
