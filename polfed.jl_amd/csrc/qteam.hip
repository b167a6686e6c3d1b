// The Clenshaw filter of Quantum-Sun operators in one launch, an instance's column
// per team (pf_team.h).
//
// The rows are the strings of 3 grain bits, then the outer spins; flip j exchanges
// the outer spin j and one grain spin, so its neighbour row is an XOR.  A block of
// the team holds an aligned range of rows:
//   grain bits | log2 W outer spins in the lane | the lane and wave in the block |
//   the block in the team (log2 T spins),
// a lane GR * W rows: X, b2 and b3 of all of them in registers for all steps, the
// grain matrix from scalar registers (a lane has whole grain blocks).  The flips of
// the lane and wave bits read b2 from LDS, whose layout [grain][lane] of W-row
// vectors makes each an XOR of the byte address and free of bank conflicts; only
// the log2 T flips of the block bits read the XCD's L2, in the same layout.
// Nothing in a step depends on another instance: the instances do not run in
// lockstep, and the jobs (longest first) are claimed by whichever team is free.
//
// A team with fewer blocks than T, or a block with more rows than it can hold,
// takes the streaming form: a lane per row, all vectors in memory.
//
// What bounds it: a step of 2^13 FP64 rows in one block takes 3.1 us, of which 45 %
// are vector instructions (22 FMAs a row), 38 % LDS reads; the rest is the latency
// of the step's serial parts with two waves per SIMD (two block barriers, the
// matrix through the scalar cache, ten rounds of LDS reads), 1.4 us for the smallest
// instances, and 0.3 - 0.7 us of team barrier.  512 threads with 256 registers
// instead of 1024 with 128: X, b2, b3 and the sums then fit without spills.
// Measured against the per-step launches (autotuned), one application:
//   64 instances of 2^13 .. 2^17 rows, orders 160 .. 306, FP64 7.9 -> 3.7 ms,
//   FP32 5.9 -> 1.9 ms; 64 of 2^11 .. 2^13 FP64 2.55 -> 0.94 ms; 3 of 2^10, order
//   60, FP64 0.33 -> 0.145 ms; 6 of 2^14 / 2^15, 4 columns, FP64 2.5 -> 1.1 ms.

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "pf_device.h"
#include "pf_internal.h"
#include "pf_qsun.h"
#include "pf_team.h"

namespace pf {

constexpr int kQsunLane = 9;  // lane and wave bits of a block: flips read from LDS
constexpr int kQsunThreads = 1 << kQsunLane;
// Most rows of a block (FP64 with 2^14 rows spilled registers: 8.5 us a step where
// two blocks of 2^13 take 3.4).
constexpr size_t qsun_rows(size_t elem) { return (size_t)kQsunThreads * (elem == 8 ? 16 : 32); }

// One operator, as the kernel reads it.  Grains below 3 spins are extended by the
// first outer spins (their flips become entries of the matrix).
struct QsunTeamOp {
  double G64[256], c64[kMaxLocPad], A64[16];
  float G32[256], c32[kMaxLocPad];
  uint64_t gsel;            // two bits per flip: its grain spin
  uint32_t gset[4];         // the flips of each grain spin
  const double* qdiag;      // Dlo[2^lb], Dhi: the diagonal of a lane's first rows
  double scale, shift;
  int64_t D;
  int32_t lgr, nf, lb, pad;
};
template <typename T> struct QsunTeamOf;
template <> struct QsunTeamOf<double> {
  static __device__ const double* G(const QsunTeamOp* o) { return o->G64; }
  static __device__ const double* c(const QsunTeamOp* o) { return o->c64; }
};
template <> struct QsunTeamOf<float> {
  static __device__ const float* G(const QsunTeamOp* o) { return o->G32; }
  static __device__ const float* c(const QsunTeamOp* o) { return o->c32; }
};

struct QsunTeamArgs {
  const QsunTeamOp* ops;
  const QsunJob* jobs;  // njobs, longest first (null: column j of `one`)
  QsunJob one;
  int64_t ldx, ldy;
  int32_t njobs, T, expect, polytype, nslots;
  uint32_t lds;         // bytes before TeamShared
  TeamCtl* ctl;
};

template <typename T>
struct QsunCoef {
  T cx, ch, cb;
  bool b3;
};
// Step j = K - k of a filter of order K.
template <typename T>
__device__ __forceinline__ QsunCoef<T> qsun_coef(int type, const double* c, int K, int j) {
  const int k = K - j;
  double alpha, beta1, dummy;
  poly_ab_dev(type, k + 1, dummy, beta1);
  if (k >= 1) poly_ab_dev(type, k, alpha, dummy);
  else alpha = type == PF_HERMITE ? 2.0 : 1.0;  // phi_1 (phi_0 = 1)
  const double ck = cload(c + k);
  const bool b3 = j >= 2 && beta1 != 0.0;
  return {(T)ck, (T)alpha, (T)beta1, b3};
}

template <int I, int N, class F>
__device__ __forceinline__ void qsun_each(F&& f) {
  if constexpr (I < N) {  // (none when I >= N)
    f(std::integral_constant<int, I>{});
    qsun_each<I + 1, N>(f);
  }
}

// The resident form: GR * W rows per lane, T = 2^NR blocks.  A step takes the GR
// planes of E rows (16 bytes) of a lane at a time: their sums h = H~ b2, then
// cx X + ch h + cb b3 over b3.  The flips go by the grain spin that they flip, so
// that the plane each LDS read adds to is known to the compiler: a read costs no
// address arithmetic (planes lie at constant offsets) but one XOR per flip.
template <typename T, int GR, int W, int NR>
__device__ __forceinline__ bool qsun_resident(const QsunTeamArgs& A, TeamShared& sh,
                                              TeamPlace& me, const QsunTeamOp* op,
                                              const QsunJob& jb) {
  // a lane's rows of one grain state: H vectors of E rows (at most 16 bytes)
  constexpr int E = W * sizeof(T) > 16 ? 16 / (int)sizeof(T) : W, H = W / E;
  constexpr uint32_t ub = E * sizeof(T);
  typedef typename VT<T, E>::t pt;
  constexpr int P = GR * H;  // planes: vector p / GR of grain state p % GR
  constexpr int lgr = GR == 16 ? 4 : 3, lw = W == 4 ? 2 : W == 2 ? 1 : 0;
  constexpr int LB = 8;  // loads in flight, local and remote
  // the diagonal: kept, or added up from its two parts in FP64 each step
  constexpr bool kDiagReg = sizeof(T) == 4;
  const int64_t D = cload(&op->D);
  const uint32_t nthr = (uint32_t)(D >> (lgr + lw + NR));
  const int lt = W > 1 ? kQsunLane : __builtin_ctz(nthr);  // (W > 1: whole blocks)
  const bool on = uni(threadIdx.x) < nthr;  // (lanes past nthr < 64 repeat others)
  const uint32_t tid = threadIdx.x & (nthr - 1u);
  constexpr uint32_t PS = kQsunThreads * ub;       // bytes of a plane in LDS
  const uint32_t ps = nthr * ub, base = tid * ub;  // in memory
  const uint32_t idx = uni(me.idx);
  auto plane = [&](uint32_t blk, int p) { return (blk * P + (uint32_t)p) * ps; };
  const int64_t row0 = (int64_t)(idx * nthr + tid) << (lgr + lw);
  __amdgpu_buffer_rsrc_t out = rsrc_of(jb.work, (uint32_t)(D * sizeof(T)));
  __amdgpu_buffer_rsrc_t in = rsrc_of(jb.work + D * (int64_t)sizeof(T), (uint32_t)(D * sizeof(T)));

  // flips 0 .. lw-1 stay in the lane, the next lt change the lane or wave, the next
  // NR the block
  const T* cp = QsunTeamOf<T>::c(op);
  const uint32_t local = ((1u << lt) - 1u) << lw;
  const uint64_t gsel = cload(&op->gsel);
  const T* Gp = QsunTeamOf<T>::G(op);

  pt x[P], u[P], v[P];  // X, b2, b3 (the last two in turns)
  double dB[W];         // diagonal of grain state 0
  T dg[kDiagReg ? GR : 1][W];
  {
    const double* X = jb.X + row0;
    const T c0 = (T)cload(jb.coefs + jb.K);
#pragma unroll
    for (int p = 0; p < P; ++p) {
      T t[E];
#pragma unroll
      for (int e = 0; e < E; ++e)
        t[e] = on ? (T)as_global(X)[((p / GR) * E + e) * GR + p % GR] : (T)0;
      if constexpr (E == 1) x[p] = t[0];
      else
#pragma unroll
        for (int e = 0; e < E; ++e) x[p][e] = t[e];
      u[p] = c0 * x[p];
      v[p] = (pt)(T)0;
      if (NR > 0 && on && jb.K > 0) bstore<pt>(u[p], out, base, plane(idx, p));
    }
    const double sc = cload(&op->scale), sf = cload(&op->shift);
    const int lb = cload(&op->lb);
    const double* dlo = cload(&op->qdiag);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int64_t r = row0 + w * GR;
      const double d = (as_global(dlo)[r & (((int64_t)1 << lb) - 1)] +
                        as_global(dlo)[((int64_t)1 << lb) + (r >> lb)] - sf) * sc;
      dB[w] = d;
#pragma unroll
      for (int g = 0; g < GR; ++g)
        if constexpr (kDiagReg) dg[g][w] = (T)(d + cload(op->A64 + g));
    }
  }
  auto step = [&](int j, pt(&u)[P], pt(&v)[P]) __attribute__((always_inline)) {
    const QsunCoef<T> f = qsun_coef<T>(A.polytype, jb.coefs, jb.K, j);
    if (!team_step_end(A.ctl, sh, me, false, [&] {
          if (on) {
#pragma unroll
            for (int p = 0; p < P; ++p) lwrite<pt>(base + p * PS, u[p]);
          }
        }))
      return false;
    {
      const __amdgpu_buffer_rsrc_t t = in;
      in = out;
      out = t;
    }
    if (!on) return true;
    uint32_t at = base;
    qsun_each<0, H>([&](auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value, p0 = q * GR;
      uint64_t z;  // opaque zero: coefficients are read again, not kept in spilled registers
      asm volatile("s_mov_b64 %0, 0" : "=s"(z));
      pt h[GR];
#pragma unroll
      for (int g = 0; g < GR; ++g) h[g] = (pt)(T)0;
      // The sums so far and the address become opaque: loads are not moved before
      // the sums of earlier ones, which would need their registers at once.
      auto fence = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < GR; g += 4)
          asm volatile("" : "+v"(h[g]), "+v"(h[g + 1]), "+v"(h[g + 2]), "+v"(h[g + 3]), "+v"(at));
      };
      // part t of the remote flips, loaded before some local work and added after it
      constexpr int kParts = NR * GR / LB;
      auto remote = [&](auto tc, auto&& work) __attribute__((always_inline)) {
        constexpr int t = decltype(tc)::value, n = t * LB / GR, g0 = t * LB % GR;
        if constexpr (t < kParts) {
          const int jr = lw + lt + n;
          const int m = 1 << ((uint32_t)(gsel >> (2 * jr)) & 3u);
          const T c = cload(cp + jr + z);
          pt r[LB];
#pragma unroll
          for (int g = 0; g < LB; ++g)
            r[g] = bload<pt>(in, at, plane(idx ^ (1u << n), p0 + ((g0 + g) ^ m)));
          work();
#pragma unroll
          for (int g = 0; g < LB; ++g) h[g0 + g] += c * r[g];
          fence();
        } else {
          work();
        }
      };
      auto grain = [&](auto gc) __attribute__((always_inline)) {
        constexpr int g0 = decltype(gc)::value * LB;
#pragma unroll
        for (int g = g0; g < g0 + LB; ++g) {
#pragma unroll
          for (int b = 0; b < GR; ++b)
            if (b != g) h[g] += cload(Gp + z + g * GR + b) * u[p0 + b];
          const double a = kDiagReg ? 0.0 : cload(op->A64 + z + g);
          pt d;
          if constexpr (E == 1) d = kDiagReg ? dg[kDiagReg ? g : 0][q] : (T)(dB[q] + a);
          else
#pragma unroll
            for (int e = 0; e < E; ++e)
              d[e] = kDiagReg ? dg[kDiagReg ? g : 0][q * E + e] : (T)(dB[q * E + e] + a);
          h[g] += d * u[p0 + g];
        }
        fence();
      };
      // the flips of the lane and wave bits that flip grain spin k
      auto flips = [&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, m = 1 << k;
        const uint32_t all = cload(&op->gset[k]);
#pragma unroll
        for (int l = 0; l < lw; ++l)
          if (all >> l & 1u) {
            const T c = cload(cp + l + z);
            const int o = ((1 << l) / E) * GR;  // (the vector of rows w ^ 2^l)
#pragma unroll
            for (int g = 0; g < GR; ++g)
              if constexpr (E > 1) {
#pragma unroll
                for (int e = 0; e < E; ++e)
                  h[g][e] += c * u[(p0 ^ o) + (g ^ m)][e ^ ((1 << l) % E)];
              } else {
                h[g] += c * u[(p0 ^ o) + (g ^ m)];
              }
            fence();
          }
        for (uint32_t set = all & local; set != 0; set &= set - 1u) {
          const int f = __builtin_ctz(set);
          const T c = cload(cp + f);
          const uint32_t from = at ^ (ub << (f - lw));
#pragma unroll
          for (int g0 = 0; g0 < GR; g0 += LB) {
            pt y[LB];
#pragma unroll
            for (int n = 0; n < LB; ++n) y[n] = lread<pt>(from + (uint32_t)(p0 + g0 + n) * PS);
#pragma unroll
            for (int n = 0; n < LB; ++n) h[(g0 + n) ^ m] += c * y[n];
          }
          fence();
        }
      };
      constexpr int kSlots = GR / LB + lgr;
      qsun_each<0, kSlots>([&](auto tc) __attribute__((always_inline)) {
        remote(tc, [&]() __attribute__((always_inline)) {
          constexpr int t = decltype(tc)::value;
          // (the largest terms last)
          if constexpr (t < lgr) flips(tc);
          else grain(std::integral_constant<int, t - lgr>{});
        });
      });
      qsun_each<kSlots, kParts>([&](auto tc) __attribute__((always_inline)) { remote(tc, [] {}); });
#pragma unroll
      for (int g = 0; g < GR; ++g) {
        pt o = f.cx * x[p0 + g] + f.ch * h[g];
        if (f.b3) o += f.cb * v[p0 + g];
        v[p0 + g] = o;
        if (NR > 0 && j < jb.K) bstore<pt>(o, out, base, plane(idx, p0 + g));
      }
    });
    return true;
  };
  auto finish = [&](const pt(&r)[P]) {
    if (!on) return;
    double* Y = jb.Y + row0;
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int e = 0; e < E; ++e)
        as_global(Y)[((p / GR) * E + e) * GR + p % GR] = (double)vget<T, E>(r[p], e);
  };
  for (int j = 1; j <= jb.K; j += 2) {
    if (!step(j, u, v)) return false;
    if (j == jb.K) {
      finish(v);
      return true;
    }
    if (!step(j + 1, v, u)) return false;
  }
  finish(u);
  return true;
}

// A lane per row, b2 and b3 in memory (any team size and D).
template <typename T>
__device__ __forceinline__ bool qsun_stream(const QsunTeamArgs& A, TeamShared& sh,
                                                      TeamPlace& me, const QsunTeamOp* op,
                                                      const QsunJob& jb) {
  constexpr uint32_t sz = sizeof(T);
  const int64_t D = op->D;
  const uint32_t bytes = (uint32_t)(D * sz);
  const int lgr = op->lgr, nf = op->nf, lb = op->lb;
  const uint32_t gr = 1u << lgr;
  const double *dlo = op->qdiag, *dhi = dlo + ((int64_t)1 << lb);
  const T *G = QsunTeamOf<T>::G(op), *c = QsunTeamOf<T>::c(op);
  for (int j = 0; j <= jb.K; ++j) {
    const QsunCoef<T> f = qsun_coef<T>(A.polytype, jb.coefs, jb.K, j);
    const __amdgpu_buffer_rsrc_t out = rsrc_of(jb.work + (j & 1) * (int64_t)bytes, bytes);
    const __amdgpu_buffer_rsrc_t b2 = rsrc_of(jb.work + (1 - (j & 1)) * (int64_t)bytes, bytes);
    for (uint32_t r = me.idx * kQsunThreads + threadIdx.x; r < D; r += me.n * kQsunThreads) {
      T o = f.cx * (T)as_global(jb.X)[r];
      if (j > 0) {
        const uint32_t a = r & (gr - 1u), r0 = r - a;
        const double d = (as_global(dlo)[r & ((1u << lb) - 1u)] + as_global(dhi)[r >> lb] -
                          op->shift) * op->scale;
        T h = (T)d * bload<T>(b2, r * sz, 0);
        for (uint32_t b = 0; b < gr; ++b)
          if (b != a) h += G[a * gr + b] * bload<T>(b2, (r0 + b) * sz, 0);
        for (int i = 0; i < nf; ++i)
          h += c[i] * bload<T>(b2, (r ^ ((1u << (op->gsel >> (2 * i) & 3u)) | (gr << i))) * sz, 0);
        o += f.ch * h;
        if (f.b3) o += f.cb * bload<T>(out, r * sz, 0);
      }
      if (j < jb.K) bstore<T>(o, out, r * sz, 0);
      else as_global(jb.Y)[r] = (double)o;
    }
    if (j < jb.K && !team_step_end(A.ctl, sh, me, false, [] {})) return false;
  }
  return true;
}

template <typename T, int NR>
__device__ __forceinline__ bool qsun_job(const QsunTeamArgs& A, TeamShared& sh, TeamPlace& me,
                                         const QsunTeamOp* op, const QsunJob& jb) {
  const int lgr = (int)cload(&op->lgr);
  const int64_t lanes = cload(&op->D) >> (NR + lgr);  // grain blocks of a block
  if (me.n == (1u << NR) && lanes >= 1) {
    constexpr bool f32 = sizeof(T) == 4;
    if (lgr == 4) {
      if (lanes <= kQsunThreads) return qsun_resident<T, 16, 1, NR>(A, sh, me, op, jb);
      if constexpr (f32)
        if (lanes <= 2 * kQsunThreads) return qsun_resident<T, 16, 2, NR>(A, sh, me, op, jb);
    } else {
      if (lanes <= kQsunThreads) return qsun_resident<T, 8, 1, NR>(A, sh, me, op, jb);
      if (lanes <= 2 * kQsunThreads) return qsun_resident<T, 8, 2, NR>(A, sh, me, op, jb);
      if constexpr (f32)
        if (lanes <= 4 * kQsunThreads) return qsun_resident<T, 8, 4, NR>(A, sh, me, op, jb);
    }
  }
  return qsun_stream<T>(A, sh, me, op, jb);
}

__device__ __forceinline__ QsunJob qsun_job_at(const QsunTeamArgs& A, uint32_t j) {
  if (A.jobs) {
    QsunJob jb;
    const QsunJob* p = A.jobs + j;
    jb.X = cload(&p->X);
    jb.Y = cload(&p->Y);
    jb.coefs = cload(&p->coefs);
    jb.work = cload(&p->work);
    jb.op = cload(&p->op);
    jb.K = cload(&p->K);
    jb.dtype = cload(&p->dtype);
    return jb;
  }
  QsunJob jb = A.one;
  jb.X += j * A.ldx;
  jb.Y += j * A.ldy;
  return jb;
}

template <int NR>
__global__ __launch_bounds__(kQsunThreads) void qsun_team_kernel(const QsunTeamArgs A) {
  TeamShared& sh = *reinterpret_cast<TeamShared*>(team_lds + A.lds);
  TeamPlace me{};
  if (!team_enter(A.ctl, (uint32_t)A.expect, (uint32_t)A.T, sh, me, [] {})) return;
  const int64_t slot = uni(sh.slot);
  if (!A.jobs && slot >= A.nslots) return;  // (uniform over the team)
  while (true) {
    if (!team_next(A.ctl, sh, me)) return;
    const uint32_t j = uni(sh.job);
    if (j >= (uint32_t)A.njobs) return;
    QsunJob jb = qsun_job_at(A, j);
    if (!A.jobs) jb.work += slot * 2 * cload(&A.ops->D) * (jb.dtype == PF_F64 ? 8 : 4);
    const QsunTeamOp* op = A.ops + jb.op;
    const bool ok = jb.dtype == PF_F64 ? qsun_job<double, NR>(A, sh, me, op, jb)
                                       : qsun_job<float, NR>(A, sh, me, op, jb);
    if (!ok) return;
    if (threadIdx.x == 0 && me.idx == 0) (void)team_add(&A.ctl->done, 1u);
  }
}

// An operator's record to device memory, by value (for a captured launch).
__global__ void qsun_record_kernel(QsunTeamOp* dst, const QsunTeamOp rec) {
  const uint32_t* s = reinterpret_cast<const uint32_t*>(&rec);
  for (uint32_t t = threadIdx.x; t < sizeof(QsunTeamOp) / 4; t += blockDim.x)
    reinterpret_cast<uint32_t*>(dst)[t] = s[t];
}
// NaN for every job when one was not finished (never a partial result)
__global__ void qsun_end_kernel(const QsunTeamArgs A) {
  if (A.ctl->done == (uint32_t)A.njobs && A.ctl->abort == 0) return;
  for (int j = 0; j < A.njobs; ++j) {
    const QsunJob jb = qsun_job_at(A, j);
    const int64_t D = A.ops[jb.op].D;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < D;
         r += (int64_t)gridDim.x * blockDim.x)
      jb.Y[r] = __builtin_nan("");
  }
}

// ------------------------------------------------------------------ host
size_t qsun_team_op_bytes() { return sizeof(QsunTeamOp); }

void qsun_team_op(const pf_op* op, void* rec) {
  QsunTeamOp& q = *static_cast<QsunTeamOp*>(rec);
  std::memset(&q, 0, sizeof(q));
  const QsunParams& P = op->qsun;
  const Affine af = op->affine(true);
  const int dg = 1 << P.Lg;
  const int lgr = std::max<int>(P.Lg, 3), fold = lgr - P.Lg, gr = 1 << lgr;
  q.D = op->D;
  q.lgr = lgr;
  q.nf = P.Lloc - fold;
  q.lb = op->qlb;
  q.qdiag = op->qdiag;
  q.scale = af.scale;
  q.shift = af.shift;
  auto put = [&](int r, int c, double v) {
    q.G64[r * gr + c] = v * af.scale;
    q.G32[r * gr + c] = (float)(v * af.scale);
  };
  for (int r = 0; r < gr; ++r) {
    double a = P.G[(r & (dg - 1)) * (dg + 1)] - P.G[0];
    for (int b = 0; b < dg; ++b) put(r, (r & ~(dg - 1)) | b, P.G[(r & (dg - 1)) * dg + b]);
    for (int j = 0; j < fold; ++j) {
      put(r, r ^ (int)P.flip[j], P.coup[j]);
      if (r >> (P.Lg + j) & 1) a += P.h[j];
    }
    q.A64[r] = a * af.scale;
  }
  for (int j = fold; j < P.Lloc; ++j) {
    const int g = __builtin_ctz(P.flip[j]);
    q.gsel |= (uint64_t)g << (2 * (j - fold));
    q.gset[g] |= 1u << (j - fold);
    q.c64[j - fold] = P.coup[j] * af.scale;
    q.c32[j - fold] = (float)(P.coup[j] * af.scale);
  }
}

// The record holds 3 grain spins, a vector's offsets 32 bits.
bool qsun_team_ok(const pf_op* op) {
  return op->qsun.Lg + op->qsun.Lloc >= 3 && op->D * 8 < ((int64_t)1 << 31);
}

// Whether a team of 2^lt blocks holds the operator, and the us of a step: measured
// 1.7 (2^11 rows, one block) to 3.1 (2^13) in FP64, 1.4 to 4.1 (2^14) in FP32, and
// 0.15 us for each doubling of the team.
bool qsun_team_fits(const pf_op* op, int dtype, int lt) {
  const int lgr = std::max<int>(op->qsun.Lg, 3);
  return (op->D >> (lgr + lt)) >= 1 && (size_t)(op->D >> lt) <= qsun_rows(dtype == PF_F64 ? 8 : 4);
}
double qsun_team_step_us(const pf_op* op, int dtype, int lt) {
  const double rows = (double)(op->D >> lt) / (1 << 13);  // of a block
  return 1.4 + 0.15 * lt + rows * (dtype == PF_F64 ? 1.9 : 1.3);
}

// A step of the per-step launches on `elems` rows x columns: launch-bound below 4.5
// us, then 1 TB/s of one vector's bytes (FP64, 3.2 M rows: 26 us for 25 MB).
double qsun_per_step_us(double elems, int dtype) {
  return std::max(4.5, elems * (dtype == PF_F64 ? 8 : 4) / 1e6);
}

// Launches the jobs (null: columns of `one`) on teams of T blocks.
static void qsun_team_launch(const pf_handle* h, QsunTeamArgs A, int T, hipStream_t st) {
  A.T = T;
  const int cus = std::max(1, h->prop.multiProcessorCount);
  const int nxcd = std::max(1, cus / 32);
  const int grid = std::max(T, cus / nxcd * nxcd);
  A.expect = grid / nxcd;
  // (64 KB of rows; more than half of a CU's LDS, so that a CU takes one block, as
  // the teams are counted)
  A.lds = 96u * 1024u;
  const size_t dyn = A.lds + sizeof(TeamShared);
#define PF_QSUN_TEAM(NR)                                                               \
  {                                                                                    \
    auto* k = qsun_team_kernel<NR>;                                                    \
    PF_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k),                       \
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn)); \
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(kQsunThreads), dyn, st, A);       \
  }
  switch (T) {
    case 1: PF_QSUN_TEAM(0) break;
    case 2: PF_QSUN_TEAM(1) break;
    case 4: PF_QSUN_TEAM(2) break;
    case 8: PF_QSUN_TEAM(3) break;
    case 16: PF_QSUN_TEAM(4) break;
    default: PF_QSUN_TEAM(5) break;
  }
#undef PF_QSUN_TEAM
  PF_HIP(hipGetLastError());
  hipLaunchKernelGGL(qsun_end_kernel, dim3(256), dim3(256), 0, st, A);
  PF_HIP(hipGetLastError());
}
void qsun_team_batch(const pf_handle* h, const void* recs,
                     const QsunJob* jobs, int njobs, int polytype, int T, void* ctl,
                     hipStream_t st) {
  QsunTeamArgs A{};
  A.ops = static_cast<const QsunTeamOp*>(recs);
  A.jobs = jobs;
  A.njobs = njobs;
  A.polytype = polytype;
  A.ctl = static_cast<TeamCtl*>(ctl);
  team_begin(ctl, nullptr, nullptr, -1, st);
  qsun_team_launch(h, A, T, st);
}

static size_t qsun_align(size_t n) { return (n + 255) & ~(size_t)255; }
size_t qsun_team_work_bytes(const pf_op* op, int dtype, int order, int ncols, int T) {
  return team_ctl_bytes() + qsun_align(sizeof(QsunTeamOp)) + qsun_align((size_t)(order + 1) * 8) +
         (size_t)std::min(ncols, 8 * (32 / T)) * 2 * op->D * (dtype == PF_F64 ? 8 : 4);
}
void qsun_team_filter(pf_op* op, int dtype, int polytype, const double* coeffs, int order,
                      const double* X, int64_t ldx, double* Y, int64_t ldy, int ncols, int T,
                      void* work, hipStream_t st) {
  char* p = static_cast<char*>(work);
  QsunTeamOp* rec = reinterpret_cast<QsunTeamOp*>(p + team_ctl_bytes());
  double* cdev = reinterpret_cast<double*>((char*)rec + qsun_align(sizeof(QsunTeamOp)));
  team_begin(p, cdev, coeffs, order, st);
  QsunTeamOp host;
  qsun_team_op(op, &host);
  hipLaunchKernelGGL(qsun_record_kernel, dim3(1), dim3(1024), 0, st, rec, host);
  PF_HIP(hipGetLastError());
  QsunTeamArgs A{};
  A.ops = rec;
  A.one = QsunJob{X, Y, cdev, (char*)cdev + qsun_align((size_t)(order + 1) * 8), 0, order, dtype, 0};
  A.ldx = ldx;
  A.ldy = ldy;
  A.njobs = ncols;
  A.nslots = std::min(ncols, 8 * (32 / T));
  A.polytype = polytype;
  A.ctl = reinterpret_cast<TeamCtl*>(p);
  qsun_team_launch(op->h, A, T, st);
}

}  // namespace pf
