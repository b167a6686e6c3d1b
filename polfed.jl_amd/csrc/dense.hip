// Dense FP64 block kernels of the block-Lanczos step: tall-skinny Gram
// products A^T B and updates B = beta B + alpha A G on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64), Cholesky-QR, small rotations and residual norms.
//
// MFMA f64 16x16x4 operand layout used here (lane l of a 64-wide wave):
//   A fragment (16 x 4): lane l holds A[l % 16][l / 16]
//   B fragment (4 x 16): lane l holds B[l / 16][l % 16]
//   C/D (16 x 16):       lane l, register v holds D[l/16 + 4*v][l % 16]
// (output layout measured on gfx950 with an in-bounds probe of known inputs).
// The contraction index k only has to agree between the A and B fragments, so
// the Gram kernel assigns k-slot l/16 to rows 4*(l/16)+q of a 16-row slab for
// the q-th of four MFMAs: each lane then loads 4 consecutive rows (32 bytes) of
// one column and 4 lanes cover a full 128-byte line.

#include <algorithm>
#include <cmath>
#include <cstring>

#include "pf_internal.h"

namespace pf {

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma16x16x4(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Row partitions of the Gram reduction, each a contiguous range of rows (616 MB, 416
// columns: 162 us with every 256th slab, 136 so; 145 with 128 ranges of twice the
// columns per wave, 153 with 512), half of it for one tile of columns, whose
// partials one block adds up.
constexpr int kGramRowBlocks = 256, kGramRowBlocks1 = 128;
constexpr int kMaxN = 64;            // widest B block of the Gram/update kernels

// WS: A has at most 16 columns; the four waves take a quarter of the slabs each and add
// their tiles in LDS (184756 x 8: 28.4 us with three waves idle, 10.1 us so).
//
// Gram partials: part[(rb * m + i) * n + j] = sum over rb's slabs of A[:, i] B[:, j].
// Grid: (kGramRowBlocks, ceil(m/(64*AT))); block: 4 waves, wave w owns the AT
// tiles of 16 A columns from i0 = 64*AT*blockIdx.y + 16*AT*w and all n columns
// of B (NT <= 4 tiles), so each B load serves AT A tiles.  Row block rb
// takes a contiguous range of slabs (16 rows), two at a time with every load issued
// before the first MFMA.  Lanes past m or n
// read a clamped column (their results are not stored); only the rows past D
// of the last, partial slab are zeroed.
template <int NT, int AT, bool WS = false>
__global__ __launch_bounds__(256) void gram_kernel(const double* __restrict__ A, int64_t lda, int m,
                                                   const double* __restrict__ B, int64_t ldb, int n,
                                                   int64_t D, double* __restrict__ part) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i0 = WS ? 0 : (blockIdx.y * 64 + w * 16) * AT;
  const int li = lane & 15, kq = lane >> 4;
  const double* pa[AT];
#pragma unroll
  for (int a = 0; a < AT; ++a) {
    const int ia = i0 + 16 * a + li;
    pa[a] = A + (int64_t)(ia < m ? ia : m - 1) * lda;
  }
  const double* pb[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int jb = t * 16 + li;
    pb[t] = B + (int64_t)(jb < n ? jb : n - 1) * ldb;
  }
  d4 acc[AT][NT];
#pragma unroll
  for (int a = 0; a < AT; ++a)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[a][t] = (d4){0.0, 0.0, 0.0, 0.0};
  // one slab's loads (rows r0..r0+3 of this lane) and MFMAs; zero rows >= D
  // only when `tail`
  auto load = [&](int64_t r0, bool tail, double (&av)[AT][4], double (&bv)[NT][4]) {
#pragma unroll
    for (int a = 0; a < AT; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) av[a][q] = (!tail || r0 + q < D) ? pa[a][r0 + q] : 0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) bv[t][q] = (!tail || r0 + q < D) ? pb[t][r0 + q] : 0.0;
  };
  auto fma = [&](const double (&av)[AT][4], const double (&bv)[NT][4]) {
#pragma unroll
    for (int a = 0; a < AT; ++a)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[a][t] = mfma16x16x4(av[a][q], bv[t][q], acc[a][t]);
  };
  const int64_t gx = WS ? 4 * gridDim.x : gridDim.x, nfull = D / 16;
  const int64_t first = WS ? 4 * blockIdx.x + w : blockIdx.x;
  const int64_t end = (first + 1) * nfull / gx;
  int64_t sl = first * nfull / gx;
  for (; sl + 1 < end; sl += 2) {
    double av0[AT][4], bv0[NT][4], av1[AT][4], bv1[NT][4];
    load(sl * 16 + 4 * kq, false, av0, bv0);
    load((sl + 1) * 16 + 4 * kq, false, av1, bv1);
    fma(av0, bv0);
    fma(av1, bv1);
  }
  if (sl < end) {  // one full slab left
    double av[AT][4], bv[NT][4];
    load(sl * 16 + 4 * kq, false, av, bv);
    fma(av, bv);
  }
  if (D % 16 != 0 && first == gx - 1) {  // the partial last slab
    double av[AT][4], bv[NT][4];
    load(nfull * 16 + 4 * kq, true, av, bv);
    fma(av, bv);
  }
  if constexpr (WS) {
    __shared__ d4 sum[3][NT][64];
    if (w > 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) sum[w - 1][t][lane] = acc[0][t];
    }
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int k = 0; k < 3; ++k) acc[0][t] += sum[k][t][lane];
  }
  // D-fragment: row (A column) i0 + 16a + kq + 4*v, column (B column) 16*t + li
  double* out = part + (int64_t)blockIdx.x * m * n;
#pragma unroll
  for (int a = 0; a < AT; ++a)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int j = t * 16 + li;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = i0 + 16 * a + kq + 4 * v;
        if (i < m && j < n) out[(int64_t)i * n + j] = acc[a][t][v];
      }
    }
}

// G[i*gsi + j*gsj] = sum_rb part[(rb*m + i)*n + j]  (fixed order:
// deterministic).  Eight lanes per entry take every eighth partial, 16 loads at a
// time, and add their sums pairwise (416 x 8 entries: 8.7 us for 128 partials with a
// lane per entry, 5.1 us so for 256).
__global__ __launch_bounds__(256) void gram_reduce_kernel(const double* __restrict__ part, int nrb,
                                                          int m, int n, double* __restrict__ G,
                                                          int64_t gsi, int64_t gsj) {
  // lanes of consecutive entries, so that each load is one line
  const int e = threadIdx.x & 31, k = threadIdx.x >> 5;
  const int64_t idx = (int64_t)blockIdx.x * 32 + e;
  const int64_t stride = (int64_t)m * n;
  __shared__ double red[8][32];
  constexpr int U = 16;
  double t = 0.0;
  if (idx < stride) {
    for (int rb = k; rb < nrb; rb += 8 * U) {
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = rb + 8 * u < nrb ? part[(rb + 8 * u) * stride + idx] : 0.0;
#pragma unroll
      for (int u = 0; u < U; ++u) t += v[u];
    }
  }
  red[k][e] = t;
  __syncthreads();
  if (k == 0 && idx < stride) {
    const double a = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
    const double b = (red[4][e] + red[5][e]) + (red[6][e] + red[7][e]);
    G[(idx / n) * gsi + (idx % n) * gsj] = a + b;
  }
}

// B = beta*B + alpha*A*G.  Block: 4 waves; a wave takes 16*RT rows in RT tiles and
// all n output columns (NT tiles of 16).  Lane l holds rows RT*(l%16) .. +RT-1 of its
// wave (tile t the rows RT*i + t), so that one load of 8*RT bytes per lane serves RT
// tiles and a fragment of G as many.  Contraction over the m columns of A in steps
// of 4: column k + l/16 of A, G(k + l/16, 16t + l%16), element (k, j) at
// G[k*gsk + j*gsj] (row-major G, gsj = 1, gives the 16 lanes of a k-slot one 128-byte
// line).  Four steps' loads are issued before their MFMAs.  Lanes past D or n read
// a clamped row or column (their results are not stored); only the contraction
// slots past m in the last steps are zeroed.  RT = 2: 614 MB, 8 columns, in 122 us
// (5.0 TB/s); one row per lane 151, four 121 but slower for 16 columns.
template <int NT, int RT>
__global__ __launch_bounds__(256) void update_kernel(const double* __restrict__ A, int64_t lda,
                                                     int m, const double* __restrict__ G,
                                                     int64_t gsk, int64_t gsj,
                                                     double* __restrict__ B, int64_t ldb, int n,
                                                     int64_t D, double alpha, double beta) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int li = lane & 15, kq = lane >> 4;
  const int64_t r0 = ((int64_t)blockIdx.x * 64 + w * 16) * RT;
  if (r0 >= D) return;
  const int64_t ra = r0 + RT * li;
  const bool tail = r0 + 16 * RT > D;  // (uniform)
  typedef double vt __attribute__((ext_vector_type(RT)));
  typedef double ut __attribute__((ext_vector_type(RT), aligned(8)));
  auto load = [&](int64_t col) {
    if (!tail) return (vt) * reinterpret_cast<const ut*>(A + ra + col * lda);
    vt v;
#pragma unroll
    for (int q = 0; q < RT; ++q) v[q] = A[(ra + q < D ? ra + q : D - 1) + col * lda];
    return v;
  };
  const double* pg[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = t * 16 + li;
    pg[t] = G + (int64_t)(j < n ? j : n - 1) * gsj;
  }
  d4 acc[RT][NT];
#pragma unroll
  for (int q = 0; q < RT; ++q)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[q][t] = (d4){0.0, 0.0, 0.0, 0.0};
  constexpr int U = 4;  // steps of 4 columns whose loads travel together
  int k = 0;
  for (; k + 4 * U <= m; k += 4 * U) {
    vt a[U];
    double g[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ka = k + 4 * u + kq;
      a[u] = load(ka);
#pragma unroll
      for (int t = 0; t < NT; ++t) g[u][t] = pg[t][ka * gsk];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[q][t] = mfma16x16x4(a[u][q], g[u][t], acc[q][t]);
  }
  for (; k < m; k += 4) {
    const int ka = k + kq;
    const bool kok = ka < m;
    const int kc = kok ? ka : m - 1;
    vt a = load(kc);
    if (!kok) a = (vt)0.0;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const double g = pg[t][kc * gsk];
#pragma unroll
      for (int q = 0; q < RT; ++q) acc[q][t] = mfma16x16x4(a[q], g, acc[q][t]);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = t * 16 + li;
    if (j >= n) continue;
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t r = r0 + RT * (kq + 4 * v) + q;  // row kq + 4v of tile q
        if (r < D) {
          double* pb = B + r + (int64_t)j * ldb;
          const double old = (beta == 0.0) ? 0.0 : beta * *pb;
          *pb = old + alpha * acc[q][t][v];
        }
      }
  }
}

// dst[r, :] = src[r, :] * M for an n x n matrix M (column-major), one row per
// thread held in N >= n registers (an array of run-time length went through
// scratch memory: 184756 x 8 took 21.7 us, 6.5 us so); TRI: M is upper triangular.
// src and dst may be the same block.  `skip`: nothing is written when it is set.
template <int N, bool TRI>
__global__ __launch_bounds__(256) void rotate_kernel(const double* src, int64_t lds, double* dst,
                                                     int64_t ldd, int64_t D, int n,
                                                     const double* __restrict__ M,
                                                     const int* __restrict__ skip) {
  __shared__ double sM[N * N];
  if (skip && *skip) return;  // (uniform)
  for (int i = threadIdx.x; i < n * n; i += blockDim.x) sM[(i / n) * N + i % n] = M[i];
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= D) return;
  double row[N];
#pragma unroll
  for (int i = 0; i < N; ++i) row[i] = i < n ? src[r + (int64_t)i * lds] : 0.0;
  if constexpr (TRI) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (j >= n) break;
      double t = 0.0;
#pragma unroll
      for (int i = 0; i <= j; ++i) t += row[i] * sM[i + j * N];
      dst[r + (int64_t)j * ldd] = t;
    }
  } else {
    for (int j = 0; j < n; ++j) {
      double t = 0.0;
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (i < n) t += row[i] * sM[i + j * N];
      dst[r + (int64_t)j * ldd] = t;
    }
  }
}

// G = the sums of nrb partials of nn <= 256 entries, in one block of 1024 threads (I:
// 1024 doubles): the threads of an entry add their partials, eight loads in flight,
// then one adds these.
__device__ __forceinline__ void sum_partials(const double* __restrict__ part, int nrb, int nn,
                                             double* I, double* G) {
  const int t = threadIdx.x, g = 1024 / nn, e = t / g, k = t % g;
  double v = 0.0;
  if (e < nn)
    for (int rb = k; rb < nrb; rb += 8 * g) {
      double x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        x[u] = rb + u * g < nrb ? part[(int64_t)(rb + u * g) * nn + e] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) v += x[u];
    }
  I[t] = v;
  __syncthreads();
  if (t < nn) {
    double sum = 0.0;
    for (int i = 0; i < g; ++i) sum += I[t * g + i];
    G[t] = sum;
  }
  __syncthreads();
}

// One pass of Cholesky-QR in one block: G = W^T W from the Gram partials (nrb > 0) or
// already summed in `part`, its factor R (G = R^T R) to Rout, R^-1 to Ri (both n x n,
// column-major, upper).  With Rin (the second pass) Rout gets R * Rin.  A pivot that
// is not above its rounding, or not finite, sets *fail (and *fail_host), and so does a
// set *prev; products are rounded (no fused multiply-add), as on a host.
__global__ __launch_bounds__(1024) void chol_kernel(const double* __restrict__ part, int nrb, int n,
                                                    const double* __restrict__ Rin,
                                                    double* Rout, double* __restrict__ Ri,
                                                    const int* prev, int* fail,
                                                    int* fail_host) {
#pragma clang fp contract(off)
  extern __shared__ double chol_lds[];
  double* G = chol_lds;             // G, then R (row j from column j on)
  double* I = chol_lds + n * n;     // partial sums, the columns' squared norms, the inverse
  const int t = threadIdx.x, nn = n * n;
  auto end = [&](int v) {
    if (t != 0) return;
    *fail = v;
    if (fail_host) *fail_host = v;
  };
  if (prev && *prev) return end(1);  // (uniform)
  if (nrb > 0) {  // n <= 16
    sum_partials(part, nrb, nn, I, G);
  } else {
    for (int i = t; i < nn; i += 1024) G[i] = part[i];
  }
  __syncthreads();
  if (t < n) I[t] = G[t * n + t];
  __syncthreads();
  const int nt = n <= 16 ? 64 : 1024;  // (one wave: its barriers cost nothing)
  if (t >= nt) return;
  for (int j = 0; j < n; ++j) {
    const double d = G[j * n + j];
    // (a repeated column leaves up to four roundings of its norm, of either sign)
    if (!(d > 4.0 * 2.220446049250313e-16 * I[j]) || d > 1.7976931348623157e308)
      return end(1);  // (uniform)
    const double r = sqrt(d);
    __syncthreads();
    if (t == 0) G[j * n + j] = r;
    else if (j + t < n) G[j * n + j + t] /= r;
    __syncthreads();
    const int m = n - 1 - j;
    for (int i = t; i < m * m; i += nt) {
      const int a = j + 1 + i / m, b = j + 1 + i % m;
      if (b >= a) G[a * n + b] -= G[j * n + a] * G[j * n + b];
    }
    __syncthreads();
  }
  if (t < n) {  // column t of the inverse
    I[t * n + t] = 1.0 / G[t * n + t];
    for (int i = t - 1; i >= 0; --i) {
      double v = 0.0;
      for (int k = i + 1; k <= t; ++k) v += G[i * n + k] * I[t * n + k];
      I[t * n + i] = -v / G[i * n + i];
    }
    for (int i = t + 1; i < n; ++i) I[t * n + i] = 0.0;
  }
  __syncthreads();
  for (int e = t; e < nn; e += nt) {
    const int i = e % n, j = e / n;
    Ri[e] = I[e];
    double v = 0.0;
    if (i <= j) {
      if (Rin)
        for (int k = i; k <= j; ++k) v += G[i * n + k] * Rin[k + j * n];
      else v = G[i * n + j];
    }
    Rout[e] = v;
  }
  end(0);
}

// The projections of a three-term step in one block (n <= 16): G = V^T W from its
// partials, a = its upper triangle mirrored, to `a` and to pinned host memory, and
// the transpose of b (by value) to `bt`; all column-major.
struct OrthoB {
  double v[16 * 16];
};
__global__ __launch_bounds__(1024) void ortho_kernel(const double* __restrict__ part, int nrb,
                                                     int n, const OrthoB b, double* a, double* bt,
                                                     double* a_host) {
  __shared__ double I[1024], G[256];
  const int t = threadIdx.x, nn = n * n;
  sum_partials(part, nrb, nn, I, G);
  if (t >= nn) return;
  const int i = t % n, j = t / n;
  const double v = G[(i < j ? i : j) * n + (i < j ? j : i)];
  a[t] = v;
  a_host[t] = v;
  bt[t] = b.v[t];
}

// Column partials of <A_j, B_j> (mode 0) or ||A_j - e_j B_j||^2 (mode 1).
__global__ __launch_bounds__(256) void coldot_kernel(const double* __restrict__ A, int64_t lda,
                                                     const double* __restrict__ B, int64_t ldb,
                                                     int64_t D, const double* __restrict__ e,
                                                     int mode, double* __restrict__ part) {
  __shared__ double red[4];
  const int c = blockIdx.y;
  double acc = 0.0;
  const double ec = mode ? e[c] : 0.0;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < D;
       r += (int64_t)gridDim.x * blockDim.x) {
    const double a = A[r + (int64_t)c * lda], b = B[r + (int64_t)c * ldb];
    if (mode) {
      const double d = a - ec * b;
      acc += d * d;
    } else {
      acc += a * b;
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[(int64_t)c * gridDim.x + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// ---------------------------------------------------------------- drivers
// G(i, j) = <A_i, B_j> stored at G[i*gsi + j*gsj] (column-major: gsi = 1,
// gsj = ldg >= m; row-major: gsi = ldg >= n, gsj = 1).
static int gram_partials(pf_handle* h, const double* A, int64_t lda, int m, const double* B,
                         int64_t ldb, int n, int64_t D, hipStream_t st) {
  const int nrb = (int)std::min<int64_t>(m <= 16 ? kGramRowBlocks1 : kGramRowBlocks, (D + 15) / 16);
  double* part = reinterpret_cast<double*>(h->partials.get((size_t)nrb * m * n * sizeof(double)));
  // Two A tiles per wave where a wide B is loaded for each of them; with one tile of
  // B, 416 columns take 136 us with one A tile per wave and 145 with two.
  const int NT = (n + 15) / 16;
  const int AT = m > 64 && NT > 1 ? 2 : 1;
  dim3 grid(nrb, (m + 64 * AT - 1) / (64 * AT)), block(256);
#define PF_GRAM(...) \
  hipLaunchKernelGGL((gram_kernel<__VA_ARGS__>), grid, block, 0, st, A, lda, m, B, ldb, n, D, part)
  if (m <= 16) {
    switch (NT) {
      case 1: PF_GRAM(1, 1, true); break;
      case 2: PF_GRAM(2, 1, true); break;
      case 3: PF_GRAM(3, 1, true); break;
      default: PF_GRAM(4, 1, true); break;
    }
  } else if (AT == 2) {
    switch (NT) {
      case 2: PF_GRAM(2, 2); break;
      case 3: PF_GRAM(3, 2); break;
      default: PF_GRAM(4, 2); break;
    }
  } else {
    switch (NT) {
      case 1: PF_GRAM(1, 1); break;
      case 2: PF_GRAM(2, 1); break;
      case 3: PF_GRAM(3, 1); break;
      default: PF_GRAM(4, 1); break;
    }
  }
#undef PF_GRAM
  PF_HIP(hipGetLastError());
  return nrb;
}
void gram(pf_handle* h, const double* A, int64_t lda, int m, const double* B, int64_t ldb, int n,
          int64_t D, double* G, int64_t gsi, int64_t gsj, hipStream_t st) {
  PF_REQUIRE(m >= 1 && n >= 1 && n <= kMaxN, "gram: 1 <= n <= 64, m >= 1");
  PF_REQUIRE(D >= 1 && lda >= D && ldb >= D, "gram: bad leading dimensions");
  PF_REQUIRE((gsi == 1 && gsj >= m) || (gsj == 1 && gsi >= n), "gram: bad output layout");
  const int nrb = gram_partials(h, A, lda, m, B, ldb, n, D, st);
  const double* part = reinterpret_cast<const double*>(h->partials.p);
  const int64_t mn = (int64_t)m * n;
  hipLaunchKernelGGL(gram_reduce_kernel, dim3((unsigned)((mn + 31) / 32)), dim3(256), 0, st, part,
                     nrb, m, n, G, gsi, gsj);
  PF_HIP(hipGetLastError());
}

// B = beta*B + alpha*A*G with G(k, j) at G[k*gsk + j*gsj] (column-major:
// gsk = 1, gsj = ldg >= m; row-major: gsk = ldg >= n, gsj = 1).
void update(const double* A, int64_t lda, int m, const double* G, int64_t gsk, int64_t gsj,
            double* B, int64_t ldb, int n, int64_t D, double alpha, double beta, hipStream_t st) {
  PF_REQUIRE(m >= 1 && n >= 1 && n <= kMaxN, "update: 1 <= n <= 64, m >= 1");
  PF_REQUIRE(D >= 1 && lda >= D && ldb >= D, "update: bad leading dimensions");
  PF_REQUIRE((gsk == 1 && gsj >= m) || (gsj == 1 && gsk >= n), "update: bad G layout");
  constexpr int RT = 2;
  dim3 grid((unsigned)((D + 64 * RT - 1) / (64 * RT))), block(256);
  const int NT = (n + 15) / 16;
#define PF_UPDATE(NTV)                                                                         \
  hipLaunchKernelGGL((update_kernel<NTV, RT>), grid, block, 0, st, A, lda, m, G, gsk, gsj, B, ldb, n, \
                     D, alpha, beta)
  switch (NT) {
    case 1: PF_UPDATE(1); break;
    case 2: PF_UPDATE(2); break;
    case 3: PF_UPDATE(3); break;
    default: PF_UPDATE(4); break;
  }
#undef PF_UPDATE
  PF_HIP(hipGetLastError());
}

// per-column reductions returned to the host (fixed order)
static void coldots_host(pf_handle* h, const double* A, int64_t lda, const double* B, int64_t ldb,
                         int64_t D, int n, const double* e_dev, int mode, double* out,
                         hipStream_t st) {
  const int nblk = (int)std::min<int64_t>(256, (D + 255) / 256);
  double* part = reinterpret_cast<double*>(h->partials.get((size_t)nblk * n * sizeof(double)));
  hipLaunchKernelGGL(coldot_kernel, dim3(nblk, n), dim3(256), 0, st, A, lda, B, ldb, D, e_dev, mode,
                     part);
  PF_HIP(hipGetLastError());
  std::vector<double> hp((size_t)nblk * n);
  PF_HIP(hipMemcpyAsync(hp.data(), part, hp.size() * sizeof(double), hipMemcpyDeviceToHost, st));
  PF_HIP(hipStreamSynchronize(st));
  for (int c = 0; c < n; ++c) {
    double t = 0.0;
    for (int b = 0; b < nblk; ++b) t += hp[(size_t)c * nblk + b];
    out[c] = t;
  }
}

template <bool TRI>
static void rotate_launch(const double* src, int64_t lds, double* dst, int64_t ldd, int64_t D,
                          int n, const double* M, const int* skip, hipStream_t st) {
  const dim3 grid((unsigned)((D + 255) / 256)), block(256);
#define PF_ROTATE(N) \
  hipLaunchKernelGGL((rotate_kernel<N, TRI>), grid, block, 0, st, src, lds, dst, ldd, D, n, M, skip)
  if (n == 1) PF_ROTATE(1);
  else if (n <= 4) PF_ROTATE(4);
  else if (n <= 8) PF_ROTATE(8);
  else if (n <= 16) PF_ROTATE(16);
  else if (n <= 32) PF_ROTATE(32);
  else PF_ROTATE(64);
#undef PF_ROTATE
  PF_HIP(hipGetLastError());
}

// Pinned results of the small factorizations: kMaxN^2 doubles and a flag.
static void qr_pinned(pf_handle* h) {
  if (!h->pinned)
    PF_HIP(hipHostMalloc(reinterpret_cast<void**>(&h->pinned),
                         ((size_t)kMaxN * kMaxN + 2) * sizeof(double)));
}

static void rotate(pf_handle* h, double* W, int64_t ldw, int64_t D, int n, const double* M_host,
                   hipStream_t st) {
  PF_REQUIRE(n >= 1 && n <= kMaxN, "rotate: 1 <= n <= 64");
  double* dM = reinterpret_cast<double*>(h->small.get((size_t)n * n * sizeof(double)));
  PF_HIP(hipMemcpyAsync(dM, M_host, (size_t)n * n * sizeof(double), hipMemcpyHostToDevice, st));
  rotate_launch<false>(W, ldw, W, ldw, D, n, dM, nullptr, st);
  // the host matrix may be freed by the caller after return
  PF_HIP(hipStreamSynchronize(st));
}

}  // namespace pf

using namespace pf;

extern "C" int pf_gram(pf_handle* h, const double* A, int64_t lda, int32_t m, const double* B,
                       int64_t ldb, int32_t n, int64_t D, double* G, int32_t ldg, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && A && B && G, "gram: null argument");
    PF_REQUIRE(ldg >= m, "gram: ldg < m");
    gram(h, A, lda, m, B, ldb, n, D, G, 1, ldg, S(stream));
  });
}

extern "C" int pf_gemm_update(pf_handle* h, const double* A, int64_t lda, int32_t m,
                              const double* G, int32_t ldg, double* B, int64_t ldb, int32_t n,
                              int64_t D, double alpha, double beta, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && A && G && B, "update: null argument");
    PF_REQUIRE((const void*)A != (const void*)B, "update: B must not alias A");
    PF_REQUIRE(ldg >= m, "update: ldg < m");
    update(A, lda, m, G, 1, ldg, B, ldb, n, D, alpha, beta, S(stream));
  });
}

extern "C" int pf_reorth(pf_handle* h, const double* V, int64_t ldv, int32_t k, double* W,
                         int64_t ldw, int32_t s, int64_t D, int32_t passes, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && V && W, "reorth: null argument");
    PF_REQUIRE(passes >= 1 && passes <= 4, "reorth: 1 <= passes <= 4");
    if (k <= 0) return;
    hipStream_t st = S(stream);
    // G = V^T W held row-major (G(i, j) at G[i*s + j]): the update's 16 lanes
    // of one contraction index then read one contiguous line of G
    double* G = reinterpret_cast<double*>(h->vecs.get((size_t)k * s * sizeof(double)));
    for (int p = 0; p < passes; ++p) {
      gram(h, V, ldv, k, W, ldw, s, D, G, s, 1, st);
      update(V, ldv, k, G, s, 1, W, ldw, s, D, -1.0, 1.0, st);
    }
  });
}

extern "C" int pf_block_qr(pf_handle* h, double* W, int64_t ldw, int64_t D, int32_t s,
                           double* R_host, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && W && R_host, "qr: null argument");
    PF_REQUIRE(s >= 1 && s <= kMaxN && D >= s && ldw >= D, "qr: bad shape");
    hipStream_t st = S(stream);
    // Two passes on the device, the first into a copy, so that W is unchanged when a
    // factorization breaks down; R and the flags go straight to pinned host memory,
    // and the one wait is at the end.
    qr_pinned(h);
    const size_t ss = (size_t)s * s;
    double* Q = reinterpret_cast<double*>(h->vecs.get(((size_t)D * s + 3 * ss + 2) * sizeof(double)));
    double* dG = Q + (size_t)D * s;
    double *R1 = dG + ss, *Ri = R1 + ss;
    int* flag = reinterpret_cast<int*>(Ri + ss);
    int* flag_host = reinterpret_cast<int*>(h->pinned + ss);
    for (int pass = 0; pass < 2; ++pass) {
      const double* A = pass ? Q : W;
      const int64_t lda = pass ? D : ldw;
      const bool fused = s <= 16;
      int nrb = 0;
      if (fused) nrb = gram_partials(h, A, lda, s, A, lda, s, D, st);
      else gram(h, A, lda, s, A, lda, s, D, dG, 1, s, st);
      const size_t lds = std::max(2 * ss, ss + 1024) * sizeof(double);
      hipLaunchKernelGGL(chol_kernel, dim3(1), dim3(1024), lds, st,
                         fused ? reinterpret_cast<const double*>(h->partials.p) : dG, nrb, s,
                         pass ? R1 : nullptr, pass ? h->pinned : R1, Ri, pass ? flag : nullptr,
                         flag + pass, pass ? flag_host : nullptr);
      PF_HIP(hipGetLastError());
      if (pass == 0) rotate_launch<true>(W, ldw, Q, D, D, s, Ri, flag, st);
      else rotate_launch<true>(Q, D, W, ldw, D, s, Ri, flag + 1, st);
    }
    PF_HIP(hipStreamSynchronize(st));
    if (*flag_host)
      throw Error{PF_ERR_NUMERIC, "qr: Gram matrix not positive definite (rank-deficient block)"};
    std::memcpy(R_host, h->pinned, ss * sizeof(double));
  });
}

extern "C" int pf_lanczos_ortho(pf_handle* h, const double* V, int64_t ldv, const double* Vp,
                                int64_t ldvp, const double* b_host, double* W, int64_t ldw,
                                int64_t D, int32_t s, double* a_host, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && V && W && a_host && (!Vp || b_host), "ortho: null argument");
    PF_REQUIRE(s >= 1 && s <= 16 && D >= 1 && ldv >= D && ldw >= D && (!Vp || ldvp >= D),
               "ortho: bad shape");
    PF_REQUIRE(V != W && Vp != W, "ortho: W must not alias V");
    hipStream_t st = S(stream);
    double* a = reinterpret_cast<double*>(h->small.get(2 * 256 * sizeof(double)));
    double* bt = a + 256;
    qr_pinned(h);
    if (!h->mark) PF_HIP(hipEventCreateWithFlags(&h->mark, hipEventDisableTiming));
    OrthoB b{};
    if (Vp)
      for (int i = 0; i < s; ++i)
        for (int j = 0; j < s; ++j) b.v[j + i * s] = b_host[i + j * s];
    const int nrb = gram_partials(h, V, ldv, s, W, ldw, s, D, st);
    hipLaunchKernelGGL(ortho_kernel, dim3(1), dim3(1024), 0, st,
                       reinterpret_cast<const double*>(h->partials.p), nrb, s, b, a, bt, h->pinned);
    PF_HIP(hipGetLastError());
    PF_HIP(hipEventRecord(h->mark, st));
    update(V, ldv, s, a, 1, s, W, ldw, s, D, -1.0, 1.0, st);
    if (Vp) update(Vp, ldvp, s, bt, 1, s, W, ldw, s, D, -1.0, 1.0, st);
    PF_HIP(hipEventSynchronize(h->mark));  // (the updates are still running)
    std::memcpy(a_host, h->pinned, (size_t)s * s * sizeof(double));
  });
}

extern "C" int pf_rotate(pf_handle* h, double* W, int64_t ldw, int64_t D, int32_t n,
                         const double* M_host, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && W && M_host && ldw >= D && D >= 1, "rotate: bad argument");
    rotate(h, W, ldw, D, n, M_host, S(stream));
  });
}

extern "C" int pf_coldots(pf_handle* h, const double* A, int64_t lda, const double* B, int64_t ldb,
                          int64_t D, int32_t n, double* out_host, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && A && B && out_host && n >= 1 && n <= 65535 && D >= 1 && lda >= D && ldb >= D,
               "coldots: bad argument");
    coldots_host(h, A, lda, B, ldb, D, n, nullptr, 0, out_host, S(stream));
  });
}

extern "C" int pf_residuals(pf_handle* h, pf_op* op, const double* psi, int64_t ld, int32_t nev,
                            double* E_host, double* res_host, pf_stream stream) {
  return guarded([&] {
    PF_REQUIRE(h && op && psi && E_host && res_host, "residuals: null argument");
    PF_REQUIRE(nev >= 1 && nev <= 65535 && ld >= op->D, "residuals: bad shape");
    hipStream_t st = S(stream);
    const int64_t D = op->D;
    // H psi with the same leading dimension as psi (the apply kernels share offsets)
    double* Hpsi = reinterpret_cast<double*>(
        h->vecs.get((size_t)ld * nev * sizeof(double) + (size_t)nev * sizeof(double)));
    double* dE = Hpsi + (size_t)ld * nev;
    int rc = pf_apply(op, PF_F64, 0, psi, ld, Hpsi, ld, nev, stream);
    if (rc != PF_OK) throw Error{rc, pf_last_error()};
    coldots_host(h, psi, ld, Hpsi, ld, D, nev, nullptr, 0, E_host, st);
    PF_HIP(hipMemcpyAsync(dE, E_host, nev * sizeof(double), hipMemcpyHostToDevice, st));
    coldots_host(h, Hpsi, ld, psi, ld, D, nev, dE, 1, res_host, st);
    for (int i = 0; i < nev; ++i) res_host[i] = std::sqrt(res_host[i]);
  });
}
