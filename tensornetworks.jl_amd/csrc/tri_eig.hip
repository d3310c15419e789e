// Eigen-decomposition of a Hermitian matrix (sides: tri_eig.hpp) spread over the whole GPU:
// Householder reduction to a real symmetric tridiagonal matrix, divide and conquer with one
// launch per phase and level, back-transformation by blocked reflectors on the matrix cores. It
// replaces two solvers for the Gram matrices of splits: the one-workgroup reduction (whose p
// steps stream the matrix through one CU: 25 ms at p = 512) and, above 512 for matrices that are
// not mostly below its noise floor (svd.hip), the block Jacobi (17-20 sweeps over the matrix).
//
// Measured (graded Gram matrices, MI355X; before -> now, eigensolver only): real 160 1.9 ->
// 0.64 ms, 512 30 -> 2.5 ms, 602 22 -> 3.1 ms, 4096 470 -> 102 ms; complex 160 2.6 -> 0.86
// ms, 512 51 -> 3.7 ms. The kept vectors' error against 64-bit LAPACK falls with it (4096,
// weights down to 1e-3 of the largest: 2.6e-7 -> 2.8e-11), since a reduction that starts at
// the large end of a graded matrix keeps its small eigenvalues' relative accuracy.
//
// Reduction. While the active matrix is larger than one workgroup's registers, one launch per
// column (tri_col_kernel): every workgroup repeats the O(n) part of the step (the pending
// rank-2 update of the pivot column, its reflector), then updates its own columns and forms
// their entries of y = A v. The launch boundary is the only grid-wide synchronisation. The
// last tail_max columns run in one workgroup with the active matrix in registers
// (tri_tail_kernel), two barriers per column.
//
// Divide and conquer. Leaves of at most 32 are solved by dc_eig.hpp's tridiagonal solver, one
// workgroup each; a merge of two blocks takes five launches shared by all merges of a level
// (deflation; secular roots; recomputed coupling vector; eigenvectors; one batched matrix
// product on the matrix cores).
#include <algorithm>
#include <cmath>

#include "dc_eig.hpp"
#include "tnh_internal.hpp"
#include "tri_eig.hpp"
#include "tri_tail.hpp"

namespace tnh {
namespace {

// ------------------------------------------------------------------ preparation

// info[0] = exponent ex of max |G_ii| (0 for a zero or non-finite diagonal), info[1] = 1
// (the status, cleared by any later failure)
__global__ __launch_bounds__(1024) void tri_scale_kernel(const double *__restrict__ G, int p, int *__restrict__ info) {
  __shared__ double red[16];
  double m = 0.0;
  for (int i = threadIdx.x; i < p; i += 1024) m = fmax(m, fabs(G[i + int64_t(i) * p]));
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) m = fmax(m, red[w]);
    info[0] = (m > 0 && m < 1e300) ? ilogb(m) : 0;
    info[1] = 1;
  }
}

// G <- 2^-ex (G + G^H) / 2 by 32 x 32 tile pairs (one workgroup per tile of the upper triangle)
template <bool CPLX>
__global__ __launch_bounds__(256) void tri_sym_kernel(double *__restrict__ G, int p, int64_t imG,
                                                      const int *__restrict__ info) {
  const int bi = blockIdx.x, bj = blockIdx.y;
  if (bi > bj) return;
  __shared__ double a[CPLX ? 2 : 1][32][33], b[CPLX ? 2 : 1][32][33];
  const double sc = ldexp(0.5, -info[0]);
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t P = p;
  for (int c = ty; c < 32; c += 8) {
    const int i = 32 * bi + tx, j = 32 * bj + c;  // tile (bi, bj)
    const int i2 = 32 * bj + tx, j2 = 32 * bi + c;  // tile (bj, bi)
    const bool ok = i < p && j < p, ok2 = i2 < p && j2 < p;
    a[0][c][tx] = ok ? G[i + j * P] : 0.0;
    b[0][c][tx] = ok2 ? G[i2 + j2 * P] : 0.0;
    if (CPLX) {
      a[CPLX][c][tx] = ok ? G[imG + i + j * P] : 0.0;
      b[CPLX][c][tx] = ok2 ? G[imG + i2 + j2 * P] : 0.0;
    }
  }
  __syncthreads();
  for (int c = ty; c < 32; c += 8) {
    const int i = 32 * bi + tx, j = 32 * bj + c;
    const int i2 = 32 * bj + tx, j2 = 32 * bi + c;
    if (i < p && j < p) {
      G[i + j * P] = sc * (a[0][c][tx] + b[0][tx][c]);
      if (CPLX) G[imG + i + j * P] = i == j ? 0.0 : sc * (a[CPLX][c][tx] - b[CPLX][tx][c]);
    }
    if (bi != bj && i2 < p && j2 < p) {
      G[i2 + j2 * P] = sc * (b[0][c][tx] + a[0][tx][c]);
      if (CPLX) G[imG + i2 + j2 * P] = sc * (b[CPLX][c][tx] - a[CPLX][tx][c]);
    }
  }
}

// ------------------------------------------------------------------ reduction

// Column step j of the reduction over the whole grid. A holds the matrix with the updates of
// steps < j - 1 applied; v_{j-1} = V[:, j-1] and y_{j-1} = A v_{j-1} (yprev) define the pending
// one, A -= w v^H + v w^H with w = tau y - |tau|^2 (v^H y) / 2 v. Every workgroup forms the
// updated pivot column j and its reflector v_j in LDS (3 (p - j) values per plane), then takes
// columns c > j in turn, one wave each: it applies the pending update, stores the column and
// sums y_j[c] = sum_i conj(A[i, c]) v_j[i] (A is Hermitian). No workgroup writes column j,
// which all of them read. Per launch A's active part is read and written once.
template <bool CPLX, int NT>
__global__ __launch_bounds__(NT) void tri_col_kernel(double *__restrict__ A, int64_t imA, int p, int j,
                                                              const double *__restrict__ yprev,
                                                              double *__restrict__ ynew, double *__restrict__ V,
                                                              int64_t imV, double *__restrict__ dd,
                                                              double *__restrict__ ee, double *__restrict__ taus) {
  constexpr int NW = NT / 64, PL = CPLX ? 2 : 1;
  extern __shared__ double lds[];
  __shared__ double red[2][NW];
  const int n = p - j, t = threadIdx.x, lane = t & 63, wave = t >> 6;  // rows j .. p - 1
  double *vpr = lds, *vpi = lds + (PL - 1) * n, *wpr = lds + PL * n, *wpi = wpr + (PL - 1) * n;
  double *vnr = lds + 2 * PL * n, *vni = vnr + (PL - 1) * n;
  const int64_t P = p;
  auto block_sum = [&](double x, int slot) {
    x = wave_sum(x);
    if (lane == 0) red[slot][wave] = x;
    __syncthreads();
    double s = 0;
    for (int w = 0; w < NW; ++w) s += red[slot][w];
    return s;
  };
  const double *acr = A + j * P + j, *aci = CPLX ? A + imA + j * P + j : nullptr;  // A[j.., j]
  // The step is a chain of reductions between reads of data that other XCDs wrote in the
  // launch before, so everything whose address is known is loaded first: this thread's entries
  // of v_{j-1}, y_{j-1} and the pivot column, and the head of the wave's first own column.
  constexpr int PC = 4, PF = 8;
  const double *vpg = j > 0 ? V + (j - 1) * P + j : acr, *ypg = j > 0 ? yprev + j : acr;
  const double *vpgi = (CPLX && j > 0) ? V + imV + (j - 1) * P + j : aci;
  const double *ypgi = (CPLX && j > 0) ? yprev + p + j : aci;
  double pv[PC], py[PC], px[PC], pvi[CPLX ? PC : 1], pyi[CPLX ? PC : 1], pxi[CPLX ? PC : 1];
#pragma unroll
  for (int q = 0; q < PC; ++q) {
    const int i = min(t + q * NT, n - 1);
    pv[q] = vpg[i];
    py[q] = ypg[i];
    px[q] = acr[i];
    if (CPLX) {
      pvi[q] = vpgi[i];
      pyi[q] = ypgi[i];
      pxi[q] = aci[i];
    }
  }
  const int cl0 = 1 + blockIdx.x * NW + wave;
  double pc[PF], pci[CPLX ? PF : 1];
  {
    const int64_t o = j * P + j + min(cl0, n - 1) * P;
#pragma unroll
    for (int q = 0; q < PF; ++q) {
      const int i = min(1 + lane + 64 * q, n - 1);
      pc[q] = A[o + i];
      if (CPLX) pci[q] = A[imA + o + i];
    }
  }
  // f(i, v, vi, y, yi) over this thread's entries, the first PC from registers
  auto each = [&](const double *g0, const double *g0i, const double *g1, const double *g1i, const double *r0,
                  const double *r0i, const double *r1, const double *r1i, auto &&f) {
#pragma unroll
    for (int q = 0; q < PC; ++q)
      if (t + q * NT < n) f(t + q * NT, r0[q], CPLX ? r0i[q] : 0.0, r1[q], CPLX ? r1i[q] : 0.0);
    for (int i = t + PC * NT; i < n; i += NT)
      f(i, g0[i], CPLX ? g0i[i] : 0.0, g1[i], CPLX ? g1i[i] : 0.0);
  };
  if (j > 0) {
    double s = 0;
    each(vpg, vpgi, ypg, ypgi, pv, pvi, py, pyi, [&](int i, double a, double c, double b, double d) {
      vpr[i] = a;
      wpr[i] = b;
      s += a * b;
      if (CPLX) {
        vpi[i] = c;
        wpi[i] = d;
        s += c * d;
      }
    });
    const double vy = block_sum(s, 0);
    const double tr = taus[j - 1], ti = CPLX ? taus[p + j - 1] : 0.0;
    const double h = 0.5 * (tr * tr + ti * ti) * vy;
    for (int i = t; i < n; i += NT) {
      const double y = wpr[i], v = vpr[i];
      if (CPLX) {
        const double yc = wpi[i], vc = vpi[i];
        wpr[i] = tr * y - ti * yc - h * v;
        wpi[i] = tr * yc + ti * y - h * vc;
      } else {
        wpr[i] = tr * y - h * v;
      }
    }
    __syncthreads();
  }
  // pivot column with the pending update, and the norm of its tail
  double xs = 0;
  {
    double vjr = 0, vji = 0, wjr = 0, wji = 0;
    if (j > 0) {
      vjr = vpr[0];
      wjr = wpr[0];
      if (CPLX) {
        vji = vpi[0];
        wji = wpi[0];
      }
    }
    each(acr, aci, acr, aci, px, pxi, px, pxi, [&](int i, double xr, double xi, double, double) {
      if (j > 0) {
        if (CPLX) {
          xr -= wpr[i] * vjr + wpi[i] * vji + vpr[i] * wjr + vpi[i] * wji;
          xi -= wpi[i] * vjr - wpr[i] * vji + vpi[i] * wjr - vpr[i] * wji;
        } else {
          xr -= wpr[i] * vjr + vpr[i] * wjr;
        }
      }
      vnr[i] = xr;
      if (CPLX) vni[i] = xi;
      if (i >= 2) xs += xr * xr + xi * xi;
    });
  }
  const double xn2 = block_sum(xs, 1);  // its barrier also publishes vnr / vni
  const double dj = vnr[0];
  const Reflector R = reflector(vnr[1], CPLX ? vni[1] : 0.0, xn2);
  __syncthreads();  // entries 0 and 1 are read before they are rewritten
  for (int i = t; i < n; i += NT) {
    const double xr = vnr[i], xi = CPLX ? vni[i] : 0.0;
    double a = i == 1 ? 1.0 : 0.0, b = 0.0;
    if (i > 1) {
      a = xr * R.sr - xi * R.si;
      b = xr * R.si + xi * R.sr;
    }
    vnr[i] = a;
    if (CPLX) vni[i] = b;
    if (blockIdx.x == 0) {
      V[j * P + j + i] = a;
      if (CPLX) V[imV + j * P + j + i] = b;
    }
  }
  if (blockIdx.x == 0 && t == 0) {
    dd[j] = dj;
    ee[j] = R.beta;
    taus[j] = R.tr;
    taus[p + j] = R.ti;
  }
  __syncthreads();
  // own columns c = j + cl, cl >= 1
  for (int cl = cl0; cl < n; cl += gridDim.x * NW) {
    double *cr = A + (j + cl) * P + j, *ci = CPLX ? A + imA + (j + cl) * P + j : nullptr;
    double vcr = 0, vci = 0, wcr = 0, wci = 0;
    if (j > 0) {
      vcr = vpr[cl];
      wcr = wpr[cl];
      if (CPLX) {
        vci = vpi[cl];
        wci = wpi[cl];
      }
    }
    double sr = 0, si = 0;
    auto entry = [&](int i, double ar, double ai) {
      if (j > 0) {
        if (CPLX) {
          ar -= wpr[i] * vcr + wpi[i] * vci + vpr[i] * wcr + vpi[i] * wci;
          ai -= wpi[i] * vcr - wpr[i] * vci + vpi[i] * wcr - vpr[i] * wci;
          ci[i] = ai;
        } else {
          ar -= wpr[i] * vcr + vpr[i] * wcr;
        }
        cr[i] = ar;
      }
      sr += ar * vnr[i];
      if (CPLX) {
        sr += ai * vni[i];
        si += ar * vni[i] - ai * vnr[i];
      }
    };
    int i0 = 1 + lane;
    if (cl == cl0) {
#pragma unroll
      for (int q = 0; q < PF; ++q)
        if (i0 + 64 * q < n) entry(i0 + 64 * q, pc[q], CPLX ? pci[q] : 0.0);
      i0 += 64 * PF;
    }
#pragma unroll 8
    for (int i = i0; i < n; i += 64) entry(i, cr[i], CPLX ? ci[i] : 0.0);
    sr = wave_sum(sr);
    if (CPLX) si = wave_sum(si);
    if (lane == 0) {
      ynew[j + cl] = sr;
      if (CPLX) ynew[p + j + cl] = si;
    }
  }
}

template <bool CPLX, int NT, int RA, int RB>
__global__ __launch_bounds__(NT) void tri_tail_kernel(const double *__restrict__ Am, int64_t imA, int p, int k0,
                                                      const double *__restrict__ yprev, double *__restrict__ V,
                                                      int64_t imV, double *__restrict__ dd, double *__restrict__ ee,
                                                      double *__restrict__ taus) {
  constexpr int TI = NT / 16, N = 16 * RB;
  static_assert(TI * RA == N, "square register tile");
  static_assert(N <= NT, "one reflector entry per thread");
  __shared__ TailShared<CPLX, NT, RA, RB> sh;
  TailRegs<CPLX, NT, RA, RB> A;
  const int t = threadIdx.x, lane = t & 63, ti = t >> 4, tj = t & 15, m = p - k0;
  const int64_t P = p;
#pragma unroll
  for (int a = 0; a < RA; ++a)
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int i = ti + TI * a, j = tj + 16 * b;
      const bool ok = i < m && j < m;
      A.r[a][b] = ok ? Am[(k0 + i) + (k0 + j) * P] : 0.0;
      if (CPLX) A.i[a][b] = ok ? Am[imA + (k0 + i) + (k0 + j) * P] : 0.0;
    }
  if (k0 > 0) {  // the update pending from column k0 - 1
    if (t < N) {
      const bool ok = t < m;
      const double a = ok ? V[(k0 - 1) * P + k0 + t] : 0.0, b = ok ? yprev[k0 + t] : 0.0;
      sh.xr[0][t] = a;
      sh.yr[t] = b;
      if (CPLX) {
        sh.xi[0][t] = ok ? V[imV + (k0 - 1) * P + k0 + t] : 0.0;
        sh.yi[t] = ok ? yprev[p + k0 + t] : 0.0;
      }
    }
    __syncthreads();
    double s = 0;
    for (int i = lane; i < m; i += 64) {
      s += sh.xr[0][i] * sh.yr[i];
      if (CPLX) s += sh.xi[0][i] * sh.yi[i];
    }
    const double tr = taus[k0 - 1], tq = CPLX ? taus[p + k0 - 1] : 0.0;
    const double h = 0.5 * (tr * tr + tq * tq) * wave_sum(s);
    double vjr[RB], vji[CPLX ? RB : 1], wjr[RB], wji[CPLX ? RB : 1];
    auto vw = [&](int i, double &vr, double &vi, double &wr, double &wi) {
      vr = sh.xr[0][i];
      const double y = sh.yr[i];
      if (CPLX) {
        vi = sh.xi[0][i];
        const double z = sh.yi[i];
        wr = tr * y - tq * z - h * vr;
        wi = tr * z + tq * y - h * vi;
      } else {
        wr = tr * y - h * vr;
      }
    };
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      double v2 = 0, w2 = 0;
      vw(tj + 16 * b, vjr[b], v2, wjr[b], w2);
      if (CPLX) {
        vji[b] = v2;
        wji[b] = w2;
      }
    }
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      double vr, vi = 0, wr, wi = 0;
      vw(ti + TI * a, vr, vi, wr, wi);
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        if (CPLX) {
          A.r[a][b] -= wr * vjr[b] + wi * vji[b] + vr * wjr[b] + vi * wji[b];
          A.i[a][b] -= wi * vjr[b] - wr * vji[b] + vi * wjr[b] - vr * wji[b];
        } else {
          A.r[a][b] -= wr * vjr[b] + vr * wjr[b];
        }
      }
    }
    __syncthreads();
  }
  if (tj == 0) {
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      sh.xr[0][ti + TI * a] = A.r[a][0];
      if (CPLX) sh.xi[0][ti + TI * a] = A.i[a][0];
    }
  }
  __syncthreads();
  tail_steps<CPLX, NT, RA, RB, 0>(sh, A, p, k0, m, V, imV, dd, ee, taus);
  if (t == 0) {
    dd[p - 1] = sh.xr[(m - 1) & 1][m - 1];
    ee[p - 1] = 0.0;
    taus[p - 1] = 0.0;
    taus[2 * p - 1] = 0.0;
  }
}

// Column steps above these sides use one 1024-thread workgroup per CU (the three vectors leave
// LDS for one), below two of 256: measured, whole solve, wide against narrow throughout: real
// 768 5.63 / 5.65 ms, 1500 15.5 / 16.6, 4096 106 / 159; complex 1500 21.6 / 19.8, 2048 36.6 / 38.7.
constexpr int kColWide = 768, kColWideCplx = 1800;

// the widest active matrix of one workgroup
constexpr int tail_max(bool cplx) { return cplx ? 128 : 192; }

template <bool CPLX, int NT, int RA, int RB>
void run_tail(hipStream_t st, const double *A, int64_t im, int p, int k0, const double *y, double *V, double *dd,
              double *ee, double *taus) {
  hipLaunchKernelGGL((tri_tail_kernel<CPLX, NT, RA, RB>), dim3(1), dim3(NT), 0, st, A, im, p, k0, y, V, im, dd, ee,
                     taus);
}

template <bool CPLX>
void launch_tail(hipStream_t st, const double *A, int64_t im, int p, int k0, const double *y, double *V, double *dd,
                 double *ee, double *taus) {
  const int m = p - k0;
  if constexpr (CPLX) {
    if (m <= 32) return run_tail<true, 256, 2, 2>(st, A, im, p, k0, y, V, dd, ee, taus);
    if (m <= 64) return run_tail<true, 256, 4, 4>(st, A, im, p, k0, y, V, dd, ee, taus);
    if (m <= 96) return run_tail<true, 256, 6, 6>(st, A, im, p, k0, y, V, dd, ee, taus);
  } else {
    static_assert(kTriMinReal > 96, "smaller real tails are not instantiated");
    if (m > 160) return run_tail<false, 512, 6, 12>(st, A, im, p, k0, y, V, dd, ee, taus);
    if (m > 128) return run_tail<false, 512, 5, 10>(st, A, im, p, k0, y, V, dd, ee, taus);
  }
  run_tail<CPLX, 512, 4, 8>(st, A, im, p, k0, y, V, dd, ee, taus);
}

// ------------------------------------------------------------------ divide and conquer

// Work arrays of the divide and conquer over Pp = leaf * 2^levels >= p positions; the positions
// past p are decoupled from T (zero off-diagonals) and hold a bound on its spectrum, so they
// sort last. Per merge of n positions starting at b the arrays hold its entries at [b, b + n).
struct DcWork {
  int p, Pp, leaf;
  double *d, *e;  // T with its off-diagonals torn between the leaves, and the untorn e
  double *lam[2];  // eigenvalues of the blocks, ascending, before and after a level
  double *Ds, *dk, *zk, *zh, *tau, *rc, *rs, *rho;
  int *src, *kpos, *dpos, *org, *finv, *rj, *ri, *mK, *mrot;
  int *info;  // [0] exponent of the scaling, [1] status
};

constexpr int kLeafMax = 32, kLeafThreads = 256;

struct Leaves {
  int leaf, levels, Pp;
};
Leaves leaves_of(int p) {
  Leaves g{p, 0, p};
  while (g.leaf > kLeafMax) {
    ++g.levels;
    g.leaf = (p + (1 << g.levels) - 1) >> g.levels;
  }
  // Up to side 512 the blocks are 32, 64, ... wide from position 0, as the one-workgroup solver's
  // are: where T is torn decides which small couplings deflate, and equal leaves lose accuracy on
  // graded matrices (a gate's tensors against 64-bit LAPACK, blocks of 32 / equal leaves, geometric
  // mean of 14 seeds: bond 70 3.3e-11 / 1.7e-10, 80 3.3e-11 / 1.2e-10, 150 8.4e-11 / 2.7e-10, 200
  // 8.8e-11 / 2.3e-10) for 0 - 5% of time (complex side 257 1.52 / 1.47 ms, 160 0.86 / 0.84, 224 1.24 /
  // 1.25). Above, equal leaves keep the padding under one per leaf; the block Jacobi that had these
  // sides was further off (bond 300: 1.7e-7, 4.0e-10 here).
  if (g.levels > 0 && p <= dc::kDcPMax) g.leaf = kLeafMax;
  g.Pp = g.leaf << g.levels;
  return g;
}

// Tears T between the leaves (d_i -= |e| on both sides), fills the padding, clears the status
// when T is not finite.
__global__ __launch_bounds__(1024) void tri_tear_kernel(DcWork w, const double *__restrict__ dd,
                                                        const double *__restrict__ ee) {
  __shared__ double red[16];
  __shared__ int bad;
  const int t = threadIdx.x;
  if (t == 0) bad = 0;
  __syncthreads();
  double m = 0;
  for (int i = t; i < w.p; i += 1024) {
    const double a = dd[i], b = i + 1 < w.p ? ee[i] : 0.0;
    if (!dc::finite(a) || !dc::finite(b)) bad = 1;
    m = fmax(m, fabs(a) + 2.0 * fabs(b));
  }
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  if ((t & 63) == 0) red[t >> 6] = m;
  __syncthreads();
  for (int q = 0; q < 16; ++q) m = fmax(m, red[q]);
  if (bad && t == 0) w.info[1] = 0;
  const double pad = 2.0 * m + 1.0;  // |T| <= max |d| + 2 max |e| <= 2 m
  for (int i = t; i < w.Pp; i += 1024) {
    double v = pad;
    const double e0 = (i > 0 && i < w.p) ? fabs(ee[i - 1]) : 0.0, e1 = i + 1 < w.p ? ee[i] : 0.0;
    if (i < w.p) {
      v = dd[i];
      if (i % w.leaf == 0) v -= e0;
      if ((i + 1) % w.leaf == 0) v -= fabs(e1);
    }
    w.d[i] = v;
    w.e[i] = e1;
  }
}

// Whether an earlier launch failed, the same answer for every thread of the workgroup. Other
// workgroups of this launch may clear the status at any time: if each wave read it for itself,
// some could leave and the others go on past the barriers with LDS entries nobody wrote, which
// index memory below. (The kernels without barriers let each thread read it.)
__device__ __forceinline__ bool failed(const DcWork &w) {
  __shared__ int status;
  if (threadIdx.x == 0) status = w.info[1];
  __syncthreads();
  return status == 0;
}

// One leaf per workgroup, by dc_eig.hpp's tridiagonal solver, which sees its positions of T only:
// with the padding among them, its deflation threshold would follow that bound on all of T instead
// of the leaf's own entries, and the small end of a graded matrix, which is where the padding
// sits, would lose its relative accuracy (a gate's tensors at bond 70, side 140: 2.9e-9 from 64-bit
// LAPACK with it, 3.4e-11 without).
__global__ __launch_bounds__(kLeafThreads) void tri_leaf_kernel(DcWork w, double *__restrict__ Q,
                                                                double *__restrict__ Q2, double *__restrict__ U) {
  __shared__ dc::DcShared sh;
  if (failed(w)) return;
  const int b = blockIdx.x * w.leaf, s = w.leaf, t = threadIdx.x, r = max(0, min(s, w.p - b));
  const int64_t P = w.Pp, o = b * (P + 1);
  for (int e = t; e < s * s; e += kLeafThreads) {
    const int i = e % s, c = e / s;
    if (i >= r || c >= r) Q[o + i + c * P] = i == c ? 1.0 : 0.0;
  }
  for (int i = r + t; i < s; i += kLeafThreads) w.lam[0][b + i] = w.d[b + i];
  for (int i = t; i < r; i += kLeafThreads) {
    sh.d[i] = w.d[b + i];
    sh.e[i] = i + 1 < r ? w.e[b + i] : 0.0;
  }
  if (t == 0) sh.status = 1;
  __syncthreads();
  if (r <= 1) {
    if (t == 0 && r == 1) {
      Q[o] = 1.0;
      w.lam[0][b] = sh.d[0];
    }
    return;
  }
  dc::dc_tridiag(dc::DcDeviceEx<kLeafThreads>{}, sh, r, P, Q + o, Q2 + o, U + o);
  __syncthreads();
  for (int i = t; i < r; i += kLeafThreads) w.lam[0][b + i] = sh.u.c.lam[i];
  if (t == 0 && sh.status == 0) w.info[1] = 0;
}

// Deflation of one merge per workgroup (n positions, halves of n / 2): the halves' eigenvalues
// merged by rank, the coupling vector z, and the scan that removes entries with a negligible
// coupling and rotates away one of two close poles (thresholds relative to the largest
// entry that is not padding). The scan is serial; it reads LDS with the
// next entry already loaded and needs neither division nor square root for an entry it keeps.
__global__ __launch_bounds__(1024) void tri_deflate_kernel(DcWork w, int n, int cur, const double *__restrict__ Q) {
  extern __shared__ double lds[];
  double *Ds = lds, *zs = lds + n;
  unsigned char *keep = reinterpret_cast<unsigned char *>(zs + n);
  __shared__ double red[2][16];
  __shared__ int cnt[1024];
  __shared__ int bad, nrot;
  if (failed(w)) return;
  const int m = blockIdx.x, b = m * n, s = n / 2, t = threadIdx.x;
  const int64_t P = w.Pp;
  const double *lam = w.lam[cur] + b;
  if (t == 0) bad = 0;
  __syncthreads();
  const double e = w.e[b + s - 1], sg = e >= 0 ? 1.0 : -1.0;
  for (int j = t; j < n; j += 1024) {
    const double D = lam[j], z = j < s ? Q[(b + s - 1) + (b + j) * P] : sg * Q[(b + s) + (b + j) * P];
    const double key = dc::order_key(D);
    if (!dc::finite(D) || !dc::finite(z)) bad = 1;
    // entries of the other half below D (the left half first among equals)
    int lo = j < s ? s : 0, hi = j < s ? n : s;
    const int base = lo;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const double o = dc::order_key(lam[mid]);
      if (j < s ? o < key : o <= key)
        lo = mid + 1;
      else
        hi = mid;
    }
    const int rank = (j < s ? j : j - s) + (lo - base);
    Ds[rank] = D;
    zs[rank] = z;
    w.src[b + rank] = j;
  }
  __syncthreads();
  if (bad) {
    if (t == 0) w.info[1] = 0;
    return;
  }
  double zn2 = 0, dmax = 0;
  for (int i = t; i < n; i += 1024) {
    const double z = zs[i];
    zn2 += z * z;
    if (b + w.src[b + i] < w.p) dmax = fmax(dmax, fabs(Ds[i]));
  }
  zn2 = wave_sum(zn2);
  for (int o = 32; o > 0; o >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, o, 64));
  if ((t & 63) == 0) {
    red[0][t >> 6] = zn2;
    red[1][t >> 6] = dmax;
  }
  __syncthreads();
  zn2 = dmax = 0;
  for (int q = 0; q < 16; ++q) {
    zn2 += red[0][q];
    dmax = fmax(dmax, red[1][q]);
  }
  const bool coupled = zn2 > 0 && e != 0.0;
  const double rho = coupled ? fabs(e) * zn2 : 0.0;
  const double tol = 8.0 * dc::kEps * fmax(dmax, rho);
  if (coupled) {
    const double zn = sqrt(zn2);
    for (int i = t; i < n; i += 1024) {
      const double z = zs[i] / zn;
      zs[i] = z;
      keep[i] = rho * fabs(z) > tol;
    }
  } else {
    for (int i = t; i < n; i += 1024) keep[i] = 0;
  }
  __syncthreads();
  if (t == 0) {
    int nr = 0;
    if (coupled) {
      int last = -1;
      double zj = 0, Dj = 0, z = zs[0], D = Ds[0];
      unsigned char kf = keep[0];
      for (int i = 0; i < n; ++i) {
        const int nx = i + 1 < n ? i + 1 : i;
        const double z1 = zs[nx], D1 = Ds[nx];
        const unsigned char k1 = keep[nx];
        if (kf) {
          const double r2 = zj * zj + z * z;
          if (last >= 0 && fabs((D - Dj) * zj * z) <= tol * r2) {  // |D_i - D_j| cs sn <= tol
            const double r = sqrt(r2), cs = z / r, sn = zj / r;
            Ds[last] = Dj * cs * cs + D * sn * sn;
            keep[last] = 0;
            w.rj[b + nr] = last;
            w.ri[b + nr] = i;
            w.rc[b + nr] = cs;
            w.rs[b + nr] = sn;
            ++nr;
            D = Dj * sn * sn + D * cs * cs;
            z = r;
            Ds[i] = D;
            zs[i] = z;
          }
          last = i;
          zj = z;
          Dj = D;
        }
        z = z1;
        D = D1;
        kf = k1;
      }
    }
    nrot = nr;
  }
  __syncthreads();
  // kept and deflated positions, each in ascending order: a contiguous chunk per thread
  const int ch = (n + 1023) / 1024, i0 = min(n, t * ch), i1 = min(n, i0 + ch);
  int mine = 0;
  for (int i = i0; i < i1; ++i) mine += keep[i];
  cnt[t] = mine;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int v = t >= o ? cnt[t - o] : 0;
    __syncthreads();
    cnt[t] += v;
    __syncthreads();
  }
  int kp = cnt[t] - mine, dp = i0 - kp;
  for (int i = i0; i < i1; ++i) {
    if (keep[i]) {
      w.kpos[b + kp] = i;
      w.dk[b + kp] = Ds[i];
      w.zk[b + kp] = zs[i];
      ++kp;
    } else {
      w.dpos[b + dp++] = i;
    }
    w.Ds[b + i] = Ds[i];
  }
  if (t == 0) {
    w.mK[m] = cnt[1023];
    w.mrot[m] = nrot;
    w.rho[m] = rho;
  }
}

// Blocks [0, nroot): a wave per secular root. The others: 64 x 64 tiles of the merges'
// eigenvectors in sorted order, Q2[:, x] = Q[:, src[x]] (zero off the child's rows).
__global__ __launch_bounds__(256) void tri_root_kernel(DcWork w, int n, int nroot, const double *__restrict__ Q,
                                                       double *__restrict__ Q2) {
  if (w.info[1] == 0) return;
  const int t = threadIdx.x, lane = t & 63;
  const int64_t P = w.Pp;
  if (int(blockIdx.x) < nroot) {
    const int a = blockIdx.x * 4 + (t >> 6);
    if (a >= w.Pp) return;
    const int m = a / n, b = m * n, j = a - b, K = w.mK[m];
    if (j >= K) return;
    int o = 0, its = 0;
    const dc::DcDeviceEx<256> ex{};
    const double tt = dc::secular_root(ex, w.dk + b, w.zk + b, w.rho[m], j, K, lane, 64, &o, &its);
    if (lane == 0) {
      w.org[a] = o;
      w.tau[a] = tt;
      if (!dc::finite(tt) || its >= 96) w.info[1] = 0;
    }
    return;
  }
  const int tn = (n + 63) / 64, s = n / 2;
  int id = blockIdx.x - nroot;
  const int m = id / (tn * tn), b = m * n;
  id %= tn * tn;
  const int r = 64 * (id % tn) + lane, c0 = 64 * (id / tn) + (t >> 6);
  if (r >= n) return;
  for (int c = c0; c < min(n, 64 * (id / tn) + 64); c += 4) {
    const int q = w.src[b + c];
    Q2[(b + r) + (b + c) * P] = ((r < s) == (q < s)) ? Q[(b + r) + (b + q) * P] : 0.0;
  }
}

// Blocks [0, nitem): a wave per item x of a merge (roots x < K, then the deflated entries):
// the Gu-Eisenstat coupling component of a root, and the item's final rank. The others: the
// deflation rotations on 64 rows of Q2 each, in order (a chain's running column in a register).
__global__ __launch_bounds__(256) void tri_couple_kernel(DcWork w, int n, int nitem, int cur,
                                                         double *__restrict__ Q2) {
  if (w.info[1] == 0) return;
  const int t = threadIdx.x, lane = t & 63;
  const int64_t P = w.Pp;
  if (int(blockIdx.x) < nitem) {
    const int a = blockIdx.x * 4 + (t >> 6);
    if (a >= w.Pp) return;
    const int m = a / n, b = m * n, x = a - b, K = w.mK[m];
    const double *dk = w.dk + b, *tau = w.tau + b;
    const int *org = w.org + b;
    if (x < K) {
      const double di = dk[x];
      double prod = lane == 0 ? (dk[org[x]] - di) + tau[x] : 1.0;
      for (int k = lane; k < K; k += 64)
        if (k != x) prod *= ((dk[org[k]] - di) + tau[k]) / (dk[k] - di);
      for (int o = 32; o > 0; o >>= 1) prod *= __shfl_xor(prod, o, 64);
      if (lane == 0) w.zh[a] = copysign(sqrt(fabs(prod) / w.rho[m]), w.zk[a]);
    }
    auto val = [&](int y) { return y < K ? dk[org[y]] + tau[y] : w.Ds[b + w.dpos[b + y - K]]; };
    const double vx = val(x), kx = dc::order_key(vx);
    int rank = 0;
    for (int y = lane; y < n; y += 64) {
      const double ky = dc::order_key(val(y));
      rank += (ky < kx) || (ky == kx && y < x);
    }
    for (int o = 32; o > 0; o >>= 1) rank += __shfl_xor(rank, o, 64);
    if (lane == 0) {
      w.finv[a] = rank;
      w.lam[cur ^ 1][b + rank] = vx;
    }
    return;
  }
  const int r = (blockIdx.x - nitem) * 256 + t;
  if (r >= w.Pp) return;
  const int m = r / n, b = m * n, nr = w.mrot[m];
  double run = 0.0;
  int held = -1;  // column whose current value is `run`
  for (int q = 0; q < nr; ++q) {
    const int cj = w.rj[b + q], ci = w.ri[b + q];
    const double cs = w.rc[b + q], sn = w.rs[b + q];
    if (held != cj) {
      if (held >= 0) Q2[r + (b + held) * P] = run;
      run = Q2[r + (b + cj) * P];
    }
    const double y = Q2[r + (b + ci) * P];
    Q2[r + (b + cj) * P] = cs * run - sn * y;
    run = sn * run + cs * y;
    held = ci;
  }
  if (held >= 0) Q2[r + (b + held) * P] = run;
}

// One column of a merge's U per workgroup: the secular eigenvector of a root, scattered to the
// sorted positions of the kept entries, or a unit vector for a deflated entry; columns in
// final order, so that the product Q2 U is the merged block's eigenvector matrix.
__global__ __launch_bounds__(256) void tri_vec_kernel(DcWork w, int n, double *__restrict__ U) {
  extern __shared__ double u[];
  __shared__ double red[4];
  if (failed(w)) return;
  const int a = blockIdx.x, m = a / n, b = m * n, x = a - b, K = w.mK[m], t = threadIdx.x;
  const int64_t P = w.Pp;
  for (int i = t; i < n; i += 256) u[i] = 0.0;
  __syncthreads();
  double f = 1.0;
  if (x < K) {
    const double *dk = w.dk + b;
    const double lo = dk[w.org[a]], tk = w.tau[a];
    double nn = 0;
    for (int i = t; i < K; i += 256) {
      const double v = w.zh[b + i] / ((dk[i] - lo) - tk);
      u[w.kpos[b + i]] = v;
      nn += v * v;
    }
    nn = wave_sum(nn);
    if ((t & 63) == 0) red[t >> 6] = nn;
    __syncthreads();
    nn = (red[0] + red[1]) + (red[2] + red[3]);
    if (!(nn > 0.0) || !dc::finite(nn)) {
      if (t == 0) w.info[1] = 0;
      return;
    }
    f = 1.0 / sqrt(nn);
  } else if (t == 0) {
    u[w.dpos[b + x - K]] = 1.0;
  }
  __syncthreads();
  double *out = U + b + (b + w.finv[a]) * P;
  for (int i = t; i < n; i += 256) out[i] = f * u[i];
}

__global__ __launch_bounds__(256) void tri_out_kernel(DcWork w, int cur, double *__restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i > w.p) return;
  const bool ok = w.info[1] != 0;
  if (i == w.p)
    out[i] = ok ? 1.0 : 0.0;
  else
    out[i] = ok ? ldexp(w.lam[cur][i], w.info[0]) : NAN;
}

// ------------------------------------------------------------------ back-transformation

// basis[:, c] = column perm[c] of the tridiagonal eigenvectors
__global__ __launch_bounds__(256) void tri_gather_kernel(const double *__restrict__ Z, int64_t ldz,
                                                         const int *__restrict__ perm, int p, int64_t tot, bool cplx,
                                                         double *__restrict__ basis) {
  const int64_t e = blockIdx.x * int64_t(256) + threadIdx.x;
  if (e >= tot) return;
  basis[e] = Z[e % p + int64_t(perm[e / p]) * ldz];
  if (cplx) basis[tot + e] = 0.0;
}

// basis <- H_0 H_1 ... H_{p-2} basis, H_k = I - tau_k v_k v_k^H: one wave per column, whose
// rows stay in registers (R per lane); the next reflector is loaded while the current one is
// applied, its dot product is a DPP wave sum. The reflectors' L2 reads are the only traffic.
template <bool CPLX, int R>
__global__ __launch_bounds__(256) void tri_back_kernel(const double *__restrict__ V, int p, int64_t imV,
                                                       const double *__restrict__ taus, double *__restrict__ X,
                                                       int64_t imX, int k) {
  const int lane = threadIdx.x & 63, c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= k) return;
  const int64_t P = p;
  double xr[R], xi[CPLX ? R : 1], nr[R], ni[CPLX ? R : 1];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = lane + 64 * r;
    xr[r] = i < p ? X[i + c * P] : 0.0;
    if (CPLX) xi[r] = 0.0;
  }
  auto load = [&](int q, double &tr, double &ti) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = lane + 64 * r;
      const bool on = i > q && i < p;  // v_q's support
      nr[r] = on ? V[i + q * P] : 0.0;
      if (CPLX) ni[r] = on ? V[imV + i + q * P] : 0.0;
    }
    tr = taus[q];
    ti = CPLX ? taus[p + q] : 0.0;
  };
  double tnr = 0, tni = 0;
  if (p >= 2) load(p - 2, tnr, tni);
  for (int q = p - 2; q >= 0; --q) {
    double vr[R], vi[CPLX ? R : 1];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      vr[r] = nr[r];
      if (CPLX) vi[r] = ni[r];
    }
    const double tr = tnr, ti = tni;
    if (q > 0) load(q - 1, tnr, tni);
    double sr = 0, si = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      sr += vr[r] * xr[r];
      if (CPLX) {
        sr += vi[r] * xi[r];
        si += vr[r] * xi[r] - vi[r] * xr[r];
      }
    }
    sr = wave_sum(sr);
    if (CPLX) si = wave_sum(si);
    const double fr = tr * sr - ti * si, fi = tr * si + ti * sr;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (CPLX) {
        xr[r] -= vr[r] * fr - vi[r] * fi;
        xi[r] -= vr[r] * fi + vi[r] * fr;
      } else {
        xr[r] -= vr[r] * fr;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = lane + 64 * r;
    if (i < p) {
      X[i + c * P] = xr[r];
      if (CPLX) X[imX + i + c * P] = xi[r];
    }
  }
}

// T factor of one panel of nb reflectors per workgroup (H_0 ... H_{nb-1} = I - V T V^H), from
// S = V^H V: T[0:j, j] = -tau_j T[0:j, 0:j] S[0:j, j], T[j, j] = tau_j. T in LDS, then to memory.
template <bool CPLX>
__global__ __launch_bounds__(256) void tri_tfac_kernel(const double *__restrict__ S, int nb, int64_t imS, int p,
                                                       const double *__restrict__ taus, double *__restrict__ T) {
  extern __shared__ double tl[];
  __shared__ double col[CPLX ? 2 : 1][128];
  const int pan = blockIdx.x, t = threadIdx.x, n2 = nb * nb;
  double *Tr = tl, *Ti = tl + n2;
  const double *Sr = S + int64_t(pan) * n2, *Si = S + imS + int64_t(pan) * n2;
  for (int e = t; e < n2; e += 256) {
    Tr[e] = 0.0;
    if (CPLX) Ti[e] = 0.0;
  }
  __syncthreads();
  for (int j = 0; j < nb; ++j) {
    const int g = pan * nb + j;
    const double tr = g < p ? taus[g] : 0.0, ti = (CPLX && g < p) ? taus[p + g] : 0.0;
    if (t < j) {
      col[0][t] = Sr[t + j * nb];
      if (CPLX) col[CPLX][t] = Si[t + j * nb];
    }
    __syncthreads();
    if (t < j) {
      double ar = 0, ai = 0;
      for (int l = t; l < j; ++l) {
        const double xr = Tr[t + l * nb], yr = col[0][l];
        ar += xr * yr;
        if (CPLX) {
          const double xi = Ti[t + l * nb], yi = col[CPLX][l];
          ar -= xi * yi;
          ai += xr * yi + xi * yr;
        }
      }
      Tr[t + j * nb] = -(tr * ar - ti * ai);
      if (CPLX) Ti[t + j * nb] = -(tr * ai + ti * ar);
    } else if (t == j) {
      Tr[j + j * nb] = tr;
      if (CPLX) Ti[j + j * nb] = ti;
    }
    __syncthreads();
  }
  for (int e = t; e < n2; e += 256) {
    T[int64_t(pan) * n2 + e] = Tr[e];
    if (CPLX) T[imS + int64_t(pan) * n2 + e] = Ti[e];
  }
}

template <bool CPLX>
void launch_back(tnh_ctx *ctx, const double *V, int p, const double *taus, double *X, int k) {
  const dim3 grid(unsigned((k + 3) / 4)), block(256);
  const int64_t im = int64_t(p) * p, imX = int64_t(p) * k;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, block, 0, ctx->stream, V, p, im, taus, X, imX, k); };
  if constexpr (CPLX)
    if (p <= 64) return go(tri_back_kernel<true, 1>);
  if (p <= 128)
    go(tri_back_kernel<CPLX, 2>);
  else if (p <= 192)
    go(tri_back_kernel<CPLX, 3>);
  else if (p <= 256)
    go(tri_back_kernel<CPLX, 4>);
  else if (p <= 512)
    go(tri_back_kernel<CPLX, 8>);
  else
    go(tri_back_kernel<CPLX, 16>);
}

// Above this side the reflectors are applied in panels on the matrix cores.
constexpr int kBackWaveMax = 1024;

int panel_width(bool cplx) { return cplx ? 64 : 128; }
int panel_count(int p, bool cplx) { return (p + panel_width(cplx) - 1) / panel_width(cplx); }

template <bool CPLX>
void reduce_matrix(tnh_ctx *ctx, double *G, int p, double *V, double *y, double *dd, double *ee, double *taus,
                   int *info) {
  const int64_t im = int64_t(p) * p;
  constexpr int PL = CPLX ? 2 : 1;
  hipLaunchKernelGGL(tri_scale_kernel, dim3(1), dim3(1024), 0, ctx->stream, G, p, info);
  const unsigned tb = unsigned((p + 31) / 32);
  hipLaunchKernelGGL(tri_sym_kernel<CPLX>, dim3(tb, tb), dim3(256), 0, ctx->stream, G, p, im, info);
  const int J = std::max(0, p - tail_max(CPLX));
  double *yb[2] = {y, y + PL * int64_t(p)};
  for (int j = 0; j < J; ++j) {
    const int n = p - j;
    auto step = [&](auto kern, int nt, int wgs) {
      const int waves = nt / 64;
      const unsigned grid = unsigned(std::min((n - 1 + waves - 1) / waves, wgs));
      hipLaunchKernelGGL(kern, dim3(grid), dim3(nt), sizeof(double) * 3 * PL * n, ctx->stream, G, im, p, j,
                         yb[(j + 1) & 1], yb[j & 1], V, im, dd, ee, taus);
    };
    if (n > (CPLX ? kColWideCplx : kColWide))
      step(tri_col_kernel<CPLX, 1024>, 1024, ctx->cu_count);
    else
      step(tri_col_kernel<CPLX, 256>, 256, 2 * ctx->cu_count);
  }
  launch_tail<CPLX>(ctx->stream, G, im, p, J, yb[(J + 1) & 1], V, dd, ee, taus);
  TNH_HIP(hipGetLastError());
}

// Carves an array out of a workspace.
template <class T>
T *carve(char *&at, int64_t n) {
  T *r = reinterpret_cast<T *>(at);
  at += (sizeof(T) * size_t(n) + 255) / 256 * 256;
  return r;
}

}  // namespace

void tri_eig_solve(tnh_ctx *ctx, double *G, int p, bool cplx, double *dout) {
  TNH_REQUIRE(p >= (cplx ? kTriMinCplx : kTriMinReal) && p <= (cplx ? kTriMaxCplx : kTriMaxReal), TNH_ERR_ARG,
              "tri_eig: side out of range");
  const int64_t pp = int64_t(p) * p;
  const int PL = cplx ? 2 : 1;
  const Leaves lv = leaves_of(p);
  const int leaf = lv.leaf, levels = lv.levels, Pp = lv.Pp;
  const int64_t qq = int64_t(Pp) * Pp;
  double *V = static_cast<double *>(ctx->workspace(640, sizeof(double) * pp * PL));
  double *Q = static_cast<double *>(ctx->workspace(641, sizeof(double) * qq));
  double *Q2 = static_cast<double *>(ctx->workspace(642, sizeof(double) * qq));
  double *U = static_cast<double *>(ctx->workspace(643, sizeof(double) * qq));
  char *at = static_cast<char *>(ctx->workspace(644, size_t(40) * 8 * (Pp + 64)));
  double *y = carve<double>(at, 2 * PL * int64_t(p));
  double *dd = carve<double>(at, p), *ee = carve<double>(at, p), *taus = carve<double>(at, 2 * int64_t(p));
  DcWork w;
  w.p = p;
  w.Pp = Pp;
  w.leaf = leaf;
  for (double **a : {&w.d, &w.e, &w.lam[0], &w.lam[1], &w.Ds, &w.dk, &w.zk, &w.zh, &w.tau, &w.rc, &w.rs, &w.rho})
    *a = carve<double>(at, Pp);
  for (int **a : {&w.src, &w.kpos, &w.dpos, &w.org, &w.finv, &w.rj, &w.ri, &w.mK, &w.mrot}) *a = carve<int>(at, Pp);
  w.info = carve<int>(at, 2);
  if (p > kBackWaveMax) fill(ctx, V, TNH_F64, pp * PL, 0.0);  // panels also read above the reflectors
  if (cplx)
    reduce_matrix<true>(ctx, G, p, V, y, dd, ee, taus, w.info);
  else
    reduce_matrix<false>(ctx, G, p, V, y, dd, ee, taus, w.info);
  // taus sits at a fixed place for tri_eig_vectors
  copy_device(ctx, ctx->workspace(645, sizeof(double) * 2 * p), taus, sizeof(double) * 2 * p);
  hipStream_t st = ctx->stream;
  hipLaunchKernelGGL(tri_tear_kernel, dim3(1), dim3(1024), 0, st, w, dd, ee);
  hipLaunchKernelGGL(tri_leaf_kernel, dim3(unsigned(Pp / leaf)), dim3(kLeafThreads), 0, st, w, Q, Q2, U);
  int cur = 0;
  for (int l = 1; l <= levels; ++l) {
    const int n = leaf << l, nm = Pp / n;
    const int tn = (n + 63) / 64, nw = (Pp + 3) / 4;
    hipLaunchKernelGGL(tri_deflate_kernel, dim3(unsigned(nm)), dim3(1024), size_t(n) * 17 + 16, st, w, n, cur, Q);
    hipLaunchKernelGGL(tri_root_kernel, dim3(unsigned(nw + nm * tn * tn)), dim3(256), 0, st, w, n, nw, Q, Q2);
    hipLaunchKernelGGL(tri_couple_kernel, dim3(unsigned(nw + (Pp + 255) / 256)), dim3(256), 0, st, w, n, nw, cur,
                       Q2);
    hipLaunchKernelGGL(tri_vec_kernel, dim3(unsigned(Pp)), dim3(256), sizeof(double) * n, st, w, n, U);
    TNH_HIP(hipGetLastError());
    Gemm g;
    g.M = g.N = g.K = n;
    g.A = Q2;
    g.B = U;
    g.C = Q;
    g.lda = g.ldb = g.ldc = Pp;
    g.sA = g.sB = g.sC = int64_t(n) * (Pp + 1);
    g.batch = nm;
    gemm(ctx, g, TNH_PREC_F64);
    cur ^= 1;
  }
  hipLaunchKernelGGL(tri_out_kernel, dim3(unsigned(p / 256 + 1)), dim3(256), 0, st, w, cur, dout);
  TNH_HIP(hipGetLastError());
}

void tri_eig_vectors(tnh_ctx *ctx, int p, bool cplx, const int *perm, int k, double *basis) {
  const int PL = cplx ? 2 : 1;
  const int Pp = leaves_of(p).Pp;
  const int64_t tot = int64_t(p) * k, pp = int64_t(p) * p;
  const double *Z = static_cast<const double *>(ctx->workspace(641, sizeof(double) * int64_t(Pp) * Pp));
  const double *V = static_cast<const double *>(ctx->workspace(640, sizeof(double) * pp * PL));
  const double *taus = static_cast<const double *>(ctx->workspace(645, sizeof(double) * 2 * p));
  hipLaunchKernelGGL(tri_gather_kernel, dim3(unsigned((tot + 255) / 256)), dim3(256), 0, ctx->stream, Z, int64_t(Pp),
                     perm, p, tot, cplx, basis);
  if (p <= kBackWaveMax) {
    if (cplx)
      launch_back<true>(ctx, V, p, taus, basis, k);
    else
      launch_back<false>(ctx, V, p, taus, basis, k);
    TNH_HIP(hipGetLastError());
    return;
  }
  // panels of reflectors, last to first: X <- X - (V T) (V^H X)
  const int nb = panel_width(cplx), full = p / nb, np = panel_count(p, cplx);
  const int64_t s2 = int64_t(np) * nb * nb;
  double *S = static_cast<double *>(ctx->workspace(646, sizeof(double) * s2 * PL));
  double *T = static_cast<double *>(ctx->workspace(647, sizeof(double) * s2 * PL));
  double *VT = static_cast<double *>(ctx->workspace(648, sizeof(double) * pp * PL));
  double *X = static_cast<double *>(ctx->workspace(649, sizeof(double) * int64_t(nb) * k * PL));
  auto opnd = [&](const double *a, int64_t off, int64_t plane, bool conj = false) {
    COperand o;
    o.re = a + off;
    o.im = cplx ? a + plane + off : nullptr;
    o.conj = conj;
    return o;
  };
  // S_b = V_b^H V_b and (V T)_b for panels b0 .. b0 + nbatch - 1 of width wd
  auto grams = [&](int b0, int nbatch, int wd) {
    Gemm g;
    g.M = g.N = wd;
    g.K = p;
    g.transA = true;
    g.lda = g.ldb = p;
    g.ldc = nb;
    g.sA = g.sB = int64_t(nb) * p;
    g.sC = int64_t(nb) * nb;
    g.batch = nbatch;
    const int64_t v0 = int64_t(b0) * nb * p, c0 = int64_t(b0) * nb * nb;
    cgemm(ctx, g, opnd(V, v0, pp, true), opnd(V, v0, pp), S + c0, cplx ? S + s2 + c0 : nullptr, TNH_F64, TNH_PREC_F64);
  };
  auto vts = [&](int b0, int nbatch, int wd) {
    Gemm g;
    g.M = p;
    g.N = g.K = wd;
    g.lda = g.ldc = p;
    g.ldb = nb;
    g.sA = g.sC = int64_t(nb) * p;
    g.sB = int64_t(nb) * nb;
    g.batch = nbatch;
    const int64_t v0 = int64_t(b0) * nb * p, c0 = int64_t(b0) * nb * nb;
    cgemm(ctx, g, opnd(V, v0, pp), opnd(T, c0, s2), VT + v0, cplx ? VT + pp + v0 : nullptr, TNH_F64, TNH_PREC_F64);
  };
  if (full) grams(0, full, nb);
  if (np > full) grams(full, 1, p - full * nb);
  const size_t tl = sizeof(double) * nb * nb * PL;
  if (cplx)
    hipLaunchKernelGGL(tri_tfac_kernel<true>, dim3(unsigned(np)), dim3(256), tl, ctx->stream, S, nb, s2, p, taus, T);
  else
    hipLaunchKernelGGL(tri_tfac_kernel<false>, dim3(unsigned(np)), dim3(256), tl, ctx->stream, S, nb, s2, p, taus, T);
  TNH_HIP(hipGetLastError());
  if (full) vts(0, full, nb);
  if (np > full) vts(full, 1, p - full * nb);
  for (int b = np - 1; b >= 0; --b) {
    const int r0 = b * nb, wd = std::min(nb, p - r0), rows = p - r0;
    const int64_t v0 = int64_t(b) * nb * p + r0, xk = int64_t(nb) * k;
    Gemm g;  // X = V_b^H basis
    g.M = wd;
    g.N = k;
    g.K = rows;
    g.transA = true;
    g.lda = g.ldb = p;
    g.ldc = nb;
    cgemm(ctx, g, opnd(V, v0, pp, true), opnd(basis, r0, tot), X, cplx ? X + xk : nullptr, TNH_F64, TNH_PREC_F64);
    Gemm h;  // basis -= (V T)_b X
    h.M = rows;
    h.N = k;
    h.K = wd;
    h.lda = h.ldc = p;
    h.ldb = nb;
    h.alpha = -1.0;
    h.beta = 1.0;
    cgemm(ctx, h, opnd(VT, v0, pp), opnd(X, 0, xk), basis + r0, cplx ? basis + tot + r0 : nullptr, TNH_F64,
          TNH_PREC_F64);
  }
}

}  // namespace tnh
