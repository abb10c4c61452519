// Davidson eigensolver for the CC Jacobian with every vector and all reduced-
// space linear algebra on the device, in FP64.
//
// Follows eT's eigen Davidson solver (run_eigen_davidson_solver,
// src/solvers/eigen_davidson_solver_class.F90:122-318, and the tools in
// src/solver_tools/davidson/): trial vectors V and their transforms AV in HBM,
// reduced matrix G = V^T A V, its lowest eigenpairs, residuals
// R = (A X - w X) / ||X|| (construct_residual_eigen_davidson_tool,
// eigen_davidson_tool_class.F90:382-461), diagonal preconditioning by the
// orbital differences, Gram-Schmidt orthonormalisation against the space
// (davidson_tool_class.F90:354), restart on the current Ritz vectors when the
// reduced dimension would exceed its maximum (default max(100, 10 n_states),
// cc_es_amplitudes_solver_factory_class.F90:307), linear-dependence threshold
// min(1e-11, 0.1 threshold) (:315).
//
// The reduced eigenproblem (non-symmetric, dimension <= 128): one wavefront does
// the Householder reduction to upper Hessenberg form and the implicitly double-
// shifted QR iteration for the eigenvalues (francis.hpp), then one wavefront per
// wanted real root the inverse iteration on G - w I with a partially pivoted LU
// (for a complex pair a +- ib, the real 2k system of u + i v).  Complex pairs are
// carried as (u, v) column pairs with real and imaginary residuals, as eT's
// Davidson tool does.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "ccsd.hpp"
#include "francis.hpp"
#include "kernels.hpp"

namespace etg {
namespace {

constexpr int kMaxRed = 128;
constexpr int kLanes = 64;

__device__ inline double sgn(double a, double b) { return b >= 0.0 ? fabs(a) : -fabs(a); }

// Adds (or takes the larger of) each lane's value and that of the lane that the
// DPP control names; lanes outside the row mask and past the row's edge add 0.
template <int kCtrl, int kRows>
__device__ inline double dpp_add(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(u)), kCtrl, kRows, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, int(u >> 32), kCtrl, kRows, 0xf, true);
  return v + __builtin_bit_cast(double, (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo));
}
template <int kCtrl, int kRows>
__device__ inline uint32_t dpp_max(uint32_t v) {
  return max(v, uint32_t(__builtin_amdgcn_update_dpp(0, int(v), kCtrl, kRows, 0xf, true)));
}

// Lane `from`'s value (from is the same in every lane).
__device__ inline double lane_value(double v, int from) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u)), from));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(u >> 32), from));
  return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}

// Sum / largest over the wavefront, in every lane.  Six DPP steps: a shuffle
// through LDS costs a round trip per step, and these reductions sit in the
// middle of serial chains.
__device__ inline double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8: lane 15 of each row of 16 has the row's sum
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);   // row_bcast 15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);   // row_bcast 31 into rows 2 and 3
  return lane_value(v, kLanes - 1);
}
__device__ inline uint32_t wave_max(uint32_t v) {
  v = dpp_max<0x111, 0xf>(v);
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);
  v = dpp_max<0x143, 0xc>(v);
  return uint32_t(__builtin_amdgcn_readlane(int(v), kLanes - 1));
}

// Orders the memory accesses of one wavefront: they execute in program order, so
// only the compiler has to keep it.
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The reduced eigensolver's team: one wavefront.
struct WaveTeam {
  __device__ int rank() const { return int(threadIdx.x); }
  __device__ int size() const { return kLanes; }
  __device__ void sync() const { wave_sync(); }
  __device__ double sum(double v) const { return wave_sum(v); }
  template <class F>
  __device__ int highest(int top, F f) const {
    for (; top > 0; top -= kLanes) {
      const int l = top - rank();
      const uint64_t hit = __ballot(l > 0 && f(l));
      if (hit != 0) return top - __builtin_ctzll(hit);
    }
    return 0;
  }
};

// H(i, j) of the k x k working matrix in LDS, column-major with the odd leading
// dimension kLdH: lanes that walk a row touch distinct banks.
constexpr int kLdH = kMaxRed + 1;
#define HH(i, j) H[(i) + (j) * kLdH]

// G - shift I into LDS, eight columns per round: their global loads are in flight together.
__device__ void load_shifted(double* H, const double* __restrict__ G, int k, int64_t ldg, double shift) {
  for (int i = threadIdx.x; i < k; i += kLanes)
    for (int j0 = 0; j0 < k; j0 += 8) {
      double g[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) g[u] = j0 + u < k ? G[i + (j0 + u) * ldg] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (j0 + u < k) HH(i, j0 + u) = g[u] - (i == j0 + u ? shift : 0.0);
    }
  wave_sync();
}

// Inverse iteration on the nm x nm matrix M (ld ldm; LDS or global; nm at most
// 64 kRows): LU with partial pivoting in place, then three solves M y = y
// starting from a fixed pattern, each normalised to unit 2-norm (largest
// component positive).  Row i of y is yv[i / 64] of lane i % 64; perm holds the
// row order of the pivoting.  For real roots M = G - (w + d) I; for a complex
// pair a +- ib the real 2k system [[G - a I, b I], [-b I, G - a I]] acting on
// [u; v] (eigenvector u + i v).
//
// One dependent chain: what costs is the latency of each of its steps.  The
// solves keep y in registers and broadcast one element per column by readlane
// (the columns of M do not depend on it and are read ahead), the pivot is the
// largest high word (20 bits of the mantissa: as stable as the largest value).
template <int kRows>
__device__ void inverse_iteration(double* M, int ldm, int nm, double anorm, int* perm, double (&yv)[kRows],
                                  int seed, int lane) {
#define MM(i, j) M[(i) + (j) * ldm]
  for (int i = lane; i < nm; i += kLanes) perm[i] = i;
  wave_sync();
  for (int c = 0; c < nm; ++c) {
    uint32_t key = 0;
    int row = c;
    for (int r = c + lane; r < nm; r += kLanes) {
      const uint32_t v = uint32_t(__builtin_bit_cast(uint64_t, MM(r, c)) >> 32) & 0x7fffffffu;
      if (v > key) {
        key = v;
        row = r;
      }
    }
    const uint32_t top = wave_max(key);
    const int p = top == 0 ? c : __builtin_amdgcn_readlane(row, __builtin_ctzll(__ballot(key == top)));
    if (p != c) {
      for (int j = lane; j < nm; j += kLanes) {
        const double tmp = MM(c, j);
        MM(c, j) = MM(p, j);
        MM(p, j) = tmp;
      }
      if (lane == 0) {
        const int tmp = perm[c];
        perm[c] = perm[p];
        perm[p] = tmp;
      }
      wave_sync();
    }
    double d = MM(c, c);
    if (d == 0.0) {
      d = 1e-300 + 1e-16 * anorm;
      wave_sync();
      if (lane == 0) MM(c, c) = d;
    }
    // rows across the lanes; at most half a wavefront of them: two lanes per row,
    // each with every other column
    const int rows = nm - c - 1;
    const int step = rows <= kLanes / 2 ? 2 : 1;
    const int first = step == 2 ? lane % (kLanes / 2) : lane, half = step == 2 ? lane / (kLanes / 2) : 0;
    for (int r = c + 1 + first; r < nm; r += kLanes) {
      const double f = MM(r, c) / d;
      // four columns per round: their loads go out before the stores
      int j = c + 1 + half;
      for (; j + 3 * step < nm; j += 4 * step) {
        const double p0 = MM(c, j), p1 = MM(c, j + step), p2 = MM(c, j + 2 * step), p3 = MM(c, j + 3 * step);
        const double a0 = MM(r, j), a1 = MM(r, j + step), a2 = MM(r, j + 2 * step), a3 = MM(r, j + 3 * step);
        MM(r, j) = a0 - f * p0;
        MM(r, j + step) = a1 - f * p1;
        MM(r, j + 2 * step) = a2 - f * p2;
        MM(r, j + 3 * step) = a3 - f * p3;
      }
      for (; j < nm; j += step) MM(r, j) -= f * MM(c, j);
      wave_sync();                                       // both lanes of the row have read MM(r, c)
      if (half == 0) MM(r, c) = f;
    }
    wave_sync();
  }
  double rd[kRows];                                      // 1 / diagonal
  int src[kRows];
#pragma unroll
  for (int s = 0; s < kRows; ++s) {
    const int i = lane + s * kLanes;
    rd[s] = i < nm ? 1.0 / MM(i, i) : 0.0;
    src[s] = i < nm ? perm[i] : i;
    yv[s] = i < nm ? 1.0 + 0.01 * ((i * 7 + seed * 3) % 11) : 0.0;
  }
  auto element = [&](const double (&v)[kRows], int c) {  // element c of a vector, to all lanes
    double e = v[0];
#pragma unroll
    for (int s = 1; s < kRows; ++s)
      if (c / kLanes == s) e = v[s];
    return lane_value(e, c % kLanes);
  };
  for (int iter = 0; iter < 3; ++iter) {
    double t[kRows];
#pragma unroll
    for (int s = 0; s < kRows; ++s) {                    // y in the pivots' order
      t[s] = 0.0;
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        const double v = __shfl(yv[u], src[s] % kLanes, kLanes);
        if (src[s] / kLanes == u) t[s] = v;
      }
    }
    // triangular solves column by column, four columns' entries read ahead
    for (int c0 = 0; c0 < nm; c0 += 4) {                 // unit lower L
      double m[4][kRows];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int s = 0; s < kRows; ++s) {
          const int i = lane + s * kLanes;
          m[q][s] = c0 + q < nm && i > c0 + q && i < nm ? MM(i, c0 + q) : 0.0;
        }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (c0 + q < nm) {
          const double yc = element(t, c0 + q);
#pragma unroll
          for (int s = 0; s < kRows; ++s) t[s] -= m[q][s] * yc;
        }
    }
    for (int c0 = nm - 1; c0 >= 0; c0 -= 4) {            // upper U
      double m[4][kRows];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int s = 0; s < kRows; ++s) {
          const int i = lane + s * kLanes;
          m[q][s] = i < c0 - q ? MM(i, c0 - q) : 0.0;
        }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (c0 - q >= 0) {
          const int c = c0 - q;
          const double yc = element(t, c) * element(rd, c);
#pragma unroll
          for (int s = 0; s < kRows; ++s) t[s] = lane + s * kLanes == c ? yc : t[s] - m[q][s] * yc;
        }
    }
    double sq = 0.0, big = 0.0;
    int ib = 0;
#pragma unroll
    for (int s = 0; s < kRows; ++s) {
      sq += t[s] * t[s];
      if (fabs(t[s]) > big) {
        big = fabs(t[s]);
        ib = lane + s * kLanes;
      }
    }
    const double nrm = sqrt(wave_sum(sq));
    for (int off = kLanes / 2; off > 0; off >>= 1) {     // the first of the largest components
      const double ob = __shfl_xor(big, off, kLanes);
      const int oi = __shfl_xor(ib, off, kLanes);
      if (ob > big || (ob == big && oi < ib)) {
        big = ob;
        ib = oi;
      }
    }
    const double sg = element(t, __builtin_amdgcn_readfirstlane(ib)) < 0.0 ? -1.0 : 1.0;
#pragma unroll
    for (int s = 0; s < kRows; ++s) yv[s] = sg * t[s] / nrm;
  }
#undef MM
}

// Eigenvalues, ordered by real part then imaginary part, the matrix's norm and
// the status (1: no convergence).  One wavefront, bound by its chain of dependent
// steps (about 0.6 us per step of the bulge chase).  With the vectors' kernel, for
// 4 roots: 95 us at k = 10, 0.27 ms at 20, 0.97 at 40, 6.7 at 100; as one kernel
// with two barriers and two round trips through LDS per step, and the roots one
// after another: 0.20, 0.54, 1.70 and 9.8 ms.
__global__ __launch_bounds__(kLanes) void reduced_eigenvalues_kernel(const double* __restrict__ G, int k,
                                                                     int ldg, double* __restrict__ wr_out,
                                                                     double* __restrict__ wi_out,
                                                                     double* __restrict__ norm_out,
                                                                     int* __restrict__ info,
                                                                     double* __restrict__ host_out) {
  __shared__ double H[kLdH * kMaxRed];
  __shared__ double wr[kMaxRed], wi[kMaxRed], ort[kMaxRed];
  const int lane = threadIdx.x;
  load_shifted(H, G, k, ldg, 0.0);

  // ---- Householder reduction to upper Hessenberg form (orthes) ----
  for (int m = 1; m < k - 1; ++m) {
    const int i0 = m + lane, i1 = i0 + kLanes;
    const double u0 = i0 < k ? HH(i0, m - 1) : 0.0, u1 = i1 < k ? HH(i1, m - 1) : 0.0;
    const double scale = wave_sum(fabs(u0) + fabs(u1));
    if (scale == 0.0) continue;
    const double s0 = u0 / scale, s1 = u1 / scale;
    double h = wave_sum(s0 * s0 + s1 * s1);
    const double x = lane_value(s0, 0);                  // the entry that stays
    const double g = -sgn(sqrt(h), x);
    h -= x * g;
    if (i0 < k) {
      ort[i0] = s0 - (lane == 0 ? g : 0.0);
      HH(i0, m - 1) = lane == 0 ? scale * g : 0.0;
    }
    if (i1 < k) {
      ort[i1] = s1;
      HH(i1, m - 1) = 0.0;
    }
    wave_sync();
    const double rh = 1.0 / h;
    // (I - u u^T / h) H: a column per lane, then H (I - u u^T / h): a row per lane
    for (int side = 0; side < 2; ++side) {
      const int st = side == 0 ? 1 : kLdH;
      for (int q = (side == 0 ? m : 0) + lane; q < k; q += kLanes) {
        double* p = side == 0 ? &HH(0, q) : &HH(q, 0);
        double f[4] = {0.0, 0.0, 0.0, 0.0};
        for (int i = m; i < k; i += 4)
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (i + u < k) f[u] += ort[i + u] * p[(i + u) * st];
        const double w = ((f[0] + f[1]) + (f[2] + f[3])) * rh;
        for (int i = m; i < k; i += 4) {
          double v[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) v[u] = i + u < k ? p[(i + u) * st] - w * ort[i + u] : 0.0;
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (i + u < k) p[(i + u) * st] = v[u];
        }
      }
      wave_sync();
    }
  }

  // ---- eigenvalues of the Hessenberg matrix (implicit double-shift QR) ----
  double anorm = 0.0;
  const int st = francis::hessenberg_eigenvalues(WaveTeam(), H, kLdH, k, wr, wi, &anorm);
  if (lane == 0) {
    *norm_out = anorm;
    *info = st;
    if (host_out) host_out[2 * kMaxRed] = double(st);
  }
  if (st != 0) return;
  for (int i = lane; i < k; i += kLanes) {
    int rank = 0;
    for (int j = 0; j < k; ++j) {
      const bool eq = wr[j] == wr[i];
      rank += wr[j] < wr[i] || (eq && (wi[j] < wi[i] || (wi[j] == wi[i] && j < i)));
    }
    wr_out[rank] = wr[i];
    wi_out[rank] = wi[i];
    if (host_out) {
      host_out[rank] = wr[i];
      host_out[kMaxRed + rank] = wi[i];
    }
  }
}

// Eigenvectors of the n_want lowest roots by inverse iteration.  Real root w:
// column w of X.  Complex pair a -+ ib (ordered a - ib first): columns w and
// w + 1 hold u and v of the eigenvector u + i v of a + ib.  Block w < n_want: the
// real root w with those after it that are numerically the same (each made
// orthogonal to the earlier ones), unless it belongs to an earlier root; block
// n_want: the complex pairs, one after another in the one 2k x 2k workspace.
// Bound by each block's chain of dependent steps: 63 us at k = 40 for 4 roots.
__global__ __launch_bounds__(kLanes) void reduced_eigenvectors_kernel(
    const double* __restrict__ G, int k, int ldg, int n_want, const double* __restrict__ wr,
    const double* __restrict__ wi, const double* __restrict__ norm, const int* __restrict__ info,
    double* __restrict__ X, int ldx, double* __restrict__ work) {
  __shared__ double H[kLdH * kMaxRed];
  __shared__ int perm[2 * kMaxRed];
  const int lane = threadIdx.x;
  if (*info != 0) return;
  const double anorm = *norm;
  if (int(blockIdx.x) < n_want) {
    // the same root: within 1e-8; a chain of them is taken with twice that, so that
    // no two roots that are the same end up in different blocks
    auto near = [&](int u, int w, double tol) { return fabs(wr[u] - wr[w]) <= tol * fmax(1.0, fabs(wr[w])); };
    auto after = [&](int w) {                            // next real root, or n_want
      for (++w; w < n_want && wi[w] != 0.0; ++w) {
      }
      return w;
    };
    int w = blockIdx.x;
    if (wi[w] != 0.0) return;
    int before = w - 1;
    while (before >= 0 && wi[before] != 0.0) --before;
    if (before >= 0 && near(before, w, 2e-8)) return;
    for (const int head = w;;) {
      const double lam = wr[w];
      load_shifted(H, G, k, ldg, lam + 1e-13 * fmax(anorm / k, fabs(lam)));
      double y[2];
      inverse_iteration<2>(H, kLdH, k, anorm, perm, y, w, lane);
      const int i0 = lane, i1 = lane + kLanes;
      for (int u = head; u < w; ++u) {
        if (wi[u] != 0.0 || !near(u, w, 1e-8)) continue;
        const double x0 = i0 < k ? X[i0 + u * int64_t(ldx)] : 0.0, x1 = i1 < k ? X[i1 + u * int64_t(ldx)] : 0.0;
        const double dp = wave_sum(x0 * y[0] + x1 * y[1]);
        y[0] -= dp * x0;
        y[1] -= dp * x1;
      }
      const double nrm = sqrt(wave_sum(y[0] * y[0] + y[1] * y[1]));
      if (i0 < k) X[i0 + w * int64_t(ldx)] = y[0] / nrm;
      if (i1 < k) X[i1 + w * int64_t(ldx)] = y[1] / nrm;
      const int next = after(w);
      if (next >= n_want || !near(w, next, 2e-8)) return;
      w = next;
      wave_sync();
    }
  }
  for (int w = 0; w < n_want; ++w) {
    const double lam = wr[w], mu = wi[w];
    if (!(mu < 0.0)) continue;
    const double a = lam + 1e-13 * fmax(anorm / k, fabs(lam)), b = -mu;
    const int n2 = 2 * k;
    for (int q = lane; q < n2 * n2; q += kLanes) {
      const int i = q % n2, j = q / n2;
      const int bi = i / k, bj = j / k, ii = i % k, jj = j % k;
      double v;
      if (bi == bj) v = G[ii + jj * int64_t(ldg)] - (ii == jj ? a : 0.0);
      else v = (ii == jj) ? (bi == 0 ? b : -b) : 0.0;
      work[i + int64_t(j) * n2] = v;
    }
    __syncthreads();
    double y[4];
    inverse_iteration<4>(work, n2, n2, anorm, perm, y, w, lane);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int i = lane + s * kLanes;
      if (i < k) X[i + w * int64_t(ldx)] = y[s];
      else if (i < n2 && w + 1 < n_want) X[i - k + (w + 1) * int64_t(ldx)] = y[s];
    }
    __syncthreads();
    ++w;                                  // the partner a + ib is done
  }
}
#undef HH

constexpr int kBlock = 256;
unsigned grid_for_d(int64_t n) { return unsigned(std::min<int64_t>((n + kBlock - 1) / kBlock, 1 << 16)); }

// R_j = AY_j - w_j Y_j - c_j Y_{p_j}  (n x s, column-major, ld n).  Real root:
// c_j = 0.  Complex pair a -+ ib in columns (j, j+1) = (u, v): R_j = Au - a u + b v,
// R_{j+1} = Av - a v - b u (eigen_davidson_tool construct_re/im_residual).
// coef = [w (s) | c (s) | p (s)] on the device.
__global__ void ritz_residual_kernel(const double* __restrict__ AY, const double* __restrict__ Y,
                                     const double* __restrict__ coef, int64_t n, int s,
                                     double* __restrict__ R) {
  for (int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; q < n * s;
       q += int64_t(gridDim.x) * blockDim.x) {
    const int j = int(q / n);
    const int64_t i = q - int64_t(j) * n;
    const int p = int(coef[2 * s + j]);
    R[q] = AY[q] - coef[j] * Y[q] - coef[s + j] * Y[i + int64_t(p) * n];
  }
}

// The residuals that become new trial vectors: column c from column src[c] >= c
// (increasing) of the block, preconditioned with root w[c].
constexpr int kMaxRoots = kMaxRed / 2 - 1;
struct NewColumns {
  int n;
  int src[kMaxRoots];
  double w[kMaxRoots];
};

// R[:, c] = R[:, src] / (w - d), guarded where the denominator vanishes (diagonal
// preconditioner).  A thread takes its element of all columns in turn: each is
// read before the column that it is in is written.
__global__ void precondition_kernel(double* R, const double* __restrict__ d, NewColumns cols, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const double di = d[i];
    for (int c = 0; c < cols.n; ++c) {
      double den = cols.w[c] - di;
      if (fabs(den) < 1e-8) den = den < 0.0 ? -1e-8 : 1e-8;
      R[i + c * n] = R[i + cols.src[c] * n] / den;
    }
  }
}

// Columns to unit norm, from their squared norms on the device (zero columns stay
// zero: they are dropped as linearly dependent).
__global__ void normalize_kernel(double* X, const double* __restrict__ sq, int64_t n) {
  double* x = X + blockIdx.y * n;
  const double s = sq[blockIdx.y];
  const double f = s > 0.0 ? 1.0 / sqrt(s) : 0.0;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    x[i] = f * x[i];
}

// T = R^-1 of the Cholesky factor R (upper) of the q x q Gram matrix, q <= 64, by
// one wavefront: lane j holds column j's row of work.  *ok = 0 (and T the identity)
// when a pivot falls below 1e-8 of its diagonal entry.  The host would need the
// matrix, its factor and two waits, 40-60 us for a few columns.
__global__ __launch_bounds__(kLanes) void cholesky_inverse_kernel(const double* __restrict__ gram, int q,
                                                                  double* __restrict__ T, double* __restrict__ ok) {
  __shared__ double A[kLanes][kLanes + 1], V[kLanes][kLanes + 1];
  const int j = threadIdx.x;
  if (j < q)
    for (int i = 0; i < q; ++i) A[i][j] = gram[i + j * q];
  const double diag = j < q ? gram[j + j * q] : 0.0;
  wave_sync();
  bool good = true;
  for (int c = 0; c < q; ++c) {
    const double pivot = A[c][c];
    if (!(pivot > 1e-8 * lane_value(diag, c))) {
      good = false;
      break;
    }
    const double r = sqrt(pivot);
    wave_sync();
    if (j >= c && j < q) A[c][j] = j == c ? r : A[c][j] / r;
    wave_sync();
    if (j > c && j < q)
      for (int i = c + 1; i <= j; ++i) A[i][j] -= A[c][i] * A[c][j];
    wave_sync();
  }
  if (j < q) {
    for (int i = q - 1; i >= 0; --i) {
      double v = i == j ? 1.0 : 0.0;
      if (good && i == j) v = 1.0 / A[j][j];
      if (good && i < j) {
        double s = 0.0;
        for (int l = i + 1; l <= j; ++l) s += A[i][l] * V[l][j];
        v = -s / A[i][i];
      }
      V[i][j] = v;
      T[i + j * q] = v;
    }
  }
  if (j == 0) *ok = good ? 1.0 : 0.0;
}

}  // namespace

namespace {

// Doubles of the reduced eigensolver's device workspace: eigenvalues (2 x 128),
// the real 2k x 2k system of a complex pair (4 x 128^2), the matrix's norm, the
// status flag.
constexpr size_t kEigenWork = 2 * kMaxRed + 4 * kMaxRed * kMaxRed + 2;

// The same workspace as a file-scope array, for the entry point that allocates
// nothing (one copy per GPU, 526 KB, held until the process ends).  Host code
// uses only the address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) double scratch[kEigenWork];

// Launches the solve with its workspace at `base` (kEigenWork doubles) and
// returns wr, wi to the host (through 2 kMaxRed + 1 doubles of pinned memory where
// the caller has some); throws on QR non-convergence.
void reduced_eigen_launch(hipStream_t stream, double* base, const double* G_dev, int64_t k, int64_t ldg,
                          int64_t n_want, double* wr, double* wi, double* X_dev, int64_t ldx,
                          double* pinned = nullptr) {
  if (k < 1 || k > kMaxRed) fail("reduced eigenproblem: dimension must be in [1, 128]");
  if (n_want < 0 || n_want > k) fail("reduced eigenproblem: invalid number of wanted roots");
  if (ldg < k || ldx < k) fail("reduced eigenproblem: leading dimension below the dimension");
  double* dwr = base;                       // wr, wi, norm, status: one copy to the host
  double* dwi = dwr + kMaxRed;
  double* dnorm = dwi + kMaxRed;
  int* dinfo = reinterpret_cast<int*>(dnorm + 1);
  double* work = dnorm + 2;                 // (2k)^2: a complex pair's system
  reduced_eigenvalues_kernel<<<1, kLanes, 0, stream>>>(G_dev, int(k), int(ldg), dwr, dwi, dnorm, dinfo, pinned);
  ETG_LAUNCH("reduced_eigenvalues");
  if (n_want > 0) {
    reduced_eigenvectors_kernel<<<unsigned(n_want + 1), kLanes, 0, stream>>>(
        G_dev, int(k), int(ldg), int(n_want), dwr, dwi, dnorm, dinfo, X_dev, int(ldx), work);
    ETG_LAUNCH("reduced_eigenvectors");
  }
  double copy[2 * kMaxRed + 2];
  if (!pinned) ETG_HIP(hipMemcpyAsync(copy, base, sizeof copy, hipMemcpyDeviceToHost, stream));
  ETG_HIP(hipStreamSynchronize(stream));
  int info = 0;
  if (!pinned) std::memcpy(&info, copy + 2 * kMaxRed + 1, sizeof info);
  const double* host = pinned ? pinned : copy;
  std::copy(host, host + k, wr);
  std::copy(host + kMaxRed, host + kMaxRed + k, wi);
  if (pinned) info = int(pinned[2 * kMaxRed]);
  if (info == 1) fail("reduced eigenproblem: QR iteration did not converge");
}

// Device address of `scratch` on the current device, looked up once per device.
double* scratch_address() {
  static std::mutex mu;
  static std::vector<double*> addr;
  int dev = 0;
  ETG_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  if (size_t(dev) >= addr.size()) addr.resize(size_t(dev) + 1, nullptr);
  if (addr[size_t(dev)] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      fail(std::string("reduced eigenproblem: no device address for the static workspace: ") +
           hipGetErrorString(e));
    addr[size_t(dev)] = static_cast<double*>(p);
  }
  return addr[size_t(dev)];
}

}  // namespace

void reduced_eigen_solve(hipStream_t stream, DeviceBuffer& workspace, const double* G_dev, int64_t k,
                         int64_t ldg, int64_t n_want, double* wr, double* wi, double* X_dev,
                         int64_t ldx, double* pinned) {
  if (k < 1 || k > kMaxRed) fail("reduced eigenproblem: dimension must be in [1, 128]");
  workspace.resize(sizeof(double) * kEigenWork);
  reduced_eigen_launch(stream, workspace.as<double>(), G_dev, k, ldg, n_want, wr, wi, X_dev, ldx, pinned);
}

void reduced_eigen_solve_noalloc(hipStream_t stream, const double* G_dev, int64_t k, int64_t ldg,
                                 int64_t n_want, double* wr, double* wi, double* X_dev, int64_t ldx) {
  if (k < 1 || k > kMaxRed)
    fail("reduced eigenproblem (no-allocation entry): dimension " + std::to_string(k) +
         " outside [1, 128], the size of its static workspace");
  reduced_eigen_launch(stream, scratch_address(), G_dev, k, ldg, n_want, wr, wi, X_dev, ldx);
}

void CCSD::reduced_eigen(const double* G_dev, int64_t k, int64_t ldg, int64_t n_want, double* wr,
                         double* wi, double* X_dev, int64_t ldx) {
  static_assert(kBlockResults + 2 * kMaxRed + 1 <= kResults, "room for the eigenvalues");
  reduced_eigen_solve(stream_, red_eig_, G_dev, k, ldg, n_want, wr, wi, X_dev, ldx,
                      red_result_.on_host() ? red_result_.as<double>() + kBlockResults : nullptr);
}

int64_t CCSD::davidson(int side, int64_t n_states, double threshold, int64_t max_iterations,
                       int64_t max_dim, Prec prec, const double* start, double* energies,
                       double* vectors, double* residual_norms) {
  require(tape_ != nullptr, "davidson: prepare_for_jacobian has not been called");
  require(have_eps_, "davidson: orbital energies required");
  require(side == 0 || side == 1, "davidson: side must be 0 (right) or 1 (left)");
  struct Clock {                          // wall time of the solve (davidson_timing)
    double& total;
    std::chrono::steady_clock::time_point t0 = std::chrono::steady_clock::now();
    ~Clock() { total += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count(); }
  } clock{dav_timing_[1]};
  const int64_t n = n_t1 + n_t2;
  require(n_states >= 1 && n_states <= std::min<int64_t>(n - 1, 62), "davidson: n_states must be in [1, 62]");
  if (max_dim <= 0) max_dim = std::max<int64_t>(100, 10 * n_states);
  max_dim = std::min<int64_t>(std::min<int64_t>(max_dim, kMaxRed), n);
  require(max_dim >= 2 * (n_states + 1),
          "davidson: maximum reduced dimension below twice the number of states plus two");
  const double lindep = std::min(1e-11, 0.1 * threshold);
  const int64_t s = n_states, s1 = n_states + 1;    // a complex pair may straddle the last root

  // HBM: Y, AY, R (n x s1), G (max_dim^2), Xr and the projection coefficients
  // (max_dim x s1 each), [w | c | partner] (3 s1), Gram-Schmidt coefficients.
  // V and AV (n x max_dim): in HBM when both fit in half of the free memory
  // (the transformation passes size their vector groups from the rest),
  // otherwise AV, and then V as well, in pinned host memory that the kernels
  // read and write over PCIe (etg_set_davidson_space overrides the choice).
  dav_Y_.resize(sizeof(double) * size_t(n) * size_t(3 * s1));
  dav_small_.resize(sizeof(double) * size_t(max_dim * max_dim + 2 * max_dim * s1 + 3 * s1 + max_dim + 2 * s1 * s1 + s1));
  {
    const size_t space = sizeof(double) * size_t(n) * size_t(max_dim);
    const size_t held = (dav_V_.on_host() ? 0 : dav_V_.bytes()) + (dav_AV_.on_host() ? 0 : dav_AV_.bytes());
    const double avail = 0.5 * double(size_t(free_memory()) + held);
    bool v_host = false, av_host = false;
    if (dav_space_ == 2) {
      v_host = av_host = true;
    } else if (dav_space_ == 0) {
      av_host = 2.0 * double(space) > avail;
      v_host = double(space) > avail;
    }
    // release first so that the other buffer can take the memory
    if (dav_V_.on_host() != v_host) dav_V_.release();
    if (dav_AV_.on_host() != av_host) dav_AV_.release();
    // pinned host memory can be refused (the system's limit on locked pages): the
    // buffer then goes to HBM after all
    auto place = [&](DeviceBuffer& b, bool host) {
      if (host) {
        try {
          b.resize_host(space);
          return;
        } catch (const Error&) {
          (void)hipGetLastError();
          b.release();
        }
      }
      b.resize(space);
    };
    place(dav_AV_, av_host);
    place(dav_V_, v_host);
  }
  double* V = dav_V_.as<double>();
  double* AV = dav_AV_.as<double>();
  double* Y = dav_Y_.as<double>();
  double* AY = Y + n * s1;
  double* Rb = Y + 2 * n * s1;
  double* G = dav_small_.as<double>();
  double* Xr = G + max_dim * max_dim;
  double* cmat = Xr + max_dim * s1;          // projection coefficients (max_dim x s1)
  double* coef = cmat + max_dim * s1;        // [w | c | partner] (3 s1)
  double* cvec = coef + 3 * s1;              // Gram-Schmidt coefficients (max_dim)
  double* gram = cvec + max_dim;             // Gram matrix of a block (s1 x s1)
  double* tmat = gram + s1 * s1;             // inverse Cholesky factor of a block (s1 x s1)
  double* sums = tmat + s1 * s1;             // squared norms of the new vectors (s1)
  double* flags = red_result_.as<double>() + 5;   // success of the two Cholesky factorisations
  diff_.resize(sizeof(double) * n);
  double* d = diff_.as<double>();
  orbital_differences(stream_, eps_.as<double>(), d, n_o, n_v, n);

  auto dot_host = [&](const double* a, const double* b) {
    double* res = red_result_.as<double>() + 3;
    dot(stream_, a, b, n, red_partial_.as<double>(), res);
    return result(res);
  };
  // Cholesky QR twice of q columns at X, through W: X T with T = R^-1, R^T R =
  // X^T X, both times (and XA T alongside, through WA, when XA is given).  It gives
  // the Q of Gram-Schmidt when every column keeps more than 1e-4 of its norm
  // against the ones before it (Cholesky pivots above 1e-8 of the diagonal); false
  // otherwise, with X and XA as they were.
  auto cholqr = [&](double* X, double* XA, int64_t q, double* W, double* WA) {
    auto factor = [&](const double* x, double* flag) {
      run_gemm(make_gemm('T', 'N', q, q, n, 1.0, x, n, x, n, 0.0, gram, q), Prec::F64);
      cholesky_inverse_kernel<<<1, kLanes, 0, stream_>>>(gram, int(q), tmat, flag);
      ETG_LAUNCH("cholesky_inverse");
    };
    auto multiply = [&](const double* x, const double* xa, double* w, double* wa) {
      run_gemm(make_gemm('N', 'N', n, q, q, 1.0, x, n, tmat, q, 0.0, w, n), Prec::F64);
      if (xa) run_gemm(make_gemm('N', 'N', n, q, q, 1.0, xa, n, tmat, q, 0.0, wa, n), Prec::F64);
    };
    factor(X, flags);
    multiply(X, XA, W, WA);
    factor(W, flags + 1);
    double ok[2];
    results(flags, 2, ok);
    if (ok[0] == 0.0 || ok[1] == 0.0) return false;
    multiply(W, WA, X, XA);
    return true;
  };
  if (start) {
    // caller's start vectors (e.g. a reduced-precision solution), orthonormalised
    // in HBM (the residual block) and then placed in the space
    ETG_HIP(hipMemcpyAsync(Rb, start, sizeof(double) * n * s, hipMemcpyDefault, stream_));
    for (int64_t j = 0; j < s; ++j) {
      for (int pass = 0; pass < 2; ++pass)
        for (int64_t i = 0; i < j; ++i) axpy(stream_, n, -dot_host(Rb + i * n, Rb + j * n), Rb + i * n, Rb + j * n);
      const double nv = std::sqrt(dot_host(Rb + j * n, Rb + j * n));
      if (!(nv > 1e-10)) fail("davidson: start vectors are linearly dependent");
      scale(stream_, Rb + j * n, n, 1.0 / nv);
    }
    ETG_HIP(hipMemcpyAsync(V, Rb, sizeof(double) * n * s, hipMemcpyDefault, stream_));
  } else {
    // unit vectors on the lowest orbital differences
    std::vector<double> hd(n);
    ETG_HIP(hipMemcpyAsync(hd.data(), d, sizeof(double) * n, hipMemcpyDeviceToHost, stream_));
    synchronize();
    std::vector<int64_t> idx(n);
    for (int64_t i = 0; i < n; ++i) idx[i] = i;
    std::partial_sort(idx.begin(), idx.begin() + s, idx.end(),
                      [&](int64_t a, int64_t b) { return hd[a] < hd[b] || (hd[a] == hd[b] && a < b); });
    fill(stream_, Rb, n * s, 0.0);
    const double one = 1.0;
    for (int64_t j = 0; j < s; ++j)
      ETG_HIP(hipMemcpyAsync(Rb + j * n + idx[j], &one, sizeof(double), hipMemcpyHostToDevice, stream_));
    ETG_HIP(hipMemcpyAsync(V, Rb, sizeof(double) * n * s, hipMemcpyDefault, stream_));
  }
  synchronize();
  int64_t k = 0, m = s;                   // space dimension, new vectors at V[:, k..k+m)
  std::vector<double> wr(max_dim), wi(max_dim), norms(s1), hcoef(3 * s1);
  double best = HUGE_VAL;                 // reduced precision: smallest largest-residual so far
  int64_t since_best = 0;
  const Prec start_prec = dav_start_prec_ < 0 ? prec : static_cast<Prec>(dav_start_prec_);
  // ETG_DAVIDSON_LOG=1: one line per iteration on stderr (progress of long solves)
  static const bool log_iterations = [] {
    const char* e = std::getenv("ETG_DAVIDSON_LOG");
    return e != nullptr && e[0] == '1';
  }();
  for (int64_t it = 1; it <= max_iterations; ++it) {
    // transforms of the new trial vectors (the start block in its own precision)
    const auto tt0 = std::chrono::steady_clock::now();
    transform_batch(side, m, V + k * n, AV + k * n, it == 1 ? start_prec : prec);
    dav_timing_[0] += std::chrono::duration<double>(std::chrono::steady_clock::now() - tt0).count();
    dav_timing_[2] += double(m);
    project_cvs(AV + k * n, m);              // eigen_davidson_solver_class.F90:187
    // G = V^T AV: new columns for all rows, new rows for the old columns
    const int64_t kn = k + m;
    run_gemm(make_gemm('T', 'N', kn, m, n, 1.0, V, n, AV + k * n, n, 0.0, G + k * max_dim, max_dim),
             Prec::F64);
    if (k > 0)
      run_gemm(make_gemm('T', 'N', m, k, n, 1.0, V + k * n, n, AV, n, 0.0, G + k, max_dim), Prec::F64);
    k = kn;
    const int64_t nw = std::min(k, s1);
    reduced_eigen(G, k, max_dim, nw, wr.data(), wi.data(), Xr, max_dim);
    // tracked columns: real roots, or complex pairs (u, v) in two columns
    int64_t se = 0;
    while (se < s && se < nw) {
      if (wi[se] < 0.0 && se + 1 < nw) {
        const double b = -wi[se];
        hcoef[se] = hcoef[se + 1] = wr[se];
        hcoef[s1 + se] = -b;
        hcoef[s1 + se + 1] = b;
        hcoef[2 * s1 + se] = double(se + 1);
        hcoef[2 * s1 + se + 1] = double(se);
        se += 2;
      } else {                            // real root (or an unpaired half: its real part)
        hcoef[se] = wr[se];
        hcoef[s1 + se] = 0.0;
        hcoef[2 * s1 + se] = double(se);
        se += 1;
      }
    }
    std::vector<double> packed(3 * se);
    for (int64_t j = 0; j < se; ++j) {
      packed[j] = hcoef[j];
      packed[se + j] = hcoef[s1 + j];
      packed[2 * se + j] = hcoef[2 * s1 + j];
    }
    // Ritz vectors and residuals
    run_gemm(make_gemm('N', 'N', n, se, k, 1.0, V, n, Xr, max_dim, 0.0, Y, n), Prec::F64);
    run_gemm(make_gemm('N', 'N', n, se, k, 1.0, AV, n, Xr, max_dim, 0.0, AY, n), Prec::F64);
    ETG_HIP(hipMemcpyAsync(coef, packed.data(), sizeof(double) * 3 * se, hipMemcpyHostToDevice, stream_));
    ritz_residual_kernel<<<grid_for_d(n * se), kBlock, 0, stream_>>>(AY, Y, coef, n, int(se), Rb);
    ETG_LAUNCH("ritz_residual");
    // squared norms of the Ritz vectors and of the residuals
    double* sq = red_result_.as<double>() + kBlockResults;
    dots(stream_, Y, n, Y, n, n, se, red_partial_.as<double>(), sq, 1);
    dots(stream_, Rb, n, Rb, n, n, se, red_partial_.as<double>(), sq + se, 1);
    std::vector<double> ynorm(2 * se);
    results(sq, 2 * se, ynorm.data());    // also waits: packed (host) is read by the copy above
    const double* rnorm = ynorm.data() + se;
    bool converged = true;
    for (int64_t j = 0; j < se; ++j) {
      const int64_t p = int64_t(hcoef[2 * s1 + j]);
      const double yy = std::sqrt(ynorm[j] + (p != j ? ynorm[p] : 0.0));
      norms[j] = std::sqrt(rnorm[j]) / yy;
      if (norms[j] >= threshold) converged = false;
    }
    for (int64_t j = 0; j < s; ++j) {
      energies[j] = hcoef[j];
      if (residual_norms) residual_norms[(it - 1) * s + j] = norms[j];
    }
    if (log_iterations) {
      double worst = 0.0;
      for (int64_t j = 0; j < s; ++j) worst = std::max(worst, norms[j]);
      std::fprintf(stderr, "davidson: iteration %lld, space %lld, %lld transformed, max residual %.3e\n",
                   (long long)it, (long long)k, (long long)m, worst);
      std::fflush(stderr);
    }
    // With reduced-precision transformations the residuals bottom out at the
    // transforms' rounding level: the solve also ends once the largest residual
    // has not improved by 10 % in 6 iterations (returned as -iterations).
    bool stalled = false;
    if (prec != Prec::F64) {
      double worst = 0.0;
      for (int64_t j = 0; j < s; ++j) worst = std::max(worst, norms[j]);
      if (worst < 0.9 * best) {
        best = worst;
        since_best = 0;
      } else {
        stalled = ++since_best >= 6;
      }
    }
    if (converged || stalled) {
      if (vectors) {
        for (int64_t j = 0; j < s; ++j) scale(stream_, Y + j * n, n, 1.0 / std::sqrt(ynorm[j]));
        host_copy_.to_host(stream_, vectors, Y, sizeof(double) * n * s);
        synchronize();
      }
      return converged ? it : -it;
    }
    // restart on the Ritz vectors when the space would overflow
    int64_t n_new = 0;
    for (int64_t j = 0; j < se; ++j) n_new += norms[j] >= threshold;
    if (k + n_new > max_dim) {
      // orthonormalise the Ritz vectors (and their transforms alike), then they
      // become the space: Cholesky QR twice (through V and AV, which are
      // replaced anyway), or one vector at a time in HBM
      if (se > 1 && cholqr(Y, AY, se, V, AV)) {
        run_gemm(make_gemm('T', 'N', se, se, n, 1.0, Y, n, AY, n, 0.0, G, max_dim), Prec::F64);
        ETG_HIP(hipMemcpyAsync(V, Y, sizeof(double) * n * se, hipMemcpyDefault, stream_));
        ETG_HIP(hipMemcpyAsync(AV, AY, sizeof(double) * n * se, hipMemcpyDefault, stream_));
        k = se;
      }
    }
    if (k + n_new > max_dim) {
      for (int64_t j = 0; j < se; ++j) {
        for (int pass = 0; pass < 2; ++pass)
          for (int64_t i = 0; i < j; ++i) {
            const double c = dot_host(Y + i * n, Y + j * n);
            axpy(stream_, n, -c, Y + i * n, Y + j * n);
            axpy(stream_, n, -c, AY + i * n, AY + j * n);
          }
        const double nv = std::sqrt(dot_host(Y + j * n, Y + j * n));
        scale(stream_, Y + j * n, n, 1.0 / nv);
        scale(stream_, AY + j * n, n, 1.0 / nv);
      }
      run_gemm(make_gemm('T', 'N', se, se, n, 1.0, Y, n, AY, n, 0.0, G, max_dim), Prec::F64);
      ETG_HIP(hipMemcpyAsync(V, Y, sizeof(double) * n * se, hipMemcpyDefault, stream_));
      ETG_HIP(hipMemcpyAsync(AV, AY, sizeof(double) * n * se, hipMemcpyDefault, stream_));
      k = se;
    }
    // preconditioned residuals of the unconverged roots, normalised, in the
    // first columns of the residual block
    NewColumns cols{};
    for (int64_t j = 0; j < se; ++j)
      if (norms[j] >= threshold) {
        cols.src[cols.n] = int(j);
        cols.w[cols.n++] = hcoef[j];
      }
    const int64_t nc = cols.n;
    if (nc > 0) {
      precondition_kernel<<<grid_for_d(n), kBlock, 0, stream_>>>(Rb, d, cols, n);
      ETG_LAUNCH("precondition");
      dots(stream_, Rb, n, Rb, n, n, nc, red_partial_.as<double>(), sums, 1);
      normalize_kernel<<<dim3(grid_for_d(n), unsigned(nc)), kBlock, 0, stream_>>>(Rb, sums, n);
      ETG_LAUNCH("normalize");
    }
    // orthogonalised against the space as one block (two passes: one read of V
    // per product however many vectors are new) ...
    if (k > 0 && nc > 0)
      for (int pass = 0; pass < 2; ++pass) {
        run_gemm(make_gemm('T', 'N', k, nc, n, 1.0, V, n, Rb, n, 0.0, cmat, max_dim), Prec::F64);
        run_gemm(make_gemm('N', 'N', n, nc, k, -1.0, V, n, cmat, max_dim, 1.0, Rb, n), Prec::F64);
      }
    // ... then against each other: Cholesky QR twice when no vector comes near
    // the span of the ones before it (through Y, free until the next Ritz
    // vectors), otherwise one vector at a time (two passes), dropping linearly
    // dependent ones
    m = 0;
    if (nc > 1 && cholqr(Rb, nullptr, nc, Y, nullptr)) m = nc;
    for (int64_t c = m; c < nc; ++c) {
      double* x = Rb + c * n;
      if (m > 0)
        for (int pass = 0; pass < 2; ++pass) {
          run_gemm(make_gemm('T', 'N', m, 1, n, 1.0, Rb, n, x, n, 0.0, cvec, max_dim), Prec::F64);
          run_gemm(make_gemm('N', 'N', n, 1, m, -1.0, Rb, n, cvec, max_dim, 1.0, x, n), Prec::F64);
        }
      const double nx = std::sqrt(dot_host(x, x));
      if (nx == 0.0 || nx < lindep) continue;
      scale(stream_, x, n, 1.0 / nx);
      if (c != m)
        ETG_HIP(hipMemcpyAsync(Rb + m * n, x, sizeof(double) * n, hipMemcpyDeviceToDevice, stream_));
      ++m;
    }
    if (m == 0) fail("davidson: no new trial vectors (linear dependence) before convergence");
    ETG_HIP(hipMemcpyAsync(V + k * n, Rb, sizeof(double) * n * m, hipMemcpyDefault, stream_));
  }
  fail("davidson: did not converge in the maximum number of iterations");
}

}  // namespace etg
