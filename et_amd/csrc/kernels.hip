// Bandwidth-bound kernels of the CCSD residual (see kernels.hpp).
#include "kernels.hpp"
#include "ladder_order.hpp"

#include <cmath>
#include <cstring>

namespace etg {
namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n, int64_t per_block = kBlock, int64_t cap = 1 << 20) {
  int64_t g = ceil_div(n, per_block);
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return unsigned(g);
}

// The same over the vectors of a batch (blockIdx.z).
inline dim3 grid_z(int64_t n, int64_t batch) { return dim3(grid_for(n), 1, unsigned(batch)); }

// Largest X with X (X + 1) / 2 <= k.
__device__ inline int64_t tri_root(int64_t k) {
  int64_t x = int64_t((sqrt(8.0 * double(k) + 1.0) - 1.0) * 0.5);
  while (x * (x + 1) / 2 > k) --x;
  while ((x + 1) * (x + 2) / 2 <= k) ++x;
  return x;
}

__device__ inline int64_t pidx(int64_t x, int64_t y) {
  const int64_t hi = x > y ? x : y, lo = x > y ? y : x;
  return hi * (hi + 1) / 2 + lo;
}

// I: index type (32-bit when the array has fewer than 2^32 elements: the
// element-wise divisions then cost a fraction of the 64-bit ones)
template <typename I>
__global__ void permute4_kernel(const double* __restrict__ x, double* __restrict__ y, I e0, I e1, I e2,
                                I e3, I s0, I s1, I s2, I s3, double alpha, double beta, int64_t sx, int64_t sy,
                                const double* z, double gamma, int64_t sz) {
  x += int64_t(blockIdx.z) * sx;
  y += int64_t(blockIdx.z) * sy;
  z += int64_t(blockIdx.z) * sz;
  const I n = e0 * e1 * e2 * e3;
  for (I idx = I(blockIdx.x) * blockDim.x + threadIdx.x; idx < n; idx += I(gridDim.x) * blockDim.x) {
    I r = idx;
    const I o0 = r % e0; r /= e0;
    const I o1 = r % e1; r /= e1;
    const I o2 = r % e2;
    const I o3 = r / e2;
    double v = alpha * x[o0 * s0 + o1 * s1 + o2 * s2 + o3 * s3];
    if (gamma != 0.0) v += gamma * z[idx];
    y[idx] = (beta == 0.0) ? v : v + beta * y[idx];
  }
}

// Permutation whose output-fastest index is not the input-fastest one: 32 x 32
// tiles of the (output dim 0, output dim p) plane go through LDS, where p is the
// output position of the input-fastest index, so reads (along dim p) and writes
// (along dim 0) are both unit-stride.  q, r: the other two output dims.
// Bound by HBM.  As in the other tiled kernels, the four loads of a lane come together and
// at clamped indices: each under its own edge condition waited for the one before (the four
// reorderings of the (H2O)8 residual 514 -> 443 us, squareup_and_u 161 -> 147, symsum_abij
// 172 -> 150; ladder_g_pm_tiled, which loops over pairs, loses by it: 1146 -> 1315).
__global__ void permute4_tiled_kernel(const double* __restrict__ x, double* __restrict__ y,
                                      int64_t e0, int64_t ep, int64_t eq, int64_t er, int64_t s0,
                                      int64_t sq, int64_t sr, int64_t yp, int64_t yq, int64_t yr,
                                      double alpha, double beta, int64_t bx, int64_t by, const double* z,
                                      double gamma, int64_t bz) {
  x += int64_t(blockIdx.z) * bx;
  y += int64_t(blockIdx.z) * by;
  z += int64_t(blockIdx.z) * bz;
  __shared__ double tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t nt0 = (e0 + 31) / 32;
  const int64_t t0 = blockIdx.x % nt0, tp = blockIdx.x / nt0;
  for (int64_t o = blockIdx.y; o < eq * er; o += gridDim.y) {
    const int64_t iq = o % eq, ir = o / eq;
    const double* xb = x + iq * sq + ir * sr;
    double* yb = y + iq * yq + ir * yr;
    double v[4], w[4] = {}, g[4] = {};
    const int64_t j0 = min(t0 * 32 + tx, e0 - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = xb[min(t0 * 32 + ty + 8 * k, e0 - 1) * s0 + min(tp * 32 + tx, ep - 1)];
    if (gamma != 0.0)
#pragma unroll
      for (int k = 0; k < 4; ++k) g[k] = z[yb - y + j0 + min(tp * 32 + ty + 8 * k, ep - 1) * yp];
    if (beta != 0.0)
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = yb[j0 + min(tp * 32 + ty + 8 * k, ep - 1) * yp];
#pragma unroll
    for (int k = 0; k < 4; ++k) tile[ty + 8 * k][tx] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t ip = tp * 32 + ty + 8 * k, i0 = t0 * 32 + tx;
      if (i0 < e0 && ip < ep) {
        double u = alpha * tile[tx][ty + 8 * k];
        if (gamma != 0.0) u += gamma * g[k];
        yb[i0 + ip * yp] = (beta == 0.0) ? u : u + beta * w[k];
      }
    }
    __syncthreads();
  }
}

__global__ void squareup_kernel(const double* __restrict__ packed, double* __restrict__ full,
                                int64_t N, int64_t sx, int64_t sy) {
  packed += int64_t(blockIdx.z) * sx;
  full += int64_t(blockIdx.z) * sy;
  const int64_t n = N * N;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < n;
       idx += int64_t(gridDim.x) * blockDim.x) {
    full[idx] = packed[pidx(idx % N, idx / N)];
  }
}

// The same through 32 x 32 LDS tiles: one workgroup per tile pair (Y block <=
// X block) reads packed elements (X, Y), Y <= X, along Y and writes full(Y, X)
// along Y and its mirror full(X, Y) along X.
__global__ __launch_bounds__(256) void squareup_tiled_kernel(const double* __restrict__ packed,
                                                             double* __restrict__ full, int64_t N, int64_t sx, int64_t sy) {
  packed += int64_t(blockIdx.z) * sx;
  full += int64_t(blockIdx.z) * sy;
  __shared__ double P[32][33];                          // P[xl][yl] = packed(X0 + xl, Y0 + yl)
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t xb = tri_root(blockIdx.x), yb = int64_t(blockIdx.x) - xb * (xb + 1) / 2;
  const int64_t X0 = xb * 32, Y0 = yb * 32;
  double p[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t X = min(X0 + ty + 8 * k, N - 1);
    p[k] = packed[X * (X + 1) / 2 + min(Y0 + tx, X)];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) P[ty + 8 * k][tx] = p[k];
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int64_t X = X0 + k, Y = Y0 + tx;              // full(Y, X), along Y
    if (X < N && Y <= X) full[Y + N * X] = P[k][tx];
    const int64_t Xr = X0 + tx, Yc = Y0 + k;            // full(Xr, Yc), along Xr
    if (Xr < N && Yc <= Xr) full[Xr + N * Yc] = P[tx][k];
  }
}

// packed element k = (X, Y), X >= Y, reads full(Y, X) (column X is contiguous in Y)
__global__ void packin_kernel(const double* __restrict__ full, double* __restrict__ packed,
                              int64_t N, double alpha, double beta, double diag_scale, int64_t sx, int64_t sy) {
  full += int64_t(blockIdx.z) * sx;
  packed += int64_t(blockIdx.z) * sy;
  const int64_t n = N * (N + 1) / 2;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t X = tri_root(k), Y = k - X * (X + 1) / 2;
    double v = alpha * full[Y + N * X];
    if (X == Y) v *= diag_scale;
    packed[k] = (beta == 0.0) ? v : v + beta * packed[k];
  }
}

// y = x + x^T through 32 x 32 LDS tiles
__global__ void symmetric_sum_kernel(const double* __restrict__ x, double* __restrict__ y,
                                     int64_t N, int64_t sx, int64_t sy) {
  x += int64_t(blockIdx.z) * sx;
  y += int64_t(blockIdx.z) * sy;
  __shared__ double tile[32][33];
  const int64_t bx = blockIdx.x, by = blockIdx.y;
  const int tx = threadIdx.x, ty = threadIdx.y;  // 32 x 8
  // load transposed block (by, bx) of x: rows by*32.., cols bx*32..
  double t[4], v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    t[k] = x[min(by * 32 + tx, N - 1) + N * min(bx * 32 + ty + 8 * k, N - 1)];
    v[k] = x[min(bx * 32 + tx, N - 1) + N * min(by * 32 + ty + 8 * k, N - 1)];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) tile[ty + 8 * k][tx] = t[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t r = bx * 32 + tx, c = by * 32 + ty + 8 * k;
    if (r < N && c < N) y[r + N * c] = v[k] + tile[tx][ty + 8 * k];
  }
}

// The same through 32 x 32 LDS tiles: one workgroup per tile pair (Y block <=
// X block) stages x(Y, X) (read along Y), x(X, Y) (along X) and, when f2 != 0,
// the two exchange terms x(p + v s, r + v q) (along p) and x(r + v q, p + v s)
// (along r) for Y = p + v q, X = r + v s, then adds to packed element
// X (X + 1) / 2 + Y, contiguous in Y for each X.  TWO: `plain` is a second array,
// added with alpha = f1 = 1, f2 = 0 (no batch).  All loads come first and at clamped
// indices: with each under its own edge condition they waited for one another, and the
// two-array form took 437 us instead of 186 at (H2O)8.
template <bool TWO>
__global__ __launch_bounds__(256) void symmetrize_and_pack_tiled_kernel(const double* __restrict__ x,
                                                                        double* __restrict__ y, int64_t n_v,
                                                                        int64_t N, double alpha, double f1,
                                                                        double f2, int64_t sx, int64_t sy,
                                                                        const double* __restrict__ plain) {
  x += int64_t(blockIdx.z) * sx;
  y += int64_t(blockIdx.z) * sy;
  __shared__ double E[TWO ? 32 : 1][33], F[TWO ? 32 : 1][33];   // of plain, as A and B
  __shared__ double A[32][33], B[32][33];              // A[xl][yl] = x(Y, X), B[yl][xl] = x(X, Y)
  __shared__ double C[32][33], D[32][33];              // C[xl][yl] = x(p + v s, r + v q), D[yl][xl] = mirror
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t xb = tri_root(blockIdx.x), yb = int64_t(blockIdx.x) - xb * (xb + 1) / 2;
  const int64_t X0 = xb * 32, Y0 = yb * 32;
  const bool exch = f2 != 0.0;
  // all loads first, none under a condition (rows past the edge repeat the last one): as
  // conditional loads each waits for the one before it
  double la[4], lb[4], lc[4], ld[4], le[4], lf[4], ly[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = ty + 8 * i;
    const int64_t Yr = min(Y0 + tx, N - 1), Xc = min(X0 + k, N - 1);    // A[k][tx] = x(Y0 + tx, X0 + k)
    la[i] = x[Yr + N * Xc];
    const int64_t Xr = min(X0 + tx, N - 1), Yc = min(Y0 + k, N - 1);    // B[k][tx] = x(X0 + tx, Y0 + k)
    lb[i] = x[Xr + N * Yc];
    if constexpr (TWO) {
      le[i] = plain[Yr + N * Xc];
      lf[i] = plain[Xr + N * Yc];
    }
    if (exch) {
      // C[k][tx]: Y = Yr = p + v q, X = Xc = r + v s  ->  x(p + v s, r + v q)
      const int64_t q = Yr / n_v, p = Yr - q * n_v, s = Xc / n_v, r = Xc - s * n_v;
      lc[i] = x[(p + n_v * s) + N * (r + n_v * q)];
      // D[k][tx]: X = Xr = r' + v s', Y = Yc = p' + v q'  ->  x(r' + v q', p' + v s')
      const int64_t q2 = Yc / n_v, p2 = Yc - q2 * n_v, s2 = Xr / n_v, r2 = Xr - s2 * n_v;
      ld[i] = x[(r2 + n_v * q2) + N * (p2 + n_v * s2)];
    }
    ly[i] = y[Xc * (Xc + 1) / 2 + min(Yr, Xc)];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = ty + 8 * i;
    A[k][tx] = la[i];
    B[k][tx] = lb[i];
    if constexpr (TWO) {
      E[k][tx] = le[i];
      F[k][tx] = lf[i];
    }
    if (exch) {
      C[k][tx] = lc[i];
      D[k][tx] = ld[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = ty + 8 * i;
    const int64_t X = X0 + k, Y = Y0 + tx;
    if (X >= N || Y > X) continue;
    double v;
    if (X == Y) {
      v = alpha * A[k][tx];
    } else {
      v = f1 * (A[k][tx] + B[tx][k]);
      if (exch) v += f2 * (C[k][tx] + D[tx][k]);
      v *= alpha;
    }
    if constexpr (TWO) v += X == Y ? E[k][tx] : E[k][tx] + F[tx][k];
    y[X * (X + 1) / 2 + Y] = ly[i] + v;
  }
}

__global__ void symmetrize_and_pack_kernel(const double* __restrict__ x, double* __restrict__ y,
                                           int64_t n_v, int64_t n_o, double alpha, double f1,
                                           double f2, int64_t sx, int64_t sy) {
  x += int64_t(blockIdx.z) * sx;
  y += int64_t(blockIdx.z) * sy;
  const int64_t N = n_v * n_o;
  const int64_t n = N * (N + 1) / 2;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t X = tri_root(k), Y = k - X * (X + 1) / 2;  // (r,s) = X, (p,q) = Y
    if (X == Y) {
      y[k] += alpha * x[Y + N * Y];
      continue;
    }
    const int64_t p = Y % n_v, q = Y / n_v, r = X % n_v, s = X / n_v;
    double v = f1 * (x[Y + N * X] + x[X + N * Y]);
    if (f2 != 0.0) v += f2 * (x[(p + n_v * s) + N * (r + n_v * q)] + x[(r + n_v * q) + N * (p + n_v * s)]);
    y[k] += alpha * v;
  }
}

// ---- steps of the direct residual taken together (the recorded program keeps them apart) ----

// full = t (N x N, symmetric) from packed storage, and u(ai, bj) = 2 t(ai, bj) - t(aj, bi).
// As squareup_tiled, with the exchange terms of the tile read along X: for i >= j they lie
// contiguously in a.
__global__ __launch_bounds__(256) void squareup_and_u_kernel(const double* __restrict__ packed, double* __restrict__ full,
                                                             double* __restrict__ u, int64_t n_v, int64_t N) {
  __shared__ double P[32][33], Q[32][33];               // P[xl][yl] = t(X, Y), Q[yl][xl] = t(aj, bi)
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t xb = tri_root(blockIdx.x), yb = int64_t(blockIdx.x) - xb * (xb + 1) / 2;
  const int64_t X0 = xb * 32, Y0 = yb * 32;
  double p[4], q[4];
  const int64_t Xr = min(X0 + tx, N - 1);               // a + v i
  const int64_t i = Xr / n_v, a = Xr - i * n_v;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t X = min(X0 + ty + 8 * k, N - 1);
    p[k] = packed[X * (X + 1) / 2 + min(Y0 + tx, X)];
    const int64_t Yc = min(Y0 + ty + 8 * k, N - 1);     // b + v j
    const int64_t j = Yc / n_v, b = Yc - j * n_v;
    q[k] = packed[pidx(a + n_v * j, b + n_v * i)];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    P[ty + 8 * k][tx] = p[k];
    Q[ty + 8 * k][tx] = q[k];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int64_t X = X0 + k, Y = Y0 + tx;              // (Y, X), along Y
    if (X < N && Y <= X) {
      full[Y + N * X] = P[k][tx];
      u[Y + N * X] = 2.0 * P[k][tx] - Q[tx][k];
    }
    const int64_t Xr = X0 + tx, Yc = Y0 + k;            // (Xr, Yc), along Xr
    if (Xr < N && Yc <= Xr) {
      full[Xr + N * Yc] = P[tx][k];
      u[Xr + N * Yc] = 2.0 * P[tx][k] - Q[k][tx];
    }
  }
}

// y(a, b, i, j) = x(ai, bj) + x(bj, ai): one 32 x 32 tile of (a, b) for one (i, j) per workgroup.
__global__ __launch_bounds__(256) void symsum_abij_kernel(const double* __restrict__ x, double* __restrict__ y,
                                                          int64_t n_v, int64_t n_o) {
  __shared__ double T[32][33];                          // T[a][b] = x(bj, ai)
  const int64_t N = n_v * n_o, nt = (n_v + 31) / 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t a0 = (blockIdx.x % nt) * 32, b0 = (blockIdx.x / nt) * 32;
  for (int64_t ij = blockIdx.y; ij < n_o * n_o; ij += gridDim.y) {
    const int64_t i = ij % n_o, j = ij / n_o;
    double t[4], v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      t[k] = x[(min(b0 + tx, n_v - 1) + n_v * j) + N * (min(a0 + ty + 8 * k, n_v - 1) + n_v * i)];
      v[k] = x[(min(a0 + tx, n_v - 1) + n_v * i) + N * (min(b0 + ty + 8 * k, n_v - 1) + n_v * j)];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) T[ty + 8 * k][tx] = t[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t a = a0 + tx, b = b0 + ty + 8 * k;
      if (a < n_v && b < n_v) y[a + n_v * b + n_v * n_v * ij] = v[k] + T[tx][ty + 8 * k];
    }
    __syncthreads();
  }
}

// F(p, q) += 2 sum_J L(J, p, q) x(J): a wavefront per element, which reads its J numbers in
// a row.  Bound by HBM (L once).  One launch for what four products of one column each
// did: residual of H2O 366 -> 350 us; the 750 MB of (H2O)8 in 186 us.
__global__ __launch_bounds__(256) void fock_coulomb_kernel(const double* __restrict__ Loo, const double* __restrict__ Lov,
                                                           const double* __restrict__ Lvo, const double* __restrict__ Lvv,
                                                           const double* __restrict__ x, int64_t J, int64_t n_o,
                                                           int64_t n_v, double* __restrict__ F) {
  const int64_t n = n_o + n_v;
  const int lane = threadIdx.x & 63;
  for (int64_t w = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6); w < n * n; w += int64_t(gridDim.x) * 4) {
    const int64_t q = w / n, p = w - q * n;
    const double* L = p < n_o ? (q < n_o ? Loo + J * (p + n_o * q) : Lov + J * (p + n_o * (q - n_o)))
                              : (q < n_o ? Lvo + J * (p - n_o + n_v * q) : Lvv + J * (p - n_o + n_v * (q - n_o)));
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t j = lane; j < J; j += 256)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j + 64 * u < J) s[u] += L[j + 64 * u] * x[j + 64 * u];
    double v = (s[0] + s[1]) + (s[2] + s[3]);
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) F[p + n * q] += 2.0 * v;
  }
}

// packin of the (a, i, b, j) order of x(a, b, i, j): packed element X = (a, i) >= Y = (b, j)
// is x(b, a, j, i), contiguous in b, times diag_scale where X = Y.
__global__ void packin_abij_kernel(const double* __restrict__ x, double* __restrict__ packed, int64_t n_v, int64_t n_o,
                                   double diag_scale) {
  const int64_t N = n_v * n_o, n = N * (N + 1) / 2;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n; k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t X = tri_root(k), Y = k - X * (X + 1) / 2;
    const int64_t i = X / n_v, a = X - i * n_v, j = Y / n_v, b = Y - j * n_v;
    const double v = x[b + n_v * a + n_v * n_v * (j + n_o * i)];
    packed[k] = X == Y ? diag_scale * v : v;
  }
}

__global__ void ladder_t_pm_kernel(const double* __restrict__ t2, double* __restrict__ tp,
                                   double* __restrict__ tm, int64_t n_o, int64_t n_v, int64_t st, int64_t sp, int64_t sm) {
  t2 += int64_t(blockIdx.z) * st;
  tp += int64_t(blockIdx.z) * sp;
  tm += int64_t(blockIdx.z) * sm;
  const int64_t op = n_o * (n_o + 1) / 2, vp = n_v * (n_v + 1) / 2;
  const int64_t om = n_o * (n_o - 1) / 2, vm = n_v * (n_v - 1) / 2;
  const int64_t n = op * vp;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < n;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const int64_t rij = idx % op, rcd = idx / op;
    const int64_t j = tri_root(rij), i = rij - j * (j + 1) / 2;
    const int64_t d = tri_root(rcd), c = rcd - d * (d + 1) / 2;
    const double x1 = t2[pidx(c + n_v * i, d + n_v * j)];
    const double x2 = t2[pidx(c + n_v * j, d + n_v * i)];
    tp[idx] = (c == d ? 0.5 : 1.0) * (x1 + x2);
    if (i < j && c < d) {
      const int64_t mij = j * (j - 1) / 2 + i, mcd = d * (d - 1) / 2 + c;
      tm[mij + om * mcd] = x1 - x2;
    }
  }
  (void)vm;
}

// t+ (op x KP) and t- (om x KM) with the contraction index in the tile-blocked
// order of ladder_order.hpp (zero at padding positions).
__global__ void ladder_t_pm_blocked_kernel(const double* __restrict__ t2, double* __restrict__ tp,
                                           double* __restrict__ tm, int64_t n_o, int64_t n_v, int64_t KP,
                                           int64_t KM, int64_t st, int64_t sp, int64_t sm) {
  t2 += int64_t(blockIdx.z) * st;
  tp += int64_t(blockIdx.z) * sp;
  tm += int64_t(blockIdx.z) * sm;
  const int64_t op = n_o * (n_o + 1) / 2, om = n_o * (n_o - 1) / 2;
  const int64_t np = op * KP, n = np + om * KM;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < n;
       idx += int64_t(gridDim.x) * blockDim.x) {
    const bool plus = idx < np;
    const int64_t q = plus ? idx : idx - np;
    const int64_t nij = plus ? op : om;
    const int64_t rij = q % nij, kk = q / nij;
    // plus: i <= j at j (j + 1) / 2 + i; minus: i < j at j (j - 1) / 2 + i
    const int64_t j = plus ? tri_root(rij) : tri_root(rij) + 1;
    const int64_t i = rij - (plus ? j * (j + 1) / 2 : j * (j - 1) / 2);
    int64_t c = 0, d = 0;
    double val = 0.0;
    if (ladder_pair_of(kk, n_v, plus, c, d)) {
      const double x1 = t2[pidx(c + n_v * i, d + n_v * j)];
      const double x2 = t2[pidx(c + n_v * j, d + n_v * i)];
      val = plus ? (c == d ? 0.5 : 1.0) * (x1 + x2) : x1 - x2;
    }
    (plus ? tp : tm)[q] = val;
  }
}

// g+ (v(v+1)/2 x npairs) and g- (v(v-1)/2 x npairs) of a G block.  For pair k = (a, b) the v x v block
// M(c, d) = G(c + v a, d + v b) gives g+_cd = M(c,d) + M(d,c) (c <= d) and
// g-_cd = M(c,d) - M(d,c) (c < d); one workgroup per tile pair (ti <= tj) reads
// the tiles M(ti, tj) and M(tj, ti) unit-stride into LDS.
__global__ void ladder_g_pm_tiled_kernel(const double* __restrict__ G, int64_t n_v, int64_t lenA,
                                         const int32_t* __restrict__ pa, const int32_t* __restrict__ pb,
                                         int64_t npairs, double* __restrict__ gp, double* __restrict__ gm) {
  __shared__ double A[32][33], B[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t vp = n_v * (n_v + 1) / 2, vm = n_v * (n_v - 1) / 2;
  const int64_t ldG = n_v * lenA;
  const int64_t tj = tri_root(blockIdx.x), ti = int64_t(blockIdx.x) - tj * (tj + 1) / 2;
  const int64_t c0 = ti * 32, d0 = tj * 32;
  for (int64_t k = blockIdx.y; k < npairs; k += gridDim.y) {
    const int64_t a = pa[k], b = pb[k];
    const double* M = G + n_v * a + ldG * n_v * b;           // M(c, d) = M[c + ldG d]
    for (int q = ty; q < 32; q += 8) {
      const int64_t c = c0 + tx, d = d0 + q;                 // A[tx][q] = M(c0+tx, d0+q)
      A[tx][q] = (c < n_v && d < n_v) ? M[c + ldG * d] : 0.0;
      const int64_t c2 = d0 + tx, d2 = c0 + q;               // B[tx][q] = M(d0+tx, c0+q)
      B[tx][q] = (c2 < n_v && d2 < n_v) ? M[c2 + ldG * d2] : 0.0;
    }
    __syncthreads();
    for (int q = ty; q < 32; q += 8) {
      const int64_t c = c0 + tx, d = d0 + q;
      if (c <= d && d < n_v) {
        const double x1 = A[tx][q], x2 = B[q][tx];           // M(c, d), M(d, c)
        gp[(d * (d + 1) / 2 + c) + vp * k] = x1 + x2;
        if (c < d) gm[(d * (d - 1) / 2 + c) + vm * k] = x1 - x2;
      }
    }
    __syncthreads();
  }
}

__global__ void ladder_gather_kernel(const double* __restrict__ wp, const double* __restrict__ wm,
                                     const int32_t* __restrict__ col, double* __restrict__ om,
                                     int64_t n_o, int64_t n_v, int64_t so, int64_t sp, int64_t sm) {
  wp += int64_t(blockIdx.z) * sp;
  wm += int64_t(blockIdx.z) * sm;
  om += int64_t(blockIdx.z) * so;
  const int64_t N = n_o * n_v;
  const int64_t n = N * (N + 1) / 2;
  const int64_t op = n_o * (n_o + 1) / 2, omn = n_o * (n_o - 1) / 2;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t X = tri_root(k), Y = k - X * (X + 1) / 2;  // X = ai, Y = bj
    const int64_t a = X % n_v, i = X / n_v, b = Y % n_v, j = Y / n_v;
    const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    const int64_t cl = col[a + n_v * b];
    double w = wp[(hi * (hi + 1) / 2 + lo) + op * cl];
    if (i != j && a != b) {
      const double sgn = ((i < j) == (a > b)) ? 1.0 : -1.0;
      w += sgn * wm[(hi * (hi - 1) / 2 + lo) + omn * cl];
    }
    om[k] += (X == Y) ? 0.5 * w : w;
  }
}

__device__ inline double block_sum(double v) {
  __shared__ double red[kBlock / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int q = 0; q < kBlock / 64; ++q) s += red[q];
  return s;  // valid in thread 0
}

// sum over X = (a, i) >= Y = (b, j), the other half of the terms being equal.  t is
// contiguous along b, g_iajb and g_ibja along j: 32 x 32 tiles of 2 g_iajb - g_ibja go
// through LDS.  Bound by HBM (24 bytes per pair): (H2O)8 1.17 -> 0.14 ms, o = 40, v = 360
// 8.4 -> 0.8, read element by element along a before.
__global__ __launch_bounds__(256) void energy_kernel(const double* __restrict__ t1, const double* __restrict__ t2,
                                                     const double* __restrict__ g, int64_t n_o, int64_t n_v,
                                                     double* __restrict__ partial) {
  __shared__ double D[32][33];                          // [b][j]
  const int64_t N = n_o * n_v, chunks = (n_v + 31) / 32;
  double acc = 0.0;
  for (int64_t item = blockIdx.x; item < N * chunks; item += gridDim.x) {
    const int64_t X = item / chunks, b0 = (item - X * chunks) * 32;
    const int64_t i = X / n_v, a = X - i * n_v;
    const int nb = int(min(int64_t(32), n_v - b0));
    for (int64_t j0 = 0; j0 <= i; j0 += 32) {
      const int nj = int(min(int64_t(32), i - j0 + 1));
      const double* g1 = g + j0 + n_o * b0 + N * (i + n_o * a);
      const double* g2 = g + j0 + n_o * a + N * (i + n_o * b0);
      for (int q = threadIdx.x; q < nj * nb; q += kBlock) {
        const int b = q / nj, j = q - b * nj;
        D[b][j] = 2.0 * g1[j + n_o * b] - g2[j + N * n_o * b];
      }
      __syncthreads();
      const int b = threadIdx.x & 31;
      const int64_t Y0 = b0 + b + n_v * j0;
      if (b < nb)
        for (int j = threadIdx.x >> 5; j < nj; j += kBlock / 32) {
          const int64_t Y = Y0 + n_v * j;
          if (Y <= X) acc += (Y < X ? 2.0 : 1.0) * (t2[X * (X + 1) / 2 + Y] + t1[X] * t1[Y]) * D[b][j];
        }
      __syncthreads();
    }
  }
  const double s = block_sum(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void sumsq_kernel(const double* __restrict__ x, const double* __restrict__ y, int64_t n,
                             double* __restrict__ partial) {
  double acc = 0.0;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < n;
       idx += int64_t(gridDim.x) * blockDim.x)
    acc += x[idx] * (y ? y[idx] : x[idx]);
  const double s = block_sum(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void finish_sum_kernel(const double* __restrict__ partial, int n, double* result) {
  double acc = 0.0;
  for (int q = threadIdx.x; q < n; q += blockDim.x) acc += partial[q];
  const double s = block_sum(acc);
  if (threadIdx.x == 0) *result = s;
}

// The same sums for several pairs: pair q = blockIdx.y of (x + q sx, y + q sy).  A
// solver's handful of dot products costs two launches (and its caller one copy to
// the host) instead of two launches, a copy and a wait each: 20-40 us apiece.
__global__ void dots_kernel(const double* __restrict__ x, int64_t sx, const double* __restrict__ y, int64_t sy,
                            int64_t n, double* __restrict__ partial) {
  x += blockIdx.y * sx;
  y += blockIdx.y * sy;
  double acc = 0.0;
  for (int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < n;
       idx += int64_t(gridDim.x) * blockDim.x)
    acc += x[idx] * y[idx];
  const double s = block_sum(acc);
  if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = s;
}

__global__ void finish_sums_kernel(const double* __restrict__ partial, int n, double* result, int64_t sr) {
  double acc = 0.0;
  for (int q = threadIdx.x; q < n; q += blockDim.x) acc += partial[int64_t(blockIdx.x) * n + q];
  const double s = block_sum(acc);
  if (threadIdx.x == 0) result[blockIdx.x * sr] = s;
}

__global__ void mp2_guess_kernel(const double* __restrict__ g, const double* __restrict__ eps,
                                 double* __restrict__ t2, int64_t n_o, int64_t n_v) {
  const int64_t N = n_o * n_v;
  const int64_t n = N * (N + 1) / 2;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t X = tri_root(k), Y = k - X * (X + 1) / 2;
    const int64_t a = X % n_v, i = X / n_v, b = Y % n_v, j = Y / n_v;
    const double d = eps[i] - eps[n_o + a] + eps[j] - eps[n_o + b];
    t2[k] = g[X + N * Y] / d;
  }
}

// Core projections; core[i] != 0 marks core occupied MOs; blockIdx.y is the vector.
// remove_core = 0, core-valence separation (cvs_projection_ccs, ccs_class.F90:1219-1250,
// cvs_projection_doubles, doubles_class.F90:287-328): zero every singles element whose
// occupied index is not a core MO and every packed doubles element (ai, bj) with neither
// i nor j a core MO.  remove_core = 1 (rm_core_projection_ccs, ccs_class.F90:1251-1280,
// rm_core_projection_doubles, doubles_class.F90:330-370): zero exactly the others.
// mode 2, ionisation (ip_projection_ccs, ccs_class.F90:1611-1640, ip_projection_doubles,
// doubles_class.F90:376-418): keep only singles into the last virtual (the bath orbital)
// and doubles with a or b the bath orbital; core is not read.
__global__ void cvs_project_kernel(double* __restrict__ x, int64_t n_t1, int64_t n, int64_t n_v,
                                   const unsigned char* __restrict__ core, int mode) {
  double* xv = x + int64_t(blockIdx.y) * n;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x) {
    bool hit;                                // an occupied core index (modes 0, 1) or the bath (2)
    if (k < n_t1) {
      hit = mode == 2 ? k % n_v == n_v - 1 : core[k / n_v] != 0;
    } else {
      const int64_t q = k - n_t1;
      const int64_t X = tri_root(q), Y = q - X * (X + 1) / 2;
      hit = mode == 2 ? (X % n_v == n_v - 1 || Y % n_v == n_v - 1) : (core[X / n_v] != 0 || core[Y / n_v] != 0);
    }
    if (hit == (mode == 1)) xv[k] = 0.0;
  }
}

__global__ void orbital_differences_kernel(const double* __restrict__ eps, double* __restrict__ x,
                                           int64_t n_o, int64_t n_v, int64_t n) {
  const int64_t N = n_o * n_v;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x) {
    if (k < N) {
      x[k] = eps[n_o + k % n_v] - eps[k / n_v];
    } else {
      const int64_t q = k - N;
      const int64_t X = tri_root(q), Y = q - X * (X + 1) / 2;
      x[k] = eps[n_o + X % n_v] - eps[X / n_v] + eps[n_o + Y % n_v] - eps[Y / n_v];
    }
  }
}

__global__ void axpy_kernel(int64_t n, double alpha, const double* __restrict__ x,
                            double* __restrict__ y) {
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x)
    y[k] += alpha * x[k];
}

__global__ void fill_kernel(double* __restrict__ x, int64_t n, double value) {
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < n;
       k += int64_t(gridDim.x) * blockDim.x)
    x[k] = value;
}

}  // namespace

void permute4(hipStream_t s, const double* x, double* y, const int64_t e[4], const int64_t st[4],
              double alpha, double beta, const Batch& b, const double* z, double gamma) {
  const int64_t n = e[0] * e[1] * e[2] * e[3];
  if (n == 0) return;
  if (z == nullptr) {
    z = y;                                      // not read
    gamma = 0.0;
  }
  int p = -1;                                   // output position of the input-fastest index
  for (int k = 0; k < 4; ++k)
    if (st[k] == 1 && e[k] > 1) p = k;
  if (p > 0 && e[0] >= 8 && e[p] >= 8) {
    int oth[2], no = 0;
    for (int k = 1; k < 4; ++k)
      if (k != p) oth[no++] = k;
    const int64_t ostride[4] = {1, e[0], e[0] * e[1], e[0] * e[1] * e[2]};
    const int64_t tiles = ceil_div(e[0], 32) * ceil_div(e[p], 32);
    const int64_t others = e[oth[0]] * e[oth[1]];
    dim3 grid(unsigned(tiles), unsigned(std::min<int64_t>(others, 65535)), unsigned(b.n));
    permute4_tiled_kernel<<<grid, kBlock, 0, s>>>(x, y, e[0], e[p], e[oth[0]], e[oth[1]], st[0],
                                                  st[oth[0]], st[oth[1]], ostride[p], ostride[oth[0]],
                                                  ostride[oth[1]], alpha, beta, b.x, b.y, z, gamma, b.z);
    ETG_LAUNCH("permute4_tiled");
    return;
  }
  // (32-bit indices: the grid-stride step stays below 2^32 - n as well)
  if (n + int64_t(kBlock) * grid_for(n) <= int64_t(UINT32_MAX))
    permute4_kernel<uint32_t><<<grid_z(n, b.n), kBlock, 0, s>>>(
        x, y, uint32_t(e[0]), uint32_t(e[1]), uint32_t(e[2]), uint32_t(e[3]), uint32_t(st[0]), uint32_t(st[1]),
        uint32_t(st[2]), uint32_t(st[3]), alpha, beta, b.x, b.y, z, gamma, b.z);
  else
    permute4_kernel<int64_t><<<grid_z(n, b.n), kBlock, 0, s>>>(x, y, e[0], e[1], e[2], e[3], st[0], st[1], st[2],
                                                               st[3], alpha, beta, b.x, b.y, z, gamma, b.z);
  ETG_LAUNCH("permute4");
}

void sort4(hipStream_t s, const double* x, const int64_t d[4], const char* perm, double* y,
           double alpha, double beta, const Batch& b, const double* z, double gamma) {
  if (std::strlen(perm) != 4) fail("sort4: permutation must have 4 digits");
  const int64_t in_stride[4] = {1, d[0], d[0] * d[1], d[0] * d[1] * d[2]};
  int64_t e[4], st[4];
  int seen = 0;
  for (int k = 0; k < 4; ++k) {
    const int q = perm[k] - '1';
    if (q < 0 || q > 3 || (seen & (1 << q))) fail(std::string("sort4: bad permutation ") + perm);
    seen |= 1 << q;
    e[k] = d[q];
    st[k] = in_stride[q];
  }
  permute4(s, x, y, e, st, alpha, beta, b, z, gamma);
}

void squareup(hipStream_t s, const double* packed, double* full, int64_t N, const Batch& b) {
  if (N >= 32) {
    const int64_t nb = ceil_div(N, 32);
    squareup_tiled_kernel<<<dim3(unsigned(nb * (nb + 1) / 2), 1, unsigned(b.n)), kBlock, 0, s>>>(packed, full, N, b.x, b.y);
    ETG_LAUNCH("squareup_tiled");
    return;
  }
  squareup_kernel<<<grid_z(N * N, b.n), kBlock, 0, s>>>(packed, full, N, b.x, b.y);
  ETG_LAUNCH("squareup");
}

void packin(hipStream_t s, const double* full, double* packed, int64_t N, double alpha, double beta,
            double diag_scale, const Batch& b) {
  packin_kernel<<<grid_z(N * (N + 1) / 2, b.n), kBlock, 0, s>>>(full, packed, N, alpha, beta, diag_scale, b.x, b.y);
  ETG_LAUNCH("packin");
}

void symmetric_sum(hipStream_t s, const double* x, double* y, int64_t N, const Batch& b) {
  if (x == y) fail("symmetric_sum: out of place only");
  dim3 grid(unsigned(ceil_div(N, 32)), unsigned(ceil_div(N, 32)), unsigned(b.n));
  symmetric_sum_kernel<<<grid, dim3(32, 8), 0, s>>>(x, y, N, b.x, b.y);
  ETG_LAUNCH("symmetric_sum");
}

void symmetrize_and_pack(hipStream_t s, const double* x, double* packed, int64_t n_v, int64_t n_o,
                         double alpha, double f1, double f2, const Batch& b) {
  const int64_t N = n_v * n_o;
  if (N >= 32) {
    const int64_t nb = ceil_div(N, 32);
    symmetrize_and_pack_tiled_kernel<false><<<dim3(unsigned(nb * (nb + 1) / 2), 1, unsigned(b.n)), kBlock, 0, s>>>(
        x, packed, n_v, N, alpha, f1, f2, b.x, b.y, nullptr);
    ETG_LAUNCH("symmetrize_and_pack_tiled");
    return;
  }
  symmetrize_and_pack_kernel<<<grid_z(N * (N + 1) / 2, b.n), kBlock, 0, s>>>(x, packed, n_v, n_o, alpha, f1, f2, b.x,
                                                                             b.y);
  ETG_LAUNCH("symmetrize_and_pack");
}

void symmetrize_and_pack_two(hipStream_t s, const double* x, const double* plain, double* packed, int64_t n_v,
                             int64_t n_o, double alpha, double f1, double f2) {
  const int64_t N = n_v * n_o, nb = ceil_div(N, 32);
  symmetrize_and_pack_tiled_kernel<true><<<unsigned(nb * (nb + 1) / 2), kBlock, 0, s>>>(x, packed, n_v, N, alpha, f1, f2, 0, 0,
                                                                                  plain);
  ETG_LAUNCH("symmetrize_and_pack_two");
}

void squareup_and_u(hipStream_t s, const double* packed, double* full, double* u, int64_t n_v, int64_t n_o) {
  const int64_t N = n_v * n_o, nb = ceil_div(N, 32);
  squareup_and_u_kernel<<<unsigned(nb * (nb + 1) / 2), kBlock, 0, s>>>(packed, full, u, n_v, N);
  ETG_LAUNCH("squareup_and_u");
}

void symsum_abij(hipStream_t s, const double* x, double* y, int64_t n_v, int64_t n_o) {
  const int64_t nt = ceil_div(n_v, 32);
  symsum_abij_kernel<<<dim3(unsigned(nt * nt), unsigned(std::min<int64_t>(n_o * n_o, 65535))), kBlock, 0, s>>>(x, y, n_v, n_o);
  ETG_LAUNCH("symsum_abij");
}

void fock_coulomb(hipStream_t s, const double* Loo, const double* Lov, const double* Lvo, const double* Lvv,
                  const double* x, int64_t n_J, int64_t n_o, int64_t n_v, double* F) {
  const int64_t n = n_o + n_v;
  fock_coulomb_kernel<<<unsigned(std::min<int64_t>(ceil_div(n * n, 4), 1 << 16)), kBlock, 0, s>>>(Loo, Lov, Lvo, Lvv, x, n_J,
                                                                                                  n_o, n_v, F);
  ETG_LAUNCH("fock_coulomb");
}

void packin_abij(hipStream_t s, const double* x, double* packed, int64_t n_v, int64_t n_o, double diag_scale) {
  const int64_t N = n_v * n_o;
  packin_abij_kernel<<<grid_for(N * (N + 1) / 2), kBlock, 0, s>>>(x, packed, n_v, n_o, diag_scale);
  ETG_LAUNCH("packin_abij");
}

void ladder_t_pm(hipStream_t s, const double* t2, double* tp, double* tm, int64_t n_o, int64_t n_v,
                 const LadderBatch& b) {
  const int64_t n = (n_o * (n_o + 1) / 2) * (n_v * (n_v + 1) / 2);
  ladder_t_pm_kernel<<<grid_z(n, b.n), kBlock, 0, s>>>(t2, tp, tm, n_o, n_v, b.vec, b.plus, b.minus);
  ETG_LAUNCH("ladder_t_pm");
}

void ladder_t_pm_blocked(hipStream_t s, const double* t2, double* tp, double* tm, int64_t n_o,
                         int64_t n_v, const LadderBatch& b) {
  const int64_t KP = ladder_blocked_len(n_v, true), KM = ladder_blocked_len(n_v, false);
  const int64_t n = (n_o * (n_o + 1) / 2) * KP + (n_o * (n_o - 1) / 2) * KM;
  ladder_t_pm_blocked_kernel<<<grid_z(n, b.n), kBlock, 0, s>>>(t2, tp, tm, n_o, n_v, KP, KM, b.vec, b.plus, b.minus);
  ETG_LAUNCH("ladder_t_pm_blocked");
}

void ladder_g_pm(hipStream_t s, const double* G, int64_t n_v, int64_t lenA, int64_t lenB,
                 const int32_t* pair_a, const int32_t* pair_b, int64_t npairs, double* gp, double* gm) {
  const int64_t n = (n_v * (n_v + 1) / 2) * npairs;
  if (n == 0) return;
  (void)lenB;
  const int64_t nt = (n_v + 31) / 32;
  dim3 grid(unsigned(nt * (nt + 1) / 2), unsigned(std::min<int64_t>(npairs, 65535)));
  ladder_g_pm_tiled_kernel<<<grid, kBlock, 0, s>>>(G, n_v, lenA, pair_a, pair_b, npairs, gp, gm);
  ETG_LAUNCH("ladder_g_pm");
}

void ladder_gather(hipStream_t s, const double* wp, const double* wm, const int32_t* col,
                   double* omega2, int64_t n_o, int64_t n_v, const LadderBatch& b) {
  const int64_t N = n_o * n_v;
  ladder_gather_kernel<<<grid_z(N * (N + 1) / 2, b.n), kBlock, 0, s>>>(wp, wm, col, omega2, n_o, n_v, b.vec, b.plus,
                                                                       b.minus);
  ETG_LAUNCH("ladder_gather");
}

void ccsd_energy(hipStream_t s, const double* t1, const double* t2, const double* g_ovov,
                 int64_t n_o, int64_t n_v, double* partial, double* result) {
  energy_kernel<<<kReduceBlocks, kBlock, 0, s>>>(t1, t2, g_ovov, n_o, n_v, partial);
  ETG_LAUNCH("energy");
  finish_sum_kernel<<<1, kBlock, 0, s>>>(partial, kReduceBlocks, result);
  ETG_LAUNCH("finish_sum");
}

void sum_squares(hipStream_t s, const double* x, int64_t n, double* partial, double* result) {
  sumsq_kernel<<<kReduceBlocks, kBlock, 0, s>>>(x, nullptr, n, partial);
  ETG_LAUNCH("sum_squares");
  finish_sum_kernel<<<1, kBlock, 0, s>>>(partial, kReduceBlocks, result);
  ETG_LAUNCH("finish_sum");
}

void dot(hipStream_t s, const double* x, const double* y, int64_t n, double* partial, double* result) {
  sumsq_kernel<<<kReduceBlocks, kBlock, 0, s>>>(x, y, n, partial);
  ETG_LAUNCH("dot");
  finish_sum_kernel<<<1, kBlock, 0, s>>>(partial, kReduceBlocks, result);
  ETG_LAUNCH("finish_sum");
}

void dots(hipStream_t s, const double* x, int64_t sx, const double* y, int64_t sy, int64_t n, int64_t count,
          double* partial, double* result, int64_t sr) {
  for (int64_t c = 0; c < count; c += kDotBatch) {
    const unsigned m = unsigned(std::min<int64_t>(count - c, kDotBatch));
    dots_kernel<<<dim3(kReduceBlocks, m), kBlock, 0, s>>>(x + c * sx, sx, y + c * sy, sy, n, partial);
    ETG_LAUNCH("dots");
    finish_sums_kernel<<<m, kBlock, 0, s>>>(partial, kReduceBlocks, result + c * sr, sr);
    ETG_LAUNCH("finish_sums");
  }
}

void mp2_guess(hipStream_t s, const double* g_vovo, const double* eps, double* t2, int64_t n_o,
               int64_t n_v) {
  const int64_t N = n_o * n_v;
  mp2_guess_kernel<<<grid_for(N * (N + 1) / 2), kBlock, 0, s>>>(g_vovo, eps, t2, n_o, n_v);
  ETG_LAUNCH("mp2_guess");
}

void orbital_differences(hipStream_t s, const double* eps, double* x, int64_t n_o, int64_t n_v,
                         int64_t n) {
  orbital_differences_kernel<<<grid_for(n), kBlock, 0, s>>>(eps, x, n_o, n_v, n);
  ETG_LAUNCH("orbital_differences");
}

void cvs_project(hipStream_t s, double* x, int64_t n_vec, int64_t n_t1, int64_t n, int64_t n_v,
                 const unsigned char* core, int mode) {
  for (int64_t v0 = 0; v0 < n_vec; v0 += 65535) {
    const dim3 g(grid_for(n, kBlock, 1 << 14), unsigned(std::min<int64_t>(n_vec - v0, 65535)));
    cvs_project_kernel<<<g, kBlock, 0, s>>>(x + v0 * n, n_t1, n, n_v, core, mode);
    ETG_LAUNCH("cvs_project");
  }
}

void axpy(hipStream_t s, int64_t n, double alpha, const double* x, double* y) {
  if (n == 0) return;
  axpy_kernel<<<grid_for(n), kBlock, 0, s>>>(n, alpha, x, y);
  ETG_LAUNCH("axpy");
}

void fill(hipStream_t s, double* x, int64_t n, double value) {
  if (n == 0) return;
  fill_kernel<<<grid_for(n), kBlock, 0, s>>>(x, n, value);
  ETG_LAUNCH("fill");
}

}  // namespace etg

// ===========================================================================
// Adjoint kernels and T1 helpers
// ===========================================================================
namespace etg {
namespace {

__device__ inline int64_t tri_root2(int64_t k) {
  int64_t x = int64_t((sqrt(8.0 * double(k) + 1.0) - 1.0) * 0.5);
  while (x * (x + 1) / 2 > k) --x;
  while ((x + 1) * (x + 2) / 2 <= k) ++x;
  return x;
}

__device__ inline int64_t pidx2(int64_t x, int64_t y) {
  const int64_t hi = x > y ? x : y, lo = x > y ? y : x;
  return hi * (hi + 1) / 2 + lo;
}

#define GRID_LOOP(var, n)                                                      \
  for (int64_t var = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; var < (n); \
       var += int64_t(gridDim.x) * blockDim.x)

__global__ void scale_kernel(double* x, int64_t n, double beta) {
  GRID_LOOP(k, n) x[k] = (beta == 0.0) ? 0.0 : beta * x[k];
}

__global__ void symmetric_sum_acc_kernel(const double* __restrict__ x, double* __restrict__ y,
                                         int64_t N, double beta, int64_t sx, int64_t sy) {
  x += int64_t(blockIdx.z) * sx;
  y += int64_t(blockIdx.z) * sy;
  __shared__ double tile[32][33];
  const int64_t bx = blockIdx.x, by = blockIdx.y;
  const int tx = threadIdx.x, ty = threadIdx.y;
  double t[4], v[4], w[4] = {};
  const int64_t rc = min(bx * 32 + tx, N - 1);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    t[k] = x[min(by * 32 + tx, N - 1) + N * min(bx * 32 + ty + 8 * k, N - 1)];
    v[k] = x[rc + N * min(by * 32 + ty + 8 * k, N - 1)];
  }
  if (beta != 0.0)
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = y[rc + N * min(by * 32 + ty + 8 * k, N - 1)];
#pragma unroll
  for (int k = 0; k < 4; ++k) tile[ty + 8 * k][tx] = t[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t r = bx * 32 + tx, c = by * 32 + ty + 8 * k;
    if (r < N && c < N) {
      const double u = v[k] + tile[tx][ty + 8 * k];
      y[r + N * c] = (beta == 0.0) ? u : u + beta * w[k];
    }
  }
}

__global__ void packsum_kernel(const double* __restrict__ full, double* __restrict__ packed,
                               int64_t N, int64_t sx, int64_t sy) {
  full += int64_t(blockIdx.z) * sx;
  packed += int64_t(blockIdx.z) * sy;
  GRID_LOOP(k, N * (N + 1) / 2) {
    const int64_t X = tri_root2(k), Y = k - X * (X + 1) / 2;
    double v = full[X + N * Y];
    if (X != Y) v += full[Y + N * X];
    packed[k] += v;
  }
}

__global__ void unpack_upper_add_kernel(const double* __restrict__ packed, double* __restrict__ full,
                                        int64_t N, double alpha, double diag_scale, int64_t sx, int64_t sy) {
  packed += int64_t(blockIdx.z) * sx;
  full += int64_t(blockIdx.z) * sy;
  GRID_LOOP(k, N * (N + 1) / 2) {
    const int64_t X = tri_root2(k), Y = k - X * (X + 1) / 2;
    double v = alpha * packed[k];
    if (X == Y) v *= diag_scale;
    full[Y + N * X] += v;
  }
}

// x(R, C) += alpha * [R == C ? p{R,R} : f1 p{R,C} + f2 p{U,W}],
// U = (R_a, C_i), W = (C_a, R_i)  (the element the psrq terms of the forward pass read)
__global__ void sympack_adjoint_kernel(const double* __restrict__ p, double* __restrict__ x,
                                       int64_t n_v, int64_t n_o, double alpha, double f1, double f2, bool acc, int64_t sx, int64_t sy) {
  p += int64_t(blockIdx.z) * sx;
  x += int64_t(blockIdx.z) * sy;
  const int64_t N = n_v * n_o;
  GRID_LOOP(idx, N * N) {
    const int64_t R = idx % N, C = idx / N;
    double v;
    if (R == C) {
      v = p[pidx2(R, R)];
    } else {
      v = f1 * p[pidx2(R, C)];
      if (f2 != 0.0) {
        const int64_t Ra = R % n_v, Ri = R / n_v, Ca = C % n_v, Ci = C / n_v;
        const int64_t U = Ra + n_v * Ci, W = Ca + n_v * Ri;
        if (U != W) v += f2 * p[pidx2(U, W)];
      }
    }
    x[idx] = acc ? x[idx] + alpha * v : alpha * v;
  }
}

// The f2 = 0 form through 32 x 32 LDS tiles (as squareup: one workgroup per
// tile pair reads packed (X, Y), Y <= X, along Y and updates x(Y, X) along Y
// and x(X, Y) along X).
__global__ __launch_bounds__(256) void sympack_adjoint_tiled_kernel(const double* __restrict__ p,
                                                                    double* __restrict__ x, int64_t N,
                                                                    double alpha, double f1, bool acc, int64_t sx,
                                                                    int64_t sy) {
  p += int64_t(blockIdx.z) * sx;
  x += int64_t(blockIdx.z) * sy;
  __shared__ double P[32][33];                          // P[xl][yl] = p(X0 + xl, Y0 + yl)
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t xb = tri_root2(blockIdx.x), yb = int64_t(blockIdx.x) - xb * (xb + 1) / 2;
  const int64_t X0 = xb * 32, Y0 = yb * 32;
  double v[4], w1[4] = {}, w2[4] = {};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t X = min(X0 + ty + 8 * k, N - 1);
    v[k] = p[X * (X + 1) / 2 + min(Y0 + tx, X)];
  }
  if (acc)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w1[k] = x[min(Y0 + tx, N - 1) + N * min(X0 + ty + 8 * k, N - 1)];
      w2[k] = x[min(X0 + tx, N - 1) + N * min(Y0 + ty + 8 * k, N - 1)];
    }
#pragma unroll
  for (int k = 0; k < 4; ++k) P[ty + 8 * k][tx] = v[k] * (X0 + ty + 8 * k == Y0 + tx ? alpha : alpha * f1);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t X = X0 + ty + 8 * k, Y = Y0 + tx;     // x(Y, X), along Y
    const double u1 = P[ty + 8 * k][tx], u2 = P[tx][ty + 8 * k];
    if (X < N && Y <= X) x[Y + N * X] = acc ? w1[k] + u1 : u1;
    const int64_t Xr = X0 + tx, Yc = Y0 + ty + 8 * k;   // x(Xr, Yc), along Xr (the diagonal once)
    if (Xr < N && Yc < Xr) x[Xr + N * Yc] = acc ? w2[k] + u2 : u2;
  }
}

// t2[{(c,i),(d,j)}] += coef * tp[ij, cd] + sgn * tm[ij, cd]
__global__ void ladder_t_pm_adjoint_kernel(const double* __restrict__ tp, const double* __restrict__ tm,
                                           double* __restrict__ t2, int64_t n_o, int64_t n_v, int64_t st, int64_t sp, int64_t sm) {
  tp += int64_t(blockIdx.z) * sp;
  tm += int64_t(blockIdx.z) * sm;
  t2 += int64_t(blockIdx.z) * st;
  const int64_t Nov = n_o * n_v;
  const int64_t op = n_o * (n_o + 1) / 2, om = n_o * (n_o - 1) / 2;
  GRID_LOOP(k, Nov * (Nov + 1) / 2) {
    const int64_t X = tri_root2(k), Y = k - X * (X + 1) / 2;
    const int64_t c = X % n_v, i = X / n_v, d = Y % n_v, j = Y / n_v;
    const int64_t il = i < j ? i : j, ih = i < j ? j : i;
    const int64_t cl = c < d ? c : d, ch = c < d ? d : c;
    const double coef = (c == d) ? 1.0 : ((i == j) ? 2.0 : 1.0);
    double v = coef * tp[(ih * (ih + 1) / 2 + il) + op * (ch * (ch + 1) / 2 + cl)];
    if (i != j && c != d) {
      const double sgn = ((c < d) == (i < j)) ? 1.0 : -1.0;
      v += sgn * tm[(ih * (ih - 1) / 2 + il) + om * (ch * (ch - 1) / 2 + cl)];
    }
    t2[k] += v;
  }
}

// G(c, a', d, b') = [a >= b] (c == d ? 2 gp[cc,k] : gp[cd,k] +- gm[cd,k]), k = col[a + v b] - col0
__global__ void ladder_g_pm_adjoint_kernel(const double* __restrict__ gp, const double* __restrict__ gm,
                                           double* __restrict__ G, int64_t n_v, int64_t a0,
                                           int64_t lenA, int64_t b0, int64_t lenB,
                                           const int32_t* __restrict__ col, int64_t col0) {
  const int64_t vp = n_v * (n_v + 1) / 2, vm = n_v * (n_v - 1) / 2;
  const int64_t rows = n_v * lenA;
  GRID_LOOP(idx, rows * n_v * lenB) {
    const int64_t r = idx % rows, q = idx / rows;
    const int64_t c = r % n_v, aa = r / n_v, d = q % n_v, bb = q / n_v;
    const int64_t a = a0 + aa, b = b0 + bb;
    double v = 0.0;
    if (a >= b) {
      const int64_t k = int64_t(col[a + n_v * b]) - col0;
      if (c == d) {
        v = 2.0 * gp[(c * (c + 1) / 2 + c) + vp * k];
      } else {
        const int64_t lo = c < d ? c : d, hi = c < d ? d : c;
        v = gp[(hi * (hi + 1) / 2 + lo) + vp * k];
        const double m = gm[(hi * (hi - 1) / 2 + lo) + vm * k];
        v += (c < d) ? m : -m;
      }
    }
    G[idx] = v;
  }
}

// adjoint of ladder_gather: for stored (i' <= j', a' >= b'):
// wp += s1 om[P1] + s2 om[P2],  wm += s1 om[P1] - s2 om[P2]
// P1 = {(a',i'),(b',j')}, P2 = {(a',j'),(b',i')}, s = 1/2 on the packed diagonal
__global__ void ladder_gather_adjoint_kernel(const double* __restrict__ om,
                                             const int32_t* __restrict__ pa,
                                             const int32_t* __restrict__ pb, double* __restrict__ wp,
                                             double* __restrict__ wm, int64_t n_o, int64_t n_v, int64_t so, int64_t sp, int64_t sm) {
  om += int64_t(blockIdx.z) * so;
  wp += int64_t(blockIdx.z) * sp;
  wm += int64_t(blockIdx.z) * sm;
  const int64_t op = n_o * (n_o + 1) / 2, omn = n_o * (n_o - 1) / 2;
  const int64_t vp = n_v * (n_v + 1) / 2;
  GRID_LOOP(idx, op * vp) {
    const int64_t r = idx % op, cl = idx / op;
    const int64_t j = tri_root2(r), i = r - j * (j + 1) / 2;       // i <= j
    const int64_t a = pa[cl], b = pb[cl];                          // a >= b
    const int64_t X1 = a + n_v * i, Y1 = b + n_v * j;
    const int64_t X2 = a + n_v * j, Y2 = b + n_v * i;
    const int64_t k1 = pidx2(X1, Y1), k2 = pidx2(X2, Y2);
    const double v1 = (X1 == Y1 ? 0.5 : 1.0) * om[k1];
    const double v2 = (k2 != k1) ? (X2 == Y2 ? 0.5 : 1.0) * om[k2] : 0.0;
    wp[idx] = v1 + v2;
    if (i != j) wm[(j * (j - 1) / 2 + i) + omn * cl] = (a != b) ? v1 - v2 : 0.0;
  }
}

__global__ void t1_xy_kernel2(const double* t1, double* X, double* Y, int64_t n_o, int64_t n_v,
                              double diag, int64_t st, int64_t sm) {
  t1 += int64_t(blockIdx.z) * st;
  X += int64_t(blockIdx.z) * sm;
  Y += int64_t(blockIdx.z) * sm;
  const int64_t n = n_o + n_v;
  GRID_LOOP(k, n * n) {
    const int64_t p = k % n, q = k / n;
    double x = (p == q) ? diag : 0.0, y = x;
    if (p >= n_o && q < n_o) x = -t1[(p - n_o) + n_v * q];  // X(o+a, i) = -t_ai
    if (p < n_o && q >= n_o) y = t1[(q - n_o) + n_v * p];   // Y(i, o+a) = t_ai
    X[k] = x;
    Y[k] = y;
  }
}

__global__ void t1_xy_adjoint_kernel(const double* Xb, const double* Yb, double* t1b, int64_t n_o,
                                     int64_t n_v, int64_t st, int64_t sm) {
  Xb += int64_t(blockIdx.z) * sm;
  Yb += int64_t(blockIdx.z) * sm;
  t1b += int64_t(blockIdx.z) * st;
  const int64_t n = n_o + n_v;
  GRID_LOOP(k, n_o * n_v) {
    const int64_t a = k % n_v, i = k / n_v;
    t1b[k] += -Xb[(n_o + a) + n * i] + Yb[i + n * (n_o + a)];
  }
}

__global__ void trace_oo_kernel2(const double* Loo, double* XJ, int64_t nJ, int64_t n_o, int64_t sx, int64_t sy) {
  Loo += int64_t(blockIdx.z) * sx;
  XJ += int64_t(blockIdx.z) * sy;
  GRID_LOOP(J, nJ) {
    double s = 0.0;
    for (int64_t k = 0; k < n_o; ++k) s += Loo[J + nJ * (k + n_o * k)];
    XJ[J] = s;
  }
}

__global__ void trace_oo_adjoint_kernel(const double* XJb, double* Loob, int64_t nJ, int64_t n_o, int64_t sx, int64_t sy) {
  XJb += int64_t(blockIdx.z) * sx;
  Loob += int64_t(blockIdx.z) * sy;
  GRID_LOOP(idx, nJ * n_o) {
    const int64_t J = idx % nJ, k = idx / nJ;
    Loob[J + nJ * (k + n_o * k)] += XJb[J];
  }
}

__global__ void fock_ov_vector_kernel2(const double* F, double* f, int64_t n_o, int64_t n_v, int64_t sx, int64_t sy) {
  F += int64_t(blockIdx.z) * sx;
  f += int64_t(blockIdx.z) * sy;
  const int64_t n = n_o + n_v;
  GRID_LOOP(k, n_o * n_v) {
    const int64_t b = k % n_v, j = k / n_v;
    f[k] = F[j + n * (n_o + b)];
  }
}

__global__ void fock_ov_vector_adjoint_kernel(const double* fb, double* Fb, int64_t n_o, int64_t n_v, int64_t sx, int64_t sy) {
  fb += int64_t(blockIdx.z) * sx;
  Fb += int64_t(blockIdx.z) * sy;
  const int64_t n = n_o + n_v;
  GRID_LOOP(k, n_o * n_v) {
    const int64_t b = k % n_v, j = k / n_v;
    Fb[j + n * (n_o + b)] += fb[k];
  }
}

__global__ void copy_sub_kernel2(const double* src, int64_t lds, double* dst, int64_t ldd, int64_t m,
                                 int64_t n, double alpha, double beta, int64_t sx, int64_t sy) {
  src += int64_t(blockIdx.z) * sx;
  dst += int64_t(blockIdx.z) * sy;
  GRID_LOOP(k, m * n) {
    const int64_t r = k % m, c = k / m;
    // alpha = 0 scales dst alone: src is dst then, and may hold anything (an infinity or
    // NaN times 0 would stay in a derivative that starts here)
    const double v = alpha == 0.0 ? 0.0 : alpha * src[r + lds * c];
    dst[r + ldd * c] = (beta == 0.0) ? v : v + beta * dst[r + ldd * c];
  }
}

// dst(m x n, ld ldd) += sum_b part[b m n + r + m c], b < nbatch
__global__ void batch_sum_acc_kernel(const double* __restrict__ part, int64_t nbatch, int64_t m,
                                     int64_t n, double* __restrict__ dst, int64_t ldd) {
  const int64_t mn = m * n;
  GRID_LOOP(k, mn) {
    double v = 0.0;
    for (int64_t b = 0; b < nbatch; ++b) v += part[k + b * mn];
    dst[(k % m) + ldd * (k / m)] += v;
  }
}

inline unsigned g2(int64_t n) { return grid_for(n); }

}  // namespace

void batch_sum_acc(hipStream_t s, const double* part, int64_t nbatch, int64_t m, int64_t n, double* dst,
                   int64_t ldd) {
  if (m * n == 0) return;
  batch_sum_acc_kernel<<<g2(m * n), kBlock, 0, s>>>(part, nbatch, m, n, dst, ldd);
  ETG_LAUNCH("batch_sum_acc");
}

void scale(hipStream_t s, double* x, int64_t n, double beta) {
  if (n == 0 || beta == 1.0) return;
  scale_kernel<<<g2(n), kBlock, 0, s>>>(x, n, beta);
  ETG_LAUNCH("scale");
}

void symmetric_sum_acc(hipStream_t s, const double* x, double* y, int64_t N, double beta, const Batch& b) {
  if (x == y) fail("symmetric_sum_acc: out of place only");
  dim3 grid(unsigned(ceil_div(N, 32)), unsigned(ceil_div(N, 32)), unsigned(b.n));
  symmetric_sum_acc_kernel<<<grid, dim3(32, 8), 0, s>>>(x, y, N, beta, b.x, b.y);
  ETG_LAUNCH("symmetric_sum_acc");
}

void packsum(hipStream_t s, const double* full, double* packed, int64_t N, const Batch& b) {
  packsum_kernel<<<grid_z(N * (N + 1) / 2, b.n), kBlock, 0, s>>>(full, packed, N, b.x, b.y);
  ETG_LAUNCH("packsum");
}

void unpack_upper_add(hipStream_t s, const double* packed, double* full, int64_t N, double alpha,
                      double diag_scale, const Batch& b) {
  unpack_upper_add_kernel<<<grid_z(N * (N + 1) / 2, b.n), kBlock, 0, s>>>(packed, full, N, alpha, diag_scale, b.x, b.y);
  ETG_LAUNCH("unpack_upper_add");
}

void symmetrize_and_pack_adjoint(hipStream_t s, const double* packed, double* x, int64_t n_v,
                                 int64_t n_o, double alpha, double f1, double f2, bool acc, const Batch& b) {
  const int64_t N = n_v * n_o;
  if (f2 == 0.0 && N >= 32) {
    const int64_t nb = ceil_div(N, 32);
    sympack_adjoint_tiled_kernel<<<dim3(unsigned(nb * (nb + 1) / 2), 1, unsigned(b.n)), kBlock, 0, s>>>(
        packed, x, N, alpha, f1, acc, b.x, b.y);
    ETG_LAUNCH("sympack_adjoint_tiled");
    return;
  }
  sympack_adjoint_kernel<<<grid_z(N * N, b.n), kBlock, 0, s>>>(packed, x, n_v, n_o, alpha, f1, f2, acc, b.x, b.y);
  ETG_LAUNCH("sympack_adjoint");
}

void ladder_t_pm_adjoint(hipStream_t s, const double* tp, const double* tm, double* t2, int64_t n_o,
                         int64_t n_v, const LadderBatch& b) {
  const int64_t N = n_o * n_v;
  ladder_t_pm_adjoint_kernel<<<grid_z(N * (N + 1) / 2, b.n), kBlock, 0, s>>>(tp, tm, t2, n_o, n_v, b.vec, b.plus, b.minus);
  ETG_LAUNCH("ladder_t_pm_adjoint");
}

void ladder_g_pm_adjoint(hipStream_t s, const double* gp, const double* gm, double* G, int64_t n_v,
                         int64_t a0, int64_t lenA, int64_t b0, int64_t lenB, const int32_t* col,
                         int64_t col0) {
  const int64_t n = n_v * lenA * n_v * lenB;
  if (n == 0) return;
  ladder_g_pm_adjoint_kernel<<<g2(n), kBlock, 0, s>>>(gp, gm, G, n_v, a0, lenA, b0, lenB, col, col0);
  ETG_LAUNCH("ladder_g_pm_adjoint");
}

void ladder_gather_adjoint(hipStream_t s, const double* omega2, const int32_t* pcol_a,
                           const int32_t* pcol_b, double* wp, double* wm, int64_t n_o, int64_t n_v,
                           const LadderBatch& b) {
  const int64_t n = (n_o * (n_o + 1) / 2) * (n_v * (n_v + 1) / 2);
  ladder_gather_adjoint_kernel<<<grid_z(n, b.n), kBlock, 0, s>>>(omega2, pcol_a, pcol_b, wp, wm, n_o, n_v, b.vec, b.plus,
                                                                 b.minus);
  ETG_LAUNCH("ladder_gather_adjoint");
}

void t1_xy(hipStream_t s, const double* t1, double* X, double* Y, int64_t n_o, int64_t n_v,
           double diag, const Batch& b) {
  const int64_t n = n_o + n_v;
  t1_xy_kernel2<<<grid_z(n * n, b.n), kBlock, 0, s>>>(t1, X, Y, n_o, n_v, diag, b.x, b.y);
  ETG_LAUNCH("t1_xy");
}

void t1_xy_adjoint(hipStream_t s, const double* Xb, const double* Yb, double* t1b, int64_t n_o,
                   int64_t n_v, const Batch& b) {
  t1_xy_adjoint_kernel<<<grid_z(n_o * n_v, b.n), kBlock, 0, s>>>(Xb, Yb, t1b, n_o, n_v, b.x, b.y);
  ETG_LAUNCH("t1_xy_adjoint");
}

void trace_oo(hipStream_t s, const double* Loo, double* XJ, int64_t nJ, int64_t n_o, const Batch& b) {
  trace_oo_kernel2<<<grid_z(nJ, b.n), kBlock, 0, s>>>(Loo, XJ, nJ, n_o, b.x, b.y);
  ETG_LAUNCH("trace_oo");
}

void trace_oo_adjoint(hipStream_t s, const double* XJb, double* Loob, int64_t nJ, int64_t n_o, const Batch& b) {
  trace_oo_adjoint_kernel<<<grid_z(nJ * n_o, b.n), kBlock, 0, s>>>(XJb, Loob, nJ, n_o, b.x, b.y);
  ETG_LAUNCH("trace_oo_adjoint");
}

void fock_ov_vector(hipStream_t s, const double* F, double* f, int64_t n_o, int64_t n_v, const Batch& b) {
  fock_ov_vector_kernel2<<<grid_z(n_o * n_v, b.n), kBlock, 0, s>>>(F, f, n_o, n_v, b.x, b.y);
  ETG_LAUNCH("fock_ov_vector");
}

void fock_ov_vector_adjoint(hipStream_t s, const double* fb, double* Fb, int64_t n_o, int64_t n_v, const Batch& b) {
  fock_ov_vector_adjoint_kernel<<<grid_z(n_o * n_v, b.n), kBlock, 0, s>>>(fb, Fb, n_o, n_v, b.x, b.y);
  ETG_LAUNCH("fock_ov_vector_adjoint");
}

void copy_sub(hipStream_t s, const double* src, int64_t lds, double* dst, int64_t ldd, int64_t m,
              int64_t n, double alpha, double beta, const Batch& b) {
  if (m * n == 0) return;
  copy_sub_kernel2<<<grid_z(m * n, b.n), kBlock, 0, s>>>(src, lds, dst, ldd, m, n, alpha, beta, b.x, b.y);
  ETG_LAUNCH("copy_sub");
}

}  // namespace etg
