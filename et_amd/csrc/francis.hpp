// Eigenvalues of a real upper Hessenberg matrix by the implicitly
// double-shifted QR iteration (J. G. F. Francis, Comput. J. 4 (1961) 265-271;
// the step and the deflation loop as stated in Golub & Van Loan, Matrix
// Computations, 4th ed., Algorithms 7.5.1 and 7.5.2).  Only the eigenvalues
// are wanted, so each similarity transformation is applied to the active
// diagonal block alone.
//
// The routine is written once for a team of lanes: on the device the team is
// one wavefront (64 lanes, scalar control computed redundantly by every lane
// from the same LDS values, row and column sweeps split across lanes); on the
// host it is one lane, so the same code is checked against LAPACK from the CPU.
//
// On the device the bulge chase is one chain of dependent steps.  A step's left
// and right updates meet only in the 3 x 3 block on the diagonal and in the one
// entry below it; every lane computes these in registers, and the other columns
// (left only) and rows (right only) are independent of each other.  So a step
// is one round of reads and one of writes, and the next reflector is made from
// registers while the writes and reads are under way.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define ETG_HD __host__ __device__
#else
#define ETG_HD
#endif

namespace etg {
namespace francis {

// Reflector I - tau v v^T with v = (1, v1, v2) that maps a (length nr = 2 or 3)
// onto alpha e1.  tau = 0 when a is already a multiple of e1.
struct Reflector {
  double tau, v1, v2, alpha;
};

ETG_HD inline Reflector make_reflector(double a0, double a1, double a2, int nr) {
  Reflector r;
  const double tail2 = nr == 3 ? a1 * a1 + a2 * a2 : a1 * a1;
  if (nr == 3 ? tail2 == 0.0 : a1 == 0.0) {
    r.tau = 0.0;
    r.v1 = r.v2 = 0.0;
    r.alpha = a0;
    return r;
  }
  const double len = std::sqrt(a0 * a0 + tail2);
  const double beta = a0 >= 0.0 ? -len : len;            // opposite sign of a0: no cancellation
  r.tau = (beta - a0) / beta;
  const double inv = 1.0 / (a0 - beta);
  r.v1 = a1 * inv;
  r.v2 = nr == 3 ? a2 * inv : 0.0;
  r.alpha = beta;
  return r;
}

// Eigenvalues of the 2 x 2 block [[a, b], [c, d]]: real pair (w1, w2, im = 0)
// or complex pair re +- i im (im > 0).
ETG_HD inline void block2_eigenvalues(double a, double b, double c, double d, double* re1, double* re2,
                                      double* im) {
  const double p = 0.5 * (a - d);
  const double disc = p * p + b * c;
  if (disc >= 0.0) {
    const double root = std::sqrt(disc);
    const double q = p >= 0.0 ? p + root : p - root;      // |q| = |p| + root
    if (q == 0.0) {
      *re1 = *re2 = d;
    } else {
      *re1 = d + q;
      *re2 = d - b * c / q;                               // (p + r)(p - r) = -bc
    }
    *im = 0.0;
  } else {
    *re1 = *re2 = d + p;
    *im = std::sqrt(-disc);
  }
}

// Team of lanes: rank, size, barrier, the sum of one value per lane, and the
// highest l in [1, top] with f(l) (0 if there is none).
struct HostTeam {
  int rank() const { return 0; }
  int size() const { return 1; }
  void sync() const {}
  double sum(double v) const { return v; }
  template <class F>
  int highest(int top, F f) const {
    while (top > 0 && !f(top)) --top;
    return top;
  }
};

// One step of the bulge chase at column c of the active block lo .. hi: the
// reflector of (x, y, z) on rows and columns c .. c + kRows - 1.  kBelow: row
// c + 3 is in the block.  On return (x, y, z) is the next step's column.
template <int kRows, bool kBelow, class Team>
ETG_HD inline void chase_step(const Team& team, double* H, int ldh, int lo, int hi, int c, double& x, double& y,
                              double& z) {
  const int me = team.rank(), lanes = team.size();
  double* D = H + c + c * ldh;                            // the diagonal block b, and t below its last column
  double b[kRows][kRows], t = 0.0;
  for (int j = 0; j < kRows; ++j)
    for (int i = 0; i < kRows; ++i) b[i][j] = D[i + j * ldh];
  if (kBelow) t = D[3 + 2 * ldh];
  // the columns right of the block (updated from the left), then the rows above
  // it (updated from the right): three entries p[0], p[st], p[2 st] each
  const int cols = kBelow ? hi - c - 2 : 0, items = cols + c - lo;
  int q = me, st = 1;
  double *p = H, p0 = 0.0, p1 = 0.0, p2 = 0.0;
  auto fetch = [&]() {
    if (q >= items) return;
    st = q < cols ? 1 : ldh;
    p = H + (q < cols ? c + (c + 3 + q) * ldh : lo + q - cols + c * ldh);
    p0 = p[0];
    p1 = p[st];
    if (kRows == 3) p2 = p[2 * st];
  };
  fetch();
  const Reflector r = make_reflector(x, y, z, kRows);
  const double tv1 = r.tau * r.v1, tv2 = r.tau * r.v2;
  for (int j = 0; j < kRows; ++j) {                       // from the left
    double w = r.tau * b[0][j] + tv1 * b[1][j];
    if (kRows == 3) w += tv2 * b[kRows - 1][j];
    b[0][j] -= w;
    b[1][j] -= w * r.v1;
    if (kRows == 3) b[kRows - 1][j] -= w * r.v2;
  }
  for (int i = 0; i < kRows; ++i) {                       // from the right
    double w = r.tau * b[i][0] + tv1 * b[i][1];
    if (kRows == 3) w += tv2 * b[i][kRows - 1];
    b[i][0] -= w;
    b[i][1] -= w * r.v1;
    if (kRows == 3) b[i][kRows - 1] -= w * r.v2;
  }
  const double wt = tv2 * t;                              // row c + 3: (0, 0, t), from the right
  while (q < items) {
    double w = r.tau * p0 + tv1 * p1;
    if (kRows == 3) w += tv2 * p2;
    p[0] = p0 - w;
    p[st] = p1 - w * r.v1;
    if (kRows == 3) p[2 * st] = p2 - w * r.v2;
    q += lanes;
    fetch();
  }
  // column c below the diagonal stays in registers: the next reflector takes it,
  // and leaves alpha and zeros
  if (me == 0) {
    if (c > lo) {
      D[-ldh] = r.alpha;
      D[1 - ldh] = 0.0;
    }
    D[0] = b[0][0];
    for (int j = 1; j < kRows; ++j)
      for (int i = 0; i < kRows; ++i) D[i + j * ldh] = b[i][j];
    if (kBelow) {
      D[3 + ldh] = -wt * r.v1;
      D[3 + 2 * ldh] = t - wt * r.v2;
    }
  }
  x = b[1][0];
  y = kRows == 3 ? b[kRows - 1][0] : 0.0;
  z = -wt;
  team.sync();
}

// Eigenvalues of the k x k upper Hessenberg matrix H (column-major, leading
// dimension ldh; overwritten) into wr, wi (complex pairs as re +- i im with the
// negative imaginary part first).  Returns 0, or 1 when an eigenvalue needs
// more than kMaxSweeps double-shift steps.  *hnorm receives the sum of the
// absolute values of H's entries on entry (the scale of the small-subdiagonal
// test and of the later inverse iteration).
template <class Team>
ETG_HD int hessenberg_eigenvalues(const Team& team, double* H, int ldh, int k, double* wr, double* wi,
                                  double* hnorm) {
  constexpr int kMaxSweeps = 80;
  constexpr double kEps = 2.220446049250313e-16;
#define ETG_H(i, j) H[(i) + (j) * ldh]
  const int me = team.rank(), lanes = team.size();
  double scale = 0.0;
  for (int j = me; j < k; j += lanes)
    for (int i = 0; i <= (j + 1 < k ? j + 1 : k - 1); ++i) scale += std::fabs(ETG_H(i, j));
  scale = team.sum(scale);
  *hnorm = scale;
  if (scale == 0.0) scale = 1.0;
  int hi = k - 1;             // the active block ends at row/column hi
  int sweeps = 0;             // double-shift steps since the last deflation
  while (hi >= 0) {
    // smallest lo such that H(lo:hi, lo:hi) has no negligible subdiagonal entry
    const int lo = team.highest(hi, [&](int l) {
      double ref = std::fabs(ETG_H(l, l)) + std::fabs(ETG_H(l - 1, l - 1));
      if (ref == 0.0) ref = scale;
      return std::fabs(ETG_H(l, l - 1)) <= kEps * ref;
    });
    team.sync();
    if (lo > 0 && me == 0) ETG_H(lo, lo - 1) = 0.0;
    team.sync();
    if (lo == hi) {                                       // one eigenvalue deflates
      if (me == 0) {
        wr[hi] = ETG_H(hi, hi);
        wi[hi] = 0.0;
      }
      hi -= 1;
      sweeps = 0;
      team.sync();
      continue;
    }
    if (lo == hi - 1) {                                   // a 2 x 2 block deflates
      double r1, r2, im;
      block2_eigenvalues(ETG_H(hi - 1, hi - 1), ETG_H(hi - 1, hi), ETG_H(hi, hi - 1), ETG_H(hi, hi), &r1, &r2,
                         &im);
      if (me == 0) {
        if (im == 0.0) {
          wr[hi - 1] = r1;
          wr[hi] = r2;
          wi[hi - 1] = wi[hi] = 0.0;
        } else {
          wr[hi - 1] = wr[hi] = r1;
          wi[hi - 1] = -im;
          wi[hi] = im;
        }
      }
      hi -= 2;
      sweeps = 0;
      team.sync();
      continue;
    }
    if (sweeps == kMaxSweeps) return 1;
    ++sweeps;
    // shifts: the eigenvalues of the trailing 2 x 2 block (sum s, product p);
    // every 10th step two unequal real shifts h + xi and h - xi / 2 off the
    // trailing entries instead.  They break the cycles of the standard shift
    // (a cyclic permutation matrix never deflates with it), and being unequal
    // they do not tie on eigenvalues placed symmetrically about h.
    // First column of (H - s1 I)(H - s2 I) on the block, written with differences
    // of diagonal entries so that it does not cancel when the block is close to
    // a multiple of I (a converging multiple eigenvalue): with the trailing
    // block [[a, b], [c, d]], (h00 - s1)(h00 - s2) = (h00 - a)(h00 - d) - b c.
    const double h00 = ETG_H(lo, lo), h10 = ETG_H(lo + 1, lo), h01 = ETG_H(lo, lo + 1);
    const double h11 = ETG_H(lo + 1, lo + 1);
    double x, y;
    if (sweeps % 10 == 0) {
      const double h = ETG_H(hi, hi);
      const double xi = std::fabs(ETG_H(hi, hi - 1)) + std::fabs(ETG_H(hi - 1, hi - 2));
      const double e = h00 - h;                           // shifts h + xi, h - xi / 2
      x = (e - xi) * (e + 0.5 * xi) + h01 * h10;
      y = h10 * (e + (h11 - h) - 0.5 * xi);
    } else {
      const double a = ETG_H(hi - 1, hi - 1), b = ETG_H(hi - 1, hi), c = ETG_H(hi, hi - 1), d = ETG_H(hi, hi);
      x = (h00 - a) * (h00 - d) - b * c + h01 * h10;
      y = h10 * ((h00 - a) + (h11 - d));
    }
    double z = h10 * ETG_H(lo + 2, lo + 1);
    const double sz = std::fabs(x) + std::fabs(y) + std::fabs(z);
    if (sz != 0.0) {
      x /= sz;
      y /= sz;
      z /= sz;
    }
    // chase the bulge down the block; (x, y, z) is the column that the next
    // reflector maps onto a multiple of e1
    int c = lo;
    for (; c + 3 <= hi; ++c) chase_step<3, true>(team, H, ldh, lo, hi, c, x, y, z);
    chase_step<3, false>(team, H, ldh, lo, hi, c, x, y, z);
    chase_step<2, false>(team, H, ldh, lo, hi, c + 1, x, y, z);
    if (me == 0) ETG_H(hi, hi - 1) = x;
    team.sync();
  }
  return 0;
#undef ETG_H
}

}  // namespace francis
}  // namespace etg
