"""The guard of the FP64 products on int8 matrix cores (et_amd/csrc/residue.hpp), built for the host:
the bound on sum |a_k b_k|, and the errors on either side of the threshold, relative to that sum.

The operands' rounding is fixed relative to the rows' norms, so without the guard rows and columns
graded in opposite directions lose digits: the unguarded errors are recorded here beside those of a
plain FP64 sum."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "residue.hpp"
using namespace etg::residue;
namespace {
struct Row { int e; float norm; };
Row scan(const double* x, long k) {
  double s = 0; uint64_t m = 0;
  for (long i = 0; i < k; ++i) {
    uint64_t b; __builtin_memcpy(&b, &x[i], 8); b &= 0x7fffffffffffffffull;
    s += x[i] * x[i]; if (b > m) m = b;
  }
  return {scale_exponent(s, m, k), scaled_norm(s, m)};
}
double value(uint32_t q) {                        // of the 8-bit float
  const int e = int(q >> 2), f = int(q & 3);
  return e == 0 ? ldexp(f, -16) : ldexp(4 + f, e - 17);
}
}
extern "C" {
int guard_bits() { return kGuardBits; }
float norm_of(const double* x, long k) { return scan(x, k).norm; }
double magnitude(double x) {                      // of an integer, in units of 2^47
  uint32_t lo, hi; to_integer(x, 0, lo, hi);
  return value(magnitude_byte(hi));
}
// the int8 product's value; q: the guard's sum; returns whether the output goes to the FP64 kernel
int product(const double* a, const double* b, long k, double* v, double* q) {
  const Row ra = scan(a, k), rb = scan(b, k);
  double hi = 0, lo = 0, sum = 0;
  for (int i = 0; i < kModuli; ++i) {
    int s = 0;
    for (long j = 0; j < k; ++j) {
      uint32_t al, ah, bl, bh;
      to_integer(a[j], ra.e, al, ah); to_integer(b[j], rb.e, bl, bh);
      s += int((signed char)(residue_byte(al, ah, i) & 0xff)) * int((signed char)(residue_byte(bl, bh, i) & 0xff));
      if (i == 0) sum += value(magnitude_byte(ah)) * value(magnitude_byte(bh));
    }
    const double r = (signed char)(residue_byte_of_sum(s, kC.md[i], kC.invd[i]) & 0xff);
    hi += r * kC.fhi[i]; lo += r * kC.flo[i];
  }
  *v = reconstruct(hi, lo, ra.e, rb.e);
  *q = ldexp(sum, 94 - ra.e - rb.e);              // of the unscaled rows
  const float m = ra.norm > rb.norm ? ra.norm : rb.norm;
  return ra.norm > 0 && rb.norm > 0 && !(float(sum) >= kThreshold * m);
}
}
'''
U = 2.0 ** -53


@pytest.fixture(scope='module')
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp('guard')
    src = d / 'guard.cpp'
    src.write_text(SRC)
    out = d / 'guard.so'
    subprocess.run(['g++', '-std=c++17', '-O2', '-shared', '-fPIC', '-I', os.path.join(ROOT, 'et_amd', 'csrc'),
                    str(src), '-o', str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    dp = ctypes.POINTER(ctypes.c_double)
    lib.norm_of.restype = ctypes.c_float
    lib.norm_of.argtypes = [dp, ctypes.c_long]
    lib.magnitude.restype = ctypes.c_double
    lib.magnitude.argtypes = [ctypes.c_double]
    lib.product.argtypes = [dp, dp, ctypes.c_long, dp, dp]
    return lib


def _product(lib, a, b):
    p = lambda x: x.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    v, q = ctypes.c_double(), ctypes.c_double()
    flag = lib.product(p(a), p(b), len(a), ctypes.byref(v), ctypes.byref(q))
    return v.value, q.value, bool(flag)


def test_magnitudes(lib):
    """The whole 2^32 of the integer's magnitude (rounded down), rounded to a quarter of a power of two: an
    eighth below to a ninth above."""
    rng = np.random.default_rng(0)
    for x in np.concatenate([2.0 ** rng.uniform(33.5, 62, 4000), 2.0 ** np.arange(34, 63.0), [2.0 ** 62]]):
        for s in (x, -x):
            r = lib.magnitude(float(np.rint(s))) / (x * 2.0 ** -47)
            assert 0.875 * (1 - 2.0 ** 32 / x) <= r <= 1.1112
    assert lib.magnitude(0.0) == 0.0 and lib.magnitude(2.0 ** 31) == 0.0


@pytest.mark.parametrize('k', [1, 63, 300, 1600])
@pytest.mark.parametrize('kind', ['normal', 'positive', 'sparse', 'one', 'lognormal'])
def test_the_sum_is_a_bound(lib, kind, k):
    rng = np.random.default_rng(k)
    for _ in range(10):
        a, b = rng.normal(size=k), rng.normal(size=k)
        if kind == 'positive':
            a, b = np.abs(a), np.abs(b)
        if kind == 'sparse':
            a[rng.random(k) < 0.9] = 0.0
        if kind == 'one':
            a[0] = 1e12
        if kind == 'lognormal':
            a, b = a * 10 ** rng.uniform(-12, 0, k), b * 10 ** rng.uniform(-12, 0, k)
        _, q, _ = _product(lib, a, b)
        assert q <= 1.24 * np.sum(np.abs(a * b)) * (1 + 1e-12)
        if kind in ('normal', 'positive') and k > 1:
            assert q >= 0.75 * np.sum(np.abs(a * b))


def test_norms(lib):
    rng = np.random.default_rng(1)
    p = lambda x: x.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    for scale in (1e-120, 1e-3, 1.0, 1.4, 2.0, 1e100):
        x = rng.normal(size=50) * scale
        f = np.linalg.norm(x / np.abs(x).max()) * np.abs(x).max()
        r = lib.norm_of(p(x), 50)
        assert 0.5 < r <= 1.000002
        lg = np.log2(f) - np.log2(r)
        assert abs(lg - np.rint(lg)) < 1e-5
    assert lib.norm_of(p(np.zeros(4)), 4) < 0
    for bad in (np.inf, np.nan):
        assert lib.norm_of(p(np.array([1.0, bad])), 2) == np.inf
    assert lib.norm_of(p(np.array([1e-200, 1e-190])), 2) == 1.0


@pytest.mark.parametrize('decades', [0, 1, 2, 3, 4, 6, 8])
def test_opposite_grading(lib, decades):
    """Rows graded 10^-d over k = 1600, columns the other way.  Where the guard keeps the int8 product its
    rms error is at most 0.82 u of sum |a b| (asked for with a quarter for chance); without it d = 8 loses
    five digits."""
    k, errs, flags, plain = 1600, [], [], []
    rng = np.random.default_rng(decades)
    g = 10.0 ** (-decades * np.arange(k) / k)
    for _ in range(40):
        a, b = rng.normal(size=k) * g, rng.normal(size=k) * g[::-1]
        v, _, flag = _product(lib, a, b)
        exact = np.sum(a.astype(np.longdouble) * b)
        s = np.sum(np.abs(a * b))
        errs.append(float((v - exact) / s))
        plain.append(float((np.add.accumulate(a * b)[-1] - exact) / s))
        flags.append(flag)
    rms = np.sqrt(np.mean(np.square(errs))) / U
    print('grading %d: int8 %.2g u, plain FP64 sum %.2g u, %d of 40 flagged'
          % (decades, rms, np.sqrt(np.mean(np.square(plain))) / U, sum(flags)))
    kept = [e for e, f in zip(errs, flags) if not f]
    if kept:
        assert np.sqrt(np.mean(np.square(kept))) < 1.25 * 0.82 * U
    if decades <= 2:
        assert not any(flags)
    if decades >= 6:
        assert all(flags) and rms > 10


def test_zero_rows_are_kept(lib):
    a, b = np.zeros(64), np.random.default_rng(0).normal(size=64)
    assert _product(lib, a, b) == (0.0, 0.0, False)
