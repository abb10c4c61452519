"""The integer arithmetic of the FP64 products on int8 matrix cores (et_amd/csrc/residue.hpp),
built for the host: residues, their sums and the reconstruction against exact integers."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "residue.hpp"
using namespace etg::residue;
extern "C" {
int modulus(int i) { return i < kModuli ? kMod[i] : 0; }
int norm_bits() { return kNormBits; }
int exponent(const double* x, long k) {
  double s = 0; uint64_t m = 0;
  for (long i = 0; i < k; ++i) {
    uint64_t b; __builtin_memcpy(&b, &x[i], 8); b &= 0x7fffffffffffffffull;
    s += x[i] * x[i]; if (b > m) m = b;
  }
  return scale_exponent(s, m, k);
}
// residue of x 2^e modulo m_i as the packs hold it
int residue(double x, int e, int i) {
  uint32_t lo, hi; to_integer(x, e, lo, hi);
  return (signed char)(residue_byte(lo, hi, i) & 0xff);
}
int sum_residue(int s, int i) { return (signed char)(residue_byte_of_sum(s, kC.md[i], kC.invd[i]) & 0xff); }
double dot(const double* a, const double* b, long k) {
  const int ea = exponent(a, k), eb = exponent(b, k);
  double hi = 0, lo = 0;
  for (int i = 0; i < kModuli; ++i) {
    int s = 0;
    for (long j = 0; j < k; ++j) s += residue(a[j], ea, i) * residue(b[j], eb, i);
    const double r = sum_residue(s, i);
    hi += r * kC.fhi[i]; lo += r * kC.flo[i];
  }
  return reconstruct(hi, lo, ea, eb);
}
}
'''


@pytest.fixture(scope='module')
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp('residue')
    src = d / 'residue.cpp'
    src.write_text(SRC)
    out = d / 'residue.so'
    subprocess.run(['g++', '-std=c++17', '-O2', '-shared', '-fPIC', '-I', os.path.join(ROOT, 'et_amd', 'csrc'),
                    str(src), '-o', str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    dp = ctypes.POINTER(ctypes.c_double)
    lib.dot.restype = ctypes.c_double
    lib.dot.argtypes = [dp, dp, ctypes.c_long]
    lib.exponent.argtypes = [dp, ctypes.c_long]
    lib.residue.argtypes = [ctypes.c_double, ctypes.c_int, ctypes.c_int]
    return lib


def _ptr(x):
    return x.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def test_residues_of_edge_integers(lib):
    """Every modulus, integers at the ends of the range and around multiples of the moduli and of 2^32."""
    edge = [0, 1, -1, 127, 128, -128, 255, 256, 2 ** 31, -2 ** 31, 2 ** 32 - 1, -2 ** 32, 2 ** 53 - 1, 1 - 2 ** 53,
            2 ** 58, -2 ** 58, 2 ** 58 - 64]
    for i in range(15):
        m = lib.modulus(i)
        for v in edge + [q * m + d for q in (-3, 1, 2 ** 20) for d in (-1, 0, 1, m // 2, m // 2 + 1)]:
            r = lib.residue(float(v), 0, i)
            assert (r - v) % m == 0 and -128 <= r <= 127
        for s in (0, 1, -1, 2 ** 31 - 1, -2 ** 31, 2 ** 30, m, -m, 128 * 128 * 131071):
            assert (lib.sum_residue(s, i) - s) % m == 0


@pytest.mark.parametrize('k', [1, 63, 64, 65, 1000])
@pytest.mark.parametrize('kind', ['normal', 'positive', 'lognormal', 'huge', 'tiny', 'zero'])
def test_products_within_the_rounding_of_the_operands(lib, kind, k):
    """|error| <= 2^-58 (|a|_2 |b|_1 + |b|_2 |a|_1) (each operand rounded by half an integer, of
    which the row's norm holds at least 2^57) + 2^-51 |a.b| (conversions and the final product)."""
    rng = np.random.default_rng(k)
    scale = {'huge': 1e180, 'tiny': 1e-180}.get(kind, 1.0)
    for _ in range(20):
        a, b = rng.normal(size=k) * scale, rng.normal(size=k) / scale
        if kind == 'positive':
            a, b = np.abs(a), np.abs(b)
        if kind == 'lognormal':
            a, b = a * 10 ** rng.uniform(-12, 0, k), b * 10 ** rng.uniform(-12, 0, k)
        if kind == 'zero':
            a = np.zeros(k)
        exact = np.sum(a.astype(np.longdouble) * b)
        n = lambda x: np.linalg.norm(x / np.abs(x).max()) * np.abs(x).max() if x.any() else 0.0
        bound = 2.0 ** -58 * (n(a) * np.abs(b).sum() + n(b) * np.abs(a).sum()) + 2.0 ** -51 * abs(exact)
        assert abs(lib.dot(_ptr(a), _ptr(b), k) - exact) <= bound


def test_scale_exponents(lib):
    """The scaled norm lies in (2^(bits - 1), 2^bits] where the squares are in range, below it elsewhere;
    rows with an infinity or NaN are marked."""
    rng = np.random.default_rng(2)
    bits = lib.norm_bits()
    for k in (1, 7, 300):
        for p in (-300, -160, -100, 0, 100, 160, 300):
            x = rng.normal(size=k) * 10.0 ** p
            big = np.abs(x).max()
            lg = np.log2(np.linalg.norm(x / big)) + np.log2(big) + lib.exponent(_ptr(x), k)
            assert lg <= bits + 1e-9
            if abs(p) <= 100:
                assert lg > bits - 1 - 1e-9
    for bad in (np.inf, -np.inf, np.nan):
        x = np.array([1.0, bad, 2.0])
        assert lib.exponent(_ptr(x), 3) == -2 ** 31
    assert lib.exponent(_ptr(np.zeros(3)), 3) == 0
