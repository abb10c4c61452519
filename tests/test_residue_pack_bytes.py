"""The last step of a residue (et_amd/csrc/residue.hpp, low_byte): for every modulus and every
23-bit byte sum the low byte is congruent to 2^23 + v, where the FP32 quotient is one off too.
Built for the host; whole numbers, compared exactly."""
import ctypes
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "residue.hpp"
using namespace etg::residue;
extern "C" long wrong(int i, long from, long to) {
  long bad = 0;
  for (long v = from; v < to; ++v) {
    const int r = (signed char)(low_byte(kBits23 + uint32_t(v), kC.invf[i], kC.c[i]) & 0xff);
    bad += ((1l << 23) + v - r) % kMod[i] != 0;
  }
  return bad;
}
'''


def test_every_byte_sum(tmp_path):
    src = tmp_path / 'low.cpp'
    src.write_text(SRC)
    out = tmp_path / 'low.so'
    subprocess.run(['g++', '-std=c++17', '-O2', '-shared', '-fPIC', '-I', os.path.join(ROOT, 'et_amd', 'csrc'),
                    str(src), '-o', str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    lib.wrong.restype = ctypes.c_long
    lib.wrong.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_long]
    # sums of 8 bytes times weights below 256, and an offset
    top = 8 * 255 * 255 + 256
    for i in range(15):
        assert lib.wrong(i, 0, top) == 0
        assert lib.wrong(i, (1 << 23) - 1000, 1 << 23) == 0
