"""The division that a projection's launch does when it norms its own rows
(csrc/model_ops.hip): h / norm as h times the rounded reciprocal, corrected
once by the remainder, equals the rounded quotient for every significand of a
16-bit h and every significand of norm. (Powers of two scale all of it exactly
while nothing leaves the normal range, which the kernel checks.)"""
import ctypes
import subprocess

import pytest

SOURCE = r"""
#include <math.h>
#include <stdint.h>
#include <string.h>
static float mantissa(uint32_t m) {
  const uint32_t u = 0x3f800000u | m;
  float f;
  memcpy(&f, &u, 4);
  return f;
}
__attribute__((target("avx2,fma"))) long mismatches(int bits) {
  long bad = 0;
#pragma omp parallel for reduction(+ : bad)
  for (uint32_t m = 0; m < (1u << 23); ++m) {
    const float norm = mantissa(m), y = 1.f / norm;
    for (uint32_t a = 0; a < (1u << bits); ++a) {
      const float h = mantissa(a << (23 - bits)), q = h * y;
      bad += fmaf(fmaf(-q, norm, h), y, q) != h / norm;
    }
  }
  return bad;
}
int supported(void) { return __builtin_cpu_supports("fma") && __builtin_cpu_supports("avx2"); }
"""


def test_corrected_reciprocal_rounds_as_the_division(tmp_path):
    src, lib = tmp_path / "q.c", tmp_path / "q.so"
    src.write_text(SOURCE)
    subprocess.run(["gcc", "-O3", "-fPIC", "-shared", "-fopenmp", "-ffp-contract=off", str(src),
                    "-o", str(lib), "-lm"], check=True)
    q = ctypes.CDLL(str(lib))
    if not q.supported():
        pytest.skip("no FMA instructions on this CPU")
    q.mismatches.restype = ctypes.c_long
    for bits in (7, 10):  # bf16 and f16 significands after the leading one
        assert q.mismatches(bits) == 0
