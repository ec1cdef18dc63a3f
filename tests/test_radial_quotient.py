"""The interpolation weight's quotient d1 / d0 of map_amd/csrc/radial.hip: for every whole d1 < d0 <=
65536, d1 * (1/d0) corrected with two fused multiply-adds has the bits of the F32 division."""
import subprocess

import pytest

SOURCE = r"""
#include <cstdio>
#include <cstring>
int main() {
  long bad = 0;
#pragma omp parallel for schedule(dynamic, 64) reduction(+ : bad)
  for (int d0 = 1; d0 <= 65536; d0++) {
    const float c = (float)d0, y = 1.0f / c;
    for (int d1 = 0; d1 < d0; d1++) {
      const float f = (float)d1;
      float q = f * y;
      q = __builtin_fmaf(__builtin_fmaf(-q, c, f), y, q);
      const float e = f / c;
      bad += memcmp(&q, &e, 4) != 0;
    }
  }
  std::printf("%ld\n", bad);
}
"""


def test_corrected_quotient_is_the_division(tmp_path):
    with open("/proc/cpuinfo") as f:
        if " fma " not in f.read():
            pytest.skip("no fused multiply-add on this CPU")
    src = tmp_path / "quotient.cpp"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O3", "-mfma", "-mavx2", "-ffp-contract=off", "-fopenmp", str(src), "-o", str(tmp_path / "q")], check=True)
    assert subprocess.run([str(tmp_path / "q")], check=True, capture_output=True, text=True).stdout.strip() == "0"
