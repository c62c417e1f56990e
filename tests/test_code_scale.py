"""The quantizers' quotient by residual (halo::CodeScale), taken from the kernel header and compiled for the host: its
codes equal rint of the IEEE division for every mantissa of the scale at every half-integer quotient (only values within an
ulp of one can round to another code; both sides scale by powers of two alike), and over random quotients at every exponent
of the scale, subnormal scales and those around 2^-60, where values are scaled up first, among them."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parents[1] / "halo-flash_amd" / "csrc" / "kernels" / "common.h"

MAIN = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#define __device__
#define __forceinline__ inline
@STRUCT@
static inline float Fb(std::uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
static inline std::uint32_t Bf(float f) { std::uint32_t u; std::memcpy(&u, &f, 4); return u; }
static inline int Want(float v, float scale) { return scale > 0.0f ? static_cast<int>(rintf(v / scale)) : 0; }
int main() {
  long ties = 0, random = 0;
#pragma omp parallel for schedule(dynamic, 4096) reduction(+ : ties)
  for (std::uint32_t m = 0; m < (1u << 23); ++m) {
    const float scale = Fb((127u << 23) | m);
    const CodeScale cs(scale);
    for (int c = 0; c < 128; ++c) {
      const std::uint32_t at = Bf((static_cast<float>(c) + 0.5f) * scale);
      for (int d = -2; d <= 2; ++d) {
        const float v = Fb(at + d);
        ties += cs.Code(v) != Want(v, scale);
      }
    }
  }
#pragma omp parallel for schedule(dynamic) reduction(+ : random)
  for (int e = 0; e < 248; ++e) {  // biased exponent of the scale: amax / 127 stays below 2^121
    std::uint64_t s = 88172645463325252ull + e;
    for (int i = 0; i < 200000; ++i) {
      s ^= s << 13, s ^= s >> 7, s ^= s << 17;
      const float scale = Fb((static_cast<std::uint32_t>(e) << 23) | (s & 0x7fffff));
      float v = scale * (static_cast<float>(static_cast<int>((s >> 23) % 2541) - 1270) / 10.0f);
      if (i % 2) v = Fb(Bf(scale * (static_cast<float>((s >> 40) % 127) + 0.5f)) + static_cast<int>(s >> 60) - 8);
      if (std::isfinite(v) && std::fabs(v) <= scale * 190.0f) random += CodeScale(scale).Code(v) != Want(v, scale);
    }
  }
  const CodeScale zero(0.0f);
  std::printf("%ld %ld %d\n", ties, random, zero.Code(0.0f));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_codes_equal_the_division(tmp_path):
    struct = re.search(r"^struct CodeScale \{.*?^\};", HEADER.read_text(), re.M | re.S)
    assert struct, "CodeScale not found"
    src, exe = tmp_path / "codes.cpp", tmp_path / "codes"
    src.write_text(MAIN.replace("@STRUCT@", struct.group(0)))
    subprocess.run(["g++", "-O3", "-march=native", "-ffp-contract=off", "-fopenmp", "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    assert out == ["0", "0", "0"], f"codes off: {out[0]} at half-integers, {out[1]} at random, zero block {out[2]}"
