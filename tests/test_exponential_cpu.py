"""The exponential behind float32 sigmoid and silu (spar_amd/csrc/hip/ops.hpp),
compiled for the host: within an ulp of the exact value in double, and the
correctly rounded float32, over the float32 arguments from -0 to -110."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent

PROGRAM = r"""
#include <cmath>
#include <cstdio>
#include <cstring>
#include "ops.hpp"
int main() {
  double worst = 0.0;
  long wrong = 0;
  auto check = [&](float x) {
    const long double exact = expl(static_cast<long double>(x));
    const double got = spar_hip::accurate_exp_nonpositive(static_cast<double>(x));
    const double error = static_cast<double>(fabsl(got - exact) / exact);
    if (error > worst) worst = error;
    if (spar_hip::rounded_exp_nonpositive(x) != static_cast<float>(exact)) {
      std::printf("%a\n", x);
      ++wrong;
    }
  };
  // every 499th float32 from -0 to -110, and one whose exponential lies within
  // 2^-47 of a rounding boundary
  for (unsigned bits = 0x80000000U; bits <= 0xc2dc0000U; bits += 499) {
    float x;
    std::memcpy(&x, &bits, sizeof x);
    check(x);
  }
  check(-0x1.03d5bep+0f);
  std::printf("worst 2^%.2f, %ld wrong\n", std::log2(worst), wrong);
  return worst <= 0x1p-52 && wrong == 0 ? 0 : 1;
}
"""


def test_exponential_of_sigmoid_is_correctly_rounded(tmp_path):
    source = tmp_path / "check.hip"
    source.write_text(PROGRAM)
    program = tmp_path / "check"
    build = subprocess.run(
        ["/opt/rocm/bin/hipcc", "--offload-host-only", "-std=c++20", "-O2", "-ffp-contract=off",
         f"-I{ROOT / 'include'}", f"-I{ROOT / 'spar_amd' / 'csrc' / 'hip'}", str(source), "-o",
         str(program)], capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0, run.stdout[-1000:] + run.stderr[-1000:]
