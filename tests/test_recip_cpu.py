"""The reciprocal of the network's sigmoid (recip_mid, tmp_amd/csrc/mlp.hip):
two Newton steps from an approximation within one unit in the last place give
the correctly rounded 1 / x, bit for bit, for every mantissa but the all-ones
one -- there only from the rounded quotient itself; else one unit below it.
(The steps scale with x by powers of two, so one binade stands for all.)"""
import subprocess

C = r"""
#include <math.h>
#include <stdio.h>
static float step(float x, float r) { return fmaf(fmaf(-x, r, 1.0f), r, r); }
int main(void) {
  for (unsigned i = 0; i < 1u << 23; i++) {
    const float x = 1.0f + i * 0x1p-23f, q = 1.0f / x;
    const float from[3] = {nextafterf(q, 0.0f), q, nextafterf(q, 2.0f)};
    for (int j = 0; j < 3; j++) {
      const float r = step(x, step(x, from[j]));
      if (r != q) printf("%a %d %a\n", x, j - 1, (double)(r - q));
    }
  }
  return 0;
}
"""


def test_two_newton_steps_give_the_quotient(tmp_path):
    src, exe = tmp_path / "r.c", tmp_path / "r"
    src.write_text(C)
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", str(src), "-o", str(exe), "-lm"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split("\n")
    assert out == ["0x1.fffffep+0 -1 -0x1p-24", "0x1.fffffep+0 1 -0x1p-24", ""]
