"""The step kernels' logarithm and sine and cosine of a turn (jja_math.h), compiled for
the host with gcc, against the C library in extended precision: -log(u) within 1 ulp
over the deviates' range, sine and cosine within 1 ulp away from zeros and 2e-16 there."""
import os
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyjjasim_amd", "csrc", "jja_math.h")

PROG = r"""
#include "%s"
#include <stdio.h>
static long double ulp(long double v) { return (long double)nextafter(fabs((double)v), INFINITY) - fabs((double)v); }
int main(void) {
  unsigned long long s = 88172645463325252ULL;
  long double wl = 0, ws = 0, wa = 0;
  for (long i = 0; i < 2000000; ++i) {
    s ^= s << 13; s ^= s >> 7; s ^= s << 17;
    uint64_t a = s >> 11;
    switch (i & 7) {                                     /* small u, u near 1, near sqrt(1/2) */
      case 1: a >>= (s >> 3) %% 53; break;
      case 2: a = (1ULL << 53) - 1 - (a >> ((s >> 3) %% 53)); break;
      case 3: a = 6369051672525773ULL + (a >> 30) - (1ULL << 22); break;
      default: break;
    }
    const double u = (double)(a + 1) * 0x1p-53;
    const long double want = -logl((long double)u);
    if (want == 0) { if (jja_neg_log(u) != 0) wl = 1e9; }
    else { long double e = fabsl(jja_neg_log(u) - want) / ulp(want); if (e > wl) wl = e; }
    const double v = (double)(s >> 11) * 0x1p-53;
    double sn, cs;
    jja_sincos_turn(v, &sn, &cs);
    /* quarter turns taken off first: an angle near 2 pi has no bits left for a sine of 1e-3 */
    const int n = (int)rint(4 * v);
    const long double t = 2.0L * 3.14159265358979323846264338327950288L * ((long double)v - 0.25L * n);
    const long double S[4] = {sinl(t), cosl(t), -sinl(t), -cosl(t)}, rs = S[n & 3], rc = S[(n + 1) & 3];
    const long double es = fabsl(sn - rs), ec = fabsl(cs - rc);
    if (es > wa) wa = es;
    if (ec > wa) wa = ec;
    if (fabsl(rs) > 1e-3L && es / ulp(rs) > ws) ws = es / ulp(rs);
    if (fabsl(rc) > 1e-3L && ec / ulp(rc) > ws) ws = ec / ulp(rc);
  }
  double sn, cs;
  jja_sincos_turn(0.25, &sn, &cs);
  printf("%%.4Lf %%.4Lf %%.3Lg %%d\n", wl, ws, wa, sn == 1.0 && fabs(cs) < 1e-30);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not available")
def test_box_muller_parts_match_libm(tmp_path):
    src = tmp_path / "t.c"
    src.write_text(PROG % HEADER)
    exe = tmp_path / "t"
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", str(exe), str(src), "-lm"], check=True)
    log_ulp, turn_ulp, turn_abs, exact = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    print(log_ulp, turn_ulp, turn_abs)
    assert float(log_ulp) <= 1.0 and float(turn_ulp) <= 1.0 and float(turn_abs) <= 2e-16 and exact == "1"
