"""The register-level DFTs of the FFT passes, compiled for the host: every
radix against a direct sum, in FP64 and FP32."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pawpyseed_amd", "csrc")
RADICES = (2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16, 18, 20, 25)

MAIN = """
#include "pp_dft.h"
#include <cmath>
#include <cstdio>
template <typename T, int R> double worst() {
  double w = 0;
  for (int one = 0; one < R; one++) {
    cplx<T> v[R];
    double in[R][2];
    for (int i = 0; i < R; i++) {  // distinct values, a unit vector's weight on one
      in[i][0] = (T)(std::sin(1.0 + i * 0.7) + (i == one ? 3.0 : 0.0));
      in[i][1] = (T)std::cos(2.0 + i * 1.3);
      v[i] = mk<T>((T)in[i][0], (T)in[i][1]);
    }
    pp::Dft<T, R>::run(v);
    double d2 = 0, n2 = 0;
    for (int k = 0; k < R; k++) {
      long double re = 0, im = 0;
      for (int i = 0; i < R; i++) {
        const long double a = 2 * M_PIl * ((i * k) % R) / R;
        re += in[i][0] * std::cos(a) - in[i][1] * std::sin(a);
        im += in[i][0] * std::sin(a) + in[i][1] * std::cos(a);
      }
      d2 += (v[k].x - re) * (v[k].x - re) + (v[k].y - im) * (v[k].y - im);
      n2 += re * re + im * im;
    }
    w = std::fmax(w, std::sqrt(d2 / n2));
  }
  return w;
}
int main() {
#define ROW(R) std::printf("%d %.3e %.3e\\n", R, worst<double, R>(), worst<float, R>());
  ROWS
}
"""


def test_register_dfts(tmp_path):
    """A radix-R DFT of two nested ones rounds by a few units of 1.1e-16
    (6e-8), normwise; a wrong root or sign gives an error of order one."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src = tmp_path / "dft.hip"
    src.write_text(MAIN.replace("ROWS", " ".join(f"ROW({r})" for r in RADICES)))
    exe = str(tmp_path / "dft")
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-I", CSRC, str(src), "-o", exe], check=True,
                   capture_output=True)
    rows = [line.split() for line in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert [int(r[0]) for r in rows] == list(RADICES)
    for r, d, f in rows:
        assert float(d) < 5e-16 and float(f) < 3e-7, (r, d, f)
