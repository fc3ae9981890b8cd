"""The compile-time unit roots of the register DFTs (``csrc/qepw_roots.h``),
compiled for the host: every root of the lengths 2 .. 16 is the double nearest
to its value."""

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "qe_python_amd" / "csrc"


def test_roots_are_correctly_rounded(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src = tmp_path / "roots.cpp"
    src.write_text("""
#include "qepw_roots.h"
#include <cstdio>
template <int M> void print() {
  constexpr qepw::UnitRoots<M> w{};
  for (int k = 0; k < M; ++k) std::printf("%d %d %a %a\\n", M, k, w.c[k], w.s[k]);
}
template <int... M> void all() { (print<M>(), ...); }
int main() { all<2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>(); }
""")
    exe = tmp_path / "roots"
    subprocess.run([cxx, "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    pi = np.longdouble("3.141592653589793238462643383279502884")
    rows = [line.split() for line in out.splitlines()]
    assert len(rows) == sum(range(2, 17))
    for m, k, c, s in rows:
        # first octant, where the 80-bit functions keep their 64 bits
        e = 8 * int(k) % (8 * int(m))
        o, j = divmod(e, int(m))
        r = pi / 4 * j / int(m)
        q = pi / 4 * (int(m) - j) / int(m)
        sr, cr, sq, cq = np.sin(r), np.cos(r), np.sin(q), np.cos(q)
        want = [(cr, sr), (sq, cq), (-sr, cr), (-cq, sq), (-cr, -sr), (-sq, -cq), (sr, -cr),
                (cq, -sq)][o]
        for got, exact in zip((float.fromhex(c), float.fromhex(s)), want):
            assert abs(np.longdouble(got) - exact) <= np.spacing(abs(np.float64(exact))) * (
                np.longdouble(0.5) + np.longdouble(2) ** -10), (m, k)
