"""Device math that is plain C++, compiled for the CPU and compared with
float64 over the whole range of its argument."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "asuna_amd", "csrc")

LOG1P = r"""
#include <cmath>
#include <cstddef>
#define __host__
#define __device__
#include "device/log1p.h"
extern "C" void log1pOf(const float* x, size_t n, int off, float* y) {
  // the reciprocal, or one of its neighbours: the hardware's is within a unit of it
  auto rcp = [&](float v) {
    const float r = 1.0f / v;
    return off ? std::nextafter(r, off > 0 ? INFINITY : 0.0f) : r;
  };
  for (size_t i = 0; i < n; ++i) y[i] = ashd::log1pPos(x[i], rcp);
}
"""


@pytest.mark.parametrize("off", [-1, 0, 1])
def test_log1p_of_every_magnitude(tmp_path, off):
    """The denoiser's log(1 + x) is within 0.54 units in the last place (its
    stated bound) from 0 and the subnormal numbers to the largest finite one,
    and infinite only at infinity."""
    (tmp_path / "l.cpp").write_text(LOG1P)
    so = str(tmp_path / "l.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-o", so,
                    str(tmp_path / "l.cpp")], check=True)
    f = C.CDLL(so).log1pOf
    f.argtypes = [C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    bits = np.concatenate([np.arange(0, 0x7F800000, 997, dtype=np.uint32),       # all magnitudes
                           np.arange(0x3E000000, 0x40800000, 13, dtype=np.uint32),  # 1/8 to 4: both sides of every branch
                           np.array([0, 1, 0x7F61B1E6, 0x7F61B1E7, 0x7F7FFFFF], np.uint32)])  # ends; 3.0e38 and next
    x = bits.view(np.float32)
    y = np.empty_like(x)
    f(x.ctypes.data, x.size, off, y.ctypes.data)
    exact = np.log1p(x.astype(np.float64))
    ulp = np.maximum(np.spacing(exact.astype(np.float32)).astype(np.float64), 2.0 ** -149)
    err = np.abs(y - exact) / ulp
    worst = int(err.argmax())
    print(f"log1p: {err[worst]:.4f} units at {x[worst]:.9g}", flush=True)
    assert err[worst] <= 0.54
    inf = np.array([np.inf], np.float32)
    f(inf.ctypes.data, 1, off, y.ctypes.data)
    assert y[0] == np.inf
