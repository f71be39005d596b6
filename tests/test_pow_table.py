"""The table-driven power of the contact-point solve (csrc/sq_pow.h) in a CPU
build: every table row against 50-digit arithmetic, the stated error over every
slice of the mantissa, and the ends of q_pow."""
import ctypes
import decimal
import os
import re
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "liggghts-public_amd", "csrc")
SHIM = """#pragma once
#include <cmath>
#include <cstring>
#define __device__
#define __forceinline__ inline
struct Idx { unsigned x; };
static Idx threadIdx = {0}, blockDim = {1};
static void __syncthreads() {}
using std::fma; using std::rint; using std::ldexp; using std::fabs;
static long long __double_as_longlong(double v) { long long b; memcpy(&b, &v, 8); return b; }
static double __hiloint2double(int hi, int lo) {
  const long long b = ((long long)hi << 32) | (unsigned)lo;
  double v; memcpy(&v, &b, 8); return v;
}
"""
MAIN = """#include "sq_pow.h"
extern "C" void powers(long n, const double *x, const double *y, double *raw, double *q) {
  static sqd::PowTab t;
  sqd::load_pow_tab(t);
  for (long k = 0; k < n; k++) {
    if (raw) raw[k] = sqd::pow_tab(t, x[k], y[k]);
    if (q) q[k] = sqd::q_pow(t, x[k], y[k]);
  }
}
"""


@pytest.fixture(scope="module")
def powers(tmp_path_factory):
    d = tmp_path_factory.mktemp("pow")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(SHIM)
    (d / "main.cpp").write_text(MAIN)
    so = str(d / "pow.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-ffp-contract=off", "-w", f"-I{d}",
                           f"-I{CSRC}", str(d / "main.cpp"), "-o", so])
    lib = ctypes.CDLL(so)
    dp = ctypes.POINTER(ctypes.c_double)

    def call(x, y, raw=True):
        x, y = (np.ascontiguousarray(a, dtype=np.float64) for a in np.broadcast_arrays(x, y))
        out = np.empty(x.size)
        p = [a.ctypes.data_as(dp) for a in (x, y, out)]
        lib.powers(ctypes.c_long(x.size), p[0], p[1], p[2] if raw else None, None if raw else p[2])
        return out

    return call


def _table(name):
    with open(os.path.join(CSRC, "sq_pow.h")) as f:
        body = re.search(name + r"\[[^\]]*\] = \{(.*?)\};", f.read(), re.S).group(1)
    return [float.fromhex(v) if "x" in v else float(v) for v in body.replace("\n", " ").split(",") if v.strip()]


def test_table_rows():
    with decimal.localcontext() as c:
        c.prec = 50
        D, ln2 = decimal.Decimal, decimal.Decimal(2).ln()
        rows = np.reshape(_table("kPowLog"), (128, 4))
        for i, (inv, head, rest, pad) in enumerate(rows):
            m = D(1) if i == 0 else (D(2) if i == 127 else 1 + (D(i) + D("0.5")) / 128)
            assert D(inv) == D(float(1 / m)) and pad == 0.0, i
            assert (head * 2.0 ** 42).is_integer(), i
            assert abs(D(head) + D(rest) + D(inv).ln() / ln2) < D(2) ** -94, i
        for j, (head, rest) in enumerate(np.reshape(_table("kPowExp"), (64, 2))):
            exact = ((D(j) / 64) * ln2).exp()
            assert D(head) == D(float(exact)) and abs(D(head) + D(rest) - exact) < D(2) ** -104, j


def _ulps(got, x, y):
    exact = np.longdouble(x) ** np.longdouble(y)  # 64-bit significand: 2^-11 of a unit here
    return float((np.abs(np.longdouble(got) - exact) / np.spacing(np.abs(exact.astype(np.float64)))).max())


def test_error(powers):
    """The exponents the solve raises to are a blockiness less two (0 to 6 for
    blockiness 2 to 8), n1 / n2 and that less two (-1.75 to 4)."""
    assert np.finfo(np.longdouble).nmant >= 63
    rng = np.random.default_rng(1)
    # every slice of the mantissa with its ends, over the bases' whole range
    slices = 1.0 + (np.arange(128)[:, None] + np.linspace(0.0, 1.0, 9)[None, :-1]) / 128
    edges = np.concatenate([slices.ravel(), np.nextafter(slices[:, 0], 0.0)[1:]])
    edges = (edges[:, None] * 2.0 ** np.arange(-39, 10)[None]).ravel()
    for lo, hi, bound in ((-2.0, 6.0, 0.52), (-20.0, 20.0, 0.55)):
        x = np.concatenate([np.repeat(edges, 4), np.exp(rng.uniform(np.log(1e-12), np.log(1e3), 600_000))])
        y = rng.uniform(lo, hi, x.size)
        y[::7] = rng.integers(int(lo), int(hi) + 1, y[::7].size)
        y[::11] = np.round(2.0 * y[::11]) / 2.0
        worst = _ulps(powers(x, y), x, y)
        print(f"exponents {lo} to {hi}: {worst:.4f} units in the last place")
        assert worst <= bound


def test_ends(powers):
    q = lambda x, y: powers(np.float64(x), np.float64(y), raw=False)[0]  # noqa: E731
    assert q(0.0, 1.5) == q(9e-13, 0.5) == q(1e-320, 3.0) == 0.0
    assert q(0.0, 0.0) == q(5.0, 1e-13) == q(1e-320, 0.0) == 1.0  # a zero exponent first
    assert q(1.0, 3.7) == q(1.0 + 5e-13, -2.0) == q(1.0 - 5e-13, 6.0) == 1.0
    assert q(1e301, 2.0) == np.inf and q(np.inf, 1.5) == np.inf
    assert q(1e301, -2.0) == q(np.inf, -1.0) == 0.0
    assert np.isnan(q(np.nan, 2.0)) and np.isnan(q(np.nan, -2.0))
    assert q(2e-12, 2.0) == pytest.approx(4e-24, rel=1e-15)
    assert q(9e299, 1.0) == pytest.approx(9e299, rel=1e-15)
