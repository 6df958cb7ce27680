"""The logarithmic means of the FP64 flux_ranocha lines (csrc/log_mean.hpp), compiled for the host, against
values in 60 digits. The device takes the same operations, with its own reciprocal."""
import ctypes
import os
import subprocess
from decimal import Decimal, getcontext

import numpy as np
import pytest

from conftest import PKG

getcontext().prec = 60
UNIT = 2.0 ** -53

SOURCE = r"""
#include "log_mean.hpp"
using namespace trixi_hip;
static double rcp(double x) { return 1.0 / x; }
extern "C" {
// pairs of nodes (density, temperature); the element's first node is r0, t0
void means(int n, const double *rl, const double *rr, const double *tl, const double *tr, const double *r0,
           const double *t0, double *rho, double *inv, double *rho_series, double *inv_series) {
  for (int i = 0; i < n; ++i) {
    double a, b, c, d;
    node_logs(rl[i], tl[i], r0[i], t0[i], rcp, a, b);
    node_logs(rr[i], tr[i], r0[i], t0[i], rcp, c, d);
    const double x = 0.5 * rl[i], y = 0.5 * rr[i], s = 0.5 * tl[i], t = 0.5 * tr[i];
    log_means<true, false>(x, y, s, t, c - a, d - b, rcp, rho[i], inv[i]);
    log_means<false, false>(x, y, s, t, 0.0, 0.0, rcp, rho_series[i], inv_series[i]);
  }
}
void logs(int n, const double *x, const double *x0, double *out) {
  for (int i = 0; i < n; ++i) {
    double other;
    node_logs(x[i], 1.0, x0[i], 1.0, rcp, out[i], other);
  }
}
int series(int which, double *c) {
  int n = 0;
  if (which == 0) for (double x : MeanSeries::s) c[n++] = x;
  if (which == 1) for (double x : MeanSeries::r) c[n++] = x;
  if (which == 2) for (double x : LogSeries::p) c[n++] = x;
  return n;
}
double max_f() { return MeanSeries::max_f; }
unsigned max_spread() { return MeanSeries::max_spread; }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("log_mean")
    (d / "t.cpp").write_text(SOURCE)
    so = str(d / "t.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas",
                    "-I" + os.path.join(PKG, "csrc"), "-shared", "-fPIC", "-o", so, str(d / "t.cpp")], check=True)
    L = ctypes.CDLL(so)
    L.max_f.restype = ctypes.c_double
    return L


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def means(lib, rl, rr, tl, tr, r0, t0):
    a = [np.ascontiguousarray(x, dtype=np.float64) for x in (rl, rr, tl, tr, r0, t0)]
    out = [np.empty(len(a[0])) for _ in range(4)]
    lib.means(len(a[0]), *[ptr(x) for x in a], *[ptr(x) for x in out])
    return out


def exact_means(x, y):
    """ln_mean(x, y) and x y / ln_mean(x, y) of two floats."""
    x, y = Decimal(float(x)), Decimal(float(y))
    if x == y:
        return x, x
    m = (y - x) / (y / x).ln()
    return m, x * y / m


def draw(rng, n, lo, hi, scale):
    """Pairs a factor 1 + lo .. 1 + hi apart and a first node between the two and a bit beyond."""
    x = scale * rng.uniform(0.5, 2.0, n)
    y = x * (1 + lo * (hi / lo) ** rng.uniform(size=n))
    first = x * (y / x) ** rng.uniform(-0.2, 1.2, n)
    swap = rng.uniform(size=n) < 0.5
    return np.where(swap, y, x), np.where(swap, x, y), first


# In units of 2^-53. Series: the sum of the two values and the last multiply-add, two roundings, rms 0.43 each of a
# value whose mantissa is spread evenly over its logarithm, 0.60 together, largest 2; the series' own part is
# below 5 % of the mean, with a few roundings of its own.
NEAR_RMS, NEAR_MAX = 0.75, 2.25
# Logarithms: y - x, the corrected quotient, the difference of the logarithms 1 each at most; each
# logarithm |l| / |L| <= 1.2 of its own rounding and 2.5 of s on at most 0.41 / 0.53 of L; the
# temperature's product and its last product 1 each.
FAR_MAX, FAR_RMS = 13.0, 2.5


@pytest.mark.parametrize("scale", [1.0, 1e-7, 1e5])
@pytest.mark.parametrize("lo,hi", [(1e-12, 1e-9), (1e-9, 1e-4), (1e-4, 0.02), (0.02, 0.1), (0.1, 0.69),
                                   (0.71, 3.0), (3.0, 100.0), (100.0, 1e8)])
def test_means_against_exact_values(lib, lo, hi, scale):
    rng = np.random.default_rng(int(1e6 * hi) % 1000003)
    n = 1500
    rl, rr, r0 = draw(rng, n, lo, hi, scale)
    tl, tr, t0 = draw(rng, n, lo, hi, 1.0 / scale)
    rho, inv, _, _ = means(lib, rl, rr, tl, tr, r0, t0)
    e_rho = np.array([float((Decimal(float(a)) - m) / m) for a, m in zip(rho, (exact_means(x, y)[0] for x, y in zip(rl, rr)))])
    e_inv = np.array([float((Decimal(float(a)) - m) / m) for a, m in zip(inv, (exact_means(x, y)[1] for x, y in zip(tl, tr)))])
    near = hi < 0.7
    for name, e in (("density", e_rho / UNIT), ("temperature", e_inv / UNIT)):
        rms, big = float(np.sqrt(np.mean(e * e))), float(np.max(np.abs(e)))
        print(f"{name} 1+[{lo:g}, {hi:g}] scale {scale:g}: rms {rms:.2f} largest {big:.2f}")
        assert rms < (NEAR_RMS if near else FAR_RMS)
        assert big < (NEAR_MAX if near else FAR_MAX)


def test_equal_values_give_themselves(lib):
    x = np.random.default_rng(3).uniform(1e-3, 1e3, 500)
    t = x[::-1].copy()
    for out, ref in zip(means(lib, x, x, t, t, x, t), (x, t, x, t)):
        assert np.array_equal(out, ref)


def test_range_is_taken_alike_on_both_paths(lib):
    """A pair in the range of the series: the same bits with and without logarithms, up to its limit; the
    high-word bound of a line keeps every pair within it."""
    rng = np.random.default_rng(4)
    f = lib.max_f()
    ratio = (1 + f) / (1 - f)
    x = rng.uniform(0.5, 2.0, 4000)
    y = x * ratio ** rng.uniform(0.0, 1 - 1e-9, 4000)
    swap = rng.uniform(size=4000) < 0.5
    x, y = np.where(swap, y, x), np.where(swap, x, y)
    rho, inv, rho_s, inv_s = means(lib, x, y, y, x, x, y)
    assert np.array_equal(rho, rho_s) and np.array_equal(inv, inv_s)
    words = (np.stack([x, y]).view(np.uint64) >> 32).astype(np.int64)
    allowed = np.abs(words[1] - words[0]) <= lib.max_spread()
    assert np.all(np.abs(y - x)[allowed] <= f * (x + y)[allowed])
    assert np.mean(allowed) > 0.5
    # the worst case of the bound: the smaller value at the start of a binade
    top = np.array([1.0]).view(np.uint64) + ((np.uint64(lib.max_spread()) << np.uint64(32)) | np.uint64(0xffffffff))
    q = float(top.view(np.float64)[0])
    assert (q - 1) / (q + 1) <= f


@pytest.mark.parametrize("which,stated", [(0, 1.3e-17), (1, 1.1e-17), (2, 7.6e-19)])
def test_series_coefficients(lib, which, stated):
    """Largest relative error of m (1 + z S), m (1 + z R) and 1 + z P over their range, from the coefficients as
    they are: one that is off in its last places shows."""
    c = (ctypes.c_double * 32)()
    c = [Decimal(v) for v in c[:lib.series(which, c)]]
    top = Decimal("0.2") if which == 2 else Decimal("0.7") / Decimal("2.7")
    top = top * top
    worst = Decimal(0)
    for i in range(1, 301):
        z = top * i / 300
        f = z.sqrt()
        at = ((1 + f) / (1 - f)).ln() / 2 / f  # atanh(f) / f
        exact = (1 / at, (1 - z) * at, at)[which]
        s = Decimal(0)
        for v in reversed(c):
            s = s * z + v
        worst = max(worst, abs((1 + z * s) / exact - 1))
    print(f"series {which}: {len(c)} coefficients, largest error {float(worst):.3g}")
    assert worst < Decimal(stated)


def test_node_logs(lib):
    """ln(x / x0), its rounding that of the larger of 1 and itself; NaN for what has no logarithm."""
    rng = np.random.default_rng(5)
    x0 = 10.0 ** rng.uniform(-200, 200, 3000)
    x = x0 * 10.0 ** (rng.uniform(-8, 8, 3000) * rng.integers(0, 2, 3000)) * rng.uniform(0.6, 1.6, 3000)
    out = np.empty_like(x)
    lib.logs(len(x), ptr(x), ptr(x0), ptr(out))
    ref = [(Decimal(float(a)) / Decimal(float(b))).ln() for a, b in zip(x, x0)]
    # e ln 2 + 2 atanh(s): the sum's rounding, and 4 units of s <= 0.2
    err = np.array([float(abs(Decimal(float(a)) - r)) / (UNIT * (abs(float(r)) + 2.0)) for a, r in zip(out, ref)])
    print(f"largest error {err.max():.2f}")
    assert err.max() < 2.0
    bad = np.array([0.0, -0.0, -1.0, np.nan, np.inf, -np.inf, 1e-310])
    out = np.empty_like(bad)
    lib.logs(len(bad), ptr(bad), ptr(np.ones_like(bad)), ptr(out))
    assert np.all(np.isnan(out))
    one = np.full(len(bad), 2.5)  # a first node without a logarithm stands as 1 (and its low word)
    lib.logs(len(bad), ptr(one), ptr(bad), ptr(out))
    assert np.all(np.abs(out - np.log(2.5)) < 1e-8)
