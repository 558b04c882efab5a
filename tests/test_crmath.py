"""The FP64 step's exp, log and pow (tempo_amd/csrc/tempo_crmath.hpp), built
for the host: every result within half a unit in the last place (plus the
2^-20 of one that a relative error of 2^-73 allows) of the value that 60
decimal digits give, over the arguments the step uses and the ends of the
range; special arguments as IEEE 754 has them."""
import ctypes
import math
import os
import shutil
import subprocess
from decimal import Decimal, localcontext

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
EXPONENTS = (1.0, 2.0, 3.0, 4.0, 7.0, 2.5, 3.5, -3.5, -3.0, -4.0, -5.0, -7.0, 1.0 / 3.0)
SHIM = """
#include "tempo_crmath.hpp"
using namespace tempo::crm;
extern "C" void shim(int what, const double* x, const double* y, double* out, int n) {
  for (int i = 0; i < n; ++i) switch (what) {
    case 0: out[i] = exp_cr(x[i]); break;
    case 1: out[i] = log_cr(x[i]); break;
    case 2: out[i] = log10_cr(x[i]); break;
    case 3: out[i] = pow_cr(x[i], y[i]); break;
    case 4: out[i] = pow_cr(10.0, y[i]); break;
%s
  }
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("crmath")
    src = d / "shim.cpp"
    src.write_text(SHIM % "\n".join(f"    case {10 + k}: out[i] = pow_cr(x[i], {e!r}); break;"
                                    for k, e in enumerate(EXPONENTS)))
    lib = d / "shim.so"
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-w",
                    f"-I{os.path.join(ROOT, 'tempo_amd', 'csrc')}", str(src), "-o", str(lib)], check=True)
    f = ctypes.CDLL(str(lib)).shim

    def call(what, x, y):
        x, y = (np.ascontiguousarray(np.broadcast_to(v, np.broadcast(x, y).shape), dtype=np.float64) for v in (x, y))
        out = np.empty_like(x)
        p = ctypes.POINTER(ctypes.c_double)
        f(what, x.ctypes.data_as(p), y.ctypes.data_as(p), out.ctypes.data_as(p), x.size)
        return out
    return call


def check(got, want):
    """got (floats) within (1/2 + 2^-20) ulp of want (Decimals)"""
    worst = 0.0
    with localcontext() as c:
        c.prec = 60
        for g, w in zip(got, want):
            ulp = Decimal(math.ulp(float(w))) if float(w) else Decimal(5e-324)
            worst = max(worst, float(abs(Decimal(float(g)) - w) / ulp))
    assert worst <= 0.5 + 2.0 ** -20, worst


N = 1500


def arguments(rng):
    return np.concatenate([np.exp(rng.uniform(-40, 40, N)), 1.0 + rng.uniform(-1e-3, 1e-3, N // 4),
                           1.0 + rng.uniform(-1, 1, N // 4) * 10.0 ** rng.uniform(-15, -4, N // 4)])


def decimals(f, *args):
    with localcontext() as c:
        c.prec = 60
        return [f(*(Decimal(float(v)) for v in a)) for a in zip(*args)]


def test_exp_log(shim):
    rng = np.random.default_rng(1)
    x = np.concatenate([rng.uniform(-700, 700, N), rng.uniform(-1, 1, N) * 10.0 ** rng.uniform(-18, 0, N)])
    check(shim(0, x, 0.0), decimals(lambda v: v.exp(), x))
    x = arguments(rng)
    check(shim(1, x, 0.0), decimals(lambda v: v.ln(), x))
    check(shim(2, x, 0.0), decimals(lambda v: v.log10(), x))


def test_pow(shim):
    rng = np.random.default_rng(2)
    x = arguments(rng)
    y = rng.uniform(-8, 8, x.size)
    check(shim(3, x, y), decimals(lambda v, w: (v.ln() * w).exp(), x, y))
    y = rng.uniform(-30, 30, N)
    check(shim(4, 10.0, y), decimals(lambda w: (Decimal(10).ln() * w).exp(), y))


@pytest.mark.parametrize("k", range(len(EXPONENTS)))
def test_pow_known_exponent(shim, k):
    rng = np.random.default_rng(10 + k)
    x = arguments(rng)
    check(shim(10 + k, x, 0.0), decimals(lambda v: (v.ln() * Decimal(EXPONENTS[k])).exp() if v != 1 else v, x))


def test_special_arguments(shim):
    inf, nan = math.inf, math.nan
    xs = [0.0, 1.0, 2.0, 0.5, -2.0, -1.0, -0.5, inf, -inf, nan, 5e-324, 1e-310, 1e300, -0.0]
    ys = [0.0, 1.0, 2.0, 3.0, -1.0, -2.0, 0.5, -0.5, inf, -inf, nan, 1100.0, -1100.0]
    x, y = (np.array(v).ravel() for v in np.meshgrid(xs, ys))
    with np.errstate(all="ignore"):
        want = np.power(x, y)
        np.testing.assert_allclose(shim(3, x, y), want, rtol=1e-15, atol=0)
        assert np.array_equal(np.signbit(shim(3, x, y))[~np.isnan(want)], np.signbit(want)[~np.isnan(want)])
        x = np.array(xs + [-1e-3, 710.0, -710.0, 746.0, -746.0, 800.0])
        np.testing.assert_allclose(shim(0, x, 0.0), np.exp(x), rtol=1e-15, atol=5e-324)
        np.testing.assert_allclose(shim(1, x, 0.0), np.log(x), rtol=1e-15, atol=0)
        np.testing.assert_allclose(shim(2, x, 0.0), np.log10(x), rtol=1e-15, atol=0)
        for k, e in enumerate(EXPONENTS):
            x = np.array([0.0, inf, 1.0, 1e-300, 1e300, nan])
            np.testing.assert_allclose(shim(10 + k, x, 0.0), np.power(x, e), rtol=1e-15, atol=5e-324)


@pytest.mark.parametrize("k", range(len(EXPONENTS)))
def test_pow_known_exponent_whole_range(shim, k):
    """arguments from the smallest to the largest for which the power is a
    normal number"""
    rng = np.random.default_rng(30 + k)
    e = EXPONENTS[k]
    ends = sorted((708.0 / abs(e) if abs(e) > 1 else 708.0, 60.0 * math.log(10.0), 250.0 * math.log(10.0) / abs(e)))
    lx = np.concatenate([rng.uniform(-ends[-1], ends[-1], N)] + [s * v + rng.uniform(-1, 1, 50) for v in ends[:-1] for s in (-1, 1)])
    lx = lx[np.abs(lx * e) < 708.0]
    x = np.exp(np.clip(lx, -708.0, 709.0))
    check(shim(10 + k, x, 0.0), decimals(lambda v: (v.ln() * Decimal(e)).exp(), x))
