"""gelu_erf (csrc/cfh_common.h), the GELU of the flow and VAE epilogues, on the CPU: its source compiled
for the host with the two hardware instructions as C functions, against erfc in double."""
from __future__ import annotations

import ctypes as C
import math
import re
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

SOURCE = (Path(__file__).resolve().parents[1] / "chain-flow_amd" / "csrc" / "cfh_common.h").read_text()
BODY = re.search(r"__device__ __forceinline__ float gelu_erf\(float x\) \{.*?\n\}\n", SOURCE, re.S).group(0)


def _exact(x):
    """x Phi(x) in double: the tail Phi(-|x|) = erfc(|x| / sqrt 2) / 2 keeps its relative precision."""
    tail = np.array([0.5 * math.erfc(abs(v) / math.sqrt(2)) for v in x])
    return np.where(x < 0, x * tail, x * (1 - tail))


@pytest.fixture(scope="module")
def gelu(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    assert cxx, "a host C++ compiler"
    d = tmp_path_factory.mktemp("gelu")
    (d / "gelu.cpp").write_text(
        "#include <math.h>\n#define __device__\n#define __forceinline__ static inline\n"
        "static float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }\n"
        "static float __builtin_amdgcn_exp2f(float x) { return exp2f(x); }\n" + BODY +
        'extern "C" void gelu(const float* x, float* y, int n) { for (int i = 0; i < n; ++i) y[i] = gelu_erf(x[i]); }\n')
    subprocess.run([cxx, "-O2", "-ffp-contract=off", "-shared", "-fPIC", str(d / "gelu.cpp"), "-o", str(d / "gelu.so")],
                   check=True)
    fn = C.CDLL(str(d / "gelu.so")).gelu

    def call(x):
        x = np.ascontiguousarray(x, dtype=np.float32)
        y = np.empty_like(x)
        p = C.POINTER(C.c_float)
        fn(x.ctypes.data_as(p), y.ctypes.data_as(p), len(x))
        return y
    return call


def test_gelu_polynomial_error():
    """The coefficients as written: t P(t) exp(-x^2 / 2) within 5.3e-8 relative of Phi(-x) for 0 <= x <= 13.4."""
    co = [float(v) for v in re.findall(r"(?:float p = |fmaf\(p, t, )(-?[0-9.]+)f", BODY)]
    scale = float(re.search(r"fmaf\(([0-9.]+)f, fabsf\(x\), 1\.0f\)", BODY).group(1))
    assert len(co) == 9
    x = np.linspace(0, 13.4, 20001)
    t = 1 / (1 + float(np.float32(scale)) * x)
    p = np.zeros_like(x)
    for c in co:
        p = p * t + float(np.float32(c))
    tail = np.array([0.5 * math.erfc(v / math.sqrt(2)) for v in x])
    assert np.abs(p * t * np.exp(-x * x / 2) / tail - 1).max() <= 5.3e-8


def test_gelu_in_float32(gelu):
    """In float32 over |x| <= 13.4.  Error: the exponent x^2 / 2 log2(e) <= 130 carries two roundings of
    2^-24 (its square, its scaling) and one of the constant, 130 * 3 * 2^-24 * ln 2 = 1.6e-5 relative in the
    tail at the far end, 1e-6 of it elsewhere from t, the ten-term polynomial and the product; below 0 that
    is relative to the result, above 0 to x times the tail, plus the last two roundings of x (1 - q).  Where
    exp(-x^2 / 2) or its product is subnormal each is off by up to half its step, 2^-149, times x."""
    x = np.linspace(-13.4, 13.4, 200001).astype(np.float32)
    x64 = x.astype(np.float64)
    tail = np.abs(x64) * np.array([0.5 * math.erfc(abs(v) / math.sqrt(2)) for v in x64])
    rel = 3 * 2.0 ** -24 * math.log(2) * x64 ** 2 * 0.7213475 + 1e-6
    bound = rel * tail + np.where(x > 0, 2 * 2.0 ** -24 * np.abs(x64), 0) + 2.0 ** -149 * (1 + np.abs(x64))
    assert (np.abs(gelu(x).astype(np.float64) - _exact(x64)) <= bound).all()


def test_gelu_rounded_to_fp16(gelu):
    """Every finite fp16 x: the fp16-rounded result is the exact value's for all but 0.02%."""
    x = np.arange(-2 ** 15, 2 ** 15).astype(np.int16).view(np.float16)
    x = x[np.isfinite(x)].astype(np.float32)
    got, ref = gelu(x).astype(np.float16), _exact(x.astype(np.float64)).astype(np.float16)
    assert (got != ref).mean() <= 2e-4


def test_gelu_of_infinities_nan_and_the_largest_values(gelu):
    """As x Phi(x) by 0.5 x (1 + erff): +inf stays, -inf gives -inf * 0 = NaN, NaN stays; past the tail's
    range x or zero."""
    y = gelu([np.inf, -np.inf, np.nan, 65504.0, -65504.0, 3e38, -3e38, 0.0, -0.0])
    assert y[0] == np.inf and np.isnan(y[1]) and np.isnan(y[2])
    assert y[3] == 65504.0 and y[4] == 0 and y[5] == np.float32(3e38) and y[6] == 0 and y[7] == 0 and y[8] == 0
