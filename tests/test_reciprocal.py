"""CPU test of the reciprocal the per-token quantiser multiplies by: the rounded quotient for every mantissa, from estimates
on either side of it, since what the hardware's estimate is worth beyond its stated accuracy is not relied on."""
import ctypes
import os
import subprocess

import pytest

from conftest import PKG

SOURCE = r"""
#include <stdint.h>
#include <string.h>
#include "abq_recip.h"

// mantissas, at one exponent, for which the result is not (float)(1 / s) from an estimate `ulps` off the rounded quotient
extern "C" long misses(int exponent, int ulps)
{
    long n = 0;
    for (uint32_t m = 0; m < (1u << 23); ++m) {
        uint32_t bits = (uint32_t)(exponent + 127) << 23 | m;
        float s, e;
        memcpy(&s, &bits, 4);
        const float want = (float)(1.0 / (double)s);
        memcpy(&bits, &want, 4);
        bits += (uint32_t)ulps;
        memcpy(&e, &bits, 4);
        n += abq::rounded_reciprocal(s, e) != want;
    }
    return n;
}
"""


@pytest.fixture(scope="module")
def misses(tmp_path_factory):
    d = tmp_path_factory.mktemp("recip")
    (d / "recip.cpp").write_text(SOURCE)
    out = str(d / "librecip.so")
    subprocess.check_call(["g++", "-O2", "-march=native", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(PKG, "csrc"),
                           str(d / "recip.cpp"), "-o", out])
    fn = ctypes.CDLL(out).misses
    fn.restype = ctypes.c_long
    return fn


# the scales of the quantiser lie between 1e-5 and 1e4
@pytest.mark.parametrize("exponent", [-17, -1, 0, 13])
@pytest.mark.parametrize("ulps", [-4, -1, 0, 1, 4])
def test_every_mantissa_rounds_like_the_quotient(misses, exponent, ulps):
    assert misses(exponent, ulps) == 0
