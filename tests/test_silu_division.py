"""The fast division of SwiGLU's g / (1 + expf(-g)) (csrc/q3vl_device.hpp,
silu_mul_n) with a reciprocal estimate that is the correctly rounded one or an
ulp off on either side, as a hardware estimate may be: over the gates that take
it, the steps have to end in the correctly rounded quotient. The bounds are
read from the source. Host arithmetic only."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "qwen3-vl-2b-inference_amd", "csrc", "q3vl_device.hpp")

STEPS = r"""
#include <math.h>
#include <stdint.h>
#include <string.h>
static float f(uint32_t b) { float x; memcpy(&x, &b, 4); return x; }
static uint32_t u(float x) { uint32_t b; memcpy(&b, &x, 4); return b; }
/* gates with bits lo .. hi - 1 whose den, |g| lie within the bounds: how many
   come out other than rounded, the first of them in *first */
long check(uint32_t lo, uint32_t hi, float gmin, float gmax, float dmax, uint32_t *first) {
    long bad = 0;
    for (uint32_t b = lo; b != hi; ++b) {
        const float g = f(b), ag = fabsf(g), den = 1.0f + expf(-g);
        if (!(den <= dmax && ag >= gmin && ag <= gmax)) continue;
        const float want = (float)((double)g / (double)den), r1 = (float)(1.0 / (double)den);
        for (int d = -1; d <= 1; ++d) {
            float r = f(u(r1) + (uint32_t)d);
            r = fmaf(fmaf(-den, r, 1.0f), r, r);
            float q = g * r;
            q = fmaf(fmaf(-den, q, g), r, q);
            q = fmaf(fmaf(-den, q, g), r, q);
            if (u(q) != u(want)) {
                if (!bad++) *first = b;
                break;
            }
        }
    }
    return bad;
}
"""


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    d = tmp_path_factory.mktemp("silu")
    (d / "steps.c").write_text(STEPS)
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", "-o", d / "steps.so", d / "steps.c", "-lm"],
                   check=True)
    lib = ctypes.CDLL(str(d / "steps.so"))
    lib.check.restype = ctypes.c_long
    lib.check.argtypes = [ctypes.c_uint32] * 2 + [ctypes.c_float] * 3 + [ctypes.POINTER(ctypes.c_uint32)]
    return lib.check


def test_fast_division_rounds_correctly(check):
    m = re.search(r"den\[i\] <= (\S+)f && ag >= (\S+)f && ag <= (\S+)f;", open(HEADER).read())
    assert m, "the bounds of the fast division"
    dmax, gmin, gmax = (float.fromhex(x) for x in m.groups())
    bits = lambda x: int(np.float32(x).view(np.uint32))  # noqa: E731
    # den takes every value of (1, 2) and beyond between 2^-25 and 2^7: the
    # binades about 1 + expf(-g) = 2 - 2^-23 whole, of the others the edges
    # and a part from within
    spans = [(bits(2.0 ** -25), bits(2.0 ** -20))]
    spans += [(bits(2.0 ** e) + o - (1 << 14 if o == 0 else 0), bits(2.0 ** e) + o + (1 << 14))
              for e in range(-40, 62) for o in (0, 0x155555, 0x2aaaab, 0x400000, 0x6abcde)]
    for sign in (0, 1 << 31):
        for lo, hi in spans:
            first = ctypes.c_uint32()
            bad = check(lo | sign, hi | sign, gmin, gmax, dmax, ctypes.byref(first))
            assert bad == 0, f"{bad} gates, the first {float(np.uint32(first.value).view(np.float32)).hex()}"
