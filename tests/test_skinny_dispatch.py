"""The few-row GEMM's predicate and its launcher agree: whatever
gemm_skinny_serves admits has a kernel. Host code only: without a device the
launcher comes as far as the runtime's own error, and hipErrorInvalidValue is
its refusal of a shape."""
import ctypes

import pytest

import q3vl_int8 as q

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="would launch (the addresses are not real)")

INVALID_VALUE = 1  # hipErrorInvalidValue


class Seg(ctypes.Structure):
    _fields_ = [("W", ctypes.c_void_p), ("S", ctypes.c_void_p), ("C", ctypes.c_void_p), ("N", ctypes.c_int)]


class SkinnyArgs(ctypes.Structure):  # GemmSkinnyArgs, csrc/q3vl_kernels.hpp
    _fields_ = [("A", ctypes.c_void_p), ("Af", ctypes.c_void_p), ("asf", ctypes.c_void_p), ("seg", Seg * 3),
                ("nseg", ctypes.c_int), ("M", ctypes.c_int), ("K", ctypes.c_int)]


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("form", ["fp32", "fragments", "swiglu"])
def test_every_admitted_shape_has_a_kernel(form, gs):
    lib = q.lib()
    serves = lib._ZN4q3vl18gemm_skinny_servesEiiibb
    serves.restype = ctypes.c_bool
    serves.argtypes = [ctypes.c_int] * 3 + [ctypes.c_bool] * 2
    launch = lib._ZN4q3vl18launch_gemm_skinnyERKNS_14GemmSkinnyArgsEibP12ihipStream_t
    launch.argtypes = [ctypes.POINTER(SkinnyArgs), ctypes.c_int, ctypes.c_bool, ctypes.c_void_p]
    fp32, swiglu = form != "fragments", form == "swiglu"
    p, bad, n = 1 << 20, [], 0
    for M in range(1, 20):
        for K in range(64, 8193, 64):
            if not serves(M, K, gs, fp32, swiglu):
                continue
            n += 1
            a = SkinnyArgs(A=p if fp32 else None, Af=None if fp32 else p, asf=None if fp32 else p,
                           nseg=2 if swiglu else 1, M=M, K=K)
            for s in a.seg:
                s.W, s.S, s.C, s.N = p, p, p, 16
            if launch(ctypes.byref(a), gs, swiglu, None) == INVALID_VALUE:
                bad.append((M, K))
    assert n > 100 and not bad, f"{len(bad)} admitted shapes without a kernel: {bad[:10]}"
