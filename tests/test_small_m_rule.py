"""Which 8-bit GEMMs of few rows run on the small-M kernel: those on which it
measured faster than the tiled kernels (csrc/launch_plan.h skinny8_faster)."""
import ctypes
import json

import pytest

from frisk_amd import runtime as rt


def kernel(m, n, k, a_type):
    out = rt.I32 if a_type == rt.I8 else rt.BF16
    d = rt.GemmDesc(m, n, k, 0, 1, a_type, a_type, out, 1, None, k, None, k, None, n, 1.0, 1.0)
    buf = ctypes.create_string_buffer(1024)
    assert rt.load().frisk_gemm_plan(ctypes.byref(d), buf, len(buf)) == rt.OK, rt.load().frisk_last_error()
    return json.loads(buf.value)["kernel"]


@pytest.mark.parametrize("a_type", [rt.E4M3, rt.I8], ids=["fp8", "int8"])
@pytest.mark.parametrize("m,n,k,small", [
    (64, 4096, 4096, True), (64, 4096, 64, True), (32, 8192, 8192, True), (64, 8192, 8192, True),
    (64, 8192, 256, False), (16, 14336, 4096, True), (32, 14336, 4096, True), (32, 14336, 512, False),
    (33, 14336, 4096, False), (64, 14336, 16384, False), (16, 16384, 64, True), (1, 16400, 4096, False),
    (8, 28672, 4096, True), (8, 28672, 2048, False), (16, 28672, 4096, False), (16, 32768, 64, True),
    (32, 32768, 4096, True), (33, 32768, 4096, False), (16, 57344, 8192, True), (32, 57344, 8192, False), (65, 4096, 4096, False)])
def test_kernel_of_few_rows(m, n, k, a_type, small):
    assert (kernel(m, n, k, a_type) == "gemm_skinny") == small
