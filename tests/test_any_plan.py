"""The tile and K slices of the any-alignment GEMM (csrc/launch_plan.h
any_plan), on shapes where the choices measured apart."""
import ctypes
import json

import pytest

from frisk_amd import runtime as rt


def plan(m, n, k, a_type, c_type, workspace=1 << 40):
    # Rows one element longer than K: no 16-byte pitch.
    d = rt.GemmDesc(m, n, k, 0, 1, a_type, a_type, c_type, 1, None, k + 1, None, k + 1, None, n, 1.0,
                    1.0, None, workspace)
    buf = ctypes.create_string_buffer(1024)
    assert rt.load().frisk_gemm_plan(ctypes.byref(d), buf, len(buf)) == rt.OK, rt.load().frisk_last_error()
    p = json.loads(buf.value)
    assert p["kernel"] == "gemm_generic"
    return p["tile_m"], p["slices"]


F16, F32, I8, FP8 = (rt.F16, rt.F16), (rt.F32, rt.F32), (rt.I8, rt.I32), (rt.E4M3, rt.BF16)


@pytest.mark.parametrize("m,n,k,types,want", [
    (1111, 3333, 1777, F16, (128, 1)),   # us 34 (64 tiles 45, two slices 40)
    (1500, 1500, 5001, F16, (128, 3)),   # 55 (unsplit 73)
    (1500, 1500, 5001, FP8, (128, 3)),   # 48 (unsplit 65)
    (1589, 256, 13953, I8, (128, 8)),    # 27 (64 tiles in two slices 34)
    (1500, 2000, 1777, F16, (128, 1)),   # 25 (64 tiles 31)
    (1024, 1024, 1001, F16, (64, 1)),    # 10 (128 tiles 21)
    (128, 4095, 4095, F32, (64, 4)),     # 48 (two slices 54)
    (200, 300, 401, F32, (64, 3)),       # 10 (unsplit 13)
    (2000, 2000, 2001, I8, (128, 1)),    # 22 (64 tiles 30)
    (5, 7, 9, F16, (64, 1))])
def test_choice(m, n, k, types, want):
    assert plan(m, n, k, *types) == want
    assert plan(m, n, k, *types, workspace=0)[1] == 1


def test_grid_holds_fewer_than_2_to_32_threads():
    # 2^24 tiles of 64 rows would be a grid of 2^32 threads.
    assert plan((1 << 30) - 1, 1, 1, *I8)[0] == 128
