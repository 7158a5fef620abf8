"""The any-alignment MFMA GEMM (frisk_gemm's route for element-aligned
operands, odd pitches and ragged K) against the fp64 / exact oracle.

Operands are views at an odd element offset and an odd pitch of buffers
filled with NaN (int8: 127), so an element read past a row, past K or past
the matrix shows in the result; outputs are views too, and what lies around
them must not change.  Tolerances are those of the aligned kernels' parity
tests: one rounding to the output type of an f32 sum."""
import itertools

import numpy as np
import pytest
import torch

from frisk_amd import runtime as rt
from oracle import gemm as G
from tests.gpu_util import decode, gen

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
PAIRS = [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
         (torch.float16, torch.float16), (torch.float16, torch.float32),
         (FP8, torch.bfloat16), (FP8, torch.float16), (FP8, torch.float32),
         (torch.int8, torch.int32), (torch.float32, torch.float32)]
TOL = {torch.bfloat16: 1e-2, torch.float16: 1e-2, torch.float32: 1e-5}
# One element, a matrix under 16 bytes, a K inside one piece, the edges of two
# 64x64 tiles (which the plan takes for all of these; 128x128:
# test_gemm_any_tiles_gpu.py) and of the 128-byte stage (128, 64 and 32
# elements), one past them, and a K that splits (16 stages and more) with a
# partial last slice.
SHAPES = [(1, 1, 1), (2, 3, 3), (5, 7, 9), (1, 129, 31), (33, 1, 127), (127, 130, 129),
          (128, 128, 128), (129, 255, 65), (3, 70, 2100), (130, 5, 4109)]


def view(rows, cols, dt, seed, pad):
    """A [rows, cols] view at an odd offset and pitch of a poisoned buffer."""
    ld = cols + pad
    n = rows * ld + 1
    g = gen(seed)
    if dt == torch.int8:
        buf = torch.full((n,), 127, dtype=dt, device="cuda")
        x = torch.randint(-127, 128, (rows, cols), generator=g, device="cuda", dtype=dt)
    else:
        buf = torch.full((n,), float("nan"), device="cuda").to(dt)
        x = torch.randn(rows, cols, generator=g, device="cuda").to(dt)
    t = buf[1:].view(rows, ld)[:, :cols]
    t.view(torch.uint8 if dt == FP8 else dt).copy_(x.view(torch.uint8) if dt == FP8 else x)
    return buf, t


def check(got, ref, out_dt):
    if out_dt == torch.int32:
        assert np.array_equal(got, ref)
    else:
        assert np.isfinite(got).all()
        assert G.row_scaled_error(got.astype(np.float64), ref) <= TOL[out_dt]


@pytest.mark.parametrize("in_dt,out_dt", PAIRS, ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("ta,tb", list(itertools.product([False, True], repeat=2)))
def test_any_alignment_every_type_and_layout(in_dt, out_dt, ta, tb):
    for i, (m, n, k) in enumerate(SHAPES):
        print(f"case any {in_dt}->{out_dt} ta={ta} tb={tb} m={m} n={n} k={k}", flush=True)
        pad = 1 + i % 3 * 2
        _, a = view(*((k, m) if ta else (m, k)), in_dt, 10 + i, pad)
        _, b = view(*((n, k) if tb else (k, n)), in_dt, 50 + i, pad)
        cbuf = torch.full((m * (n + pad) + 1,), 77, device="cuda").to(out_dt)
        c = cbuf[1:].view(m, n + pad)[:, :n]
        assert rt.gemm_plan(a, b, c, trans_a=ta, trans_b=tb)["kernel"] == "gemm_generic"
        A, B = decode(a), decode(b)
        ref = G.gemm_int(A, B, trans_a=ta, trans_b=tb) if in_dt == torch.int8 else \
            G.gemm_fp64(A, B, trans_a=ta, trans_b=tb)
        for ws in (True, False):  # split over K where the plan splits, and unsplit
            rt.gemm(a, b, c, trans_a=ta, trans_b=tb, workspace=ws)
            torch.cuda.synchronize()
            check(decode(c), ref, out_dt)
            around = cbuf[1:].view(m, n + pad)[:, n:]
            assert bool((around == 77).all()) and float(cbuf[0]) == 77
        rt.gemm(a, b, c, trans_a=ta, trans_b=tb, clear_accum=False)
        torch.cuda.synchronize()
        if out_dt in (torch.int32, torch.float32):
            check(decode(c), 2 * ref, out_dt)


def test_any_alignment_takes_a_short_workspace():
    # The same request with a workspace too small for its split runs unsplit,
    # and without device allocation it gives the split's bits.
    m, n, k = 64, 200, 6001
    _, a = view(m, k, torch.bfloat16, 1, 1)
    _, b = view(n, k, torch.bfloat16, 2, 1)
    need = rt.gemm_workspace_bytes(a, b, torch.empty(m, n, dtype=torch.bfloat16, device="cuda"),
                                   trans_b=True)
    assert 0 < need <= rt.NOALLOC_SCRATCH_BYTES
    outs = []
    for ws in (True, False, torch.empty(need // 2, dtype=torch.uint8, device="cuda"),
               torch.empty(need + 8, dtype=torch.uint8, device="cuda")[8:]):
        c = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        rt.gemm(a, b, c, trans_b=True, workspace=ws)
        outs.append(c)
    na = torch.empty_like(outs[0])
    rt.gemm_noalloc(a, b, na, trans_b=True)
    torch.cuda.synchronize()
    assert torch.equal(outs[1], outs[2]) and torch.equal(outs[1], outs[3])
    assert torch.equal(outs[0], na)
    check(decode(outs[0]), decode(a) @ decode(b).T, torch.bfloat16)
