"""The any-alignment GEMM on 128x128 tiles (every type pair and layout), their
K slices, and operands that reach past 2^31 bytes, against the fp64 / exact
oracle on a sample of the rows.  Operands and outputs are views as in
test_gemm_any_gpu.py; tolerances are that file's."""
import itertools

import numpy as np
import pytest
import torch

from frisk_amd import runtime as rt
from oracle import gemm as G
from tests.gpu_util import decode, gen
from tests.test_gemm_any_gpu import FP8, PAIRS, check, view

pytestmark = pytest.mark.gpu


def sample(m):
    """Rows at the edges of the 128-row tiles and their 32-row quarters, the
    last ones, and some between."""
    edge = [r for t in range(0, m, 128) for r in (t, t + 31, t + 32, t + 63, t + 64, t + 127)]
    return sorted({r for r in edge + [m - 1, m - 2, m // 3] if 0 <= r < m})


def run(m, n, k, in_dt, out_dt, ta, tb, pad, tile, slices=None):
    print(f"case any {in_dt}->{out_dt} ta={ta} tb={tb} m={m} n={n} k={k}", flush=True)
    _, a = view(*((k, m) if ta else (m, k)), in_dt, m + k, pad)
    _, b = view(*((n, k) if tb else (k, n)), in_dt, n + k, pad)
    cbuf = torch.full((m * (n + pad) + 1,), 77, device="cuda").to(out_dt)
    wide = cbuf[1:].view(m, n + pad)
    c = wide[:, :n]
    p = rt.plan_of(rt.gemm_desc(a, b, c, trans_a=ta, trans_b=tb)) if slices is None else \
        rt.gemm_plan(a, b, c, trans_a=ta, trans_b=tb)
    assert p["kernel"] == "gemm_generic" and p["tile_m"] == tile, p
    rows = sample(m)
    pick = torch.tensor(rows, device="cuda")
    bytes_ = a.view(torch.uint8) if in_dt == FP8 else a
    part = (bytes_[:, pick] if ta else bytes_[pick]).contiguous()
    A, B = decode(part.view(FP8) if in_dt == FP8 else part), decode(b)
    ref = G.gemm_int(A, B, trans_a=ta, trans_b=tb) if in_dt == torch.int8 else \
        G.gemm_fp64(A, B, trans_a=ta, trans_b=tb)
    rt.gemm(a, b, c, trans_a=ta, trans_b=tb, workspace=slices is not None)
    torch.cuda.synchronize()
    check(decode(c[pick].contiguous()), ref, out_dt)
    if out_dt in (torch.int32, torch.float32):
        rt.gemm(a, b, c, trans_a=ta, trans_b=tb, clear_accum=False, workspace=slices is not None)
        torch.cuda.synchronize()
        check(decode(c[pick].contiguous()), 2 * ref, out_dt)
    assert bool((wide[:, n:] == 77).all()) and float(cbuf[0]) == 77
    return p


@pytest.mark.parametrize("in_dt,out_dt", PAIRS, ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("ta,tb", list(itertools.product([False, True], repeat=2)))
def test_128_tiles_every_type_and_layout(in_dt, out_dt, ta, tb):
    # One element of K, one past a 128-byte stage (f32 32, 16-bit 64, 8-bit 128
    # elements) and many stages with a ragged last one.
    for i, k in enumerate((1, 33, 65, 129, 1777)):
        run(1111, 3333, k, in_dt, out_dt, ta, tb, 1 + i % 3 * 2, 128)


@pytest.mark.parametrize("m,n,k,in_dt,out_dt", [
    (1500, 1500, 5001, torch.float16, torch.float16), (1500, 1500, 5001, torch.bfloat16, torch.float32),
    (1500, 1500, 5001, FP8, torch.bfloat16), (1589, 256, 13953, torch.int8, torch.int32),
    (256, 4097, 1111, torch.float32, torch.float32)], ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_128_tiles_in_slices(m, n, k, in_dt, out_dt, ta, tb):
    p = run(m, n, k, in_dt, out_dt, ta, tb, 1, 128, slices=True)
    assert p["slices"] > 1 and p["workspace_bytes"] > 0, p


@pytest.mark.parametrize("in_dt,out_dt", [(torch.bfloat16, torch.float32), (torch.int8, torch.int32)],
                         ids=lambda x: str(x).replace("torch.", ""))
@pytest.mark.parametrize("ta", [False, True])
def test_operand_past_2_to_31_bytes(in_dt, out_dt, ta):
    """A 16-byte aligned A whose rows lie so far apart that a tile's 32-bit
    offsets do not reach: 64-bit addresses, K-major and M-major."""
    m, n, k = (272, 48, 80) if not ta else (80, 48, 272)
    rows, cols = (k, m) if ta else (m, k)
    es = torch.empty((), dtype=in_dt).element_size()
    ld = (1 << 31) // (255 * es) // 16 * 16 + 4096
    buf = torch.empty(rows * ld, dtype=in_dt, device="cuda")
    a = buf.view(rows, ld)[:, :cols]
    g = gen(7)

    def mat(r, c):
        if in_dt == torch.int8:
            return torch.randint(-127, 128, (r, c), generator=g, device="cuda", dtype=in_dt)
        return torch.randn(r, c, generator=g, device="cuda").to(in_dt)

    a.copy_(mat(rows, cols))
    b = mat(n, k)
    c = torch.empty(m, n, dtype=out_dt, device="cuda")
    assert (rows - 1) * ld * es > 1 << 31
    assert rt.gemm_plan(a, b, c, trans_a=ta, trans_b=True)["kernel"] == "gemm_generic"
    A, B = decode(a.contiguous()), decode(b)
    ref = G.gemm_int(A, B, trans_a=ta, trans_b=True) if in_dt == torch.int8 else \
        G.gemm_fp64(A, B, trans_a=ta, trans_b=True)
    for ws in (True, False):
        c.fill_(0)
        rt.gemm(a, b, c, trans_a=ta, trans_b=True, workspace=ws)
        torch.cuda.synchronize()
        check(decode(c), ref, out_dt)
        assert np.abs(ref).max() > 0
