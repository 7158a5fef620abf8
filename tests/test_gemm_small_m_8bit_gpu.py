"""The small-M kernel on 8-bit inputs (M <= 64, A [M, K], B [N, K]) against
the exact integer product (int8) and the fp64 oracle (fp8, whose MFMAs align
the products of one instruction before adding them: 2e-2 of a row's largest
value, and one rounding of the output)."""
import numpy as np
import pytest
import torch

from frisk_amd import runtime as rt
from oracle import gemm as G
from tests.gpu_util import Guarded, decode, gen

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
# K inside one 16-byte piece and one 64-byte step, whole batches and a tail;
# N partial in the last tile, one round of 16-column tiles (4096), wider
# columns (8192: 32, 16328: 64); M at each tile height and one past it.  Past
# 32 rows the wide ones (24584, 8200) run on 128x128 tiles.
SHAPES = [(1, 16, 16), (5, 40, 48), (16, 4096, 1040), (17, 72, 2064), (32, 8192, 256), (33, 24584, 80),
          (64, 4096, 192), (64, 8200, 64), (16, 16328, 80), (32, 8200, 1040), (64, 8184, 1040)]


@pytest.mark.parametrize("in_dt,out_dt", [(FP8, torch.bfloat16), (FP8, torch.float16),
                                          (FP8, torch.float32), (torch.int8, torch.int32)],
                         ids=lambda x: str(x).replace("torch.", ""))
def test_small_m_8bit(in_dt, out_dt):
    for m, n, k in SHAPES:
        print(f"case small-M {in_dt}->{out_dt} m={m} n={n} k={k}", flush=True)
        g = gen(m + n + k)
        if in_dt == torch.int8:
            a, b = (torch.randint(-127, 128, (r, k), generator=g, device="cuda", dtype=in_dt) for r in (m, n))
            sa = sb = 1.0
        else:
            a, b = (torch.randn(r, k, generator=g, device="cuda").to(in_dt) for r in (m, n))
            sa, sb = 0.5, 0.25
        c = Guarded((m, (n + 15) // 16 * 16), out_dt)
        c.t.zero_()
        out = c.t[:, :n]
        kw = dict(trans_b=True, scale_a=sa, scale_b=sb)
        want = "gemm_128" if m > 32 and n >= 8200 else "gemm_skinny"
        assert rt.gemm_plan(a, b, out, trans_b=True)["kernel"] == want
        ref = G.gemm_int(decode(a), decode(b), trans_b=True) if in_dt == torch.int8 else \
            G.gemm_fp64(decode(a), decode(b), trans_b=True) * (sa * sb)
        for times in (1, 2):  # C = A.B, then C += A.B
            rt.gemm(a, b, out, clear_accum=times == 1, **kw)
            torch.cuda.synchronize()
            assert c.guards_intact() and not bool(c.t[:, n:].any())
            if in_dt == torch.int8:
                assert np.array_equal(decode(out), times * ref)
            else:
                assert G.row_scaled_error(decode(out), times * ref) <= 2e-2
