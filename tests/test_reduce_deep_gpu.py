"""Axis-0 sums of many rows, bit-exact with the oracle's tree: runs and blocks
past the 256 rows a thread's short counter takes.  Of the largest, a sample of
the columns is compared (each column is a tree of its own)."""
import pytest
import torch

from frisk_amd import runtime as rt
from oracle import tileops as T
from tests.gpu_util import gen
from tests.test_tileops_gpu import TORCH, assert_same_bits, bits_of

pytestmark = pytest.mark.gpu

# (rows, cols, workspace).  Without one, 1024 >> cvb row groups of 256 rows a
# block (cols 2: 1024 groups, 5: 512, 40: 128): one row, a third and a few rows
# past whole blocks, and 32 blocks less one row; then 8192 columns, 256 strips
# of 32 groups with runs of 2^11 rows.  With one, two passes whose first runs
# 8 groups of 2^9 rows a block.
CASES = [(262145, 2, False), (174763, 5, False), (65542, 40, False), ((1 << 23) - 1, 1, False),
         (33001, 8192, False), (20501, 12000, True)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,cols,workspace", CASES, ids=lambda v: str(v))
def test_sum_over_many_rows(dtype, rows, cols, workspace):
    print(f"case deep sum {dtype} {rows}x{cols} workspace={workspace}", flush=True)
    x = torch.randn(rows, cols, generator=gen(rows), device="cuda").to(TORCH[dtype])
    pick = torch.arange(cols) if cols <= 40 else \
        torch.tensor([0, 1, 63, 64, 4093, cols // 2 + 1, cols - 2, cols - 1])
    src = x[:, pick.to(x.device)].float().cpu().numpy()
    want = T.to_bits(dtype, T.reduce(src, "sum", 0, dtype))
    out = torch.empty(cols, dtype=TORCH[dtype], device="cuda")
    rt.reduce(x, out, "sum", axis=0, workspace=workspace)
    torch.cuda.synchronize()
    assert_same_bits(dtype, bits_of(dtype, out[pick.to(x.device)].contiguous()), want)
