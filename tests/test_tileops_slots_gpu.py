"""Copies and fills where the slots a thread takes change: one, two and four of
short rows, and rows on either side of the limit between shared workgroups and
a workgroup a row (64 slots of 8 for 4-byte elements, 128 else), with whole
and ragged last slots.  Conversions are round to nearest even, as torch's."""
import pytest
import torch

from frisk_amd import runtime as rt
from tests.gpu_util import gen

pytestmark = pytest.mark.gpu

T = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "f64": torch.float64,
     "i8": torch.int8}
# 600 columns: 2 rows a pass, so 2 x 512 (conversions) or 2 x 256 (copies) rows
# per slot a thread; 17 columns: 64 rows a pass.
SHAPES = [(3, 600), (700, 600), (2100, 600), (5001, 600), (40001, 17), (70001, 17), (140001, 17),
          (500, 504), (500, 512), (500, 513), (700, 1024), (700, 1025)]


@pytest.mark.parametrize("src,dst", [("f32", "bf16"), ("bf16", "f32"), ("f32", "f32"), ("f16", "f16"),
                                     ("i8", "i8"), ("f64", "f64"), ("bf16", "f16")])
def test_copy_slots(src, dst):
    for r, c in SHAPES:
        print(f"case slots {src}->{dst} {r}x{c}", flush=True)
        g = gen(r + c)
        x = torch.randint(-100, 100, (r, c + 3), generator=g, device="cuda", dtype=torch.int8) if src == "i8" \
            else torch.randn(r, c + 3, generator=g, device="cuda").to(T[src])
        x = x[:, 1:c + 1]
        wide = torch.full((r, c + 2), 7, device="cuda", dtype=T[dst])
        out = wide[:, 1:c + 1]
        rt.copy(x, out)
        torch.cuda.synchronize()
        assert torch.equal(out, x.to(T[dst]))
        rt.fill(out, 3.0)
        torch.cuda.synchronize()
        assert bool((out == 3).all()) and bool((wide[:, 0] == 7).all()) and bool((wide[:, c + 1] == 7).all())
