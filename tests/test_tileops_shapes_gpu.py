"""Tile ops at the sizes where a launch shape changes, on views at odd element
offsets and pitches, bit-exact with the oracle: rows shared by 4 or 16 waves,
axis-0 strips of one and two passes with partial runs and blocks, and copies
and fills whose short rows share a workgroup."""
import numpy as np
import pytest
import torch

from frisk_amd import runtime as rt
from oracle import tileops as T
from tests.test_tileops_gpu import (TORCH, assert_same_bits, bits_of, device_from_bits, seed_of, values)

pytestmark = pytest.mark.gpu

# Axis 1: one wave a row, four (at least 256 slots and under 2048 rows) and
# sixteen, with a partial last chunk and runs of no chunk.
ROWS = [(2100, 1500), (600, 2049), (3, 16385), (40, 28653), (1, 70001)]
# Axis 0: under 256 rows (one, a few and 32 runs of eight), two passes (partial
# last block; one block; narrow with many blocks, whose longest run without a
# workspace is 256 rows; strips that leave part of a round empty), and the same
# in one pass of 1024 threads.  (Longer runs: test_reduce_deep_gpu.py.)
COLS = [(1, 900), (26, 1433), (112, 1587), (255, 70), (256, 515), (449, 665), (17921, 9),
        (600, 12801), (3000, 12805)]


def odd_view(dtype, x):
    """x as a view one element into a buffer with an odd pitch."""
    r, c = x.shape
    buf = torch.zeros(r * (c + 3) + 1, dtype=TORCH[dtype], device="cuda")
    v = buf[1:].view(r, c + 3)[:, :c]
    v.copy_(device_from_bits(dtype, T.to_bits(dtype, x)).view(r, c))
    return v


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("kind", ["sum", "max", "min"])
@pytest.mark.parametrize("axis,shape", [(1, s) for s in ROWS] + [(0, s) for s in COLS],
                         ids=lambda v: str(v).replace(" ", ""))
def test_reduce_launch_shapes(dtype, kind, axis, shape):
    print(f"case reduce {dtype} {kind} axis{axis} {shape}", flush=True)
    src = values(dtype, shape, seed=seed_of(dtype, kind, axis, shape), specials=kind != "sum")
    want = T.to_bits(dtype, T.reduce(src, kind, axis, dtype))
    n = shape[0] if axis == 1 else shape[1]
    x = device_from_bits(dtype, T.to_bits(dtype, src)).view(shape)
    for t, ws in ((x, True), (x, False), (odd_view(dtype, src), True)):
        dst = torch.empty(n, dtype=TORCH[dtype], device="cuda")
        rt.reduce(t, dst, kind, axis=axis, workspace=ws)
        torch.cuda.synchronize()
        assert_same_bits(dtype, bits_of(dtype, dst), want, f"workspace={ws}")


@pytest.mark.parametrize("src,dst", [("f32", "bf16"), ("bf16", "f32"), ("f16", "e4m3"), ("e4m3", "f16"),
                                     ("bf16", "bf16"), ("f32", "f32"), ("e4m3", "e4m3")])
@pytest.mark.parametrize("shape", [(1, 5), (1000, 1), (130, 17), (77, 128), (9, 2048), (5, 2057), (3, 9001)],
                         ids=lambda v: str(v).replace(" ", ""))
def test_copy_and_fill_short_and_odd_rows(src, dst, shape):
    print(f"case copy {src}->{dst} {shape}", flush=True)
    r, c = shape
    bits = T.to_bits(src, values(src if src != "e4m3" else "f16", shape, seed=r + c))
    s = torch.zeros(r * (c + 3) + 1, dtype=TORCH[src], device="cuda").view(torch.uint8)
    es = s.numel() // (r * (c + 3) + 1)
    view = s.view(TORCH[src])[1:].view(r, c + 3)[:, :c]
    view.view(torch.uint8).copy_(device_from_bits(src, bits).view(r, c).view(torch.uint8)) if es == 1 else \
        view.copy_(device_from_bits(src, bits).view(r, c))
    buf = torch.full((r * (c + 5) * 4 + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    eb = torch.empty((), dtype=TORCH[dst]).element_size()
    wide = buf[:((r * (c + 5) + 1) * eb)].view(TORCH[dst])[1:].view(r, c + 5)
    out = wide[:, :c]
    rt.copy(view, out)
    torch.cuda.synchronize()
    want = T.convert(src, dst, bits) if src != dst else bits
    assert_same_bits(dst, bits_of(dst, out), want.reshape(shape))
    guard = bits_of(dst, wide)[:, c:]
    assert np.all(guard.view(np.uint8) == 0xA5)
    rt.fill(out, 1.5)
    torch.cuda.synchronize()
    assert np.all(bits_of(dst, out) == T.to_bits(dst, np.float32([1.5]))[0])
    assert np.all(bits_of(dst, wide)[:, c:].view(np.uint8) == 0xA5)
