"""Attention with few queries (decode steps, seq_q <= 32) against the fp64
oracle: the kernel whose waves divide the keys, and its key splits over a
workspace.  Tolerances as in test_attn_gpu.py (one rounding of a probability
and one of the output)."""
import ctypes

import numpy as np
import pytest
import torch

from frisk_amd import runtime as rt
from oracle import attention as A
from oracle import gemm as G
from tests.gpu_util import Guarded, gen

pytestmark = pytest.mark.gpu

LSE_TOL = {torch.bfloat16: 4e-3, torch.float16: 1e-3}
# (batch, heads, seq_q, seq_k): fewer blocks of 64 keys than waves, one past
# and one short of a block, a whole round of blocks, more queries than keys,
# the most queries of the kernel, and lengths that split over the workspace.
# (The shortest run the query-tiled kernel, by head_dim: plan::attn_few; the
# fewest keys of this one, and more heads than one round of its workgroups.)
CASES = [(1, 1, 1, 1), (1, 2, 1, 63), (2, 1, 3, 65), (1, 3, 1, 1024), (1, 2, 32, 33), (1, 1, 32, 7),
         (2, 2, 17, 300), (1, 2, 1, 4097), (1, 1, 5, 9000), (1, 2, 32, 129), (2, 1, 32, 193), (1, 1, 1, 193),
         (3, 100, 2, 706)]


def call(q, k, v, o, lse, causal, ws, **kw):
    """frisk_attn_fwd_ws with `ws` bytes of scratch (None: frisk_attn_fwd)."""
    d = rt.attn_desc(q, k, v, o, causal=causal, lse=lse, **kw)
    lib = rt.load()
    need = lib.frisk_attn_workspace_size(ctypes.byref(d))
    assert need >= 0
    if ws is None:
        rc = lib.frisk_attn_fwd(ctypes.byref(d), None)
    else:
        buf = Guarded((max(need, 16),), torch.uint8)
        rc = lib.frisk_attn_fwd_ws(ctypes.byref(d), buf.t.data_ptr(), max(need, 16), None)
    assert rc == rt.OK, lib.frisk_last_error()
    torch.cuda.synchronize()
    assert ws is None or buf.guards_intact()
    return need


@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("kt", [False, True], ids=["k", "kt"])
def test_few_queries(d, causal, kt):
    torch.cuda.synchronize()
    split = 0
    for i, (b, h, sq, sk) in enumerate(CASES):
        dt, out = ((torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32))[i % 2]
        if kt and sk % 2:
            sk += 1
        print(f"case few queries d{d} b{b} h{h} sq{sq} sk{sk} causal={causal} kt={kt} {dt}", flush=True)
        g = gen(100 * d + i)
        q, k, v = (torch.randn(b, h, n, d, generator=g, device="cuda").to(dt) for n in (sq, sk, sk))
        ref, rlse = A.attention_fp64(q.double().cpu().numpy(), k.double().cpu().numpy(),
                                     v.double().cpu().numpy(), causal=causal, scale=d ** -0.5)
        kk = k
        if kt:  # rows of sk keys, 16-byte pitch
            pitch = (sk + 7) // 8 * 8
            kk = torch.full((b, h, d, pitch), float("nan"), device="cuda").to(dt)[..., :sk]
            kk.copy_(k.transpose(-1, -2))
        live = np.isfinite(rlse)
        for ws in (None, True):
            o, lse = Guarded((b, h, sq, d), out), Guarded((b, h, sq), torch.float32)
            split += call(q, kk, v, o.t, lse.t, causal, ws, k_transposed=kt) > 0
            assert o.guards_intact() and lse.guards_intact()
            got, l = o.t.double().cpu().numpy(), lse.t.cpu().numpy()
            if live.any():
                assert G.row_scaled_error(got[live], ref[live]) <= 1e-2
                assert np.abs(l[live] - rlse[live]).max() <= LSE_TOL[dt]
            assert np.all(got[~live] == 0) and np.all(np.isneginf(l[~live]))
    assert split > 0  # some case splits its keys


def test_few_queries_repeat_bitwise_and_through_the_binding():
    # The binding allocates the scratch; heads interleaved (BSHD) as a KV
    # cache keeps them.  Every call gives the same bits.
    q, k, v = (torch.randn(2, n, 4, 128, generator=gen(n), device="cuda").to(torch.bfloat16)
               .transpose(1, 2) for n in (1, 3000, 3000))
    outs = []
    for _ in range(3):
        o = torch.empty(2, 1, 4, 128, dtype=torch.bfloat16, device="cuda").transpose(1, 2)
        rt.attn_fwd(q, k, v, o, causal=True)
        outs.append(o)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    ref, _ = A.attention_fp64(q.double().cpu().numpy(), k.double().cpu().numpy(),
                              v.double().cpu().numpy(), causal=True, scale=128 ** -0.5)
    assert G.row_scaled_error(outs[0].double().cpu().numpy(), ref) <= 1e-2


@pytest.mark.parametrize("as_handle", [False, True])
def test_scratch_belongs_to_the_stream_of_the_call(monkeypatch, as_handle):
    """On another stream than the current one, the scratch of a call comes
    from that stream's pool: a tensor of the current stream never reuses it
    while the kernels run."""
    side = torch.cuda.Stream()
    stream = side.cuda_stream if as_handle else side
    seen, empty = [], torch.empty

    def recorded(*a, **kw):
        seen.append(torch.cuda.current_stream().cuda_stream)
        return empty(*a, **kw)

    g = gen(5)
    q = torch.randn(1, 1, 1, 128, generator=g, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn(1, 1, 4096, 128, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    a = torch.randn(2, 13418, generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randn(13418, 210, generator=g, device="cuda").to(torch.bfloat16)
    x = torch.randn(8192, 1024, generator=g, device="cuda")
    outs = [torch.zeros_like(q), torch.zeros(2, 210, device="cuda"), torch.zeros(1024, device="cuda")]
    calls = [lambda o, **kw: rt.attn_fwd(q, k, v, o, **kw), lambda o, **kw: rt.gemm(a, b, o, **kw),
             lambda o, **kw: rt.reduce(x, o, "max", axis=0, **kw)]
    ref = [call_(torch.zeros_like(o)) for call_, o in zip(calls, outs)]
    torch.cuda.synchronize()
    monkeypatch.setattr(torch, "empty", recorded)
    for call_, o in zip(calls, outs):
        call_(o, stream=stream)
    monkeypatch.undo()
    torch.cuda.synchronize()
    assert seen == [side.cuda_stream] * 3
    assert all(torch.equal(o, r) for o, r in zip(outs, ref))
