"""Which attention kernel a call gets (csrc/launch_plan.h): the target's launch
contract reports what the library launches."""
import ctypes
import os
import subprocess

import pytest

import frisk_amd as F
from frisk_amd import runtime as rt

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "frisk_amd", "csrc")


@pytest.fixture(scope="module")
def few(tmp_path_factory):
    """plan::attn_few on 256 CUs for (heads, queries, keys, head_dim) tuples."""
    d = tmp_path_factory.mktemp("plan")
    src = d / "plan.cpp"
    src.write_text(f"""#include "{CSRC}/launch_plan.h"
#include <cstdio>
#include <cstdlib>
int main(int n, char** v) {{
  for (int i = 1; i + 3 < n; i += 4)
    printf("%d ", frisk::plan::attn_few(atoll(v[i]), atoll(v[i + 1]), atoll(v[i + 2]), atoll(v[i + 3]), KT, 256));
}}""")
    for kt in (0, 1):
        subprocess.run(["g++", "-std=c++17", f"-DKT={kt}", str(src), "-o", str(d / f"plan{kt}")], check=True)
    return lambda calls, kt=False: [x == "1" for x in subprocess.run(
        [str(d / f"plan{int(kt)}"), *(str(x) for c in calls for x in c)], check=True, capture_output=True,
        text=True).stdout.split()]


@pytest.mark.parametrize("d,waves", [(16, 16), (32, 16), (64, 8), (128, 4)])
def test_few_queries_need_enough_keys_for_their_heads(few, d, waves):
    first = {16: 193, 32: 193, 64: 129, 128: 65}[d]      # one round of workgroups
    many = 385 if d == 128 else 705                      # several
    for bh, keys in ((1, first), (256, first), (257, many), (8192, many)):
        assert few([(bh, 1, keys, d), (bh, 32, keys, d), (bh, 1, keys - 1, d), (bh, 32, keys - 1, d),
                    (bh, 33, keys, d)]) == [True, True, False, False, False]
    # A grid of workgroups holds fewer than 2^32 threads.
    most = (1 << 32) // (64 * waves)
    assert few([(most - 1, 1, 4096, d), (most, 1, 4096, d)]) == [True, False]


def test_transposed_keys_at_head_dim_128_in_one_round_of_heads(few):
    calls = [(256, 2, 4096, 128), (257, 2, 4096, 128), (1024, 32, 512, 128), (257, 2, 4096, 64)]
    assert few(calls) == [True] * 4 and few(calls, kt=True) == [True, False, False, True]
    plans = [F.frisk.attention_launch_plan(b, q, d, seq_k=k, k_transposed=True)["kernel"] for b, q, k, d in calls]
    assert plans == ["attn_fewq", "attn_fwd", "attn_fwd", "attn_fewq"]


def contract(bh, sq, sk, d):
    L = F.frisk.attention_launch_plan(bh, sq, d, seq_k=sk)
    return L["kernel"], L["waves"]


@pytest.mark.parametrize("d,waves", [(16, 16), (32, 16), (64, 8), (128, 4)])
def test_launch_contract_reports_the_few_query_kernel(few, d, waves):
    calls = [(bh, sq, sk, d) for bh in (1, 256, 8192) for sq in (1, 32, 33) for sk in (64, 200, 1000)]
    for c, is_few in zip(calls, few(calls)):
        kernel, got = contract(*c)
        assert kernel == ("attn_fewq" if is_few else "attn_fwd")
        assert got == waves if is_few else got in (4, 8)
    # The keys default to the queries: a square problem of few queries has few keys.
    assert F.frisk.attention_launch_plan(64, 32, d)["kernel"] == "attn_fwd"


def test_waves_requested_are_those_of_the_query_tiled_kernel():
    assert rt.requested_waves(F.frisk.attention_launch_plan(128, 4096, 128)) == 8
    assert rt.requested_waves(F.frisk.attention_launch_plan(8, 4, 16, seq_k=4096)) == 0


@pytest.mark.parametrize("bh,sq,sk,d", [(2, 1, 4096, 128), (256, 1, 832, 64), (2, 32, 9000, 16),
                                        (2, 33, 9000, 128), (2, 1, 768, 128), (8192, 1, 512, 64)])
def test_scratch_only_for_the_few_query_kernel(bh, sq, sk, d):
    a = rt.AttnDesc(bh, 1, sq, sk, d, rt.BF16, 0, 1.0, 0, sq * d, sq * d, d, 0, sk * d, sk * d, d,
                    0, sk * d, sk * d, d, 0, sq * d, sq * d, d, None, rt.BF16, 0, 0)
    need = rt.load().frisk_attn_workspace_size(ctypes.byref(a))
    assert need >= 0, rt.load().frisk_last_error()
    if contract(bh, sq, sk, d)[0] != "attn_fewq" or sk <= rt.FEW_KEYS:
        assert need == 0
