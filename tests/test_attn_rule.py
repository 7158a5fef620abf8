"""Which attention kernel a call gets (csrc/launch_plan.h)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "frisk_amd", "csrc")


@pytest.fixture(scope="module")
def few(tmp_path_factory):
    """plan::attn_few on 256 CUs for (heads, queries, keys, head_dim) tuples."""
    d = tmp_path_factory.mktemp("plan")
    src, exe = d / "plan.cpp", d / "plan"
    src.write_text(f"""#include "{CSRC}/launch_plan.h"
#include <cstdio>
#include <cstdlib>
int main(int n, char** v) {{
  for (int i = 1; i + 3 < n; i += 4)
    printf("%d ", frisk::plan::attn_few(atoll(v[i]), atoll(v[i + 1]), atoll(v[i + 2]), atoll(v[i + 3]), 256));
}}""")
    subprocess.run(["g++", "-std=c++17", str(src), "-o", str(exe)], check=True)
    return lambda calls: [x == "1" for x in subprocess.run(
        [str(exe), *(str(x) for c in calls for x in c)], check=True, capture_output=True,
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
