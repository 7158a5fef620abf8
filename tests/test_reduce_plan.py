"""The launch geometry of axis-0 reductions (csrc/launch_plan.h), read by a
host program."""
import ctypes
import os
import subprocess

import pytest

from frisk_amd import runtime as rt

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "frisk_amd", "csrc")


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """run(expression over r (rows), c (cols), shapes) -> list of int lists."""
    def go(fields, shapes):
        d = tmp_path_factory.mktemp("plan")
        src, exe = d / "plan.cpp", d / "plan"
        src.write_text(f"""#include "{CSRC}/launch_plan.h"
#include <cstdio>
#include <cstdlib>
using namespace frisk::plan;
int main(int n, char** v) {{
  for (int i = 1; i + 1 < n; i += 2) {{
    const int64_t r = atoll(v[i]), c = atoll(v[i + 1]);
    for (const long long x : {{{", ".join(f"(long long)({f})" for f in fields)}}}) printf("%lld ", x);
    puts("");
  }}
}}""")
        subprocess.run(["g++", "-std=c++17", str(src), "-o", str(exe)], check=True)
        out = subprocess.run([str(exe), *(str(x) for s in shapes for x in s)], check=True,
                             capture_output=True, text=True).stdout
        return [[int(x) for x in line.split()] for line in out.strip().split("\n")]
    return go


SHAPES = [(256, 3), (100000, 3), (40000, 5), (262145, 2), ((1 << 23) - 1, 1), (70000, 40),
          (300000, 64), (131072, 2048), (65536, 12800), (33000, 8192), (16384, 32768), (600, 12801),
          (1024, 65536), (4097, 70000)]


def test_one_pass_covers_the_rows_on_live_threads(run):
    fields = ["cols_pass(r, c, true, 1024)." + f for f in ("threads", "cvb_log2", "b_log2", "blocks", "strips")]
    for (rows, cols), (threads, cvb, b, blocks, strips) in zip(SHAPES, run(fields, SHAPES)):
        slots, groups = -(-cols // 4), threads >> cvb
        # No strip is wider than the slots there are, unless the rows give
        # fewer runs of eight than there are threads: at most one thread in two
        # of a workgroup has no column.
        assert (1 << cvb) < 2 * slots or groups <= -(-rows // 8), (rows, cols)
        assert strips << cvb >= slots and blocks * (groups << b) >= rows
        assert (blocks - 1) * (groups << b) < rows
        # Runs past 256 rows only in 256 threads and a full round of strips,
        # within their counter's 22 levels; blocks within 12 levels.
        if b > 8:
            assert threads == 256 and strips >= 256 and blocks == 1 and b - 2 <= 22, (rows, cols)
        assert blocks < 1 << 12
        if blocks == 1 and threads == 1024:
            assert groups << b < 4 * rows or b == 3  # few idle row groups


@pytest.mark.parametrize("dtype,kind", [(rt.F32, rt.REDUCE_SUM), (rt.F32, rt.REDUCE_MAX),
                                        (rt.BF16, rt.REDUCE_SUM)])
def test_workspace_query_asks_only_for_what_the_launch_reads(run, dtype, kind):
    """The size is 0 exactly where frisk_reduce runs one pass, so no caller
    allocates scratch nobody reads and no workspace is too short for it."""
    plan = f"cols_two_pass(r, c, {str(kind == rt.REDUCE_SUM).lower()}, {str(dtype == rt.F32).lower()})"
    lib = rt.load()
    for (rows, cols), (two,) in zip(SHAPES, run([plan], SHAPES)):
        d = rt.ReduceDesc(rows, cols, dtype, kind, 0, 1, 16, cols, 16, 1)
        assert (lib.frisk_reduce_workspace_size(ctypes.byref(d)) > 0) == bool(two), (rows, cols)


def test_one_pass_where_its_strips_fill_the_chip():
    lib = rt.load()

    def size(rows, cols, kind=rt.REDUCE_SUM, dtype=rt.F32):
        d = rt.ReduceDesc(rows, cols, dtype, kind, 0, 1, 16, cols, 16, 1)
        return lib.frisk_reduce_workspace_size(ctypes.byref(d))

    assert size(1024, 65536) == 0 and size(4096, 32768, rt.REDUCE_MAX) == 0 and size(300, 14000) == 0
    assert size(32768, 16384) == 0  # an f32 sum of long runs
    assert size(16384, 13000) > 0 and size(600, 12801, dtype=rt.F16) > 0 and size(100000, 3) > 0
