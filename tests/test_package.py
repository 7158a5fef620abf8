"""The package without its compiled extension."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_submodules_import_before_the_extension_is_built():
    """`from frisk_amd import build` (how a fresh checkout is built) and
    `runtime` work without frisk_ffi; its names still say what is missing."""
    code = """
import sys
sys.modules["frisk_amd.frisk_ffi"] = None  # as if not built
from frisk_amd import build, runtime
assert build.build_all and runtime.gemm
try:
    from frisk_amd import context
except ImportError as e:
    assert "is not built" in str(e), e
else:
    raise AssertionError("context resolved")
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT, timeout=300)
