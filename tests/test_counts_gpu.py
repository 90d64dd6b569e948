"""Reference counts stay at their ceiling in the kernels that sum a block's
references (count_check.hip, built with the library by __graft_entry__.build)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import __graft_entry__  # noqa: E402


@pytest.mark.gpu
def test_counts_past_the_ceiling_do_not_grow():
    exe = __graft_entry__.COUNT_CHECK
    if not os.path.exists(exe):
        __graft_entry__.build()
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
