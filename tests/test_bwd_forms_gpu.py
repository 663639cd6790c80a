"""Both forms of the 16-bit backward, each over the sizes of the backward tests
whatever the dispatch would choose there: tests/bwd_switch_check.py in a child
process with the form pinned (small grids take the split form by themselves,
large ones the 128-row form)."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.parametrize("split", ["0", "1"])
def test_backward_form_vs_oracle(device, split):
    env = {k: v for k, v in os.environ.items() if not k.startswith("PMKL_ATTN")}
    res = subprocess.run([sys.executable, str(ROOT / "tests" / "bwd_switch_check.py")], cwd=str(ROOT),
                         env={**env, "PMKL_ATTN_BWDSPLIT": split}, capture_output=True, text=True, timeout=110)
    print(res.stdout[-3000:], flush=True)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
