"""The forms of the 16-bit backward, each over the sizes of the backward tests
whatever the dispatch would choose there: tests/bwd_switch_check.py in a child
process with the form pinned (small grids take the split form by themselves,
large ones the 128-row form or, at head_dim 64, the eight-wave one)."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent


def test_backward_form_rule(device):
    """The split form where it is the faster (bf16, 256 CUs): not on a single tile
    of streamed rows, not where the 128-row workgroups fill the CUs."""
    from pmkl_amd import capi

    def form(BH, S, D, causal, with_o=True):
        ptrs = list(range(0x1000, 0xb000, 0x1000))
        ptrs[4] *= with_o
        name = capi.attn_bwd_kernel_name(capi.make_bwd_args(
            *ptrs, 0, 0, dtype=capi.PMKL_DTYPE_BF16, batch=1, heads=BH, seq_len=S, head_dim=D,
            is_causal=causal))
        return tuple(int(x) for x in name.split(">")[0].split(", ")[3:])

    for BH, S, D, causal in ((1, 65, 128, True), (128, 100, 64, True), (96, 129, 64, True), (64, 320, 64, True),
                             (128, 256, 64, True), (64, 512, 64, True), (1, 80, 64, False), (128, 128, 128, False),
                             (16, 2047, 128, True), (256, 128, 32, False), (32, 2047, 32, True)):
        assert form(BH, S, D, causal) == (2, 4), (BH, S, D, causal)
    for BH, S, D, causal in ((1, 1, 128, True), (1, 64, 128, True), (4, 33, 64, False), (16, 64, 32, True),
                             (192, 100, 64, True), (128, 129, 64, True), (85, 320, 64, True), (1, 65, 64, False),
                             (192, 128, 128, False), (64, 512, 128, True), (72, 512, 64, True), (300, 128, 32, False)):
        assert form(BH, S, D, causal) == (1, 4), (BH, S, D, causal)
    # eight waves: an even number of 128-row workgroups per CU, long sequences
    for BH, S, causal in ((24, 2047, False), (32, 2048, False), (6, 8192, False), (16, 8192, False), (24, 8192, False),
                          (16, 8192, True), (28, 4096, True)):
        assert form(BH, S, 64, causal) == (1, 8), (BH, S, causal)
    for BH, S, causal in ((64, 1024, False), (40, 2047, False), (64, 2048, False), (20, 8192, False), (8, 8192, True),
                          (12, 8192, True), (64, 2048, True), (24, 8192, True), (64, 8192, False)):
        assert form(BH, S, 64, causal) == (1, 4), (BH, S, causal)
    assert form(36, 1024, 64, False) == (1, 8) and form(36, 1024, 64, False, with_o=False) == (1, 4)
    assert form(26, 4096, 64, True) == (1, 8) and form(26, 4096, 64, True, with_o=False) == (1, 4)
    assert form(24, 2047, 32, False) == form(24, 2047, 128, False) == (1, 4)


@pytest.mark.parametrize("split, waves", [("0", "4"), ("0", "8"), ("1", "4")])
def test_backward_form_vs_oracle(device, split, waves):
    env = {k: v for k, v in os.environ.items() if not k.startswith("PMKL_ATTN")}
    res = subprocess.run([sys.executable, str(ROOT / "tests" / "bwd_switch_check.py")], cwd=str(ROOT),
                         env={**env, "PMKL_ATTN_BWDSPLIT": split, "PMKL_ATTN_BWDWAVES": waves}, capture_output=True, text=True, timeout=110)
    print(res.stdout[-3000:], flush=True)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
