"""The fp32 kernels' 32-row blocks and their four-way split of the streamed
tiles, at the sizes where they can go wrong: one row, the edges of a block,
fewer tiles than waves, tiles that do not divide by four.  Forward, and the
backward with and without the forward's output, against the float64 oracle
with the tolerances of the other fp32 tests."""
from __future__ import annotations

import pytest

from tests.test_attn_bwd_gpu import _check, _run, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_split_edges(device, D, causal):
    import torch

    import pmkl_amd
    from pmkl_amd.workloads import small_inputs
    from tests.parity import check_outputs

    for i, (B, H, S) in enumerate([(1, 3, 1), (2, 1, 31), (1, 9, 32), (1, 2, 33), (1, 1, 97), (3, 1, 128),
                                   (1, 2, 129), (1, 1, 290)]):
        tag = f"fp32 split B{B} H{H} S{S} D{D} causal={causal}"
        _say(f"case {tag}")
        q, k, v = small_inputs(B, H, S, D, "fp32", seed=9100 + i)
        o, m, l = pmkl_amd.attn_fwd(q.to(device), k.to(device), v.to(device), is_causal=causal)
        torch.cuda.synchronize()
        check_outputs(q, k, v, o, m, l, "fp32", causal=causal, label=tag)
        for with_o in (False, True):
            if with_o and S == 1:   # dq is 0: only rounding noise to compare
                continue
            got, ref, fl = _run(B, H, S, D, "fp32", causal, seed=9200 + i, with_o=with_o)
            _check(got, ref, "fp32", f"{tag} with_o={with_o}", fl)
