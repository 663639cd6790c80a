"""The 16-bit backward's split form (two waves per 32 owned rows) at the sizes
where it can go wrong: one row, the edges of a wave's rows, of a workgroup's 64
and of the 64 and 128 streamed rows, an odd number of tiles; and the 128-row
form beside it on grids too large for the split.  With and without the
forward's output, against the float64 oracle with the tolerances of the other
backward tests."""
from __future__ import annotations

import pytest

from tests.test_attn_bwd_gpu import _check, _run, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_backward_split_edges(device, D, causal, dtype):
    # (B, H, S, heads checked); 600 x 1 and 600 x 2 128-row workgroups are past
    # the split's rule
    for i, (B, H, S, heads) in enumerate([(1, 1, 1, None), (1, 3, 31, None), (2, 1, 33, None), (1, 2, 64, None),
                                          (1, 1, 65, None), (1, 2, 127, None), (1, 2, 129, None), (1, 1, 193, None),
                                          (1, 1, 321, None), (100, 6, 65, [0, 599]), (100, 6, 193, [7, 598])]):
        tag = f"{dtype} B{B} H{H} S{S} D{D} causal={causal}"
        for with_o in (False, True):
            if with_o and S == 1:   # dq is 0: only rounding noise to compare
                continue
            _say(f"case {tag} with_o={with_o}")
            got, ref, fl = _run(B, H, S, D, dtype, causal, seed=9300 + i, with_o=with_o, heads=heads)
            _check(got, ref, dtype, f"{tag} with_o={with_o}", fl)


def test_forward_small_item_count(device):
    """Head_dim 128 on 128-row work items: the sizes at which the rule begins,
    ragged tiles, both masks."""
    import torch

    import pmkl_amd
    from pmkl_amd.workloads import small_inputs
    from tests.parity import check_outputs

    for i, (B, H, S, dtype, causal) in enumerate([(1, 1, 385, "bf16", False), (1, 2, 353, "fp16", True),
                                                  (2, 1, 511, "bf16", True), (1, 1, 641, "fp16", False),
                                                  (1, 1, 1025, "bf16", True)]):
        tag = f"{dtype} B{B} H{H} S{S} D128 causal={causal}"
        _say(f"case {tag}")
        q, k, v = small_inputs(B, H, S, 128, dtype, seed=9400 + i)
        qd, kd, vd = (x.to(device) for x in (q, k, v))
        o, m, l = pmkl_amd.attn_fwd(qd, kd, vd, is_causal=causal)
        torch.cuda.synchronize()
        args = pmkl_amd.capi.make_args(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), o.data_ptr(), m.data_ptr(),
                                       l.data_ptr(), dtype=pmkl_amd.torch_dtype_to_pmkl(qd.dtype), batch=B, heads=H,
                                       seq_len=S, head_dim=128, is_causal=causal)
        assert "attn_fwd_w64_kernel" in pmkl_amd.capi.attn_fwd_kernel_name(args)
        assert "1, 4>" in pmkl_amd.capi.attn_fwd_kernel_name(args)
        check_outputs(q, k, v, o, m, l, dtype, causal=causal, label=tag)
