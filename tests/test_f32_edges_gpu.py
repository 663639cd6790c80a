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


@pytest.mark.parametrize("D, B, H", [(64, 24, 32), (32, 48, 32)])
def test_fp32_forward_128_row_workgroups(device, D, B, H):
    """Full attention over 96 to 128 keys with many heads: the 128-row kernel
    (256 CUs), at both ends of the range; the key-split kernel beside it."""
    import torch

    import pmkl_amd
    from pmkl_amd import capi
    from pmkl_amd.workloads import small_inputs
    from tests.parity import check_outputs

    def name(heads, S, causal=False):
        f32 = capi.PMKL_DTYPE_F32
        return capi.attn_fwd_kernel_name(capi.make_args(*range(0x1000, 0x7000, 0x1000), dtype=f32, batch=1, heads=heads,
                                                        seq_len=S, head_dim=D, is_causal=causal))

    for S in (96, 128):
        assert name(B * H, S).startswith("attn_fwd_f32_kernel"), name(B * H, S)
        tag = f"fp32 B{B} H{H} S{S} D{D} full"
        _say(f"case {tag}")
        q, k, v = small_inputs(B, H, S, D, "fp32", seed=9700 + S)
        o, m, l = pmkl_amd.attn_fwd(q.to(device), k.to(device), v.to(device), is_causal=False)
        torch.cuda.synchronize()
        check_outputs(q, k, v, o, m, l, "fp32", causal=False, label=tag)
    for heads, S, causal in ((B * H, 95, False), (B * H, 129, False), (B * H, 128, True), (B * H - 1, 128, False)):
        assert name(heads, S, causal).startswith("attn_fwd_f32_split_kernel"), (heads, S, causal)
