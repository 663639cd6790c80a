"""The 16-bit backward in the form that the dispatch chooses, with and without
the forward's output: the split form (two waves per 32 owned rows) from S 65 on
at the edges of a wave's rows, of a workgroup's 64 and of the 64 and 128
streamed rows and an odd number of tiles; the 128-row form below and on grids
too large for the split (test_bwd_forms_gpu.py pins either at all sizes).  Against the float64 oracle
with the tolerances of the other backward tests; with the forward's output
against the same oracle with its row term moved to <dout, O> (_move_row_term)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle
from tests.test_attn_bwd_gpu import _check, _np, _run, _say

pytestmark = pytest.mark.gpu


def _move_row_term(ref, q, k, v, do, o, m, l, causal, heads):
    """The oracle's dq, dk with D_i = <dout_i, o_i>, o as the forward stored it,
    for its D_i = sum_j P_ij dP_ij.  A kernel that is handed O computes that one.
    The two differ by more than a rounding of the gradient: the stored 16-bit m
    and l are off by up to 2^-9 in bf16, so sum_j P_ij is 1 + O(2^-8 + |m| 2^-9),
    and the oracle's D_i is off by as much of itself, all in one direction
    (B1 H2 S64 D32 full bf16: dq 1.19 of its bound from that alone)."""
    dq, dk, dv = (x.copy() for x in ref)
    sc = oracle.default_scale(q.shape[-1])
    for n, h in enumerate(range(q.shape[0]) if heads is None else heads):
        s = sc * q[h] @ k[h].T
        if causal:
            s[np.triu_indices(s.shape[0], 1)] = -np.inf
        p = np.exp(s - m[h][:, None]) / l[h][:, None]
        shift = sc * p * ((p * (do[h] @ v[h].T)).sum(axis=1) - (do[h] * o[h]).sum(axis=1))[:, None]
        dq[n] += shift @ k[h]
        dk[n] += shift.T @ q[h]
    return dq, dk, dv


def _run_with_o(B, H, S, D, dtype, causal, seed, heads):
    """_run, handing the backward the forward's output."""
    import torch

    import pmkl_amd
    from pmkl_amd.workloads import small_inputs, torch_dtype

    q, k, v = small_inputs(B, H, S, D, dtype, seed=seed)
    rng = np.random.Generator(np.random.PCG64(seed + 17))
    do = torch.from_numpy(rng.standard_normal((B, H, S, D)).astype(np.float32)).to(torch_dtype(dtype))
    qd, kd, vd, dod = (x.to("cuda:0") for x in (q, k, v, do))
    o, m, l = pmkl_amd.attn_fwd(qd, kd, vd, is_causal=causal)
    got = pmkl_amd.attn_bwd(dod, qd, kd, vd, m, l, is_causal=causal, out=o)
    torch.cuda.synchronize()
    q, k, v, do, o = (_np(t).reshape(B * H, S, D) for t in (q, k, v, do, o))
    m, l = (_np(t).reshape(B * H, S) for t in (m, l))
    ref = _move_row_term(oracle.attn_bwd(q, k, v, do, m, l, causal=causal, heads=heads), q, k, v, do, o, m, l, causal,
                         heads)
    got = [_np(x).reshape(B * H, S, D) for x in got]
    return got if heads is None else [x[list(heads)] for x in got], ref


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
            if with_o:
                got, ref = _run_with_o(B, H, S, D, dtype, causal, seed=9300 + i, heads=heads)
            else:
                got, ref, _ = _run(B, H, S, D, dtype, causal, seed=9300 + i, heads=heads)
            _check(got, ref, dtype, f"{tag} with_o={with_o}")


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


def test_forward_small_item_count_rule(device):
    """Head_dim 128 causal: where 128-row work items and their order over the XCDs
    are the faster (256 CUs), and the results on a plain order with two items per
    workgroup."""
    import torch

    import pmkl_amd
    from pmkl_amd import capi
    from pmkl_amd.workloads import small_inputs
    from tests.parity import check_outputs

    def name(BH, S):
        return capi.attn_fwd_kernel_name(capi.make_args(*range(0x1000, 0x7000, 0x1000), dtype=capi.PMKL_DTYPE_BF16,
                                                        batch=1, heads=BH, seq_len=S, head_dim=128))

    for BH, S, form, xcd in ((32, 1800, ", 1, 4>", False), (32, 1500, ", 1, 4>", False), (32, 2047, ", 1, 4>", True),
                             (64, 1024, ", 1, 4>", True), (16, 1500, ", 1, 4>", True), (48, 1030, ", 1, 8>", True),
                             (49, 1200, ", 1, 8>", False), (40, 1200, ", 1, 8>", False), (38, 1200, ", 1, 4>", False)):
        assert form in name(BH, S) and ("xcd order" in name(BH, S)) == xcd, (BH, S, name(BH, S))
    q, k, v = small_inputs(2, 16, 1500, 128, "bf16", seed=9450)
    o, m, l = pmkl_amd.attn_fwd(q.to(device), k.to(device), v.to(device))
    torch.cuda.synchronize()
    heads = lambda t: t[:, [0, 7, 15]]
    check_outputs(*map(heads, (q, k, v)), *(heads(t).contiguous() for t in (o, m, l)), "bf16", causal=True,
                  label="bf16 B2 H16 S1500 D128")
