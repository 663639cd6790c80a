"""The fp32 backward a row per wave: where the dispatch takes it (sequences that
leave most of a 32-row tile empty; measured there up to 8 times faster than the
tiles), its results against the float64 oracle, and a call with more heads than
a launch of the tile kernels could hold."""
from __future__ import annotations

import pytest

from tests.test_attn_bwd_gpu import _check, _run, _say

pytestmark = pytest.mark.gpu


def _name(BH, S, D, causal=True):
    from pmkl_amd import capi

    args = capi.make_bwd_args(*(range(0x1000, 0xb000, 0x1000)), 0, 0, dtype=capi.PMKL_DTYPE_F32, batch=1, heads=BH,
                              seq_len=S, head_dim=D, is_causal=causal)
    return capi.attn_bwd_kernel_name(args)


def test_fp32_backward_rows_or_tiles(device):
    # (heads, S, head_dim): rows where they are the faster, on a device of 256 CUs
    for BH, S, D in ((1, 1, 32), (65536, 4, 32), (256, 8, 32), (64, 14, 32), (8192, 6, 64), (384, 8, 64), (128, 14, 64),
                     (32, 28, 64), (16, 33, 64), (65536, 7, 128), (384, 8, 128), (64, 16, 128), (16, 36, 128)):
        assert "attn_bwd_f32_row_dq_kernel" in _name(BH, S, D), (BH, S, D)
    for BH, S, D in ((1024, 8, 32), (1, 16, 32), (1024, 8, 64), (1024, 8, 128), (192, 14, 64), (64, 24, 64), (1, 37, 64), (128, 16, 128),
                     (1, 48, 128)):
        assert "attn_bwd_f32_dq_kernel" in _name(BH, S, D), (BH, S, D)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_backward_rows_vs_oracle(device, D, causal):
    for i, (B, H, S) in enumerate([(1, 1, 1), (2, 3, 2), (1, 5, 5), (3, 1, 8), (1, 2, 12), (1, 2, 16), (1, 3, 28),
                                   (2, 2, 31), (1, 1, 36)]):
        tag = f"fp32 rows B{B} H{H} S{S} D{D} causal={causal}"
        _say(f"case {tag} {_name(B * H, S, D, causal)}")
        for with_o in (False, True):
            if with_o and S == 1:   # dq is 0: only rounding noise to compare
                continue
            got, ref, fl = _run(B, H, S, D, "fp32", causal, seed=9600 + i, with_o=with_o)
            _check(got, ref, "fp32", f"{tag} with_o={with_o}", fl)


def test_fp32_backward_more_than_2_24_heads(device):
    """S = 1: dv = dout (P = 1), dq = dk = 0 up to rounding."""
    import torch

    import pmkl_amd

    B, D = (1 << 24) + 3, 32
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(1, 1, 1, D, device="cuda", generator=g) for _ in range(3))
    o, m, l = pmkl_amd.attn_fwd(q, k, v)
    wide = lambda t: t.expand(B, *t.shape[1:])
    dout = torch.randn(B, 1, 1, D, device="cuda", generator=g)
    dq, dk, dv = pmkl_amd.attn_bwd(dout, wide(q), wide(k), wide(v), wide(m).contiguous(), wide(l).contiguous(),
                                   out=wide(o))
    torch.cuda.synchronize()
    assert float((dv - dout).abs().max()) < 1e-5
    assert float(dq.abs().max()) < 1e-4 and float(dk.abs().max()) < 1e-4
