"""Child-process check of the 16-bit backward's forms (run by
tests/test_bwd_forms_gpu.py with PMKL_ATTN_BWDSPLIT and PMKL_ATTN_BWDWAVES set;
the library reads them once per process): the cases of test_attn_bwd_gpu.py on the form that the
switches pin, and more of them where that form can go wrong.  Exits 0 when all
pass."""
from __future__ import annotations

import os
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT))


def main() -> int:
    import torch

    import pmkl_amd
    from tests import test_attn_bwd_gpu as t

    ks = 2 if os.environ["PMKL_ATTN_BWDSPLIT"] == "1" else 1
    eight = ks == 1 and os.environ["PMKL_ATTN_BWDWAVES"] == "8"
    raw, launched = pmkl_amd.capi.attn_bwd_raw, set()

    def named(args, stream=None):   # every backward call of the cases below names its kernels first
        name = pmkl_amd.capi.attn_bwd_kernel_name(args)
        assert name.count(f", {ks}, {8 if eight and args.head_dim == 64 else 4}>") == 2, name
        launched.add(name.split(" grid")[0])
        return raw(args, stream)

    pmkl_amd.capi.attn_bwd_raw = named
    dev = torch.device("cuda:0")
    for dtype in ("bf16", "fp16"):
        for D in (64,) if eight else (32, 64, 128):
            for causal in (True, False):
                t.test_bwd_small_shapes_vs_oracle(dev, dtype, D, causal)
                # edges of a wave's rows and of a tile, odd and even counts of tiles, more than two per workgroup
                for B, H, S in ((1, 3, 31), (1, 2, 127), (1, 2, 129), (1, 1, 193), (1, 1, 321), (1, 2, 449), (1, 1, 700)):
                    tag = f"{dtype} B{B} H{H} S{S} D{D} causal={causal}"
                    t._say(f"case {tag}")
                    got, ref, _ = t._run(B, H, S, D, dtype, causal, seed=9500 + S, ml_dtype=torch.float32)
                    t._check(got, ref, dtype, tag)
            t.test_bwd_strided_views_without_copies(dev, dtype, D)
            if D > 32:
                t.test_bwd_with_forward_output(dev, dtype, D)
        for causal in (True, False) if not eight else ():
            t.test_bwd_float_ml_from_64_row_kernel(dev, dtype, causal)
    if not eight:   # head_dim 128
        t.test_bwd_larger_heads_sampled(dev)
    t.test_bwd_closed_form_constant_v(dev)
    assert len(launched) == (4 if eight else 12), launched   # dtypes x head_dims x masks
    return 0


if __name__ == "__main__":
    sys.exit(main())
