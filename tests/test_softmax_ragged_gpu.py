"""Row softmax with rows that are no whole number of 16-byte vectors: the last
vector of a row is moved back to end with it and shares elements with the one
before.  Row lengths around the vector, the row group and the chunk edges,
unaligned bases and strides, every type pair's store width, in place, and
special values among the shared elements, against the float64 oracle."""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_softmax_gpu import _check, _run, _say, _tdt

pytestmark = pytest.mark.gpu

W = {"fp32": 4, "fp16": 8, "bf16": 8}


@pytest.mark.parametrize("in_dt,out_dt", [("fp32", "fp32"), ("fp16", "fp16"), ("bf16", "bf16"), ("bf16", "fp32"),
                                          ("fp32", "fp16")])
def test_ragged_rows(device, in_dt, out_dt):
    w = W[in_dt]
    for n in sorted({w - 1, w, w + 1, 2 * w - 1, 2 * w + 1, 8 * w + 3, 64 * w - 1, 64 * w + 1, 1023}):
        for stride, offset in ((n, 0), (n + 1, 1), (n + w, 3)):
            for is_log in (False, True):
                label = f"softmax {in_dt}->{out_dt} n={n} stride={stride} offset={offset} log={is_log}"
                _say(f"case {label}")
                y, x = _run(71, n, stride, in_dt, out_dt, is_log, seed=n + stride, offset=offset)
                _check(y, x, n, out_dt, is_log, label)
        if in_dt == out_dt:
            y, x = _run(71, n, n, in_dt, out_dt, False, seed=n, in_place=True)
            _check(y, x, n, out_dt, False, f"softmax {in_dt} n={n} in place")


@pytest.mark.parametrize("dt", ["fp32", "bf16"])
def test_ragged_special_values(device, dt):
    import torch

    n = 5 * W[dt] + 2   # the last vector shares W - 2 elements with the one before
    x = np.random.Generator(np.random.PCG64(3)).uniform(-3, 3, size=(6, n))
    x[0, -3] = -np.inf            # among the shared elements
    x[1, :] = -np.inf
    x[1, -4] = 2.0                # the only finite one
    x[2, -3] = np.nan
    x[3, 0] = np.nan
    x[4, -1] = 80.0
    xt = torch.from_numpy(x.astype(np.float32)).to(_tdt(dt))
    for is_log in (False, True):
        y, x64 = _run(6, n, n, dt, dt, is_log, seed=0, xt=xt)
        _check(y, x64, n, dt, is_log, f"softmax {dt} special values log={is_log}")
