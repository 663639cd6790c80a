"""The fp32 backward's hidden keys and queries add nothing, whatever they hold:
an infinity or a NaN in one row of q, k, v or dout reaches exactly the gradients
of the rows that see it (and the rows past S, which the kernels read as zero,
reach none).  Against a float64 reference that visits visible pairs only."""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_attn_bwd_gpu import TOL, _say, _term_floors

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _forward(q, k, v, causal):
    o, m, l = np.zeros_like(q), np.zeros(q.shape[:2]), np.zeros(q.shape[:2])
    for h in range(q.shape[0]):
        for i in range(q.shape[1]):
            n = i + 1 if causal else q.shape[1]
            s = k[h, :n] @ q[h, i] / np.sqrt(q.shape[2])
            m[h, i] = s.max()
            p = np.exp(s - m[h, i])
            l[h, i] = p.sum()
            o[h, i] = (p / l[h, i]) @ v[h, :n]
    return o, m, l


def _backward(q, k, v, do, o, m, l, causal):
    sc = 1 / np.sqrt(q.shape[2])
    dq, dk, dv = (np.zeros_like(q) for _ in range(3))
    for h in range(q.shape[0]):
        for i in range(q.shape[1]):
            n = i + 1 if causal else q.shape[1]
            p = np.exp(sc * (k[h, :n] @ q[h, i]) - m[h, i]) / l[h, i]
            dp = v[h, :n] @ do[h, i]
            ds = sc * p * (dp - (do[h, i] @ o[h, i] if o is not None else p @ dp))
            dq[h, i] = ds @ k[h, :n]
            dk[h, :n] += np.outer(ds, q[h, i])
            dv[h, :n] += np.outer(p, do[h, i])
    return dq, dk, dv


# (tensor, row counted from the end if negative, element or None for the row, value)
PLANTED = [("k", 45, None, NAN), ("k", -1, 3, INF), ("v", 45, 5, -INF), ("v", -1, None, NAN), ("q", 20, None, NAN),
           ("q", 45, 7, INF), ("do", 45, None, NAN), ("do", 50, 2, INF), ("do", 50, 2, -INF), ("k", 40, None, -INF)]


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_fp32_backward_nonfinite_rows(device, D, causal):
    import torch

    import pmkl_amd

    H = 2
    for S in (77, 160, 290):
        rng = np.random.Generator(np.random.PCG64(S + D))
        clean = {n: rng.standard_normal((H, S, D)).astype(np.float32).astype(np.float64) for n in ("q", "k", "v", "do")}
        for name, row, element, value in PLANTED:
            x = {n: a.copy() for n, a in clean.items()}
            if (name, value) == ("k", -INF):   # a key whose scores are all -inf: P = 0
                x["q"] = np.abs(x["q"])
            _, m0, l0 = _forward(x["q"], x["k"], x["v"], causal)
            floors = _term_floors(x["q"], x["k"], x["v"], x["do"], m0, l0, causal)
            x[name][0, row, slice(None) if element is None else element] = value
            with np.errstate(all="ignore"):
                o, m, l = _forward(x["q"], x["k"], x["v"], causal)
                dev = lambda a: torch.from_numpy(a.astype(np.float32)).to(device)[None]
                o, m, l = (a.astype(np.float32).astype(np.float64) for a in (o, m, l))
                for with_o in (False, True):
                    tag = f"fp32 S{S} D{D} causal={causal} {name}[{row}, {element}] = {value} with_o={with_o}"
                    _say(f"case {tag}")
                    want = _backward(x["q"], x["k"], x["v"], x["do"], o if with_o else None, m, l, causal)
                    got = pmkl_amd.attn_bwd(dev(x["do"]), dev(x["q"]), dev(x["k"]), dev(x["v"]), dev(m), dev(l),
                                            is_causal=causal, out=dev(o) if with_o else None)
                    torch.cuda.synchronize()
                    assert not causal or any(np.isfinite(w).any() for w in want), tag
                    for g, w, fl, grad in zip(got, want, floors, ("dq", "dk", "dv")):
                        g = g[0].cpu().numpy().astype(np.float64)
                        fin = np.isfinite(w)
                        assert np.array_equal(g[~fin], w[~fin], equal_nan=True), f"{tag}: {grad} not finite elsewhere"
                        err = np.abs(g[fin] - w[fin])
                        assert (err <= TOL["fp32"] * max(fl, 1.0)).all(), f"{tag}: {grad} off by {err.max()}"


@pytest.mark.parametrize("D", [32, 64, 128])
def test_fp32_forward_row_of_minus_infinities(device, D):
    """The first query sees one key, whose score is -inf: m = -inf and l, o NaN,
    as the sums of exp(-inf - -inf) are; the other rows give that key no weight."""
    import torch

    import pmkl_amd

    for H, S in ((2, 77), (2, 290), (600, 130)):
        rng = np.random.Generator(np.random.PCG64(S + D))
        q, k, v = (rng.standard_normal((H, S, D)).astype(np.float32).astype(np.float64) for _ in range(3))
        q = np.abs(q)
        k[:, 0] = -INF
        with np.errstate(all="ignore"):
            want = _forward(q[:2], k[:2], v[:2], True)
        got = pmkl_amd.attn_fwd(*(torch.from_numpy(x.astype(np.float32)).to(device)[None] for x in (q, k, v)))
        torch.cuda.synchronize()
        for g, w, name in zip(got, want, ("o", "m", "l")):
            g = g[0, :2].cpu().numpy().astype(np.float64)
            fin = np.isfinite(w)
            assert fin.any() and not fin.all()
            assert np.array_equal(g[~fin], w[~fin], equal_nan=True), f"H{H} S{S} D{D}: {name} not finite elsewhere"
            assert (np.abs(g[fin] - w[fin]) <= 1e-5 * np.abs(w[fin]).max()).all(), f"H{H} S{S} D{D}: {name}"
