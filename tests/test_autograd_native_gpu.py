"""The native autograd entry on device tensors against the Python autograd
function it stands in for: same outputs and gradients bit for bit, and the same
behaviour where PyTorch hooks into autograd."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def _inputs(dtype, packed=False, B=2, H=3, S=77, D=64, seed=5):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    if packed:
        qkv = mk(B, S, 3, H, D)
        q, k, v = (qkv[:, :, i].transpose(1, 2).detach().requires_grad_(True) for i in range(3))
    else:
        q, k, v = (mk(B, H, S, D).requires_grad_(True) for _ in range(3))
    return q, k, v, mk(B, H, S, D)


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("packed", [False, True])
def test_same_as_python_function(device, dtype, packed):
    import torch
    from pmkl_amd.pmkl_function import fused_self_attention, fused_self_attention_

    for causal in (True, False):
        q, k, v, do = _inputs(getattr(torch, dtype), packed)
        a = fused_self_attention(q, k, v, causal)
        b = fused_self_attention_.apply(q, k, v, causal)
        assert all(torch.equal(x, y) and x.requires_grad == y.requires_grad for x, y in zip(a, b))
        for seed in (do, do[..., :1].expand_as(do), do.transpose(1, 2).contiguous().transpose(1, 2)):
            ga = torch.autograd.grad(a[0], (q, k, v), seed, retain_graph=True)
            gb = torch.autograd.grad(b[0], (q, k, v), seed, retain_graph=True)
            assert all(torch.equal(x, y) for x, y in zip(ga, gb))
        # the gradients of m and l are ignored; alone they give zeros
        ga = torch.autograd.grad((a[1].sum() + a[2].sum()), (q, k, v), retain_graph=True)
        assert all(not g.any() for g in ga)
        torch.autograd.grad(a[0], (q,), do)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(a[0], (q,), do)


def test_hooks_transforms_and_modes(device):
    import torch
    from pmkl_amd.pmkl_function import fused_self_attention, fused_self_attention_

    q, k, v, do = _inputs(torch.bfloat16)
    want = torch.autograd.grad(fused_self_attention_.apply(q, k, v, True)[0], (q, k, v), do)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        out = fused_self_attention(q, k, v, True)[0]
    assert len(packed) == 6
    got = torch.autograd.grad(out, (q, k, v), do)
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    # torch.func gets the Python function, whose kernels refuse its wrapper tensors
    f = torch.func.grad(lambda q: (fused_self_attention(q, k.detach(), v.detach(), True)[0] * do).sum())
    with pytest.raises(RuntimeError, match="data pointer"):
        f(q.detach())
    # no graph without grad mode; keywords and the default of debug
    with torch.no_grad():
        assert not fused_self_attention(q=q, k=k, v=v, is_casual=True)[0].requires_grad
    # a saved input changed in place is refused
    out = fused_self_attention(q, k, v, True)[0]
    with torch.no_grad():
        k.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(do)


def test_side_stream(device):
    import torch
    from pmkl_amd.pmkl_function import fused_self_attention

    q, k, v, do = _inputs(torch.float16, S=300)
    want = torch.autograd.grad(fused_self_attention(q, k, v, True)[0], (q, k, v), do)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = torch.autograd.grad(fused_self_attention(q, k, v, True)[0], (q, k, v), do)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(got, want))


def test_gradient_strides_of_single_dimensions(device):
    """A dimension of size 1 may carry any stride; such a gradient gives the
    result of its contiguous copy."""
    import torch
    from pmkl_amd.pmkl_function import fused_self_attention

    for B, H, S in ((1, 3, 40), (2, 1, 40), (1, 1, 40), (2, 3, 1)):
        q, k, v, do = _inputs(torch.bfloat16, B=B, H=H, S=S, D=32)
        st = [7 if n == 1 else x for n, x in zip(do.shape[:3], do.stride())] + [1]
        odd = do.as_strided(do.shape, st)
        a = torch.autograd.grad(fused_self_attention(q, k, v, True)[0], (q, k, v), odd)
        b = torch.autograd.grad(fused_self_attention(q, k, v, True)[0], (q, k, v), do)
        assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_saved_tensors_that_come_back_different(device):
    """What a saved-tensor hook returns is checked before a kernel gets its pointer."""
    import torch
    from pmkl_amd.pmkl_function import fused_self_attention

    q, k, v, do = _inputs(torch.bfloat16)
    for unpack in (lambda t: t[..., :1], lambda t: t.float() if t.dim() == 4 else t[..., :1], lambda t: t.cpu()):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = fused_self_attention(q, k, v, True)[0]
        with pytest.raises(RuntimeError, match="came back"):
            torch.autograd.grad(out, (q, k, v), do)
