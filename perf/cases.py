"""Performance cases of the framework: what its users call, over the sizes they call it with.

Four kinds of work, each through a public entry point:

  fwd      inference: `pmkl_pytorch_ext.fused_self_attention_fw`, or, with "buffers", `pmkl_amd.attn_fwd` into output
           buffers that the program keeps (row max and row sum in float32)
  train    a training step's attention: `pmkl_function.fused_self_attention` and autograd's gradients of q, k and v
  op       the operator pair without autograd: `fused_self_attention_fw`, then `fused_self_attention_bw`, which is not
           handed the forward's output
  softmax  `pmkl_amd.softmax` over the last dimension of a score matrix

`draw` gives further cases over the ranges that the listed ones stand for: every data type, head_dim 32, 64 and 128,
causal and full, contiguous tensors and views of one packed projection, sequences from a few rows to 16,384.
"""
import math

import torch

import pmkl_amd
import pmkl_function
import pmkl_pytorch_ext

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

# Largest work of one pass, of the largest listed cases: multiply-adds x 2 of attention in 16 and in 32 bits, elements of
# one [B, H, S, D] tensor, elements of a softmax.
MAX_FLOPS = {2: 14 * 128 * 128 * 4096 * 4097 / 2, 4: 14 * 64 * 64 * 1024 * 1025 / 2}
MAX_ELEMENTS = {2: 128 * 4096 * 128, 4: 64 * 1024 * 128}
MAX_SOFTMAX = 131072 * 1024


def _attention(name, kind, dtype, B, H, S, D, causal, packed=False, buffers=False):
    return {"name": name, "kind": kind, "dtype": dtype, "B": B, "H": H, "S": S, "D": D, "causal": causal,
            "packed": packed, "buffers": buffers}


def _softmax(name, dtype, rows, n, log):
    return {"name": name, "kind": "softmax", "dtype": dtype, "rows": rows, "n": n, "log": log}


def listed():
    return [
        # One short prompt in float32, the smallest call: its latency is what a user sees.
        _attention("fwd_f32_128", "fwd", "fp32", 1, 4, 128, 64, True),
        # The float32 training shape of the operator's own test: small, full attention, head_dim 128.
        _attention("train_f32_128", "train", "fp32", 2, 16, 128, 128, False),
        # The float32 shape of the forward's own GPU test: an ordinary batch at S = 1,024.
        _attention("fwd_f32_1k", "fwd", "fp32", 4, 16, 1024, 64, True),
        # The same batch in training, for programs that train in float32.
        _attention("train_f32_1k", "train", "fp32", 4, 16, 1024, 64, True),
        # Prefill of a large decoder layer in bfloat16, the benchmark's headline shape, into kept buffers.
        _attention("fwd_bf16_4k", "fwd", "bf16", 4, 32, 4096, 128, True, buffers=True),
        # Training of the same layer: the largest case.
        _attention("train_bf16_4k", "train", "bf16", 4, 32, 4096, 128, True),
        # Training of a mid-sized decoder in float16; q, k and v are views of one packed projection.
        _attention("train_f16_1k", "train", "fp16", 8, 16, 1024, 64, True, packed=True),
        # Training with many short sequences and small heads.
        _attention("train_f16_256", "train", "fp16", 64, 8, 256, 32, True),
        # Training of an encoder over 196 patches and a class token: full attention, odd length.
        _attention("train_bf16_197", "train", "bf16", 16, 12, 197, 64, False, packed=True),
        # The operator pair on a long odd sequence with few heads; its backward forms the row terms itself.
        _attention("op_bf16_2047", "op", "bf16", 2, 8, 2047, 128, True),
        # Wide float32 score rows, all aligned.
        _softmax("softmax_f32_1024", "fp32", 131072, 1024, False),
        # Score rows of the 197-long sequences: odd length, so most rows start unaligned.
        _softmax("softmax_bf16_197", "bf16", 151296, 197, False),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(max(low, high))))))


def draw(rng):
    kind = rng.choices(["fwd", "train", "op", "softmax"], [0.35, 0.4, 0.1, 0.15])[0]
    dtype = rng.choices(["fp32", "fp16", "bf16"], [0.3, 0.35, 0.35])[0]
    if kind == "softmax":
        n = _log_int(rng, 4, 1024)
        return {"kind": kind, "dtype": dtype, "rows": _log_int(rng, 12, MAX_SOFTMAX // 1024), "n": n,
                "log": rng.random() < 0.3}
    size = DTYPES[dtype].itemsize
    D = rng.choice([32, 64, 64, 128, 128])
    causal = rng.random() < 0.65
    if size == 4:
        S = _log_int(rng, 16, 2048)
    else:
        S = _log_int(rng, 16, 16384 if kind == "fwd" else 8192)
    pairs = S * (S + 1) // 2 if causal else S * S
    heads = min(MAX_FLOPS[size] / (14 * D * pairs), MAX_ELEMENTS[size] / (S * D), 2048)
    BH = _log_int(rng, 1, max(1, int(heads)))
    H = max(1, min(BH, rng.choice([1, 2, 4, 5, 8, 12, 16, 32])))
    B = max(1, BH // H)
    return {"kind": kind, "dtype": dtype, "B": B, "H": H, "S": S, "D": D, "causal": causal,
            "packed": rng.random() < 0.4, "buffers": kind == "fwd" and rng.random() < 0.5}


def prepare(case, seed):
    dtype = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)

    if case["kind"] == "softmax":
        return {"case": case, "x": normal(case["rows"], case["n"]) * 4}
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    if case["packed"]:   # one projection [B, S, 3, H, D], as a fused QKV layer writes it
        qkv = normal(B, S, 3, H, D)
        q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    else:
        q, k, v = normal(B, H, S, D), normal(B, H, S, D), normal(B, H, S, D)
    state = {"case": case, "q": q, "k": k, "v": v}
    if case["kind"] != "fwd":
        state["dout"] = normal(B, H, S, D)
    if case["kind"] == "train":
        for name in "qkv":
            state[name].requires_grad_(True)
    if case["buffers"]:
        state["out"] = torch.empty((B, H, S, D), dtype=dtype, device="cuda")
        state["out_m"] = torch.empty((B, H, S), dtype=torch.float32, device="cuda")
        state["out_l"] = torch.empty((B, H, S), dtype=torch.float32, device="cuda")
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "softmax":
        return pmkl_amd.softmax(state["x"], is_log=case["log"])
    q, k, v = state["q"], state["k"], state["v"]
    if kind == "train":
        out, m, l = pmkl_function.fused_self_attention(q, k, v, case["causal"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
    elif kind == "op":
        out, m, l = pmkl_pytorch_ext.fused_self_attention_fw(q, k, v, case["causal"])
        dq, dk, dv = pmkl_pytorch_ext.fused_self_attention_bw(state["dout"], q, k, v, m, l, case["causal"])
    elif case["buffers"]:
        out, m, l = pmkl_amd.attn_fwd(q, k, v, is_causal=case["causal"], out=state["out"], out_m=state["out_m"],
                                      out_l=state["out_l"])
    else:
        out, m, l = pmkl_pytorch_ext.fused_self_attention_fw(q, k, v, case["causal"])
    if kind == "fwd":
        return {"out": out, "m": m, "l": l}
    return {"out": out, "m": m, "l": l, "dq": dq, "dk": dk, "dv": dv}


def work(case):
    size = DTYPES[case["dtype"]].itemsize
    if case["kind"] == "softmax":
        elements = case["rows"] * case["n"]
        # per element a difference, an exponential, a sum, a product and the maximum
        return {"bytes": 2 * elements * size, "flops": 5 * elements}
    rows = case["B"] * case["H"] * case["S"]
    pairs = rows * (case["S"] + 1) // 2 if case["causal"] else rows * case["S"]
    row_size = 4 if case["buffers"] else size
    if case["kind"] == "fwd":      # q, k, v; out, m, l.  Two products.
        return {"bytes": 4 * rows * case["D"] * size + 2 * rows * row_size, "flops": 4 * case["D"] * pairs}
    # q, k, v, dout; out, m, l, dq, dk, dv.  Two products forward, five backward.
    return {"bytes": 8 * rows * case["D"] * size + 2 * rows * size, "flops": 14 * case["D"] * pairs}


def tolerance(case):
    # About four times the distance from the 64-bit results: 4e-7 / 2.5e-4 / 2.2e-3 forward and softmax (the rounding of the
    # stored outputs in 16 bits; ten times in 32, where the distance grows with the row length), 8e-7 / 7e-4 / 5.6e-3
    # backward, which reads the row max and row sum as stored.
    if case["kind"] in ("train", "op"):
        return {"rel": {"fp32": 1e-5, "fp16": 3e-3, "bf16": 2e-2}[case["dtype"]]}
    return {"rel": {"fp32": 4e-6, "fp16": 1e-3, "bf16": 8e-3}[case["dtype"]]}


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "softmax":
        x = state["x"].double()
        return torch.log_softmax(x, -1) if case["log"] else torch.softmax(x, -1)
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    heads = {n: state[n].detach().double().reshape(B * H, S, D) for n in ("q", "k", "v", "dout") if n in state}
    scale = 1.0 / math.sqrt(D)
    hidden = torch.ones(S, S, dtype=torch.bool, device="cuda").triu_(1) if case["causal"] else None
    parts = []
    step = max(1, (1 << 26) // (S * S))
    for at in range(0, B * H, step):
        q, k, v = (heads[n][at:at + step] for n in "qkv")
        s = torch.matmul(q, k.transpose(1, 2).contiguous()).mul_(scale)
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        m = s.amax(-1)
        p = s.sub_(m[..., None]).exp_()
        l = p.sum(-1)
        p.div_(l[..., None])
        got = [torch.matmul(p, v), m, l]
        if case["kind"] != "fwd":
            dout = heads["dout"][at:at + step]
            ds = torch.matmul(dout, v.transpose(1, 2).contiguous())
            ds.sub_((dout * got[0]).sum(-1, keepdim=True)).mul_(p)
            got += [torch.matmul(ds, k).mul_(scale), torch.matmul(ds.transpose(1, 2).contiguous(), q).mul_(scale),
                    torch.matmul(p.transpose(1, 2).contiguous(), dout)]
        parts.append(got)
    whole = [torch.cat(p) for p in zip(*parts)]
    names = ("out", "m", "l", "dq", "dk", "dv")
    return {n: t.reshape(B, H, S, D) if t.dim() == 3 else t.reshape(B, H, S) for n, t in zip(names, whole)}
