"""What a user of the attention path runs, as cases to be timed: training steps (forward and backward through autograd),
prefill and decode forwards, the padded-batch module, block-sparse attention and attention with a learned bias, from one
prompt of a few dozen tokens to batches that fill the GPU.  Every case goes through the package's public entry points.

A case is a dict of plain values:
  path      train / infer   packed self-attention (flash_attn_unpadded_qkvpacked_func), with / without a backward
            decode          a few new tokens per sequence against a cache of keys (flash_attn_unpadded_kvpacked_func)
            padded          the FlashAttention module on a padded batch with a key padding mask, evaluation
            sparse          block-sparse self-attention, training step (flash_blocksparse_attn_func)
            bias            self-attention with a learned bias shared by the batch, training step
  dtype     fp16 / bf16;   B, H, D: batch entries, heads, head dim;   N: longest sequence (decode: longest cache)
  min_frac  the sequence lengths are spread evenly between min_frac * N and N (1: all equal)
  p, causal, rotary, alibi, new (tokens per sequence of a decode step), density (of the block layout): options of the path
"""
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("flash-attention_amd"))  # the package's folder in the repository this runs in

from flash_attn.flash_attention import FlashAttention  # noqa: E402
from flash_attn.flash_attn_interface import (flash_attn_unpadded_kvpacked_func,  # noqa: E402
                                             flash_attn_unpadded_qkvpacked_func,
                                             flash_attn_unpadded_qkvpacked_rotary_func)
from flash_attn.flash_blocksparse_attn_interface import convert_blockmask, flash_blocksparse_attn_func  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one short prompt of an interactive user: nothing but launches and host work
        dict(name="prompt_short", path="infer", dtype="fp16", B=1, H=12, D=64, N=61, min_frac=1.0, causal=True),
        # one token for each of eight conversations of a serving process, caches of uneven length
        dict(name="decode_b8", path="decode", dtype="bf16", B=8, H=16, D=128, N=4096, min_frac=0.25, new=1),
        # prompts of a serving process, 128-wide heads, uneven lengths
        dict(name="prefill_d128", path="infer", dtype="bf16", B=4, H=16, D=128, N=3001, min_frac=0.2, causal=True),
        # encoder evaluation on a padded batch: unpad, attend, pad
        dict(name="padded_eval", path="padded", dtype="fp16", B=32, H=16, D=64, N=512, min_frac=0.5),
        # BERT training on packed sequences of 256 to 512 tokens with dropout
        dict(name="bert_train", path="train", dtype="fp16", B=8, H=12, D=64, N=512, min_frac=0.5, p=0.1),
        # the big-batch BERT-like step of the published benchmark script (1004 to 1023 tokens, padding mask, dropout)
        dict(name="batch64_train", path="train", dtype="fp16", B=64, H=16, D=64, N=1023, min_frac=0.982, p=0.1),
        # the headline workload: a plain fp16 step at 2048 tokens
        dict(name="plain_train", path="train", dtype="fp16", B=8, H=12, D=64, N=2048, min_frac=1.0),
        # GPT-2 sized training: causal, with rotary embedding at the usual context, plain at a long one
        dict(name="gpt_rotary_train", path="train", dtype="bf16", B=8, H=12, D=64, N=1024, min_frac=1.0, causal=True, rotary=True),
        dict(name="gpt_long_train", path="train", dtype="bf16", B=8, H=12, D=64, N=4096, min_frac=1.0, causal=True),
        # a model with 128-wide heads, causal
        dict(name="d128_train", path="train", dtype="bf16", B=16, H=12, D=128, N=2048, min_frac=1.0, causal=True),
        # long documents under a fixed block layout at the interface's own granularity (16 queries x 256 keys)
        dict(name="sparse_train", path="sparse", dtype="fp16", B=4, H=16, D=64, N=4096, min_frac=1.0, density=0.25),
        # attention with a learned (1, heads, N, N) bias, ragged batch, small heads
        dict(name="bias_train", path="bias", dtype="fp16", B=8, H=8, D=32, N=701, min_frac=0.6),
    ]


def _lens(c):
    """Sequence lengths of a case, longest first (prepare() shuffles them)."""
    lo, hi, B = max(1, round(c["min_frac"] * c["N"])), c["N"], c["B"]
    return [hi - (hi - lo) * i // max(1, B - 1) for i in range(B)]


def _active_blocks(c):
    """(rows of 16 queries, columns of 256 keys, active blocks) of a sparse case's layout: the diagonal and as many others
    as make up the density."""
    rows, cols = -(-c["N"] // 16), -(-c["N"] // 256)
    diagonal = rows
    return rows, cols, diagonal + max(0, round((c["density"] - diagonal / (rows * cols)) * rows * cols))


def _flops(c):
    lens = _lens(c)
    if c["path"] == "decode":
        return sum(4.0 * c["H"] * c["D"] * c["new"] * n for n in lens)
    if c["path"] == "sparse":
        rows, cols, active = _active_blocks(c)
        scores = sum(float(n) * n for n in lens) * active / (rows * cols)
    else:
        scores = sum(n * (n + 1) / 2.0 if c.get("causal") else float(n) * n for n in lens)
    return 4.0 * c["H"] * c["D"] * scores * (1.0 if c["path"] in ("infer", "padded") else 3.5)


def work(case):
    """The products of the forward (two) and of the backward (five), and every input read and output written once."""
    lens, row = _lens(case), case["H"] * case["D"] * 2
    total = sum(lens)
    if case["path"] == "decode":
        nbytes = (2 * total + 2 * case["B"] * case["new"]) * row
    elif case["path"] == "padded":
        nbytes = 3 * total * row + case["B"] * case["N"] * (row + 1)  # the valid rows of qkv, the whole padded output
    elif case["path"] == "infer":
        nbytes = 4 * total * row
    else:
        nbytes = 8 * total * row  # q, k, v, dout; out, dq, dk, dv
        if case["path"] == "bias":
            nbytes += 2 * case["H"] * case["N"] ** 2 * 2
    return {"bytes": float(nbytes), "flops": _flops(case)}


def tolerance(case):
    # Results, probabilities and score gradients are rounded to the element type between fp32 sums.  Measured against the
    # closed form in 64 bits (D 32 .. 128, up to 1021 tokens, causal or not, with a bias): out, dq, dk, dv, dbias are off by
    # 2.2e-4 .. 3.2e-4 of their norm in fp16 and 1.8e-3 .. 2.6e-3 in bf16, single values by up to 0.008 and 0.075 of the
    # root mean square (causal: the first rows attend to few keys).  Four times that.
    return {"rel": 1.2e-3, "max": 0.03} if case["dtype"] == "fp16" else {"rel": 1e-2, "max": 0.3}


def draw(rng):
    def log_int(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    path = rng.choice(["train", "train", "train", "infer", "infer", "decode", "padded", "sparse", "bias"])
    c = dict(path=path, dtype=rng.choice(["fp16", "bf16"]), H=rng.choice([8, 12, 16]), D=rng.choice([32, 64, 64, 128]),
             min_frac=rng.choice([1.0, round(rng.uniform(0.2, 0.95), 3)]))
    most_flops, batch = 4e11, (1, 64)
    if path == "train":
        c.update(N=log_int(100, 6000), p=rng.choice([0.0, 0.0, 0.1]), causal=rng.random() < 0.5)
        if c["p"] == 0.0 and c["causal"]:
            c.update(rng.choice([{}, {"rotary": True}, {"alibi": True}]))
    elif path == "infer":
        c.update(N=log_int(16, 8000), causal=rng.random() < 0.7)
    elif path == "decode":
        c.update(D=rng.choice([64, 128]), N=log_int(200, 12000), new=rng.choice([1, 1, 1, 2, 5]))
        most_flops = 1e9 * c["new"]  # (bound by the bytes of the cache: 1 GB)
    elif path == "padded":
        c.update(dtype="fp16", D=rng.choice([32, 64]), N=log_int(64, 1500), min_frac=round(rng.uniform(0.3, 0.9), 3))
    elif path == "sparse":
        c.update(D=64, N=log_int(1000, 8000), min_frac=1.0, density=round(rng.uniform(0.15, 0.4), 3))
        batch = (1, 8)
    else:
        c.update(D=rng.choice([32, 64]), N=log_int(100, 1100))
        batch = (1, 8)
    c["B"] = 1
    one = _flops(c)
    most = max(1, min(batch[1], int(most_flops / one)))
    c["B"] = log_int(1, most) if most > 1 else 1
    return c


def prepare(case, seed):
    dev, dtype = torch.device("cuda", torch.cuda.current_device()), _DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    path, B, H, D, N = case["path"], case["B"], case["H"], case["D"], case["N"]
    lens = torch.tensor(_lens(case), dtype=torch.int32)[torch.randperm(B, generator=host)]
    total = int(lens.sum())

    def normal(*shape):
        return torch.randn(*shape, device=dev, dtype=torch.float32, generator=gen).to(dtype)

    def cumulative(n):
        return torch.cat([n.new_zeros(1), n.cumsum(0, dtype=torch.int32)]).to(dev)

    s = {"case": case, "seed": seed, "cu": cumulative(lens), "gen": torch.cuda.default_generators[dev.index]}
    if path == "decode":
        s.update(q=normal(B * case["new"], H, D), kv=normal(total, 2, H, D),
                 cu_q=cumulative(torch.full((B,), case["new"], dtype=torch.int32)))
        return s
    if path == "padded":
        s["qkv"] = normal(B, N, 3, H, D)
        s["mask"] = type("Mask", (), {"bool_matrix": (torch.arange(N)[None, :] < lens[:, None]).to(dev)})
        s["module"] = FlashAttention(attention_dropout=0.1).eval()
        return s
    s["qkv"] = normal(total, 3, H, D)
    if path == "infer":
        return s
    s["qkv"].requires_grad_()
    s["dout"] = normal(total, H, D)
    if case.get("rotary"):
        angle = torch.outer(torch.arange(N, device=dev, dtype=torch.float32),
                            10000.0 ** (-torch.arange(0, D, 2, device=dev, dtype=torch.float32) / D))
        s["rotary"] = (torch.cos(angle).to(dtype), torch.sin(angle).to(dtype))
    if case.get("alibi"):
        s["alibi"] = 2.0 ** (-8.0 * torch.arange(1, H + 1, device=dev, dtype=torch.float32) / H)
    if path == "bias":
        s["bias"] = normal(1, H, N, N).requires_grad_()
    if path == "sparse":
        rows, cols, active = _active_blocks(case)
        layout = torch.zeros(rows, cols, dtype=torch.bool)
        layout[torch.arange(rows), torch.arange(rows) // 16] = True
        free = (~layout).flatten().nonzero().flatten()
        layout.view(-1)[free[torch.randperm(free.numel(), generator=host)[: active - rows]]] = True
        s["layout"] = convert_blockmask(layout.to(dev), causal=False)  # once per layout, as the modules keep it
    return s


def run(state):
    s, c = state, state["case"]
    path, N = c["path"], c["N"]
    if path == "decode":
        with torch.no_grad():
            return flash_attn_unpadded_kvpacked_func(s["q"], s["kv"], s["cu_q"], s["cu"], c["new"], N, 0.0)
    if path == "infer":
        with torch.no_grad():
            return flash_attn_unpadded_qkvpacked_func(s["qkv"], s["cu"], N, 0.0, causal=c["causal"])
    if path == "padded":
        with torch.no_grad():
            return s["module"](s["qkv"], key_padding_mask=s["mask"])[0]
    wanted = (s["qkv"],)
    if path == "sparse":
        out = flash_blocksparse_attn_func(s["qkv"], s["cu"], s["layout"], 0.0, N, convert_mask=False)
    elif path == "bias":
        out = flash_attn_unpadded_qkvpacked_func(s["qkv"], s["cu"], N, 0.0, attn_bias=s["bias"])
        wanted = (s["qkv"], s["bias"])
    elif c.get("rotary"):
        out = flash_attn_unpadded_qkvpacked_rotary_func(s["qkv"], *s["rotary"], s["cu"], N, 0.0, causal=c["causal"])
    else:
        p = c.get("p", 0.0)
        if p > 0.0:
            s["gen"].manual_seed(s["seed"])  # a reproducible step: the mask follows the generator
        out = flash_attn_unpadded_qkvpacked_func(s["qkv"], s["cu"], N, p, causal=c.get("causal", False), alibi_slopes=s.get("alibi"))
    return (out,) + torch.autograd.grad(out, wanted, s["dout"])
