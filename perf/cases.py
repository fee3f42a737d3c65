"""The workloads whose time counts: attention calls as a program that uses this package makes them.

Every case goes through the public functions, ``flash_attention_fn`` and ``flash_attention_qkvpacked_fn``:
a training case is one forward and backward through autograd and returns the output and every gradient, an
inference case is one forward without gradients and returns the output.

A case is a dict of plain values:
  mode    "train" or "infer"
  packed  q, k, v come as one (B, S, 3, H, D) tensor
  B, H, M, N, D, causal, dtype ("bf16" or "fp16")
  bias    "none"
          "dense"   a trainable (B, H, M, N) bias of type bias_dtype
          "shared"  a trainable (1, H, M, N) bias of type bias_dtype, one table for the whole batch
          "alibi"   AlibiBias with fixed slopes, the bias is formed from the indices
          "alibi_tensor"  the same bias as a trainable (1, H, M, N) tensor of type bias_dtype (B is 1)
          "padding"       a bool mask (B, 1, 1, N): False behind the end of each sequence
          "padding_dense" the same mask written out as (B, H, M, N)
"""
import math

import torch

from triton_flashattn_amd import AlibiBias, flash_attention_fn, flash_attention_qkvpacked_fn

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(mode, B, H, M, N, D, causal=False, dtype="bf16", bias="none", bias_dtype="bf16", packed=False):
    return {"mode": mode, "packed": packed, "B": B, "H": H, "M": M, "N": N, "D": D, "causal": causal, "dtype": dtype,
            "bias": bias, "bias_dtype": bias_dtype}


def listed():
    cases = {
        # A training step of a small model, bias parameter in fp32: nothing but launches and host work.
        "train_tiny": _case("train", 2, 4, 128, 128, 64, bias="dense", bias_dtype="fp32"),
        # One generated token per sequence against a key/value cache: a stream over the cache.
        "decode": _case("infer", 8, 16, 1, 4097, 128),
        # Encoding a batch of short sequences of different lengths.
        "encode_padded": _case("infer", 32, 12, 197, 197, 64, bias="padding"),
        # The forward over a long prompt or document.
        "prefill_long": _case("infer", 1, 32, 8192, 8192, 128, causal=True),
        # Language-model training at an ordinary length, fp16, head dim 64.
        "train_causal": _case("train", 4, 16, 2048, 2048, 64, causal=True, dtype="fp16"),
        # ... and on long sequences whose length is no multiple of anything.
        "train_long": _case("train", 1, 16, 6001, 6001, 128, causal=True),
        # A bias with a gradient for every score: what this package is for (the benchmark's workload).
        "train_bias": _case("train", 2, 16, 4096, 4096, 128, bias="dense"),
        # A learned table of relative positions, one for the whole batch, on image-like sequences.
        "train_shared_bias": _case("train", 32, 12, 197, 197, 64, bias="shared", bias_dtype="fp32"),
        # Packed self-attention over padded sequences; the mask is written out, as the plain interface has it.
        "train_packed_mask": _case("train", 8, 12, 1024, 1024, 64, causal=True, bias="padding_dense", packed=True),
        # Cross attention from few queries to many keys, distance penalty as a trainable tensor ...
        "train_cross_bias": _case("train", 1, 32, 1024, 8192, 128, bias="alibi_tensor"),
        # ... and with fixed slopes, computed from the indices.
        "train_cross_alibi": _case("train", 1, 32, 1024, 8192, 128, bias="alibi"),
        # A head dim between those of the kernels.
        "train_head_dim_80": _case("train", 8, 16, 257, 257, 80),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A sequence length: half of them multiples of 64, the others whatever comes."""
    n = _log_int(rng, lo, hi)
    return max(lo, n // 64 * 64) if rng.random() < 0.5 else n


_MAX_FLOPS, _MAX_BYTES = 9.0e11, 3.4e9  # what the largest listed case takes, nearly


def draw(rng):
    kind = rng.choice(["tiny", "decode", "encode", "prefill", "causal", "bias", "shared", "mask", "cross", "head_dim"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "tiny":
        S = _length(rng, 16, 256)
        c = _case("train", rng.randint(1, 4), rng.randint(1, 8), S, S, rng.choice([32, 64]), dtype=dtype, bias="dense",
                  bias_dtype=rng.choice([dtype, "fp32"]))
    elif kind == "decode":
        c = _case("infer", _log_int(rng, 1, 32), rng.choice([8, 12, 16, 32]), rng.choice([1, 1, 1, 4, 7, 16]),
                  _length(rng, 256, 16384), rng.choice([64, 128]), dtype=dtype, bias=rng.choice(["none", "none", "padding"]))
    elif kind == "encode":
        S = _length(rng, 64, 1024)
        c = _case("infer", _log_int(rng, 4, 64), rng.choice([8, 12, 16]), S, S, rng.choice([32, 64, 128]), dtype=dtype,
                  bias=rng.choice(["padding", "padding", "none"]))
    elif kind == "prefill":
        S = _length(rng, 1024, 16384)
        c = _case("infer", rng.randint(1, 4), rng.choice([8, 16, 32]), S, S, rng.choice([64, 128]), causal=True, dtype=dtype)
    elif kind == "causal":
        S = _length(rng, 512, 8192)
        c = _case("train", rng.randint(1, 8), rng.choice([8, 12, 16, 32]), S, S, rng.choice([64, 128]),
                  causal=rng.random() < 0.75, dtype=dtype)
    elif kind == "bias":
        M = _length(rng, 256, 4096)
        N = M if rng.random() < 0.5 else _length(rng, 256, 4096)
        c = _case("train", rng.randint(1, 4), rng.choice([8, 12, 16]), M, N, rng.choice([32, 64, 128]), dtype=dtype,
                  bias="dense", bias_dtype=rng.choice([dtype, dtype, "fp32"]))
    elif kind == "shared":
        S = _length(rng, 49, 577)
        c = _case("train", _log_int(rng, 4, 64), rng.choice([8, 12, 16]), S, S, rng.choice([32, 64]), dtype=dtype,
                  bias="shared", bias_dtype=rng.choice([dtype, "fp32"]))
    elif kind == "mask":
        S = _length(rng, 128, 2048)
        c = _case("train", rng.randint(2, 16), rng.choice([8, 12, 16]), S, S, rng.choice([64, 128]), causal=rng.random() < 0.5,
                  dtype=dtype, bias=rng.choice(["padding", "padding_dense"]), packed=rng.random() < 0.5)
    elif kind == "cross":
        c = _case("train", 1, rng.choice([8, 16, 32]), _length(rng, 64, 1024), _length(rng, 1024, 8192), rng.choice([64, 128]),
                  dtype=dtype, bias=rng.choice(["alibi", "alibi_tensor"]), bias_dtype=dtype)
    else:
        S = _length(rng, 128, 1024)
        c = _case("train", rng.randint(1, 16), rng.choice([8, 12, 16]), S, S, rng.choice([40, 72, 80, 96]), dtype=dtype,
                  causal=rng.random() < 0.25)
    while c["B"] > 1 and (work(c)["flops"] > _MAX_FLOPS or work(c)["bytes"] > _MAX_BYTES):
        c["B"] -= 1
    while c["H"] > 1 and (work(c)["flops"] > _MAX_FLOPS or work(c)["bytes"] > _MAX_BYTES):
        c["H"] //= 2
    return c


def prepare(case, seed):
    """Normal q, k, v and upstream gradients, a bias of the size that trained tables have, sequences that fill
    between half and all of the padded length."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    B, H, M, N, D = (case[n] for n in ("B", "H", "M", "N", "D"))
    dt = _DTYPES[case["dtype"]]
    train = case["mode"] == "train"

    def normal(*shape, dtype=dt):
        return torch.randn(*shape, device=dev, generator=g).to(dtype)

    if case["packed"]:
        inputs = [normal(B, M, 3, H, D)]
    else:
        inputs = [normal(B, M, H, D), normal(B, N, H, D), normal(B, N, H, D)]
    for t in inputs:
        t.requires_grad_(train)
    wanted = list(inputs) if train else []

    kind, bias = case["bias"], None
    if kind in ("dense", "shared"):
        bias = normal(B if kind == "dense" else 1, H, M, N, dtype=_DTYPES[case["bias_dtype"]]).requires_grad_(train)
    elif kind in ("alibi", "alibi_tensor"):
        slopes = (2.0 ** (-8.0 * (torch.arange(H, device=dev) + 1) / H)).float()
        bias = AlibiBias(slopes)
        if kind == "alibi_tensor":
            bias = bias.materialize(M, N, _DTYPES[case["bias_dtype"]]).requires_grad_(train)
    elif kind in ("padding", "padding_dense"):
        lengths = torch.randint((N + 1) // 2, N + 1, (B,), device=dev, generator=g)
        bias = (torch.arange(N, device=dev)[None, :] < lengths[:, None])[:, None, None, :]
        if kind == "padding_dense":
            bias = bias.expand(B, H, M, N).contiguous()
    if isinstance(bias, torch.Tensor) and bias.requires_grad:
        wanted.append(bias)
    return {"call": flash_attention_qkvpacked_fn if case["packed"] else flash_attention_fn, "inputs": inputs, "bias": bias,
            "causal": case["causal"], "wanted": wanted, "dout": normal(B, M, H, D) if train else None}


def run(state):
    if state["dout"] is None:
        with torch.no_grad():
            return state["call"](*state["inputs"], state["bias"], state["causal"])
    out = state["call"](*state["inputs"], state["bias"], state["causal"])
    grads = torch.autograd.grad(out, state["wanted"], state["dout"])
    return (out.detach(),) + tuple(grads)


def work(case):
    """Two matrix products forward and five backward, over the scores that can be visible; q, k, v, the bias and
    the upstream gradient read once, the output and the gradients written once."""
    B, H, M, N, D = (case[n] for n in ("B", "H", "M", "N", "D"))
    train = case["mode"] == "train"
    seen = 0.5 if case["causal"] else 1.0
    flops = 4.0 * B * H * M * N * D * seen * (3.5 if train else 1.0)
    rows = 2 * D * H * (2 * B * M + 2 * B * N)  # q and out, k and v
    if train:
        rows += 2 * D * H * (2 * B * M + 2 * B * N)  # dout and dq, dk and dv
    es = {"bf16": 2, "fp16": 2, "fp32": 4}[case["bias_dtype"]]
    bias = {"none": 0, "dense": B * H * M * N * es * seen, "shared": H * M * N * es * seen, "alibi": 4 * H,
            "alibi_tensor": H * M * N * es * seen, "padding": B * N, "padding_dense": B * H * M * N * seen}[case["bias"]]
    if train and case["bias"] in ("dense", "shared", "alibi_tensor"):
        bias *= 2  # and its gradient
    return {"bytes": float(rows + bias), "flops": flops}


def tolerance(case):
    """Against an evaluation of the same inputs in 64 bits, outputs and gradients are off by 2.0e-3 to 2.6e-3 in bf16
    and 2.6e-4 to 3.4e-4 in fp16 (42 cases, every kind above; the roundings of P, dS and the results); four times that."""
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.4e-3}
