"""The work that users of this package have it do, as cases that can be timed and whose outputs can be compared.

    listed()           the cases
    draw(rng)          one more case from the ranges that the listed ones stand for
    prepare(case, seed)  what a program holds before the call: tensors on the GPU, slopes, state buffers
    run(state)         one pass through the public entry points
    work(case)         bytes and operations a pass cannot do without
    tolerance(case)    how far a correct implementation at the same precision may be off

A case is one of five kinds of use:
    train    an attention layer's forward and backward on whole sequences: `lightning_attn` and autograd
    prompt   the forward of a prompt that leaves the KV state behind: `lasp_fuse_parallel`'s launch shim
    decode   one new token for every sequence of a batch, the KV states updated in place: `lasp_fuse`'s launch shim
    chunk    one rank's share of a longer sequence, forward and backward, with the states that came from the
             neighbouring ranks: `lasp_fuse_parallel`'s launch shims
    chain    all chunks of a sequence-parallel group, forward and backward, through the `lasp_fuse` operator, one
             process playing every rank
"""
import importlib
import math

import torch

import lasp_amd

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
# The largest pass: forward and backward of 65536 tokens on 16 heads of 128 bf16 features.
MOST_BYTES = 65536 * 16 * 128 * 2 * 11


def _case(kind, b, h, n, d=128, e=128, dtype="bf16", decay=True, chunks=1):
    return {"kind": kind, "b": b, "h": h, "n": n, "d": d, "e": e, "dtype": dtype, "decay": decay, "chunks": chunks}


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # one token for each of 32 sequences: a serving loop's step, which reads and writes every KV state
        named("decode_b32_h16", "decode", 32, 16, 1),
        # the prompt of one request, of no particular length, before such steps
        named("prompt_h16_n2000", "prompt", 1, 16, 2000),
        # the smallest training call: one short sequence on few heads, as in unit tests and small experiments
        named("train_h8_n256", "train", 1, 8, 256),
        # a batch of short sequences in fp16: fine-tuning on short texts
        named("train_fp16_b8_h12_n512", "train", 8, 12, 512, dtype="fp16"),
        # single precision, the correctness configuration of the benchmark: b=2, h=12, n=2048
        named("train_fp32_b2_h12_n2048", "train", 2, 12, 2048, dtype="fp32"),
        # heads of 64 features, as many models have them
        named("train_d64_b4_h16_n4096", "train", 4, 16, 4096, d=64, e=64),
        # queries and keys wider than one launch takes: two feature slices whose outputs add up
        named("train_d256_h8_n8192", "train", 1, 8, 8192, d=256),
        # a batch padded to its longest text, whose length is no multiple of anything
        named("train_b3_h12_n5003", "train", 3, 12, 5003),
        # eight sequence-parallel chunks of 2048 tokens, the benchmark's chunked configuration: b=2, h=12
        named("chain_b2_h12_8x2048", "chain", 2, 12, 2048, chunks=8),
        # one rank's 16384 tokens of a 32-head model with states from both neighbours
        named("chunk_h32_n16384", "chunk", 1, 32, 16384),
        # a long sequence without decay (a linear transformer's feature map, elu + 1) in chunks of 16384
        named("chain_nodecay_h16_8x16384", "chain", 1, 16, 16384, decay=False, chunks=8),
        # the headline configuration: 65536 tokens on 16 heads, forward and backward in one pass
        named("train_h16_n65536", "train", 1, 16, 65536),
    ]


def _between(rng, lo, hi):
    """Log-uniform in [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choices(["train", "prompt", "decode", "chunk", "chain"], [50, 15, 10, 15, 10])[0]
        dtype = rng.choices(["bf16", "fp16", "fp32"], [60, 20, 20])[0]
        h = rng.choice([4, 8, 12, 16, 20, 24, 32])
        b = rng.choice([1, 1, 1, 2, 3, 4, 6, 8])
        d, e = rng.choices([(128, 128), (64, 64), (128, 64), (96, 96), (80, 80), (256, 128), (192, 128)], [60, 14, 6, 6, 4, 6, 4])[0]
        decay = rng.random() < 0.85
        chunks = 1
        if kind == "decode":
            b, n, d, e, decay = _between(rng, 1, 64), 1, min(d, 128), min(e, 128), True
        elif kind == "prompt":
            n, d, e = _between(rng, 16, 32768), min(d, 128), min(e, 128)
        elif kind == "chunk":
            n, d, e = _between(rng, 512, 32768), min(d, 128), min(e, 128)
        elif kind == "chain":
            n, d, e, chunks = _between(rng, 512, 16384), min(d, 128), min(e, 128), rng.choice([2, 4, 8])
        else:
            n = _between(rng, 64, 65536)
        if rng.random() < 0.6:  # lengths that are whole blocks, and lengths that are not
            n = max(n // 64, 1) * 64 if n >= 64 else n
        case = _case(kind, b, h, n, d, e, dtype, decay, chunks)
        # (single precision is bound by arithmetic, at about four times the time a byte)
        if work(case)["bytes"] * (4 if dtype == "fp32" else 1) <= MOST_BYTES:
            return case


def _slopes(case, dev):
    if not case["decay"]:
        return torch.zeros(case["h"], 1, 1, device=dev)
    return lasp_amd.build_slope_tensor(case["h"]).to(dev)


def _chain_group(chunks):
    """One process plays the `chunks` ranks of a sequence-parallel group."""
    if lasp_amd.get_sequence_parallel_world_size() != chunks:
        lasp_amd.destroy_parallel_groups()
        lasp_amd.initialize_lasp(1, chunks)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    b, h, n, d, e = (case[k] for k in "bhnde")
    dtype = DTYPES[case["dtype"]]

    def normal(width):
        return torch.randn(b, h, n, width, generator=g, device=dev)

    def qk():
        x = normal(d)
        x = x / math.sqrt(d) if case["decay"] else (torch.nn.functional.elu(x) + 1) / d  # a non-negative feature map without decay
        return x.to(dtype)

    def ve():
        return (normal(e) / math.sqrt(e)).to(dtype)

    kind = case["kind"]
    state = {"kind": kind, "s": _slopes(case, dev)}
    learns = kind in ("train", "chain")
    parts = []
    for _ in range(case["chunks"]):
        q, k, v = [t.requires_grad_(learns) for t in (qk(), qk(), ve())]
        parts.append((q, k, v, ve() if learns or kind == "chunk" else None))
    state["parts"] = parts

    def kv(std):
        return torch.randn(b, h, d, e, generator=g, device=dev) * std

    if kind == "decode":
        state["KV"] = kv(0.02)
    elif kind == "prompt":
        state["KV"] = kv(0.0)
    elif kind == "chunk":
        state["KV"], state["DKV"] = kv(0.02), kv(0.02)
    elif kind == "chain":
        state["KV"], state["DKV"] = kv(0.0), kv(0.0)
        state["chunks"] = case["chunks"]
        _chain_group(case["chunks"])
    return state


def run(state):
    kind, s = state["kind"], state["s"]
    if kind == "chain":
        outs, dos, leaves = [], [], []
        for c, (q, k, v, do) in enumerate(state["parts"]):
            q.grad = k.grad = v.grad = None
            lasp_amd.set_sequence_parallel_rank(c)
            outs.append(lasp_amd.lasp_fuse(q, k, v, s, state["KV"], state["DKV"]))
            dos.append(do)
            leaves += [q, k, v]
        torch.autograd.backward(outs, dos)
        return outs, [t.grad for t in leaves], state["KV"], state["DKV"]

    q, k, v, do = state["parts"][0]
    if kind == "train":
        q.grad = k.grad = v.grad = None
        o = lasp_amd.lightning_attn(q, k, v, s)
        o.backward(do)
        return o, q.grad, k.grad, v.grad
    if kind == "decode":
        fuse = importlib.import_module("lasp_amd.lasp_fuse")  # (the package's attribute of that name is the operator)
        return fuse.lasp_forward(q, k, v, s, state["KV"]), state["KV"]
    parallel = importlib.import_module("lasp_amd.lasp_fuse_parallel")
    o, kv, kv_out = parallel.lasp_forward(q, k, v, s, state["KV"])
    if kind == "prompt":
        return o, kv_out
    dq, dk, dv, dkv_out = parallel.lasp_backward(q, k, v, s, do, kv, state["KV"], state["DKV"])
    return o, kv_out, dq, dk, dv, dkv_out


def work(case):
    """The forward reads q, k, v and writes o; the backward, which cannot start before the loss is known, reads q, k, v and
    do and writes dq, dk, dv.  Operations: the recurrence token by token (2 d e to update a state and 2 d e to apply it),
    which no blocking undercuts."""
    b, h, n, d, e, chunks = (case[k] for k in ("b", "h", "n", "d", "e", "chunks"))
    rows, size, state = b * h * n * chunks, BYTES[case["dtype"]], 4 * b * h * d * e
    nbytes, flops = rows * size * (2 * d + 2 * e), rows * 4 * d * e
    if case["kind"] in ("train", "chunk", "chain"):
        nbytes += rows * size * (4 * d + 3 * e)
        flops += rows * 10 * d * e
    passes = 2 if case["kind"] in ("chunk", "chain") else 1  # states go both ways where there is a backward
    if case["kind"] != "train":
        nbytes += 2 * state * passes * chunks
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the outputs are off from the same recurrence in 64 bits (largest relative 2-norm over the
    kinds of case: bf16 3.3e-3, fp16 4.1e-4, fp32 3.3e-7; largest single difference 2.9e-2, 3.2e-3, 3.2e-6)."""
    rel = {"bf16": 1.2e-2, "fp16": 1.6e-3, "fp32": 1.4e-6}[case["dtype"]]
    return {"rel": rel, "max": 10 * rel}
