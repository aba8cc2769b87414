#!/usr/bin/env python3
"""Benchmark of the hot path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--no-extras]

One step = forward + backward of causal decayed linear attention through the
public operator (lightning_attn + autograd) on the headline workload (TNL-1B head shape):
b=1, h=16, n=65536, d=e=128, bf16, Q/K/V/dO ~ N(0,1)/sqrt(d), slopes
2^(-8(i+1)/16); inputs are resident in HBM before the timed region.
Prints ONE JSON line (metric = fwd+bwd tokens/s) that also carries
  roofline     -- la_bwd3, the dominant kernel, against the HBM roof: algorithmic
                  bytes per launch / its mean launch duration (HIP events around
                  every launch, on the launch stream); roofline_fwd: the same for la_apply.
                  `traffic` is read from the rocprofv3 counter summary under profiles/
                  and is null when that summary was taken with another segment plan or another
                  state of the kernels' source.
  cpu_baseline -- the CPU oracle (fp32 torch port of the same recurrence) timed on
                  the host cores on a bounded number of passes of the same workload.
  other_configs -- forward+backward times of the other benchmark configurations
                  (0: fp32; 1: single pass and as 8 chunks through lasp_fuse and
                  lasp_fuse_parallel; 3: one chunk with incoming KV; 4: 1M tokens as
                  64 chunks, with and without decay), each with tokens/s and canonical
                  TFLOP/s, each timed after 100 ms of the same work.

Order of the run: the other configurations; W warm-up and K timed steps of the headline step as they
come (`ms_per_step_unsettled`); a settling phase (--settle-ms, default 150 ms of the headline step,
untimed); then the W warm-up steps and the K timed steps behind `value` (`warmup_effective` counts
every untimed step before them).  The settling
phase is there because the part answers every change of load with a power-management transient:
for about 30 ms after these kernels start -- from idle or straight after other GPU work -- every
kernel runs 5-30 % slower, back to back with no gaps between them, and then settles.  A training
job sits in the settled regime, so that is what the timed steps measure; `settle_ms` is
recorded in the output, and --settle-ms 0 shows the transient.
"""
import argparse
import hashlib
import json
import os
import re
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

B, H, N, D = 1, 16, 65536, 128
FLOP_FWD_PER_TH = 98304        # 2Bd + 2Be + 4de at B=64, d=e=128
FLOP_BWD_PER_TH = 245760       # 6Bd + 4Be + 10de
BYTES_FWD_PER_TH = 1024        # read Q,K,V + write O, bf16
BYTES_BWD_PER_TH = 1792        # read Q,K,V,dO + write dQ,dK,dV
HBM_PEAK_GBS = 8000.0
MFMA_BF16_PEAK_TFLOPS = 2500.0
F32_PRODUCTS = 6  # bf16 products that the fp32 kernels make of one
HBM_PROFILE = os.path.join(ROOT, "profiles", "pmc_hbm_bytes_config2.txt")


def slopes(h):
    return torch.tensor([2.0 ** (-8.0 * (i + 1) / h) for i in range(h)], dtype=torch.float32).reshape(h, 1, 1)


def make_inputs(device, n=N, seed=2):
    g = torch.Generator().manual_seed(seed)
    mk = lambda: (torch.randn(B, H, n, D, generator=g) / D ** 0.5).to(torch.bfloat16)
    q, k, v, do = mk(), mk(), mk(), mk()
    return [t.to(device) for t in (q, k, v, do)]


def device_inputs(dev, b, h, n, d, dtype, seed, scale):
    g = torch.Generator(device=dev).manual_seed(seed)
    return [(torch.randn(b, h, n, d, generator=g, device=dev) * scale).to(dtype) for _ in range(4)]


def kernel_code():
    """A short hash of the sweep kernels' source without its comments."""
    code = hashlib.sha256()
    for name in ("lasp_common.h", "lasp_mfma.hip"):
        with open(os.path.join(ROOT, "lasp_amd", "csrc", name)) as f:
            code.update("".join(re.sub(r"//.*", "", f.read()).split()).encode())
    return code.hexdigest()[:16]


def read_traffic_profile(path=HBM_PROFILE):
    """HBM bytes per launch from the committed rocprofv3 FETCH_SIZE / WRITE_SIZE summary.

    The file states the segment plan it was taken with (`plan: seg_len=.. n_seg=..`), the kernels' source (`code: ..`, see
    kernel_code), the scale factor of each counter (from a plain device copy of known size) and one
    `traffic <kernel> fetch_kib=.. write_kib=..` line per kernel.  Returns {"seg_len", "n_seg", "code", "kernels": {name: bytes}}
    or None if there is no such file."""
    try:
        text = open(path).read()
    except OSError:
        return None
    plan = re.search(r"plan:\s*seg_len=(\d+)\s+n_seg=(\d+)", text)
    scale = re.search(r"scale:\s*fetch=([0-9.]+)\s+write=([0-9.]+)", text)
    code = re.search(r"^code:\s*(\w+)", text, flags=re.M)
    if not plan or not scale or not code:
        return None
    f_scale, w_scale = float(scale.group(1)), float(scale.group(2))
    kernels = {}
    for m in re.finditer(r"^traffic\s+(\S+)\s+fetch_kib=([0-9.]+)\s+write_kib=([0-9.]+)", text, flags=re.M):
        kernels[m.group(1)] = int((float(m.group(2)) * f_scale + float(m.group(3)) * w_scale) * 1024)
    return {"seg_len": int(plan.group(1)), "n_seg": int(plan.group(2)), "code": code.group(1), "kernels": kernels}


CEILING_PROFILE = os.path.join(ROOT, "profiles", "stream_probe_hbm_ceiling.txt")


def read_ceiling_profile(path=CEILING_PROFILE):
    """{"4:3": GB/s, ...} from the committed summary of `bench.py --stream-probe` (lines `ceiling mix=R:W gbs=...`),
    or None if there is no such file."""
    try:
        text = open(path).read()
    except OSError:
        return None
    found = {m.group(1): float(m.group(2)) for m in re.finditer(r"^ceiling\s+mix=(\d+:\d+)\s+gbs=([0-9.]+)", text, flags=re.M)}
    return found or None


def stream_probe(dev, mib_each, iters):
    """What the memory system sustains for the sweeps' access pattern with no arithmetic: R read and W write
    streams of `mib_each` MiB through lasp_stream_probe, best grid of a small sweep, next to a plain device copy."""
    from lasp_amd import _abi

    n = mib_each << 20
    bufs = [torch.empty(n, dtype=torch.uint8, device=dev).fill_(1) for _ in range(10)]
    rows = []

    def timed(fn):
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(iters):
            fn()
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) / iters

    ms = timed(lambda: bufs[1].copy_(bufs[0]))
    rows.append({"mix": "copy_", "reads": 1, "writes": 1, "grid": None, "us": ms * 1e3, "gbs": 2 * n / ms / 1e6})
    for r, w in ((1, 0), (2, 0), (4, 0), (0, 1), (1, 1), (3, 1), (4, 3), (7, 3)):
        best = None
        for grid in (512, 1024, 2048, 4096, 8192):
            ms = timed(lambda: _abi.stream_probe(bufs[:r], bufs[r:r + w], grid))
            if best is None or ms < best[1]:
                best = (grid, ms)
        rows.append({"mix": f"{r}:{w}", "reads": r, "writes": w, "grid": best[0], "us": best[1] * 1e3,
                     "gbs": (r + w) * n / best[1] / 1e6})
    return rows


def cpu_cores():
    cores = int(os.environ.get("OMP_NUM_THREADS", "0")) or (os.cpu_count() or 1)
    return min(cores, os.cpu_count() or cores)


def cpu_time_passes(fn, budget_s, max_passes):
    passes, t0 = 0, time.perf_counter()
    while True:
        fn()
        passes += 1
        if time.perf_counter() - t0 >= budget_s or passes >= max_passes:
            break
    return (time.perf_counter() - t0) / passes, passes


def cpu_baseline():
    """Oracle port (oracle/lasp_oracle.py: ref_chunked, fp32, block 64) on all host cores: the headline
    workload for about 10 s, configurations 0 and 3 for a few seconds each."""
    from oracle import lasp_oracle as O

    cores = cpu_cores()
    torch.set_num_threads(cores)
    q, k, v, do = [t.float() for t in make_inputs("cpu")]
    s = slopes(H)
    O.ref_chunked(q[:, :, :1024], k[:, :, :1024], v[:, :, :1024], s, do[:, :, :1024])  # warm the thread pool
    dt, passes = cpu_time_passes(lambda: O.ref_chunked(q, k, v, s, do, block=64, dtype=torch.float32), 10.0, 16)
    out = {
        "value": B * N / dt,
        "unit": "tokens/s",
        "cores": cores,
        "kind": "port",
        "sample": f"{passes} fwd+bwd passes of the full workload (b={B} h={H} n={N} d={D}), fp32 torch, {dt:.2f} s each",
        "gflops": (FLOP_FWD_PER_TH + FLOP_BWD_PER_TH) * B * H * N / dt / 1e9,
    }
    del q, k, v, do
    g = torch.Generator().manual_seed(0)
    q0, k0, v0, do0 = [torch.randn(2, 12, 2048, 128, generator=g) for _ in range(4)]
    dt0, p0 = cpu_time_passes(lambda: O.ref_chunked(q0, k0, v0, slopes(12), do0, block=64, dtype=torch.float32), 3.0, 64)
    g = torch.Generator().manual_seed(3)
    q3, k3, v3, do3 = [torch.randn(1, 32, 16384, 128, generator=g) / D ** 0.5 for _ in range(4)]
    kv3 = torch.randn(1, 32, 128, 128, generator=g) * 0.02
    dt3, p3 = cpu_time_passes(lambda: O.ref_chunked(q3, k3, v3, slopes(32), do3, kv3, None, block=64,
                                                    dtype=torch.float32), 4.0, 16)
    out["other_configs"] = {
        "config0_fp32": {"tokens_per_s": 2 * 2048 / dt0, "ms": dt0 * 1e3, "passes": p0},
        "config3_chunk_with_kv_in": {"tokens_per_s": 16384 / dt3, "ms": dt3 * 1e3, "passes": p3},
    }
    return out


def gpu_time(fn, iters, warm=3, settle_ms=100.0):
    """Mean wall time of `fn` in ms over `iters` back-to-back calls, after `warm` first calls and
    `settle_ms` of the same work (the part's clocks settle some tens of ms after the load changes)."""
    for _ in range(warm):
        fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    while (time.perf_counter() - t0) * 1e3 < settle_ms:
        for _ in range(4):
            fn()
        torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(iters):
        fn()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / iters * 1e3


def rates(ms, b, h, n):
    th = b * h * n
    return {
        "fwd_bwd_ms": ms,
        "tokens_per_s": b * n / (ms * 1e-3),
        "tflops": (FLOP_FWD_PER_TH + FLOP_BWD_PER_TH) * th / (ms * 1e-3) / 1e12,
        "algorithmic_gbs": None,
    }


def with_bytes(r, b, h, n, elem_bytes):
    r["algorithmic_gbs"] = (BYTES_FWD_PER_TH + BYTES_BWD_PER_TH) * (elem_bytes / 2) * b * h * n / (r["fwd_bwd_ms"] * 1e-3) / 1e9
    return r


def single_pass_step(lasp_amd, q, k, v, do, s):
    def step():
        q.grad = k.grad = v.grad = None
        lasp_amd.lightning_attn(q, k, v, s).backward(do)

    return step


def chain_step(lasp_amd, op, parts, s, KV, DKV):
    """Forward over the chunks in order, backward in reverse, through a public chunk operator with the
    loopback standing in for the neighbouring ranks (one process plays every sequence-parallel rank)."""
    chunks = len(parts)

    grads = [p[3] for p in parts]

    def step():
        outs = []
        for c, (q, k, v, _do) in enumerate(parts):
            q.grad = k.grad = v.grad = None
            lasp_amd.set_sequence_parallel_rank(c)
            outs.append(op(q, k, v, s, KV, DKV))
        # one backward over the whole chain, as a model that sums the chunks' losses would run it: autograd
        # visits the chunk operators last-created first, which is the order the dKV chain needs
        torch.autograd.backward(outs, grads)

    return step


def graph_of(step):
    """One HIP graph holding everything `step` launches. The library's entry points allocate nothing and
    clear no memory with memset nodes, so a whole forward + backward chain records cleanly; torch's
    allocator serves the temporaries from the graph's own pool."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    torch.cuda.synchronize()
    return graph


def split_chunks(tensors, chunks):
    """Contiguous per-chunk leaves (each rank of a real run owns its chunk as a tensor of its own)."""
    n = tensors[0].shape[2]
    step = n // chunks
    parts = []
    for c in range(chunks):
        sl = slice(c * step, (c + 1) * step)
        q, k, v, do = [t[:, :, sl].contiguous() for t in tensors]
        parts.append((q.requires_grad_(True), k.requires_grad_(True), v.requires_grad_(True), do))
    return parts


def other_configs(dev):
    """Forward+backward times of benchmark configurations 0, 1, 3 and 4 (synthetic inputs of their shapes)."""
    import importlib

    import lasp_amd

    LF = importlib.import_module("lasp_amd.lasp_fuse")
    out = {}

    # configuration 0: fp32, b=2 h=12 n=2048, single pass
    b, h, n = 2, 12, 2048
    q, k, v, do = device_inputs(dev, b, h, n, D, torch.float32, 10, 1.0)
    for t in (q, k, v):
        t.requires_grad_(True)
    r = with_bytes(rates(gpu_time(single_pass_step(lasp_amd, q, k, v, do, slopes(h).to(dev)), 50), b, h, n), b, h, n, 4)
    r["frac_bf16_mfma_peak"] = r["tflops"] * F32_PRODUCTS / MFMA_BF16_PEAK_TFLOPS
    out["config0_fp32_single_pass"] = r
    del q, k, v, do

    # configuration 1: bf16, b=2 h=12 n=16384; single pass, then 8 chunks of 2048 with KV / DKV carry
    b, h, n, chunks = 2, 12, 16384, 8
    tensors = device_inputs(dev, b, h, n, D, torch.bfloat16, 11, 1.0)
    s = slopes(h).to(dev)
    q, k, v, do = tensors
    ql, kl, vl = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out["config1_single_pass"] = with_bytes(rates(gpu_time(single_pass_step(lasp_amd, ql, kl, vl, do, s), 30), b, h, n), b, h, n, 2)
    del ql, kl, vl
    parts = split_chunks(tensors, chunks)
    KV = torch.empty(b, h, D, D, device=dev)
    DKV = torch.empty_like(KV)
    for name in ("lasp_fuse", "lasp_fuse_parallel"):
        lasp_amd.destroy_parallel_groups()
        lasp_amd.initialize_lasp(1, chunks)
        try:
            step = chain_step(lasp_amd, getattr(lasp_amd, name), parts, s, KV, DKV)
            ms = gpu_time(step, 20)
            # the same chain replayed from one HIP graph: takes the host's launch work out of the figure
            graph = graph_of(step)
            graph_ms = gpu_time(graph.replay, 20)
            del graph
        finally:
            lasp_amd.destroy_parallel_groups()
        r = with_bytes(rates(ms, b, h, n), b, h, n, 2)
        r["chunks"] = chunks
        r["vs_single_pass"] = ms / out["config1_single_pass"]["fwd_bwd_ms"]
        r["hip_graph_replay_ms"] = graph_ms
        out[f"config1_chain_{name}"] = r
    del tensors, parts, q, k, v, do

    # configuration 3: bf16, b=1 h=32, one chunk of 16384 with incoming KV ~ N(0, 0.02), DKV_in = 0,
    # through lasp_fuse's launch shims (KV and DKV updated in place)
    b, h, n = 1, 32, 16384
    q, k, v, do = device_inputs(dev, b, h, n, D, torch.bfloat16, 13, D ** -0.5)
    s = slopes(h).to(dev)
    g = torch.Generator(device=dev).manual_seed(14)
    kv_in = torch.randn(b, h, D, D, generator=g, device=dev) * 0.02
    KV, DKV = torch.empty_like(kv_in), torch.empty_like(kv_in)

    def step3():
        KV.copy_(kv_in)
        DKV.zero_()
        LF.lasp_forward(q, k, v, s, KV)
        LF.lasp_backward(q, k, v, s, do, kv_in, DKV)

    out["config3_chunk_with_kv_in"] = with_bytes(rates(gpu_time(step3, 30), b, h, n), b, h, n, 2)
    del q, k, v, do

    # configuration 4a: bf16, b=1 h=16 n=1 048 576 as 64 chunks of 16384 through lasp_fuse
    b, h, chunks, step = 1, 16, 64, 16384
    n = chunks * step
    s = slopes(h).to(dev)
    parts = []
    for c in range(chunks):
        q, k, v, do = device_inputs(dev, b, h, step, D, torch.bfloat16, 1000 + c, D ** -0.5)
        parts.append((q.requires_grad_(True), k.requires_grad_(True), v.requires_grad_(True), do))
    KV = torch.empty(b, h, D, D, device=dev)
    DKV = torch.empty_like(KV)
    lasp_amd.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, chunks)
    try:
        ms = gpu_time(chain_step(lasp_amd, lasp_amd.lasp_fuse, parts, s, KV, DKV), 3, warm=1)
    finally:
        lasp_amd.destroy_parallel_groups()
    r = with_bytes(rates(ms, b, h, n), b, h, n, 2)
    r["chunks"] = chunks
    out["config4a_1m_tokens_chain_lasp_fuse"] = r

    # configuration 4b: the same chain without decay (s = 0), q and k passed through elu(x) + 1
    with torch.no_grad():
        for q, k, _v, _do in parts:
            for t in (q, k):
                t.copy_(torch.nn.functional.elu(t.float() * D ** 0.5) + 1)
    s0 = torch.zeros(h, 1, 1, device=dev)
    lasp_amd.initialize_lasp(1, chunks)
    try:
        ms = gpu_time(chain_step(lasp_amd, lasp_amd.lasp_fuse, parts, s0, KV, DKV), 3, warm=1)
    finally:
        lasp_amd.destroy_parallel_groups()
    r = with_bytes(rates(ms, b, h, n), b, h, n, 2)
    r["chunks"] = chunks
    out["config4b_1m_tokens_no_decay_chain_lasp_fuse"] = r
    del parts
    torch.cuda.empty_cache()
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-extras", action="store_true", help="skip the other configurations (profiling runs)")
    ap.add_argument("--settle-ms", type=float, default=150.0,
                    help="run the headline step untimed for this long before the warm-up steps (see the module docstring)")
    ap.add_argument("--chain-only", action="store_true",
                    help="run only configuration 1's 8-chunk chain through lasp_fuse and print its time (profiling runs)")
    ap.add_argument("--stream-probe", action="store_true",
                    help="run only the streaming-bandwidth probe (read:write mixes with no arithmetic) and print its table")
    ap.add_argument("--probe-mib", type=int, default=1024, help="size of each stream of the probe, MiB")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also run one plain 1 GiB device copy (reference point for rocprofv3 byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        sys.exit("bench.py: this build runs on ONE GPU (no collectives, no sharding); use --gpus 1")
    if not torch.cuda.is_available():
        sys.exit("bench.py: no GPU visible")

    import lasp_amd
    from lasp_amd import _abi

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)

    if args.stream_probe:
        rows = stream_probe(dev, args.probe_mib, 20)
        print(f"# streaming probe: streams of {args.probe_mib} MiB each, 16 KiB pieces, 16-byte accesses, "
              f"non-temporal stores; best of grids 512..8192; {torch.cuda.get_device_name(dev)}")
        for r in rows:
            print(f"ceiling mix={r['mix']} gbs={r['gbs']:.0f}  # footprint {(r['reads'] + r['writes']) * args.probe_mib} MiB, "
                  f"{r['us']:.1f} us per launch, grid {r['grid']}")
        print(json.dumps({"stream_probe": rows, "mib_each": args.probe_mib}))
        return

    if args.chain_only:
        b, h, n, chunks = 2, 12, 16384, 8
        parts = split_chunks(device_inputs(dev, b, h, n, D, torch.bfloat16, 11, 1.0), chunks)
        KV = torch.empty(b, h, D, D, device=dev)
        lasp_amd.initialize_lasp(1, chunks)
        ms = gpu_time(chain_step(lasp_amd, lasp_amd.lasp_fuse, parts, slopes(h).to(dev), KV, torch.empty_like(KV)),
                      args.steps, warm=args.warmup, settle_ms=args.settle_ms)
        lasp_amd.destroy_parallel_groups()
        print(json.dumps({"workload": "config 1 as 8 chunks of 2048 tokens through lasp_fuse (loopback), forward + backward",
                          "ms_per_step": ms, "steps": args.steps, "chunk_plan": _abi.plan(b, h, n // chunks, D, D, torch.bfloat16)[:2]}))
        return

    # the headline inputs are made (on the host, seeded) before anything runs on the GPU, so that no idle
    # stretch separates the other configurations from the headline's warm-up
    q, k, v, do = make_inputs(dev)
    extras = None if args.no_extras else other_configs(dev)
    q.requires_grad_(True)
    k.requires_grad_(True)
    v.requires_grad_(True)
    s = slopes(H).to(dev)
    assert _abi.kernel_path(B, H, N, D, D, torch.bfloat16) == _abi.PATH_MFMA
    seg_len, n_seg, _ = _abi.plan(B, H, N, D, D, torch.bfloat16)

    if args.copy_calibration:
        src = torch.empty(1 << 29, dtype=torch.bfloat16, device=dev).fill_(1.0)  # 1 GiB
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst

    step = single_pass_step(lasp_amd, q, k, v, do, s)

    def fwd_only():
        with torch.no_grad():
            lasp_amd.lightning_attn(q, k, v, s)

    for _ in range(3):  # first calls: library load, kernel attributes, allocator growth
        step()
    torch.cuda.synchronize()
    # the driver's regime as it stands: W warm-up steps, then K timed steps, before any settling
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_step_unsettled = (time.perf_counter() - t0) / args.steps * 1e3
    settle_steps = 0
    t0 = time.perf_counter()
    while (time.perf_counter() - t0) * 1e3 < args.settle_ms:
        for _ in range(10):
            step()
        torch.cuda.synchronize()
        settle_steps += 10
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ms_step = dt / args.steps * 1e3

    # forward alone
    fwd_only()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        fwd_only()
    torch.cuda.synchronize()
    ms_fwd = (time.perf_counter() - t0) / args.steps * 1e3

    # per-kernel durations: the same K steps again with every launch bracketed by events
    _abi.profile_begin(16 * args.steps + 16)
    for _ in range(args.steps):
        step()
    prof = _abi.profile_end()
    th = B * H * N
    kernel_sum_ms = sum(ms for ms, cnt in prof.values()) / args.steps

    profile = read_traffic_profile()
    same_plan = profile is not None and (profile["seg_len"], profile["n_seg"], profile["code"]) == (seg_len, n_seg, kernel_code())

    ceilings = read_ceiling_profile()

    def roof(kernel, cls, alg_bytes, mix):
        ms, cnt = prof[cls]
        avg_ms = ms / max(cnt, 1)
        achieved = alg_bytes / (avg_ms * 1e-3) / 1e9
        extra = {}
        if ceilings and mix in ceilings:
            # what a kernel that only streams this read:write mix reached on this part (profiles/)
            extra = {"measured_ceiling": ceilings[mix], "measured_ceiling_mix": mix,
                     "frac_of_measured_ceiling": achieved / ceilings[mix],
                     "measured_ceiling_source": os.path.relpath(CEILING_PROFILE, ROOT)}
        return {
            **extra,
            "kernel": kernel, "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": profile["kernels"].get(kernel) if same_plan else None,
            "traffic_source": os.path.relpath(HBM_PROFILE, ROOT) if same_plan else None,
            "algorithmic_bytes_per_launch": alg_bytes, "avg_launch_ms": avg_ms, "launches": cnt,
        }

    flop_step = (FLOP_FWD_PER_TH + FLOP_BWD_PER_TH) * th
    tflops = flop_step / (ms_step * 1e-3) / 1e12

    out = {
        "metric": "fwd+bwd tokens/s, causal decayed linear attention, h=16 d=128 n=64K, 1 MI355X",
        "value": B * N / (ms_step * 1e-3),
        "unit": "tokens/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "settle_ms": args.settle_ms,
        "settle_steps": settle_steps,
        # untimed steps that ran before the timed ones: first calls, the unsettled measurement (W + K), settling, W
        "warmup_effective": 3 + args.warmup + args.steps + settle_steps + args.warmup,
        "ms_per_step": ms_step,
        # K steps timed straight after 3 first calls and W warm-up steps, before the settling phase
        "ms_per_step_unsettled": ms_step_unsettled,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic",
        "config": {
            "workload": "TNL-1B attention head shape: lightning_attn fwd+bwd, b=1 h=16 n=65536 d=e=128, single pass, no KV state",
            "seg_len": seg_len,
            "n_seg": n_seg,
        },
        "fwd_ms": ms_fwd,
        "fwd_tokens_per_s": B * N / (ms_fwd * 1e-3),
        "fwd_tflops": FLOP_FWD_PER_TH * th / (ms_fwd * 1e-3) / 1e12,
        "fwd_bwd_tflops": tflops,
        "frac_bf16_mfma_peak": tflops / MFMA_BF16_PEAK_TFLOPS,
        "step_algorithmic_gbs": (BYTES_FWD_PER_TH + BYTES_BWD_PER_TH) * th / (ms_step * 1e-3) / 1e9,
        "frac_hbm_peak_step": (BYTES_FWD_PER_TH + BYTES_BWD_PER_TH) * th / (ms_step * 1e-3) / 1e9 / HBM_PEAK_GBS,
        "kernel_ms": {name: {"total_ms": ms, "launches": cnt} for name, (ms, cnt) in prof.items() if cnt},
        "kernel_sum_ms_per_step": kernel_sum_ms,
        # dominant kernel: la_bwd3 (one launch = the whole backward sweep: reads Q,K,V,dO, writes dQ,dK,dV)
        "roofline": roof("la_bwd3", "bwd3", BYTES_BWD_PER_TH * th, "4:3"),
        # second kernel: la_apply (one launch = the forward sweep: reads Q,K,V, writes O)
        "roofline_fwd": roof("la_apply", "apply", BYTES_FWD_PER_TH * th, "3:1"),
    }
    if extras is not None:
        out["other_configs"] = extras
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline()
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
