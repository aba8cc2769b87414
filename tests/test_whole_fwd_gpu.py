"""Operators whose forward and backward run in one launch each although the plan has several segments: no states are kept, and the
backward starts from the incoming state.  At both sides of the lines, with and without states, against the oracle."""
import pytest
import torch

import lasp_amd
from lasp_amd import _abi, _native
from lasp_amd.utils import seq_parallel_manager as spm
from tests.helpers import make_inputs, oracle

pytestmark = pytest.mark.gpu

# one rounding of an input-sized operand per product and one of the result: 2^-9 (bf16), 2^-12 (fp16), a few of them
REL = {torch.bfloat16: 1.2e-2, torch.float16: 1.6e-3}


def profiled(call):
    _abi.profile_begin()
    out = call()
    torch.cuda.synchronize()
    return out, {name: count for name, (_, count) in _abi.profile_end().items() if count}


def close(got, want, dtype, what):
    diff, want = (got.detach().cpu().double() - want).flatten(2), want.double().flatten(2)
    rel = diff.norm(dim=2) / want.norm(dim=2)
    assert float(rel.max()) < REL[dtype], (what, float(rel.max()), int(rel.argmax()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e,whole", [
    (2, 12, 2048, 128, 128, True), (1, 16, 1408, 128, 128, True), (1, 16, 1409, 128, 128, False),
    (1, 30, 2111, 128, 128, True), (2, 40, 1601, 96, 80, True),  # a partial last block, narrow rows
    (1, 32, 2816, 128, 128, True),                               # 44 blocks, the fewest that a forward cuts into eight segments, the most
    (1, 90, 2100, 128, 64, True), (2, 12, 2048, 64, 64, False),  # more (b, h) than places for two segments; the 64-wide kernels
])
def test_attention(gpu_device, b, h, n, d, e, whole, dtype):
    inp = make_inputs(b, h, n, d, e, dtype, seed=n + h, scale=0.3, state=False)
    s = torch.linspace(0.3, 0.0, h)
    leaves = [inp[x].to(gpu_device).requires_grad_(True) for x in "qkv"]
    assert _abi.kernel_path(b, h, n, d, e, dtype) == _abi.PATH_MFMA

    def run():
        o = lasp_amd.lightning_attn(*leaves, s.to(gpu_device).view(h, 1, 1))
        o.backward(inp["do"].to(gpu_device))
        return o

    o, launches = profiled(run)
    assert (launches == {"fused": 2}) == whole, launches
    ref = oracle(inp, s)
    for x, name in zip((o, *(t.grad for t in leaves)), ("o", "dq", "dk", "dv")):
        close(x, ref[name], dtype, name)
    with torch.no_grad():  # no backward: the same launch
        again, launches = profiled(lambda: lasp_amd.lightning_attn(*leaves, s.to(gpu_device).view(h, 1, 1)))
    assert torch.equal(again, o) or not whole


@pytest.mark.parametrize("operator", ["lasp_fuse", "lasp_fuse_parallel"])
def test_a_chain(gpu_device, operator):
    """Three chunks of a chain: states travel both ways, the buffers end as documented."""
    b, h, n, d, chunks, dtype = 2, 12, 1800, 128, 3, torch.bfloat16
    inp = make_inputs(b, h, n * chunks, d, d, dtype, seed=4, scale=0.3, state=False)
    s = torch.linspace(0.2, 0.0, h)
    fuse = getattr(lasp_amd, operator)
    KV, DKV = [torch.full((b, h, d, d), float("nan"), device=gpu_device) for _ in range(2)]
    spm.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, chunks)
    try:
        def run():
            outs, leaves = [], []
            for c in range(chunks):
                lasp_amd.set_sequence_parallel_rank(c)
                part = [inp[x][:, :, c * n:(c + 1) * n].to(gpu_device).requires_grad_(True) for x in "qkv"]
                outs.append(fuse(*part, s.to(gpu_device).view(h, 1, 1), KV, DKV))
                leaves.append(part)
            torch.autograd.backward(outs, [inp["do"][:, :, c * n:(c + 1) * n].to(gpu_device) for c in range(chunks)])
            return outs, leaves

        (outs, leaves), launches = profiled(run)
    finally:
        spm.destroy_parallel_groups()
    # backwards; forwards only of a chunk that no state leaves (lasp_fuse keeps the last one's in the caller's buffer)
    assert launches["fused"] == (chunks if operator == "lasp_fuse" else chunks + 1), launches
    assert "bwd3" not in launches, launches
    ref = oracle(inp, s)
    close(torch.cat(outs, 2), ref["o"], dtype, "o")
    for i, name in enumerate(("dq", "dk", "dv")):
        close(torch.cat([p[i].grad for p in leaves], 2), ref[name], dtype, name)
    if operator == "lasp_fuse":  # the last chunk's state
        close(KV, ref["kv_out"], dtype, "KV")


def test_shims_keep_their_states(gpu_device):
    """What the launch shims return is for a caller to hand on: the states are left as planned."""
    b, h, n, d = 2, 12, 2048, 128
    assert _abi.load().lasp_whole_ok(b, h, n, d, d, 1, 1) == 1
    q, k, v = [torch.randn(b, h, n, d, device=gpu_device).to(torch.bfloat16) / 11 for _ in range(3)]
    kv = torch.randn(b, h, d, d, device=gpu_device)
    s = torch.linspace(0.2, 0.0, h, device=gpu_device)
    (o, states, seg_len), launches = profiled(lambda: _native.chunk_fwd(q, k, v, s, kv_in=kv, kv_out=torch.empty_like(kv)))
    assert "fused" not in launches and states.numel() * 4 == _abi.plan(b, h, n, d, d, torch.bfloat16)[2]
    over = kv.clone()  # a state updated in place: nothing orders the readers and the writer of a single launch
    (o2, none, _), launches = profiled(lambda: _native.chunk_fwd(q, k, v, s, kv_in=over, kv_out=over, keep=False))
    assert "fused" not in launches and torch.equal(o2, o)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("operator", ["lasp_fuse", "lasp_fuse_parallel"])
@pytest.mark.parametrize("b,h,n,d", [(2, 12, 2048, 128), (1, 40, 1700, 96)])
def test_a_state_that_leaves_is_a_sum_of_segments(gpu_device, operator, b, h, n, d, dtype):
    """Without decay every product is exact in 32 bits and only the sums round, like random walks over 16 tokens' partial sums of the
    size reached: segments of 256 tokens (16 roundings, then 8 of the scan) leave about sqrt(16 / 2 + 8 / 2) * 2^-25 = 1.0e-7; one
    accumulator over 2048 tokens sqrt(128 / 2) * 2^-25 = 2.4e-7 (measured 1.0e-7 to 1.3e-7, and 2.9e-7)."""
    assert _abi.load().lasp_whole_ok(b, h, n, d, d, _abi.DTYPE_CODE[dtype], 1) == 1
    g = torch.Generator().manual_seed(n)
    q, k, v = [torch.randn(b, h, n, d, generator=g) for _ in range(3)]
    q, k, v = [t.to(dtype).to(gpu_device) for t in (q / d, (torch.nn.functional.elu(k) + 1) / d, v / d ** 0.5)]
    s = torch.zeros(h, 1, 1, device=gpu_device)
    KV, DKV = [torch.full((b, h, d, d), float("nan"), device=gpu_device) for _ in range(2)]
    spm.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, 2)
    try:
        for c in range(2):  # the same chunk twice: what leaves the first one enters the second
            lasp_amd.set_sequence_parallel_rank(c)
            getattr(lasp_amd, operator)(q.clone().requires_grad_(True), k, v, s, KV, DKV)
            if c == 0 and operator == "lasp_fuse":
                first = KV.clone()
    finally:
        spm.destroy_parallel_groups()
    if operator == "lasp_fuse_parallel":  # (its buffer holds what entered the last chunk)
        first = KV
    want = k.double().transpose(2, 3) @ v.double()
    assert float((first.double() - want).norm() / want.norm()) < 1.7e-7
