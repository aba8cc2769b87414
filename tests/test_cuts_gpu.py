"""The single-launch kernels cut a (b, h) into segments that are shorter the longer the walk before them, for heads whose decay reaches
far, and into equal ones for the others: both in one call, at sizes from one block on."""
import pytest
import torch

from lasp_amd import _abi
from tests.helpers import make_inputs, oracle

pytestmark = pytest.mark.gpu

# one rounding of an input-sized operand per product and one of the result: 2^-9 (bf16), 2^-12 (fp16), a few of them
REL = {torch.bfloat16: 1.2e-2, torch.float16: 1.6e-3}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e", [
    (1, 6, 64, 128, 128), (1, 6, 65, 128, 128), (2, 4, 256, 128, 128),  # one block, two, four
    (1, 5, 1000, 128, 128), (4, 8, 1024, 128, 128),                     # six segments forwards, the last three of one block
    (5, 32, 500, 128, 128), (1, 130, 128, 128, 128),                    # one segment each, and in the backward a cut last round
    (1, 16, 1024, 64, 64), (3, 40, 700, 64, 48),                        # the 64-wide kernels
    (1, 6, 900, 96, 40), (1, 3, 600, 192, 128),                         # narrow rows, slices of wide ones
])
@pytest.mark.parametrize("state", [True, False])
def test_every_head(gpu_device, b, h, n, d, e, dtype, state):
    inp = make_inputs(b, h, n, d, e, dtype, seed=n + h, scale=0.3, state=state, state_std=0.5)
    dev = {k: (v.to(gpu_device) if v is not None else None) for k, v in inp.items()}
    s = torch.tensor([0.0, 0.004, 0.02, 0.06, 0.2, 0.7])[torch.arange(h) % 6]  # reaches from all blocks to one
    sd = s.to(gpu_device)
    assert _abi.kernel_path(b, h, n, d, e, dtype) == _abi.PATH_MFMA_FUSED
    kvo, dkvo = (torch.empty_like(dev["kv"]) for _ in range(2)) if state else (None, None)
    o, _, _ = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], sd, dev["kv"], kvo)
    dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], sd, dev["do"], dev["kv"], dev["dkv"], dkvo)
    ref = oracle(inp, s)
    for name, x in dict(o=o, dq=dq, dk=dk, dv=dv, kv_out=kvo, dkv_out=dkvo).items():
        if x is None:
            continue
        diff, want = (x.cpu().double() - ref[name]).flatten(2), ref[name].double().flatten(2)
        rel = diff.norm(dim=2) / want.norm(dim=2)
        assert float(rel.max()) < REL[dtype], (name, float(rel.max()), int(rel.argmax()))


@pytest.mark.parametrize("n", [3, 64, 200, 256])
def test_a_state_in_place(gpu_device, n):
    """A chunk of one planned segment may leave its state over the incoming one: no other workgroup reads it then."""
    inp = make_inputs(1, 6, n, 128, 128, torch.bfloat16, seed=n, scale=0.3, state=True, state_std=0.5, device=gpu_device)
    s = torch.linspace(0.0, 0.3, 6, device=gpu_device)
    assert _abi.inplace_ok(1, 6, n, 128, 128, torch.bfloat16, 0, False)
    apart, over = torch.empty_like(inp["kv"]), inp["kv"].clone()
    o = _abi._chunk_fwd_exact(inp["q"], inp["k"], inp["v"], s, inp["kv"], apart)[0]
    o2 = _abi._chunk_fwd_exact(inp["q"], inp["k"], inp["v"], s, over, over)[0]
    assert torch.equal(o, o2) and torch.equal(apart, over)
