"""Heads with d > 128 in 16 bits: the library sweeps q and k in slices of 128 features (the last one may be narrower),
adds the slices' parts of O and dV in place and keeps one state per slice."""
import pytest
import torch

import lasp_amd
from helpers import check, in_place_bits, make_inputs, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,e", [(136, 128), (192, 64), (256, 128), (320, 40), (1024, 128)])
@pytest.mark.parametrize("n,seg", [(1, 0), (65, 0), (500, 0), (500, 64), (1152, 128), (2600, 0)])
def test_feature_slices(gpu_device, n, seg, d, e, dtype):
    from lasp_amd import _abi

    inp = make_inputs(1, 3, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.tensor([0.4, 0.02, 0.0])
    kvo, dkvo = torch.empty_like(dev["kv"]), torch.empty_like(dev["dkv"])
    o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], s.to(gpu_device), dev["kv"], kvo, seg)
    ref = oracle(inp, s)
    for kept in (states, None):  # the forward's states, and states rebuilt in the backward
        dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], s.to(gpu_device), dev["do"], dev["kv"], dev["dkv"], dkvo,
                                    kept, seg_len)
        got = dict(o=o, kv_out=kvo, dq=dq, dk=dk, dv=dv, dkv_out=dkvo)
        # the bound of every 16-bit parity test; O and dV are rounded once more per slice (2^-9 each)
        check(got, ref, 2e-2, what=f"n={n} seg={seg} d={d} e={e} {dtype} kept={kept is not None}")


@pytest.mark.parametrize("d", [192, 256])
@pytest.mark.parametrize("n,seg", [(500, 64), (1152, 128), (65, 0)])
def test_states_updated_in_place(gpu_device, n, seg, d):
    """Every slice parks the incoming state of a head outside the scan (slope 0.4: gone within 64 tokens) in its own part of
    the workspace, and reads it in a sweep that starts after all slices' outgoing states have replaced the incoming ones."""
    inp = make_inputs(1, 3, n, d, 128, torch.bfloat16, seed=n + d, scale=0.3, state=True, state_std=1.0, device=gpu_device)
    for i, (a, r) in enumerate(in_place_bits(inp, torch.tensor([0.4, 0.02, 0.0], device=gpu_device), seg)):
        assert torch.equal(a, r), i


def test_wide_operator_chain(gpu_device):
    """Two chunks through lasp_fuse with d = 192: the whole state travels as one message and KV / DKV are updated in place."""
    inp = make_inputs(1, 2, 600, 192, 64, torch.bfloat16, seed=5, scale=0.3, state=False)
    s = torch.tensor([0.3, 0.01])
    ref = oracle(inp, s)
    lasp_amd.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, 2)
    try:
        KV = torch.empty(1, 2, 192, 64, device=gpu_device)
        DKV = torch.empty_like(KV)
        leaves, outs, dos = [], [], []
        for c, sl in enumerate((slice(0, 300), slice(300, 600))):
            lasp_amd.set_sequence_parallel_rank(c)
            q, k, v = [inp[x][:, :, sl].to(gpu_device).contiguous().requires_grad_(True) for x in ("q", "k", "v")]
            outs.append(lasp_amd.lasp_fuse(q, k, v, s.to(gpu_device), KV, DKV))
            dos.append(inp["do"][:, :, sl].to(gpu_device))
            leaves.append((q, k, v))
        torch.autograd.backward(outs, dos)
    finally:
        lasp_amd.destroy_parallel_groups()
    got = dict(o=torch.cat([o.detach() for o in outs], 2), kv_out=KV, dkv_out=DKV)
    for i, name in enumerate(("dq", "dk", "dv")):
        got[name] = torch.cat([x[i].grad for x in leaves], 2)
    check(got, ref, 2e-2, what="two-chunk lasp_fuse chain, d = 192")
