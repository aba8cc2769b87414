"""Heads of at most 64 features run on the 64-wide 16-bit kernels: the pre-pass takes two 64-token blocks per step (a
segment of 64 or 192 tokens ends in half a step), rows narrower than 64, ragged lengths, few and many segments."""
import pytest
import torch

from helpers import check, in_place_bits, make_inputs, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,e", [(64, 64), (56, 64), (64, 24), (8, 16)])
@pytest.mark.parametrize("n,seg", [(1, 0), (63, 0), (128, 64), (129, 64), (447, 192), (1000, 64), (1088, 192), (3000, 1088)])
def test_rows_of_up_to_64_features(gpu_device, n, seg, d, e, dtype):
    from lasp_amd import _abi

    b, h = 2, 3
    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.tensor([0.4, 0.02, 0.0])
    kvo, dkvo = torch.empty_like(dev["kv"]), torch.empty_like(dev["dkv"])
    o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], s.to(gpu_device), dev["kv"], kvo, seg)
    ref = oracle(inp, s)
    for kept in (states, None):  # the forward's states, and states rebuilt in the backward
        dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], s.to(gpu_device), dev["do"], dev["kv"], dev["dkv"], dkvo,
                                    kept, seg_len)
        got = dict(o=o, kv_out=kvo, dq=dq, dk=dk, dv=dv, dkv_out=dkvo)
        # the bound of every 16-bit parity test: roundings of 2^-9 in inputs, decayed keys, scores and states
        check(got, ref, 2e-2, what=f"n={n} seg={seg} d={d} e={e} {dtype} kept={kept is not None}")


@pytest.mark.parametrize("d,e", [(64, 64), (56, 24)])
@pytest.mark.parametrize("n,seg", [(500, 64), (1152, 128), (65, 0)])
def test_states_updated_in_place(gpu_device, n, seg, d, e):
    """Two waves hold each column block of the state that a single workgroup reads and replaces; heads outside the scan
    (slope 0.4) find the incoming state in the workspace."""
    inp = make_inputs(2, 3, n, d, e, torch.bfloat16, seed=n + d, state=True, state_std=1.0, device=gpu_device)
    for i, (a, r) in enumerate(in_place_bits(inp, torch.tensor([0.4, 0.02, 0.0], device=gpu_device), seg)):
        assert torch.equal(a, r), i
