"""The 128-wide 16-bit sweeps where their pipeline of three sets of tiles begins and ends: one to six blocks per segment, with and
without a partial last one, entered by a state from memory, gathered or walked for, whole rows, narrow ones and slices."""
import pytest
import torch

from helpers import check, make_inputs, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,e", [(128, 128), (128, 72), (200, 128)])
@pytest.mark.parametrize("n,seg", [(n, seg) for n in (64, 65, 128, 191, 192, 256, 321, 384) for seg in (0, 64, 128, 192, 384)
                                   if seg < n + 64])
def test_few_blocks(gpu_device, n, seg, d, e, dtype):
    from lasp_amd import _abi

    inp = make_inputs(1, 3, n, d, e, dtype, seed=n + seg + d + e, scale=0.3, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.tensor([0.4, 0.02, 0.0])
    kvo, dkvo = torch.empty_like(dev["kv"]), torch.empty_like(dev["dkv"])

    def run():
        o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], s.to(gpu_device), dev["kv"], kvo, seg)
        dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], s.to(gpu_device), dev["do"], dev["kv"], dev["dkv"], dkvo,
                                    states, seg_len)
        return dict(o=o, kv_out=kvo.clone(), dq=dq, dk=dk, dv=dv, dkv_out=dkvo.clone())

    got = run()
    # the bound of every 16-bit parity test: a few roundings of 2^-9, of the products' operands and the output; in fp16 of an eighth each
    check(got, oracle(inp, s), 2e-2 if dtype == torch.bfloat16 else 2e-2 / 8, what=f"n={n} seg={seg} d={d} e={e} {dtype}")
    for _ in range(3):  # no sum depends on which wave comes first
        for name, x in run().items():
            assert torch.equal(x, got[name]), name
