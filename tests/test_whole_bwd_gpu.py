"""The backward of a chunk in one launch where the forward takes several: on both sides of the line between the two, in either
element type, with a partial last block, narrow rows and an outgoing state that lies over the incoming one."""
import pytest
import torch

from helpers import check, make_inputs, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e", [
    (1, 16, 1408, 128, 128), (1, 16, 1409, 128, 128),  # the last length that takes it, and the first that does not
    (2, 12, 2048, 128, 128), (1, 20, 1601, 128, 128),  # several segments; three of 20 (b, h) on half of the XCDs
    (3, 12, 2500, 96, 96), (1, 25, 2111, 128, 72),     # narrow rows
    (2, 30, 2177, 128, 128),                           # one segment per (b, h)
])
@pytest.mark.parametrize("decay", [True, False])
def test_matches_oracle_and_the_three_kernels(gpu_device, b, h, n, d, e, dtype, decay):
    from lasp_amd import _abi

    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.linspace(0.4, 0.003, h) if decay else torch.zeros(h)
    sd = s.to(gpu_device)
    o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], sd, dev["kv"], torch.empty_like(dev["kv"]))

    def run(in_place):
        # an outgoing state over the incoming one takes the three kernels, if it is not copied away first
        dkv_in = dev["dkv"].clone()
        dkv_out = dkv_in if in_place else torch.empty_like(dkv_in)
        _abi.profile_begin()
        dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], sd, dev["do"], dev["kv"], dkv_in, dkv_out, states, seg_len)
        launches = {name: count for name, (_, count) in _abi.profile_end().items() if count}
        over = in_place and _abi.inplace_ok(b, h, n, d, e, dtype, seg_len, True)
        assert (launches == {"fused": 1}) == (n <= 88 * b * h and not over), launches
        return dict(dq=dq, dk=dk, dv=dv, dkv_out=dkv_out)

    got, apart = run(False), run(True)
    want = oracle(inp, s)
    # the bound of every 16-bit parity test: a few roundings of 2^-9 (2^-12 in fp16), of the products' operands and the output
    for out in (got, apart):
        check(out, {k: want[k] for k in out}, 2e-2, what=f"b={b} h={h} n={n} d={d} e={e} {dtype}")
    for name, x in run(False).items():  # no sum depends on which workgroup comes first
        assert torch.equal(x, got[name]), name
