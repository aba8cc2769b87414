"""A backward that is given the forward's segment states takes the state entering the chunk from them: what the buffer `kv_in`
holds by then does not matter, as where the forward has updated it in place.  (Plans of up to four segments of whole rows gather
own states, which leave the incoming one out, and read `kv_in`.)"""
import pytest
import torch

from helpers import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e", [
    (2, 12, 2048, 128, 128), (1, 20, 1601, 128, 128),  # chunks whose backward is one launch: several segments
    (3, 12, 2500, 96, 96), (1, 25, 2111, 128, 72),     # narrow rows
    (5, 16, 1700, 96, 96),                             # narrow rows, one segment of the backward per (b, h)
    (1, 6, 2048, 128, 128), (1, 3, 3000, 64, 64), (1, 3, 1500, 192, 64),  # three kernels
])
@pytest.mark.parametrize("explicit", [False, True])
def test_incoming_state_comes_from_the_kept_states(gpu_device, b, h, n, d, e, dtype, explicit):
    from lasp_amd import _abi

    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0, device=gpu_device)
    s = torch.linspace(0.4, 0.0, h, device=gpu_device)  # heads outside the scan, in it, and without decay
    seg_len, n_seg, _ = _abi.plan(b, h, n, d, e, dtype)
    assert n_seg > 4 or (d, e) != (128, 128)
    kv_in = inp["kv"].clone()
    o, states, used = _abi._chunk_fwd_exact(inp["q"], inp["k"], inp["v"], s, kv_in, torch.empty_like(kv_in))
    assert used == seg_len

    def grads(kv, kept=states):
        return _abi._chunk_bwd_exact(inp["q"], inp["k"], inp["v"], s, inp["do"], kv, inp["dkv"], torch.empty_like(inp["dkv"]),
                                     kept, seg_len if explicit else 0)

    want = grads(kv_in)
    for held in (torch.full_like(kv_in, 3.0), torch.full_like(kv_in, float("nan"))):
        for name, x, r in zip(("dq", "dk", "dv"), grads(held), want):
            assert torch.equal(x, r), name
    # Without the pointer as well, but for heads whose state dies within the shortest segment: they stand outside the scan, and
    # are taken to have started from nothing.
    dq = grads(None)[0]
    outside = s * 1.4426950408889634 * (n - (n_seg - 1) * seg_len) > 24
    assert outside.any() and not outside.all()
    _, without, _ = _abi._chunk_fwd_exact(inp["q"], inp["k"], inp["v"], s, None, torch.empty_like(kv_in))
    assert torch.equal(dq[:, ~outside], want[0][:, ~outside])
    assert torch.equal(dq[:, outside], grads(None, without)[0][:, outside])
