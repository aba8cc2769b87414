"""The fp32 sweeps leave out the state update of a segment's last block: segments of one block, of several, and ones that end in a
partial block, for every number of feature tiles, against the oracle in 64 bits."""
import pytest
import torch

from lasp_amd import _abi
from tests.helpers import NORM_F32, check_norm, make_inputs, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,e", [(128, 128), (60, 64), (96, 72), (128, 64)])
@pytest.mark.parametrize("n,seg", [(32, 64), (40, 64), (65, 64), (96, 64), (200, 64), (224, 128), (320, 256), (333, 320)])
def test_every_token_of_a_last_block(gpu_device, d, e, n, seg):
    h = 3
    inp = make_inputs(2, h, n, d, e, torch.float32, seed=n + d, scale=0.2, state=True, state_std=0.3)
    dev = {k: t.to(gpu_device) for k, t in inp.items()}
    s = torch.tensor([0.0, 0.01, 0.4])
    sd = s.to(gpu_device)
    kv_out, dkv_out = (torch.empty_like(dev["kv"]) for _ in range(2))
    o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], sd, dev["kv"], kv_out, seg)
    dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], sd, dev["do"], dev["kv"], dev["dkv"], dkv_out, states, seg_len)
    got, ref = dict(o=o, kv_out=kv_out, dq=dq, dk=dk, dv=dv, dkv_out=dkv_out), oracle(inp, s)
    check_norm(got, ref, NORM_F32, what=f"n={n} seg={seg} d={d} e={e}")
    # the last block of every segment on its own: few tokens, whose errors the whole would hide.  (A few hundred tokens' sums
    # round as often as theirs; a 2-norm over 1 to 32 of them scatters, hence three times the bound.)
    for t0 in range(0, n, seg):
        t1 = min(t0 + seg, n)
        for lo, hi in ((t0, min(t0 + 32, t1)), (t0 + (t1 - t0 - 1) // 32 * 32, t1)):  # last going backwards, and forwards
            part = lambda out: {k: x[:, :, lo:hi] for k, x in out.items() if k in ("o", "dq", "dk", "dv")}
            check_norm(part(got), part(ref), 3 * NORM_F32, what=f"tokens {lo}..{hi}")
