"""DKV states that lie further apart than the forward's segments: as far as the sweeps start and half as far, in whole and partial pieces,
for heads that the scan takes and heads that it leaves out, one piece from the other end of the chunk and many."""
import pytest
import torch

from helpers import check, make_inputs, oracle

pytestmark = pytest.mark.gpu

# As in the other 16-bit parity tests: a few roundings of 2^-9; in fp16 of an eighth.
TOL = {torch.bfloat16: 2e-2, torch.float16: 2e-2 / 8}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e,seg_len", [
    (1, 16, 1088, 128, 128, 64), (2, 8, 1100, 128, 128, 64),  # four of the forward's segments each; the last piece one block and 12 tokens
    (1, 12, 897, 128, 128, 64), (1, 16, 641, 128, 64, 64),    # three; one token in the last one
    (1, 12, 1999, 128, 128, 64),                              # sweeps over six, pieces of three
    (2, 16, 449, 128, 128, 64), (1, 20, 520, 128, 128, 64),   # two pieces, three
    (1, 8, 700, 256, 128, 64), (1, 10, 1300, 192, 128, 64), (1, 16, 385, 200, 72, 64),  # slices
    (1, 8, 3784, 128, 128, 0), (1, 16, 1536, 192, 128, 0),    # default plans
])
@pytest.mark.parametrize("decay", [(0.4, 0.003), (0.9, 0.08), (0.0, 0.0)])
def test_matches_oracle(gpu_device, b, h, n, d, e, seg_len, dtype, decay):
    from lasp_amd import _abi

    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.linspace(*decay, h)
    sd = s.to(gpu_device)
    what = f"b={b} h={h} n={n} d={d} e={e} {dtype} {decay}"

    def run(carried, in_place=False):
        kv, dkv = (dev["kv"], dev["dkv"].clone()) if carried else (None, None)
        out = dkv if in_place else torch.full_like(dev["kv"], float("nan")) if carried else None
        o, states, seg = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], sd, kv, None if kv is None else torch.empty_like(kv), seg_len)
        dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], sd, dev["do"], kv, dkv, out, states, seg)
        got = dict(dq=dq, dk=dk, dv=dv)
        return dict(got, dkv_out=out) if carried else got

    want, got = oracle(inp, s), run(True)
    check(got, {k: want[k] for k in got}, TOL[dtype], what=what)
    for name, x in run(True, in_place=True).items():
        assert torch.equal(x, got[name]), (what, name)
    bare = dict(inp, kv=torch.zeros_like(inp["kv"]), dkv=torch.zeros_like(inp["dkv"]))
    want, got = oracle(bare, s), run(False)
    check(got, {k: want[k] for k in got}, TOL[dtype], what=what + ", no states")
