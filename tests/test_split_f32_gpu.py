"""The fp32 MFMA kernels multiply numbers split into three bf16 parts: lengths around their 32-token blocks, and numbers for
which a split could go wrong, against the oracle in 64 bits."""
import pytest
import torch

import lasp_amd
from lasp_amd import _abi
from oracle import lasp_oracle as O
from tests.helpers import check, make_inputs

pytestmark = pytest.mark.gpu

# An output element is rounded 48 times in the state term and 12 in the intra-block term, a state 12 times a block (at most 9
# blocks here), each time by at most 2^-24 of a partial sum; operands and decays add a few such roundings.
TOL = 180 * 2.0 ** -24
H = 4


def _run(inp, s, seg):
    dev = {k: (t.cuda() if t is not None else None) for k, t in inp.items()}
    s = s.cuda()
    kv_out, dkv_out = (torch.empty_like(dev["kv"]) for _ in range(2)) if dev["kv"] is not None else (None, None)
    o, states, seg_len = _abi._chunk_fwd_exact(dev["q"], dev["k"], dev["v"], s, kv_in=dev["kv"], kv_out=kv_out, seg_len=seg)
    dq, dk, dv = _abi._chunk_bwd_exact(dev["q"], dev["k"], dev["v"], s, dev["do"], kv_in=dev["kv"], dkv_in=dev["dkv"],
                                       dkv_out=dkv_out, kv_seg_states=states, seg_len=seg_len)[:3]
    return dict(o=o, kv_out=kv_out, dq=dq, dk=dk, dv=dv, dkv_out=dkv_out)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 97, 260])
@pytest.mark.parametrize("state", [True, False])
def test_lengths(n, state):
    inp = make_inputs(1, H, n, 128, 128, torch.float32, seed=n, scale=0.1, state=state)
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], inp["kv"], inp["dkv"], dtype=torch.float64)
    check(_run(inp, s, 64), ref, TOL, what=f"n={n}")


def test_features_of_any_size():
    """Features of q and k whose sizes differ by 2^80 and cancel in q . k."""
    inp = make_inputs(1, H, 130, 128, 128, torch.float32, seed=5, scale=0.1, state=False)
    size = 2.0 ** torch.linspace(-40, 40, 128).round()
    inp["q"], inp["k"] = inp["q"] * size, inp["k"] / size
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], dtype=torch.float64)
    got = _run(inp, s, 64)
    for out, by in (("dq", size), ("dk", 1 / size)):
        got[out], ref[out] = got[out].cpu() * by, ref[out] * by.double()
    check(got, ref, TOL, names=("o", "dq", "dk", "dv"))


def test_lowest_value():
    """The lowest finite number has no bf16 neighbour that rounding could take it to."""
    inp = make_inputs(1, H, 96, 128, 128, torch.float32, seed=6, scale=0.01, state=False)
    inp["v"][:, :, 40, 3] = torch.finfo(torch.float32).min
    inp["k"][:, :, 41, 5] = torch.finfo(torch.float32).min
    inp["do"][:] = 0
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], dtype=torch.float64)
    got = _run(inp, s, 64)
    assert torch.isfinite(got["o"]).all()
    check(got, ref, TOL, names=("o",))


def test_nan_stays_behind():
    """A NaN of a token reaches its own output and none of the blocks before it."""
    inp = make_inputs(1, H, 96, 128, 128, torch.float32, seed=7, scale=0.1, state=False)
    s = lasp_amd.build_slope_tensor(H)
    clean = _run(inp, s, 64)["o"]
    for name in ("q", "k", "v"):
        bad = dict(inp, **{name: inp[name].clone()})
        bad[name][:, :, 70, 9] = float("nan")
        o = _run(bad, s, 64)["o"]
        assert torch.isnan(o[:, :, 70]).any(-1).all()
        assert torch.equal(o[:, :, :64], clean[:, :, :64])
