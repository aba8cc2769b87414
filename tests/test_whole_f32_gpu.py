"""float32 calls without states that run as one segment per (b, h): around the line of the rule that chooses it, against the
oracle in 64 bits and against the call in segments."""
import pytest
import torch

import lasp_amd
from lasp_amd import _abi
from oracle import lasp_oracle as O
from tests.helpers import check, make_inputs

pytestmark = pytest.mark.gpu

# As in segments of 64 tokens (180 roundings), and 12 more for each further block of a state's sum
def tol(n):
    return (180 + 12 * (n // 32)) * 2.0 ** -24


@pytest.mark.parametrize("b,h,n,d,e", [(4, 12, 128, 128, 128), (6, 8, 97, 128, 128), (24, 8, 321, 128, 128), (12, 16, 130, 64, 64),
                                       (16, 10, 200, 80, 96), (10, 16, 255, 100, 70)])
def test_one_segment(b, h, n, d, e):
    wide = (128, 128) if e == 70 else (d, e)  # (rows that are no multiple of 4 are padded)
    whole = _abi.stateless_seg_len(b, h, n, *wide, torch.float32)
    assert whole >= n and whole % 64 == 0
    inp = {k: t for k, t in make_inputs(b, h, n, d, e, torch.float32, seed=n, scale=0.1, state=False).items() if t is not None}
    s = lasp_amd.build_slope_tensor(h)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], None, None, dtype=torch.float64)
    dev = {k: t.cuda() for k, t in inp.items()}
    leaves = [dev[x].requires_grad_() for x in "qkv"]
    o = lasp_amd.lightning_attn(*leaves, s.cuda())
    grads = torch.autograd.grad(o, leaves, dev["do"])
    check(dict(o=o, dq=grads[0], dk=grads[1], dv=grads[2]), {k: ref[k] for k in ("o", "dq", "dk", "dv")}, tol(n), what=f"{b} {h} {n} {d} {e}")
    with torch.no_grad():
        o2, states, seg = _abi.chunk_fwd(*leaves, s.cuda())
        assert seg == whole and states is None
        assert torch.equal(o, o2)
        # the state that is asked for only in the backward, under the forward's segment length
        dkv = torch.empty(b, h, d, e, device="cuda")
        again = _abi.chunk_bwd(*leaves, s.cuda(), dev["do"], dkv_out=dkv, kv_seg_states=states, seg_len=seg)
        for a, c in zip(grads, again):
            assert torch.equal(a, c)
        # asked for in the forward: the default plan, as ever
        kv = torch.empty(b, h, d, e, device="cuda")
        assert _abi.chunk_fwd(*leaves, s.cuda(), kv_out=kv)[2] == _abi.plan(b, h, n, *wide, torch.float32)[0] < n
    check(dict(dkv_out=dkv, kv_out=kv), {k: ref[k] for k in ("dkv_out", "kv_out")}, tol(n), what="states")


def test_where_segments_stay():
    f32 = torch.float32
    for shape in [(2, 12, 2048, 128, 128), (1, 96, 1024, 128, 128), (1, 16, 1024, 128, 128), (1, 96, 1024, 64, 64), (1, 512, 4096, 128, 128)]:
        assert _abi.stateless_seg_len(*shape, f32) == 0
    assert _abi.stateless_seg_len(1, 192, 512, 128, 128, torch.bfloat16) == 0
    assert _abi.stateless_seg_len(1, 192, 512, 126, 128, f32) == 0 == _abi.stateless_seg_len(1, 192, 512, 0, 128, f32)
