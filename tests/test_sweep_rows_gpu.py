"""Backward sweeps over several of the forward's segments in a row: whole and partial rows of segments, on both sides of the rule that
takes them, in either element type, for every width that has them, from kept states and from states of the backward's own."""
import pytest
import torch

from helpers import bwd_rows, check, make_inputs, oracle

pytestmark = pytest.mark.gpu

# The bound of every 16-bit parity test: a few roundings of 2^-9, of the products' operands and the output; in fp16 as many, of an
# eighth each.
TOL = {torch.bfloat16: 2e-2, torch.float16: 2e-2 / 8}


# (b, h, n, d, e, seg_len): segments in a row, as the rule has them
SHAPES = {
    (1, 4, 7168, 128, 128, 0): 2, (1, 4, 6800, 128, 128, 0): 2,      # rows of the library's own segments; a ragged last one
    (1, 5, 2600, 128, 128, 192): 1,                                  # one round as it is
    (1, 2, 8129, 96, 80, 256): 1,                                    # ... of narrow rows, one token in the last segment
    (1, 16, 1600, 192, 128, 0): 2, (1, 3, 4161, 256, 72, 128): 2,    # slices
    (1, 10, 2570, 128, 128, 256): 2,                                 # a last segment too small to count
    (1, 7, 1280, 128, 64, 64): 2, (1, 1, 4096, 128, 128, 64): 1,
    (1, 3, 520, 128, 128, 64): 1, (1, 6, 2049, 64, 64, 192): 1,      # the last one: heads that never take it
    (1, 27, 309, 128, 128, 64): 3, (1, 27, 309, 256, 72, 64): 3,     # a second row of two segments, the last ragged
    (1, 9, 553, 96, 80, 64): 2, (1, 41, 309, 96, 80, 64): 5,         # narrow rows
    (1, 27, 919, 128, 128, 64): 8,                                   # the most in a row, twice
    (1, 41, 431, 128, 128, 64): 7, (1, 41, 492, 128, 128, 64): 8,    # rows that are the whole chunk
    (1, 57, 2225, 128, 128, 512): 5, (1, 57, 1378, 256, 64, 192): 8,  # rows of 40 blocks, and of 24 of a slice: the longest
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e,seg_len", SHAPES)
@pytest.mark.parametrize("decay", [True, False])
def test_matches_oracle(gpu_device, b, h, n, d, e, seg_len, dtype, decay):
    from lasp_amd import _abi

    segment = _abi.plan(b, h, n, d, e, dtype, seg_len)[0]
    assert bwd_rows(b, h, n, d, e, dtype, seg_len) == SHAPES[b, h, n, d, e, seg_len] * segment
    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.linspace(0.4, 0.003, h) if decay else torch.zeros(h)  # heads that the scan leaves out, and heads that it does not
    sd = s.to(gpu_device)
    what = f"b={b} h={h} n={n} d={d} e={e} {dtype}"

    def run(carried, kept, seg):
        kv, dkv = (dev["kv"], dev["dkv"].clone()) if carried else (None, None)
        out = torch.empty_like(dev["kv"]) if carried else None
        o, states, seg = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], sd, kv, None if kv is None else torch.empty_like(kv), seg)
        dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], sd, dev["do"], kv, dkv, out, states if kept else None, seg)
        got = dict(dq=dq, dk=dk, dv=dv)
        return dict(got, dkv_out=out) if carried else got

    want = oracle(inp, s)
    got = run(True, True, seg_len)
    check(got, {k: want[k] for k in got}, TOL[dtype], what=what)
    for name, x in run(True, False, seg_len).items():  # the states are the same ones
        assert torch.equal(x, got[name]), (what, name)
    other = 2560 if n > 2560 else 512  # swept one by one
    check(got, run(True, True, other), TOL[dtype], what=what + ", other segments")

    bare = dict(inp, kv=torch.zeros_like(inp["kv"]), dkv=torch.zeros_like(inp["dkv"]))
    want, got = oracle(bare, s), run(False, True, seg_len)
    check(got, {k: want[k] for k in got}, TOL[dtype], what=what + ", no states")


def test_results_do_not_depend_on_the_launch(gpu_device):
    from lasp_amd import _abi

    inp = make_inputs(1, 4, 7168, 128, 128, torch.bfloat16, seed=3, scale=0.3, state=True, state_std=1.0, device=gpu_device)
    s = torch.linspace(0.3, 0.0, 4, device=gpu_device)

    def run():
        o, states, seg = _abi.chunk_fwd(inp["q"], inp["k"], inp["v"], s, inp["kv"], torch.empty_like(inp["kv"]), 0)
        return _abi.chunk_bwd(inp["q"], inp["k"], inp["v"], s, inp["do"], inp["kv"], inp["dkv"], torch.empty_like(inp["dkv"]), states, seg)

    first = run()
    for x, y in zip(first, run()):
        assert torch.equal(x, y)
