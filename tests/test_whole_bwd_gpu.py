"""The backward of a chunk in one launch where the forward takes several: on both sides of the lines between the two, in either
element type, with a partial last block, narrow rows and an outgoing state that lies over the incoming one."""
import ctypes

import pytest
import torch

from helpers import check, make_inputs, oracle

pytestmark = pytest.mark.gpu

# The bound of every 16-bit parity test: a few roundings of 2^-9, of the products' operands and the output; in fp16 as many, of an
# eighth each.
TOL = {torch.bfloat16: 2e-2, torch.float16: 2e-2 / 8}


def profiled(call):
    """What `call` returns, and the kernels it launched."""
    from lasp_amd import _abi

    _abi.profile_begin()
    out = call()
    return out, {name: count for name, (_, count) in _abi.profile_end().items() if count}


def another_length(seg_len):
    """A segment length that is not the plan's: the three kernels are taken."""
    return 192 if seg_len == 256 else 256


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e,one", [
    (1, 16, 1408, 128, 128, True), (1, 16, 1409, 128, 128, False),  # the last length that takes it, and the first that does not
    (2, 12, 2048, 128, 128, True), (1, 20, 1601, 128, 128, True),   # several segments; three of 20 (b, h) on half of the XCDs
    (3, 12, 2500, 96, 96, True), (1, 25, 2111, 128, 72, False),     # narrow rows
    (2, 30, 2177, 128, 128, True),                                  # one segment per (b, h)
    (6, 14, 1700, 96, 96, True), (1, 83, 1700, 128, 128, True),     # ... of 81 to 85, more than one XCD has places for: some are cut
])
@pytest.mark.parametrize("decay", [True, False])
def test_matches_oracle_and_the_three_kernels(gpu_device, b, h, n, d, e, one, dtype, decay):
    from lasp_amd import _abi

    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0)
    dev = {k: v.to(gpu_device) for k, v in inp.items()}
    s = torch.linspace(0.4, 0.003, h) if decay else torch.zeros(h)
    sd = s.to(gpu_device)

    def run(in_place=False, seg_len=0):
        kvo = torch.empty_like(dev["kv"])
        o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], sd, dev["kv"], kvo, seg_len)
        # an outgoing state over the incoming one takes the three kernels, if it is not copied away first
        dkv_in = dev["dkv"].clone()
        dkv_out = dkv_in if in_place else torch.empty_like(dkv_in)
        (dq, dk, dv), launches = profiled(lambda: _abi.chunk_bwd(
            dev["q"], dev["k"], dev["v"], sd, dev["do"], dev["kv"], dkv_in, dkv_out, states, seg_len))
        over = in_place and _abi.inplace_ok(b, h, n, d, e, dtype, seg_len, True)
        planned = seg_len == _abi.plan(b, h, n, d, e, dtype)[0]
        assert (launches == {"fused": 1}) == (one and planned and not over), launches
        return dict(dq=dq, dk=dk, dv=dv, dkv_out=dkv_out)

    what = f"b={b} h={h} n={n} d={d} e={e} {dtype}"
    got, three = run(), run(seg_len=another_length(_abi.plan(b, h, n, d, e, dtype)[0]))
    want = oracle(inp, s)
    for out in (got, run(in_place=True), three):
        check(out, {k: want[k] for k in out}, TOL[dtype], what=what)
    check(got, three, TOL[dtype], what=what + ", one launch and three kernels")
    for name, x in run().items():  # no sum depends on which workgroup comes first
        assert torch.equal(x, got[name]), name


@pytest.mark.parametrize("b,h,n,d,e,one", [
    (5, 16, 6144, 128, 128, True), (5, 16, 6145, 128, 128, False),    # one round of whole rows, the longest chunk
    (7, 12, 2560, 128, 128, True), (7, 12, 2561, 128, 128, False),    # more than an XCD has places for
    (8, 12, 4096, 128, 128, True), (8, 12, 4097, 128, 128, False),    # more rounds than one
    (3, 43, 5120, 128, 128, True), (8, 18, 4608, 128, 128, False),    # ... of more than 128 (b, h): scanned, gathered
    (1, 28, 1792, 128, 64, True), (1, 28, 2464, 128, 64, False),      # narrow rows, one round
    (7, 12, 6144, 96, 96, True), (7, 12, 6145, 96, 96, False),        # ... and more
    (2, 12, 2048, 64, 64, False), (2, 12, 2048, 192, 128, False),     # the 64-wide kernels, slices
])
def test_lines_between_the_two(gpu_device, b, h, n, d, e, one):
    """Only where the lines lie, and that both sides of them agree."""
    from lasp_amd import _abi

    g = torch.Generator(device=gpu_device).manual_seed(n + b * h)
    mk = lambda w: (torch.randn(b, h, n, w, generator=g, device=gpu_device) / w ** 0.5).to(torch.bfloat16)
    q, k, v, do = mk(d), mk(d), mk(e), mk(e)
    kv, dkv = [torch.randn(b, h, d, e, generator=g, device=gpu_device) for _ in range(2)]
    s = torch.linspace(0.3, 0.002, h, device=gpu_device)
    seg_len = _abi.plan(b, h, n, d, e, torch.bfloat16)[0]

    def run(seg):
        out = torch.empty_like(dkv)
        grads, launches = profiled(lambda: _abi._chunk_bwd_exact(q, k, v, s, do, kv, dkv, out, None, seg))
        return (*grads, out), launches

    got, launches = run(0)
    assert (launches == {"fused": 1}) == one, launches
    explicit, launches = run(seg_len)  # the plan's own length, given: the same
    assert (launches == {"fused": 1}) == one, launches
    other, launches = run(another_length(seg_len))
    assert "fused" not in launches
    for name, x, y, z in zip(("dq", "dk", "dv", "dkv_out"), got, explicit, other):
        assert torch.equal(x, y), name
        diff, want = (x.float() - z.float()).flatten(2), z.float().flatten(2)
        # each within 4e-3 of the sums in 64 bits (2-norm), three times that
        assert float((diff.norm(dim=2) / want.norm(dim=2)).max()) < 1.2e-2, name


@pytest.mark.parametrize("over", ["kv_in", "dkv_in", "part of kv_in", "twin over kv_in"])
@pytest.mark.parametrize("kept", [True, False])
def test_an_outgoing_state_over_an_incoming_one_takes_three_kernels(gpu_device, over, kept):
    """In one launch nothing orders the workgroup that writes the one and those that read the other."""
    from lasp_amd import _abi

    b, h, n, d, e = 2, 12, 2048, 128, 128
    inp = make_inputs(b, h, n, d, e, torch.bfloat16, seed=9, scale=0.3, state=True, state_std=1.0, device=gpu_device)
    s = torch.linspace(0.4, 0.003, h, device=gpu_device)
    seg_len, n_seg, state_bytes = _abi.plan(b, h, n, d, e, torch.bfloat16)
    assert n_seg > 4  # gathered states are refused in place
    size = b * h * d * e
    states = _abi.chunk_fwd(inp["q"], inp["k"], inp["v"], s, inp["kv"], torch.empty_like(inp["kv"]))[1]
    lib = _abi.load()
    bwd = lib.lasp_chunk_bwd_twin
    bwd.restype = ctypes.c_int
    bwd.argtypes = [ctypes.c_void_p] * 14 + [ctypes.c_size_t] + [ctypes.c_int] * 2 + [ctypes.c_int64] + [ctypes.c_int] * 4 + [ctypes.c_void_p]

    def run(where):
        room = torch.empty(2 * size, device=gpu_device)  # kv_in, and what may lie half over it
        room[:size] = inp["kv"].flatten()
        dkv_in, dkv_out, twin = inp["dkv"].clone(), torch.empty_like(inp["dkv"]), None
        if where == "kv_in":
            dkv_out = room[:size]
        elif where == "part of kv_in":
            dkv_out = room[size // 2:size // 2 + size]
        elif where == "dkv_in":
            dkv_out = dkv_in
        elif where == "twin over kv_in":
            twin = room[:size]
        grads = [torch.empty_like(inp[x]) for x in "qkv"]
        ws = torch.empty(2 * state_bytes // 4, device=gpu_device)
        p = lambda t: None if t is None else t.data_ptr()
        rc, launches = profiled(lambda: bwd(
            p(inp["q"]), p(inp["k"]), p(inp["v"]), p(s), p(inp["do"]), p(room), p(dkv_in), *map(p, grads), p(dkv_out), p(twin),
            p(states) if kept else None, p(ws), 2 * state_bytes, b, h, n, d, e, 1, seg_len, _abi._raw_stream(gpu_device)))
        assert rc == 0, lib.lasp_last_error()
        if twin is not None:
            assert torch.equal(twin, dkv_out.flatten())
        return dict(zip(("dq", "dk", "dv", "dkv_out"), (*grads, dkv_out.view(b, h, d, e)))), launches

    apart, launches = run(None)
    assert launches == {"fused": 1}
    got, launches = run(over)
    assert "fused" not in launches and launches["bwd3"] == 1
    check(got, apart, 2e-2, what=over)
