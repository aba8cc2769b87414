"""float32 rows narrower than 128 features on the MFMA kernels (lasp_narrow_fwd, lasp_narrow_bwd): widths around their tiles of 32
features and vectors of 4, lengths around their blocks of 32 tokens, against the oracle in 64 bits; nothing is written beside
the outputs; results do not depend on which of the two Python paths took the call."""
import pytest
import torch

import lasp_amd
from lasp_amd import _abi, _native
from oracle import lasp_oracle as O
from tests.helpers import NORM_F32, check, check_norm, make_inputs

pytestmark = pytest.mark.gpu

# as for rows of 128 features: an output element is rounded 60 times at most, a state 12 times a block (at most 9 blocks here),
# each time by at most 2^-24 of a partial sum; operands and decays add a few such roundings
TOL = 180 * 2.0 ** -24
H = 3
WIDTHS = [(4, 4), (32, 36), (64, 64), (64, 60), (68, 8), (96, 96), (80, 80), (100, 124), (128, 64), (64, 128), (124, 128)]


def _run(inp, s, seg, cached=True):
    dev = {k: (t.cuda() if t is not None else None) for k, t in inp.items()}
    s = s.cuda()
    kv_out, dkv_out = (torch.empty_like(dev["kv"]) for _ in range(2)) if dev["kv"] is not None else (None, None)
    o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], s, kv_in=dev["kv"], kv_out=kv_out, seg_len=seg)
    dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], s, dev["do"], kv_in=dev["kv"], dkv_in=dev["dkv"],
                                dkv_out=dkv_out, kv_seg_states=states if cached else None, seg_len=seg_len)
    return dict(o=o, kv_out=kv_out, dq=dq, dk=dk, dv=dv, dkv_out=dkv_out)


@pytest.mark.parametrize("d,e", WIDTHS)
@pytest.mark.parametrize("n,state", [(1, True), (33, False), (128, True), (260, True)])
def test_widths(d, e, n, state):
    inp = make_inputs(1, H, n, d, e, torch.float32, seed=n + d + e, scale=0.1, state=state)
    assert not _abi._pad_to_mfma(inp["q"], inp["v"])
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], inp["kv"], inp["dkv"], dtype=torch.float64)
    for cached in (True, False):
        got = _run(inp, s, 64, cached)
        check(got, ref, TOL, what=f"d={d} e={e} n={n} cached={cached}")
        check_norm(got, ref, NORM_F32, what=f"d={d} e={e} n={n} cached={cached}")


@pytest.mark.parametrize("d,e", WIDTHS)
def test_as_padded_to_128(d, e):
    """The same numbers as from rows that are padded with zeros: to the bit, since zeros add nothing."""
    inp = make_inputs(2, H, 200, d, e, torch.float32, seed=d * e, scale=0.1, state=True)
    dev = {k: t.cuda() for k, t in inp.items()}
    s = lasp_amd.build_slope_tensor(H).cuda()
    got = _run(inp, s.cpu(), 64)

    def rows(t):
        return _abi._pad_last(t, 128)

    kv, dkv = (_abi._pad_state(dev[x], d, e) for x in ("kv", "dkv"))
    kv_out, dkv_out = torch.empty_like(kv), torch.empty_like(dkv)
    args = rows(dev["q"]), rows(dev["k"]), rows(dev["v"]), s
    o, states, seg = _abi._chunk_fwd_exact(*args, kv_in=kv, kv_out=kv_out, seg_len=64)
    dq, dk, dv = _abi._chunk_bwd_exact(*args, rows(dev["do"]), kv_in=kv, dkv_in=dkv, dkv_out=dkv_out, kv_seg_states=states, seg_len=seg)
    want = dict(o=o[..., :e], dq=dq[..., :d], dk=dk[..., :d], dv=dv[..., :e], kv_out=kv_out[:, :, :d, :e], dkv_out=dkv_out[:, :, :d, :e])
    for name, t in want.items():
        assert torch.equal(got[name], t), name


@pytest.mark.parametrize("d,e", [(64, 64), (36, 100), (80, 96)])
def test_neighbouring_memory(d, e):
    """Outputs between guard bands, through the C entry points."""
    b, n, guard, code = 1, 70, 4096, _abi.DTYPE_CODE[torch.float32]
    inp = {k: t.cuda() for k, t in make_inputs(b, H, n, d, e, torch.float32, seed=1, scale=0.1, state=True).items()}
    s = lasp_amd.build_slope_tensor(H).cuda()
    seg, _, nbytes = _abi.plan(b, H, n, d, e, torch.float32, 64)
    lib, stream = _abi.load(), torch.cuda.current_stream().cuda_stream

    def guarded(count):
        return torch.full((guard + count + guard,), 7.25, device="cuda")

    def inner(t):
        return t.data_ptr() + 4 * guard

    def whole(t):
        return bool((t[:guard] == 7.25).all() and (t[-guard:] == 7.25).all())

    o, dq, dk, dv = (guarded(b * H * n * w) for w in (e, d, d, e))
    kv, dkv, twin = (guarded(b * H * d * e) for _ in range(3))
    states, ws = guarded(nbytes // 4), guarded(nbytes // 4)
    p = {k: t.data_ptr() for k, t in inp.items()}
    assert lib.lasp_narrow_fwd(p["q"], p["k"], p["v"], s.data_ptr(), p["kv"], inner(kv), inner(twin), inner(o), inner(states), b, H, n, d, e,
                               code, seg, stream) == 0
    assert lib.lasp_narrow_bwd(p["q"], p["k"], p["v"], s.data_ptr(), p["do"], p["kv"], p["dkv"], inner(dq), inner(dk), inner(dv),
                               inner(dkv), None, inner(states), inner(ws), nbytes, b, H, n, d, e, code, seg, stream) == 0
    torch.cuda.synchronize()
    assert all(whole(t) for t in (o, dq, dk, dv, kv, dkv, twin, states, ws))
    assert torch.equal(kv, twin)


@pytest.mark.parametrize("d,e", [(64, 64), (96, 80)])
def test_native_and_python_paths_agree(d, e):
    inp = {k: t.cuda() for k, t in make_inputs(2, H, 300, d, e, torch.float32, seed=2, scale=0.1, state=False).items() if t is not None}
    s = lasp_amd.build_slope_tensor(H).cuda()
    leaves = [inp[x].requires_grad_() for x in "qkv"]
    o = _native.ext().attention(*leaves, s)
    assert o is not None
    grads = torch.autograd.grad(o, leaves, inp["do"])
    with torch.no_grad():
        o2, states, seg = _abi.chunk_fwd(*leaves, s)
        grads2 = _abi.chunk_bwd(*leaves, s, inp["do"], kv_seg_states=states, seg_len=seg)
    for a, c in zip((o, *grads), (o2, *grads2)):
        assert torch.equal(a, c)


def _shifted(t):
    """The same numbers in a view that starts 4 bytes past a multiple of 16."""
    room = torch.empty(t.numel() + 1, device="cuda")
    out = room[1:].view(t.shape).copy_(t)
    assert out.data_ptr() % 16 == 4
    return out


@pytest.mark.parametrize("native", [True, False])
def test_rows_that_start_off_a_vector(native):
    inp = {k: t.cuda() for k, t in make_inputs(1, H, 70, 64, 36, torch.float32, seed=3, scale=0.1, state=False).items() if t is not None}
    s = lasp_amd.build_slope_tensor(H).cuda()
    seen = []
    for place in (torch.clone, _shifted):
        q, k, v, do = (place(inp[x]) for x in ("q", "k", "v", "do"))
        if native:
            leaves = [t.requires_grad_() for t in (q, k, v)]
            o = _native.ext().attention(*leaves, s)
            seen.append((o, *torch.autograd.grad(o, leaves, do)))
        else:
            o, states, seg = _abi.chunk_fwd(q, k, v, s)
            seen.append((o, *_abi.chunk_bwd(q, k, v, s, do, kv_seg_states=states, seg_len=seg)))
    assert all(torch.equal(a, c) for a, c in zip(*seen))


def _overlapping(state, apart):
    """`state` and room for another that starts `apart` floats after it, in one buffer."""
    first, second = max(-apart, 0), max(apart, 0)
    room = torch.zeros(state.numel() + abs(apart), device="cuda")
    views = [room[at:at + state.numel()].view(state.shape) for at in (first, second)]
    views[0].copy_(state)
    return views


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("apart", [4, -4, 64 * 36])
def test_states_that_lie_partly_over_each_other(native, apart):
    """As where rows are padded; states of full rows are refused."""
    inp = {k: t.cuda() for k, t in make_inputs(1, H, 300, 64, 36, torch.float32, seed=4, scale=0.1, state=True).items()}
    s = lasp_amd.build_slope_tensor(H).cuda()
    calls = _native if native else _abi

    def run(pair):
        kv, kv_out = pair(inp["kv"])
        o, _, _ = calls.chunk_fwd(inp["q"], inp["k"], inp["v"], s, kv_in=kv, kv_out=kv_out)
        dkv, dkv_out = pair(inp["dkv"])
        grads = calls.chunk_bwd(inp["q"], inp["k"], inp["v"], s, inp["do"], kv_in=inp["kv"], dkv_in=dkv, dkv_out=dkv_out)
        return (o, kv_out, *grads, dkv_out)

    got, want = run(lambda t: _overlapping(t, apart)), run(lambda t: (t.clone(), torch.empty_like(t)))
    assert all(torch.equal(a, c) for a, c in zip(got, want))
    full = torch.zeros(1, H, 64, 128, device="cuda")
    kv, kv_out = _overlapping(torch.zeros(1, H, 128, 128, device="cuda"), apart)
    with pytest.raises(_abi.LaspError, match="overlaps"):
        calls.chunk_fwd(full, full, full, s, kv_in=kv, kv_out=kv_out)


@pytest.mark.parametrize("d,e,b,n", [(64, 64, 16, 1800), (96, 80, 32, 600)])
def test_segments_of_512_tokens_cut_in_two(d, e, b, n):
    """The default plan where it halves a segment that has a CU to itself."""
    h = 4
    assert _abi.plan(b, h, n, d, e, torch.float32, 0)[0] == 256
    assert _abi.plan(b, h, n, 128, 128, torch.float32, 0)[0] == 512
    inp = make_inputs(b, h, n, d, e, torch.float32, seed=n, scale=0.1, state=True)
    s = lasp_amd.build_slope_tensor(h)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], inp["kv"], inp["dkv"], dtype=torch.float64)
    check(_run(inp, s, 0), ref, (60 + 12 * -(-n // 32)) * 2.0 ** -24, what=f"d={d} e={e} n={n}")
