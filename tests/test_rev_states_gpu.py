"""DKV states of backwards whose sweeps go over several of the forward's segments in a row: in whole and partial rows, for heads that the
scan takes and heads that it leaves out, one row from the other end of the chunk and many."""
import pytest
import torch

from helpers import bwd_rows, check, make_inputs, oracle

pytestmark = pytest.mark.gpu

# As in the other 16-bit parity tests: a few roundings of 2^-9; in fp16 of an eighth.
TOL = {torch.bfloat16: 2e-2, torch.float16: 2e-2 / 8}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e,seg_len", [
    (1, 16, 1088, 128, 128, 64), (2, 8, 1100, 128, 128, 64),  # four of the forward's segments each; the last row one segment, one and 12 tokens
    (1, 12, 897, 128, 128, 64), (1, 16, 641, 128, 64, 64),    # three; one token in the last one
    (1, 12, 1999, 128, 128, 64),                              # six
    (2, 16, 449, 128, 128, 64), (1, 20, 520, 128, 128, 64),   # two rows, three
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


@pytest.mark.parametrize("b,h,n,d,e,seg_len", [(1, 16, 1088, 128, 128, 64), (2, 16, 449, 128, 128, 64), (1, 10, 1300, 192, 128, 64),
                                               (1, 12, 1999, 96, 128, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_state_that_leaves_is_a_sum_of_the_same_pieces(gpu_device, b, h, n, d, e, seg_len, dtype):
    """DKV_out has the bits that a call of few heads gives, whose sweeps go over one segment each: it is a sum of the forward's segments,
    whatever row the sweeps go over.  The gradients do not depend on whether it is asked for."""
    from lasp_amd import _abi

    assert bwd_rows(b, h, n, d, e, dtype, seg_len) > seg_len and bwd_rows(1, 1, n, d, e, dtype, seg_len) == seg_len
    dev = make_inputs(b, h, n, d, e, dtype, seed=n + d, scale=0.3, state=True, state_std=1.0, device=gpu_device)
    s = torch.linspace(0.05, 0.0, h, device=gpu_device)

    def run(part, s, leaves=True):
        out = torch.full_like(part["kv"], float("nan")) if leaves else None
        return out, _abi.chunk_bwd(part["q"], part["k"], part["v"], s, part["do"], part["kv"], part["dkv"], out, None, seg_len)

    whole, grads = run(dev, s)
    for i in range(h):
        one, _ = run({k: v[:1, i:i + 1].contiguous() for k, v in dev.items()}, s[i:i + 1].contiguous())
        assert torch.equal(one, whole[:1, i:i + 1]), i
    for name, x, y in zip(("dq", "dk", "dv"), grads, run(dev, s, leaves=False)[1]):
        assert torch.equal(x, y), name


def chunk_bwd_over(fill, inp, s, kv_in, dkv_in, dkv_out, seg_len):
    """lasp_chunk_bwd without kept states, in a workspace that holds `fill` everywhere: (dq, dk, dv)."""
    from lasp_amd import _abi

    q, v = inp["q"], inp["v"]
    b, h, n, d, e = *q.shape, v.shape[-1]
    seg_len, _, nbytes = _abi.plan(b, h, n, d, e, q.dtype, seg_len)
    ws = torch.full((2 * nbytes // 4,), fill, device=q.device)
    dq, dk, dv = [torch.empty_like(t) for t in (q, q, v)]
    p = lambda t: None if t is None else t.data_ptr()
    rc = _abi.load().lasp_chunk_bwd(p(q), p(inp["k"]), p(v), p(s), p(inp["do"]), p(kv_in), p(dkv_in), p(dq), p(dk), p(dv), p(dkv_out),
                                    None, p(ws), 2 * nbytes, b, h, n, d, e, _abi.DTYPE_CODE[q.dtype], seg_len,
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _abi.load().lasp_last_error()
    return dq, dk, dv


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,e,seg_len", [
    (2, 24, 320, 128, 128, 64), (1, 64, 449, 256, 128, 64),  # five segments, eight with one token in the last
    (1, 41, 431, 96, 80, 64),                                # narrow rows
    (4, 16, 1536, 512, 128, 0),                              # the library's own plan
])
def test_one_row_of_segments(gpu_device, b, h, n, d, e, seg_len, dtype):
    """A sweep over the whole chunk: no head, whatever the next one or the workspace holds, leaves anything but its own sum."""
    assert bwd_rows(b, h, n, d, e, dtype, seg_len) == (-(-n // seg_len) * seg_len if seg_len else n)
    inp = make_inputs(b, h, n, d, e, dtype, seed=n + d + e, scale=0.3, state=True, state_std=1.0)
    # every state dies within the chunk; the slowest is at 2^-25 after it, which a head 2^20 times as large would show
    s = torch.linspace(0.5, 25 / (1.4427 * n), h)
    loud = torch.arange(b * h).view(b, h) % 3 == 1
    if dtype == torch.bfloat16:
        inp["do"][loud] *= 2.0 ** 20
        inp["dkv"][loud] *= 2.0 ** 20
    dev, sd = {k: v.to(gpu_device) for k, v in inp.items()}, s.to(gpu_device)
    what = f"b={b} h={h} n={n} d={d} e={e} {dtype}"

    def run(do, carried, fill=float("nan")):
        kv, dkv = (dev["kv"], dev["dkv"]) if carried else (None, None)
        out = torch.full_like(dev["kv"], float("nan"))
        grads = chunk_bwd_over(fill, dict(dev, do=do), sd, kv, dkv, out, seg_len)
        bare = chunk_bwd_over(fill, dict(dev, do=do), sd, kv, dkv, None, seg_len)  # (the outgoing state not wanted)
        return dict(zip(("dq", "dk", "dv"), grads), dkv_out=out), dict(zip(("dq", "dk", "dv"), bare))

    for carried in (True, False):
        want = oracle(inp if carried else dict(inp, kv=torch.zeros_like(inp["kv"]), dkv=torch.zeros_like(inp["dkv"])), s)
        got, bare = run(dev["do"], carried)
        check(got, {k: want[k] for k in got}, TOL[dtype], what=what)
        check(bare, {k: want[k] for k in bare}, TOL[dtype], what=what + ", no outgoing state")
        # heads that overflow leave the others' bits alone
        do = dev["do"].clone()
        do[loud.to(gpu_device)] = float("inf")
        for name, x in run(do, carried, fill=0.0)[0].items():
            assert torch.equal(x[~loud.to(gpu_device)], got[name][~loud.to(gpu_device)]), (what, name)
