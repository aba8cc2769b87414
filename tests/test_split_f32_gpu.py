"""The fp32 MFMA kernels multiply numbers split into three bf16 parts: lengths around their 32-token blocks, and numbers for
which a split could go wrong, against the oracle in 64 bits."""
import pytest
import torch

import lasp_amd
from lasp_amd import _abi
from oracle import lasp_oracle as O
from tests.helpers import NORM_F32, check, check_norm, make_inputs

pytestmark = pytest.mark.gpu

# An output element is rounded 48 times in the state term and 12 in the intra-block term, a state 12 times a block (at most 9
# blocks here), each time by at most 2^-24 of a partial sum; operands and decays add a few such roundings.
TOL = 180 * 2.0 ** -24
H = 4


def _run(inp, s, seg):
    dev = {k: (t.cuda() if t is not None else None) for k, t in inp.items()}
    s = s.cuda()
    kv_out, dkv_out = (torch.empty_like(dev["kv"]) for _ in range(2)) if dev["kv"] is not None else (None, None)
    o, states, seg_len = _abi.chunk_fwd(dev["q"], dev["k"], dev["v"], s, kv_in=dev["kv"], kv_out=kv_out, seg_len=seg)
    dq, dk, dv = _abi.chunk_bwd(dev["q"], dev["k"], dev["v"], s, dev["do"], kv_in=dev["kv"], dkv_in=dev["dkv"],
                                dkv_out=dkv_out, kv_seg_states=states, seg_len=seg_len)
    return dict(o=o, kv_out=kv_out, dq=dq, dk=dk, dv=dv, dkv_out=dkv_out)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 97, 260])
@pytest.mark.parametrize("state", [True, False])
def test_lengths(n, state):
    inp = make_inputs(1, H, n, 128, 128, torch.float32, seed=n, scale=0.1, state=state)
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], inp["kv"], inp["dkv"], dtype=torch.float64)
    got = _run(inp, s, 64)
    check(got, ref, TOL, what=f"n={n}")
    check_norm(got, ref, NORM_F32, what=f"n={n}")


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
    check_norm(got, ref, NORM_F32, names=("o", "dq", "dk", "dv"))


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("value", [1.0077972, 0.7071068, 0.1, 3.14159265])
def test_equal_numbers(d, value):
    """Every product is the same, and so is what it leaves out: nothing averages.  The omitted partial products are at most 2^-22 of
    a product, in each of the up to three products that an output passes through, beside the roundings of the sums, all of one sign."""
    n = 64
    inp = {x: torch.full((1, H, n, d), value) for x in ("q", "k", "v", "do")}
    inp.update(kv=None, dkv=None)
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], dtype=torch.float64)
    check_norm(_run(inp, s, 64), ref, 3 * 2.0 ** -22 + NORM_F32, what=f"{value}")


@pytest.mark.parametrize("n,d", [(1, 128), (3, 128), (3, 64)])
def test_short_sums(n, d):
    """Sums of one or a few products, in which no error averages: features of which one is not zero."""
    inp = make_inputs(16, H, n, d, d, torch.float32, seed=n, state=False)
    for x in ("q", "k"):
        inp[x][..., 1:] = 0
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], dtype=torch.float64)
    check_norm(_run(inp, s, 64), ref, NORM_F32, what=f"n={n} d={d}")


@pytest.mark.parametrize("power", [-109, -115, -120])
def test_small_operands(power):
    """Numbers below 2^-110 have parts under bf16's smallest, 2^-133: they are held to 2^-134 (to the bit above), here in q and in what
    is made of it and k, whose size makes up for it: rows, weighted rows and states, each off by 2^-134 of 2^power."""
    inp = make_inputs(1, H, 130, 128, 128, torch.float32, seed=9, state=False)
    inp["q"], inp["k"] = inp["q"] * 2.0 ** power, inp["k"] * 2.0 ** 100
    s = lasp_amd.build_slope_tensor(H)
    ref = O.ref_chunked(inp["q"], inp["k"], inp["v"], s, inp["do"], dtype=torch.float64)
    got = _run(inp, s, 64)
    tol = NORM_F32 + (3 * 2.0 ** (-134 - power) if power < -110 else 0)
    check_norm(got, ref, tol, names=("o", "dk", "dv"))
    check_norm(got, ref, NORM_F32, names=("dq",))


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


T, CLEAN = 70, 64  # a token in the middle of a 32-token block, and where its block starts
# what an input of token T reaches: outputs from there on (forwards), up to there (backwards), or its own only
REACH = {("q", "o"): "own", ("k", "o"): "later", ("do", "dq"): "own", ("v", "dq"): "later", ("k", "dv"): "own", ("q", "dv"): "earlier",
         ("v", "dk"): "own", ("do", "dk"): "earlier"}


@pytest.mark.parametrize("d,e", [(128, 128), (64, 96)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("name", ["q", "k", "v", "do"])
def test_nonfinite_inputs_stay_where_they_are_seen(name, value, d, e):
    """A NaN or an infinity of a token reaches no token that does not see it, in its own block neither: where it is a factor of
    the scores.  As a summed row (V, and K, Q, dO in their gradients) it meets the masked scores, which are zero, inside a product, and
    other tokens of its block become NaN; no token of the blocks before (after, backwards) does."""
    inp = make_inputs(1, H, 128, d, e, torch.float32, seed=7, scale=0.1, state=False)
    s = lasp_amd.build_slope_tensor(H)
    clean = _run(inp, s, 64)
    bad = dict(inp, **{name: inp[name].clone()})
    bad[name][:, :, T, 9] = value
    got = _run(bad, s, 64)
    for (source, out), reach in REACH.items():
        if source != name:
            continue
        seen = {"own": slice(T, T + 1), "later": slice(T, None), "earlier": slice(0, T + 1)}[reach]
        assert not torch.isfinite(got[out][:, :, T]).all(-1).any(), out
        same = got[out] == clean[out]
        same[:, :, seen] = True
        assert same.all(), (out, (~same).any(-1).nonzero()[:8].tolist())
    if name == "v":
        assert torch.equal(got["o"][:, :, :CLEAN], clean["o"][:, :, :CLEAN])


@pytest.mark.parametrize("d,e", [(128, 128), (64, 96)])
def test_masked_scores_that_overflow(d, e):
    """Finite inputs whose product is too large for fp32 only between tokens that do not see each other."""
    inp = make_inputs(1, H, 128, d, e, torch.float32, seed=8, scale=0.1, state=False)
    inp["q"][:, :, T, 3], inp["do"][:, :, T, 3] = 1e20, 1e20
    s = lasp_amd.build_slope_tensor(H)
    clean = _run(inp, s, 64)
    inp["k"][:, :, T + 5, 3], inp["v"][:, :, T + 5, 3] = 1e20, 1e20
    got = _run(inp, s, 64)
    for out in ("o", "dq"):
        assert torch.isfinite(got[out][:, :, :T + 5]).all()
        assert torch.equal(got[out][:, :, :T + 5], clean[out][:, :, :T + 5]), out
    for out in ("dk", "dv"):
        assert torch.isfinite(got[out][:, :, T + 1:]).all(), out
