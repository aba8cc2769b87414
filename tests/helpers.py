"""Shared helpers for the parity tests (inputs by seed, oracle calls, error metric)."""
import torch

from oracle import lasp_oracle as O

TOL = {torch.float32: 1e-3, torch.bfloat16: 2e-2, torch.float16: 2e-2}
NAMES = ("o", "kv_out", "dq", "dk", "dv", "dkv_out")


def make_inputs(b, h, n, d, e, dtype, seed, scale=1.0, state=True, state_std=0.02, device="cpu"):
    """Seeded N(0, scale^2) q, k, v, do rounded to `dtype`; fp32 states N(0, state_std^2)."""
    g = torch.Generator().manual_seed(seed)
    mk = lambda *shape: (torch.randn(*shape, generator=g) * scale).to(dtype)
    q, k, v, do = mk(b, h, n, d), mk(b, h, n, d), mk(b, h, n, e), mk(b, h, n, e)
    kv = dkv = None
    if state:
        kv = torch.randn(b, h, d, e, generator=g) * state_std
        dkv = torch.randn(b, h, d, e, generator=g) * state_std
    out = dict(q=q, k=k, v=v, do=do, kv=kv, dkv=dkv)
    return {k_: (t.to(device) if t is not None else None) for k_, t in out.items()}


def oracle(inp, s, block=64, dtype=torch.float64):
    """Oracle on the SAME (already rounded) inputs, in fp64 unless told otherwise."""
    c = {k_: (t.detach().cpu() if t is not None else None) for k_, t in inp.items()}
    return O.ref_chunked(c["q"], c["k"], c["v"], s.cpu(), c["do"], c["kv"], c["dkv"], block=block, dtype=dtype)


def check(got: dict, ref: dict, tol: float, names=NAMES, what=""):
    """Asserts the parity bound on every (batch, head) slice of every output: the worst slice's
    max|x - ref| / max|ref| must not exceed `tol`.  The whole-tensor figure goes into the message."""
    errs, whole = {}, {}
    for name in names:
        if name in got and got[name] is not None:
            errs[name] = O.rel_err(got[name], ref[name])
            whole[name] = O.rel_err_whole(got[name], ref[name])
    bad = {k_: v_ for k_, v_ in errs.items() if not (v_ <= tol)}
    assert not bad, f"{what}: worst (b,h) slice over {tol}: {bad} (per-head: {errs}; whole tensor: {whole})"
    return errs


# What the three-part products of the fp32 MFMA kernels leave, as a 2-norm over an output's: some 60 roundings of 2^-25 (of 2^-24 at
# most) of a partial sum, which add up like a random walk to 2.3e-7, and a few of operands and decays; measured 0.7e-7 to 2.2e-7 (n = 1 ...
# 2048).  A product that lost its third parts (2^-17 of an operand) would show 5e-6 and more.
NORM_F32 = 1e-6


def check_norm(got: dict, ref: dict, tol: float, names=NAMES, what=""):
    """Asserts |x - ref| <= tol |ref| in 2-norms over each whole output."""
    errs = {name: float((got[name].cpu().double() - ref[name].double()).norm() / ref[name].double().norm())
            for name in names if got.get(name) is not None}
    assert all(v_ <= tol for v_ in errs.values()), f"{what}: 2-norm over {tol}: {errs}"


def in_place_bits(inp, s, seg):
    """Outputs of a forward and two backwards (the forward's states, rebuilt ones) whose states are updated in place, each
    with that of separate buffers.  Where the library does not take a shape in place in a direction, that one is left out."""
    from lasp_amd import _abi

    shape = (*inp["q"].shape, inp["v"].shape[-1], inp["q"].dtype)
    takes = {backward: _abi.inplace_ok(*shape, seg, backward) for backward in (False, True)}
    assert takes[False]

    def run(in_place):
        buffers = lambda x, backward: (x, x if in_place and takes[backward] else torch.empty_like(x))
        kv, kv_out = buffers(inp["kv"].clone(), False)
        o, states, seg_len = _abi._chunk_fwd_exact(inp["q"], inp["k"], inp["v"], s, kv_in=kv, kv_out=kv_out, seg_len=seg)
        got = [o, kv_out]
        for kept in (states, None):
            dkv, dkv_out = buffers(inp["dkv"].clone(), True)
            got += _abi._chunk_bwd_exact(inp["q"], inp["k"], inp["v"], s, inp["do"], kv_in=inp["kv"], dkv_in=dkv,
                                         dkv_out=dkv_out, kv_seg_states=kept, seg_len=seg_len)
            got.append(dkv_out)
        return got

    return list(zip(run(True), run(False)))


def bwd_rows(b, h, n, d, e, dtype, seg_len):
    """Tokens of a backward sweep as the library has them, see lasp_bwd_rows."""
    import ctypes

    from lasp_amd import _abi

    row = ctypes.c_int(-1)
    rc = _abi.load().lasp_bwd_rows(b, h, ctypes.c_int64(n), d, e, _abi.DTYPE_CODE[dtype], seg_len, ctypes.byref(row))
    assert rc == 0, rc
    return row.value
