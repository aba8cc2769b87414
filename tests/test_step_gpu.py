"""A few tokens under their states (lasp_step.hip): outputs and states against the recurrence in 64 bits, in place or not,
with and without an incoming or outgoing state, at every edge of the kernel's slabs and row groups."""
import pytest
import torch

import lasp_amd
from lasp_amd import _abi, _native

pytestmark = pytest.mark.gpu


def _recurrence(q, k, v, s, kv):
    q, k, v, kv = [t.double().cpu() for t in (q, k, v, kv)]
    lam = torch.exp(-s.double().cpu().reshape(1, -1, 1, 1))
    out = []
    for t in range(q.shape[2]):
        kv = kv + k[:, :, t, :, None] * v[:, :, t, None, :]
        out.append(torch.matmul(q[:, :, t, None, :], kv))
        kv = lam * kv
    return torch.cat(out, 2), kv


# one rounding of the output (2^-9 for bf16, 2^-12 for fp16), or the rounding of fp32 sums of up to 128 terms
REL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 1e-6}


@pytest.mark.parametrize("b,h,n,d,e", [(1, 1, 1, 128, 128), (32, 16, 1, 128, 128), (3, 5, 1, 80, 96), (2, 3, 4, 128, 64),
                                       (1, 2, 3, 40, 36), (1, 3, 2, 1, 4), (2, 2, 4, 127, 100)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_a_few_tokens(gpu_device, b, h, n, d, e, dtype):
    g = torch.Generator(device=gpu_device).manual_seed(n * 1000 + d)
    mk = lambda w: torch.randn(b, h, n, w, generator=g, device=gpu_device).to(dtype)
    q, k, v = mk(d), mk(d), mk(e)
    s = lasp_amd.build_slope_tensor(h).to(gpu_device)
    # a state that starts 4 bytes off a 16-byte boundary
    room = torch.randn(b * h * d * e + 1, generator=g, device=gpu_device)
    kv = room[1:].view(b, h, d, e)
    before = kv.clone()
    want_o, want_kv = _recurrence(q, k, v, s, before)

    _abi.profile_begin(16)
    out = torch.empty_like(before)
    o, states, _ = _native.chunk_fwd(q, k, v, s, kv_in=kv, kv_out=out, keep=False)
    launches = {name: n for name, (_, n) in _abi.profile_end().items() if n}
    assert launches == {"fused": 1} and states is None
    assert torch.equal(kv, before)
    rel = lambda a, w: float((a.double().cpu() - w).norm() / w.norm())
    assert rel(o, want_o) < REL[dtype] and rel(out, want_kv) < 1e-6

    o2, _, _ = _native.chunk_fwd(q, k, v, s, kv_in=kv, kv_out=kv, keep=False)  # in place
    assert torch.equal(o2, o) and torch.equal(kv, out)
    want_o, want_kv = _recurrence(q, k, v, s, torch.zeros_like(before))
    o3, _, _ = _native.chunk_fwd(q, k, v, s, kv_out=out, keep=False)  # no incoming state
    assert rel(o3, want_o) < REL[dtype] and rel(out, want_kv) < 1e-6
    o4, _, _ = _native.chunk_fwd(q, k, v, s, keep=False)  # no state at all
    assert torch.equal(o4, o3)


def test_states_of_a_few_fp32_tokens_are_kept_for_a_backward(gpu_device):
    """A call that keeps its states (autograd) still leaves what the backward reads."""
    q, k, v, do = [torch.randn(1, 2, 3, 128, device=gpu_device) for _ in range(4)]
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    kv = torch.randn(1, 2, 128, 128, device=gpu_device)
    o, states, seg_len = _native.chunk_fwd(q, k, v, s, kv_in=kv, kv_out=torch.empty_like(kv))
    assert states is not None
    kept = _native.chunk_bwd(q, k, v, s, do, kv_in=kv, kv_seg_states=states, seg_len=seg_len)
    rebuilt = _native.chunk_bwd(q, k, v, s, do, kv_in=kv, seg_len=seg_len)
    assert all(torch.equal(a, b) for a, b in zip(kept, rebuilt))
