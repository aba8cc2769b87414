"""Chunks of which the caches keep only the ends of the segments give the bits of their heads' own, smaller calls, of which they keep
everything."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,n,d,e,seg_len,dtype", [
    (16, 22016, 128, 128, 1024, torch.bfloat16),  # blocks of either kind in a segment; the scan
    (16, 23000, 128, 128, 1088, torch.float16),   # a partial last block in a short last segment
    (64, 5500, 128, 128, 1408, torch.bfloat16),   # four segments, gathered
    (24, 18003, 96, 128, 1216, torch.bfloat16),   # narrow rows
    (8, 44001, 256, 128, 1088, torch.bfloat16),   # slices
    (16, 22000, 128, 128, 4352, torch.bfloat16),  # dQ's loads too
    (256, 2100, 128, 128, 64, torch.bfloat16),    # segments of one block, none of which stays
])
def test_same_bits_as_smaller_calls(gpu_device, h, n, d, e, seg_len, dtype):
    from lasp_amd import _abi

    g = torch.Generator(device=gpu_device).manual_seed(n + d)
    mk = lambda w: (torch.randn(1, h, n, w, generator=g, device=gpu_device) * 0.3).to(dtype)
    q, k, v, do = mk(d), mk(d), mk(e), mk(e)
    s = torch.linspace(0.4, 0.002, h, device=gpu_device)

    def run(lo, hi):
        x = [t[:, lo:hi].contiguous() for t in (q, k, v, do)]
        o, states, seg = _abi.chunk_fwd(*x[:3], s[lo:hi].contiguous(), seg_len=seg_len)
        if seg_len < 4352:  # (dQ's loads are as usual, and how many segments a sweep goes over depends on the heads)
            return dict(o=o)
        return dict(zip(("o", "dq", "dk", "dv"), (o, *_abi.chunk_bwd(*x[:3], s[lo:hi].contiguous(), x[3], kv_seg_states=states, seg_len=seg))))

    whole = run(0, h)
    for lo in range(0, h, h // 4):
        for name, x in run(lo, lo + h // 4).items():
            assert torch.equal(x, whole[name][:, lo:lo + h // 4]), (name, lo)
