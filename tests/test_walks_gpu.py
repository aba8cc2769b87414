"""Walks over the blocks before (after) a segment, of every length from none to seven: the last few (b, h) of these backwards are cut, eight
blocks for heads whose decay reaches far at 0, 3, 5, 6 and 7, for the others into equal segments whose walks end at the reach.  The products
of a walk block are split over two blocks' time, so that odd and even walks end differently."""
import pytest
import torch

import lasp_amd
from oracle import lasp_oracle as O

pytestmark = pytest.mark.gpu

# one rounding of an input-sized operand per product and one of the result: 2^-9 (bf16), 2^-12 (fp16), a few of them
REL = {torch.bfloat16: 1.2e-2, torch.float16: 1.6e-3}


@pytest.mark.parametrize("h,n,d,e,dtype", [
    (82, 450, 128, 128, torch.bfloat16),  # eight blocks, the last with two tokens
    (81, 448, 128, 128, torch.float16),   # seven whole ones, cut at 0, 3, 5 and 6
    (83, 130, 96, 72, torch.bfloat16),    # narrow rows, walks of none, one and two
])
@pytest.mark.parametrize("slope", [0.0, 0.01, 0.07, 0.2])  # walks to the chunk's end; as far as the decay reaches, four blocks and two
def test_walks_of_every_length(gpu_device, h, n, d, e, dtype, slope):
    g = torch.Generator().manual_seed(h + n)
    mk = lambda w: (torch.randn(1, h, n, w, generator=g) / w ** 0.5).to(dtype)
    q, k, v, do = mk(d), mk(d), mk(e), mk(e)
    s = torch.full((h, 1, 1), slope)
    ref = O.ref_chunked(q, k, v, s, do, dtype=torch.float64)
    leaves = [t.to(gpu_device).requires_grad_(True) for t in (q, k, v)]
    out = lasp_amd.lightning_attn(*leaves, s.to(gpu_device))
    out.backward(do.to(gpu_device))
    for x, name in zip((out.detach(), *(t.grad for t in leaves)), ("o", "dq", "dk", "dv")):
        diff, want = x.double().cpu() - ref[name], ref[name]
        rel = diff.flatten(2).norm(dim=2) / want.flatten(2).norm(dim=2)
        assert float(rel.max()) < REL[dtype], (name, float(rel.max()), int(rel.argmax()))
