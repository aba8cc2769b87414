"""What the 16-bit backward's kernels rely on in the rule for its sweeps (lasp_bwd_rows), over shapes on all sides of it: no GPU."""
import ctypes
import itertools

import pytest
import torch

from helpers import bwd_rows
from lasp_amd import _abi


@pytest.mark.parametrize("d,e", [(128, 128), (96, 80), (192, 128), (256, 72), (512, 128), (64, 64)])
def test_rows(d, e):
    seen, dtype = set(), torch.bfloat16
    for bh, n, seg_len in itertools.product((1, 2, 3, 5, 8, 13, 16, 24, 27, 41, 57, 64, 80, 96, 300),
                                            (65, 309, 431, 520, 919, 1344, 1536, 2225, 3757, 4096, 8192, 16384, 65536), (0, 64, 128, 192, 256, 512, 1024)):
        segment, n_seg, _ = _abi.plan(1, bh, n, d, e, dtype, seg_len)
        row = bwd_rows(1, bh, n, d, e, dtype, seg_len)
        if row == 0:
            continue
        m = row // segment
        assert row == m * segment and 1 <= m <= min(8, n_seg) and (m == 1 or row <= 64 * (24 if d > 128 else 40)), (bh, n, seg_len, row)
        seen.add((m, row >= n))
    if (d, e) == (64, 64):
        assert {x[0] for x in seen} == {1}  # two workgroups share a CU: one segment each
    else:
        assert {x[0] for x in seen} == set(range(1, 9)) and any(x[1] and x[0] > 1 for x in seen)


def test_where_there_are_none():
    assert bwd_rows(2, 12, 2048, 128, 128, torch.bfloat16, 0) == 0                                    # one launch
    assert bwd_rows(2, 12, 2048, 128, 128, torch.bfloat16, _abi.plan(2, 12, 2048, 128, 128, torch.bfloat16)[0]) == 0  # ... the plan's length
    assert bwd_rows(2, 12, 512, 128, 128, torch.bfloat16, 0) == 0 and bwd_rows(1, 64, 8192, 128, 128, torch.bfloat16, 2048) == 0  # gathered
    assert bwd_rows(1, 16, 4096, 128, 128, torch.float32, 0) == 0
    assert bwd_rows(2, 12, 2048, 128, 128, torch.bfloat16, 192) > 0
    lib, n = _abi.load(), ctypes.c_int64
    assert lib.lasp_bwd_rows(0, 1, n(1), 128, 128, 1, 0, None) < 0 and lib.lasp_bwd_rows(1, 16, n(8192), 128, 128, 1, 0, None) == 0
