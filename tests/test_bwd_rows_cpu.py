"""What the 16-bit backward's kernels rely on in the rule for its sweeps and DKV states (lasp_bwd_rows), over shapes on all sides of it: no GPU."""
import ctypes
import itertools

import pytest
import torch

from helpers import bwd_rows
from lasp_amd import _abi


@pytest.mark.parametrize("d,e", [(128, 128), (96, 80), (192, 128), (256, 72), (512, 128), (64, 64)])
def test_rows_and_pieces(d, e):
    seen, dtype = set(), torch.bfloat16
    for bh, n, seg_len in itertools.product((1, 2, 3, 5, 8, 13, 16, 24, 27, 41, 57, 64, 80, 96, 300),
                                            (65, 309, 431, 520, 919, 1344, 1536, 2225, 3757, 4096, 8192, 16384, 65536), (0, 64, 128, 192, 256, 512, 1024)):
        segment, n_seg, nbytes = _abi.plan(1, bh, n, d, e, dtype, seg_len)
        row, piece = bwd_rows(1, bh, n, d, e, dtype, seg_len, False)
        assert (row == 0) == (piece == 0)
        if row == 0:
            continue
        m, states = row // segment, lambda tokens: -(-n // tokens) * bh * 4 * 128 * 128 * -(-d // 128)
        assert row == m * segment and 1 <= m <= min(8, n_seg) and (m == 1 or row <= 64 * (24 if d > 128 else 40)), (bh, n, seg_len, row)
        assert row % piece == 0 and states(piece) <= nbytes, (bh, n, seg_len, row, piece)
        # where a state leaves the sweeps are the same and the workspace is filled: one state for each piece of the forward's
        kept = bwd_rows(1, bh, n, d, e, dtype, seg_len, True)
        assert kept[0] == row and piece % kept[1] == 0 and segment % kept[1] == 0 and states(kept[1]) == nbytes, (bh, n, seg_len, kept)
        seen.add((m, piece > kept[1], row >= n, piece >= n))
    if (d, e) == (64, 64):
        assert {x[:2] for x in seen} == {(1, False)}  # two workgroups share a CU: one segment each
    else:
        assert {x[0] for x in seen} == set(range(1, 9))
        assert any(x[1] for x in seen) and any(x[2] and not x[3] for x in seen) and any(x[3] and x[0] > 1 for x in seen)


def test_where_there_are_none():
    rows = lambda *a: bwd_rows(*a, False)
    assert rows(2, 12, 2048, 128, 128, torch.bfloat16, 0) == (0, 0)                                    # one launch
    assert rows(2, 12, 2048, 128, 128, torch.bfloat16, _abi.plan(2, 12, 2048, 128, 128, torch.bfloat16)[0]) == (0, 0)  # ... the plan's length
    assert rows(2, 12, 512, 128, 128, torch.bfloat16, 0) == (0, 0) and rows(1, 64, 8192, 128, 128, torch.bfloat16, 2048) == (0, 0)  # gathered
    assert rows(1, 16, 4096, 128, 128, torch.float32, 0) == (0, 0)
    assert rows(2, 12, 2048, 128, 128, torch.bfloat16, 192)[0] > 0
    lib, n = _abi.load(), ctypes.c_int64
    assert lib.lasp_bwd_rows(0, 1, n(1), 128, 128, 1, 0, 0, None, None) < 0 and lib.lasp_bwd_rows(1, 16, n(8192), 128, 128, 1, 0, 0, None, None) == 0
