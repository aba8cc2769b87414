"""Argument checks of the calls that leave the outgoing state in two places, and of the few-token call (host code only)."""
import ctypes

import pytest

from lasp_amd import _abi

P = ctypes.c_void_p
MB = 1 << 20


@pytest.mark.parametrize("backward", [False, True])
def test_a_twin_overlaps_nothing(backward):
    lib = _abi.load()
    size = 2 * 128 * 128 * 4

    def call(out, twin):
        state = [P(1 * MB), P(out) if out else None, P(twin)]  # incoming, outgoing, twin
        if backward:
            dq, dk, dv = P(20 * MB), P(21 * MB), P(22 * MB)
            return lib.lasp_chunk_bwd_twin(P(10 * MB), P(11 * MB), P(12 * MB), P(13 * MB), P(14 * MB), None, state[0], dq, dk,
                                           dv, state[1], state[2], None, P(30 * MB), ctypes.c_size_t(64 * MB), 1, 2,
                                           ctypes.c_int64(512), 128, 128, 1, 128, None)
        return lib.lasp_chunk_fwd_twin(P(10 * MB), P(11 * MB), P(12 * MB), P(13 * MB), *state, P(20 * MB), P(30 * MB), 1, 2,
                                       ctypes.c_int64(512), 128, 128, 1, 128, None)

    for twin in (1 * MB, 1 * MB + size - 4, 2 * MB, 2 * MB - 4):
        assert call(2 * MB, twin) == -8 and b"twin" in lib.lasp_last_error(), twin
    assert call(2 * MB, 1 * MB + size + 2) == -6   # next to both, but on no 4-byte boundary
    assert call(0, 3 * MB) == -1                   # a twin of a state that is not wanted
    assert call(2 * MB, 2 * MB + size) == -7       # passes these checks; none of these addresses is device memory


def test_few_token_call_refuses_other_shapes():
    lib = _abi.load()
    step = lambda n, d, e, o=20 * MB: lib.lasp_step_fwd(P(10 * MB), P(11 * MB), P(12 * MB), P(13 * MB), None, None, P(o) if o else None,
                                                        1, 2, ctypes.c_int64(n), d, e, 1, None)
    assert step(5, 128, 128) == -2 and step(1, 136, 128) == -2 and step(1, 128, 126) == -2
    assert b"lasp_step_fwd" in lib.lasp_last_error()
    assert step(1, 128, 128, 0) == -1
    assert step(4, 128, 128) == -7
