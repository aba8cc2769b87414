"""The native extension's answer to calls that it leaves to the Python path, as far as it can be had without a GPU."""
import torch

from lasp_amd import _native


def test_a_chunk_without_state_buffers_is_left_to_the_python_path():
    t, s, KV = torch.zeros(1, 2, 4, 8), torch.zeros(2), torch.zeros(1, 2, 8, 8)
    for kv, dkv in ((None, None), (KV, None), (None, KV)):
        assert _native.ext().takes(t, t, t, s, kv, dkv) is False
