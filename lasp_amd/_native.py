"""Loads lasp_amd/_lasp_torch.so, the native PyTorch side of the library (lasp_amd/csrc/lasp_torch.cpp).

Its functions take an operator's usual case from the Python call to the enqueued kernels and the autograd node, and
return None for any other, which the callers then hand to the Python path over ctypes (`_abi`, `_chain`)."""
from __future__ import annotations

import os

import torch  # noqa: F401  (the extension links against torch's libraries: they have to be in the process first)

from . import _abi

_EXT_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lasp_torch.so")
_ext = None


def ext():
    """The extension module, loaded once; raises if it has not been built."""
    global _ext
    if _ext is None:
        if not os.path.exists(_EXT_PATH):
            raise _abi.LaspError(f"{_EXT_PATH} is missing: build it with `python -m lasp_amd.build`")
        _abi.load()
        from . import _chain, _lasp_torch

        _lasp_torch.bind(_abi.LaspError, _chain.before_native_backward, _chain.after_backward, _chain.after_native_forward)
        _ext = _lasp_torch
    return _ext


def chunk_fwd(q, k, v, s, kv_in=None, kv_out=None, keep=True):
    """`_abi.chunk_fwd` under the default plan, natively where the extension takes the call.  keep=False: the caller has
    no use for the segment states, and None may be returned in their place."""
    if q.is_cuda:
        done = ext().chunk_fwd(q, k, v, s, kv_in, kv_out, 0, keep)
        if done is not None:
            return done
    return _abi.chunk_fwd(q, k, v, s, kv_in=kv_in, kv_out=kv_out)


def chunk_bwd(q, k, v, s, do, kv_in=None, dkv_in=None, dkv_out=None, kv_seg_states=None, seg_len=0):
    """`_abi.chunk_bwd`, natively where the extension takes the call."""
    if q.is_cuda:
        done = ext().chunk_bwd(q, k, v, s, do, kv_in, dkv_in, dkv_out, kv_seg_states, seg_len)
        if done is not None:
            return done
    return _abi.chunk_bwd(q, k, v, s, do, kv_in=kv_in, dkv_in=dkv_in, dkv_out=dkv_out, kv_seg_states=kv_seg_states,
                          seg_len=seg_len)
