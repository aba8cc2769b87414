"""Shared machinery of the lasp_* operators: one autograd Function that runs a chunk
through the C ABI and passes the d x e state along the sequence-parallel chain.

Choreography (forward: rank r-1 -> r -> r+1, backward reversed) follows
lasp/lasp_fuse.py:478-532 and lasp/lasp_fuse_parallel.py:1073-1137: receive the
incoming state unless first in the chain, keep it for backward, run the chunk
(which leaves the outgoing state in the caller's KV buffer), send that on unless
last; backward mirrors this with DKV.  KV and DKV receive no gradient.

The reference zeroes KV, receives into it and clones it (lasp/lasp_fuse.py:485-496).
Here the received state lands in a tensor of its own (`state_take`), which is both the
kernel's input and the copy kept for backward, and the first rank passes "no incoming
state" instead of a zeroed buffer: the caller's KV is only ever written, with KV_out,
so what it holds on entry does not matter and no zero / copy / clone kernels run per chunk.
"""
from __future__ import annotations

import torch

from . import _native
from .utils import seq_parallel_manager as spm


def feature_slices(d: int):
    """Column ranges the public wrappers cut q and k into.

    One kernel launch takes d <= 128, so wider heads are processed as 128-wide
    slices whose outputs add up (Q K^T is a sum over feature slices), as
    lasp/lightning_attention.py:513-529 does.
    """
    width = 128
    return [(lo, min(lo + width, d)) for lo in range(0, d, width)]


class Exchange:
    """Where a chunk sits in its chain: whom it receives states from and sends them to.

    rebind: the outgoing state goes to a new tensor and the caller's KV / DKV buffer is left
    holding the INCOMING state, which is what lasp_fuse_parallel's `KV = ...` rebinding does
    (lasp/lasp_fuse_parallel.py:941-942,1099-1106); otherwise the buffer receives the outgoing
    state in place (lasp/lasp_fuse.py:126-127,352-353).
    tag: feature-slice index, keeps the loopback messages of different slices apart.
    """

    __slots__ = ("group", "rank", "world", "prev_rank", "next_rank", "rebind", "tag")

    def __init__(self, rebind, tag=0):
        self.group = spm.get_sequence_parallel_group()
        self.rank = spm.get_sequence_parallel_rank()
        self.world = spm.get_sequence_parallel_world_size()
        self.prev_rank = spm.get_seq_parallel_send_rank()
        self.next_rank = spm.get_seq_parallel_receive_rank()
        self.rebind, self.tag = rebind, tag

    def _outgoing(self, buffer, incoming, wanted):
        if not self.rebind:
            return buffer
        if incoming is None:
            buffer.zero_()
        else:
            buffer.copy_(incoming)
        return torch.empty_like(buffer) if wanted else None  # the last rank's outgoing state goes nowhere

    def before_forward(self, KV, barrier):
        """(state entering the chunk or None, tensor for the state that leaves it or None)."""
        if barrier and not isinstance(self.group, spm.LoopbackGroup):
            torch.distributed.barrier()
        kv_in = spm.state_take(KV, self.prev_rank, self.group, tag=self.tag) if self.rank > 0 else None
        return kv_in, self._outgoing(KV, kv_in, self.rank < self.world - 1)

    def twin(self, buffer, outgoing):
        """A tensor for a second copy of the outgoing state, or None: where the caller keeps `outgoing` in its buffer and
        the loopback would park a copy of it, the kernels write that copy beside the original."""
        if outgoing is not buffer or not isinstance(self.group, spm.LoopbackGroup):
            return None
        return torch.empty_like(buffer)

    def after_forward(self, kv_out, twin=None):
        if self.rank < self.world - 1:
            spm.state_send(kv_out if twin is None else twin, self.next_rank, self.group, tag=self.tag,
                           give=self.rebind or twin is not None)


def before_backward(x: Exchange, DKV):
    """The same for the backward of the chunk, whose states travel the other way."""
    dkv_in = None
    if x.rank < x.world - 1:
        dkv_in = spm.state_take(DKV, x.next_rank, x.group, dst=x.rank, tag=x.tag)
    return dkv_in, x._outgoing(DKV, dkv_in, x.rank > 0)


def after_backward(x: Exchange, dkv_out, twin=None):
    if x.rank > 0:
        spm.state_send(dkv_out if twin is None else twin, x.prev_rank, x.group, src=x.rank, tag=x.tag,
                       give=x.rebind or twin is not None)


@torch.no_grad()
def after_native_forward(x: Exchange, kv_out, twin=None):
    """Exchange.after_forward, called by the extension between the kernels of a chunk and the saving of its tensors."""
    x.after_forward(kv_out, twin)


def before_native_backward(x: Exchange, DKV):
    """before_backward for the native node: the outgoing state's twin comes third (see Exchange.twin)."""
    dkv_in, dkv_out = before_backward(x, DKV)
    return dkv_in, dkv_out, x.twin(DKV, dkv_out) if x.rank > 0 else None


class ChunkFunction(torch.autograd.Function):
    """forward(q, k, v, s, KV, DKV, cache_states, barrier, rebind=False, tag=0) -> o

    KV / DKV: caller-owned float32 (b, h, d, e) buffers, or None for the stateless
    single-device operator (then nothing is sent or received).
    cache_states: keep the per-segment incoming states for backward (the
    lasp_fuse_parallel trade, lasp/lasp_fuse_parallel.py:1103) instead of
    recomputing them (lasp_fuse, whose backward re-runs the kv recurrence,
    lasp/lasp_fuse.py:237-260).
    rebind, tag: see Exchange.
    """

    @staticmethod
    def forward(ctx, q, k, v, s, KV, DKV, cache_states, barrier, rebind=False, tag=0):
        chained = KV is not None
        ctx.chained = chained
        if not chained:
            o, states, seg_len = _native.chunk_fwd(q, k, v, s)
            ctx.save_for_backward(q, k, v, s, states if cache_states else None)
            ctx.seg_len = seg_len
            return o

        x = Exchange(rebind, tag)
        kv_in, kv_out = x.before_forward(KV, barrier)
        o, states, seg_len = _native.chunk_fwd(q, k, v, s, kv_in=kv_in, kv_out=kv_out)
        # DKV is a scratch buffer that later backward calls overwrite in place, so it is
        # kept by reference rather than as a version-checked saved tensor.
        ctx.save_for_backward(q, k, v, s, states if cache_states else None, kv_in)
        ctx.dkv_buffer = DKV
        ctx.seg_len = seg_len
        ctx.exchange = x
        x.after_forward(kv_out)
        return o

    @staticmethod
    def backward(ctx, do):
        none = (None,) * 7
        if not ctx.chained:
            q, k, v, s, states = ctx.saved_tensors
            dq, dk, dv = _native.chunk_bwd(q, k, v, s, do, kv_seg_states=states, seg_len=ctx.seg_len)
            return (dq, dk, dv) + none

        q, k, v, s, states, kv_in = ctx.saved_tensors
        dkv_in, dkv_out = before_backward(ctx.exchange, ctx.dkv_buffer)
        dq, dk, dv = _native.chunk_bwd(q, k, v, s, do, kv_in=kv_in, dkv_in=dkv_in, dkv_out=dkv_out,
                                    kv_seg_states=states, seg_len=ctx.seg_len)
        after_backward(ctx.exchange, dkv_out)
        return (dq, dk, dv) + none


def native_chunk(q, k, v, s, KV, DKV, barrier, rebind=False):
    """A chunk of a chain as ChunkFunction runs it (states kept for backward), through the native autograd node;
    None where the extension does not take the call."""
    if not q.is_cuda:
        return None
    ext = _native.ext()
    if not ext.takes(q, k, v, s, KV, DKV):
        return None
    x = Exchange(rebind)
    with torch.no_grad():  # as in a Function's forward: the buffers take no part in the graph, whatever they require
        kv_in, kv_out = x.before_forward(KV, barrier)
        twin = x.twin(KV, kv_out) if x.rank < x.world - 1 else None
    return ext.chunk(q, k, v, s, kv_in, kv_out, twin, DKV, x)


def run_sliced(q, k, v, ed, KV, DKV, cache_states, barrier, rebind=False):
    """Applies ChunkFunction per feature slice of q/k and adds the outputs (the library slices 16-bit heads itself, see
    native_chunk)."""
    d = q.shape[-1]
    parts = feature_slices(d)
    if len(parts) == 1:
        return ChunkFunction.apply(q, k, v, ed, KV, DKV, cache_states, barrier, rebind, 0)
    out = None
    for tag, (lo, hi) in enumerate(parts):
        q1, k1 = q[..., lo:hi], k[..., lo:hi]
        if KV is None:
            o = ChunkFunction.apply(q1, k1, v, ed, None, None, cache_states, barrier, rebind, tag)
        else:
            kv1 = KV[:, :, lo:hi].contiguous()
            dkv1 = DKV[:, :, lo:hi].contiguous()
            o = ChunkFunction.apply(q1, k1, v, ed, kv1, dkv1, cache_states, barrier, rebind, tag)
            KV[:, :, lo:hi].copy_(kv1)
        out = o if out is None else out + o
    return out
