"""The native autograd node (lasp_amd/csrc/lasp_torch.cpp) against the Python autograd Function, which reaches the same kernels
over ctypes: the same bits, graphs that can be kept or not, and the calls that it leaves to the Python path."""
import contextlib

import pytest
import torch

import lasp_amd
from lasp_amd import _abi, _native
from lasp_amd._chain import ChunkFunction

pytestmark = pytest.mark.gpu


def _leaves(dev, b, h, n, d, e, dtype, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    mk = lambda w: (torch.randn(b, h, n, w, generator=g, device=dev) / w ** 0.5).to(dtype)
    return [mk(w).requires_grad_(True) for w in (d, d, e)], mk(e)


@contextlib.contextmanager
def _over_ctypes():
    """ChunkFunction's calls (of the forward and, on autograd's thread, of the backward) go to `_abi` and not to the extension,
    whose plans, workspaces and argument order are what is compared."""
    calls = []
    abi_call = lambda name: lambda *args, **kw: (calls.append(name), getattr(_abi, name)(*args, **kw))[1]
    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(_native, "chunk_fwd", abi_call("chunk_fwd"))
        patch.setattr(_native, "chunk_bwd", abi_call("chunk_bwd"))
        yield
    assert set(calls) == {"chunk_fwd", "chunk_bwd"}


@pytest.mark.parametrize("b,h,n,d,e,dtype", [(1, 2, 1, 128, 128, torch.bfloat16), (2, 3, 300, 64, 40, torch.float16),
                                             (1, 4, 4096, 128, 128, torch.bfloat16), (1, 2, 777, 128, 128, torch.float32),
                                             (1, 2, 500, 256, 128, torch.bfloat16)])
def test_native_node_gives_the_bits_of_the_python_function(gpu_device, b, h, n, d, e, dtype):
    (q, k, v), do = _leaves(gpu_device, b, h, n, d, e, dtype)
    s = lasp_amd.build_slope_tensor(h).to(gpu_device)
    o = lasp_amd.lightning_attn(q, k, v, s)
    assert "LaspChunk" in o.grad_fn.name()
    native = torch.autograd.grad(o, (q, k, v), do, retain_graph=True)
    again = torch.autograd.grad(o, (q, k, v), do)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, (q, k, v), do)
    with _over_ctypes():
        op = ChunkFunction.apply(q, k, v, s, None, None, True, False)
        python = torch.autograd.grad(op, (q, k, v), do)
    assert torch.equal(o, op)
    for a, b_, c in zip(native, again, python):
        assert torch.equal(a, c) and torch.equal(b_, c)
    with torch.no_grad():
        assert lasp_amd.lightning_attn(q, k, v, s).grad_fn is None


def test_calls_that_stay_with_the_python_path(gpu_device):
    """Non-contiguous inputs and expanded gradients run natively; slopes on the host and widths that need padding do not:
    all give the values of the plain call."""
    (q, k, v), do = _leaves(gpu_device, 1, 2, 200, 128, 128, torch.bfloat16)
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    want = lasp_amd.lightning_attn(q, k, v, s)
    strided = lasp_amd.lightning_attn(q.transpose(1, 2).contiguous().transpose(1, 2), k, v, s)
    assert torch.equal(strided, want)
    assert torch.equal(lasp_amd.lightning_attn(q, k, v, s.cpu()), want)
    gs = torch.autograd.grad(want.float().sum(), (q, k, v))
    gd = torch.autograd.grad(lasp_amd.lightning_attn(q, k, v, s), (q, k, v), torch.ones_like(want))
    assert all(torch.equal(a, b) for a, b in zip(gs, gd))
    (q, k, v), _ = _leaves(gpu_device, 1, 2, 100, 60, 36, torch.bfloat16)
    assert lasp_amd.lightning_attn(q, k, v, s).shape == v.shape


@pytest.mark.parametrize("name,rebind", [("lasp_fuse", False), ("lasp_fuse_parallel", True)])
def test_native_chain_gives_the_bits_of_the_python_function(gpu_device, name, rebind):
    _compare_chains(gpu_device, name, rebind, 1100, 128, 128, torch.bfloat16)


@pytest.mark.parametrize("n,d,e,dtype", [(3, 128, 128, torch.bfloat16), (200, 128, 128, torch.float16), (200, 64, 40, torch.bfloat16),
                                         (4096, 128, 128, torch.bfloat16), (2500, 64, 64, torch.bfloat16),
                                         (300, 128, 128, torch.float32)])
def test_chain_on_every_kind_of_kernel_that_leaves_a_state(gpu_device, n, d, e, dtype):
    """The copy of the outgoing state that the kernels write for the next rank, against the one that the Python path makes."""
    _compare_chains(gpu_device, "lasp_fuse", False, n, d, e, dtype)


def _compare_chains(gpu_device, name, rebind, n, d, e, dtype):
    results = []
    s = lasp_amd.build_slope_tensor(4).to(gpu_device)
    for native in (True, False):
        lasp_amd.destroy_parallel_groups()
        lasp_amd.initialize_lasp(1, 3)
        with contextlib.ExitStack() as stack:
            stack.callback(lasp_amd.destroy_parallel_groups)
            if not native:
                stack.enter_context(_over_ctypes())
            KV = torch.empty(1, 4, d, e, device=gpu_device)
            DKV = torch.empty_like(KV)
            outs, leaves, dos = [], [], []
            for c in range(3):
                lasp_amd.set_sequence_parallel_rank(c)
                (q, k, v), do = _leaves(gpu_device, 1, 4, n, d, e, dtype, seed=c)
                if native:
                    outs.append(getattr(lasp_amd, name)(q, k, v, s, KV, DKV))
                else:
                    outs.append(ChunkFunction.apply(q, k, v, s, KV, DKV, True, False, rebind))
                dos.append(do)
                leaves += [q, k, v]
            assert ("LaspChunk" in outs[0].grad_fn.name()) == native
            torch.autograd.backward(outs, dos)
            assert not lasp_amd.loopback_pending()
            results.append([*outs, *[t.grad for t in leaves], KV, DKV])
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_a_receive_without_a_sender_raises_from_the_backward(gpu_device):
    """An error of the state exchange on autograd's thread arrives as the Python exception it is."""
    lasp_amd.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, 2)
    try:
        (q, k, v), do = _leaves(gpu_device, 1, 2, 64, 128, 128, torch.bfloat16)
        KV = torch.empty(1, 2, 128, 128, device=gpu_device)
        lasp_amd.set_sequence_parallel_rank(0)
        o = lasp_amd.lasp_fuse(q, k, v, lasp_amd.build_slope_tensor(2).to(gpu_device), KV, torch.empty_like(KV))
        with pytest.raises(RuntimeError, match="loopback recv"):
            o.backward(do)
    finally:
        lasp_amd.destroy_parallel_groups()


def test_a_state_of_another_shape_is_refused(gpu_device):
    """A received state is read as (b, h, d, e) floats: one that another chunk left with fewer raises, in both directions."""
    from lasp_amd._abi import LaspError
    from lasp_amd.utils import seq_parallel_manager as spm

    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    zeros = lambda *shape, **k: torch.zeros(*shape, device=gpu_device, **k)
    for received in (zeros(1, 2, 64, 128), zeros(1, 2, 128, 128, dtype=torch.bfloat16), zeros(1, 2, 128, 256)[..., ::2],
                     torch.zeros(1, 2, 128, 128)):
        lasp_amd.destroy_parallel_groups()
        lasp_amd.initialize_lasp(1, 2)
        try:
            (q, k, v), do = _leaves(gpu_device, 1, 2, 200, 128, 128, torch.bfloat16)
            KV = torch.empty(1, 2, 128, 128, device=gpu_device)
            DKV = torch.empty_like(KV)
            lasp_amd.set_sequence_parallel_rank(0)
            o = lasp_amd.lasp_fuse(q, k, v, s, KV, DKV)
            spm.state_send(received, 0, spm.get_sequence_parallel_group(), src=1, give=True)
            with pytest.raises(LaspError, match="dkv_in must be"):
                o.backward(do)
            lasp_amd.set_sequence_parallel_rank(1)
            spm.state_recv(torch.empty_like(KV), 0, spm.get_sequence_parallel_group())  # the one that the call above left
            spm.state_send(received, 1, spm.get_sequence_parallel_group(), src=0, give=True)
            with pytest.raises(LaspError, match="kv_in must be"):
                lasp_amd.lasp_fuse(q, k, v, s, KV, DKV)
        finally:
            lasp_amd.destroy_parallel_groups()


@pytest.mark.parametrize("name", ["lasp_fuse", "lasp_fuse_parallel"])
def test_calls_without_state_buffers(gpu_device, name):
    """Without a DKV a forward still runs, and the backward of a group of one; without either the call is the stateless one."""
    op = getattr(lasp_amd, name)
    (q, k, v), do = _leaves(gpu_device, 1, 2, 200, 128, 128, torch.bfloat16)
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    o = lasp_amd.lightning_attn(q, k, v, s)
    want = torch.autograd.grad(o, (q, k, v), do)
    lasp_amd.destroy_parallel_groups()
    KV = torch.empty(1, 2, 128, 128, device=gpu_device)
    with torch.no_grad():
        assert torch.equal(op(q, k, v, s, KV, None), o)
    stateless = op(q, k, v, s, None, None)
    assert torch.equal(stateless, o)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(stateless, (q, k, v), do), want))
    if name == "lasp_fuse":
        assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(op(q, k, v, s, KV, None), (q, k, v), do), want))


@pytest.mark.parametrize("name", ["lasp_fuse", "lasp_fuse_parallel", "lasp_cache"])
def test_state_buffers_that_require_a_gradient(gpu_device, name):
    """They are scratch: they may be leaves that require a gradient, receive none, and their in-place changes are counted."""
    op = getattr(lasp_amd, name)
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    lasp_amd.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, 2)
    try:
        outs, dos = [], []
        KV, DKV = [torch.zeros(1, 2, 128, 128, device=gpu_device, requires_grad=True) for _ in range(2)]
        for c in range(2):
            lasp_amd.set_sequence_parallel_rank(c)
            (q, k, v), do = _leaves(gpu_device, 1, 2, 100, 128, 128, torch.bfloat16, seed=c)
            outs.append(op(q, k, v, s, *(() if name != "lasp_cache" else (None,)), KV, DKV))
            assert "LaspChunk" in outs[-1].grad_fn.name()
            dos.append(do)
        assert name == "lasp_fuse" or KV._version == 2
        torch.autograd.backward(outs, dos)
        assert name == "lasp_fuse" or DKV._version == 2
        assert KV.grad is None and DKV.grad is None
    finally:
        lasp_amd.destroy_parallel_groups()


@pytest.mark.parametrize("name", ["lasp_fuse", "lasp_fuse_parallel"])
def test_a_checkpointed_chunk_sends_its_state_again(gpu_device, name, monkeypatch):
    """torch.utils.checkpoint ends a recomputed forward from a hook on its last saved tensor.  The chunk has sent its state by
    then, as the Python Function has: the next rank, which recomputes too, waits for it."""
    from lasp_amd.utils import seq_parallel_manager as spm
    from torch.utils.checkpoint import checkpoint

    sent = []
    state_send = spm.state_send
    monkeypatch.setattr(spm, "state_send", lambda t, dst, *a, **k: (sent.append(dst), state_send(t, dst, *a, **k)))
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    op = getattr(lasp_amd, name)
    python = lambda q, k, v, s, KV, DKV: ChunkFunction.apply(q, k, v, s, KV, DKV, True, False, name != "lasp_fuse")
    results = []
    for call, checkpointed in ((op, False), (op, True), (python, True)):
        lasp_amd.destroy_parallel_groups()
        lasp_amd.initialize_lasp(1, 2)
        del sent[:]
        try:
            (q, k, v), do = _leaves(gpu_device, 1, 2, 300, 128, 128, torch.bfloat16)
            KV = torch.zeros(1, 2, 128, 128, device=gpu_device)
            DKV = torch.zeros_like(KV)
            run = lambda q, k, v: call(q, k, v, s, KV, DKV)
            lasp_amd.set_sequence_parallel_rank(0)
            o = checkpoint(run, q, k, v, use_reentrant=False) if checkpointed else run(q, k, v)
            spm.state_send(torch.ones_like(KV), 0, spm.get_sequence_parallel_group(), src=1)
            o.backward(do)
            assert sent == ([1, 0, 1] if checkpointed else [1, 0])
            results.append([o, q.grad, k.grad, v.grad])
        finally:
            lasp_amd.destroy_parallel_groups()
    for r in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], r))


def test_saved_tensor_hooks_see_what_the_node_keeps(gpu_device):
    """Offloaded to the host and back, the node's tensors give the same gradients."""
    (q, k, v), do = _leaves(gpu_device, 1, 2, 3000, 128, 128, torch.bfloat16)
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    want = torch.autograd.grad(lasp_amd.lightning_attn(q, k, v, s), (q, k, v), do)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.to(gpu_device)):
        o = lasp_amd.lightning_attn(q, k, v, s)
    assert len(packed) == 5  # q, k, v, s and the segment states
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, (q, k, v), do), want))


@pytest.mark.parametrize("name", ["lightning_attn", "lasp_fuse", "lasp_fuse_parallel"])
def test_compiled_autograd_runs_the_backward(gpu_device, name):
    """The node has the rules that compiled autograd asks for; a second run of the same shapes is served by what it compiled."""
    from torch._dynamo import compiled_autograd

    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    chunks = 1 if name == "lightning_attn" else 2
    results = []
    for how in ("eager", "compiled", "compiled"):
        lasp_amd.destroy_parallel_groups()
        lasp_amd.initialize_lasp(1, chunks)
        try:
            outs, dos, leaves = [], [], []
            KV = torch.zeros(1, 2, 128, 128, device=gpu_device)
            DKV = torch.zeros_like(KV)
            for c in range(chunks):
                lasp_amd.set_sequence_parallel_rank(c)
                (q, k, v), do = _leaves(gpu_device, 1, 2, 2500, 128, 128, torch.bfloat16, seed=c)
                outs.append(getattr(lasp_amd, name)(q, k, v, s, *(() if chunks == 1 else (KV, DKV))))
                dos.append(do)
                leaves += [q, k, v]
            if how == "eager":
                torch.autograd.backward(outs, dos)
            else:
                with compiled_autograd._enable(torch.compile(backend="eager")):
                    torch.autograd.backward(outs, dos)
            assert not lasp_amd.loopback_pending()
            results.append([*outs, *[t.grad for t in leaves], KV, DKV])
        finally:
            lasp_amd.destroy_parallel_groups()
    for r in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], r))


def test_the_interpreter_lock_is_free_during_a_call(gpu_device):
    """Another thread gets to run while a call allocates and launches.  The lock is not taken from a thread that keeps it here
    (the switch interval is longer than the test), so a tick inside a call means that the call had let go of it."""
    import sys
    import threading
    import time

    (q, k, v), do = _leaves(gpu_device, 1, 16, 65536, 128, 128, torch.bfloat16)
    q, k, v = q.detach(), k.detach(), v.detach()
    s = lasp_amd.build_slope_tensor(16).to(gpu_device)
    ext = _native.ext()
    calls = {
        "attention": lambda: ext.attention(q, k, v, s),
        "chunk_fwd": lambda: ext.chunk_fwd(q, k, v, s, None, None, 0, True),
        "chunk_bwd": lambda: ext.chunk_bwd(q, k, v, s, do, None, None, None, None, 0),
    }
    ticks, done = [], threading.Event()

    def tick():
        while not done.is_set():
            ticks.append(time.perf_counter_ns())
            time.sleep(0)

    interval = sys.getswitchinterval()
    sys.setswitchinterval(600.0)
    other = threading.Thread(target=tick)
    other.start()
    try:
        for name, call in calls.items():
            seen = False
            for _ in range(20):
                torch.cuda.synchronize()
                torch.cuda.empty_cache()  # the call has to ask the driver for its outputs
                begin = time.perf_counter_ns()
                out = call()
                end = time.perf_counter_ns()
                assert out is not None
                del out
                seen = any(begin < t < end for t in ticks[-100000:])
                if seen:
                    break
            assert seen, name
    finally:
        done.set()
        sys.setswitchinterval(interval)
        other.join()


class _NoGradient(torch.autograd.Function):
    """x -> x whose backward has no gradient to give."""

    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


def test_an_output_without_a_gradient_counts_as_one_of_zeros(gpu_device):
    """Also in a chain, where the chunk still passes its neighbours' states on."""
    (q, k, v), do = _leaves(gpu_device, 1, 2, 100, 128, 128, torch.bfloat16)
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    _NoGradient.apply(lasp_amd.lightning_attn(q, k, v, s)).backward(do)
    assert all(torch.equal(t.grad, torch.zeros_like(t)) for t in (q, k, v))
    lasp_amd.destroy_parallel_groups()
    lasp_amd.initialize_lasp(1, 2)
    try:
        grads = []
        for silent in (True, False):
            KV = torch.empty(1, 2, 128, 128, device=gpu_device)
            DKV = torch.empty_like(KV)
            outs, leaves, dos = [], [], []
            for c in range(2):
                lasp_amd.set_sequence_parallel_rank(c)
                (q, k, v), do = _leaves(gpu_device, 1, 2, 100, 128, 128, torch.bfloat16, seed=c)
                o = lasp_amd.lasp_fuse(q, k, v, s, KV, DKV)
                outs.append(_NoGradient.apply(o) if silent and c == 1 else o)
                dos.append(do if c == 0 else torch.zeros_like(do))
                leaves += [q, k, v]
            torch.autograd.backward(outs, dos)
            assert not lasp_amd.loopback_pending()
            grads.append([t.grad for t in leaves])
        assert all(torch.equal(a, b) for a, b in zip(*grads))
    finally:
        lasp_amd.destroy_parallel_groups()


def test_transforms_see_the_operator(gpu_device):
    """Forward-mode differentiation and vmap, for which the operator has no rule, are refused; a traced call replays."""
    (q, k, v), do = _leaves(gpu_device, 1, 2, 70, 128, 128, torch.bfloat16)
    s = lasp_amd.build_slope_tensor(2).to(gpu_device)
    import torch.autograd.forward_ad as fwad

    with fwad.dual_level(), pytest.raises(RuntimeError):
        lasp_amd.lightning_attn(fwad.make_dual(q.detach(), do), k, v, s)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: lasp_amd.lightning_attn(x, k.detach(), v.detach(), s))(q.detach()[None])
    traced = torch.jit.trace(lasp_amd.lightning_attn, (q, k, v, s), check_trace=False)
    q2 = torch.randn_like(q)
    assert torch.equal(traced(q2, k, v, s), lasp_amd.lightning_attn(q2, k, v, s))
