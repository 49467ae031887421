"""QTensor.fwd through the native host path (candle_amd/csrc/cq_host.cpp) and through the Python one: the same results, refusals and side effects."""
import threading

import pytest
import torch

from candle_amd import _lib
from candle_amd import quantized as q
from candle_amd.quantized import GgmlDType, QMatMul, QTensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
N, K = 96, 512


def weight(fmt=GgmlDType.Q4K):
    g = torch.Generator(device=DEV).manual_seed(1)
    return QTensor.quantize(torch.randn(N, K, generator=g, device=DEV), fmt)


def both(call, monkeypatch):
    """What `call` returns or raises on the native path and on the Python path."""
    out = []
    for native in (True, False):
        with monkeypatch.context() as m:
            if not native:
                m.setattr(_lib, "qmatmul", None)
            try:
                out.append(call())
            except Exception as e:
                out.append((type(e), str(e)))
    return out


@pytest.mark.parametrize("fmt", [GgmlDType.Q8_0, GgmlDType.Q4K, GgmlDType.Q3K, GgmlDType.Q5_1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_same_results(fmt, dtype, monkeypatch):
    w = weight(fmt)
    w.fwd(torch.ones(64, K, device=DEV))                     # sizes the stream's workspace
    for shape in ((1, K), (16, K), (1, 1, K), (2, 3, K), (3, 1, 7, K)):
        x = torch.randn(shape, device=DEV).to(dtype)
        assert _lib.qmatmul(x, w.storage._data, w.storage._dtype, w._shape, q._workspaces) is not None
        a, b = both(lambda: w.fwd(x), monkeypatch)
        assert a.shape == b.shape == (*shape[:-1], N) and a.dtype == dtype and torch.equal(a, b), shape
        offset = torch.randn(x.numel() + 16, device=DEV).to(dtype)[16:].view(shape)        # not where an allocation begins
        assert torch.equal(*both(lambda: w.fwd(offset), monkeypatch)), shape
    y = w.fwd(torch.randn(2, K, device=DEV, requires_grad=True))
    assert not y.requires_grad and QMatMul.from_qtensor(w).forward(x).dtype == dtype


def test_same_refusals(monkeypatch):
    w, x = weight(), torch.randn(4, K, device=DEV)
    w.fwd(x)
    stored = weight(GgmlDType.Q8K)
    calls = [lambda: w.fwd(x.cpu()), lambda: w.fwd(x[0]), lambda: w.fwd(x[:, :256]), lambda: w.fwd(torch.randn(K, 4, device=DEV).t()), lambda: w.fwd(x.double()),
             lambda: w.fwd(torch.randn(4, 2 * K, device=DEV)), lambda: stored.fwd(x), lambda: w.fwd(torch.randn(4 * K + 1, device=DEV)[1:].view(4, K)),
             lambda: torch.vmap(w.fwd)(x.view(2, 2, K)), lambda: w.fwd(x.to_sparse())]
    for i, call in enumerate(calls):
        a, b = both(call, monkeypatch)
        assert isinstance(a, tuple) and a == b, (i, a, b)
    for empty in ((0, K), (2, 0, K)):
        a, b = both(lambda: w.fwd(torch.empty(empty, device=DEV)), monkeypatch)
        assert a.shape == b.shape == (*empty[:-1], N)


def test_the_python_path_takes_what_is_not_ordinary():
    """A subclass, a function mode, a new stream, a workspace that is too small or locked: left alone, and the call still returns."""
    w, x = weight(), torch.randn(4, K, device=DEV)
    want = w.fwd(x)
    native = lambda t: _lib.qmatmul(t, w.storage._data, w.storage._dtype, w._shape, q._workspaces)
    assert torch.equal(native(x), want)

    class Sub(torch.Tensor):
        pass

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert native(x.as_subclass(Sub)) is None and native(x.cpu()) is None
    with Mode():
        assert native(x) is None and torch.equal(w.fwd(x), want)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        assert native(x) is None                             # no workspace of this stream yet
        a = w.fwd(x)
        b = native(x)                                        # now there is one
    s.synchronize()
    assert torch.equal(a, want) and torch.equal(b, want)
    slot = q._workspaces[(0, torch.cuda.current_stream().cuda_stream)]
    big = torch.randn(2048, K, device=DEV)
    if _lib.lib().cq_qmatmul_workspace_bytes(12, 2048, K, N) > slot.buf.numel():
        assert native(big) is None
    got = []
    with slot.lock:
        assert native(x) is None                             # another call is being enqueued
        t = threading.Thread(target=lambda: got.append(w.fwd(x)))
        t.start()
        t.join(0.2)
        assert t.is_alive() and not got                      # ... and this one waits for it
    t.join(10)
    assert torch.equal(got[0], want) and not slot.lock.locked()


@pytest.mark.parametrize("fmt", [GgmlDType.Q8_0, GgmlDType.Q4K])
def test_workspace_of_just_enough_bytes(fmt):
    """A buffer of the stream that is missing or a byte too small is left to Python, unlocked; one of exactly the bytes that the library asks for is taken, and nothing
    behind it is written."""
    w, x = weight(fmt), torch.randn(200, K, device=DEV)
    want, need = w.fwd(x), _lib.lib().cq_qmatmul_workspace_bytes(int(fmt), 200, K, N)
    assert need > 1
    slot, memory = q._Workspace(), torch.full((need + 4096,), 255, dtype=torch.uint8, device=DEV)
    mine = {(0, torch.cuda.current_stream().cuda_stream): slot}
    native = lambda: _lib.qmatmul(x, w.storage._data, w.storage._dtype, w._shape, mine)
    for buf in (None, memory[:need - 1], memory[:0]):
        slot.buf = buf
        assert native() is None and not slot.lock.locked()
    slot.buf = memory[:need]
    assert torch.equal(native(), want) and not slot.lock.locked() and bool((memory[need:] == 255).all())
    assert _lib.qmatmul(x, w.storage._data, w.storage._dtype, w._shape, {}) is None


def test_threads_share_a_stream():
    """Several threads on one stream: calls of more than one launch do not get between each other's."""
    w = weight()
    xs = [torch.randn(24, K, device=DEV) for _ in range(4)]
    want = [w.fwd(x) for x in xs]
    bad = []

    def run(i):
        for _ in range(50):
            if not torch.equal(w.fwd(xs[i]), want[i]):
                bad.append(i)
    ts = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_captured_calls_replay():
    w, x = weight(), torch.randn(24, K, device=DEV)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        w.fwd(x)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            y = w.fwd(x)
    for seed in range(3):
        x.copy_(torch.randn(24, K, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, w.fwd(x)), seed
