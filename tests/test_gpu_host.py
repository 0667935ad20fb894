"""The host module's calls (one per layer call) against the Python autograd
functions they stand for: bit for bit over the forms both take, and what autograd
promises of a node kept: hooks on saved tensors, version checks, partial
gradients, one differentiation; transforms, tracing and forward mode stay with
the Python functions."""
import sys
import threading
import time

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.checkpoint import checkpoint

import moc
from moc import MoC, api
from moc import _lib
from tests._parity import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32


def _layer(dtype, K=16, S=4, D=130, Z=128, act="silu", route="softmax"):
    torch.manual_seed(K + S)
    m = MoC(D, Z, S, K, activation=act, init_std=0.3, router_activation=route).to(DEV, dtype)
    with torch.no_grad():
        m.router.copy_(randn(gen(K), K, Z, scale=0.05))
    return m


def _python(m, x, z, cu=None, longest=None):
    return api._MoCLayerFunction.apply(x, z, m.router, m.conv_bases, m.activation,
                                       m.router_activation, cu, longest, None, None)


FORMS = {
    "plain": lambda t: t,
    "strided": lambda t: torch.cat((t, t), -1)[..., :t.shape[-1]],
    "offset": lambda t: torch.cat((t.flatten()[:2], t.flatten()))[2:].view(t.shape),
    "transposed": lambda t: t.transpose(0, 1).contiguous().transpose(0, 1),
}
DYS = {
    "rows": lambda y, g: randn(g, *y.shape).to(y),
    "one": lambda y, g: randn(g, 1).to(y).expand_as(y),
    "row": lambda y, g: randn(g, y.shape[-1]).to(y).expand_as(y),
    "strided": lambda y, g: randn(g, *y.shape[:-1], 2 * y.shape[-1]).to(y)[..., ::2],
}


@pytest.mark.parametrize("dtype,K,S,route", [(BF, 16, 4, "softmax"), (BF, 12, 3, "exp"), (F32, 16, 4, "exp"),
                                             (F32, 4, 2, "softmax"), (BF, 32, 8, "softmax")])
@pytest.mark.parametrize("form", list(FORMS))
def test_layer_bit_for_bit(dtype, K, S, route, form):
    m, g = _layer(dtype, K, S, route=route), gen(3)
    x, z = (FORMS[form](randn(g, 2, 37, n).to(DEV, dtype)).detach().requires_grad_() for n in (130, 128))
    wrt = [x, z, m.router, m.conv_bases]
    for dy in DYS.values():
        y, state = m(x, z)
        ref = _python(m, x, z)
        assert state is None and type(y.grad_fn).__name__ == "_MoCLayerFunctionBackward"
        d = dy(y, gen(5))
        assert torch.equal(y, ref)
        for a, b in zip(torch.autograd.grad(y, wrt, d), torch.autograd.grad(ref, wrt, d)):
            assert a.dtype == b.dtype and torch.equal(a, b)
    with torch.no_grad():
        y, state = m(x, z, output_final_state=True)
        assert torch.equal(y, ref) and torch.equal(state, api._final_state(x, None, S))


@pytest.mark.parametrize("cu_dt", [torch.int32, torch.int64])
@pytest.mark.parametrize("lead", [False, True])
def test_packed_and_functional_bit_for_bit(cu_dt, lead):
    m, g = _layer(BF), gen(4)
    lengths = [1, 30, 7, 64]
    N = sum(lengths)
    cu = torch.tensor([0, *lengths]).cumsum(0).to(DEV, cu_dt)
    x, z, a = (randn(g, N, n).to(DEV, BF).requires_grad_() for n in (130, 128, 16))
    dy = randn(g, N, 130).to(DEV, BF)
    up = (lambda t: t[None]) if lead else (lambda t: t)
    y = up(m(up(x), up(z), cu_seqlens=cu, max_seqlen=64)[0]) if not lead else m(x[None], z[None], cu_seqlens=cu,
                                                                                max_seqlen=64)[0]
    ref = up(_python(m, x, z, cu, 64))
    got = torch.autograd.grad(y, [x, z, m.router, m.conv_bases], up(dy))
    want = torch.autograd.grad(ref, [x, z, m.router, m.conv_bases], up(dy))
    assert torch.equal(y, ref) and all(torch.equal(p, q) for p, q in zip(got, want))
    y = moc.moc_triton(up(x), up(a), m.conv_bases, activation="silu", cu_seqlens=cu, max_seqlen=64)[0]
    ref = up(api._MoCFunction.apply(x, a, m.conv_bases, "silu", cu, 64, None, None))
    got = torch.autograd.grad(y, [x, a, m.conv_bases], up(dy))
    want = torch.autograd.grad(ref, [x, a, m.conv_bases], up(dy))
    assert torch.equal(y, ref) and all(torch.equal(p, q) for p, q in zip(got, want))


def test_partial_gradients_and_frozen_inputs():
    m, g = _layer(BF), gen(6)
    x, z = randn(g, 2, 20, 130).to(DEV, BF), randn(g, 2, 20, 128).to(DEV, BF)
    dy = randn(g, 2, 20, 130).to(DEV, BF)
    zz = z.clone().requires_grad_()
    full = torch.autograd.grad(_python(m, x, zz), [zz, m.router, m.conv_bases], dy)
    for i, t in enumerate([zz, m.router, m.conv_bases]):
        assert torch.equal(torch.autograd.grad(m(x, zz)[0], [t], dy)[0], full[i])
    m.requires_grad_(False)
    y, _ = m(x, zz)
    assert torch.equal(torch.autograd.grad(y, [zz], dy)[0], full[0])
    assert not m(x, z)[0].requires_grad


def test_autograd_promises():
    m, g = _layer(BF), gen(7)
    x, z = (randn(g, 2, 20, n).to(DEV, BF).requires_grad_() for n in (130, 128))
    # one differentiation
    y, _ = m(x, z)
    dx, = torch.autograd.grad(y, [x], torch.ones_like(y).requires_grad_(), create_graph=True)
    with pytest.raises(RuntimeError, match="differentiate twice"):
        dx.sum().backward()
    # saved-tensor hooks see every saved tensor and may move it
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1],
                                                  lambda t: t.to(DEV)):
        y, _ = m(x, z)
    assert len(seen) >= 5
    want = torch.autograd.grad(_python(m, x, z), [x, z], torch.ones_like(y))
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, [x, z], torch.ones_like(y)), want))
    # a graph is used once, and its saved tensors are not written to in between
    y, _ = m(x, z)
    torch.autograd.grad(y, [x], torch.ones_like(y))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, [x], torch.ones_like(y))
    y, _ = m(x, z)
    with torch.no_grad():
        z.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(y, [x], torch.ones_like(y))


@pytest.mark.parametrize("dtype", [BF, F32])
def test_checkpointed_layer(dtype):
    """A checkpoint's saved tensors are unpacked once: the nodes of the host module
    and of the Python functions."""
    m, g = _layer(dtype), gen(13)
    x, z = (randn(g, 2, 20, n).to(DEV, dtype).requires_grad_() for n in (130, 128))
    cu = torch.tensor([0, 20, 40], dtype=torch.int32)
    xp, zp = x.detach().flatten(0, 1).requires_grad_(), z.detach().flatten(0, 1).requires_grad_()
    dy = randn(g, 2, 20, 130).to(DEV, dtype)
    want = torch.autograd.grad(m(x, z)[0], [x, z], dy)
    calls = {"host": (lambda a, b: m(a, b)[0], x, z), "python": (lambda a, b: _python(m, a, b), x, z),
             "offsets on the host": (lambda a, b: m(a, b, cu_seqlens=cu.to(DEV), max_seqlen=20, cu_seqlens_cpu=cu)[0],
                                     xp, zp),
             "functional": (lambda a, b: moc.moc_triton(a, b[..., :16].softmax(-1), m.conv_bases)[0], x, z)}
    for name, (f, a, b) in calls.items():
        d = dy.view(a.shape)
        got = torch.autograd.grad(checkpoint(f, a, b, use_reentrant=False), [a, b], d)
        ref = torch.autograd.grad(f(a, b), [a, b], d)
        assert all(torch.equal(u, v) for u, v in zip(got, ref)), name
        if name != "functional":
            assert all(torch.equal(u.view_as(v), v) for u, v in zip(got, want)), name


def test_watched_calls_stay_with_python():
    m, g = _layer(BF), gen(8)
    x, z = (randn(g, 2, 20, n).to(DEV, BF) for n in (130, 128))
    H = _lib.host()
    args = (m.router, m.conv_bases, 1, 1, None)
    assert H.layer(x, z, *args) is not None
    with torch.autograd.forward_ad.dual_level():
        assert H.layer(torch.autograd.forward_ad.make_dual(x, x), z, *args) is None
    inside = []
    torch.func.vmap(lambda t: (inside.append(H.layer(t[None], z[:1], *args)), t)[1])(x)
    torch.func.grad(lambda t: (inside.append(H.layer(t, z, *args)), t.sum())[1])(x)
    torch.jit.trace(lambda t: (inside.append(H.layer(t, z, *args)), t)[1], (x,), check_trace=False)
    class Seen(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, call, kwargs=None):
            self.ops += 1
            return func(*call, **(kwargs or {}))

    with Seen() as seen:
        inside.append(H.layer(x, z, *args))
        y, _ = m(x, z)
    assert seen.ops > 0 and torch.equal(y, m(x, z)[0])
    assert len(inside) == 4 and all(v is None for v in inside)
    assert H.layer(x.cpu(), z, *args) is None and H.layer(x.half(), z, *args) is None
    assert H.layer(x[:, :0], z[:, :0], *args) is None and H.layer(x, z[:, :5], *args) is None


class Tagged(torch.Tensor):
    """A subclass without __torch_dispatch__: nothing in its dispatch keys."""


def test_subclasses_keep_their_type():
    m, g = _layer(BF), gen(11)
    x, z = randn(g, 2, 20, 130).to(DEV, BF), randn(g, 2, 20, 128).to(DEV, BF)
    a = randn(g, 2, 20, 16).to(DEV, BF)
    tx, H = x.as_subclass(Tagged), _lib.host()
    assert H.layer(tx, z, m.router, m.conv_bases, 1, 1, None) is None
    assert H.layer(x, z.as_subclass(Tagged), m.router, m.conv_bases, 1, 1, None) is None
    assert H.func(x, a.as_subclass(Tagged), m.conv_bases, 1, None) is None
    assert H.stateful(x, z, m.router.as_subclass(Tagged), m.conv_bases, None, 1, 1, True) is None
    for grad in (True, False):
        with torch.set_grad_enabled(grad):
            for got, want in ((m(tx, z)[0], m(x, z)[0]),
                              (moc.moc_triton(tx, a, m.conv_bases)[0], moc.moc_triton(x, a, m.conv_bases)[0])):
                assert type(got) is Tagged and type(want) is torch.Tensor
                assert torch.equal(got.as_subclass(torch.Tensor), want)
    with torch.no_grad():
        y, cache = m.step(tx[:, :1], z[:, :1], cache=torch.zeros(2, 130, 4, device=DEV, dtype=BF))
        assert type(y) is Tagged
    # what is no tensor gets the Python functions' error, not an argument error
    with pytest.raises(AttributeError):
        moc.moc_triton(x[0], a[0], m.conv_bases, cu_seqlens=[0, 20], max_seqlen=20)


@pytest.mark.parametrize("dtype", [BF, F32])
def test_stateful_bit_for_bit(dtype):
    m, g = _layer(dtype), gen(9)
    x, z = randn(g, 3, 9, 130).to(DEV, dtype), randn(g, 3, 9, 128).to(DEV, dtype)
    c0 = randn(g, 3, 130, 4).to(DEV, dtype)
    with torch.no_grad():
        y, state = m(x, z, cache=c0, output_final_state=True)
        w = api.ops.router_forward(z, m.router, routing=1)
        ref, fin = api.ops.launch_forward_prefill(x, w, m.conv_bases, c0, activation_flag=1, final_state=True,
                                                  routing=3)
        assert torch.equal(y, ref) and torch.equal(state, fin)
        assert m(x, z, cache=c0)[1] is None
    # a step writes the cache it is given and returns it, also with gradients on
    for cache in (c0.clone(), c0.transpose(1, 2).contiguous().transpose(1, 2)):
        one, two = cache.clone(memory_format=torch.preserve_format), cache
        logits = api.ops.router_forward(z[:, :1], m.router)
        ref = api._step(x[:, :1], logits, m.conv_bases, one, "silu", "softmax")
        y, out = m.step(x[:, :1], z[:, :1], cache=two, output_final_state=True)
        assert out is two and torch.equal(one, two)
        if dtype == F32:  # the same two launches
            assert torch.equal(y, ref)
        else:  # the one-launch step rounds its weights as another kernel does
            assert (y - ref).float().abs().max() <= 2.0 ** -7 * ref.float().abs().max()


@pytest.mark.parametrize("dtype,B,T,D,K,S,one", [
    (BF, 2, 2, 130, 16, 4, False), (BF, 2, 3, 130, 16, 4, True), (BF, 3, 6, 130, 32, 8, False),
    (F32, 2, 7, 130, 16, 8, True), (F32, 1, 1024, 4096, 16, 4, True), (F32, 1, 1025, 4096, 16, 4, False),
    (F32, 1, 1025, 4096, 16, 3, True), (F32, 2, 600, 4098, 20, 3, False), (BF, 1, 1025, 4096, 32, 8, True)])
def test_prompt_state(dtype, B, T, D, K, S, one):
    """A prompt's state from the forward launch, or the plain forward's rows where
    those are cheaper: the same y and state."""
    m, g = _layer(dtype, K, S, D), gen(T)
    x, z = randn(g, B, T, D).to(DEV, dtype), randn(g, B, T, 128).to(DEV, dtype)
    with torch.no_grad():
        out = _lib.host().stateful(x, z, m.router, m.conv_bases, None, 1, 1, True)
        assert (out is not None) == one
        y, state = m(x, z, output_final_state=True)
        w = api.ops.router_forward(z, m.router, routing=1)
        ref = api.ops.launch_forward(x, w, m.conv_bases, activation_flag=1, routing=3)
    assert torch.equal(y, ref) and torch.equal(state, api._final_state(x, None, S))


def _step(m, x, z, dy):
    y, _ = m(x, z)
    return [y.detach(), *torch.autograd.grad(y, [x, z, m.router, m.conv_bases], dy)]


@pytest.mark.parametrize("dtype", [BF, F32])
def test_streams_and_threads(dtype):
    """Forward and backward of four threads at once, each on a stream of its own."""
    m, g = _layer(dtype), gen(10)
    sets = [tuple(randn(g, 2, 300, n).to(DEV, dtype) for n in (130, 128, 130)) for _ in range(4)]
    sets = [(x.requires_grad_(), z.requires_grad_(), dy) for x, z, dy in sets]
    want = [_step(m, *s) for s in sets]
    torch.cuda.synchronize()
    got = [None] * 4
    together = threading.Barrier(4)

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            together.wait()
            for _ in range(20):
                got[i] = _step(m, *sets[i])
        s.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(torch.equal(u, v) for a, b in zip(got, want) for u, v in zip(a, b))


def test_other_threads_run_during_a_call():
    """The calls run without the interpreter lock: with no switch forced (an
    interval of 100 s), another thread counts on only while a call is inside."""
    m, g = _layer(BF), gen(12)
    x, z = randn(g, 2, 2000, 130).to(DEV, BF), randn(g, 2, 2000, 128).to(DEV, BF)
    w = randn(g, 2, 2000, 16).to(DEV, BF)
    c0 = randn(g, 2, 130, 4).to(DEV, BF)
    H = _lib.host()
    calls = {"layer": lambda: H.layer(x, z, m.router, m.conv_bases, 1, 1, None),
             "func": lambda: H.func(x, w, m.conv_bases, 1, None),
             "stateful": lambda: H.stateful(x, z, m.router, m.conv_bases, c0, 1, 1, True)}
    count, stop = [0], []

    def other():
        while not stop:
            count[0] += 1
            time.sleep(0)  # gives the lock up and waits for it again

    before = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    try:
        sys.setswitchinterval(100.0)
        thread.start()
        for name, call in calls.items():
            ran = 0
            for _ in range(30):
                torch.cuda.empty_cache()  # the call allocates from the device: long enough to switch
                at = count[0]
                with torch.set_grad_enabled(name != "stateful"):
                    out = call()
                ran += count[0] - at
                assert out is not None
                del out
            assert ran > 0, name
    finally:
        stop.append(1)
        sys.setswitchinterval(before)
        thread.join()
