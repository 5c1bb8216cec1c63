"""The eager route of csrc/host.cpp against the Python Functions it takes the place of: the same results bit for bit
over types, sizes, layouts and the ways gradients are asked for, and the same calls refused."""
import pytest
import torch
from torch.autograd import forward_ad

import genbmm_amd as genbmm
from genbmm_amd import _lib, genmul

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
STREAM = (11, 4)


def log_python(a, b):
    return genmul.LogMatMul.apply(a, b, genmul.PATH_AUTO if a.dtype == torch.float32 else genmul.PATH_RECIP)


PAIRS = {"log": (genbmm.logbmm, log_python), "max": (genbmm.maxbmm, genmul.MaxMatMul.apply),
         "prodmax": (genbmm.prodmaxbmm, genmul.ProdMaxMatMul.apply),
         "sample": (lambda a, b: genbmm.samplebmm(a, b, STREAM), lambda a, b: genmul.SampleMatMul.apply(a, b, STREAM))}


def operands(gpu, B, M, K, N, dtype):
    torch.manual_seed(B + M + K + N)
    return [torch.randn(*s).to(gpu, dtype) for s in ((B, M, K), (B, K, N), (B, M, N))]


def native(a, b):
    return _lib.host().plain(a, b)


@pytest.mark.parametrize("op", list(PAIRS))
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,M,K,N", [(1, 1, 1, 1), (3, 7, 5, 9), (2, 130, 97, 101), (0, 3, 4, 5), (2, 3, 0, 5), (2, 0, 4, 5)])
def test_results(gpu, op, dtype, B, M, K, N):
    a, b, g = operands(gpu, B, M, K, N, dtype)
    new, old = PAIRS[op]
    assert native(a, b)
    with torch.no_grad():
        assert torch.equal(new(a, b), old(a, b))
    for needs in ("ab", "a", "b"):
        x, y = a.clone().requires_grad_("a" in needs), b.clone().requires_grad_("b" in needs)
        wrt = [t for t in (x, y) if t.requires_grad]
        # (a gradient of another type: values that the result's type does not hold)
        for grad in (g, torch.randn_like(g, dtype=torch.float64), g.transpose(1, 2).contiguous().transpose(1, 2),
                     g[:1, :1, :1].expand_as(g) if g.numel() else g):
            if op == "prodmax" and M == 0:      # no factors to read the gradient from: refused
                for f in (new, old):
                    with pytest.raises(RuntimeError, match="genbmm_prodmax_bwd"):
                        torch.autograd.grad(f(x, y), wrt, grad)
                continue
            got = torch.autograd.grad(new(x, y), wrt, grad)
            want = torch.autograd.grad(old(x, y), wrt, grad)
            assert all(torch.equal(p, q) for p, q in zip(got, want))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("part", ["ab", "a", "b"])
@pytest.mark.parametrize("B,M,K,N", [(3, 7, 5, 9), (2, 128, 128, 128), (2, 130, 97, 101)])
def test_second_order(gpu, dtype, part, B, M, K, N):
    a, b, g = operands(gpu, B, M, K, N, dtype)
    got = []
    for f in PAIRS["log"]:
        x, y, h = (t.clone().requires_grad_() for t in (a, b, g))
        first = torch.autograd.grad(f(x, y), (x, y), h, create_graph=True)
        asked = [first["ab".index(c)] for c in part]
        got.append(torch.autograd.grad(asked, (x, y, h), [torch.cos(t).detach() for t in asked]))
    assert all(torch.equal(p, q) for p, q in zip(*got))


@pytest.mark.parametrize("op", list(PAIRS))
def test_without_the_extension(gpu, op, monkeypatch):
    """Where it was not built for this torch the Python Functions carry the call."""
    a, b, g = operands(gpu, 2, 40, 33, 50, torch.float32)

    def run():
        x, y = a.clone().requires_grad_(), b.clone().requires_grad_()
        out = PAIRS[op][0](x, y)
        return type(out.grad_fn).__name__, [out.detach()] + list(torch.autograd.grad(out, (x, y), g))

    name, want = run()
    monkeypatch.setattr(_lib, "_host", False)
    python, got = run()
    assert "MatMulBackward" not in name
    assert "MatMulBackward" in python
    assert all(torch.equal(p, q) for p, q in zip(got, want))


def test_what_takes_the_route(gpu):
    a, b, _ = operands(gpu, 2, 6, 5, 7, torch.float32)
    assert native(a, b) and native(torch.nn.Parameter(a), b)
    wide = operands(gpu, 2, 6, 4096, 7, torch.float32)

    class Sub(torch.Tensor):
        pass

    for x, y in ((a.cpu(), b.cpu()), (a.double(), b.double()), (a, b.half()), (a[0], b[0]), (a, b[:1]), (a, b[:, :4]),
                 (a.transpose(1, 2).contiguous().transpose(1, 2), b), (a.as_subclass(Sub), b), (wide[0], wide[1]),
                 (torch.complex(a, a).conj().imag, b), (a.int(), b.int())):
        assert not native(x, y)


def refusal(f, *args):
    """(type, message) of what f raises."""
    with pytest.raises(Exception) as e:
        f(*args)
    return e.type, str(e.value)


def same_refusal(attempt, fs, kind, words):
    """Every f of fs refused by `attempt`, with one type and one message that says `words`."""
    got = [refusal(attempt, f) for f in fs]
    assert got[0][0] is kind and words in got[0][1] and all(x == got[0] for x in got), got


@pytest.mark.parametrize("op", list(PAIRS))
def test_refused_as_before(gpu, op):
    a, b, g = operands(gpu, 2, 6, 5, 7, torch.float32)

    def forward_mode(f, which=0):
        with forward_ad.dual_level():
            x = [a, b]
            x[which] = forward_ad.make_dual(x[which], x[which])
            f(*x)

    def batched(f):
        x = a.clone().requires_grad_()
        torch.autograd.grad(f(x, b), x, torch.stack([g, g]), is_grads_batched=True)

    def twice(f):
        x = a.clone().requires_grad_()
        out = f(x * 1, b)
        torch.autograd.grad(out, x, g)
        torch.autograd.grad(out, x, g)

    def changed(f):
        x = (a * 1).requires_grad_()
        out = f(x, b)
        with torch.no_grad():
            x.add_(1)
        torch.autograd.grad(out, x, g)

    def tangent(f):
        x = a.clone().requires_grad_()
        out = f(x, b)
        with forward_ad.dual_level():
            torch.autograd.grad(out, x, forward_ad.make_dual(g, g))

    fs = PAIRS[op]
    same_refusal(forward_mode, fs, NotImplementedError, "jvp")
    same_refusal(lambda f: forward_mode(f, 1), fs, NotImplementedError, "jvp")
    same_refusal(batched, fs, RuntimeError, "doesn't have storage")
    same_refusal(lambda f: torch.func.vmap(f)(torch.stack([a, a]), torch.stack([b, b])), fs, RuntimeError, "setup_context")
    same_refusal(lambda f: torch.func.grad(lambda t: f(t, b).sum())(a), fs, RuntimeError, "setup_context")
    same_refusal(twice, fs, RuntimeError, "a second time")
    if op == "log":
        same_refusal(changed, fs, RuntimeError, "modified by an inplace operation")    # saved for the backward
        same_refusal(tangent, fs, NotImplementedError, "jvp")


@pytest.mark.parametrize("op", list(PAIRS))
def test_hooks_traces_streams_threads(gpu, op):
    import threading

    a, b, g = operands(gpu, 2, 40, 33, 50, torch.float32)
    new, old = PAIRS[op]
    x = a.clone().requires_grad_()
    want = torch.autograd.grad(old(x, b), x, g)[0]
    with torch.autograd.graph.save_on_cpu():
        out = new(x, b)
    assert torch.equal(torch.autograd.grad(out, x, g)[0], want)
    traced = torch.jit.trace(new, (a, b), check_trace=False)          # a Python Function records itself; a native one would not
    assert "^" in str(traced.graph) and torch.equal(traced(a, b), old(a, b))
    got = {}

    def work(i):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            y = a.clone().requires_grad_()
            got[i] = torch.autograd.grad(new(y, b), y, g)[0]
        s.synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(torch.equal(got[i], want) for i in range(4))


@pytest.mark.parametrize("op", list(PAIRS))
@pytest.mark.parametrize("unpack", [lambda t: t.cpu(), lambda t: t.double(), lambda t: t[..., :1],
                                    lambda t: torch.stack([t, t], -1)[..., 0]])
def test_what_a_saved_tensor_hook_may_not_return(gpu, op, unpack):
    a, b, g = operands(gpu, 2, 6, 5, 7, torch.float32)
    x = a.clone().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        out = PAIRS[op][0](x, b)
    with pytest.raises(RuntimeError, match="expected|must be"):
        torch.autograd.grad(out, x, g)
