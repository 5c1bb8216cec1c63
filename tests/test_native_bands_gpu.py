"""The eager route of csrc/host.cpp for banded products against the Python Functions it takes the place of: the same
results bit for bit over types, sizes and the ways gradients are asked for, and the same calls refused."""
import threading

import pytest
import torch
from torch.autograd import forward_ad

import genbmm_amd as genbmm
from genbmm_amd import _lib, sparse

pytestmark = pytest.mark.gpu

BAND = (2, 3, 4, 1)
OPS = {"band_mul": ("multiply", sparse.bandedbmm), "band_log": ("multiply_log", sparse.bandedlogbmm),
       "band_max": ("multiply_max", sparse.bandedmaxbmm)}


def pair(op, band=BAND):
    """(by the class's method, by the Python Function)"""
    method, fn = OPS[op]
    a_lu, a_ld, b_lu, b_ld = band

    def new(a, b):
        return getattr(genbmm.BandedMatrix(a, a_lu, a_ld), method)(genbmm.BandedMatrix(b, b_lu, b_ld)).data

    return new, lambda a, b: fn(_lib.dense(a), a_lu, a_ld, _lib.dense(b), b_lu, b_ld, a_lu + b_ld, a_ld + b_lu)


def operands(gpu, B, n, dtype=torch.float32, band=BAND):
    torch.manual_seed(B + n)
    wa, wb = band[0] + band[1] + 1, band[2] + band[3] + 1
    return [torch.randn(B, n, w).to(gpu, dtype) for w in (wa, wb, wa + wb - 1)]


def native(a, b, band=BAND, op="band_mul"):
    a_lu, a_ld, b_lu, b_ld = band
    return getattr(_lib.host(), op)(a, a_lu, a_ld, b, b_lu, b_ld) is not None


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,n,band", [(1, 1, (0, 0, 0, 0)), (3, 17, BAND), (2, 130, (32, 32, 20, 33)), (0, 4, BAND), (2, 0, BAND),
                                      (1, 20, (70, 70, 5, 5))])
def test_results(gpu, op, dtype, B, n, band):
    a, b, g = operands(gpu, B, n, dtype, band)
    new, old = pair(op, band)
    assert native(a, b, band, op)
    with torch.no_grad():
        assert torch.equal(new(a, b), old(a, b))
    for needs in ("ab", "a", "b"):
        x, y = a.clone().requires_grad_("a" in needs), b.clone().requires_grad_("b" in needs)
        wrt = [t for t in (x, y) if t.requires_grad]
        for grad in (g, torch.randn_like(g, dtype=torch.float64), g.transpose(1, 2).contiguous().transpose(1, 2),
                     g[:1, :1, :1].expand_as(g) if g.numel() else g):
            got, want = (torch.autograd.grad(f(x, y), wrt, grad) for f in (new, old))
            assert all(torch.equal(p, q) for p, q in zip(got, want))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("part", ["ab", "a", "b"])
def test_second_order(gpu, dtype, part):
    a, b, g = operands(gpu, 2, 40, dtype)
    got = []
    for f in pair("band_log"):
        x, y, h = (t.clone().requires_grad_() for t in (a, b, g))
        first = torch.autograd.grad(f(x, y), (x, y), h, create_graph=True)
        asked = [first["ab".index(c)] for c in part]
        got.append(torch.autograd.grad(asked, (x, y, h), [torch.cos(t).detach() for t in asked]))
    assert all(torch.equal(p, q) for p, q in zip(*got))


@pytest.mark.parametrize("op", list(OPS))
def test_without_the_extension(gpu, op, monkeypatch):
    a, b, g = operands(gpu, 2, 40)

    def run():
        x, y = a.clone().requires_grad_(), b.clone().requires_grad_()
        out = pair(op)[0](x, y)
        return type(out.grad_fn).__name__, [out.detach()] + list(torch.autograd.grad(out, (x, y), g))

    name, want = run()
    monkeypatch.setattr(_lib, "_host", False)
    python, got = run()
    assert "MulBackward" not in name and "MulBackward" in python
    assert all(torch.equal(p, q) for p, q in zip(got, want))


def test_what_takes_the_route(gpu):
    a, b, _ = operands(gpu, 2, 6)
    assert native(a, b) and native(torch.nn.Parameter(a), b)

    class Sub(torch.Tensor):
        pass

    for x, y, band in ((a.cpu(), b.cpu(), BAND), (a.double(), b.double(), BAND), (a, b.half(), BAND), (a[0], b[0], BAND), (a, b[:1], BAND),
                       (a, b[:, :4], BAND), (a, b, (3, 3, 4, 1)), (a, b, (-1, 6, 4, 1)), (a.as_subclass(Sub), b, BAND), (a.int(), b.int(), BAND),
                       (a.transpose(1, 2).contiguous().transpose(1, 2), b, BAND), (torch.complex(a, a).conj().imag, b, BAND)):
        assert not native(x, y, band)
    wide = operands(gpu, 2, 6, band=(80, 80, 70, 70))       # sparse._dense_pays may take these
    assert not native(*wide[:2], (80, 80, 70, 70)) and native(*wide[:2], (80, 80, 70, 70), "band_max")


def refusal(f, *args):
    with pytest.raises(Exception) as e:
        f(*args)
    return e.type, str(e.value)


def same_refusal(attempt, fs, kind, words):
    got = [refusal(attempt, f) for f in fs]
    assert got[0][0] is kind and words in got[0][1] and all(x == got[0] for x in got), got


@pytest.mark.parametrize("op", list(OPS))
def test_refused_as_before(gpu, op):
    a, b, g = operands(gpu, 2, 6)

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

    fs = pair(op)
    same_refusal(forward_mode, fs, NotImplementedError, "jvp")
    same_refusal(lambda f: forward_mode(f, 1), fs, NotImplementedError, "jvp")
    same_refusal(batched, fs, RuntimeError, "doesn't have storage")
    same_refusal(lambda f: torch.func.vmap(f)(torch.stack([a, a]), torch.stack([b, b])), fs, RuntimeError, "setup_context")
    same_refusal(lambda f: torch.func.grad(lambda t: f(t, b).sum())(a), fs, RuntimeError, "setup_context")
    same_refusal(twice, fs, RuntimeError, "a second time")
    same_refusal(changed, fs, RuntimeError, "modified by an inplace operation")
    if op == "band_log":
        same_refusal(tangent, fs, NotImplementedError, "jvp")


@pytest.mark.parametrize("op", list(OPS))
def test_hooks_traces_streams_threads(gpu, op):
    a, b, g = operands(gpu, 2, 40)
    new, old = pair(op)
    x = a.clone().requires_grad_()
    want = torch.autograd.grad(old(x, b), x, g)[0]
    with torch.autograd.graph.save_on_cpu():
        out = new(x, b)
    assert torch.equal(torch.autograd.grad(out, x, g)[0], want)
    traced = torch.jit.trace(new, (a, b), check_trace=False)
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


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("unpack", [lambda t: t.cpu(), lambda t: t.double(), lambda t: t[..., :1],
                                    lambda t: torch.stack([t, t], -1)[..., 0]])
def test_what_a_saved_tensor_hook_may_not_return(gpu, op, unpack):
    a, b, g = operands(gpu, 2, 6)
    x = a.clone().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        out = pair(op)[0](x, b)
    with pytest.raises(RuntimeError, match="expected|must be"):
        torch.autograd.grad(out, x, g)
