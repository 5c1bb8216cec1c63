"""Operands and gradients that carry torch's lazy negative bit - the imaginary part of a conjugate, whose memory
holds the values with the other sign - against the same values written out: equal bit for bit."""
import pytest
import torch

import genbmm_amd as genbmm
from genbmm_amd import _lib, genmul, ops, sparse

pytestmark = pytest.mark.gpu

STREAM = (11, 4)


@pytest.fixture(autouse=True, params=[True, False], ids=["extension", "python"])
def extension(request, monkeypatch):
    """With the host extension, whose checks look at the bit as well, and without it."""
    assert _lib.host() is not None
    if not request.param:
        monkeypatch.setattr(_lib, "_host", False)


def lazy(t):
    """t's values, contiguous, with the negative bit set: the storage holds -t."""
    x = torch._neg_view((-t).contiguous())
    assert x.is_neg() and x.is_contiguous() and torch.equal(x, t)
    return x


def same(got, want):
    assert len(got) == len(want) and all(torch.equal(p, q) for p, q in zip(got, want))


def first_order(f, ts, g):
    xs = [t.clone().requires_grad_() for t in ts]
    out = f(*xs)
    return [out.detach()] + list(torch.autograd.grad(out, xs, g))


DENSE = {"log": genbmm.logbmm, "max": genbmm.maxbmm, "prodmax": genbmm.prodmaxbmm,
         "sample": lambda a, b: genbmm.samplebmm(a, b, STREAM)}
DTYPES = [torch.float32, torch.float64, torch.float16, torch.bfloat16]


@pytest.mark.parametrize("op", list(DENSE))
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,M,K,N", [(1, 1, 1, 1), (2, 7, 5, 9), (1, 3, 4100, 2)])
def test_dense(gpu, op, dtype, B, M, K, N):
    torch.manual_seed(B + M + K + N)
    a, b, g = (torch.randn(*s).to(gpu, dtype) for s in ((B, M, K), (B, K, N), (B, M, N)))
    f = DENSE[op]
    want = first_order(f, (a, b), g)
    same(first_order(f, (a, b), lazy(g)), want)
    for x, y in ((lazy(a), b), (a, lazy(b)), (lazy(a), lazy(b))):
        same([f(x, y)], want[:1])
    leaf = (-a).requires_grad_()          # the gradient goes through the view
    same(torch.autograd.grad(f(torch._neg_view(leaf), b), leaf, g), [-want[1]])


def test_as_a_program_meets_it(gpu):
    """.imag of a conjugate: of one element it counts as contiguous, and nothing wrote it out."""
    z = torch.complex(torch.randn(1, 1, 1), torch.randn(1, 1, 1)).to(gpu)
    g = z.conj().imag
    assert g.is_neg() and g.is_contiguous()
    a, b = torch.randn(1, 1, 1, device=gpu), torch.randn(1, 1, 1, device=gpu)
    for f in DENSE.values():
        same(first_order(f, (a, b), g), first_order(f, (a, b), g.clone()))
        assert torch.equal(f(g, b), f(g.clone(), b))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,M,K,N", [(2, 7, 5, 9), (2, 128, 128, 128)])
def test_second_order(gpu, dtype, B, M, K, N):
    torch.manual_seed(M)
    a, b, g, ua, ub = (torch.randn(*s).to(gpu, dtype) for s in ((B, M, K), (B, K, N), (B, M, N), (B, M, K), (B, K, N)))

    def run(g, us):
        x, y, h = a.clone().requires_grad_(), b.clone().requires_grad_(), torch.zeros_like(g).requires_grad_()
        first = torch.autograd.grad(genbmm.logbmm(x, y), (x, y), g + h, create_graph=True)
        return torch.autograd.grad(first, (x, y, h), us)

    same(run(g, [lazy(ua), lazy(ub)]), run(g, [ua, ub]))


BANDED = {"mul": lambda x, y: x.multiply(y), "log": lambda x, y: x.multiply_log(y), "max": lambda x, y: x.multiply_max(y),
          "sample": lambda x, y: x.multiply_sample(y, STREAM)}


@pytest.mark.parametrize("op", list(BANDED))
@pytest.mark.parametrize("dtype", DTYPES)
def test_banded(gpu, op, dtype):
    torch.manual_seed(3)
    a, b = torch.randn(2, 9, 4).to(gpu, dtype), torch.randn(2, 9, 3).to(gpu, dtype)
    g = torch.randn(2, 9, 6).to(gpu, dtype)

    def f(x, y):
        return BANDED[op](genbmm.BandedMatrix(x, 2, 1), genbmm.BandedMatrix(y, 1, 1)).data

    want = first_order(f, (a, b), g)
    same(first_order(f, (a, b), lazy(g)), want)
    same([f(lazy(a), lazy(b))], want[:1])
    leaf = (-a).requires_grad_()
    same(torch.autograd.grad(f(torch._neg_view(leaf), b), leaf, g), [-want[1]])
    direct = {"mul": sparse.bandedbmm, "log": sparse.bandedlogbmm, "max": sparse.bandedmaxbmm}
    if op in direct:                      # the Functions themselves, by the reference's names
        h = lambda x, y: direct[op](x, 2, 1, y, 1, 1, 3, 2)
        x, y = lazy(a).requires_grad_(), lazy(b).requires_grad_()
        out = h(x, y)
        same([out.detach()] + list(torch.autograd.grad(out, (x, y), g)), want)


def test_banded_second_order_and_structure(gpu):
    torch.manual_seed(4)
    a, b, g = torch.randn(2, 9, 4, device=gpu), torch.randn(2, 9, 3, device=gpu), torch.randn(2, 9, 6, device=gpu)
    ua, ub = torch.randn_like(a), torch.randn_like(b)

    def run(us):
        x, y, h = (t.clone().requires_grad_() for t in (a, b, g))
        out = genbmm.BandedMatrix(x, 2, 1).multiply_log(genbmm.BandedMatrix(y, 1, 1)).data
        return torch.autograd.grad(torch.autograd.grad(out, (x, y), h, create_graph=True), (x, y, h), us)

    same(run([lazy(ua), lazy(ub)]), run([ua, ub]))
    m = genbmm.BandedMatrix(a, 2, 1)
    n = genbmm.BandedMatrix(lazy(a), 2, 1)
    other = genbmm.BandedMatrix(b, 1, 1)
    for f in (lambda x: x.transpose(), lambda x: x.band_shift(1), lambda x: x.band_pad(2), lambda x: x.col_shift(1),
              lambda x: x._expand(3, 3), lambda x: x.op(other, torch.add), lambda x: x.multiply_back(other, None, lazy(g))):
        assert torch.equal(f(n).data, f(m).data)
    assert torch.equal(n.to_dense(), m.to_dense())
    dense = m.to_dense()
    assert torch.equal(genbmm.banddiag(lazy(dense), 2, 1)[0], genbmm.banddiag(dense, 2, 1)[0])


def test_traced_operators(gpu):
    torch.manual_seed(5)
    a, b, g = torch.randn(2, 7, 5, device=gpu), torch.randn(2, 5, 9, device=gpu), torch.randn(2, 7, 9, device=gpu)
    for f in (ops.logbmm, ops.maxbmm, ops.prodmaxbmm, lambda x, y: ops.samplebmm(x, y, *STREAM)):
        want = first_order(f, (a, b), g)
        same(first_order(f, (a, b), lazy(g)), want)
        same([f(lazy(a), lazy(b))], want[:1])


def test_refused_where_nothing_writes_it_out(gpu):
    """The dense Functions take operands in the library's form only; a saved tensor that a hook replaced is not the
    forward's."""
    a, b, g = torch.randn(2, 7, 5, device=gpu), torch.randn(2, 5, 9, device=gpu), torch.randn(2, 7, 9, device=gpu)
    for f in (genmul.LogMatMul, genmul.MaxMatMul, genmul.ProdMaxMatMul, genmul.SampleMatMul):
        with pytest.raises(RuntimeError, match="negative"):
            f.apply(lazy(a), b)
    with pytest.raises(RuntimeError, match="negative"):
        _lib.addr(lazy(a))
    for f in (genbmm.logbmm, genmul.LogMatMul.apply):
        x = a.clone().requires_grad_()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: torch._neg_view(t)):
            out = f(x, b)
        with pytest.raises(RuntimeError, match="negative"):
            torch.autograd.grad(out, x, g)
