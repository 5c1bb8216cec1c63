"""Many small and odd shapes through the arg-max products and their backward: the group
sweep + resolve (64- and 32-column panels, ragged K), the (line, k-range) backward with
one to sixty-four ranges, and samplebmm's three sweeps.  Seeded, so the cases are fixed."""
import random

import numpy as np
import pytest
import torch

import oracle
import genbmm_amd as genbmm
from genbmm_amd import _lib

pytestmark = pytest.mark.gpu


def _shapes(seed, count, kmax):
    rng = random.Random(seed)
    edge = [1, 2, 3, 7, 8, 9, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 130]
    out = []
    for _ in range(count):
        M = rng.choice(edge + [rng.randint(1, 200)])
        N = rng.choice(edge + [rng.randint(1, 200)])
        K = rng.choice([1, 2, 7, 8, 9, 15, 16, 17, 127, 128, 129, 255, 256, 257, 263, 511, 512, 513, rng.randint(1, kmax)])
        B = rng.randint(1, 3)
        if B * M * K * N > 6_000_000:
            K = max(1, 6_000_000 // (B * M * N))
        out.append((B, M, K, N))
    return out


def grid(*shape):
    return torch.round(torch.randn(*shape) * 4) / 4


@pytest.mark.parametrize("prod", [False, True])
def test_max_products_on_many_shapes(gpu, prod):
    torch.manual_seed(5)
    for B, M, K, N in _shapes(11 + prod, 40, 700):
        a, b = grid(B, M, K), grid(B, K, N)
        g = grid(B, M, N).clamp(-4, 4)
        ad, bd = a.to(gpu).requires_grad_(True), b.to(gpu).requires_grad_(True)
        out = (genbmm.prodmaxbmm if prod else genbmm.maxbmm)(ad, bd)
        sv, si = oracle.seq_maxbmm_fwd(a, b, prod)
        assert torch.equal(out.detach().cpu(), sv), (B, M, K, N)
        ga, gb = torch.autograd.grad(out, (ad, bd), g.to(gpu))
        wa, wb = oracle.seq_argmax_bwd(a if prod else K, b, si, g, prod)
        assert torch.equal(ga.cpu(), wa) and torch.equal(gb.cpu(), wb), (B, M, K, N)


def test_argmax_backward_with_many_k_ranges(gpu):
    """K from one range of 128 cells to more than 64 of them (several workgroups per line)."""
    lib = _lib.load()
    torch.manual_seed(6)
    for B, M, K, N in [(1, 5, 1, 9), (2, 70, 129, 33), (1, 40, 1000, 70), (1, 9, 4097, 17), (1, 3, 8200, 5),
                       (1, 2, 9000, 130)]:
        idx = torch.randint(-1, K, (B, M, N), dtype=torch.int32)
        g = torch.randn(B, M, N)
        ga = torch.full((B, M, K), float("nan"), device=gpu)
        gb = torch.full((B, K, N), float("nan"), device=gpu)
        assert lib.genbmm_argmax_bwd(_lib.ptr(idx.to(gpu)), _lib.ptr(g.to(gpu)), _lib.ptr(ga), _lib.ptr(gb),
                                     B, M, K, N, _lib.stream_of(ga)) == 0
        wa, wb = oracle.seq_argmax_bwd(K, torch.zeros(B, K, N), idx, g, False)
        assert torch.equal(ga.cpu(), wa) and torch.equal(gb.cpu(), wb), (B, M, K, N)


@pytest.mark.parametrize("prod", [False, True])
def test_argmax_backward_of_every_row_length(gpu, prod):
    """Rows of 1 to 68 cells: whole chunks of 32, whole pieces of four, single cells, in every combination,
    rows of odd length (so that pieces start at any cell).  Bit for bit as the ordered sums."""
    torch.manual_seed(8)
    for N in range(1, 69):
        a, b, g = grid(2, 5, 9), grid(2, 9, N), grid(2, 5, N)
        for dt in (torch.float32, torch.float16):
            ad, bd = a.to(gpu, dt).requires_grad_(True), b.to(gpu, dt).requires_grad_(True)
            ga, gb = torch.autograd.grad((genbmm.prodmaxbmm if prod else genbmm.maxbmm)(ad, bd), (ad, bd), g.to(gpu, dt))
            _, si = oracle.seq_maxbmm_fwd(a, b, prod)
            wa, wb = oracle.seq_argmax_bwd(a if prod else 9, b, si, g, prod)
            assert torch.equal(ga.cpu(), wa.to(dt)) and torch.equal(gb.cpu(), wb.to(dt)), (N, dt)

def test_sample_on_many_shapes(gpu):
    """Every index brackets its uniform in the float64 CDF; shapes on both sides of the
    matrix-core limits (M, N >= 96, K >= 16), of the 62 slabs that its six-bit tag counts
    (K <= 992; K = 993, 1008, 1040: seven bits) and of its 126-slab limit (K <= 2016; the last
    shape has a matrix-core forward and, with K = 2020, the two-level sweep on the vector ALU
    behind it)."""
    lib = _lib.load()
    torch.manual_seed(7)
    shapes = _shapes(13, 14, 400) + [(1, 96, 16, 96), (1, 97, 993, 100), (1, 130, 992, 96), (2, 100, 500, 131),
                                     (1, 128, 1040, 160), (2, 256, 1008, 128), (1, 128, 2016, 96), (1, 96, 2020, 128)]
    for B, M, K, N in shapes:
        a, b = 2 * torch.randn(B, M, K), 2 * torch.randn(B, K, N)
        ad, bd = a.to(gpu), b.to(gpu)
        out = torch.empty(B, M, N, device=gpu)
        idx = torch.empty(B, M, N, dtype=torch.int32, device=gpu)
        stats = torch.empty(lib.genbmm_samplebmm_stats_size(B, M, K, N), device=gpu)
        assert lib.genbmm_samplebmm_fwd(_lib.ptr(ad), _lib.ptr(bd), _lib.ptr(out), _lib.ptr(idx), _lib.ptr(stats),
                                        77, 3, B, M, K, N, _lib.stream_of(ad)) == 0
        u = oracle.philox_uniform(0, B * M * N, 77, 3).view(B, M, N).double()
        cdf = oracle.sample_cdf64(a, b)
        got = idx.cpu().long()
        assert int(got.min()) >= 0 and int(got.max()) < K, (B, M, K, N)
        hi = torch.gather(cdf, 2, got.unsqueeze(2)).squeeze(2)
        lo = torch.where(got > 0, torch.gather(cdf, 2, (got - 1).clamp(min=0).unsqueeze(2)).squeeze(2),
                         torch.zeros_like(hi))
        ok = (lo - 2e-5 <= u) & (u <= hi + 2e-5)
        assert bool(ok.all()), ((B, M, K, N), float((~ok).float().mean()))
        want = oracle.sample_index_from_cdf(cdf, u).long()
        assert float((got != want).float().mean()) < 5e-3, (B, M, K, N)


@pytest.mark.parametrize("shape", [(2, 128, 200, 160), (2, 256, 512, 128)])
@pytest.mark.parametrize("scale", [0.05, 2.0, 12.0, 40.0, 100.0, 400.0])
def test_sample_on_flat_and_peaked_distributions(gpu, scale, shape):
    """From nearly uniform to one-term-takes-all (at the largest scales the winning term leads by
    hundreds: the remainder the matrix-core sweep hands to the resolve step, six mantissa bits
    short, must still name the right term), with masked terms (-inf, -1e9), on shapes that take
    the matrix-core sweep (and its exact fix-up where S underflows): 13 and 32 slabs."""
    lib = _lib.load()
    torch.manual_seed(int(scale * 10))
    B, M, K, N = shape
    a, b = scale * torch.randn(B, M, K), scale * torch.randn(B, K, N)
    a[:, ::3, ::5] = float("-inf")
    b[:, 1::7, ::2] = -1e9
    a[1, 5, :] = float("-inf")          # a row without any mass: out = -inf, index 0
    ad, bd = a.to(gpu), b.to(gpu)
    out = torch.empty(B, M, N, device=gpu)
    idx = torch.empty(B, M, N, dtype=torch.int32, device=gpu)
    stats = torch.empty(lib.genbmm_samplebmm_stats_size(B, M, K, N), device=gpu)
    assert lib.genbmm_samplebmm_fwd(_lib.ptr(ad), _lib.ptr(bd), _lib.ptr(out), _lib.ptr(idx), _lib.ptr(stats),
                                    5, 11, B, M, K, N, _lib.stream_of(ad)) == 0
    u = oracle.philox_uniform(0, B * M * N, 5, 11).view(B, M, N).double()
    want_out, want_idx = oracle.seq_samplebmm_fwd(a, b, u.float())
    got = idx.cpu().long()
    live = torch.ones(B, M, N, dtype=torch.bool)
    live[1, 5, :] = False
    assert bool((got[~live] == 0).all()) and bool((out.cpu()[~live] == want_out[~live]).all())
    assert torch.allclose(out.cpu()[live], want_out[live], rtol=1e-5, atol=1e-5)
    cdf = oracle.sample_cdf64(a, b)
    hi = torch.gather(cdf, 2, got.unsqueeze(2)).squeeze(2)
    lo = torch.where(got > 0, torch.gather(cdf, 2, (got - 1).clamp(min=0).unsqueeze(2)).squeeze(2), torch.zeros_like(hi))
    # fp32 prefix sums over K terms (the reference's too): K roundings of 2^-24 of the running mass;
    # and the masses are exp(a + b - out) with `out` rounded to fp32: 2^-24 |out| in the exponent
    tol = max(2e-5, 2.0 * K * 2.0 ** -24, 2.0 * float(want_out[live].abs().max()) * 2.0 ** -23)
    viol = torch.maximum(lo - u, u - hi).clamp(min=0)
    ok = (viol <= tol) | ~live
    assert bool(ok.all()), (float((~ok).float().mean()), float(viol[live].max()), tol)
    # a sampled term always has mass (never a masked one)
    picked = torch.gather(a.unsqueeze(-1) + b.unsqueeze(-3), 2, got.unsqueeze(2)).squeeze(2)
    assert bool((picked[live] > -1e8).all())

# Edges of the whole-item log kernels (tiles of 16, groups of four rows per wave, 64 columns per chunk, the sizes at
# which another instantiation takes over, the largest items) and of the 128-wide tiles on narrower extents behind them.
_LOG_EDGES = [(3, 1, 1, 1), (3, 15, 16, 17), (2, 17, 33, 31), (2, 32, 33, 48), (2, 49, 48, 47), (2, 64, 63, 64), (2, 65, 64, 1),
              (2, 16, 65, 64), (1, 95, 96, 97), (2, 97, 16, 95), (1, 128, 100, 64), (1, 5, 128, 127), (1, 128, 1, 128),
              (1, 100, 80, 100), (1, 96, 97, 96), (1, 104, 100, 97), (2, 33, 130, 35), (2, 130, 33, 40), (600, 33, 129, 64),
              (2, 70, 200, 90), (1, 40, 512, 33)]


@pytest.mark.parametrize("B,M,K,N", _LOG_EDGES)
def test_log_products_at_the_edges_of_their_kernels(gpu, B, M, K, N):
    """Against float64 (a few roundings of values around 10: 1e-5), and the half types against the float kernels
    on the same widened values, rounded once."""
    torch.manual_seed(M + K + N)
    a, b, g = torch.randn(B, M, K), torch.randn(B, K, N), torch.randn(B, M, N)
    want = oracle.logbmm_grads64(a, b, g)
    ad, bd = a.to(gpu).requires_grad_(True), b.to(gpu).requires_grad_(True)
    out = genbmm.logbmm(ad, bd)
    for got, ref in zip((out.detach(),) + torch.autograd.grad(out, (ad, bd), g.to(gpu)), want):
        assert torch.allclose(got.cpu().double(), ref, rtol=1e-5, atol=1e-5), (B, M, K, N)
    lib = _lib.load()
    for dt, sfx in ((torch.float16, "_f16"), (torch.bfloat16, "_bf16")):
        half = [x.to(gpu, dt) for x in (a, b, g)]
        wide = [x.float() for x in half]
        res = []
        for sfx_, (x, y, gg) in ((sfx, half), ("", wide)):
            o, gx, gy = torch.empty_like(gg), torch.empty_like(x), torch.empty_like(y)
            ws = torch.empty(lib.genbmm_logbmm_stats_size(B, M, K, N), device=gpu)
            assert getattr(lib, "genbmm_logbmm_fwd" + sfx_)(*map(_lib.ptr, (x, y, o, ws)), B, M, K, N, _lib.stream_of(x)) == 0
            if sfx_ == "":
                o_float, o = o, res[0].float()      # the half backward reads `out` as stored
            assert getattr(lib, "genbmm_logbmm_bwd" + sfx_)(*map(_lib.ptr, (x, y, o, gg, ws, gx, gy)), B, M, K, N,
                                                            _lib.stream_of(x)) == 0
            if sfx_ == "":
                assert torch.equal(res[0], o_float.to(dt)), (dt, B, M, K, N)
                assert torch.equal(res[1], gx.to(dt)) and torch.equal(res[2], gy.to(dt)), (dt, B, M, K, N)
            res += [o, gx, gy]


@pytest.mark.parametrize("B,M,K,N", [(3, 17, 20, 33), (2, 65, 70, 50), (2, 100, 100, 60), (2, 120, 128, 40)])
def test_log_items_that_cannot_be_factored(gpu, B, M, K, N):
    """Rows 200 apart, a masked row and a masked column (-inf), a row at the floor: cells (forward) and items (backward)
    that the factored form does not carry.  The other items keep their bits."""
    torch.manual_seed(7)
    a, b, g = torch.randn(B, M, K), torch.randn(B, K, N), torch.randn(B, M, N)
    clean = [x.to(gpu) for x in (a, b, g)]
    a[0, 3, : K // 2] -= 200
    b[0, K // 2 :] -= 200
    a[0, 5], b[0, :, 7], a[0, 6] = -float("inf"), -float("inf"), -1e9
    g[0, 5], g[0, :, 7], g[0, 6] = 0, 0, 0
    outs = []
    for x, y, z in (clean, [t.to(gpu) for t in (a, b, g)]):
        x, y = x.requires_grad_(True), y.requires_grad_(True)
        o = genbmm.logbmm(x, y)
        outs.append((o.detach(),) + torch.autograd.grad(o, (x, y), z))
    for u, v in zip(*outs):
        assert torch.equal(u[1:], v[1:])
    want = torch.logsumexp(a[0].double().unsqueeze(2) + b[0].double().unsqueeze(0), 1)
    got = outs[1][0][0].cpu().double()
    live = torch.ones(M, N, dtype=torch.bool)
    live[5], live[6], live[:, 7] = False, False, False
    assert torch.allclose(got[live], want[live], rtol=1e-5, atol=1e-5)
    assert bool((got[5] == -float("inf")).all()) and bool((got[:, 7][live[:, 0]] == -float("inf")).all())


ITEMS = [(3, 20, 31, 17), (2, 3, 2, 5), (2, 48, 40, 33), (2, 64, 64, 64), (2, 65, 70, 50), (2, 96, 90, 72), (2, 128, 100, 64),
         (2, 128, 16, 128), (2, 2, 128, 1), (3, 128, 4, 4), (3, 9, 5, 16), (2, 3, 4, 128), (2, 32, 128, 32), (2, 128, 32, 32),
         (2, 32, 32, 128), (2, 128, 32, 128), (2, 66, 2, 67)]


def _log_grads(gpu, a, b, g, dt):
    x, y = a.to(gpu, dt).requires_grad_(True), b.to(gpu, dt).requires_grad_(True)
    o = genbmm.logbmm(x, y)
    return [o.detach()] + list(torch.autograd.grad(o, (x, y), g.to(gpu, dt)))


@pytest.mark.parametrize("dt, eps", [(torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("kind", ["one", "most"])
@pytest.mark.parametrize("shape", ITEMS)
def test_log_items_with_cells_that_cannot_be_factored(gpu, shape, kind, dt, eps):
    """One such cell (its row and its column of the gradients are formed again, the others are not), and most of them.
    A weight exp(a + b - out) is as good as its exponent: |a + b| and |out| stay below 256, so 3 x 2^-25 x 256 = 2.3e-5
    and a few units of rounding; a gradient is off by at most that share of its sum over |g|.  Half types add
    the rounding of `out`, which the weights are formed from (up to eps x |out|), and of the result."""
    torch.manual_seed(11)
    B, M, K, N = shape
    a, b, g = torch.randn(B, M, K), torch.randn(B, K, N), torch.randn(B, M, N)
    if kind == "most":
        a, b = 20 * a, 20 * b
    else:
        a[0, 1, 0] += 60
        b[0, 1, 0] += 60
    a, b, g = (t.to(dt).float() for t in (a, b, g))
    got = [t.double().cpu() for t in _log_grads(gpu, a, b, g, dt)]
    x, y = a.double().requires_grad_(True), b.double().requires_grad_(True)
    out = torch.logsumexp(x.unsqueeze(3) + y.unsqueeze(1), 2)
    want = torch.autograd.grad(out, (x, y), g.double(), retain_graph=True)
    size = torch.autograd.grad(out, (x, y), g.abs().double())
    most = float(out.detach().abs().max())
    assert most < 256
    assert bool(((got[0] - out).abs() <= 2e-5 + (2.0 ** -23 + eps) * out.abs()).all())
    share = 4e-5 + (0.0 if dt == torch.float32 else np.expm1(eps * most) + eps)
    for p, q, s in zip(got[1:], want, size):
        assert bool(((p - q).abs() <= share * s + 1e-6).all()), float(((p - q).abs() - share * s).max())


# (shape, checksum of the indices, checksum of the results' bit patterns): what (77, 3) draws, taken on this GPU
PINNED = [
    ((3, 32, 32, 32), 75771211, 5024752994044624),
    ((5, 20, 31, 17), 21829264, 1533337294056679),
    ((2, 3, 7, 5), 841, 238548035912),
    ((3, 39, 39, 39), 200200960, 11141693888447905),
    ((4, 33, 50, 40), 339369046, 14925593276291406),
    ((2, 64, 64, 64), 1063904730, 36168368379317341),
    ((2, 48, 64, 16), 35921555, 1265989910378496),
    ((2, 64, 64, 65), 1105184507, 37307711455305653),
    ((2, 95, 90, 94), 3625213043, 86771139876725177),
    ((2, 128, 16, 128), 1204188941, 165470003316713310),
    ((2, 88, 173, 83), 5097526939, 65001696922925094),
    ((1, 50, 300, 200), 7289323424, 54278549119542690),
    ((40, 60, 60, 160), 56095483104, 2078153295314331851),
    ((3, 96, 97, 72), 4839040713, 108602366278520920),
    ((2, 128, 100, 64), 3389913281, 75868209950720266),
    ((3, 96, 96, 96), 6064557672, 139651555690366767),
    ((1, 97, 993, 100), 23311339183, 51548700677893467),
    ((1, 96, 2020, 128), 53009622172, 57440072148626388),
]


@pytest.mark.parametrize("shape, draws, bits", PINNED)
def test_pinned_draws_stay_the_same(gpu, shape, draws, bits):
    """A (seed, offset) names its draws: they and the result whose last bits they hang on are those they always were,
    with cells that the factored sums cannot serve among them (a term that leads by e^60, a row and a column
    without mass)."""
    lib = _lib.load()
    B, M, K, N = shape
    gen = torch.Generator().manual_seed(B + 3 * M + 5 * K + 7 * N)
    a, b = (torch.randint(-3000, 3000, s, generator=gen).float() / 512 for s in ((B, M, K), (B, K, N)))
    a[0, 1, 0] += 60
    b[0, 1, 0] += 60
    a[-1, 2, :] = float("-inf")
    a[-1, :, 0] = -1e9
    ad, bd = a.to(gpu), b.to(gpu)
    out = torch.empty(B, M, N, device=gpu)
    idx = torch.empty(B, M, N, dtype=torch.int32, device=gpu)
    stats = torch.empty(lib.genbmm_samplebmm_stats_size(B, M, K, N), device=gpu)
    assert lib.genbmm_samplebmm_fwd(_lib.ptr(ad), _lib.ptr(bd), _lib.ptr(out), _lib.ptr(idx), _lib.ptr(stats),
                                    77, 3, B, M, K, N, _lib.stream_of(ad)) == 0
    w = (torch.arange(B * M * N) % 9973 + 1).view(B, M, N)
    assert int((idx.cpu().long() * w).sum()) == draws
    assert int((out.cpu().view(torch.int32).long() * w).sum()) == bits
