"""Both gradients of the banded (+,x) and log products on 32 x 32 blocks (csrc/banded_grads.h): bands of one to three
blocks per row on either side, matrices cut anywhere inside a block, several workgroups per item and several items per
workgroup's round, values at both ends of the float range, values that are not finite, and the half types.  Against the
float64 sequential restatement of the reference's kernels (oracle.seq_band_bwd), every cell to 1e-5 of the sum of its
terms' magnitudes (a sum of up to 65 products in fp32, each within 2^-22, stays below 2^-17 of it)."""
import numpy as np
import pytest
import torch

import oracle
from genbmm_amd import _lib

pytestmark = pytest.mark.gpu
P = _lib.ptr

SHAPES = [(64, 33, 16, 16, 16, 16), (3, 257, 32, 32, 32, 32), (1, 96, 31, 33, 32, 32), (2, 129, 32, 31, 0, 64), (1, 31, 32, 32, 32, 32),
          (5, 200, 64, 0, 0, 32), (2, 500, 2, 3, 32, 32), (2, 333, 40, 20, 1, 1), (1, 2000, 20, 12, 9, 40), (130, 64, 32, 32, 32, 32),
          (1, 1, 30, 30, 30, 30), (300, 65, 32, 32, 32, 32)]


def bands(B, n, W, scale=1.0):
    return torch.rand(B, n, W) * 2 - 1 if scale == 1.0 else (torch.rand(B, n, W) * 2 - 1) * scale


def run(gpu, a, b, g, band, mode, suffix=""):
    lib = _lib.load()
    a_lu, a_ld, b_lu, b_ld = band
    B, n, _ = a.shape
    a, b, g = a.to(gpu), b.to(gpu), g.to(gpu)
    out, ga, gb = torch.empty_like(g), torch.full_like(a, float("nan")), torch.full_like(b, float("nan"))
    ws = torch.empty(max(1, lib.genbmm_banded_workspace_size(*band, B, n)), device=gpu) if mode == 0 else None
    s = _lib.stream_of(a)
    assert getattr(lib, "genbmm_banded_fwd" + suffix)(P(a), a_lu, a_ld, P(b), b_lu, b_ld, P(out), None, P(ws), B, n, mode, s) == 0
    assert getattr(lib, "genbmm_banded_bwd" + suffix)(P(a), a_lu, a_ld, P(b), b_lu, b_ld, P(out), None, P(ws), P(g), P(ga), P(gb),
                                                      B, n, mode, s) == 0
    return ga.cpu(), gb.cpu()


def reference(a, b, g, band, mode):
    return oracle.seq_band_bwd(a.double(), band[0], band[1], b.double(), band[2], band[3], g.double(), mode, dtype=np.float64)


def near(got, want, scale):
    assert bool(((got.double() - want).abs() <= 1e-5 * scale + 1e-44).all()), float(((got.double() - want).abs() / (scale + 1e-44)).max())


@pytest.mark.parametrize("B,n,a_lu,a_ld,b_lu,b_ld", SHAPES)
@pytest.mark.parametrize("mode", [0, 3])
def test_gradients_of_block_bands(gpu, B, n, a_lu, a_ld, b_lu, b_ld, mode):
    torch.manual_seed(n + mode)
    band = (a_lu, a_ld, b_lu, b_ld)
    a, b = bands(B, n, a_lu + a_ld + 1), bands(B, n, b_lu + b_ld + 1)
    g = torch.randn(B, n, a.shape[2] + b.shape[2] - 1)
    got = run(gpu, a, b, g, band, mode)
    if B > 8:       # the oracle is sequential: a few items, the ends among them
        pick = [0, 1, B // 2, B - 2, B - 1]
        a, b, g, got = a[pick], b[pick], g[pick], [x[pick] for x in got]
    want = reference(a, b, g, band, mode)
    scale = reference(a if mode == 0 else a.abs(), b if mode == 0 else b.abs(), g.abs(), band, mode)
    for x, y, z in zip(got, want, scale):
        near(x, y, z.double())


@pytest.mark.parametrize("tiny,huge", [(1e-37, 1e30), (1e-30, 1e-3), (1e-20, 1e20)])
def test_gradients_at_both_ends_of_the_range(gpu, tiny, huge):
    """Operands and gradients far apart in magnitude, denormals among them: the parts of a small factor are as exact as
    a large one's."""
    torch.manual_seed(3)
    band = (32, 32, 30, 34)
    a, b, g = bands(2, 150, 65), bands(2, 150, 65), torch.randn(2, 150, 129)
    a[0] *= tiny
    b[0] *= huge
    g[1, 40:90] *= tiny
    b[1, :, 20:40] *= huge
    got, want = run(gpu, a, b, g, band, 3), reference(a, b, g, band, 3)
    for x, y, z in zip(got, want, reference(a.abs(), b.abs(), g.abs(), band, 3)):
        near(x, y, z.double())


@pytest.mark.parametrize("mode", [0, 3])
def test_gradients_that_are_not_finite(gpu, mode):
    """An infinite or NaN gradient reaches the cells it is a term of and no other; the others of such a line (a row of the
    gradient's band) may be the exact way's, in which infinity meets no zero of a staged block, and lines without such
    cells keep their bits.  (Infinities within 31 cells of a row's end are left out: a staged block may hold them beside a
    neighbouring line, times zero, and that line is then the exact way's as well.)  Sums of the log product that its forward could not factor are the exact way's."""
    torch.manual_seed(4)
    band = (32, 32, 32, 32)
    a, b, g = bands(2, 200, 65), bands(2, 200, 65), torch.randn(2, 200, 129)
    clean, clean_want = run(gpu, a, b, g, band, mode), reference(a, b, g, band, mode)
    g[0, 50, 70], g[0, 120, 64], g[1, 100, 30] = float("inf"), float("nan"), 1e36
    got, want = run(gpu, a, b, g, band, mode), reference(a, b, g, band, mode)
    small = torch.where(torch.isfinite(g), g, torch.zeros(()))
    scale = reference(a if mode == 0 else a.abs(), b if mode == 0 else b.abs(), small.abs(), band, mode)
    for x, y, z, c, cy in zip(got, want, scale, clean, clean_want):
        assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(torch.isinf(x), torch.isinf(y))
        fin = torch.isfinite(y)
        near(x[fin], y[fin], z.double()[fin])
        kept = ((y == cy).all(2))
        assert bool(kept.any()) and not bool(kept.all()) and torch.equal(x[kept], c[kept])
    if mode == 0:
        a[0, 60:80] -= 300.0 * (torch.arange(65) > 30)
        g = torch.randn(2, 200, 129)
        # The exact way's weight is exp(a + b - out) of values around 300: a + b, out and the difference are rounded
        # by up to 2^-24 300 each, 5.4e-5 of the weight together, and so may every term of a sum be.
        got, want, scale = run(gpu, a, b, g, band, 0), reference(a, b, g, band, 0), reference(a, b, g.abs(), band, 0)
        for x, y, z in zip(got, want, scale):
            assert bool(((x.double() - y).abs() <= 6e-5 * z.double() + 1e-30).all())


@pytest.mark.parametrize("dt,suffix", [(torch.float16, "_f16"), (torch.bfloat16, "_bf16")])
def test_half_gradients_are_the_float_kernels_rounded_once(gpu, dt, suffix):
    torch.manual_seed(5)
    for band, n in (((32, 32, 32, 32), 300), ((20, 12, 30, 2), 95)):
        a, b = bands(3, n, band[0] + band[1] + 1).to(dt), bands(3, n, band[2] + band[3] + 1).to(dt)
        g = torch.randn(3, n, a.shape[2] + b.shape[2] - 1).to(dt)
        for mode in (0, 3):
            half, full = run(gpu, a, b, g, band, mode, suffix), run(gpu, a.float(), b.float(), g.float(), band, mode)
            for x, y in zip(half, full):
                assert torch.equal(x, y.to(dt)), (band, mode)
