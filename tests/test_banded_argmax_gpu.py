"""The band max product's backward where its addressing changes: strips whose cells all lie inside the matrix, and
rows so long that a strip's offsets do not fit 32 bits."""
import numpy as np
import pytest
import torch

import oracle
from genbmm_amd import _lib
from genbmm_amd.sparse import BandedMatrix

pytestmark = pytest.mark.gpu


# a first and a last strip beside inner ones, rows of whole and partial chunks of 16 cells, one chunk and less,
# a band of several parts of 128 diagonals, one-sided bands
@pytest.mark.parametrize("n,a_lu,a_ld,b_lu,b_ld", [
    (300, 9, 6, 7, 9), (300, 8, 8, 7, 9), (270, 3, 4, 4, 4), (270, 2, 1, 3, 2), (330, 32, 32, 32, 32), (700, 100, 160, 3, 130),
    (400, 0, 40, 0, 30), (400, 40, 0, 30, 0)])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
def test_inner_strips(gpu, n, a_lu, a_ld, b_lu, b_ld, dt):
    """Bit for bit the sequential oracle's sums; the bands' cells outside the matrix take part in nothing."""
    torch.manual_seed(n + a_lu)
    B = 3
    a = torch.randint(-8, 9, (B, n, a_lu + a_ld + 1)) / 4.0        # ties
    b = torch.randint(-8, 9, (B, n, b_lu + b_ld + 1)) / 4.0
    g = torch.randn(B, n, a.shape[2] + b.shape[2] - 1).to(dt)
    X = BandedMatrix(a.to(gpu, dt).requires_grad_(True), a_lu, a_ld)
    Y = BandedMatrix(b.to(gpu, dt).requires_grad_(True), b_lu, b_ld)
    ga, gb = torch.autograd.grad(X.multiply_max(Y).data, (X.data, Y.data), g.to(gpu))
    wa, wb = oracle.seq_band_bwd(a, a_lu, a_ld, b, b_lu, b_ld, g.float(), 1, dtype=np.float32)
    assert torch.equal(ga.cpu(), wa.to(dt)) and torch.equal(gb.cpu(), wb.to(dt))


def test_rows_beyond_32_bit_offsets(gpu):
    """2^25 diagonals on 17 rows.  Gradients are small whole numbers: exact in any order."""
    n, a_lu, a_ld, b_lu, b_ld = 17, 1 << 24, 1 << 24, 1, 1
    Wa, Wb, r_lu = a_lu + a_ld + 1, b_lu + b_ld + 1, a_lu + b_ld
    Wo = Wa + Wb - 1
    idx = torch.zeros(1, n, Wo, dtype=torch.int32, device=gpu)    # cells outside the matrix: 0
    g = torch.ones(1, n, Wo, device=gpu)                          # (whose gradient goes nowhere)
    ga, gb = torch.empty(1, n, Wa, device=gpu), torch.empty(1, n, Wb, device=gpu)
    want_a, want_b = {}, {}
    rng = np.random.default_rng(5)
    for i in range(n):
        for o in range(n):
            j = o - i + r_lu
            k = int(rng.integers(max(0, j - Wb + 1), min(j, Wa - 1) + 1))
            v = int(rng.integers(1, 9))
            idx[0, i, j], g[0, i, j] = k, v
            want_a[i, k] = want_a.get((i, k), 0) + v
            want_b[o, k - j + Wb - 1] = want_b.get((o, k - j + Wb - 1), 0) + v
    p = _lib.ptr
    # (the operands themselves are not read)
    assert _lib.load().genbmm_banded_bwd(p(ga), a_lu, a_ld, p(gb), b_lu, b_ld, p(None), p(idx), p(None), p(g), p(ga), p(gb),
                                         1, n, 1, _lib.stream_of(ga)) == 0
    for got, want in ((ga, want_a), (gb, want_b)):
        assert int(got.count_nonzero()) == len(want)
        rows, cols = zip(*want)
        assert got[0, list(rows), list(cols)].tolist() == list(want.values())
