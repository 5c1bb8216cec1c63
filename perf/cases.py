"""What the performance of this package is measured on.

Every case is one training step's use of one product, through the package's public functions:
the forward product, and the gradients with respect to both operands for an incoming gradient
(`second` cases: the second-order terms as well).  That is how a structured-prediction model calls
it: partition functions and marginals (logbmm, multiply_log), best paths (maxbmm, multiply_max),
sampled paths (samplebmm) and plain band products (multiply).

`listed()` holds the benchmark configurations of bench_configs.py, a ragged one and a bfloat16 one;
`draw()` spreads sizes, batches, bandwidths and element types over the ranges in between.
"""
import math

import torch

import genbmm_amd as genbmm

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_DENSE = {"log": genbmm.logbmm, "max": genbmm.maxbmm, "prodmax": genbmm.prodmaxbmm}


def listed():
    return [
        # A small chain: 16 sequences, 64 states.  The smallest call: launches and host work.
        _dense("log_small", "log", 16, 64, 64, 64),
        # A linear-chain CRF step: 512 (sequence, position) pairs, 128 states.
        _dense("log_chain", "log", 512, 128, 128, 128),
        # The bottom level of a chain's reduction tree: very many products of 32 states.
        _dense("log_skinny", "log", 8192, 32, 32, 32),
        # Large state spaces (the benchmark of bench.py).
        _dense("log_large", "log", 64, 512, 512, 512),
        # State counts that come from data, not from a tile: odd, unequal, nothing aligned.
        _dense("log_ragged", "log", 48, 251, 173, 301),
        # Mixed-precision training: the large step on bfloat16 potentials.
        _dense("log_bf16", "log", 64, 512, 512, 512, "bfloat16"),
        # A loss on marginals (entropy, risk): first- and second-order gradients of the CRF step.
        _dense("log_second", "second", 512, 128, 128, 128),
        # Best paths: maxbmm (and, drawn, prodmaxbmm on probabilities) on a grid with ties.
        _dense("max", "max", 256, 256, 256, 256),
        # Sampled paths.
        _dense("sample", "sample", 64, 512, 512, 512),
        # Alignments as banded matrices: 4096 positions, 32 diagonals either side, in the three semirings.
        _band("band_mul", "band_mul", 64, 4096, 32, 32, 32, 32),
        _band("band_log", "band_log", 64, 4096, 32, 32, 32, 32),
        _band("band_max", "band_max", 64, 4096, 32, 32, 32, 32),
    ]


def _dense(name, op, B, M, K, N, dtype="float32"):
    case = {"op": op, "B": B, "M": M, "K": K, "N": N, "dtype": dtype}
    return dict(case, name=name) if name else case


def _band(name, op, B, n, a_lu, a_ld, b_lu, b_ld):
    case = {"op": op, "B": B, "n": n, "a_lu": a_lu, "a_ld": a_ld, "b_lu": b_lu, "b_ld": b_ld, "dtype": "float32"}
    return dict(case, name=name) if name else case


def _loguniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


# (terms b*m*k*n of the largest listed case, share of the draws) of each dense product
_DENSE_RANGE = {"log": (64 * 512**3, 6), "second": (512 * 128**3, 1), "max": (256**4, 1), "prodmax": (256**4, 1),
                "sample": (64 * 512**3, 1)}
_SMALLEST = 16 * 64**3
_MOST_CELLS = 64 * 3 * 512**2      # of a, b and out together
_BAND_OPS = ("band_mul", "band_log", "band_max")


def draw(rng):
    ops = [op for op, (_, share) in _DENSE_RANGE.items() for _ in range(share)] + list(_BAND_OPS)
    op = rng.choice(ops)
    if op in _BAND_OPS:
        # bandwidths on either side of the diagonal apart, sequences from sentences to documents
        bands = [_loguniform(rng, 2, 32) for _ in range(4)]
        n = _loguniform(rng, 128, 4096)
        return _band(None, op, max(1, min(512, _loguniform(rng, 2**14, 64 * 4096) // n)), n, *bands)
    dtype = rng.choice(("float32", "float32", "float32", "float32", "bfloat16", "float16")) if op == "log" else "float32"
    most, _ = _DENSE_RANGE[op]
    low = 64 if op == "second" else 32
    if rng.random() < 0.4:          # one state space
        M = K = N = _loguniform(rng, low, 512)
    else:                           # three that are of the same order
        base = _loguniform(rng, low, 512)
        M, K, N = (max(low, min(512, int(base * rng.uniform(0.6, 1.5)))) for _ in range(3))
    terms = _loguniform(rng, _SMALLEST, most)
    cells = M * K + K * N + M * N
    B = max(1, min(terms // (M * K * N), _MOST_CELLS // cells, 8192))
    return _dense(None, op, B, M, K, N, dtype)


def prepare(case, seed):
    op, B = case["op"], case["B"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    if op in _BAND_OPS:
        n = case["n"]
        wa, wb = case["a_lu"] + case["a_ld"] + 1, case["b_lu"] + case["b_ld"] + 1
        # Uniform[-1, 1): similarity scores
        a = torch.rand(B, n, wa, generator=gen, device="cuda") * 2 - 1
        b = torch.rand(B, n, wb, generator=gen, device="cuda") * 2 - 1
        g = normal(B, n, wa + wb - 1)
    else:
        M, K, N = case["M"], case["K"], case["N"]
        a, b, g = normal(B, M, K), normal(B, K, N), normal(B, M, N)
        if op == "max":             # scores on a grid of eighths: ties are common
            a, b = torch.round(a * 8) / 8, torch.round(b * 8) / 8
        elif op == "prodmax":       # probabilities in (0, 1]
            a = 1 - torch.rand(B, M, K, generator=gen, device="cuda")
            b = 1 - torch.rand(B, K, N, generator=gen, device="cuda")
        elif op == "sample":        # log-potentials of a trained model: peaked
            a, b = 2 * a, 2 * b
    state = {"case": case, "a": a.to(dtype).requires_grad_(), "b": b.to(dtype).requires_grad_(), "g": g.to(dtype)}
    if op == "sample":              # the gradient of the sum counts the drawn terms; the draw is pinned,
        state["g"] = torch.ones_like(g)     # as a reproducible run's is
        state["stream"] = (seed, 0)
    elif op == "second":
        state["g"].requires_grad_()
        state["u"] = (normal(B, M, K), normal(B, K, N))
    return state


def run(state):
    case, a, b, g = state["case"], state["a"], state["b"], state["g"]
    op = case["op"]
    if op in _BAND_OPS:
        x = genbmm.BandedMatrix(a, case["a_lu"], case["a_ld"])
        y = genbmm.BandedMatrix(b, case["b_lu"], case["b_ld"])
        product = {"band_mul": x.multiply, "band_log": x.multiply_log, "band_max": x.multiply_max}[op]
        out = product(y).data
    elif op == "sample":
        out = genbmm.samplebmm(a, b, stream=state["stream"])
    elif op == "second":
        out = genbmm.logbmm(a, b)
        first = torch.autograd.grad(out, (a, b), g, create_graph=True)
        second = torch.autograd.grad(first, (a, b, g), state["u"])
        return (out,) + first + second
    else:
        out = _DENSE[op](a, b)
    return (out,) + torch.autograd.grad(out, (a, b), g)


def exact(case, seed):
    """What `run` returns for these inputs, by plain torch in float64.  A maximum compares sums (products)
    rounded once to float32, as its definition has it, and takes the lowest index that attains it; the
    gradients of a drawn path have no such value."""
    state = prepare(case, seed)
    op = case["op"]
    a, b = (state[x].detach().double().requires_grad_() for x in "ab")
    g = state["g"].detach().double()
    if op == "second":
        g.requires_grad_()
        out = _log_product(a, b)
        first = torch.autograd.grad(out, (a, b), g, create_graph=True)
        return (out,) + first + torch.autograd.grad(first, (a, b, g), [u.double() for u in state["u"]])
    if op in ("max", "prodmax"):
        return _best_product(a.detach(), b.detach(), g, op == "prodmax")
    if op in _BAND_OPS:
        wa, wb = case["a_lu"] + case["a_ld"] + 1, case["b_lu"] + case["b_ld"] + 1
        rows = _band_rows(b, case["b_ld"], wb)
        if op == "band_max":
            return _best_band(a.detach(), rows.detach(), g, case)
        # inputs within [-1, 1): exponentials need no shift
        x, y = (a, rows) if op == "band_mul" else (a.exp(), torch.where(_band_cells(rows, case), rows.exp(), 0))
        out = torch.zeros(*a.shape[:2], wa + wb - 1, dtype=torch.float64, device=a.device)
        for i, cols, pos in _band_terms(case):
            out[:, cols, i : i + wb] += x[:, cols, i : i + 1] * y[:, pos]
        if op == "band_log":        # cells without a term hold 0
            out = torch.where(out > 0, torch.where(out > 0, out, 1).log(), 0)
    else:
        out = _log_product(a, b)
    if op == "sample":
        return out.detach(), None, None
    return (out.detach(),) + torch.autograd.grad(out, (a, b), g)


def _log_product(a, b):
    ma, mb = a.detach().amax(2, keepdim=True), b.detach().amax(1, keepdim=True)
    return torch.bmm((a - ma).exp(), (b - mb).exp()).log() + ma + mb


def _best_product(a, b, g, prod):
    out, ga, gb = torch.empty_like(g), torch.zeros_like(a), torch.zeros_like(b)
    K = a.shape[2]
    step = max(1, 2**28 // (a.shape[1] * K * b.shape[2]))
    ks = torch.arange(K, device=a.device).view(1, 1, K, 1)
    for i in range(0, a.shape[0], step):
        x, y, s = a[i : i + step].unsqueeze(3), b[i : i + step].unsqueeze(1), slice(i, i + step)
        terms = (x * y if prod else x + y).float()
        best = terms.amax(2, keepdim=True)
        idx = torch.where(terms == best, ks, K).amin(2)
        out[s] = best.squeeze(2)
        gs = g[s]
        if prod:
            ga[s].scatter_add_(2, idx, gs * b[s].gather(1, idx))
            gb[s].scatter_add_(1, idx, gs * a[s].gather(2, idx))
        else:
            ga[s].scatter_add_(2, idx, gs)
            gb[s].scatter_add_(1, idx, gs)
    return out, ga, gb


def _band_rows(b, ld, width):
    """rows[:, p, j]: the band's cell of dense row p and column p - ld + j (0 where there is none)."""
    n = b.shape[1]
    j = torch.arange(width, device=b.device)
    col = torch.arange(n, device=b.device).unsqueeze(1) - ld + j
    ok = (col >= 0) & (col < n)
    return torch.where(ok, b[:, col.clamp(0, n - 1), (width - 1 - j).expand_as(col)], 0)


def _band_cells(rows, case):
    """Which cells of _band_rows are cells of the matrix."""
    col = torch.arange(case["n"], device=rows.device).unsqueeze(1) - case["b_ld"] + torch.arange(rows.shape[2], device=rows.device)
    return (col >= 0) & (col < case["n"])


def _band_terms(case):
    """(diagonal i of a, its columns, the dense rows they meet b in): out[c, i + j] takes a[c, i] and rows[c + i - a_lu, j]."""
    n = case["n"]
    for i in range(case["a_lu"] + case["a_ld"] + 1):
        shift = i - case["a_lu"]
        low, high = max(0, -shift), min(n, n - shift)
        if low < high:
            yield i, slice(low, high), slice(low + shift, high + shift)


def _best_band(a, rows, g, case):
    wb, cells = rows.shape[2], _band_cells(rows, case)
    best, at = torch.full_like(g, -1e9), torch.zeros_like(g, dtype=torch.int64)
    for i, cols, pos in _band_terms(case):
        terms = torch.where(cells[pos], a[:, cols, i : i + 1] + rows[:, pos], -2e9).float().double()
        old = best[:, cols, i : i + wb]
        at[:, cols, i : i + wb] = torch.where(terms > old, i, at[:, cols, i : i + wb])
        best[:, cols, i : i + wb] = torch.maximum(terms, old)
    ga, grows = torch.zeros_like(a), torch.zeros_like(rows)
    for i, cols, pos in _band_terms(case):
        won = torch.where((at[:, cols, i : i + wb] == i) & cells[pos], g[:, cols, i : i + wb], 0)
        ga[:, cols, i] = won.sum(2)
        grows[:, pos] += won
    # back from rows to columns: cell (c, k) of b lies in dense row c + k - b_lu
    n = case["n"]
    k = torch.arange(wb, device=a.device)
    row = torch.arange(n, device=a.device).unsqueeze(1) + k - case["b_lu"]
    ok = (row >= 0) & (row < n)
    gb = torch.where(ok, grows[:, row.clamp(0, n - 1), (wb - 1 - k).expand_as(row)], 0)
    return torch.where(best > -1e9, best, 0), ga, gb


def work(case):
    """Operations: a multiply-add (a compare and an add) per term and result for every sum a pass
    needs - log products: one forward, two backward, eight in the second order; max products:
    one forward, the gradients a scatter of g; the sample product: the forward's.  Bytes: operands and
    incoming gradients read once, results and gradients written once."""
    op, B = case["op"], case["B"]
    size = 4 if case["dtype"] == "float32" else 2
    if op in _BAND_OPS:
        wa, wb = case["a_lu"] + case["a_ld"] + 1, case["b_lu"] + case["b_ld"] + 1
        a, b, out = B * case["n"] * wa, B * case["n"] * wb, B * case["n"] * (wa + wb - 1)
        terms = B * case["n"] * wa * wb
    else:
        M, K, N = case["M"], case["K"], case["N"]
        a, b, out, terms = B * M * K, B * K * N, B * M * N, B * M * K * N
    if op == "second":
        return {"bytes": size * (4 * a + 4 * b + 3 * out), "flops": 2 * (1 + 2 + 8) * terms}
    sums = 3 if op in ("log", "band_log", "band_mul") else 1
    return {"bytes": size * (2 * a + 2 * b + 2 * out), "flops": 2 * sums * terms + (0 if sums == 3 else 2 * out)}


def tolerance(case):
    """Four times what the path differs by from itself in double precision on the same inputs."""
    op, dtype = case["op"], case["dtype"]
    if dtype == "bfloat16":         # 0.0012 (result), 0.0017 ... 0.009 (gradients, formed from a rounded result)
        return {"rel": 2e-2, "max": 0.8}
    if dtype == "float16":
        return {"rel": 3e-3, "max": 0.1}
    if op == "sample":
        # 5e-8 (result); a uniform within rounding of a partial sum draws the next term, which moves one
        # count of the gradients from a cell to its neighbour
        return {"rel": 2e-2, "max": 0.99}
    if op in ("log", "second"):     # 5e-8 (result), 4.7e-7 and 1.6e-5 at the largest of a gradient
        return {"rel": 2e-6, "max": 6e-5}
    return {"rel": 6e-7, "max": 1e-5}   # 1.5e-7 and 2.6e-6: sums of at most 512 products
