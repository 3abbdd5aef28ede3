"""The front program of the LU (csrc/fronts.h) where it can go wrong: fronts at
the edges of their 8-row tiles and at the largest size, one row more (the band
programs take over), source singletons of both kinds, a supply row longer than
one chunk, chains, and packed blocks.  The CPU tests check the program and its
CPU execution against numpy; the GPU tests compare factors and solutions bit for
bit with that execution, which runs the same operations in the same order (a
quotient by reciprocal and exact-remainder correction is the rounded quotient)."""

import numpy as np
import pytest

from vajax_amd.sparse import SparseLU


def _csr(A):
    ip = np.concatenate([[0], np.cumsum((A != 0).sum(axis=1))]).astype(np.int32)
    return ip, np.nonzero(A)[1].astype(np.int32), A[A != 0]


def _dense(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(-1, 1, (n, n)) + n * np.eye(n)


def _arrow(blocks, k, border, seed):
    """`blocks` dense blocks of k rows, each coupled to a dense border."""
    n = blocks * k + border
    A = np.zeros((n, n))
    b0 = blocks * k
    rng = np.random.default_rng(seed)
    for i in range(blocks):
        s = slice(i * k, (i + 1) * k)
        A[s, s] = rng.uniform(-1, 1, (k, k))
        A[s, b0:] = rng.uniform(-1, 1, (k, border))
        A[b0:, s] = rng.uniform(-1, 1, (border, k))
    A[b0:, b0:] = rng.uniform(-1, 1, (border, border))
    return A + (k + border) * blocks * np.eye(n)


def _sources(n, seed):
    """A ladder of n nodes with a grounded source at one end and a rail: nodes
    0..n-1, rail n, branch rows n+1 (node 0) and n+2 (rail)."""
    rng = np.random.default_rng(seed)
    A = np.zeros((n + 3, n + 3))

    def g(i, j, v):
        A[i, i] += v
        A[j, j] += v
        A[i, j] -= v
        A[j, i] -= v * 1.5  # unsymmetric

    for i in range(n - 1):
        g(i, i + 1, rng.uniform(1e-3, 1e-2))
    for i in range(n):
        g(i, n, rng.uniform(1e-4, 1e-3))
        A[i, i] += 1e-12
    for node, br in ((0, n + 1), (n, n + 2)):
        A[node, br] = A[br, node] = 1.0
    return A


CASES = {f"dense{n}": (lambda n=n: _dense(n, n)) for n in (1, 2, 7, 8, 9, 16, 17, 24, 25, 31, 32, 33,
                                                          40, 41, 57, 63, 64, 65)}
CASES.update({
    "arrow8x20+24": lambda: _arrow(8, 20, 24, 1),
    "arrow40x9+31": lambda: _arrow(40, 9, 31, 2),
    "arrow130x3+5": lambda: _arrow(130, 3, 5, 3),
    "arrow6x40+24": lambda: _arrow(6, 40, 24, 4),
    "diagonal": lambda: np.diag(np.arange(1.0, 30.0)),
    "sources1": lambda: _sources(1, 5),
    "sources40": lambda: _sources(40, 6),
    "sources5000": None,  # the rail's row takes two chunks
})


def _case(name):
    if name != "sources5000":
        return _csr(CASES[name]())
    n = 5000
    rng = np.random.default_rng(7)
    rows, cols, vals = [], [], []

    def add(i, j, v):
        rows.append(i), cols.append(j), vals.append(v)

    for i in range(n):
        add(i, i, 3e-2 + rng.uniform(0, 1e-3))
        if i + 1 < n:
            v = rng.uniform(1e-3, 1e-2)
            add(i, i + 1, -v), add(i + 1, i, -1.5 * v)
        add(i, n, -1e-4), add(n, i, -2e-4)
    add(n, n, 1.0), add(n, n + 1, 1.0), add(n + 1, n, 1.0)
    order = np.lexsort((cols, rows))
    r = np.array(rows)[order]
    ip = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n + 2))]).astype(np.int32)
    return ip, np.array(cols, np.int32)[order], np.array(vals)[order]


def _residual(ip, ix, a, x, b):
    r = np.add.reduceat(a * x[ix], ip[:-1]) - b
    scale = np.add.reduceat(np.abs(a * x[ix]), ip[:-1]) + np.abs(b)
    return float(np.max(np.abs(r) / scale))


@pytest.mark.parametrize("name", list(CASES))
def test_front_program_on_the_cpu(name):
    ip, ix, a = _case(name)
    lu = SparseLU(ip, ix)
    lu.analyze(a)
    lu.check_schedules()
    b = np.random.default_rng(3).standard_normal(len(ip) - 1)
    # diagonally weighted matrices: componentwise backward error of a few eps
    # per row entry
    assert _residual(ip, ix, a, lu.solve_cpu(a, b), b) <= 65 * 2.3e-16 * 4
    assert _residual(ip, ix, a, lu.solve_cpu(a, b, 1), b) <= 65 * 6e-8 * 4


@pytest.mark.parametrize("rows,front", [(64, True), (65, False)])
def test_later_analyses_of_a_handle_keep_its_kind_of_program(rows, front):
    ip, ix, a = _csr(_dense(rows, 9))
    lu = SparseLU(ip, ix)
    b = np.random.default_rng(3).standard_normal(rows)
    for width in (None, None, 8):  # a setter between the second and the third
        if width:
            lu.set_band_width(width)
        lu.analyze(a)
        lu.check_schedules()
        assert (lu.info()["fact_task_targets"] == 0) == front
        assert _residual(ip, ix, a, lu.solve_cpu(a, b), b) <= 65 * 2.3e-16 * 4
        a = a * np.random.default_rng(4).uniform(0.9, 1.1, len(a))


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_front_program_matches_its_cpu_execution(name):
    import torch

    print(name, flush=True)
    ip, ix, a = _case(name)
    n = len(ip) - 1
    lu = SparseLU(ip, ix)
    lu.analyze(a)
    a2 = a * np.random.default_rng(4).uniform(0.9, 1.1, len(a))
    d = torch.as_tensor(a2, device="cuda")
    b = np.random.default_rng(5).standard_normal(n)
    bd = torch.as_tensor(b, device="cuda")
    x = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
    for _ in range(2):  # the second pass starts from the first one's leftovers
        assert lu.refactor(d, 0) == 0
        lu.solve(d, bd, x, 0)
        assert np.array_equal(lu.download(), lu.refactor_cpu(a2, 0))
        assert np.array_equal(x.cpu().numpy(), lu.solve_cpu(a2, b, 0))
    assert lu.refactor(d, 1) == 0
    lu.solve(d, bd, x, 2)
    assert _residual(ip, ix, a2, x.cpu().numpy(), b) <= 65 * 2.3e-16 * 4
    # the right-hand side's buffer takes the solution
    lu.refactor(d, 0)
    lu.solve(d, bd, x, 0)
    lu.solve(d, bd, bd, 0)
    assert torch.equal(x, bd)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 0.0])
def test_bad_pivots_are_reported(bad):
    """A zero pivot, an infinite or a NaN entry reach the pivot monitor."""
    import torch

    from vajax_amd import _lib as L

    for name in ("dense9", "arrow6x40+24", "sources40"):
        print(name, bad, flush=True)
        ip, ix, a = _case(name)
        lu = SparseLU(ip, ix)
        lu.analyze(a)
        a2 = a.copy()
        if bad == 0.0:
            a2[:] = 0.0
        else:
            a2[len(a2) // 2] = bad
        assert lu.refactor(torch.as_tensor(a2, device="cuda"), 0) == L.VJX_WARN_PIVOT
        assert lu.refactor(torch.as_tensor(a, device="cuda"), 0) == 0
