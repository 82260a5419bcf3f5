"""The factor and operator-forming kernels at the edges of their tiles: leaf sizes around the
16-row MFMA tiles, the 64-row builds and the 128-row limit, ranks around 16 and 32, leaves that
pass through (rank >= rows), and roots on either side of the LDS build (143 rows in Float64);
the refined solve's residual around its 4096-row chunks.  Random generators, D made dominant,
against the CPU oracle: two backward-stable solvers differ by at most about cond(A) eps, held to
50 cond eps as the golden fixtures are, with cond from the dense expansion."""
import numpy as np
import pytest

from conftest import H, random_hss, rect_hss

pytestmark = pytest.mark.gpu
EPS = 2.220446049250313e-16


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def dominant(h, s):
    """Adds s to the diagonal of every leaf block."""
    if h.leafnode:
        h.D += s * np.eye(h.D.shape[0])
    else:
        dominant(h.A11, s)
        dominant(h.A22, s)
    return h


SIZES = [  # leaf rows, ku, kv
    ([16, 16, 16, 16], 3, 3),
    ([17, 15, 16, 33], 5, 4),
    ([64, 64, 64, 64], 16, 16),
    ([65, 63, 64, 66], 17, 15),
    ([128, 128, 127, 128], 33, 20),
    ([96, 113, 128, 97], 48, 31),
    ([20, 20, 40, 40], 24, 8),       # the first two leaves pass through
    ([64, 64], 60, 30),              # root of 120 rows
    ([150], 0, 0),                   # the root alone: in memory
    ([143], 0, 0),                   # and in LDS
    ([50, 1, 40, 2], 1, 1),
]


@pytest.mark.parametrize("ms,ku,kv", SIZES)
def test_factor_sizes(hip, oracle, ms, ku, kv):
    rng = np.random.default_rng(sum(ms) + 7 * ku + kv)
    h = dominant(rect_hss(rng, ms, ms, ku, kv), 4.0 * ku * kv * np.sqrt(max(ms)))
    nodes, blob = H.pack(h)
    n = sum(ms)
    B = rng.standard_normal((n, 5))
    Xo = oracle.ulvfactsolve(nodes, blob, B)
    cond = np.linalg.cond(oracle.matmul(nodes, blob, np.eye(n)))
    A = hip.HipHssMatrix((nodes, blob))
    F = A.ulvfactor("fp64")
    assert rel(F.solve(B), Xo) <= 50 * cond * EPS
    F.close()
    # batched with itself: the same operators whatever shares the launches
    Fs = hip.ulvfactor_batch([A, A], "fp64")
    for f in Fs:
        assert rel(f.solve(B), Xo) <= 50 * cond * EPS
        f.close()
    F = A.ulvfactor("fp32")
    X, rep = F.solve(B, tol=1e-10, max_iter=30, report=True)
    F.close()
    R = oracle.matmul(nodes, blob, X) - B
    assert np.max(np.linalg.norm(R, axis=0) / np.linalg.norm(B, axis=0)) <= 1e-10


@pytest.mark.parametrize("n,nrhs", [(4095, 1), (4096, 3), (4097, 2)])
def test_refined_residual_chunks(hip, oracle, n, nrhs):
    rng = np.random.default_rng(n)
    _, h = random_hss(rng, n, 128, 0, "cauchy", 1e-8)
    nodes, blob = H.pack(dominant(h, 8.0 * n))
    B = rng.standard_normal((n, nrhs))
    A = hip.HipHssMatrix((nodes, blob))
    F = A.ulvfactor("fp32")
    X, rep = F.solve(B, tol=1e-10, max_iter=20, report=True)
    F.close()
    R = oracle.matmul(nodes, blob, X) - B
    worst = float(np.max(np.linalg.norm(R, axis=0) / np.linalg.norm(B, axis=0)))
    assert worst <= 1e-10
    # the reported residual is this one, to the rounding of both products (a few eps ||A|| ||x|| / ||b||)
    assert abs(rep["rel_residual"] - worst) <= 1e-13


def test_pool_reuse(hip, oracle, c1):
    """Factors of other sizes in the memory of closed ones: the same bits as the first time."""
    nodes, blob = c1["nodes"], c1["blob"]
    rng = np.random.default_rng(3)
    A = hip.HipHssMatrix((nodes, blob))
    B = rng.standard_normal((2001, 4))
    h = dominant(rect_hss(rng, [64, 60, 50, 64], [64, 60, 50, 64], 9, 7), 4000.0)
    A2 = hip.HipHssMatrix(H.pack(h))
    first = A.solve(B)
    keep = A.ulvfactor("fp64")
    for _ in range(3):
        A2.solve(rng.standard_normal((238, 3)))
        F = A.ulvfactor("fp64")
        assert np.array_equal(F.solve(B), first)
        F.close()
        assert np.array_equal(A.solve(B), first)
    assert np.array_equal(keep.solve(B), first)
    keep.close()
