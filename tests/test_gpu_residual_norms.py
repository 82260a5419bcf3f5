"""The relative residual that refinement decides by, where it is large enough to be told from
rounding: a Float32 factor's first solve (about 1e-7 on these diagonally dominant matrices), against
the oracle's product.  Both products are off by about 1e-15, so 1e-5 of the value holds them, and a
lost row of 8193 moves it by 6e-5.  Rows around the chunks of the single solve (4096) and around
the batch's thread counts (256 and 1024 threads, four rows each; the choice at 2048 rows on average)."""
import numpy as np
import pytest

from conftest import H
from test_gpu_factor_sizes import dominant

pytestmark = pytest.mark.gpu
SCALE = np.array([1.0, 1e8, 1e-6])
_made = {}


def matrix(n):
    if n not in _made:
        # 1/(x - y) on an even grid: entries of at most n/2, so 8 n on the diagonal dominates
        K = H.KernelMatrix(np.linspace(-1.0, 1.0, n), "cauchy", 1.0)
        rcl = H.bisection_cluster(n, 128)
        _made[n] = H.pack(dominant(H.compress(K, rcl, rcl, 1e-6, 1e-6), 8.0 * n))
    return _made[n]


def relres(oracle, pack, X, B):
    R = oracle.matmul(*pack, X) - B
    return np.linalg.norm(R, axis=0) / np.linalg.norm(B, axis=0)


@pytest.mark.parametrize("n", [300, 4096, 4097, 8193])
def test_single(hip, oracle, n):
    pack = matrix(n)
    B = np.random.default_rng(n).standard_normal((n, 3)) * SCALE
    F = hip.HipHssMatrix(pack).ulvfactor("fp32")
    for cols in ([0, 1, 2], [0], [1], [2]):
        X, rep = F.solve(B[:, cols], tol=1e-3, max_iter=5, report=True)
        assert rep["iterations"] == 0
        want = relres(oracle, pack, X, B[:, cols]).max()
        assert 1e-9 < want < 1e-5
        assert abs(rep["rel_residual"] - want) <= 1e-5 * want
    F.close()


@pytest.mark.parametrize("ns", [[255], [1024], [1025], [2048], [2049], [4097], [8193], [300, 8193], [256] * 9 + [8193]])
def test_batch(hip, oracle, ns):
    import torch
    packs = [matrix(n) for n in ns]
    A = [hip.HipHssMatrix(p) for p in packs]
    rng = np.random.default_rng(sum(ns))
    B = [rng.standard_normal((n, 3)) * SCALE for n in ns]
    Bt = [torch.from_numpy(np.ascontiguousarray(b.T)).to("cuda:0") for b in B]
    X = [torch.zeros_like(b) for b in Bt]
    torch.cuda.synchronize()
    F = hip.ulvfactor_batch(A, "fp32")
    ptr = lambda ts: [t.data_ptr() for t in ts]
    plan = hip.Plan(F, [3] * len(ns), ptr(Bt), ns, ptr(X), ns, refinement=True)

    def worst():
        torch.cuda.synchronize()
        return max(relres(oracle, p, x.cpu().numpy().T, b).max() for p, x, b in zip(packs, X, B))

    rep = plan.execute(tol=1e-3)
    assert rep["iterations"] == 0
    want = worst()
    assert 1e-9 < want < 1e-5
    assert abs(rep["rel_residual"] - want) <= 1e-5 * want
    rep = plan.execute(tol=1e-12)  # x += d of every row
    assert rep["iterations"] >= 1 and worst() <= 1e-12
    plan.close()
