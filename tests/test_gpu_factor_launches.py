"""The compact-WY blocks of the per-reflector kernel's nodes: adjacent levels in one launch, and
only those levels where the blocked kernel takes others."""
import numpy as np
import pytest

from conftest import H, rect_hss
from test_gpu_factor_sizes import EPS, dominant, rel

pytestmark = pytest.mark.gpu


def records(hip, A, prec):
    hip.prof_reset()
    hip.prof_enable(True)
    try:
        F = A.ulvfactor(prec)
        return F, hip.prof_records()
    finally:
        hip.prof_enable(False)
        hip.prof_reset()


def of(recs, kernel):
    return [(r["level"], r["nwork"]) for r in recs if r["kernel"] == kernel]


@pytest.mark.parametrize("ms,ku,kv,prec,wy", [
    ([40] * 8, 6, 5, "fp32", [(0, 14)]),    # every level: 8 + 4 + 2 nodes
    ([128] * 4, 8, 70, "fp64", [(0, 4)]),   # 198 rows of [D; V'] at the leaves, 86 above
    ([40] * 8, 6, 5, "fp64", []),
])
def test_wy_launches(hip, oracle, ms, ku, kv, prec, wy):
    rng = np.random.default_rng(sum(ms) + kv)
    nodes, blob = H.pack(dominant(rect_hss(rng, ms, ms, ku, kv), 4.0 * ku * kv * np.sqrt(max(ms))))
    n = sum(ms)
    F, recs = records(hip, hip.HipHssMatrix((nodes, blob)), prec)
    assert of(recs, "k_ulv_wy") == wy
    B = rng.standard_normal((n, 3))
    Xo = oracle.ulvfactsolve(nodes, blob, B)
    cond = np.linalg.cond(oracle.matmul(nodes, blob, np.eye(n)))
    if prec == "fp64":
        assert rel(F.solve(B), Xo) <= 50 * cond * EPS
    else:
        X = F.solve(B, tol=1e-12, max_iter=30)
        assert rel(X, Xo) <= 50 * cond * EPS + 1e-12 * cond
    F.close()
