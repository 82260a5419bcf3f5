"""The root's LU in memory (a root block too large for LDS), in each of its builds: few roots,
more than an XCD's L2 holds, and one for every CU; a root-only matrix is its own root.  Against
numpy, held to the growth-free bound of partial pivoting, m eps cond; singular columns are reported
from each build."""
import numpy as np
import pytest

from conftest import H

pytestmark = pytest.mark.gpu
EPS = 2.220446049250313e-16

CASES = [("fp64", 144, 1), ("fp64", 300, 2), ("fp64", 300, 64), ("fp64", 200, 136), ("fp64", 193, 250),
         ("fp32", 203, 1), ("fp32", 320, 88), ("fp32", 257, 136)]


def root(D):
    return H.pack(H.HssMatrix(D=D, rootnode=True))


@pytest.mark.parametrize("prec,m,count", CASES)
def test_root_lu(hip, prec, m, count):
    rng = np.random.default_rng(m + count)
    Ds = [rng.standard_normal((m, m)) for _ in range(min(count, 3))]
    mats = [hip.HipHssMatrix(root(D)) for D in Ds]
    b = rng.standard_normal((m, 2))
    facts = hip.ulvfactor_batch([mats[i % len(mats)] for i in range(count)], prec)
    for i in sorted({0, 1, 2, count // 2, count - 1} & set(range(count))):
        D = Ds[i % len(Ds)]
        x = facts[i].solve(b, tol=1e-12, max_iter=40) if prec == "fp32" else facts[i].solve(b)
        want = np.linalg.solve(D, b)
        assert np.linalg.norm(x - want) <= (m * EPS + (1e-12 if prec == "fp32" else 0.0)) * np.linalg.cond(D) * np.linalg.norm(want)
    for f in facts:
        f.close()


@pytest.mark.parametrize("prec,m,count", CASES)
def test_singular_root_in_memory(hip, prec, m, count):
    d = np.arange(1.0, m + 1)
    good = hip.HipHssMatrix(root(np.diag(d)))
    for bad in (0, m // 2, m - 1):
        e = d.copy()
        e[bad] = 0.0
        A = hip.HipHssMatrix(root(np.diag(e)))
        with pytest.raises(H.SingularException, match=rf"\({bad + 1}\).*matrix {count - 1}"):
            hip.ulvfactor_batch([good] * (count - 1) + [A], prec)
