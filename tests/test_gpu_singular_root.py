"""Singular roots of more than one row and a branch: the root's LU stops at the first zero (or
NaN) pivot, and the kernel that forms the root's inverse, enqueued behind it, still applies every
row exchange, so all of them have to be in range.  Pass-through leaves (ku = m) make the root block
diag(D1, D2), so the failing column is known."""
import numpy as np
import pytest

from conftest import H, rect_hss

pytestmark = pytest.mark.gpu


def diagonal_root(half, bad=None, value=0.0):
    d = np.arange(1.0, 2 * half + 1)
    if bad is not None:
        d[bad] = value
    eye, z = np.eye(half), np.zeros((half, half))
    a = H.HssMatrix(D=np.diag(d[:half]), U=eye, V=eye)
    b = H.HssMatrix(D=np.diag(d[half:]), U=eye, V=eye)
    return d, H.HssMatrix(A11=a, A22=b, B12=z, B21=z, rootnode=True)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("half", [2, 17, 64])
def test_singular_root_column(hip, half, prec):
    d, h = diagonal_root(half)
    good = hip.HipHssMatrix(H.pack(h))
    rng = np.random.default_rng(half)
    b = rng.standard_normal((2 * half, 3))
    # blocks of this size in the memory pool that hold another factor's data
    for _ in range(2):
        other = hip.HipHssMatrix(H.pack(rect_hss(rng, [half, half], [half, half], half, half)))
        other.ulvfactor(prec).close()
    for bad in (0, half - 1, half, 2 * half - 1):
        for value in (0.0, np.nan):
            A = hip.HipHssMatrix(H.pack(diagonal_root(half, bad, value)[1]))
            with pytest.raises(H.SingularException, match=rf"\({bad + 1}\)"):
                A.ulvfactor(prec)
            with pytest.raises(H.SingularException, match=rf"\({bad + 1}\).*matrix 1"):
                hip.ulvfactor_batch([good, A], prec)
    F = good.ulvfactor(prec)
    X = F.solve(b, tol=1e-14, max_iter=10) if prec == "fp32" else F.solve(b)
    F.close()
    # diagonal systems: a division and, in Float32, refinement to 1e-14
    assert np.max(np.abs(X - b / d[:, None]) * d[:, None]) <= 1e-13 * np.max(np.abs(b))
