"""Rounding of the product Y' D in the ULV factor (Y the reflectors of U, D a leaf's block): with
D = c 11' + I and U = 1, every term of a column's sum is the same number t, and the reflector takes
all of c 11' out of the rows that are eliminated, so an error of p eps in the sums is an error of
about p cond(A) eps in the solution.  With t = 1 the additions are exact, which gives the error of
everything else (the reflector's scale and tau, the update with Y).  t = 1 + f 2^-46 makes each
addition to a partial sum in [64 t, 128 t) round the same way by up to half a unit: one running sum
over the 128 rows adds up to 14 eps.  Partial sums of 16 rows lose at most 2.7 eps in the sums
and 1.5 in adding them up."""
import numpy as np
import pytest

from conftest import H

pytestmark = pytest.mark.gpu
EPS = 2.220446049250313e-16


def solution(A, b):
    """A \\ b, refined with residuals in extended precision."""
    x = np.linalg.solve(A, b).astype(np.longdouble)
    Al, bl = A.astype(np.longdouble), b.astype(np.longdouble)
    for _ in range(5):
        x += np.linalg.solve(A, (bl - Al @ x).astype(np.float64))
    return x


def error(hip, f):
    """Error of A \\ 1 with terms t = 1 + f 2^-46, in units of cond(A) eps."""
    m = 128
    scale = 1.0 / (1.0 + np.sqrt(float(m)))  # the reflector of U = 1 is [scale, .., scale, 1]
    c = (1.0 + f * 2.0 ** -46) / scale
    one = np.ones((m, 1))
    leaf = lambda: H.HssMatrix(D=np.full((m, m), c) + np.eye(m), U=one, V=one)
    half = np.full((1, 1), 0.5)
    h = H.HssMatrix(A11=leaf(), A22=leaf(), B12=half, B21=half, rootnode=True)
    A = H.full(h)
    b = np.ones((2 * m, 1))
    x = solution(A, b)
    err = float(np.linalg.norm(hip.HipHssMatrix(H.pack(h)).solve(b) - x) / np.linalg.norm(x))
    return err / (np.linalg.cond(A) * EPS)


@pytest.mark.parametrize("f", [0.1, 0.2, 0.3, 0.4, 0.45, 0.49, 0.6, 0.7, 0.8])
def test_sums_of_the_reflector_product(hip, f):
    assert error(hip, f) <= error(hip, 0.0) + 4.2
