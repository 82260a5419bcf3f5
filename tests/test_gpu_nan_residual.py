"""A solve whose residual is NaN has not converged: the refined single solve (both correction
methods), the batched plan and the server say so alike, and the other columns and requests are
refined as if it were not there."""
import numpy as np
import pytest

from conftest import H, random_hss

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def problem():
    _, h = random_hss(np.random.default_rng(5), 600, 64, 0, "cauchy", 1e-8)
    rng = np.random.default_rng(6)
    return H.pack(h), rng.standard_normal((600, 3))


def residuals(oracle, nodes, blob, X, B):
    R = oracle.matmul(nodes, blob, X) - B
    return np.linalg.norm(R, axis=0) / np.linalg.norm(B, axis=0)


@pytest.mark.parametrize("method", ["ir", "gmres"])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_nan_column_single(hip, oracle, problem, prec, method):
    import torch
    (nodes, blob), B = problem
    F = hip.HipHssMatrix((nodes, blob)).ulvfactor(prec)
    Bn = B.copy()
    Bn[17, 1] = np.nan
    with pytest.raises(hip.NotConverged):
        F.solve(Bn, tol=1e-10, max_iter=4, method=method)
    with pytest.raises(hip.NotConverged):
        F.solve(np.full((600, 1), np.nan), tol=1e-10, max_iter=4, method=method)
    Bt = torch.from_numpy(np.ascontiguousarray(Bn.T)).to("cuda:0")
    X = torch.zeros_like(Bt)
    torch.cuda.synchronize()
    with pytest.raises(hip.NotConverged):
        F.solve_dev(3, Bt.data_ptr(), 600, X.data_ptr(), 600, tol=1e-10, max_iter=4, method=method)
    torch.cuda.synchronize()
    good = [0, 2]
    assert np.max(residuals(oracle, nodes, blob, X.cpu().numpy().T[:, good], B[:, good])) <= 1e-10


def test_nan_from_the_factor(hip):
    """A leaf whose eliminated block is exactly zero: its L has a zero diagonal, and only the root's
    pivots are looked at."""
    rng = np.random.default_rng(7)
    u = rng.standard_normal((8, 2))
    a = H.HssMatrix(D=np.zeros((8, 8)), U=u, V=u)
    b = H.HssMatrix(D=np.eye(8), U=u, V=u)
    h = H.HssMatrix(A11=a, A22=b, B12=np.eye(2), B21=np.eye(2), rootnode=True)
    A = hip.HipHssMatrix(H.pack(h))
    with pytest.raises((hip.NotConverged, H.SingularException)):
        A.ulvfactor("fp32").solve(np.ones((16, 1)), tol=1e-10, max_iter=3)


def test_nan_request_in_plan_and_server(hip, oracle, problem):
    import torch
    (nodes, blob), B = problem
    A = hip.HipHssMatrix((nodes, blob))
    Bt = torch.from_numpy(np.ascontiguousarray(B.T)).to("cuda:0")
    Bn = Bt.clone()
    Bn[1, 5] = float("nan")
    Xt, Xn = torch.zeros_like(Bt), torch.zeros_like(Bt)
    torch.cuda.synchronize()
    F = [A.ulvfactor("fp32"), A.ulvfactor("fp32")]
    ptr = lambda *t: [x.data_ptr() for x in t]
    plan = hip.Plan(F, [3, 3], ptr(Bn, Bt), [600, 600], ptr(Xn, Xt), [600, 600], refinement=True)
    with pytest.raises(hip.NotConverged):
        plan.execute(tol=1e-10, max_iter=4)
    torch.cuda.synchronize()
    assert np.max(residuals(oracle, nodes, blob, Xt.cpu().numpy().T, B)) <= 1e-10
    plan.close()
    srv = hip.Server(1 << 30, prec="fp32", tol=1e-10, max_iter=4, max_inflight=4)
    mid = srv.admit(A)
    Xt.zero_()
    torch.cuda.synchronize()
    tn = srv.submit(mid, 3, Bn.data_ptr(), 600, Xn.data_ptr(), 600)
    tg = srv.submit(mid, 3, Bt.data_ptr(), 600, Xt.data_ptr(), 600)
    while srv.step() > 0:
        pass
    rn, rg = srv.poll(tn), srv.poll(tg)
    assert rn["status"] == 2 and np.isnan(rn["rel_residual"])
    assert rg["status"] == 1 and rg["rel_residual"] <= 1e-10
    torch.cuda.synchronize()
    assert np.max(residuals(oracle, nodes, blob, Xt.cpu().numpy().T, B)) <= 1e-10
    srv.close()
