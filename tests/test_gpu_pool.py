"""Memory kept from destroyed factors, on the device: given back by trim, and a server's factors are
counted at what they hold whatever blocks the pool has (the pool itself is tested on the CPU in
test_pool.py)."""
import numpy as np
import pytest

from conftest import H, random_hss

pytestmark = pytest.mark.gpu


def test_trim_and_accounting(hip):
    import torch
    _, h = random_hss(np.random.default_rng(9), 16384, 64, 0, "cauchy", 1e-8)
    pack = H.pack(h)
    ctx = hip.Context(0)
    A = hip.HipHssMatrix(pack, ctx)

    def used():
        srv = hip.Server(1 << 30, prec="fp64", ctx=ctx)
        srv.admit(A)
        n = srv.used_bytes()
        srv.close()
        return n

    first = used()
    F = A.ulvfactor("fp64")
    size = F.device_bytes()
    assert first <= size <= first * (1 + 1 / 16) * (1 + 1 / 8) + 8192
    B = np.random.default_rng(1).standard_normal((16384, 2))
    X = F.solve(B)
    F.close()
    before = torch.cuda.mem_get_info()[0]
    ctx.trim()
    assert torch.cuda.mem_get_info()[0] - before >= size
    # the same count and the same bits with the pool empty, and with larger blocks in it
    assert used() == first
    _, h2 = random_hss(np.random.default_rng(10), 17000, 64, 0, "cauchy", 1e-8)
    hip.HipHssMatrix(H.pack(h2), ctx).ulvfactor("fp64").close()
    assert used() == first
    F = A.ulvfactor("fp64")
    assert np.array_equal(F.solve(B), X)
    F.close()
