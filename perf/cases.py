"""The work that is timed: HSS products and ULV solves as a program calls them.

A case is a dict of plain values:

  op       "matvec"     C = alpha A B + beta C on device arrays (mul!, src/matmul.jl:18)
           "solve"      X = A \\ B with a resident Float64 factor, device arrays
           "mixed"      X = A \\ B with a resident Float32 factor refined to 1e-10 in Float64
           "backslash"  X = A \\ B from the matrix alone: factor, solve, release
                        (ulvfactsolve, src/ulvfactor.jl:10), device arrays
           "ldiv"       the same from and to host arrays, the call hssA \\ b itself
           "batch"      many matrices of uneven size solved together by a kept plan
           "factors"    many matrices of uneven size factored together, solved once, released
           "serve"      requests on resident Float32 factors through the serving loop
  kernel   "log": log|x - y| on sorted uniform points of [-1, 1]; "cauchy": 1/(x - y) on points as
           `grid` says
  diag     the diagonal: 1, or for solves with the log kernel -24, past the logarithm of the
           closest pairs (a regularised fit): with 1 some point sets give a matrix so close to
           singular that no two correct solves agree and a Float32 factor does not refine
  n        size of the matrix (of the largest one where there are many)
  nrhs     right-hand sides (the most of one request where there are many)

The matrices are HSS approximations of kernel matrices, built here from the points alone
(nested skeletons of kernel columns sampled near and far), so that both sides of a comparison
get the same generators whatever the library's own compressors do.
"""
from __future__ import annotations

import importlib
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parents[1]
PKG = "hssmatrices_jl_amd"


def listed():
    log = dict(kernel="log", tol=1e-9, grid="uniform", diag=-24.0)
    c1 = dict(kernel="cauchy", n=2001, leaf=64, tol=1e-6, grid="even", diag=1.0, nrhs=1)
    many = dict(kernel="cauchy", n=16384, low=1024, count=32, leaf=64, tol=1e-8, grid="spread", diag=1.0, nrhs=32)
    return [
        # the Cauchy kernel on a 2001-point grid, the reference's test matrix, with one vector:
        # the smallest calls, where launches and latency are what a caller waits for
        dict(c1, name="matvec-cauchy-2001", op="matvec", alpha=1.0, beta=0.0),
        dict(c1, name="solve-cauchy-2001", op="solve"),
        # hssA \\ b on that matrix as the reference is called: host vector in, host vector out
        dict(c1, name="ldiv-cauchy-2001", op="ldiv"),
        # a ragged size with a few vectors, updating C (mul! with alpha and beta)
        dict(log, name="update-log-23171", op="matvec", n=23171, leaf=64, nrhs=7, diag=1.0, alpha=-1.0, beta=0.5),
        # one right-hand side against a large resident factor, as inside an outer iteration
        dict(log, name="solve-log-40009", op="solve", n=40009, leaf=128, nrhs=1),
        # the n = 65536 log kernel with a block of 64 vectors: product, solve with the resident
        # factor, and factor + solve
        dict(log, name="matvec-log-65536", op="matvec", n=65536, leaf=128, nrhs=64, diag=1.0, alpha=1.0, beta=0.0),
        dict(log, name="solve-log-65536", op="solve", n=65536, leaf=128, nrhs=64),
        dict(log, name="backslash-log-65536", op="backslash", n=65536, leaf=128, nrhs=64),
        # mixed precision on the same matrix, the largest block
        dict(log, name="mixed-log-65536", op="mixed", n=65536, leaf=128, nrhs=128),
        # uneven Cauchy instances: solved together by a kept plan, and factored together
        dict(many, name="batch-cauchy-32", op="batch"),
        dict(many, name="factors-cauchy-32", op="factors"),
        # a burst of requests on resident Float32 factors
        dict(log, name="serve-log-16", op="serve", n=32768, low=4096, count=6, requests=16, leaf=128, nrhs=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: any operation, size, width and leaf size of them."""
    op = rng.choice(["matvec", "matvec", "solve", "solve", "backslash", "mixed", "ldiv", "batch", "factors", "serve"])
    c = dict(op=op, kernel="log", n=_log_int(rng, 2001, 65536), leaf=rng.choice([64, 96, 128]), tol=1e-9, grid="uniform",
             diag=-24.0, nrhs=_log_int(rng, 1, 64))
    if op == "matvec":
        c.update(diag=1.0, alpha=rng.choice([1.0, -1.0]), beta=rng.choice([0.0, 0.5]))
        if rng.random() < 0.5:
            c.update(kernel="cauchy", grid=rng.choice(["even", "spread"]), tol=rng.choice([1e-6, 1e-8]))
    elif op == "mixed":
        c.update(nrhs=_log_int(rng, 1, 128))
    elif op == "ldiv":
        c.update(n=_log_int(rng, 1024, 8192), nrhs=_log_int(rng, 1, 16))
    elif op in ("batch", "factors"):
        c.update(kernel="cauchy", diag=1.0, grid="spread", tol=1e-8, n=_log_int(rng, 4096, 16384), low=1024,
                 count=rng.randint(8, 32), leaf=64, nrhs=_log_int(rng, 4, 32))
    elif op == "serve":
        c.update(n=_log_int(rng, 8192, 32768), low=4096, count=rng.randint(2, 6), requests=rng.randint(4, 16), leaf=128,
                 nrhs=_log_int(rng, 2, 32))
    return c


# ---------------------------------------------------------------------------
# trees and generators
# ---------------------------------------------------------------------------
def _tree(n, leaf):
    """Breadth-first bisection tree: [start, stop, left, right, parent, depth] a node (a range
    longer than `leaf` is split after its first half, rounded up)."""
    nodes = [[0, n, -1, -1, -1, 0]]
    i = 0
    while i < len(nodes):
        a, b, d = nodes[i][0], nodes[i][1], nodes[i][5]
        if b - a > leaf:
            h = a + (b - a + 1) // 2
            nodes[i][2], nodes[i][3] = len(nodes), len(nodes) + 1
            nodes.append([a, h, -1, -1, i, d + 1])
            nodes.append([h, b, -1, -1, i, d + 1])
        i += 1
    return nodes


def _points(case, n, rng):
    if case["grid"] == "even":
        return np.linspace(-1.0, 1.0, n)
    if case["grid"] == "spread":  # one point a cell, no two closer than a twentieth of a cell; shifted
        return (np.arange(n) + 0.025 + 0.95 * rng.random(n)) * (2.0 / n) - 1.0 + 0.5 * rng.random()
    return np.sort(rng.uniform(-1.0, 1.0, n))


def _kernel(kind, d, diag):
    """Entries of the kernel at differences d = x - y; a zero difference is the diagonal."""
    z = d == 0
    v = torch.where(z, torch.ones_like(d), d)
    v = torch.log(v.abs()) if kind == "log" else torch.reciprocal(v)
    return torch.where(z, torch.full_like(d, diag), v)


def _offsets(n, near, ratio):
    """Distances 1, 2, .. `near`, then geometric ones up to n."""
    o = list(range(1, near + 1))
    while o[-1] < n:
        o.append(max(o[-1] + 1, int(o[-1] * ratio)))
    return torch.tensor(o[:-1] if len(o) > near else o)


def _interpolate(Y, tol):
    """Y (nodes x rows x columns; unused rows zero): each node's skeleton rows, chosen by row
    pivoting until the largest remaining row is at most tol times the first, and U with
    Y ~ U Y[skeleton].  Returns (pivots, U, ranks)."""
    N, c, _ = Y.shape
    Y = Y.clone()
    at = torch.arange(N, device=Y.device)
    rank = torch.zeros(N, dtype=torch.long, device=Y.device)
    live = torch.ones(N, dtype=torch.bool, device=Y.device)
    first, piv, low = None, [], []
    for _ in range(c):
        n2 = (Y * Y).sum(2)
        big, p = n2.max(1)
        big = big.sqrt()
        first = big if first is None else first
        live = live & (big > tol * first)
        if not bool(live.any()):
            break
        q = Y[at, p] * (live / big.clamp_min(1e-300))[:, None]
        t = torch.bmm(Y, q[:, :, None].contiguous())[:, :, 0]
        Y = Y - t[:, :, None] * q[:, None, :]
        Y[at, p] = torch.where(live[:, None], torch.zeros_like(q), Y[at, p])
        piv.append(p)
        low.append(t)
        rank += live
    piv, L = torch.stack(piv, 1), torch.stack(low, 2)
    k = L.shape[2]
    Lp = torch.gather(L, 1, piv[:, :, None].expand(-1, -1, k)).tril()
    on = torch.arange(k, device=Y.device)[None] < rank[:, None]
    Lp = torch.where(on[:, :, None] & on[:, None, :], Lp, torch.zeros_like(Lp)) + torch.diag_embed((~on).to(Lp.dtype))
    U = torch.linalg.solve_triangular(Lp, L, upper=False, left=False)
    return piv, U, rank


class Matrix:
    """Generators of one HSS matrix: the node list with D, U, V, B12, B21, R, W on the host."""

    def __init__(self, n, nodes):
        self.n, self.nodes = n, nodes
        self.gen = [dict() for _ in nodes]
        self.ku = [0] * len(nodes)
        self.kv = [0] * len(nodes)

    def entries(self):
        return sum(a.size for g in self.gen for a in g.values())


def _build(kind, points, leaf, tol, diag, device):
    """The HSS matrices of the given point sets, all levels of all of them together."""
    mats = [Matrix(len(x), _tree(len(x), leaf)) for x in points]
    base = np.concatenate([[0], np.cumsum([len(x) for x in points])])
    xs = torch.from_numpy(np.concatenate(points)).to(device)
    rows = {}  # (matrix, node) -> its candidate point indices (global), for rows and columns
    depth = max(nd[5] for m in mats for nd in m.nodes)
    host = {}
    for d in range(depth, 0, -1):
        level = [(i, j) for i, m in enumerate(mats) for j, nd in enumerate(m.nodes) if nd[5] == d]
        for side, near, ratio in (("u", 40, 1.12), ("v", 44, 1.13)):
            cand = []
            for i, j in level:
                a, b, l, r = mats[i].nodes[j][:4]
                cand.append(np.arange(a, b) + base[i] if l < 0 else np.concatenate([rows[i, l, side], rows[i, r, side]]))
            c = max(len(v) for v in cand)
            C = torch.zeros(len(level), c, dtype=torch.long)
            M = torch.zeros(len(level), c, dtype=torch.bool)
            for t, v in enumerate(cand):
                C[t, :len(v)] = torch.from_numpy(v)
                M[t, :len(v)] = True
            lo = torch.tensor([base[i] for i, _ in level])[:, None]
            hi = torch.tensor([base[i + 1] for i, _ in level])[:, None]
            a = torch.tensor([mats[i].nodes[j][0] + base[i] for i, j in level])[:, None]
            b = torch.tensor([mats[i].nodes[j][1] + base[i] for i, j in level])[:, None]
            o = _offsets(max(m.n for m in mats), near, ratio)[None]
            P = torch.cat([a - o, b - 1 + o], 1)
            ok = ((P >= lo) & (P < hi)).to(device)
            P = P.clamp(lo, hi - 1).to(device)
            C, M = C.to(device), M.to(device)
            dif = xs[C][:, :, None] - xs[P][:, None, :]
            Y = _kernel(kind, dif if side == "u" else -dif, diag)
            Y = torch.where(M[:, :, None] & ok[:, None, :], Y, torch.zeros_like(Y))
            piv, U, rank = _interpolate(Y, tol)
            sk = torch.gather(C, 1, piv).cpu().numpy()
            U, rank = U.cpu().numpy(), rank.cpu().numpy()
            for t, (i, j) in enumerate(level):
                m, k = mats[i], int(rank[t])
                (m.ku if side == "u" else m.kv)[j] = k
                rows[i, j, side] = sk[t, :k]
                host[i, j, side] = U[t, :len(cand[t]), :k]
    for i, m in enumerate(mats):
        x = points[i]
        for j, (a, b, l, r, _, _) in enumerate(m.nodes):
            g = m.gen[j]
            if l < 0:
                if j > 0:
                    g["U"], g["V"] = host[i, j, "u"], host[i, j, "v"]
                continue
            for key, p, q in (("B12", l, r), ("B21", r, l)):
                I, J = rows[i, p, "u"] - base[i], rows[i, q, "v"] - base[i]
                dif = x[I][:, None] - x[J][None]
                g[key] = np.log(np.abs(dif)) if kind == "log" else 1.0 / dif
            if j > 0:
                for s, k, name in (("u", m.ku, "R"), ("v", m.kv, "W")):
                    m.gen[l][name], m.gen[r][name] = host[i, j, s][:k[l]], host[i, j, s][k[l]:]
        leaves = [j for j, nd in enumerate(m.nodes) if nd[2] < 0]
        w = max(m.nodes[j][1] - m.nodes[j][0] for j in leaves)
        at = torch.tensor([[min(m.nodes[j][0] + t, m.n - 1) for t in range(w)] for j in leaves]).to(device) + int(base[i])
        D = _kernel(kind, xs[at][:, :, None] - xs[at][:, None, :], diag).cpu().numpy()
        for t, j in enumerate(leaves):
            s = m.nodes[j][1] - m.nodes[j][0]
            m.gen[j]["D"] = D[t, :s, :s]
    return mats


def _sizes(case):
    """The matrices' sizes: n, or `count` of them log-uniform in [low, n], the same for every seed."""
    if "count" not in case:
        return [case["n"]]
    rng = np.random.default_rng(17)
    ns = np.round(np.exp(rng.uniform(math.log(case["low"]), math.log(case["n"]), case["count"]))).astype(int)
    ns[0] = case["n"]
    return [int(v) for v in ns]


def _device():
    return "cuda:0" if torch.cuda.is_available() else "cpu"


def _matrices(case, seed):
    rng = np.random.default_rng([int(seed), 17])
    return _build(case["kernel"], [_points(case, n, rng) for n in _sizes(case)], case["leaf"], case["tol"], case["diag"],
                  _device())


def _requests(case):
    """(matrix, right-hand sides) of every request, the same for every seed."""
    rng = np.random.default_rng(23)
    if case["op"] == "serve":
        return [(int(rng.integers(case["count"])), int(min(case["nrhs"], rng.geometric(1.0 / 8)))) for _ in range(case["requests"])]
    if "count" in case:
        return [(i, int(rng.integers(1, case["nrhs"] + 1))) for i in range(case["count"])]
    return [(0, case["nrhs"])]


def _vectors(case, seed, mats):
    """Normal right-hand sides, one (nrhs x n) array a request: the columns of B, contiguous."""
    g = torch.Generator().manual_seed(int(seed) * 7919 + 5)
    return [torch.randn(k, mats[i].n, dtype=torch.float64, generator=g) for i, k in _requests(case)]


# ---------------------------------------------------------------------------
# the library's side
# ---------------------------------------------------------------------------
def _hip():
    if PKG not in sys.modules:
        d = ROOT / "hssmatrices.jl_amd"
        spec = importlib.util.spec_from_file_location(PKG, d / "__init__.py", submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[PKG] = mod
        spec.loader.exec_module(mod)
    return importlib.import_module(PKG + ".hip")


def _pack(m):
    """Node table and generator blob of a Matrix (column-major blocks, breadth-first)."""
    dt = importlib.import_module(PKG + ".hssmatrix").NODE_DTYPE
    t = np.zeros(len(m.nodes), dtype=dt)
    blob, at = [], 0
    height = [0] * len(m.nodes)
    for j in range(len(m.nodes) - 1, -1, -1):
        if m.nodes[j][2] >= 0:
            height[j] = 1 + max(height[m.nodes[j][2]], height[m.nodes[j][3]])
    for j, (a, b, l, r, p, d) in enumerate(m.nodes):
        q = t[j]
        q["parent"], q["left"], q["right"], q["depth"], q["height"] = p, l, r, d, height[j]
        q["m"] = q["n"] = b - a
        q["ku"], q["kv"] = m.ku[j], m.kv[j]
        q["row_off"] = q["col_off"] = a
        for key in ("D", "U", "V", "B12", "B21", "R", "W"):
            v = m.gen[j].get(key)
            q["off_" + key] = -1 if v is None or v.size == 0 else at
            if v is not None and v.size:
                blob.append(np.asfortranarray(v).ravel(order="F"))
                at += v.size
    return t, np.concatenate(blob)


def prepare(case, seed):
    hip = _hip()
    mats = _matrices(case, seed)
    rhs = _vectors(case, seed, mats)
    op = case["op"]
    A = [hip.HipHssMatrix(_pack(m)) for m in mats]
    s = dict(case=case, hip=hip, A=A)
    if op == "ldiv":
        s["b"] = np.asfortranarray(rhs[0].numpy().T)
        return s
    s["B"] = [b.to("cuda:0") for b in rhs]
    s["X"] = [torch.zeros_like(b) for b in s["B"]]
    req = _requests(case)
    s["nrhs"] = [k for _, k in req]
    s["ld"] = [mats[i].n for i, _ in req]
    if op == "matvec" and case["beta"] != 0.0:
        s["X"][0].copy_(torch.flip(s["B"][0], [1]))
    elif op == "solve":
        s["F"] = [A[0].ulvfactor("fp64")]
    elif op == "mixed":
        s["F"] = [A[0].ulvfactor("fp32")]
    elif op == "batch":
        s["F"] = hip.ulvfactor_batch(A, "fp64")
        s["plan"] = hip.Plan(s["F"], s["nrhs"], _ptr(s["B"]), s["ld"], _ptr(s["X"]), s["ld"], refinement=True)
    elif op == "serve":
        s["server"] = hip.Server(64 << 30, prec="fp32", tol=1e-10, max_inflight=64)
        s["id"] = [s["server"].admit(a) for a in A]
        s["on"] = [i for i, _ in req]
    torch.cuda.synchronize()
    return s


def _ptr(ts):
    return [t.data_ptr() for t in ts]


def run(s):
    op, hip, A = s["case"]["op"], s["hip"], s["A"]
    if op == "ldiv":
        return hip.ulvfactsolve(A[0], s["b"])
    B, X, nrhs, ld = s["B"], s["X"], s["nrhs"], s["ld"]
    if op == "matvec":
        A[0].matmul_dev(nrhs[0], s["case"]["alpha"], B[0].data_ptr(), ld[0], s["case"]["beta"], X[0].data_ptr(), ld[0])
    elif op == "solve":
        s["F"][0].solve_dev(nrhs[0], B[0].data_ptr(), ld[0], X[0].data_ptr(), ld[0])
    elif op == "mixed":
        s["F"][0].solve_dev(nrhs[0], B[0].data_ptr(), ld[0], X[0].data_ptr(), ld[0], tol=1e-10, max_iter=10)
    elif op == "backslash":
        F = A[0].ulvfactor("fp64")
        F.solve_dev(nrhs[0], B[0].data_ptr(), ld[0], X[0].data_ptr(), ld[0])
        F.close()
    elif op == "batch":
        s["plan"].execute(tol=1e-10)
    elif op == "factors":
        F = hip.ulvfactor_batch(A, "fp64")
        hip.solve_batch_dev(F, nrhs, _ptr(B), ld, _ptr(X), ld)
        for f in F:
            f.close()
    else:
        srv = s["server"]
        t = [srv.submit(s["id"][s["on"][i]], nrhs[i], B[i].data_ptr(), ld[i], X[i].data_ptr(), ld[i]) for i in range(len(B))]
        while srv.step() > 0:
            pass
        for k in t:
            srv.poll(k)
    return X


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its values in plain numpy
# ---------------------------------------------------------------------------
def _factor_sizes(m):
    """(entries, factor flops) of the ULV factor in the reference's form: per node the QL
    reflectors of U, the LQ reflectors, the triangles and the blocks applied to b and V."""
    ent = fl = 0
    red = {}
    for j in range(len(m.nodes) - 1, -1, -1):
        a, b, l, r = m.nodes[j][:4]
        n = b - a if l < 0 else red[l] + red[r]
        if j == 0:
            return ent + n * n, fl + 2.0 / 3.0 * n ** 3
        k = min(m.ku[j], n)
        nk, kv = n - k, m.kv[j]
        red[j] = k
        ent += n * k + n * nk + nk * (nk + 1) // 2 + k * nk + kv * nk
        fl += 2.0 * n * k * k + 4.0 * n * n * k + 2.0 * n * nk * nk + 4.0 * n * nk * (k + kv)


def work(case):
    """Each input (generators, factor, right-hand sides) read once and each output written once;
    a refined solve is counted as one Float64 solve."""
    mats = _matrices(case, 0)
    req = _requests(case)
    op = case["op"]
    byt = fl = 0.0
    for i, k in req:
        m = mats[i]
        byt += 8.0 * m.n * k * (3 if op == "matvec" and case["beta"] != 0.0 else 2)
        fl += 2.0 * k * (m.entries() if op == "matvec" else _factor_sizes(m)[0])
    for i in {i for i, _ in req}:
        m = mats[i]
        if op in ("ldiv", "backslash", "factors"):
            byt += 8.0 * m.entries()
            fl += _factor_sizes(m)[1]
        else:
            byt += (4.0 if op in ("mixed", "serve") else 8.0) * (m.entries() if op == "matvec" else _factor_sizes(m)[0])
    return {"bytes": byt, "flops": fl}


def _mul(m, B):
    """A B (B n x k) by the tree: z up, f down."""
    nd, g = m.nodes, m.gen
    z, f = [None] * len(nd), [None] * len(nd)
    for j in range(len(nd) - 1, 0, -1):
        a, b, l, r = nd[j][:4]
        z[j] = g[j]["V"].T @ B[a:b] if l < 0 else g[l]["W"].T @ z[l] + g[r]["W"].T @ z[r]
    C = np.zeros_like(B)
    for j, (a, b, l, r, _, _) in enumerate(nd):
        if l < 0:
            C[a:b] = g[j]["D"] @ B[a:b] + (g[j]["U"] @ f[j] if j else 0.0)
        else:
            f[l] = g[j]["B12"] @ z[r] + (g[l]["R"] @ f[j] if j else 0.0)
            f[r] = g[j]["B21"] @ z[l] + (g[r]["R"] @ f[j] if j else 0.0)
    return C


def _solver(m):
    """x = A \\ b by eliminating the leaves: with f a node's incoming term, a leaf has
    x = D^-1 (b - U f) and z = V' x = a - G f; a branch couples its children's z and f."""
    nd, g = m.nodes, m.gen
    N = len(nd)
    G, lu, inv = [None] * N, [None] * N, [None] * N
    for j in range(N - 1, -1, -1):
        l, r = nd[j][2], nd[j][3]
        if l < 0:
            inv[j] = np.linalg.inv(g[j]["D"])
            if j:
                lu[j] = inv[j] @ g[j]["U"]
                G[j] = g[j]["V"].T @ lu[j]
        else:
            kl, kr = m.kv[l], m.kv[r]
            M = np.eye(kl + kr)
            M[:kl, kl:] = G[l] @ g[j]["B12"]
            M[kl:, :kl] = G[r] @ g[j]["B21"]
            inv[j] = np.linalg.inv(M)
            if j:
                lu[j] = inv[j] @ np.vstack([G[l] @ g[l]["R"], G[r] @ g[r]["R"]])
                G[j] = np.vstack([g[l]["W"], g[r]["W"]]).T @ lu[j]

    def solve(b):
        z, f, h = [None] * N, [None] * N, [None] * N
        for j in range(N - 1, -1, -1):
            a, e, l, r = nd[j][:4]
            if l < 0:
                h[j] = inv[j] @ b[a:e]
                z[j] = g[j]["V"].T @ h[j] if j else None
            else:
                h[j] = inv[j] @ np.vstack([z[l], z[r]])
                z[j] = np.vstack([g[l]["W"], g[r]["W"]]).T @ h[j] if j else None
        x = np.zeros_like(b)
        for j, (a, e, l, r, _, _) in enumerate(nd):
            y = h[j] - lu[j] @ f[j] if j else h[j]
            if l < 0:
                x[a:e] = y
            else:
                zl, zr = y[:m.kv[l]], y[m.kv[l]:]
                f[l] = g[j]["B12"] @ zr + (g[l]["R"] @ f[j] if j else 0.0)
                f[r] = g[j]["B21"] @ zl + (g[r]["R"] @ f[j] if j else 0.0)
        return x

    return solve


def exact(case, seed):
    mats = _matrices(case, seed)
    rhs = _vectors(case, seed, mats)
    if case["op"] == "matvec":
        B = rhs[0].numpy().T.copy()
        C = case["alpha"] * _mul(mats[0], B)
        if case["beta"] != 0.0:
            C += case["beta"] * B[::-1]
        return [np.ascontiguousarray(C.T)]
    out = []
    solvers = {}
    for (i, _), b in zip(_requests(case), rhs):
        b = b.numpy().T.copy()
        if i not in solvers:
            solvers[i] = _solver(mats[i])
        x = solvers[i](b)
        for _ in range(4):  # refined in Float64 from here on
            x = x + solvers[i](b - _mul(mats[i], x))
        out.append(x if case["op"] == "ldiv" else np.ascontiguousarray(x.T))
    return out[0] if case["op"] == "ldiv" else out
