"""MINRES solves that run as one resident launch (diagonal preconditioner) against the stepwise kernels,
which a preconditioner with an entry off the diagonal still takes, and against the FP64 residual.

The matrices have eigenvalues of at least 1 in magnitude by diagonal dominance, so an error is at most the
residual, rtol |b| for each route."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-9


def _matrix(n, kind, seed):
    """Symmetric, row sums of the off-diagonal part below |diagonal| - 1; indefinite where signed."""
    import scipy.sparse as sps

    rng = np.random.default_rng(seed)
    if kind == "diagonal":
        A = sps.csr_matrix((n, n))
    elif kind == "band":  # short rows, neighbours only
        k = min(2, n - 1)
        A = sps.diags([rng.uniform(-1, 1, n - d) for d in range(1, k + 1)], list(range(1, k + 1)), shape=(n, n))
    elif kind == "arrow":  # two full rows: more columns in one block than a thread prefetches
        A = sps.lil_matrix((n, n))
        A[0, 1:] = rng.uniform(-1, 1, n - 1) / n
        A[n // 2, n // 2 + 1:] = rng.uniform(-1, 1, n - n // 2 - 1) / n
    else:  # scattered columns, rows of uneven length
        A = sps.random(n, n, density=min(1.0, kind / n), random_state=seed, data_rvs=lambda m: rng.uniform(-1, 1, m))
        A = sps.triu(A, 1)
    A = sps.csr_matrix(A)
    A = A + A.T
    d = 1.0 + np.asarray(abs(A).sum(axis=1)).ravel() + rng.uniform(0, 1, n)
    sign = np.where(np.arange(n) < (2 * n + 2) // 3, 1.0, -1.0)
    return sps.csr_matrix(A + sps.diags(sign * d)), d


@pytest.mark.parametrize("n,kind", [(1, "diagonal"), (15, "diagonal"), (16, "band"), (17, 3), (129, "band"),
                                    (1023, 6), (1025, 12), (5000, "arrow"), (4099, 40), (30011, 9)])
def test_resident_route_matches_stepwise(n, kind):
    import scipy.sparse as sps
    import torch

    from nfempy_amd.solvers import MinresIR

    print(f"[minres grid] n={n} {kind}", flush=True)
    A, d = _matrix(n, kind, seed=n)
    A.sort_indices()
    dev = lambda a, t: torch.tensor(np.ascontiguousarray(a), dtype=t, device="cuda")
    rp, ci = dev(A.indptr, torch.int32), dev(A.indices, torch.int32)
    v64 = dev(A.data, torch.float64)
    v32 = v64.to(torch.float32)
    b = np.random.default_rng(n + 1).standard_normal(n)
    pinv = dev(1.0 / d, torch.float32)
    # the same diagonal, and one stored zero off it: only the stepwise kernels take such a preconditioner
    P = sps.csr_matrix(sps.diags(1.0 / d)).tocoo()
    extra = n - 1
    order = np.lexsort((np.append(P.col, 0), np.append(P.row, extra)))
    rows, cols = np.append(P.row, extra)[order], np.append(P.col, 0)[order]
    vals = np.append(P.data, 0.0)[order]
    ptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    pc = (dev(ptr, torch.int32), dev(cols, torch.int32), dev(vals, torch.float32))
    got = {}
    for name, kw in (("resident", {"pinv": pinv}), ("stepwise", {"pc": pc})):
        s = MinresIR(rp, ci, v32, v64, **kw)
        for _ in range(2):  # the second solve meets the first one's work space
            x, info = s.solve(dev(b, torch.float64), rtol=RTOL)
            x = x.cpu().numpy()
            assert info["converged"], (name, info)
            assert np.linalg.norm(b - A @ x) <= 1.1 * RTOL * np.linalg.norm(b), name
        solved, declined = s.resident_counts()
        # what the preconditioner is, is known before a launch: nothing is tried and declined
        assert declined == 0 and (solved > 0) == (name == "resident"), (name, solved, declined)
        got[name] = info["iterations"], x
        s.close()
    # the same recurrence, tested every 16 iterations: roundings can move a stop by one test per outer step
    (it_r, x_r), (it_s, x_s) = got["resident"], got["stepwise"]
    assert abs(it_r - it_s) <= 32
    assert np.linalg.norm(x_r - x_s) <= 2.2 * RTOL * np.linalg.norm(b)


def test_iteration_limit_and_zero_rhs():
    import torch

    from nfempy_amd.solvers import MinresIR

    A, d = _matrix(2000, 10, seed=5)
    A.sort_indices()
    dev = lambda a, t: torch.tensor(np.ascontiguousarray(a), dtype=t, device="cuda")
    v64 = dev(A.data, torch.float64)
    s = MinresIR(dev(A.indptr, torch.int32), dev(A.indices, torch.int32), v64.to(torch.float32), v64,
                 pinv=dev(1.0 / d, torch.float32))
    b = dev(np.random.default_rng(6).standard_normal(2000), torch.float64)
    x, info = s.solve(b, rtol=1e-14, max_inner=3, max_outer=2)
    assert not info["converged"] and info["iterations"] == 6 and info["residual"] < 1.0
    x, info = s.solve(torch.zeros_like(b))
    assert float(x.abs().max()) == 0.0 and info["iterations"] == 0
    s.close()


def test_exact_breakdown_is_finite():
    """The identity ends the Lanczos process after one step."""
    import torch

    from nfempy_amd.solvers import MinresIR

    n = 300
    ar = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    one = torch.ones(n, dtype=torch.float64, device="cuda")
    s = MinresIR(ar, ar[:-1].contiguous(), one.to(torch.float32), one, pinv=one.to(torch.float32))
    b = torch.linspace(-1, 2, n, dtype=torch.float64, device="cuda")
    x, info = s.solve(b, rtol=1e-12)
    assert info["converged"] and float((x - b).norm() / b.norm()) <= 1e-12
    s.close()


@pytest.mark.parametrize("pc", ["diag", "twogrid", "learned"])
def test_batch_over_resident_sizes(pc):
    """Instances of one block, of many, more blocks than fit one launch: FP64 residuals, and each instance
    bitwise what it is alone (its block count follows from its own size); then, with an instance that the
    two-grid cycle leaves to the stepwise kernels (11 cubed: 216 aggregates), the whole batch there."""
    import torch

    from nfempy_amd.batch import DarcyBatch

    specs = [(2, 1), (9, 2), (5, 2), (9, 2), (7, 1), (1, 2), (9, 2), (11, 1)]
    b = DarcyBatch(specs, seed=4, workers=1)
    b.assemble()
    print(f"[minres grid] batch {pc}", flush=True)
    mixed, mixed_infos, _ = b.solve_batched(rtol=1e-8, pc=pc)
    assert (b.last_resident[0] > 0) == (pc == "diag")  # the limit is one of the cycle's
    xs, infos, _ = b.solve_batched(list(range(7)), rtol=1e-8, pc=pc)
    assert b.last_resident[0] == sum(i["outer"] for i in infos) and b.last_resident[1] == 0
    xs.append(mixed[7])
    infos.append(mixed_infos[7])
    for i in range(7):  # both within rtol of the solution, times the conditioning
        assert mixed_infos[i]["converged"]
        assert float((mixed[i] - xs[i]).norm() / xs[i].norm()) <= 1e-6
    for i in range(len(specs)):
        assert infos[i]["converged"], (i, infos[i])
        y = b.fp64_system(i)
        n = len(y["rowptr"]) - 1
        A = torch.sparse_csr_tensor(y["rowptr"].long(), y["col"].long(), y["vals64"], size=(n, n))
        res = float((y["b"] - A @ xs[i]).norm() / y["b"].norm())
        assert res <= 1.1e-8, (i, res)
    for i in (1, 2, 3, 6):
        alone, info, _ = b.solve_batched([i], rtol=1e-8, pc=pc)
        assert b.last_resident == (info[0]["outer"], 0)
        assert info[0]["iterations"] == infos[i]["iterations"]
        assert torch.equal(alone[0], xs[i]), i


@pytest.mark.parametrize("n", [1, 2, 3, 5, 9])
def test_elasticity_resident_matches_stepwise(n):
    """The resident solve takes the 3 x 3 block operator; without it the stepwise kernels run. Both end at
    an FP64 residual of 1e-9; the system's conditioning separates their solutions by more."""
    import torch

    from nfempy_amd.elasticity import ElasticitySystem
    from nfempy_amd.mesh import Mesh, unit_cube
    from nfempy_amd.spaces import ProductSpace

    mesh = Mesh.from_blocks(3, *unit_cube(n))
    space = ProductSpace({"s": (3, 3, "BDM", 1, mesh), "u": (3, 3, "Lagrange", 0, mesh),
                          "t": (3, 3, "Lagrange", 0, mesh)})
    space.make_subspaces_discontinuous({"u": True, "t": True})
    space.build_structures({"s": [1], "u": [1], "t": [1]}, {"s": [2, 3, 4, 5, 6, 7]})
    r = np.random.default_rng(n)
    lam, mu = (np.exp(0.5 * r.standard_normal(6 * n ** 3)) for _ in range(2))
    rhs = lambda x, y, z: np.array([0.3 * np.ones_like(x), 0.7 * np.ones_like(x), np.ones_like(x)]
                                   + [np.zeros_like(x)] * 3)
    y = ElasticitySystem(space, {"lambda": lam, "mu": mu, "rhs": rhs})
    for fp64 in (True, False):
        y.assemble("A", fp64=fp64)
    got = {}
    for block3 in (True, False):
        y.use_block3 = block3
        print(f"[minres grid] elasticity n={n} blocks={block3}", flush=True)
        x, info = y.solve(rtol=1e-9)
        assert info["converged"] and info["residual"] <= 1e-9, info
        assert y.last_resident == ((info["outer"], 0) if block3 else (0, 0)), (n, y.last_resident)
        rp, col, _, v64 = y.full("A")
        A = torch.sparse_csr_tensor(rp.long(), col.long(), v64, size=(y.n, y.n))
        res = float((-y.rhs64 - A @ x).norm() / y.rhs64.norm())
        assert res <= 1.1e-9, res
        got[block3] = x, info["iterations"]
    assert abs(got[True][1] - got[False][1]) <= 48
    err = float((got[True][0] - got[False][0]).norm() / got[False][0].norm())
    assert err <= 1e-6, err
