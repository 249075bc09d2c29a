"""Routes of the MINRES solves: what is refused before a route is chosen, which route a solve takes, and
what it does when the device does not give it the resident one."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(specs, pc="twogrid", seed=3):
    """(DarcyBatch, MinresBatch, right-hand sides, BatchTwoGrid or None) with the preconditioner set up."""
    from nfempy_amd.batch import DarcyBatch

    b = DarcyBatch(specs, seed=seed, workers=1)
    b.assemble()
    return _batch_of(b, *range(len(specs)), pc=pc)


def _batch_of(b, *idx, pc="twogrid"):
    """The same of some instances of a batch."""
    import torch

    from nfempy_amd.batch_pc import BatchTwoGrid
    from nfempy_amd.learned import default_weights_path, load_params
    from nfempy_amd.solvers import MinresBatch

    systems = [b.fp64_system(i) for i in idx]
    mb = MinresBatch(systems)
    tg = None
    if pc != "diag":
        theta = load_params(default_weights_path()) if pc == "learned" else None
        tg = BatchTwoGrid([b.instances[i]["system"] for i in idx], mb.offsets, theta=theta)
        mb.set_pc(tg.setup([s["vals64"] for s in systems]))
        mb._tg = tg  # the descriptors point into its arrays
    return b, mb, torch.cat([s["b"] for s in systems]), tg


def _elasticity(n):
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
    return y


def _elasticity_solver(y):
    """(MinresIR with the 3 x 3 blocks and the two-grid descriptor, descriptor)."""
    from nfempy_amd import _native as nat
    from nfempy_amd.solvers import MinresIR

    desc = y.twogrid().setup()
    rp, col, v32, v64 = y.full("A")
    b3 = y.ops["A"]["block3"]
    nat.call("nfx_md_scatter", int(v32.numel()), nat.ptr(v32), nat.ptr(b3["dest"]), 0, nat.ptr(b3["bval"]),
             nat.stream_handle())
    return MinresIR(rp, col, v32, v64, block3=(b3["n_blocks"], b3["browptr"], b3["bcol"], b3["bval"]),
                    tg=desc), desc


def _copy(struct):
    out = type(struct)()
    ctypes.memmove(ctypes.byref(out), ctypes.byref(struct), ctypes.sizeof(struct))
    return out


def test_incomplete_preconditioners_are_refused():
    """A descriptor with a null array, or smoother couplings that the blocks cannot take, comes back as an
    argument error before any kernel reads it, whichever route the solve would take."""
    import torch

    print("[routes] batch descriptors", flush=True)
    b, mb, rhs, tg = _batch([(2, 1), (2, 2)])
    for g, good in enumerate(tg._descs):
        names = [n for n, t in good._fields_ if t is ctypes.c_void_p]
        for name in names:
            arr = (type(good) * len(tg._descs))(*[_copy(d) for d in tg._descs])
            if name == "wo" or (name.startswith("fb_") and good.n_fb == 0):
                continue
            setattr(arr[g], name, None)
            with pytest.raises(ValueError, match="nfx_batch_tg"):
                mb.set_pc(arr)
        if good.nb == 4:
            arr = (type(good) * len(tg._descs))(*[_copy(d) for d in tg._descs])
            arr[g].wo = arr[g].wd
            with pytest.raises(ValueError, match="couplings"):
                mb.set_pc(arr)
    mb.set_pc(tg._descs)  # the complete groups still solve
    x, infos = mb.solve(rhs, rtol=1e-8)
    assert all(i["converged"] for i in infos)
    mb.close()

    print("[routes] elasticity descriptor", flush=True)
    y = _elasticity(2)
    s, desc = _elasticity_solver(y)
    for name in ("dinv", "nbr", "sblk", "winv", "agg_ptr", "agg_mem", "agg_of", "ainv", "work"):
        s.tg = _copy(desc)
        setattr(s.tg, name, None)
        with pytest.raises(ValueError, match="incomplete descriptor"):
            s.solve(-y.rhs64)
    s.tg = _copy(desc)
    x, info = s.solve(torch.zeros_like(y.rhs64))  # nothing to solve: nothing read
    assert info["residual"] == 0.0
    x, info = s.solve(-y.rhs64, rtol=1e-8)
    assert info["converged"]
    s.close()


# ---- which route ran ------------------------------------------------------------------------------
LDS = 158 * 1024  # bytes of a block, as nfx_grid.h has them
SHARE = 128 * 1024  # bytes of an instance per block, as nfx_bm_grid.hip has them


def _batch_layout(A):
    """(values in LDS, columns beyond what the threads hold) of each block of an instance without a two-grid cycle: how
    nfx_bm_grid.hip lays out its LDS."""
    n = A.shape[0]
    blocks = -(-(6 * A.nnz + 40 * n) // SHARE)
    out = set()
    for r in range(blocks):
        S = A[n * r // blocks:n * (r + 1) // blocks]
        R, H = S.shape[0], len(np.unique(S.indices))
        base = 4 * (2 * R + 1) + 24 * R + 4 + 4 * ((S.nnz + 1) // 2)
        assert base + 8 * ((n + 31) // 32) + 4 * H <= LDS and base + 8 * H <= LDS
        listed = H > 4 * 1024
        out.add((base + (8 if listed else 4) * H + 4 * S.nnz <= LDS, listed))
    return out


@pytest.mark.parametrize("n,kind,layout", [(8000, 1, (True, False)), (8000, 2, (True, True)),
                                           (20000, 9, (False, True))])
def test_batch_layouts_match_stepwise(n, kind, layout):
    """Scattered systems whose blocks meet few or many columns, and hold their values in LDS or not: the resident
    route against the stepwise one and the FP64 residual."""
    import torch

    from nfempy_amd.solvers import MinresBatch
    from tests.test_gpu_minres_grid import _matrix

    print(f"[routes] layout n={n} {kind}", flush=True)
    A, d = _matrix(n, kind, seed=n + kind)
    A.sort_indices()
    assert layout in _batch_layout(A)
    dev = lambda a, t: torch.tensor(np.ascontiguousarray(a), dtype=t, device="cuda")
    v64 = dev(A.data, torch.float64)
    b = np.random.default_rng(n).standard_normal(n)
    got = {}
    for launches in (-1, 0):
        mb = MinresBatch([{"rowptr": dev(A.indptr, torch.int32), "col": dev(A.indices, torch.int32),
                           "vals32": v64.to(torch.float32), "vals64": v64, "pinv": dev(1.0 / d, torch.float32)}])
        mb.set_resident(launches)
        x, infos = mb.solve(dev(b, torch.float64), rtol=1e-9)
        x = x.cpu().numpy()
        assert infos[0]["converged"]
        assert mb.resident_counts() == ((infos[0]["outer"], 0) if launches else (0, 0))
        assert np.linalg.norm(b - A @ x) <= 1.1e-9 * np.linalg.norm(b)
        got[launches] = x
        mb.close()
    # eigenvalues of at least 1 in magnitude: an error is at most the residual, 1e-9 |b| for each route
    assert np.linalg.norm(got[-1] - got[0]) <= 2.2e-9 * np.linalg.norm(b)


def _elasticity_layout(bp, bc, mem, E, ns, n_agg):
    """(values in LDS, columns beyond what the threads hold) of the blocks of an elasticity solve on the 3 x 3
    block rows (bp, bc): nfx_el_grid.hip's layout."""
    nb, nu = len(bp) - 1, 3 * E
    F, n = ns // 9, 3 * nb
    size = lambda k: (2 * int(bp[-1]) + 64 * n) // k + (48 << 10)
    blocks = 16
    while blocks < 256 and (-(-E // blocks) > 12 or size(blocks) > LDS):
        blocks *= 2
    assert -(-E // blocks) <= 34 and size(blocks) <= LDS and n_agg <= 128
    out = set()
    for k in range(blocks):
        f = np.arange(3 * (F * k // blocks), 3 * (F * (k + 1) // blocks))
        c = mem[E * k // blocks:E * (k + 1) // blocks]
        rows = np.concatenate([f, ns // 3 + c, (ns + nu) // 3 + c])
        RB, nz = len(rows), int((bp[rows + 1] - bp[rows]).sum())
        H = len(np.unique(np.concatenate([bc[bp[r]:bp[r + 1]] for r in rows])))
        words = 2 * RB + 1 + 15 * RB + 27 * len(f) + 3 * 1024 + 6 * 384 + 12 * 128 + 384 + 129 + 256
        base = 4 * words + 4 * ((nz + 1) // 2)
        assert base + 8 * ((nb + 31) // 32) + 4 * H <= LDS and base + 16 * H <= LDS
        listed = 3 * H > 4 * 1024
        out.add((base + 12 * H + (4 * H if listed else 0) + 36 * nz <= LDS, listed))
    return out


@pytest.mark.parametrize("n,shuffled,layout", [(5, False, (True, False)), (10, False, (False, False)),
                                               (10, True, (False, True))])
def test_elasticity_layouts_are_resident(n, shuffled, layout):
    """Systems whose blocks hold their values in LDS, and the largest that is resident, whose blocks do not;
    with its faces numbered in any order a block meets more columns than its threads hold. FP64 residuals."""
    import scipy.sparse as sps
    import torch

    from nfempy_amd.solvers import MinresIR

    print(f"[routes] elasticity layout n={n} {shuffled}", flush=True)
    y = _elasticity(n)
    desc = _copy(y.twogrid().setup())
    rp, col, v32, v64 = (v.cpu().numpy() for v in y.full("A"))
    A = sps.csr_matrix((v64, col, rp), shape=(y.n, y.n))
    F = y.n_s // 9
    p = np.random.default_rng(n).permutation(F) if shuffled else np.arange(F)
    rows = np.concatenate([(9 * p[:, None] + np.arange(9)).ravel(), np.arange(y.n_s, y.n)])
    A = A[rows][:, rows].tocsr()
    A.sort_indices()
    B = A.tobsr((3, 3))
    B.sort_indices()
    mem = y.twogrid().agg_mem.cpu().numpy()
    seen = _elasticity_layout(B.indptr, B.indices, mem, y.E, y.n_s, desc.n_agg)
    print(f"[routes] {seen}", flush=True)
    assert layout in seen
    dev = lambda a, t: torch.tensor(np.ascontiguousarray(a), dtype=t, device="cuda")
    i32, f32, f64 = torch.int32, torch.float32, torch.float64
    dinv = y.twogrid().dinv32.view(F, 81)[torch.tensor(p, device="cuda")].contiguous()
    desc.dinv = dinv.data_ptr()
    block3 = (len(B.indices), dev(B.indptr, i32), dev(B.indices, i32),
              dev(B.data.reshape(-1, 9).T.ravel(), f32))
    s = MinresIR(dev(A.indptr, i32), dev(A.indices, i32), dev(A.data, f32), dev(A.data, f64), block3=block3, tg=desc)
    b = -y.rhs64.cpu().numpy()[rows]
    x, info = s.solve(dev(b, f64), rtol=1e-8, inner_rtol=3e-4)
    assert info["converged"] and s.resident_counts() == (info["outer"], 0)
    s.close()
    assert np.linalg.norm(b - A @ x.cpu().numpy()) <= 1.1e-8 * np.linalg.norm(b)


def _single(n=4000, stream=None):
    import torch

    from nfempy_amd.solvers import MinresIR
    from tests.test_gpu_minres_grid import _matrix

    A, d = _matrix(n, 6, seed=n)
    A.sort_indices()
    dev = lambda a, t: torch.tensor(np.ascontiguousarray(a), dtype=t, device="cuda")
    v64 = dev(A.data, torch.float64)
    s = MinresIR(dev(A.indptr, torch.int32), dev(A.indices, torch.int32), v64.to(torch.float32), v64,
                 pinv=dev(1.0 / d, torch.float32), stream=stream)
    return s, dev(np.random.default_rng(n).standard_normal(n), torch.float64)


def test_stepwise_where_no_launch_is_allowed():
    """None, one, and as many launches as a solve wants: the counts say what ran, every solve converges."""
    print("[routes] single", flush=True)
    s, b = _single()
    full, info = s.solve(b, rtol=1e-10)
    outer = info["outer"]
    assert outer > 1 and s.resident_counts() == (outer, 0)
    s.set_resident(0)
    x, info = s.solve(b, rtol=1e-10)
    assert info["converged"] and s.resident_counts() == (outer, 0)
    s.set_resident(1)  # the second inner solve is declined
    x, info = s.solve(b, rtol=1e-10)
    assert info["converged"] and s.resident_counts() == (outer + 1, 1)
    s.set_resident()
    x, info = s.solve(b, rtol=1e-10)
    assert s.resident_counts() == (2 * outer + 1, 1) and bool((x == full).all())
    s.close()

    print("[routes] elasticity", flush=True)
    y = _elasticity(3)
    s, _ = _elasticity_solver(y)
    s.set_resident(1)
    x, info = s.solve(-y.rhs64, rtol=1e-9, inner_rtol=3e-4)
    assert info["converged"] and info["outer"] > 1 and s.resident_counts() == (1, 1)
    s.close()

    print("[routes] batch over two launches", flush=True)
    _, mb, rhs, _ = _batch([(9, 2), (5, 2), (9, 2), (9, 2), (3, 1)])
    mb.set_resident(1)
    x, infos = mb.solve(rhs, rtol=1e-8)
    solved, declined = mb.resident_counts()
    assert all(i["converged"] and i["outer"] > 1 for i in infos[:4])
    assert 0 < solved < 5 and solved + declined == 5  # the first refinement step; the later ones do not try
    mb.close()


def test_given_up_waits_end_stepwise():
    """A launch without its last block: the others give up their wait for it, the launch ends, the solve goes on
    with the stepwise kernels."""
    print("[routes] single", flush=True)
    s, b = _single()
    s.set_resident(absent=True)
    x, info = s.solve(b, rtol=1e-9)
    assert info["converged"] and s.resident_counts() == (0, 1)
    s.set_resident()
    x, info = s.solve(b, rtol=1e-9)
    assert s.resident_counts() == (info["outer"], 1)
    s.close()

    print("[routes] elasticity", flush=True)
    y = _elasticity(3)
    s, _ = _elasticity_solver(y)
    s.set_resident(absent=True)
    x, info = s.solve(-y.rhs64, rtol=1e-8)
    assert info["converged"] and s.resident_counts() == (0, 1)
    s.close()

    print("[routes] batch", flush=True)
    _, mb, rhs, _ = _batch([(7, 2), (6, 2)])
    mb.set_resident(absent=True)
    x, infos = mb.solve(rhs, rtol=1e-8)
    solved, declined = mb.resident_counts()
    assert all(i["converged"] and i["outer"] > 1 for i in infos)
    assert (solved, declined) == (1, 1)  # the first refinement step: the smaller system's block was left out
    mb.close()


def test_two_threads_on_two_streams():
    """Two host threads, each with its own solver and stream: every answer is the one that the solver gives
    alone (bitwise, as long as no launch was declined)."""
    import threading

    import torch

    print("[routes] two threads", flush=True)
    pair, want, got = [], [], [[], []]
    for n in (4000, 9001):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            s, b = _single(n, stream=st)
            want.append(s.solve(b, rtol=1e-9)[0])
        pair.append((s, b, st))
    torch.cuda.synchronize()

    def work(i):
        s, b, st = pair[i]
        with torch.cuda.stream(st):
            for _ in range(8):
                got[i].append(s.solve(b, rtol=1e-9))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    for i, (s, b, _) in enumerate(pair):
        assert len(got[i]) == 8 and all(info["converged"] for _, info in got[i])
        solved, declined = s.resident_counts()
        print(f"[routes] solver {i}: {solved} resident, {declined} declined", flush=True)
        assert solved > 0
        for x, _ in got[i]:
            if declined == 0:
                assert torch.equal(x, want[i])
            else:
                assert float((x - want[i]).norm()) <= 2.2e-9 * float(b.norm())
        s.close()


def test_a_batch_keeps_one_route():
    """The route is that of the whole batch, whichever instances still iterate: with an instance that the cycle
    leaves to the stepwise kernels (11 cubed: 216 aggregates) the others' results are bitwise the same while
    it iterates, when it starts from its solution, and when the batch is kept from resident launches; alone
    on the stepwise route each instance is bitwise what it is there."""
    import torch

    print("[routes] one route", flush=True)
    specs = [(4, 1), (5, 2), (11, 1), (3, 2)]
    b, mb, rhs, _ = _batch(specs)
    x, infos = mb.solve(rhs, rtol=1e-8)
    assert all(i["converged"] for i in infos) and mb.resident_counts() == (0, 0)
    part = lambda v, i: v[int(mb.offsets[i]):int(mb.offsets[i + 1])]
    start = torch.zeros_like(rhs)
    part(start, 2).copy_(part(x, 2))
    again, infos2 = mb.solve(rhs, x=start, rtol=1e-8)
    assert infos2[2]["iterations"] == 0 and mb.resident_counts() == (0, 0)
    for i in (0, 1, 3):
        assert torch.equal(part(again, i), part(x, i)), i
    mb.close()
    for i in (0, 1, 3):
        _, one, rhs1, _ = _batch_of(b, i)
        one.set_resident(0)
        alone, info = one.solve(rhs1, rtol=1e-8)
        assert info[0]["iterations"] == infos[i]["iterations"] and torch.equal(alone, part(x, i)), i
        one.close()


@pytest.mark.parametrize("spec,count,resident", [((9, 2), 6, True), ((9, 2), 7, False), ((5, 2), 96, True),
                                                 ((5, 2), 103, False)])
def test_a_batch_is_resident_where_its_launches_pay(spec, count, resident):
    """Instances of 9 cubed of degree 2 take 87 blocks, two a launch of 256: three launches pay, four, two
    thirds full, do not. Instances of 5 cubed take 15 blocks: six launches for 1,440 of them pay, 1,545 would be seven."""
    print(f"[routes] launches of {count}", flush=True)
    b, mb, rhs, _ = _batch([spec] * count)
    x, infos = mb.solve(rhs, rtol=1e-8)
    assert all(i["converged"] for i in infos)
    assert mb.resident_counts() == ((sum(i["outer"] for i in infos), 0) if resident else (0, 0))
    mb.close()


CHILD = """
import sys
sys.path.insert(0, {root!r})
from tests.test_gpu_resident_routes import _single
s, b = _single()
for _ in range(2):
    x, info = s.solve(b, rtol=1e-9)
    assert info["converged"], info
print("counts", *s.resident_counts(), flush=True)
s.close()
"""


def test_a_second_process_solves_beside_this_one():
    """A device gives cooperative launches to one process at a time: in a second one the launch is refused and
    the solve runs stepwise; the device is not asked again at once."""
    import os
    import subprocess
    import sys

    print("[routes] second process", flush=True)
    s, b = _single()
    s.solve(b, rtol=1e-9)
    assert s.resident_counts()[0] > 0  # this process holds them
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-u", "-c", CHILD.format(root=root)], capture_output=True, text=True,
                         timeout=100)
    print(out.stdout, out.stderr[-500:], flush=True)
    assert out.returncode == 0, out.stderr[-2000:]
    solved, declined = (int(v) for v in out.stdout.split("counts")[1].split())
    assert (solved, declined) == (0, 1) or declined == 0  # refused once, or the device serves both
    x, info = s.solve(b, rtol=1e-9)
    assert info["converged"]
    s.close()


def test_a_batch_is_planned_by_its_first_solve():
    """Creating a batch reads none of its arrays and holds the stepwise vectors only; a system too large to be
    resident (2 M rows) adds nothing to them when it is solved."""
    import torch

    from nfempy_amd.solvers import MinresBatch
    from tests.test_gpu_minres_grid import _matrix

    print("[routes] plan", flush=True)
    A, d = _matrix(3000, 6, seed=1)
    A.sort_indices()
    dev = lambda a, t: torch.tensor(np.ascontiguousarray(a), dtype=t, device="cuda")
    v64 = dev(A.data, torch.float64)
    sy = {"rowptr": dev(A.indptr, torch.int32), "col": dev(A.indices, torch.int32), "vals32": v64.to(torch.float32),
          "vals64": v64, "pinv": dev(1.0 / d, torch.float32)}
    b = dev(np.random.default_rng(2).standard_normal(3000), torch.float64)
    mb = MinresBatch([sy])
    want, info = mb.solve(b)
    mb.close()
    rp = sy["rowptr"].clone()
    sy["rowptr"].zero_()
    mb = MinresBatch([sy])
    sy["rowptr"].copy_(rp)
    x, info2 = mb.solve(b)
    assert mb.resident_counts() == (info2[0]["outer"], 0) and torch.equal(x, want)
    mb.close()

    print("[routes] memory", flush=True)
    n = 2_000_000
    ar = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    v = torch.linspace(1, 2, n, dtype=torch.float64, device="cuda")
    sy = {"rowptr": ar, "col": ar[:-1].contiguous(), "vals32": v.to(torch.float32), "vals64": v}
    b = torch.ones_like(v)
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    mb = MinresBatch([sy])
    x, info = mb.solve(b, x=x)
    used = free - torch.cuda.mem_get_info()[0]
    assert info[0]["converged"] and mb.resident_counts() == (0, 0)
    assert used <= 12.6 * 4 * n, used  # 10 FP32 vectors and one of FP64, and the tiles' words
    mb.close()


@pytest.mark.parametrize("n", [1, 2, 4])
def test_elasticity_solution_against_a_direct_solve(n):
    """The resident solve against scipy's sparse LU of the same FP64 matrix: an error is at most the residual
    over the smallest eigenvalue in magnitude (the matrix is symmetric)."""
    import scipy.sparse as sps
    import scipy.sparse.linalg as spla

    print(f"[routes] elasticity against LU n={n}", flush=True)
    y = _elasticity(n)
    x, info = y.solve(rtol=1e-10)
    assert info["converged"] and y.last_resident == (info["outer"], 0)
    rp, col, _, v64 = (v.cpu().numpy() for v in y.full("A"))
    A = sps.csc_matrix(sps.csr_matrix((v64, col, rp), shape=(y.n, y.n)))
    assert abs(A - A.T).max() <= 1e-13 * abs(A).max()
    b = -y.rhs64.cpu().numpy()
    lu = spla.splu(A)
    want = lu.solve(b)
    want += lu.solve(b - A @ want)
    inverse = spla.LinearOperator(A.shape, matvec=lu.solve, dtype=np.float64)
    lowest = abs(spla.eigsh(A, k=1, sigma=0.0, OPinv=inverse, which="LM", return_eigenvectors=False)[0])
    err, bound = np.linalg.norm(x.cpu().numpy() - want), 1e-10 * np.linalg.norm(b) / lowest
    print(f"[routes] error {err:.2e}, bound {bound:.2e}, |x| {np.linalg.norm(want):.2e}", flush=True)
    assert err <= 1.1 * bound
