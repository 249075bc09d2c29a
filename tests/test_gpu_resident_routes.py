"""Routes of the MINRES solves: what is refused before a route is chosen, which route a solve takes, and
what it does when the device does not give it the resident one."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(specs, pc="twogrid", seed=3):
    """(DarcyBatch, MinresBatch, right-hand sides, BatchTwoGrid or None) with the preconditioner set up."""
    import torch

    from nfempy_amd.batch import DarcyBatch
    from nfempy_amd.batch_pc import BatchTwoGrid
    from nfempy_amd.learned import default_weights_path, load_params
    from nfempy_amd.solvers import MinresBatch

    b = DarcyBatch(specs, seed=seed, workers=1)
    b.assemble()
    systems = [b.fp64_system(i) for i in range(len(specs))]
    mb = MinresBatch(systems)
    tg = None
    if pc != "diag":
        theta = load_params(default_weights_path()) if pc == "learned" else None
        tg = BatchTwoGrid([inst["system"] for inst in b.instances], mb.offsets, theta=theta)
        mb.set_pc(tg.setup([s["vals64"] for s in systems]))
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
