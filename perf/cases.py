"""What is timed: the work that a program built on this package has it do, through its public calls.

Assembly of mixed Darcy systems (one system, or a batch in one set of launches) and of dual-mixed
elasticity, the solves that follow them, a training step of the learned smoother, and a time step of
the mixed-dimensional model. Meshes are the structured simplex meshes of the benchmark and the tests
(n x n x 2 triangles, n x n x n x 6 tetrahedra), coefficients are the log-normal fields the benchmark
uses, drawn on the device from the seed.

``listed`` holds the cases, ``draw`` gives more of the same ranges; see each kind's functions below.
"""

import functools
import math

import numpy as np
import torch

DEV = "cuda"


# ---- the cases ------------------------------------------------------------------------------------
def listed():
    return [
        # the reference's own 2-D case: both precisions, as a program that will solve needs them;
        # a few microseconds of kernel, so launches and the host path count
        _assembly("darcy2d-rt1-both-32", 2, 1, 32, "both"),
        # the benchmark's warm assembly (196,608 tetrahedra)
        _assembly("darcy3d-rt1-f32-32", 3, 1, 32, "f32"),
        # second-degree elements on an odd mesh (41,154 tetrahedra)
        _assembly("darcy3d-rt2-f32-19", 3, 2, 19, "f32"),
        # dual-mixed elasticity: operator and residual (10,368 tetrahedra)
        {"name": "elasticity-assembly-12", "kind": "elasticity_assembly", "n": 12, "operator": "A", "precision": "f32",
         "sigma": 0.5},
        # 24 systems of both degrees in one set of launches
        {"name": "batch-assembly-24", "kind": "batch_assembly", "count": 24, "lo": 4, "hi": 12, "mix": 1, "sigma": 1.0},
        # the driver flow of the reference: coefficients as Python callables, scatter, KSP solve, host
        # vectors in and out, on its 2-D case
        {"name": "driver2d-32", "kind": "driver", "n": 32, "sigma": 1.0},
        # block-preconditioned MINRES to 1e-8 on a small second-degree system (3,072 tetrahedra)
        _solve("minres3d-rt2-8", 3, 2, 8),
        # preconditioner set-up and solve to 1e-8 with the learned two-grid preconditioner, at the
        # benchmark's size
        {"name": "learned-solve-32", "kind": "learned_solve", "n": 32, "sigma": 2.0},
        # dual-mixed elasticity: two-grid set-up and solve to 1e-8 (3,072 tetrahedra)
        {"name": "elasticity-solve-8", "kind": "elasticity_solve", "n": 8, "sigma": 0.5},
        # 12 systems of both degrees solved together with the batched two-grid preconditioner
        {"name": "batch-solve-12", "kind": "batch_solve", "count": 12, "lo": 4, "hi": 9, "mix": 1, "sigma": 1.0},
        # one backward-Euler step of the mixed-dimensional model
        {"name": "mixed-dim-step-16", "kind": "mixed_dim", "n": 16, "fractures": 5, "dt": 1e-3},
        # forward, loss and backward of the learned smoother (24,576 cells)
        {"name": "train-16", "kind": "train", "n": 16, "samples": 12, "sigma": 2.0},
    ]


def draw(rng):
    kind = rng.choice(["assembly", "assembly", "elasticity_assembly", "batch_assembly", "driver", "solve",
                       "learned_solve", "elasticity_solve", "batch_solve", "mixed_dim", "train"])

    def size(lo, hi):
        return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))

    def sigma(hi):
        return round(rng.uniform(0.3 * hi, hi), 3)

    if kind == "assembly":
        dim, degree = rng.choice([(2, 1), (2, 2), (3, 1), (3, 2)])
        hi = {(2, 1): 181, (2, 2): 90, (3, 1): 32, (3, 2): 19}[(dim, degree)]
        precision = rng.choice(["f32", "f64", "both"])
        if precision != "f32":
            hi = int(hi * 0.75)
        return _assembly(None, dim, degree, size(6 if dim == 2 else 3, hi), precision,
                         rng.choice(["cell", "cell", "point"]), sigma(2.0))
    if kind == "elasticity_assembly":
        return {"kind": kind, "n": size(3, 12), "operator": rng.choice(["A", "A", "P"]),
                "precision": rng.choice(["f32", "f32", "f64"]), "sigma": sigma(0.5)}
    if kind == "batch_assembly":
        return {"kind": kind, "count": size(4, 24), "lo": rng.randint(3, 5), "hi": rng.randint(6, 11),
                "mix": rng.randint(2, 10 ** 6), "sigma": sigma(2.0)}
    if kind == "driver":
        return {"kind": kind, "n": size(8, 48), "sigma": sigma(1.0)}
    if kind == "solve":
        dim, degree = rng.choice([(2, 1), (2, 2), (3, 1), (3, 2)])
        hi = {(2, 1): 64, (2, 2): 32, (3, 1): 24, (3, 2): 9}[(dim, degree)]
        return _solve(None, dim, degree, size(8 if dim == 2 else 4, hi), sigma(1.0))
    if kind == "learned_solve":
        return {"kind": kind, "n": size(6, 31), "sigma": sigma(2.0)}
    if kind == "elasticity_solve":
        return {"kind": kind, "n": size(3, 8), "sigma": sigma(0.5)}
    if kind == "batch_solve":
        return {"kind": kind, "count": size(3, 12), "lo": rng.randint(3, 5), "hi": rng.randint(6, 8),
                "mix": rng.randint(2, 10 ** 6), "sigma": sigma(1.0)}
    if kind == "mixed_dim":
        return {"kind": kind, "n": size(8, 16), "fractures": rng.randint(2, 5),
                "dt": float("%.3g" % 10.0 ** rng.uniform(-3.3, -2.0))}
    return {"kind": "train", "n": size(5, 16), "samples": rng.choice([8, 12, 13]), "sigma": sigma(2.0)}


def _assembly(name, dim, degree, n, precision, coefficients="cell", sigma=2.0):
    """Warm assembly: CSR values and residual with the Dirichlet term, pattern kept. ``coefficients``:
    one value per cell, or one per quadrature point."""
    c = {"kind": "assembly", "dim": dim, "degree": degree, "n": n, "precision": precision,
         "coefficients": coefficients, "sigma": sigma}
    return {"name": name, **c} if name else c


def _solve(name, dim, degree, n, sigma=1.0):
    """Preconditioner, MINRES and FP64 refinement to 1e-8 on an assembled system."""
    c = {"kind": "solve", "dim": dim, "degree": degree, "n": n, "sigma": sigma}
    return {"name": name, **c} if name else c


# ---- sizes ----------------------------------------------------------------------------------------
def _sizes(dim, degree, n):
    """Elements, rows and CSR entries of the mixed Darcy system on the structured mesh."""
    if dim == 2:
        E, F, Fb = 2 * n * n, 3 * n * n + 2 * n, 4 * n
        nf, ni, npr = (1, 0, 1) if degree == 1 else (2, 2, 3)
        nl = 3 * nf + ni + npr
    else:
        E, F, Fb = 6 * n ** 3, 12 * n ** 3 + 6 * n * n, 12 * n * n
        nf, ni, npr = (1, 0, 1) if degree == 1 else (3, 3, 4)
        nl = 4 * nf + ni + npr
    nnz = nf * ((F - Fb) * (2 * nl - nf) + Fb * nl) + (ni + npr) * E * nl
    return E, nf * F + (ni + npr) * E, nnz


def _specs(case):
    """(n, degree) of a batch's systems: uneven sizes, both degrees, fixed by the case."""
    r = np.random.default_rng(case["mix"])
    return list(zip(r.integers(case["lo"], case["hi"] + 1, case["count"]).tolist(),
                    r.integers(1, 3, case["count"]).tolist()))


def work(case):
    kind = case["kind"]
    if kind in ("assembly", "batch_assembly"):
        specs = [(3,) + s for s in _specs(case)] if kind == "batch_assembly" else [
            (case["dim"], case["degree"], case["n"])]
        out = {"bytes": 0, "flops": 0}
        for dim, *rest in specs:
            degree, n = (rest[1], rest[0]) if kind == "batch_assembly" else rest
            E, N, nnz = _sizes(dim, degree, n)
            for size in {"f32": (4,), "f64": (8,), "both": (4, 8)}[case.get("precision", "f32")]:
                # vertex ids, vertices, coefficient, facet ids and signs in; values and residual out
                out["bytes"] += E * (4 * (dim + 1) * 2 + 1 + size * (dim + 1)) + size * (nnz + N)
                out["flops"] += 12 * nnz
        return out
    if kind in ("elasticity_assembly", "elasticity_solve"):
        n = case["n"]
        E, F = 6 * n ** 3, 12 * n ** 3 + 6 * n * n
        N, nnz = 9 * F + 6 * E, 662 * E
        if kind == "elasticity_assembly":
            size = 8 if case["precision"] == "f64" else 4
            return {"bytes": 241 * E + size * (nnz + N), "flops": 29376 * E}
        return {"bytes": 16 * nnz + 16 * N, "flops": 4 * nnz}
    if kind == "batch_solve":
        tot = [_sizes(3, k, n) for n, k in _specs(case)]
        N, nnz = sum(t[1] for t in tot), sum(t[2] for t in tot)
    elif kind == "train":
        E = 6 * case["n"] ** 3
        agg = max(1, case["n"] // 2) ** 3
        net = E * (2 * 8 * 64 + 4 * 2 * 128 * 64)
        return {"bytes": E * (16 + 40 + 16 + 4 * case["samples"]) + 4 * 33730 * 2,
                "flops": 3 * net + 2 * case["samples"] * (agg ** 2 + 15 * E)}
    elif kind == "mixed_dim":
        _, N, nnz = _sizes(3, 1, case["n"])
    else:
        dim, degree = {"driver": (2, 1), "learned_solve": (3, 1)}.get(kind) or (case["dim"], case["degree"])
        _, N, nnz = _sizes(dim, degree, case["n"])
    return {"bytes": 12 * nnz + 16 * N, "flops": 2 * nnz}


def tolerance(case):
    """Assembled values: the rounding of their precision, measured against 64 bits. Solves stop at a
    relative residual of 1e-8: two correct ones differ in the unknowns by that times the system's
    conditioning. Training: activations are stored in bf16, so a gradient carries its rounding."""
    kind = case["kind"]
    if kind in ("assembly", "elasticity_assembly"):
        return {"rel": 1e-12} if case["precision"] == "f64" else {"rel": 1e-6}
    if kind == "batch_assembly":
        return {"rel": 1e-6}
    if kind == "train":
        return {"rel": 4e-3, "max": 0.1}
    return {"rel": 1e-6, "max": 1e-4}


# ---- meshes and spaces: built once for a size, as a program does ------------------------------------
@functools.lru_cache(maxsize=4)
def _darcy_space(dim, degree, n):
    from nfempy_amd.mesh import Mesh, unit_cube, unit_square
    from nfempy_amd.pattern import build_pattern
    from nfempy_amd.spaces import ProductSpace

    mesh = Mesh.from_blocks(dim, *(unit_square(n) if dim == 2 else unit_cube(n)))
    space = ProductSpace({"u": (dim, 1, "RT", degree, mesh), "p": (dim, 1, "Lagrange", degree - 1, mesh)})
    space.make_subspaces_discontinuous({"p": True})
    space.build_structures({"u": [1], "p": [1]}, {"u": [2, 3, 4, 5] if dim == 2 else [2, 3, 4, 5, 6, 7]})
    dest, sign = space.reference_destinations()
    return space, build_pattern(space.n_dof, dest, sign)


def _darcy_system(dim, degree, n):
    from nfempy_amd.device import DarcySystem

    space, pattern = _darcy_space(dim, degree, n)
    return DarcySystem(space, device=DEV, pattern=pattern)


def _field(sysd, seed, ell, sigma):
    """Gaussian field at the cell centres, as the benchmark draws it."""
    from nfempy_amd.fields import grf_device

    return grf_device(sysd.coords64[sysd.cells.long()].mean(dim=1), seed=seed, ell=ell, sigma=sigma, n_features=256)


def _darcy_data(sysd, seed, coefficients="cell", ell=0.1, sigma=1.0):
    """Inverse permeability, source and boundary pressure as the assembly's arguments."""
    from nfempy_amd.device import CoefficientArg

    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    rand = lambda *s: torch.rand(*s, generator=gen, device=DEV, dtype=torch.float64)
    kinv = torch.exp(-_field(sysd, seed, ell, sigma))
    source = 1.0 + 0.5 * rand(sysd.E)
    pd = CoefficientArg(rand(sysd.F * sysd.nqf).contiguous(), sysd.nqf, 1)
    if coefficients == "point":
        kinv = (kinv[:, None] * (1.0 + 0.2 * rand(sysd.E, sysd.nq))).reshape(-1).contiguous()
        source = (source[:, None] * (1.0 + 0.2 * rand(sysd.E, sysd.nq))).reshape(-1).contiguous()
        return CoefficientArg(kinv, sysd.nq, 1), CoefficientArg(source, sysd.nq, 1), pd
    return CoefficientArg(kinv.contiguous(), 1, 0), CoefficientArg(source, 1, 0), pd


def _elasticity_system(case, seed):
    from nfempy_amd.elasticity import ElasticitySystem

    space = _elasticity_space(case["n"])
    E = 6 * case["n"] ** 3
    r = np.random.default_rng(seed)
    lam, mu = (np.exp(case["sigma"] * r.standard_normal(E)) for _ in range(2))
    force = r.uniform(0.25, 1.0, 3)
    rhs = lambda x, y, z: np.array([f * np.ones_like(x) for f in force] + [np.zeros_like(x)] * 3)
    return ElasticitySystem(space, {"lambda": lam, "mu": mu, "rhs": rhs}), lam, mu, force


@functools.lru_cache(maxsize=2)
def _elasticity_space(n):
    from nfempy_amd.mesh import Mesh, unit_cube
    from nfempy_amd.spaces import ProductSpace

    mesh = Mesh.from_blocks(3, *unit_cube(n))
    space = ProductSpace({"s": (3, 3, "BDM", 1, mesh), "u": (3, 3, "Lagrange", 0, mesh),
                          "t": (3, 3, "Lagrange", 0, mesh)})
    space.make_subspaces_discontinuous({"u": True, "t": True})
    space.build_structures({"s": [1], "u": [1], "t": [1]}, {"s": [2, 3, 4, 5, 6, 7]})
    return space


def _driver_functions(case, seed):
    """Permeability, source and boundary pressure as callables of the coordinates."""
    a, b, c = np.random.default_rng(seed).uniform(0.2, 1.0, 3)
    kappa = lambda x, y, z: np.exp(case["sigma"] * a * np.sin(3.0 * x) * np.cos(2.0 * y))
    rhs = lambda x, y, z: np.array([2 * np.pi ** 2 * np.sin(np.pi * x) * np.sin(np.pi * y) + b])
    p = lambda x, y, z: np.array([c * x * (1.0 - y)])
    return kappa, rhs, p


# ---- prepare and run --------------------------------------------------------------------------------
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_assembly(case, seed):
    sysd = _darcy_system(case["dim"], case["degree"], case["n"])
    return {"run": _run_assembly, "sys": sysd, "data": _darcy_data(sysd, seed, case["coefficients"], sigma=case["sigma"]),
            "fp64": {"f32": (False,), "f64": (True,), "both": (True, False)}[case["precision"]]}


def _run_assembly(s):
    return [dict(zip(("values", "residual"), s["sys"].assemble(*s["data"], fp64=fp64))) for fp64 in s["fp64"]]


def _prepare_elasticity_assembly(case, seed):
    sysd = _elasticity_system(case, seed)[0]
    return {"run": _run_elasticity_assembly, "sys": sysd, "which": case["operator"],
            "fp64": case["precision"] == "f64"}


def _run_elasticity_assembly(s):
    values, residual = s["sys"].assemble(s["which"], fp64=s["fp64"])
    return {"values": values, "residual": residual} if s["which"] == "A" else {"values": values}


def _prepare_batch(case, seed):
    from nfempy_amd.batch import DarcyBatch

    return DarcyBatch(_specs(case), seed=1000 * (seed % 100000), ell=0.1, sigma=case["sigma"], workers=1)


def _prepare_batch_assembly(case, seed):
    batch = _prepare_batch(case, seed)
    batch.capture()
    return {"run": _run_batch_assembly, "batch": batch}


def _run_batch_assembly(s):
    s["batch"].assemble()
    return [{"values": i["vals"], "residual": i["rhs"]} for i in s["batch"].instances]


def _prepare_driver(case, seed):
    from nfempy_amd.assembly import SequentialAssembler
    from nfempy_amd.mesh import Mesh, unit_square
    from nfempy_amd.spaces import ProductSpace
    from nfempy_amd.weak_forms import LaplaceDualWeakForm, LaplaceDualWeakFormBCDirichlet

    mesh = Mesh.from_blocks(2, *unit_square(case["n"]))
    space = ProductSpace({"u": (2, 1, "RT", 1, mesh), "p": (2, 1, "Lagrange", 0, mesh)})
    space.make_subspaces_discontinuous({"p": True})
    space.build_structures({"u": [1], "p": [1]}, {"u": [2, 3, 4, 5]})
    kappa, rhs, p = _driver_functions(case, seed)
    form = LaplaceDualWeakForm(space)
    form.functions = {"rhs": rhs, "kappa": kappa}
    form.scatter(None, None)  # the pattern and the device arrays, which the space then keeps
    return {"run": _run_driver, "space": space, "forms": (LaplaceDualWeakForm, LaplaceDualWeakFormBCDirichlet),
            "assembler": SequentialAssembler, "kappa": kappa, "rhs": rhs, "p": p}


def _run_driver(s):
    import warnings

    from nfempy_amd.assembly import Mat
    from nfempy_amd.ksp import KSP

    space = s["space"]
    A, rg = Mat(), np.zeros(space.n_dof)
    A.createAIJ([space.n_dof, space.n_dof])
    form, bc = (cls(space) for cls in s["forms"])
    form.functions, bc.functions = {"rhs": s["rhs"], "kappa": s["kappa"]}, {"p": s["p"]}
    u = space.discrete_spaces["u"]
    assembler = s["assembler"](space, A, rg)
    alpha = np.zeros(space.n_dof)
    assembler.form_to_input_list = {"mixed": ["form", range(len(u.elements)), form, alpha],
                                    "dirichlet": ["bc_form", range(len(u.bc_elements)), bc, alpha]}
    assembler.scatter_forms()
    A.assemble()
    ksp = KSP().create()
    ksp.setOperators(A)
    b, x = A.createVecLeft(), A.createVecRight()
    b.array[:] = -rg
    ksp.setType("preonly")
    ksp.getPC().setType("lu")
    ksp.setTolerances(rtol=1e-8)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)
        ksp.solve(b, x)
    return {"residual": rg, "flux": x.array[:u.n_dof], "pressure": x.array[u.n_dof:]}


def _assembled(dim, degree, n, seed, ell=0.1, sigma=1.0):
    sysd = _darcy_system(dim, degree, n)
    data = _darcy_data(sysd, seed, ell=ell, sigma=sigma)
    for fp64 in (True, False):
        sysd.assemble(*data, fp64=fp64)
    return sysd, data


def _split(x, n_u):
    return {"flux": x[:n_u], "pressure": x[n_u:]}


def _prepare_solve(case, seed):
    sysd, data = _assembled(case["dim"], case["degree"], case["n"], seed, sigma=case["sigma"])
    return {"run": _run_solve, "sys": sysd, "data": data}


def _run_solve(s):
    from nfempy_amd.solvers import MinresIR, darcy_preconditioner

    y = s["sys"]
    sign, pinv = darcy_preconditioner(y.rowptr, y.col, y.vals64, y.n, y.n_u)
    solver = MinresIR(y.rowptr, y.col, y.vals32, y.vals64, sign, pinv)
    x, _ = solver.solve(-y.rhs64, rtol=1e-8, max_inner=100000)
    solver.close()
    return _split(x, y.n_u)


def _prepare_learned_solve(case, seed):
    from nfempy_amd.learned import Fgmres, LearnedSchurPC, default_weights_path, load_params

    sysd, data = _assembled(3, 1, case["n"], seed, ell=0.05, sigma=case["sigma"])
    pc = LearnedSchurPC(sysd, load_params(default_weights_path()))
    pc.setup()
    return {"run": _run_learned_solve, "sys": sysd, "data": data, "pc": pc, "solver": Fgmres(sysd.n, 40)}


def _run_learned_solve(s):
    from nfempy_amd.learned import solve_learned

    s["pc"].setup()
    x, _ = solve_learned(s["sys"], s["pc"], -s["sys"].rhs64, rtol=1e-8, solver=s["solver"])
    return _split(x, s["sys"].n_u)


def _prepare_elasticity_solve(case, seed):
    sysd = _elasticity_system(case, seed)[0]
    for fp64 in (True, False):
        sysd.assemble("A", fp64=fp64)
    sysd.twogrid()
    return {"run": _run_elasticity_solve, "sys": sysd}


def _run_elasticity_solve(s):
    x, _ = s["sys"].solve(rtol=1e-8)
    cut = s["sys"].field_bounds
    return {name: x[a:b] for name, a, b in zip(("stress", "displacement", "rotation"), cut, cut[1:])}


def _prepare_batch_solve(case, seed):
    batch = _prepare_batch(case, seed)
    batch.assemble()
    batch.solve_batched(rtol=1e-2, pc="learned")  # the cold structure of the preconditioner
    return {"run": _run_batch_solve, "batch": batch}


def _run_batch_solve(s):
    s["batch"].assemble()
    return s["batch"].solve_batched(rtol=1e-8, pc="learned")[0]


def _prepare_mixed_dim(case, seed):
    from nfempy_amd.mixed_dim import MixedDimDarcy

    a, b = np.random.default_rng(seed).uniform(0.5, 1.5, 2)
    model = MixedDimDarcy(_fractures(case["n"], case["fractures"]), dt=case["dt"], kappa_matrix=float(a),
                          p_boundary=lambda x, y, z: b * (1.0 - x) + 0.2 * y)
    model.setup()
    x = torch.zeros(model.N, dtype=torch.float64, device=DEV)
    for _ in range(2):  # a state inside the run, not its first step
        x, _ = model.step(x)
    return {"run": _run_mixed_dim, "model": model, "x": x}


@functools.lru_cache(maxsize=2)
def _fractures(n, count):
    from nfempy_amd.mixed_dim import FractureNetwork

    return FractureNetwork(n, count=count, seed=2026)


def _run_mixed_dim(s):
    x, _ = s["model"].step(s["x"])
    return _split(x, s["model"].n_u)


def _prepare_train(case, seed):
    from nfempy_amd.learned import LearnedSchurPC, SmootherTrainer, default_weights_path, load_params

    sysd, data = _assembled(3, 1, case["n"], seed, ell=0.05, sigma=case["sigma"])
    pc = LearnedSchurPC(sysd, coarse_fp16=False)
    trainer = SmootherTrainer(pc, load_params(default_weights_path()), n_random=case["samples"], seed=seed)
    pc.setup()
    return {"run": _run_train, "sys": sysd, "data": data, "pc": pc, "trainer": trainer, "e": trainer.samples()}


def _run_train(s):
    pc, trainer = s["pc"], s["trainer"]
    pc.schur(s["sys"].vals64)
    pc.forward()
    pc.coarse()
    loss = trainer.loss_and_gamma(s["e"])
    return {"loss": loss, "gradient": trainer.backward(), "smoother_diag": pc.Wd, "smoother_off": pc.Wo}


# ---- the same in 64 bits, from the plan's numbering and reference basis --------------------------------
def exact(case, seed):
    f = globals().get("_exact_" + case["kind"])
    return None if f is None else f(case, seed)


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a)).to(DEV)


def _scatter(n, rowptr, col, dest, sign, K, upper=False):
    """CSR values of element matrices K at rows and columns dest; entries not in the pattern are left out."""
    rp = rowptr.long()
    keys = torch.repeat_interleave(torch.arange(n, device=DEV), rp[1:] - rp[:-1]) * n + col.long()
    want = (dest[:, :, None] * n + dest[:, None, :]).reshape(-1)
    vals = (K * sign[:, :, None] * sign[:, None, :]).reshape(-1)
    at = torch.searchsorted(keys, want).clamp(max=len(keys) - 1)
    ok = keys[at] == want
    if upper:
        ok &= (dest[:, :, None] <= dest[:, None, :]).reshape(-1)
    return torch.zeros(len(keys), dtype=torch.float64, device=DEV).index_add_(0, at[ok], vals[ok])


def _geometry(points, cells):
    X = _dev(points)[cells.long()]
    J = (X[:, 1:] - X[:, :1]).transpose(1, 2)  # (E, 3, dim)
    return J, torch.sqrt(torch.linalg.det(J.transpose(1, 2) @ J))


def _quadrature_values(c, E, nq):
    a = c.arr.to(torch.float64)
    return a[:, None].expand(E, nq) if c.sq == 0 and c.se == 1 else (
        a.expand(E, nq) if c.se == 0 else a.reshape(E, nq))


def _exact_darcy(sysd, data):
    """(values, residual) of [[M, -B^T], [B, 0]] with the Dirichlet facet term."""
    E, nb, nq = sysd.E, sysd.nb, sysd.nq
    mesh = sysd.u_sp.mesh
    J, det = _geometry(mesh.points, sysd.cells)
    w = _dev(sysd.qweights)
    tab = sysd.u_el.tabulate(sysd.qpoints)
    phi, div = _dev(tab[0]), _dev(np.einsum("kqjk->qj", tab[1:]))
    psi = _dev(sysd.p_el.tabulate(sysd.qpoints)[0, :, :, 0])
    kinv, f = (_quadrature_values(c, E, nq) for c in data[:2])
    P = torch.einsum("ecd,qad->eqac", J, phi)
    M = torch.einsum("eq,eqac,eqbc->eab", kinv * w / det[:, None], P, P)
    B = torch.einsum("q,qa,qk->ka", w, div, psi).expand(E, -1, -1)
    K = torch.zeros((E, sysd.nl, sysd.nl), dtype=torch.float64, device=DEV)
    K[:, :nb, :nb], K[:, nb:, :nb], K[:, :nb, nb:] = M, B, -B.transpose(1, 2)
    dest, sign = _dev(sysd.ref_dest.astype(np.int64)), _dev(sysd.ref_sign)
    vals = _scatter(sysd.n, sysd.rowptr, sysd.col, dest, sign, K)
    rg = torch.zeros(sysd.n, dtype=torch.float64, device=DEV)
    rg.index_add_(0, dest[:, nb:].reshape(-1), -torch.einsum("eq,q,e,qk->ek", f, w, det, psi).reshape(-1))
    # facets: sum_q w |F| p_D psi . n, n the outward unit normal of the neighbour cell
    fn, ne = sysd.bc_facet.long(), sysd.bc_neigh.long()
    X = _dev(mesh.points)[fn]
    T = X[:, 1:] - X[:, :1]
    detf = torch.sqrt(torch.linalg.det(T @ T.transpose(1, 2)))
    if sysd.dim == 2:
        nrm = torch.stack([T[:, 0, 1], -T[:, 0, 0], torch.zeros_like(detf)], 1)
    else:
        nrm = torch.linalg.cross(T[:, 0], T[:, 1])
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    inside = _dev(mesh.points)[sysd.cells.long()[ne]].mean(1) - X.mean(1)
    nrm = nrm * -torch.sign((nrm * inside).sum(1, keepdim=True))
    trace = sysd.bc_trace64[sysd.bc_combo.long()]  # (F, nqf, fd, dim)
    flux = torch.einsum("fcd,fqad,fc->fqa", J[ne], trace, nrm) / det[ne][:, None, None]
    pd = data[2].arr.to(torch.float64).reshape(sysd.F, sysd.nqf)
    r = torch.einsum("q,f,fq,fqa->fa", sysd.bc_fw64, detf, pd, flux)
    rows = sysd.bc_rows.long()
    rg.index_add_(0, (rows & ((1 << 28) - 1)).reshape(-1),
                  torch.where((rows >> 30) & 1 == 1, -r, r).reshape(-1))
    return vals, rg


def _exact_assembly(case, seed):
    s = _prepare_assembly(case, seed)
    values, residual = _exact_darcy(s["sys"], s["data"])
    return [{"values": values, "residual": residual} for _ in s["fp64"]]


def _exact_batch_assembly(case, seed):
    from nfempy_amd.device import CoefficientArg

    out = []
    for inst in _prepare_batch(case, seed).instances:
        y = inst["system"]
        zero = CoefficientArg(torch.zeros(y.F * y.nqf, dtype=torch.float64, device=DEV), y.nqf, 1)
        values, residual = _exact_darcy(y, (inst["kinv"], inst["f"], zero))
        out.append({"values": values, "residual": residual})
    return out


def _exact_elasticity_assembly(case, seed):
    y, lam, mu, force = _elasticity_system(case, seed)
    space = _elasticity_space(case["n"])
    points, weights = space.quadrature[3]
    tab = y.s_sp.element.tabulate(points)
    J, det = _geometry(y.s_sp.mesh.points, y.cells)
    w, lam, mu = _dev(weights), _dev(lam), _dev(mu)
    phi = torch.einsum("ecd,qad->eqac", J, _dev(tab[0])) / det[:, None, None, None]
    div = _dev(np.einsum("kqjk->qj", tab[1:]))
    E, nb = len(det), phi.shape[2]
    K = torch.zeros((E, 42, 42), dtype=torch.float64, device=DEV)
    dw = det[:, None] * w
    mass = torch.einsum("eq,eqac,eqbc->eab", dw, phi, phi) / (2 * mu)[:, None, None]
    flat = phi.reshape(E, len(w), -1)  # entry 3 a + c: direction c of basis a pairs with stress row c
    K[:, :36, :36] -= torch.einsum("eq,eqi,eqj->eij", dw * (lam / (2 * mu * (2 * mu + 3 * lam)))[:, None], flat, flat)
    for c in range(3):
        K[:, c:36:3, c:36:3] += mass
    if case["operator"] == "A":
        ub = torch.einsum("q,qa->a", w, div)
        first = torch.einsum("eq,eqac->eac", dw, phi)
        skew = {0: [(2, 1, 1.0), (1, 2, -1.0)], 1: [(0, 2, 1.0), (2, 0, -1.0)], 2: [(1, 0, 1.0), (0, 1, -1.0)]}
        for c in range(3):
            K[:, 36 + c, c:36:3] += ub
            K[:, c:36:3, 36 + c] += ub
            for row, d, s in skew[c]:
                K[:, 39 + c, row:36:3] -= s * first[:, :, d]
                K[:, row:36:3, 39 + c] -= s * first[:, :, d]
    else:
        dd = torch.einsum("q,qa,qb->ab", w, div, div)[None] / det[:, None, None]
        for c in range(3):
            K[:, c:36:3, c:36:3] += dd
        vol = det * w.sum()
        for i in range(36, 42):
            K[:, i, i] = vol
    dest, sign = _dev(y.ref_dest.astype(np.int64)), _dev(y.ref_sign)
    op = y.ops[case["operator"]]
    out = {"values": _scatter(y.n, op["rowptr"], op["col"], dest, sign, K, upper=True)}
    if case["operator"] == "A":
        rg = torch.zeros(y.n, dtype=torch.float64, device=DEV)
        r = -(det * w.sum())[:, None] * _dev(force)
        out["residual"] = rg.index_add_(0, dest[:, 36:39].reshape(-1), r.reshape(-1))
    return out


def _solve64(n, n_u, rowptr, col, vals, b):
    """x of A x = b in 64 bits: MINRES on diag(I, -I) A with a block-diagonal preconditioner, repeated
    on the residual."""
    rp, ci = rowptr.long(), col.long()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), rp[1:] - rp[:-1])
    sign = torch.ones(n, dtype=torch.float64, device=DEV)
    sign[n_u:] = -1.0
    A = torch.sparse_csr_tensor(rp, ci, vals * sign[rows], size=(n, n))
    diag = torch.zeros(n, dtype=torch.float64, device=DEV)
    on = rows == ci
    diag[rows[on]] = vals[on]
    sub = (rows >= n_u) & (ci < n_u)
    prec = diag.clone()
    prec[n_u:] = 0.0
    prec.index_add_(0, rows[sub], vals[sub] ** 2 / diag[ci[sub]])
    pinv = 1.0 / prec.abs()
    b = b * sign
    x = torch.zeros_like(b)
    for _ in range(4):
        r = b - A @ x
        if float(r.norm()) <= 1e-13 * float(b.norm()):
            break
        x = x + _minres64(A, pinv, r, 1e-9)
    return x


def _minres64(A, pinv, b, tol, most=20000):
    one = torch.ones((), dtype=torch.float64, device=DEV)
    x, w, w2 = torch.zeros_like(b), torch.zeros_like(b), torch.zeros_like(b)
    r1, r2, y = b, b, pinv * b
    beta = beta1 = torch.sqrt(b @ y)
    oldb = dbar = eps = one * 0.0
    phibar, cs, sn = beta1, -one, one * 0.0
    for it in range(most):
        v = y / beta
        y = A @ v
        if it:
            y = y - (beta / oldb) * r1
        alfa = v @ y
        y = y - (alfa / beta) * r2
        r1, r2 = r2, y
        y = pinv * r2
        oldb, beta = beta, torch.sqrt(r2 @ y)
        oldeps, delta = eps, cs * dbar + sn * alfa
        gbar, eps, dbar = sn * dbar - cs * alfa, sn * beta, -cs * beta
        gamma = torch.sqrt(gbar * gbar + beta * beta)
        cs, sn = gbar / gamma, beta / gamma
        phi, phibar = cs * phibar, sn * phibar
        w1, w2 = w2, w
        w = (v - oldeps * w1 - delta * w2) / gamma
        x = x + phi * w
        if it % 100 == 99 and float(phibar) <= tol * float(beta1):
            break
    return x


def _exact_solved(sysd, data):
    values, residual = _exact_darcy(sysd, data)
    return _split(_solve64(sysd.n, sysd.n_u, sysd.rowptr, sysd.col, values, -residual), sysd.n_u)


def _exact_solve(case, seed):
    return _exact_solved(*_assembled(case["dim"], case["degree"], case["n"], seed, sigma=case["sigma"]))


def _exact_learned_solve(case, seed):
    return _exact_solved(*_assembled(3, 1, case["n"], seed, ell=0.05, sigma=case["sigma"]))


def _exact_batch_solve(case, seed):
    from nfempy_amd.device import CoefficientArg

    out = []
    for inst in _prepare_batch(case, seed).instances:
        y = inst["system"]
        zero = CoefficientArg(torch.zeros(y.F * y.nqf, dtype=torch.float64, device=DEV), y.nqf, 1)
        values, residual = _exact_darcy(y, (inst["kinv"], inst["f"], zero))
        out.append(_solve64(y.n, y.n_u, y.rowptr, y.col, values, -residual))
    return out


def _exact_driver(case, seed):
    from nfempy_amd.device import CoefficientArg

    y = _darcy_system(2, 1, case["n"])
    kappa, rhs, p = _driver_functions(case, seed)
    at = lambda f, x: _dev(np.asarray(f(x[..., 0].ravel(), x[..., 1].ravel(), x[..., 2].ravel())).reshape(-1))
    data = (CoefficientArg(1.0 / at(kappa, y.xq), y.nq, 1), CoefficientArg(at(rhs, y.xq), y.nq, 1),
            CoefficientArg(at(p, y.bc_xq), y.nqf, 1))
    values, residual = _exact_darcy(y, data)
    x = _solve64(y.n, y.n_u, y.rowptr, y.col, values, -residual)
    out = _split(x.cpu().numpy(), y.n_u)
    return {"residual": residual.cpu().numpy(), **out}


def _exact_train(case, seed):
    """Loss, smoother and gradient by automatic differentiation, weights as the layers hold them (bf16)."""
    s = _prepare_train(case, seed)
    y, pc, e = s["sys"], s["pc"], s["e"].to(torch.float64)
    values, _ = _exact_darcy(y, s["data"])
    nbr, agg = pc.g.nbr.long().reshape(-1, 4), pc.g.agg_of.long()
    has = nbr >= 0
    q = nbr.clamp(min=0)
    pos = lambda a: a.long().reshape(-1, 4)
    at = lambda p: torch.where(p >= 0, values[p.clamp(min=0)], torch.zeros((), dtype=torch.float64, device=DEV))
    pb, pqb, pm = pos(pc.g.pos_b), pos(pc.g.pos_qb), pos(pc.g.pos_m)
    m = torch.where(pm >= 0, at(pm), torch.ones((), dtype=torch.float64, device=DEV))
    sd, so = (at(pb) ** 2 / m).sum(1), torch.where(has, at(pb) * at(pqb) / m, torch.zeros_like(m))
    a = torch.where(has, -so / torch.sqrt(sd[:, None] * sd[q]), torch.zeros_like(so))
    cnt = has.sum(1)
    lr = torch.where(has, (sd[q] / sd[:, None]).log().abs(), torch.zeros_like(so))
    least = torch.where(has, a, torch.full_like(a, math.inf)).min(1).values
    feats = torch.stack([a.sum(1), a.max(1).values, torch.where(cnt > 0, least, torch.zeros_like(sd)),
                         (sd + so.sum(1)) / sd, lr.sum(1) / cnt.clamp(min=1), lr.max(1).values, cnt / 4.0,
                         torch.ones_like(sd)], 1)
    theta = pc.theta32.to(torch.float64).clone()
    shapes = [(8, 64), (64,)] + [(64, 64), (64, 64), (64,)] * 4 + [(64,), (1,), (64,), (1,)]
    parts, off = [], 0
    for k, shape in enumerate(shapes):
        v = theta[off:off + math.prod(shape)].reshape(shape)
        off += math.prod(shape)
        if len(shape) == 2 or k in (14, 16):
            v = v.to(torch.float32).to(torch.bfloat16).to(torch.float64)
        parts.append(v.clone().requires_grad_(True))
    h = torch.relu(feats @ parts[0] + parts[1])
    for l in range(4):
        wh, wm, bias = parts[2 + 3 * l: 5 + 3 * l]
        msg = sum(a[:, j:j + 1] * h[q[:, j]] for j in range(4))
        h = h + torch.relu(h @ wh + msg @ wm + bias)
    ud, cd, ue, ce = parts[14:]
    wd = (0.65 + h @ ud + cd) / sd
    wo = torch.where(has, a * ((h @ ue)[:, None] + (h @ ue)[q] + ce) / torch.sqrt(sd[:, None] * sd[q]),
                     torch.zeros_like(a))
    mul = lambda d, o, v: d * v + sum(o[:, j] * v[:, q[:, j]] for j in range(4))
    Ac = torch.zeros((pc.g.n_agg,) * 2, dtype=torch.float64, device=DEV)
    Ac.index_put_((agg, agg), sd, accumulate=True)
    Ac.index_put_((agg[:, None].expand(-1, 4)[has], agg[q][has]), so[has], accumulate=True)
    Se = mul(sd, so, e)
    v = e - mul(wd, wo, Se)
    c = torch.zeros((len(e), pc.g.n_agg), dtype=torch.float64, device=DEV).index_add_(1, agg, mul(sd, so, v))
    u = v - torch.linalg.solve(Ac, c.T).T[:, agg]
    loss = ((u * mul(sd, so, u)).sum(1) / (e * Se).sum(1)).mean()
    grads = torch.autograd.grad(loss, parts)
    return {"loss": loss.detach(), "gradient": torch.cat([g.reshape(-1) for g in grads]),
            "smoother_diag": wd.detach(), "smoother_off": wo.detach().reshape(-1)}
