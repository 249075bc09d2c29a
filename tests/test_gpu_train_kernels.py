"""The training step's kernels on synthetic cell graphs at the sizes where their tiling can go
wrong (one node, one less and one more than a tile, a ragged last tile, more tiles than blocks),
against the FP64 oracle."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(E, seed):
    """A ring with chords (every node up to 4 neighbours, symmetric couplings) and its S in ELL form."""
    rng = np.random.default_rng(seed)
    nbr = -np.ones((E, 4), np.int64)
    soff = np.zeros((E, 4))
    for k, step in ((0, 1), (2, 7)):
        if E <= 2 * step:
            continue
        c = -rng.uniform(0.1, 0.3, E)
        p = np.arange(E)
        q = (p + step) % E
        nbr[p, k], soff[p, k] = q, c
        nbr[q, k + 1], soff[q, k + 1] = p, c
    sdiag = 0.2 + np.abs(soff).sum(1) + rng.uniform(0.0, 0.5, E)
    return nbr, sdiag, soff


def _dev(a, dt):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=dt)


def _bf(t):
    import torch

    return t.view(torch.bfloat16).double().cpu().numpy()


@pytest.mark.parametrize("E", [1, 3, 31, 63, 64, 65, 750, 40001])
def test_network_backward_sizes(E):
    """Gradient per parameter group against the FP64 backward on the device's own activations: FP32
    sums of up to E terms, relative L2 error 1e-4 (eps * sqrt(E) is 1.2e-5 at 40,001)."""
    import torch
    import oracle.learned as ol
    from nfempy_amd import _native as nat
    from nfempy_amd.learned import param_layout

    nbr, sdiag, soff = _graph(E, E)
    rng = np.random.default_rng(E + 1)
    lay, n_par = param_layout()
    theta = (rng.standard_normal(n_par) * 0.15).astype(np.float32)
    f32, f64, i32 = torch.float32, torch.float64, torch.int32
    d = {"nbr": _dev(nbr, i32), "sd": _dev(sdiag, f64), "so": _dev(soff, f64), "t32": _dev(theta, f32)}
    d["t16"] = d["t32"].to(torch.bfloat16).view(torch.int16).contiguous()
    new = lambda n, dt: torch.zeros(n, dtype=dt, device="cuda")
    a, x, sd32, so32 = new(4 * E, f32), new(8 * E, f32), new(E, f32), new(4 * E, f32)
    h, m, z = new(5 * E * 64, torch.int16), new(4 * E * 64, torch.int16), new(5 * E * 64, f32)
    Wd, Wo = new(E, f32), new(4 * E, f32)
    s = nat.stream_handle()
    nat.call("nfx_gnn_features", E, nat.ptr(d["nbr"]), nat.ptr(d["sd"]), nat.ptr(d["so"]), nat.ptr(a), nat.ptr(x),
             nat.ptr(sd32), nat.ptr(so32), s)
    nat.call("nfx_gnn_forward", E, nat.ptr(d["nbr"]), nat.ptr(a), nat.ptr(x), nat.ptr(d["t32"]), nat.ptr(d["t16"]),
             nat.ptr(h), nat.ptr(m), nat.ptr(z), nat.ptr(d["sd"]), nat.ptr(Wd), nat.ptr(Wo), s)
    gd, go = rng.standard_normal(E).astype(np.float32), rng.standard_normal((E, 4)).astype(np.float32)
    go[nbr < 0] = 0.0
    gdd, god = _dev(gd, f32), _dev(go, f32)
    dh, dm, grad = new(E * 64, f32), new(E * 64, f32), new(n_par, f32)
    part = torch.full((nat.call("nfx_gnn_backward_workspace", E),), float("nan"), dtype=f32, device="cuda")
    nat.call("nfx_gnn_backward", E, nat.ptr(d["nbr"]), nat.ptr(a), nat.ptr(x), nat.ptr(d["t16"]), nat.ptr(h),
             nat.ptr(m), nat.ptr(z), nat.ptr(d["sd"]), nat.ptr(gdd), nat.ptr(god), nat.ptr(dh), nat.ptr(dm),
             nat.ptr(part), nat.ptr(grad), s)
    torch.cuda.synchronize()
    # forward: smoother entries within 2e-2 of the Jacobi scale of the bf16-emulating oracle
    Wd_or, Wo_or, cache = ol.forward(theta.astype(np.float64), nbr, sdiag, soff, emulate_bf16=True)
    assert (np.abs(Wd.cpu().numpy() - Wd_or) * sdiag).max() < 2e-2
    assert np.abs(Wo.cpu().numpy().reshape(E, 4) - Wo_or).max() * sdiag.min() < 2e-2
    hh, mm = _bf(h).reshape(5, E, 64), _bf(m).reshape(4, E, 64)
    zz = z.double().cpu().numpy().reshape(5, E, 64)
    q = np.where(nbr >= 0, nbr, 0)
    cache.update(h=list(hh), m=list(mm), z0=zz[0], z=list(zz[1:]), s=hh[4][:, None, :] + hh[4][q],
                 a=a.double().cpu().numpy().reshape(E, 4), x=x.double().cpu().numpy().reshape(E, 8))
    want = ol.backward(theta.astype(np.float64), cache, gd.astype(np.float64), go.astype(np.float64))
    got = grad.cpu().numpy().astype(np.float64)
    for name, (o, shape) in lay.items():
        k = int(np.prod(shape))
        w, g = want[o:o + k], got[o:o + k]
        assert np.linalg.norm(g - w) <= 1e-4 * max(np.linalg.norm(w), 1e-3), (name, E)


@pytest.mark.parametrize("sizes", [(1,), (12, 1, 51), (102, 103), (250, 7, 400), (3,) * 300])
def test_coarse_operator_aggregate_sizes(sizes):
    """P^T S P against numpy for aggregates of one cell, just below and above the cells a wave
    holds at once (102), several batches, and many small ones; FP64 sums (1e-13 of the row)."""
    import torch
    from nfempy_amd import _native as nat

    E, n_agg = sum(sizes), len(sizes)
    nbr, sdiag, soff = _graph(E, n_agg)
    rng = np.random.default_rng(E)
    agg_of = rng.permutation(np.repeat(np.arange(n_agg), sizes))
    mem = np.argsort(agg_of, kind="stable")
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    i32, f64 = torch.int32, torch.float64
    d = [_dev(a, i32) for a in (ptr, mem, agg_of, nbr)] + [_dev(sdiag, f64), _dev(soff, f64)]
    Ac = torch.zeros((n_agg, n_agg), dtype=f64, device="cuda")
    nat.call("nfx_coarse_dense", n_agg, *(nat.ptr(t) for t in d), nat.ptr(Ac), nat.stream_handle())
    torch.cuda.synchronize()
    want = np.zeros((n_agg, n_agg))
    np.add.at(want, (agg_of, agg_of), sdiag)
    p, j = np.nonzero(nbr >= 0)
    np.add.at(want, (agg_of[p], agg_of[nbr[p, j]]), soff[p, j])
    scale = np.abs(sdiag).sum()
    assert np.abs(Ac.cpu().numpy() - want).max() <= 1e-13 * scale


@pytest.mark.parametrize("n", [1, 255, 257, 150001])
def test_flux_row_sum_bound(n):
    """max_i sum_j |M_ij| / M_ii over tridiagonal rows (more rows than the kernel's grid covers in
    one pass for the largest), a maximum: exact up to the FP32 rounding of each row's quotient."""
    import torch
    from nfempy_amd import _native as nat

    rng = np.random.default_rng(n)
    diag, off = rng.uniform(1.0, 2.0, n), rng.uniform(-0.4, 0.4, n)
    vals = np.stack([diag, off, np.roll(off, 1)])  # slot-major; row i couples to i + 1 and i - 1
    pos = np.arange(3 * n).reshape(3, n).copy()
    pos[1, n - 1] = pos[2, 0] = -1
    col = np.stack([np.arange(n), np.minimum(np.arange(n) + 1, n - 1), np.maximum(np.arange(n) - 1, 0)])
    i32 = torch.int32
    dpos, dcol, ddiag = _dev(pos, i32), _dev(col, i32), _dev(np.arange(n), i32)
    dv = _dev(vals, torch.float64)
    coef = torch.empty(3 * n, dtype=torch.float32, device="cuda")
    bound = torch.full((1,), 7.0, dtype=torch.float32, device="cuda")
    nat.call("nfx_flux_sweep_coef", n, 3, nat.ptr(dpos), nat.ptr(dcol), nat.ptr(ddiag), nat.ptr(dv), 0.0,
             nat.ptr(coef), nat.ptr(bound), nat.stream_handle())
    torch.cuda.synchronize()
    s = diag + np.where(pos[1] >= 0, np.abs(vals[1]), 0) + np.where(pos[2] >= 0, np.abs(vals[2]), 0)
    assert np.float32((s / diag).max()) == pytest.approx(bound.item(), rel=1.2e-7)
