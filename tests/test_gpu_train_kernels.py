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
