"""The row kernel's parts of the reference table (all of it, the reference tensors, the values at the quadrature
points) against the element kernel: every combination of coefficients per element and per point, on meshes of
one tile, of a ragged last tile and of more tiles than a block takes."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,degree,n", [(2, 1, 5), (2, 2, 1), (2, 2, 23), (3, 1, 3), (3, 2, 1), (3, 2, 7)])
@pytest.mark.parametrize("kappa_at,f_at", [("cell", "cell"), ("point", "point"), ("point", "cell"), ("cell", "point")])
def test_rows_match_the_element_kernel(dim, degree, n, kappa_at, f_at):
    """Both sum a few dozen products an entry in other orders: 64 eps of the largest value of a row's scale."""
    import torch

    from nfempy_amd.device import DarcySystem
    from tests._cases import product_darcy_space

    y = DarcySystem(product_darcy_space(dim, n, degree))
    r = np.random.default_rng(7 * dim + degree + n)
    draw = lambda at: np.exp(r.standard_normal((y.E, y.nq) if at == "point" else y.E))
    kappa, f = draw(kappa_at), draw(f_at)
    for fp64, eps in ((False, 2.0 ** -23), (True, 2.0 ** -52)):
        print(f"[row tables] {dim} {degree} {n} {kappa_at} {f_at} {fp64}", flush=True)
        v, g = (t.clone() for t in y.assemble_elements(kappa, f, fp64=fp64))
        ve, ge = y.assemble_elements(kappa, f, fp64=fp64, method="element")
        torch.cuda.synchronize()
        assert float((v - ve).abs().max()) <= 64 * eps * float(ve.abs().max())
        assert float((g - ge).abs().max()) <= 64 * eps * float(ge.abs().max())
