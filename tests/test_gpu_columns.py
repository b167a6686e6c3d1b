"""Column-major maps of wide blocks (four columns per lane, csrc/ops.hip) against the
oracle's sparse matrix: column counts that leave one, two and three columns to the
last group, both arithmetics, and every term of the recurrence."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from oracle import models as om

pytestmark = pytest.mark.gpu


# one application: two dozen roundings of O(1) terms, as the narrow blocks' test
@pytest.mark.parametrize("dtype,tol", [("f64", 1e-13), ("f32", 1e-5)])
@pytest.mark.parametrize("J2,ncols", [(0.0, 44), (0.5, 41), (0.0, 42), (0.5, 43)])
def test_wide_column_blocks_match_oracle(dev, dtype, tol, J2, ncols):
    from polfed_amd.operators import SpinChainOperator
    L, Lup = 17, 8  # 24310 rows: 95 groups of 256 for each four columns
    bonds, Js, Ds = (om.j1j2_bonds(L, 1.0, J2, 0.9, 1.1, "open") if J2 else
                     om.xxz_bonds(L, 0.8, 0.7, "periodic"))
    h = np.random.default_rng(3).uniform(-1, 1, L)
    op = SpinChainOperator(L, Lup, bonds, Js, Ds, h, device=dev)
    H = om.spin_half_hamiltonian(L, bonds, Js, Ds, h, Lup).tocsr()
    g = float(abs(H).sum(axis=1).max())
    op.set_rescale(-g, 1.1 * g)
    Ht = (H - 0.05 * g * sp.identity(op.D, format="csr")) / (1.05 * g)
    rng = np.random.default_rng(ncols)
    X, B2, B3 = (rng.standard_normal((op.D, ncols)) for _ in range(3))
    tdt = torch.float64 if dtype == "f64" else torch.float32
    put = lambda M: dev.to_device(M).to(tdt)
    got = lambda t: dev.to_host(t.to(torch.float64))
    rel = lambda a, b: np.max(np.abs(a - b)) / np.max(np.abs(b))
    Xd, b2, b3 = put(X), put(B2), put(B3)
    assert rel(got(op.apply(b2, dtype=dtype)), H @ B2) < tol
    assert rel(got(op.apply(b2, rescaled=True, dtype=dtype)), Ht @ B2) < tol
    out = torch.empty_like(Xd)
    op.recurrence(out, b2, b3, 0.3, Xd, dtype=dtype)
    assert rel(got(out), 0.3 * X + 2.0 * (Ht @ B2) - B3) < tol
    op.finalsum(b2, b3, 0.4, out, Xd, dtype=dtype)
    assert rel(got(out), 0.4 * X + Ht @ B2 - B3) < tol
