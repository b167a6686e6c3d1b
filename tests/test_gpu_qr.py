"""Cholesky-QR on the device (csrc/dense.hip) against numpy's QR: block widths at the
edges of its register and reduction variants, padded leading dimensions, and blocks
whose first or second factorization breaks down; the three-term projection of a
block step against numpy."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s", [1, 2, 4, 5, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("D", [70, 5003])
def test_block_qr_matches_numpy(dev, s, D):
    from polfed_amd import NumericBreakdown
    from polfed_amd import blockops as bo
    rng = np.random.default_rng(s + D)
    W = rng.standard_normal((D, s)) * np.logspace(0, -3, s)
    pad = torch.full((s, D + 5), np.nan, dtype=torch.float64, device=dev.torch_device)
    pad[:, :D] = dev.to_device(W)
    Q = pad[:, :D]
    R = bo.block_qr(dev, Q)
    Qn, Rn = np.linalg.qr(W)
    sign = np.sign(np.diag(Rn))
    q = dev.to_host(Q)
    # two passes: orthogonal to a few roundings of D-term sums
    assert np.max(np.abs(q.T @ q - np.eye(s))) < 1e-13
    assert np.max(np.abs(q - Qn * sign)) < 1e-10
    assert np.max(np.abs(R - Rn * sign[:, None])) < 1e-11 * np.max(np.abs(Rn))
    assert np.array_equal(R, np.triu(R))
    assert torch.isnan(pad[:, D:]).all()
    bad = [np.zeros((D, s)), np.full((D, s), np.inf)]
    if s > 1:
        bad.append(np.repeat(W[:, :1], s, axis=1) * np.where(np.arange(s) == s - 1, 0.0, 1.0))
    for B in bad:
        Bd = dev.to_device(B)
        keep = Bd.clone()
        with pytest.raises(NumericBreakdown):
            bo.block_qr(dev, Bd)
        assert torch.equal(Bd, keep)


@pytest.mark.parametrize("s", [1, 3, 8, 16, 17])
@pytest.mark.parametrize("D", [40, 5003])
def test_lanczos_ortho_matches_numpy(dev, s, D):
    from polfed_amd import blockops as bo
    rng = np.random.default_rng(s + D)
    V, Vp, W, B = (rng.standard_normal((D, s)) / np.sqrt(D) for _ in range(4))
    b = np.triu(B[:s])
    a = V.T @ W
    a = np.triu(a) + np.triu(a, 1).T
    for prev in (False, True):
        Wd = dev.to_device(W)
        got = bo.lanczos_ortho(dev, dev.to_device(V), dev.to_device(Vp) if prev else None,
                               b if prev else None, Wd)
        assert np.max(np.abs(got - a)) < 1e-14
        assert np.max(np.abs(dev.to_host(Wd) - (W - V @ a - (Vp @ b.T if prev else 0.0)))) < 1e-14


@pytest.mark.parametrize("D", [1, 15, 17, 31, 127, 129, 4097])
def test_gram_and_update_edges(dev, D):
    """Rows at the edges of slabs, row pairs and row ranges; odd leading dimensions."""
    from polfed_amd import blockops as bo
    rng = np.random.default_rng(D)
    for m, n in ((1, 1), (16, 8), (17, 1), (70, 17), (130, 64), (65, 33)):
        A, B, G = rng.standard_normal((D, m)), rng.standard_normal((D, n)), rng.standard_normal((m, n))
        pad = torch.full((m, D + 3), np.nan, dtype=torch.float64, device=dev.torch_device)
        pad[:, :D] = dev.to_device(A)
        out = torch.full((n, D + 1), 7.0, dtype=torch.float64, device=dev.torch_device)
        out[:, :D] = dev.to_device(B)
        got = dev.to_host(bo.gram(dev, pad[:, :D], out[:, :D]))
        assert np.max(np.abs(got - A.T @ B)) < 1e-13 * max(D, 10)
        bo.update(dev, pad[:, :D], dev.to_device(G), out[:, :D], alpha=-0.5, beta=2.0)
        assert np.max(np.abs(dev.to_host(out[:, :D]) - (2.0 * B - 0.5 * A @ G))) < 1e-13 * max(m, 10)
        assert (out[:, D:] == 7.0).all()
