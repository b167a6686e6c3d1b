"""The one-launch filter of spin chains (a team of blocks per column, csrc/team.hip)
against the oracle's Clenshaw, at the sizes where its tables change: a whole small
sector in one block, the cut at ten low sites, odd sectors, open and periodic
chains (the periodic ones run folded), one and two coupling values, every number
of blocks per column in the resident and the streaming form, and column counts
that leave teams idle or take further rounds."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from oracle import clenshaw as oc
from oracle import dos as odos
from oracle import models as om

pytestmark = pytest.mark.gpu

# FP64: a few hundred roundings of |b_k| <= O(1) terms, 1e-12 as for the per-step
# filter; FP32 likewise 5e-4 (tests/test_gpu_ops.py uses the same bounds)
TOL = {"f64": 1e-12, "f32": 5e-4}

CASES = [
    # name, L, Lup, J2, boundary, columns, blocks per column
    ("two_sites", 2, 1, 0.0, "periodic", 2, [1]),
    ("tiny_xxz", 12, 6, 0.0, "periodic", 3, [1]),
    ("tiny_13_bonds", 13, 5, 0.0, "periodic", 1, [1]),
    ("tiny_j1j2", 11, 5, 0.5, "periodic", 9, [1]),
    ("one_high_site_pair", 12, 4, 0.3, "open", 2, [1]),
    ("cut_open", 14, 5, 0.0, "open", 5, [1, 2, 8, 32]),
    ("cut_ring", 15, 7, 0.0, "periodic", 9, [1, 4, 16]),
    ("cut_ring_j1j2", 14, 7, 0.5, "periodic", 3, [1, 2, 32]),
    ("few_particles", 20, 4, 0.0, "periodic", 17, [1, 8, 32]),
    ("many_particles", 16, 12, 0.5, "open", 2, [2, 16]),
    # the most groups per wave (blocks of eight waves in FP64), and too many
    ("ring_xxz_full", 18, 9, 0.0, "periodic", 1, [2, 4, 8]),
    ("ring_j1j2_full", 18, 9, 0.5, "periodic", 1, [4, 8, 16]),
]


def _chain(dev, L, Lup, J2, boundary, seed):
    from polfed_amd.operators import SpinChainOperator
    if J2:
        bonds, Js, Ds = om.j1j2_bonds(L, 1.0, J2, 0.9, 1.1, boundary)
    else:
        bonds, Js, Ds = om.xxz_bonds(L, 0.8, 0.7, boundary)
    h = om.resolve_fields(L, 0.0, 1.5, rng=np.random.default_rng(seed))
    op = SpinChainOperator(L, Lup, bonds, Js, Ds, h, device=dev)
    H = om.spin_half_hamiltonian(L, bonds, Js, Ds, h, Lup).tocsr()
    g = float(abs(H).sum(axis=1).max())
    op.set_rescale(-g, 1.1 * g)
    a, b = 1.05 * g, 0.05 * g
    return op, ((H - b * sp.identity(H.shape[0], format="csr")) / a).tocsr()


def _rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_team_filter_matches_oracle(dev, case):
    name, L, Lup, J2, boundary, s, teams = case
    op, Ht = _chain(dev, L, Lup, J2, boundary, len(name))
    X = np.random.default_rng(L).standard_normal((op.D, s))
    Xd = dev.to_device(X)
    for K, poly in ((1, "Chebyshev"), (2, "Chebyshev"), (40, "Chebyshev"), (9, "Legendre"),
                    (6, "Hermite")):
        c = oc.filter_coefficients(0.1, K) if poly == "Chebyshev" else \
            np.random.default_rng(K).standard_normal(K + 1) * 0.1
        ref = oc.clenshaw_apply(lambda Z: Ht @ Z, c, X, poly)
        for dt in ("f64", "f32"):
            outs = []
            for T in teams:
                op.set_tuning(team=T)
                Y = torch.full_like(Xd, np.nan)
                op.filter(c, Xd, Y, dtype=dt, polytype=poly)
                outs.append(dev.to_host(Y))
                assert _rel(outs[-1], ref) < TOL[dt], (K, poly, dt, T)
    op.set_tuning(team=-1)


def test_team_filter_in_place_and_strided(dev):
    """The result may replace X; leading dimensions beyond D; an overlap that is
    not column by column takes the per-step launches, which copy X first."""
    op, Ht = _chain(dev, 15, 7, 0.0, "periodic", 3)
    D, s = op.D, 4
    X = np.random.default_rng(1).standard_normal((D, s))
    c = oc.filter_coefficients(-0.2, 30)
    ref = oc.clenshaw_apply(lambda Z: Ht @ Z, c, X)
    op.set_tuning(team=8)
    buf = torch.zeros((s + 1, D + 7), dtype=torch.float64, device=dev.torch_device)
    for shift in (0, 1):  # in place, then one column further
        buf[:s, :D] = dev.to_device(X)
        op.filter(c, buf[:s, :D], buf[shift:s + shift, :D])
        assert _rel(dev.to_host(buf[shift:s + shift, :D].contiguous()), ref) < 1e-12, shift


def test_team_filter_more_couplings_than_classes(dev):
    """Three coupling values: no team tables, the filter still works."""
    from polfed_amd.operators import SpinChainOperator
    L, Lup = 13, 6
    bonds, Js, Ds = om.xxz_bonds(L, 1.0, 1.0, "periodic")
    Js = [0.5 + 0.25 * (i % 3) for i in range(len(Js))]
    h = np.random.default_rng(5).uniform(-1, 1, L)
    op = SpinChainOperator(L, Lup, bonds, Js, Ds, h, device=dev)
    H = om.spin_half_hamiltonian(L, bonds, Js, Ds, h, Lup).tocsr()
    g = float(abs(H).sum(axis=1).max())
    op.set_rescale(-g, g)
    op.set_tuning(team=1)
    X = np.random.default_rng(2).standard_normal((op.D, 3))
    c = oc.filter_coefficients(0.3, 25)
    Y = dev.to_host(op.filter(c, dev.to_device(X)))
    assert _rel(Y, oc.clenshaw_apply(lambda Z: (H / g) @ Z, c, X)) < 1e-12


# moments are averages of products of such vectors: the per-step moments' bounds
@pytest.mark.parametrize("dtype,tol", [("f64", 1e-12), ("f32", 2e-4)])
@pytest.mark.parametrize("case", CASES[1:], ids=[c[0] for c in CASES[1:]])
def test_team_moments_match_oracle(dev, case, dtype, tol):
    """Every moment, odd and even counts of them: FP64 takes two per step."""
    name, L, Lup, J2, boundary, s, teams = case
    op, Ht = _chain(dev, L, Lup, J2, boundary, len(name))
    P = np.random.default_rng(L).standard_normal((op.D, s))
    Pd = dev.to_device(P)
    for N in (2, 3, 40):
        ref = odos.dos_moments(lambda v: Ht @ v, N, P)
        for T in teams:
            op.set_tuning(team=T)
            mu = op.kpm_moments(N, Pd, dtype=dtype)
            assert np.max(np.abs(mu - ref)) / op.D < tol, (N, T)
