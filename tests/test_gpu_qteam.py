"""The one-launch Quantum-Sun filter (a team of blocks per column, csrc/qteam.hip)
against the oracle's Clenshaw: every grain size (those below three spins are
extended by outer spins), rows per block from one grain block to more than a block
holds (the streaming form), every number of blocks, odd column counts, uneven
orders and idle instances, both arithmetics in one call, the other polynomials,
and columns in place."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from oracle import clenshaw as oc
from oracle import models as om

pytestmark = pytest.mark.gpu

# FP64: a few hundred roundings of |b_k| <= O(1) terms, as for the per-step forms
TOL = {"f64": 1e-12, "f32": 5e-4}

# grain spins, outer spins, blocks per column
SIZES = [(3, 1, [1, 2]), (3, 5, [1, 4, 32]), (3, 7, [1, 8]), (3, 10, [1, 2, 16]), (3, 12, [2, 32]),
         (1, 2, [1]), (1, 9, [1, 8]), (2, 6, [1, 4]), (2, 10, [1]), (4, 3, [1, 8]), (4, 9, [1, 4])]


def _op(dev, Lg, Lloc, seed):
    from polfed_amd.operators import QSunOperator
    rng = np.random.default_rng(seed)
    hz, nb = rng.random(Lloc) + 0.5, rng.integers(0, Lg, size=Lloc)
    cp = 0.75 ** np.arange(Lloc)
    x = rng.standard_normal((1 << Lg, 1 << Lg))
    G = (x + x.T) / 3.0
    H = sp.csr_matrix(om.qsun_hamiltonian_from_draws(Lloc, Lg, 1.0, hz, nb, cp, G))
    g = float(abs(H).sum(axis=1).max())
    op = QSunOperator(Lloc, Lg, 1.0, hz, nb, cp, G, device=dev)
    op.set_rescale(-g, 1.1 * g)
    return op, ((H - 0.05 * g * sp.identity(H.shape[0], format="csr")) / (1.05 * g)).tocsr()


def _rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("Lg,Lloc,teams", SIZES)
def test_qsun_team_filter_matches_oracle(dev, Lg, Lloc, teams):
    op, Ht = _op(dev, Lg, Lloc, 7 * Lg + Lloc)
    X = np.random.default_rng(Lloc).standard_normal((op.D, 3))
    Xd = dev.to_device(X)
    for K, poly in ((0, "Chebyshev"), (1, "Chebyshev"), (2, "Chebyshev"), (31, "Chebyshev"),
                    (9, "Legendre"), (6, "Hermite")):
        c = np.random.default_rng(K).standard_normal(K + 1) * 0.1
        ref = oc.clenshaw_apply(lambda Z: Ht @ Z, c, X, poly)
        for dt in ("f64", "f32"):
            for T in teams:
                op.set_tuning(team=T)
                Y = torch.full_like(Xd, np.nan)
                op.filter(c, Xd, Y, dtype=dt, polytype=poly)
                assert _rel(dev.to_host(Y), ref) < TOL[dt], (K, poly, dt, T)
    Y = Xd.clone()
    op.filter(c, Y, Y, dtype="f64", polytype=poly)
    assert _rel(dev.to_host(Y), ref) < TOL["f64"]


@pytest.mark.parametrize("team", [-1, 1, 4, 32])
def test_qsun_team_batch_matches_oracle(dev, team):
    """More jobs than teams, uneven orders, an idle instance, mixed arithmetic, one
    instance in place, two that share their input."""
    from polfed_amd.batch import QSunBatch
    pairs = [_op(dev, 3 if i % 4 else 2, 5 + i % 3, i) for i in range(11)]
    ops = [p[0] for p in pairs]
    batch = QSunBatch(ops, 2)
    cs = [np.random.default_rng(i).standard_normal(3 + 5 * i) * 0.1 for i in range(len(ops))]
    batch.set_filter(cs)
    batch.set_tuning(team=team)
    X = [dev.to_device(np.random.default_rng(50 + i).standard_normal((op.D, 2)))
         for i, op in enumerate(ops)]
    same = [i for i in range(len(ops)) if ops[i].D == ops[3].D and i != 3]
    X[same[0]] = X[3]
    host = [dev.to_host(x).copy() for x in X]
    Y = [torch.full_like(x, np.nan) for x in X]
    Y[5] = X[5]
    dts = ["f32" if i % 3 == 1 else "f64" for i in range(len(ops))]
    batch.filter([None if i == 2 else (X[i], Y[i], dts[i]) for i in range(len(ops))])
    for i, (_, Ht) in enumerate(pairs):
        if i == 2:
            assert torch.isnan(Y[i]).all()
            continue
        ref = oc.clenshaw_apply(lambda Z: Ht @ Z, cs[i], host[i], "Chebyshev")
        assert _rel(dev.to_host(Y[i]), ref) < TOL[dts[i]], i


def test_qsun_team_batch_overlapping_blocks(dev):
    """An output that is another instance's input: the copies of the per-step form."""
    from polfed_amd.batch import QSunBatch
    pairs = [_op(dev, 3, 6, 20 + i) for i in range(2)]
    batch = QSunBatch([p[0] for p in pairs], 1)
    cs = [np.linspace(0.1, 0.4, 20), np.linspace(0.3, 0.2, 9)]
    batch.set_filter(cs)
    batch.set_tuning(team=1)
    X = [dev.to_device(np.random.default_rng(i).standard_normal((pairs[0][0].D, 1))) for i in (0, 1)]
    host = [dev.to_host(x).copy() for x in X]
    batch.filter([(X[0], X[1], "f64"), (X[1], X[0], "f64")])
    for i in (0, 1):
        ref = oc.clenshaw_apply(lambda Z: pairs[i][1] @ Z, cs[i], host[i], "Chebyshev")
        assert _rel(dev.to_host(X[1 - i]), ref) < TOL["f64"]
