"""Performance cases of the POLFED hot path on one GPU.

Each case is one call (or the two calls that always follow each other) that a
program using this package makes: the polynomial filter of the block-Lanczos
solve on spin chains, the same on a batch of Quantum-Sun instances and on a
packed sparse matrix, the KPM moments of the density of states, the operator
application of the user hooks, the reorthogonalization and QR of a Lanczos
block, and the extremal-eigenvalue probes.  ``listed`` gives the fixed cases,
``draw`` more of the same ranges, ``prepare`` what a program holds before the
call (operators, launch plans, input blocks on the device), ``run`` one pass
and ``exact`` the same values from plain torch in FP64.

FP32-arithmetic results come back from the package in FP64 containers; a pass
hands them on as float32, the precision they have.
"""
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent


def _package():
    """The repository's package (directory ``polfed.jl_amd``, imported as polfed_amd)."""
    if "polfed_amd" not in sys.modules:
        pkg = ROOT / "polfed.jl_amd"
        spec = importlib.util.spec_from_file_location(
            "polfed_amd", pkg / "__init__.py", submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["polfed_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["polfed_amd"]


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the reference's CPU-runnable size, one vector: every step is tiny and
        # latency counts; order of its nev=50 solve
        dict(name="filter_xxz14_vec", kind="filter", L=14, Lup=7, J2=0.0, periodic=True, s=1,
             dtype="f64", order=402),
        # odd everything: open chain off half filling, an odd block
        dict(name="filter_open17_b5", kind="filter", L=17, Lup=7, J2=0.0, periodic=False, s=5,
             dtype="f64", order=601),
        # the plain FP64 solve at L=20, block 8 (a stretch of its order-12621 filter)
        dict(name="filter_xxz20_b8", kind="filter", L=20, Lup=10, J2=0.0, periodic=True, s=8,
             dtype="f64", order=400),
        # the precision workload, L=22 block 16: its two filters
        dict(name="filter_xxz22_b16_f32", kind="filter", L=22, Lup=11, J2=0.0, periodic=True,
             s=16, dtype="f32", order=200),
        dict(name="filter_xxz22_b16", kind="filter", L=22, Lup=11, J2=0.0, periodic=True, s=16,
             dtype="f64", order=200),
        # the largest: J1-J2 L=24, block 32, FP32 filter, past the caches
        dict(name="filter_j1j2_24_b32_f32", kind="filter", L=24, Lup=12, J2=0.5, periodic=True,
             s=32, dtype="f32", order=40),
        # density of states: the default 250 moments on a chunk of FP64 probes
        dict(name="kpm_xxz20", kind="kpm", L=20, Lup=10, J2=0.0, periodic=True, R=32, N=250,
             dtype="f64"),
        # 64 disorder realizations of the Quantum Sun, single vectors, uneven
        # sizes and orders, one batched application
        dict(name="qsun_batch64", kind="batch", n=64, lloc_min=10, lloc_max=14, s=1, dtype="f64",
             order=300),
        # polfed(matrix): the packed sparse operator, two coupling values
        dict(name="packed_j1j2_18_b6", kind="packed", L=18, Lup=9, J2=0.5, periodic=True, s=6,
             dtype="f64", order=300),
        # user hooks and residuals: one operator application on caller's blocks
        dict(name="apply_xxz22_b16", kind="apply", L=22, Lup=11, J2=0.0, periodic=True, s=16,
             dtype="f64"),
        # late Lanczos iteration of the L=20 solve: CGS2 against the basis, then QR
        dict(name="reorth_xxz20_b8", kind="reorth", D=184756, k=416, s=8),
        # spectral bounds of a chain before the solve: two whole Lanczos runs
        dict(name="extrema_xxz18", kind="extrema", L=18, Lup=9, J2=0.0, periodic=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _chain(rng, lo, hi):
    """A chain of lo..hi sites at or near half filling."""
    L = rng.randint(lo, hi)
    return dict(L=L, Lup=max(1, L // 2 - rng.choice([0, 0, 1, 2])), J2=rng.choice([0.0, 0.0, 0.5]),
                periodic=rng.random() < 0.75)


def draw(rng):
    kind = rng.choice(["filter", "filter", "filter", "kpm", "batch", "packed", "apply", "reorth",
                       "extrema"])
    dtype = rng.choice(["f64", "f64", "f32"])
    if kind == "filter":
        c = dict(kind=kind, **_chain(rng, 10, 23), s=_log_int(rng, 1, 32), dtype=dtype)
        most = 6e10 / (math.comb(c["L"], c["Lup"]) * c["s"] * len(_bonds(c)))
        return dict(c, order=max(20, min(_log_int(rng, 40, 1000), int(most))))
    if kind == "kpm":
        c = dict(kind=kind, **_chain(rng, 12, 21), R=_log_int(rng, 8, 64), dtype=dtype)
        most = 6e10 / (math.comb(c["L"], c["Lup"]) * c["R"] * len(_bonds(c)))
        return dict(c, N=max(20, min(_log_int(rng, 50, 500), int(most))))
    if kind == "batch":
        lo = rng.randint(7, 12)
        return dict(kind=kind, n=_log_int(rng, 3, 64), lloc_min=lo, lloc_max=lo + rng.randint(0, 2),
                    s=rng.choice([1, 1, 1, 2, 4]), dtype=dtype, order=_log_int(rng, 60, 300))
    if kind == "packed":
        c = dict(kind=kind, **_chain(rng, 11, 19), s=_log_int(rng, 1, 16), dtype=dtype)
        return dict(c, order=_log_int(rng, 40, 300))
    if kind == "apply":
        return dict(kind=kind, **_chain(rng, 12, 22), s=_log_int(rng, 1, 32), dtype=dtype)
    if kind == "reorth":
        s = _log_int(rng, 1, 16)
        return dict(kind=kind, D=_log_int(rng, 3000, 300000), k=s * _log_int(rng, 2, 320 // s), s=s)
    return dict(kind=kind, **_chain(rng, 10, 19))


# ------------------------------------------------------------ models, in numpy
def _bonds(case):
    """(site i, site j, J, Delta), 1-based sites; second neighbours with J2."""
    L, out = case["L"], []
    for dist, J in ((1, 1.0), (2, case["J2"])):
        if J:
            for i in range(1, (L if case["periodic"] else L - dist) + 1):
                out.append((i, (i + dist - 1) % L + 1, J, 1.0))
    return out


def _fields(case, seed):
    return 2.0 * (2.0 * np.random.default_rng(seed).random(case["L"]) - 1.0)


def _bounds(case, h):
    """An interval that holds the spectrum."""
    r = sum(abs(J) * (abs(d) / 4 + 0.5) for _, _, J, d in _bonds(case)) + float(np.abs(h).sum()) / 2
    return -r, r


def _delta_coefficients(order, target=0.1):
    """The solver's default filter: c_n = (2 - [n=0]) cos(n acos t), p(t) = 1."""
    n = np.arange(order + 1)
    a = np.cos(n * math.acos(target))
    c = np.where(n == 0, 1.0, 2.0) * a
    return c / float(c @ a)


def _block(n, D, seed, salt=0):
    """n columns of unit length, (n, D) on the device."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1000003 + salt)
    X = torch.randn((n, D), dtype=torch.float64, device="cuda", generator=g)
    return X / X.norm(dim=1, keepdim=True)


def _device():
    _package()
    from polfed_amd.device import default_device
    return default_device()


def _chain_operator(case, seed, dev):
    from polfed_amd.operators import SpinChainOperator
    h = _fields(case, seed)
    b = _bonds(case)
    op = SpinChainOperator(case["L"], case["Lup"], [(i, j) for i, j, _, _ in b],
                           [J for _, _, J, _ in b], [d for _, _, _, d in b], h, device=dev)
    op.set_rescale(*_bounds(case, h))
    return op


def _connectivity(case, seed):
    """Basis states, diagonal and per bond (J/2, rows, columns) on the device."""
    L = case["L"]
    s = torch.arange(1 << L, dtype=torch.int64, device="cuda")
    pop = torch.zeros_like(s)
    for k in range(L):
        pop += (s >> k) & 1
    s = s[pop == case["Lup"]].contiguous()
    del pop
    z = lambda k: ((s >> k) & 1).double() - 0.5  # noqa: E731
    diag = torch.zeros(len(s), dtype=torch.float64, device="cuda")
    for k, hk in enumerate(_fields(case, seed)):
        diag += float(hk) * z(k)
    links = []
    for i, j, J, d in _bonds(case):
        diag += J * d * z(i - 1) * z(j - 1)
        rows = torch.nonzero(((s >> (i - 1)) & 1) != ((s >> (j - 1)) & 1)).reshape(-1)
        cols = torch.searchsorted(s, s[rows] ^ ((1 << (i - 1)) | (1 << (j - 1))))
        links.append((J / 2, rows, cols))
    return diag, links


def _qsun_draws(case, i, seed):
    """Instance i of a batch: (L_loc, disorder, neighbours, couplings, grain)."""
    rng = np.random.default_rng([seed, i])
    lloc = case["lloc_min"] + i % (case["lloc_max"] - case["lloc_min"] + 1)
    disorder = rng.random(lloc) + 0.5
    neighbors = rng.integers(0, 3, size=lloc)
    couplings = 0.75 ** (np.arange(lloc) + 0.4 * rng.random(lloc) - 0.2)
    x = rng.standard_normal((8, 8))
    return lloc, disorder, neighbors, couplings, (x + x.T) / math.sqrt(2.0) / 3.0


def _qsun_bound(d):
    return float(np.linalg.norm(d[4], 2)) + float(d[1].sum()) / 2 + float(d[3].sum()) / 4


def _qsun_orders(case):
    """Uneven orders: larger instances take longer polynomials."""
    span = case["lloc_max"] - case["lloc_min"] + 1
    return [case["order"] // 3 + (2 * case["order"] // 3) * (i % span + 1) // span + i % 7
            for i in range(case["n"])]


# ------------------------------------------------------------------- the calls
def prepare(case, seed):
    dev = _device()
    kind = case["kind"]
    if kind == "reorth":
        D, k, s = case["D"], case["k"], case["s"]
        return dict(case=case, dev=dev, V=_block(k, D, seed), W=_block(s, D, seed, 1))
    if kind == "batch":
        from polfed_amd.batch import QSunBatch
        from polfed_amd.operators import QSunOperator
        ops = []
        for i in range(case["n"]):
            lloc, hz, nb, cp, G = d = _qsun_draws(case, i, seed)
            op = QSunOperator(lloc, 3, 1.0, hz, nb, cp, G, device=dev)
            op.set_rescale(-_qsun_bound(d), _qsun_bound(d))
            ops.append(op)
        batch = QSunBatch(ops, case["s"])
        batch.set_filter([_delta_coefficients(K) for K in _qsun_orders(case)])
        batch.autotune(case["dtype"], nsteps=6)
        X = [_block(case["s"], op.D, seed, i) for i, op in enumerate(ops)]
        return dict(case=case, batch=batch, X=X, Y=[torch.empty_like(x) for x in X])
    if kind == "packed":
        from polfed_amd.operators import PackedOperator
        diag, links = _connectivity(case, seed)
        D = len(diag)
        values = sorted({w for w, _, _ in links})
        starts, flat, at = [], [], 0
        for v in values:  # per value: the columns of each row, ascending
            key = torch.cat([r * D + c for w, r, c in links if w == v]).sort().values
            count = torch.bincount(key // D, minlength=D).cumsum(0).cpu().numpy()
            starts.append(at + np.concatenate([[0], count]))
            flat.append((key % D).cpu().numpy().astype(np.int32))
            at += len(flat[-1])
        op = PackedOperator(diag.cpu().numpy(), values, np.array(starts), np.concatenate(flat),
                            device=dev)
        op.set_rescale(*_bounds(case, _fields(case, seed)))
    else:
        op = _chain_operator(case, seed, dev)
    state = dict(case=case, dev=dev, op=op)
    if kind == "kpm":
        op.ensure_tuned(min(case["R"], 32 if case["dtype"] == "f64" else 64), case["dtype"], 3)
        state["P"] = _block(case["R"], op.D, seed)
    elif kind == "apply":
        state["X"] = _block(case["s"], op.D, seed)
        if case["dtype"] == "f32":
            state["X"] = state["X"].float()
    elif kind == "extrema":
        state["x"] = _block(1, op.D, seed)[0].contiguous()
    else:
        op.ensure_tuned(case["s"], case["dtype"], 3)
        state["c"] = _delta_coefficients(case["order"])
        state["X"] = _block(case["s"], op.D, seed)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    f32 = case.get("dtype") == "f32"
    if kind in ("filter", "packed"):
        Y = state["op"].filter(state["c"], state["X"], dtype=case["dtype"])
        return Y.float() if f32 else Y
    if kind == "kpm":
        mu = state["op"].kpm_moments(case["N"], state["P"], dtype=case["dtype"])
        return mu.astype(np.float32) if f32 else mu
    if kind == "batch":
        state["batch"].filter([(x, y, case["dtype"]) for x, y in zip(state["X"], state["Y"])])
        return [y.float() if f32 else y for y in state["Y"]]
    if kind == "apply":
        return state["op"].apply(state["X"], rescaled=True, dtype=case["dtype"])
    if kind == "reorth":
        from polfed_amd import blockops
        W = state["W"].clone()
        blockops.reorth(state["dev"], state["V"], W, passes=2)
        return W, blockops.block_qr(state["dev"], W)
    from polfed_amd import lanczos_extrema
    return lanczos_extrema(state["op"], state["x"], device=state["dev"])


# ------------------------------------------------- what a pass cannot do without
def _chain_flops(case, cols):
    """Per operator application: half of the bonds flip, one multiply-add each,
    the diagonal and the two vector terms of the recurrence."""
    return math.comb(case["L"], case["Lup"]) * cols * (len(_bonds(case)) + 6.0)


def work(case):
    kind = case["kind"]
    esz = 4 if case.get("dtype") == "f32" else 8
    if kind == "batch":
        b = f = 0.0
        span = case["lloc_max"] - case["lloc_min"] + 1
        for i, K in enumerate(_qsun_orders(case)):
            lloc = case["lloc_min"] + i % span
            rows = float(2 ** (3 + lloc)) * case["s"]
            b += rows * (8 + esz)
            f += K * rows * 2.0 * (lloc + 8 + 3)
        return {"bytes": b, "flops": f}
    if kind == "reorth":
        D, k, s = case["D"], case["k"], case["s"]
        return {"bytes": 8.0 * D * (k + 2 * s), "flops": 8.0 * D * k * s + 8.0 * D * s * s}
    D = math.comb(case["L"], case["Lup"])
    if kind == "extrema":
        its = 60  # two runs of about this many single-vector iterations
        return {"bytes": 8.0 * D * 2 * its, "flops": 2 * its * (_chain_flops(case, 1) + 4.0 * D * its)}
    if kind == "kpm":
        return {"bytes": 8.0 * D * case["R"], "flops": case["N"] / 2 * _chain_flops(case, case["R"])}
    if kind == "apply":
        return {"bytes": 2.0 * esz * D * case["s"], "flops": _chain_flops(case, case["s"])}
    return {"bytes": D * case["s"] * (8.0 + esz),
            "flops": case["order"] * _chain_flops(case, case["s"])}


# ---------------------------------------------------------- the same, in 64 bits
def _apply_links(diag, links, X):
    """H X on rows of X (columns of the block) from the bond lists."""
    Y = diag * X
    for w, rows, cols in links:
        Y[:, rows] += w * X[:, cols]
    return Y


def _clenshaw(apply, c, X):
    b1, b2 = torch.zeros_like(X), torch.zeros_like(X)
    for ck in c[:0:-1]:
        b1, b2 = 2.0 * apply(b1) - b2 + float(ck) * X, b1
    return apply(b1) - b2 + float(c[0]) * X




def exact(case, seed):
    kind = case["kind"]
    if kind == "reorth":
        V, W = _block(case["k"], case["D"], seed), _block(case["s"], case["D"], seed, 1)
        for _ in range(2):
            W = W - (W @ V.t()) @ V
        Q, R = torch.linalg.qr(W.t().cpu())
        sign = torch.where(torch.diagonal(R) < 0, -1.0, 1.0).double()
        return (Q * sign).t().contiguous(), (R * sign[:, None]).numpy()
    if kind == "batch":
        out = []
        for i, K in enumerate(_qsun_orders(case)):
            lloc, hz, nb, cp, G = d = _qsun_draws(case, i, seed)
            D, a = 2 ** (3 + lloc), _qsun_bound(d)
            r = torch.arange(D, device="cuda")
            dz = torch.zeros(D, dtype=torch.float64, device="cuda")
            for j in range(lloc):
                dz += float(hz[j]) * (((r >> (3 + j)) & 1).double() - 0.5)
            flips = [(0.25 * float(cp[j]), r ^ ((1 << (3 + j)) | (1 << int(nb[j]))))
                     for j in range(lloc)]
            Gd = torch.from_numpy(G).cuda()

            def apply(X):
                Y = dz * X + (X.reshape(-1, 8) @ Gd.t()).reshape(X.shape)
                for w, idx in flips:
                    Y = Y + w * X[:, idx]
                return Y / a

            out.append(_clenshaw(apply, _delta_coefficients(K), _block(case["s"], D, seed, i)))
        return out
    diag, links = _connectivity(case, seed)
    D = len(diag)
    Emin, Emax = _bounds(case, _fields(case, seed))
    a = (Emax - Emin) / 2
    if kind == "extrema":
        return _extremes(diag, links, _block(1, D, seed))
    scaled = [(w / a, r, c) for w, r, c in links]
    diag = (diag - (Emax + Emin) / 2) / a
    if kind == "apply":
        X = _block(case["s"], D, seed)
        X = X.float().double() if case["dtype"] == "f32" else X
        return _apply_links(diag, scaled, X)
    if kind == "kpm":
        P = _block(case["R"], D, seed)
        t0, t1 = P, _apply_links(diag, scaled, P)
        mu = [float((P * t0).sum()), float((P * t1).sum())]
        for _ in range(2, case["N"]):
            t0, t1 = t1, 2.0 * _apply_links(diag, scaled, t1) - t0
            mu.append(float((P * t1).sum()))
        return np.array(mu) * (D / case["R"])
    return _clenshaw(lambda X: _apply_links(diag, scaled, X), _delta_coefficients(case["order"]),
                     _block(case["s"], D, seed))


def _extremes(diag, links, v, most=300):
    """Smallest and largest eigenvalue by Lanczos with full reorthogonalization."""
    V = torch.zeros((most + 1, len(diag)), dtype=torch.float64, device="cuda")
    V[0] = v[0] / v[0].norm()
    al, be = [], []
    for k in range(min(most, len(diag) - 1)):
        w = _apply_links(diag, links, V[k:k + 1])[0]
        al.append(float(w @ V[k]))
        for _ in range(2):
            w = w - (V[:k + 1] @ w) @ V[:k + 1]
        be.append(float(w.norm()))
        if be[-1] < 1e-10:
            break
        V[k + 1] = w / be[-1]
    n = len(al)
    T = np.diag(al) + np.diag(be[:n - 1], 1) + np.diag(be[:n - 1], -1)
    e = np.linalg.eigvalsh(T)
    return float(e[0]), float(e[-1])
