"""The calls whose speed this repository watches, through its public entry points.

What a program that uses the library spends its time on, from the smallest
chain of the tests (L=10, D=8) to the benchmark's bond dimension (D=1024):

* "heff"        one product with a site's effective Hamiltonian on device
                vectors (Context.heff_apply_device), in every precision the
                library contracts in: the inner step of every eigensolve;
* "eig"         the local eigensolver seam on host vectors (Context.eig_lowest);
* "ground"      a short schedule of the variational driver from a random start
                with its default options (FindVariationalGroundState: SVD gauge
                moves, full eigensolves, <H> and <H^2>);
* "sweep"       a one-site sweep (left and right pass) with the benchmark's options
                (QR gauge, capped eigensolves) from a random start;
* "sweep2"      the same with two-site updates (their splits are singular value
                decompositions);
* "expectation" <H> of a chain: the left zipper over all sites;
* "batch"       sweeps of many chains in lockstep from a random start.

Environments are those of random matrix product states (random isometries
contracted with the MPO, so the "nothing placed" channels are the identity, as
in any canonical chain); chains start from seeded random tensors.  Contexts are
used as they are created (no tuning table).
"""
import math

import numpy as np
import torch

import tensornetworks_amd as tn
from tensornetworks_amd import models
from tensornetworks_amd.dmrg import create_h2

PRECISION = {"fp64": tn.TN_FP64, "fp32": tn.TN_FP32, "bf16": tn.TN_BF16, "bf16x3": tn.TN_BF16X3}
OPERAND_BYTES = {"fp64": 8, "fp32": 4, "bf16": 2, "bf16x3": 6}


def listed():
    return [
        # one apply at the bulk site of the smallest test chain (S=1/2, D=8):
        # launches and the wait are all there is
        {"name": "heff_d2_D8_fp64", "kind": "heff", "model": "xxz", "d": 2, "D1": 8, "D2": 8, "precision": "fp64"},
        # an ordinary ragged site (bond dimensions as the truncation leaves them), FP64
        {"name": "heff_d2_300x210_fp64", "kind": "heff", "model": "xxz", "d": 2, "D1": 300, "D2": 210,
         "precision": "fp64"},
        # FP32 contractions, S=1, ragged, between the small chains and the benchmark
        {"name": "heff_d3_500x420_fp32", "kind": "heff", "model": "xxz", "d": 3, "D1": 500, "D2": 420,
         "precision": "fp32"},
        # the benchmark's bulk site (S=1 with Dz, D=1024) in its headline precision
        {"name": "heff_d3_D1024_bf16x3", "kind": "heff", "model": "xxz", "d": 3, "D1": 1024, "D2": 1024,
         "precision": "bf16x3"},
        # the same site in FP64: the precision of every reference result, and the largest apply
        {"name": "heff_d3_D1024_fp64", "kind": "heff", "model": "xxz", "d": 3, "D1": 1024, "D2": 1024,
         "precision": "fp64"},
        # a program that keeps its own sweep and calls the eigensolver per site: small and ordinary
        {"name": "eig_d2_D16", "kind": "eig", "model": "xxz", "d": 2, "D1": 16, "D2": 16, "nev": 2},
        {"name": "eig_d3_192x160", "kind": "eig", "model": "xxz", "d": 3, "D1": 192, "D2": 160, "nev": 1},
        # the smallest chain of the tests through the variational driver, default options
        {"name": "ground_L10_D8", "kind": "ground", "d": 2, "L": 10, "D": 8},
        # a production sweep at moderate D: QR gauge, partial re-orthogonalisation
        {"name": "sweep_L14_D256", "kind": "sweep", "d": 3, "L": 14, "D": 256},
        # two-site sweep at fixed Dmax
        {"name": "sweep2_L16_D96", "kind": "sweep2", "d": 2, "L": 16, "D": 96},
        # the energy of a finished chain
        {"name": "expectation_L24_D256", "kind": "expectation", "d": 2, "L": 24, "D": 256},
        # many small chains of different length and bond dimension in lockstep
        {"name": "batch_24_chains", "kind": "batch", "chains": 24, "Lmin": 8, "Lmax": 28, "Dmin": 16, "Dmax": 96},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["heff"] * 6 + ["eig", "ground", "sweep", "sweep2", "expectation", "batch"])
    d = rng.choice([2, 3])
    if kind == "heff":
        D1 = _log(rng, 6, 1000)
        D2 = max(4, min(1000, int(D1 * rng.uniform(0.6, 1.4))))
        return {"kind": kind, "model": rng.choice(["xxz", "xxz", "xxz", "tfim", "long3"]) if D1 < 400 else "xxz", "d": d,
                "D1": D1, "D2": D2, "precision": rng.choice(["fp64", "fp64", "fp32", "bf16x3", "bf16x3", "bf16"])}
    if kind == "eig":
        D1 = _log(rng, 6, 180)
        return {"kind": kind, "model": "xxz", "d": d, "D1": D1, "D2": max(6, int(D1 * rng.uniform(0.7, 1.3))),
                "nev": rng.choice([1, 2])}
    if kind in ("ground", "sweep"):
        return {"kind": kind, "d": d, "L": rng.randint(6, 14), "D": _log(rng, 6, 40 if kind == "ground" else 240)}
    if kind == "sweep2":
        return {"kind": kind, "d": 2, "L": rng.randint(6, 16), "D": _log(rng, 6, 90)}
    if kind == "expectation":
        return {"kind": kind, "d": d, "L": rng.randint(8, 24), "D": _log(rng, 6, 250)}
    return {"kind": kind, "chains": rng.randint(4, 24), "Lmin": 6, "Lmax": rng.randint(8, 28), "Dmin": 8,
            "Dmax": rng.randint(16, 96)}


# ---------------------------------------------------------------------------
def _bulk(model, d):
    """Bulk block of the chain's MPO, (Dw, Dw, d, d)."""
    if model == "tfim":
        return models.tfim_bulk_W(d, 1.0, 0.7)
    if model == "long3":  # interactions over up to three sites, Dw = 8
        return models.long_range_bulk_W(d, 1.0, 0.5, 3)
    return models.xxz_bulk_W(d, 1.0, 1.0, 0.0, 0.1 if d == 3 else 0.0)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _isometry(g, rows, cols):
    q, r = torch.linalg.qr(torch.randn(rows, cols, dtype=torch.float64, device="cuda", generator=g))
    return q * torch.sign(torch.diagonal(r))


def _environment(g, W, d, D, start):
    """Environment (bra, w, ket) of a random canonical block that ends on a bond
    of dimension D: isometries A[i1][m][i2] contracted with W one site at a time."""
    Dw = W.shape[0]
    F = torch.zeros(1, Dw, 1, dtype=torch.float64, device="cuda")
    F[0, start, 0] = 1.0
    full = False
    while not full:
        D1 = F.shape[0]
        full = D1 == D
        D2 = min(D, D1 * d)
        A = _isometry(g, D1 * d, D2)
        T = (F.reshape(D1 * Dw, D1) @ A.reshape(D1, d * D2)).reshape(D1, Dw, d, D2)
        T = torch.einsum("awnb,wvmn->amvb", T, W).reshape(D1 * d, Dw * D2)
        F = (A.T @ T).reshape(D2, Dw, D2)
    return F


def _site(case, seed):
    """(W, L, R, x): one site's operator, its environments (bra, w, ket) and a
    unit vector x[a][m][b], as device tensors."""
    d, D1, D2 = case["d"], case["D1"], case["D2"]
    W = torch.from_numpy(_bulk(case["model"], d)).cuda()
    g = _generator(seed)
    L = _environment(g, W, d, D1, 0)
    R = _environment(g, W.permute(1, 0, 2, 3).contiguous(), d, D2, W.shape[0] - 1)
    x = torch.randn(D1, d, D2, dtype=torch.float64, device="cuda", generator=g)
    return W, L, R, x / x.norm()


def _ref(x):
    """x[a][m][b] as the library's flat site tensor psi[m + d*(a + D1*b)]."""
    return x.permute(2, 0, 1).contiguous().reshape(-1)


def _bind(case, seed):
    W, L, R, x = _site(case, seed)
    ctx = tn.Context(0)
    host = [F.permute(2, 0, 1).contiguous().reshape(-1).cpu().numpy() for F in (L, R)]
    ctx.site_bind(W.cpu().numpy(), host[0], host[1], case["d"], case["D1"], case["D2"],
                  PRECISION[case.get("precision", "fp64")])
    return ctx, _ref(x)


def _options(case):
    if case["kind"] == "batch":
        return tn.SweepOpts.default(precision=tn.TN_FP32, env_precision=tn.TN_FP32, refine=0, gauge=1, eig_tol=1e-8,
                                    max_krylov=24, max_restarts=0, reorth=1)
    if case["kind"] == "sweep":
        return tn.SweepOpts.default(refine=0, gauge=1, eig_tol=1e-8, max_krylov=24, max_restarts=0, reorth=1,
                                    time_heff=0)
    return tn.SweepOpts.default(eig_tol=1e-12)


def _couplings(seed, n):
    """Couplings of the batched workload (J, Jz, hz per chain)."""
    return models.random_xxz_couplings(n, seed)


def _members(case):
    """Length and bond dimension of every chain of a batch."""
    n, size = case["chains"], 1000003 * case["chains"] + case["Lmax"] + case["Dmax"]
    return [w[:2] for w in models.batched_workload(n, size, (case["Lmin"], case["Lmax"]),
                                                   (case["Dmin"], case["Dmax"]))]


def _chain(ctx, L, d, D, couplings):
    """A chain with its bonds as two gauge passes leave them (they cut the bonds
    at the ends to what a site can carry)."""
    J, Jz, hz = couplings
    ch = tn.Chain(ctx, models.xxz_mpo(L, 0.5 * (d - 1), Jxy=J, Jz=Jz, hz=hz, Dz=0.1 if d == 3 else 0.0), D)
    ch.initialize(1, 1)
    ch.normalize_qr(1)
    ch.normalize_qr(0)
    return ch


def _isometries(case, seed):
    """Left-canonical random chain: A[a][m][b] per site."""
    L, d, D = case["L"], case["d"], case["D"]
    g = _generator(seed)
    bonds = [1]
    for i in range(L):
        bonds.append(1 if i == L - 1 else min(D, bonds[-1] * d, d ** min(L - 1 - i, 40)))
    return [_isometry(g, bonds[i] * d, bonds[i + 1]).reshape(bonds[i], d, bonds[i + 1]) for i in range(L)]


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "heff":
        state["ctx"], state["x"] = _bind(case, seed)
        state["y"] = torch.empty_like(state["x"])
    elif kind == "eig":
        state["ctx"], x = _bind(case, seed)
        state["x"] = x.cpu().numpy()
    elif kind in ("ground", "sweep", "sweep2"):
        state["ctx"] = tn.Context(0)
        state["options"] = _options(case)
        state["seed"] = seed
        state["chain"] = _chain(state["ctx"], case["L"], case["d"], case["D"], _couplings(seed, 1)[0])
        if kind == "ground":
            state["H2"] = create_h2(state["chain"].Ws)
    elif kind == "expectation":
        state["ctx"] = tn.Context(0)
        sites = _isometries(case, seed)
        ch = tn.Chain(state["ctx"], models.xxz_mpo(case["L"], 0.5 * (case["d"] - 1)), case["D"])
        for i, A in enumerate(sites):
            ch.set_site(i, A.shape[0], A.shape[2], _ref(A).cpu().numpy())
        state["chain"] = ch
    else:
        state["ctx"] = tn.Context(0)
        state["options"] = _options(case)
        state["seed"] = seed
        state["chains"] = [_chain(state["ctx"], L, 2, D, w)
                           for (L, D), w in zip(_members(case), _couplings(seed, case["chains"]))]
        state["batch"] = tn.Batch(state["ctx"], state["chains"], max_krylov=state["options"].max_krylov)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return state


def _in_phase(v, guess):
    """An eigenvector's sign is free: the one with a non-negative overlap."""
    return v if np.dot(v, guess) >= 0 else -v


def _restart(ch, seed, options):
    """A random right-canonical state and its environments."""
    ch.initialize(1, seed)
    ch.normalize_qr(1)
    ch.load_caches(options)


def run(state):
    kind = state["case"]["kind"]
    if kind == "heff":
        state["ctx"].heff_apply_device(state["x"].data_ptr(), state["y"].data_ptr(), state["x"].numel())
        return state["y"]
    if kind == "eig":
        nev = state["case"]["nev"]
        e, X, _, _ = state["ctx"].eig_lowest(state["x"], tol=1e-12, maxit=200, nev=nev)
        if nev == 1:
            return e, _in_phase(X, state["x"])
        return e, _in_phase(X[:, 0], state["x"]), _in_phase(X[:, 1], state["x"])
    if kind == "expectation":
        return state["chain"].expectation()
    options, case = state["options"], state["case"]
    if kind == "batch":
        for k, ch in enumerate(state["chains"]):
            _restart(ch, 7919 * state["seed"] + k, options)
        for _ in range(2):
            state["batch"].sweep(0, options)
            energies = state["batch"].sweep(1, options)
        return energies
    ch = state["chain"]
    bonds = range(case["L"] - 1)
    if kind == "ground":
        ch.initialize(1, state["seed"])
        result = tn.FindVariationalGroundState(ch, [tn.ScheduleLine(2, case["D"])], options, state["H2"])
        return [result.energy] + [ch.bond_sv(b) for b in bonds]
    _restart(ch, state["seed"], options)
    st = tn.SweepStats()
    if kind == "sweep":
        ch.sweep(0, options, st)
        ch.sweep(1, options, st)
        return st.energy  # QR gauge moves keep no singular values
    ch.sweep2(0, case["D"], 0.0, options, st)
    ch.sweep2(1, case["D"], 0.0, options, st)
    return [st.energy] + [ch.bond_sv(b) for b in bonds]


# ---------------------------------------------------------------------------
def _bonds(L, d, D):
    return [min(D, d ** min(i, L - i, 40)) for i in range(L + 1)]


def _site_work(d, Dw, D1, D2, elem, vec):
    """One product with the effective Hamiltonian: two contractions over the
    channels that are not the identity; every operand once."""
    ch = max(Dw - 1, 1)
    flops = 2.0 * ch * d * D1 * D2 * (D1 + D2)
    return {"bytes": elem * Dw * (D1 * D1 + D2 * D2) + 2.0 * vec * d * D1 * D2, "flops": flops}


def work(case):
    kind = case["kind"]
    total = {"bytes": 0.0, "flops": 0.0}

    def add(w, times=1.0):
        total["bytes"] += times * w["bytes"]
        total["flops"] += times * w["flops"]

    if kind == "heff":
        add(_site_work(case["d"], _bulk(case["model"], case["d"]).shape[0], case["D1"], case["D2"],
                       OPERAND_BYTES[case["precision"]], 8))
    elif kind == "eig":  # some 20 products per eigenpair at the least, the vectors in and out
        add(_site_work(case["d"], _bulk(case["model"], case["d"]).shape[0], case["D1"], case["D2"], 8, 8),
            20 * case["nev"])
    elif kind == "expectation":  # one environment update per site
        b = _bonds(case["L"], case["d"], case["D"])
        for i in range(case["L"]):
            add(_site_work(case["d"], 5, b[i], b[i + 1], 8, 8))
    else:
        # per site and direction: a product per Krylov vector (ten at the least
        # from a random start), an environment update, and a gauge move (an
        # orthogonalisation, or a decomposition of about four times its work)
        if kind == "batch":
            chains, sweeps, elem = [(L, 2, D) for L, D in _members(case)], 2, 4
        else:
            chains, sweeps, elem = [(case["L"], case["d"], case["D"])], 2 if kind == "ground" else 1, 8
        heavy = 4.0 if kind in ("sweep2", "ground") else 1.0
        for L, d, D in chains:
            b = _bonds(L, d, D)
            two = 1 if kind == "sweep2" else 0
            for i in range(L - two):
                D1, D2 = b[i], b[i + 1 + two]
                add(_site_work(d * d if two else d, 5, D1, D2, elem, 8), 2 * sweeps * 10)
                add(_site_work(d, 5, b[i], b[i + 1], elem, 8), 2 * sweeps)
                rows, cols = (D1 * d, d * D2) if two else (D1 * d, D2)
                add({"bytes": 16.0 * rows * cols, "flops": heavy * 2.0 * rows * cols * min(rows, cols)}, 2 * sweeps)
    return total


# ---------------------------------------------------------------------------
def _heff(W, L, R, x):
    D1, d, D2 = x.shape
    Dw1, Dw2 = W.shape[0], W.shape[1]
    T = (x.reshape(D1 * d, D2) @ R.permute(2, 1, 0).reshape(D2, Dw2 * R.shape[0])).reshape(D1, d, Dw2, D2)
    T = torch.einsum("anvb,wvmn->wamb", T, W).reshape(Dw1 * D1, d * D2)
    return (L.reshape(D1, Dw1 * D1) @ T).reshape(D1, d, D2)


def _lowest(apply, start, steps):
    """Lowest eigenpair by Lanczos with two Gram-Schmidt passes per step."""
    v = start / start.norm()
    V = torch.empty(steps, start.numel(), dtype=torch.float64, device="cuda")
    T = torch.zeros(steps, steps, dtype=torch.float64)
    k = steps
    for j in range(steps):
        V[j] = v
        w = apply(v)
        c = V[:j + 1] @ w
        w = w - V[:j + 1].T @ c
        c2 = V[:j + 1] @ w
        w = w - V[:j + 1].T @ c2
        T[j, j] = (c + c2)[j].item()
        b = w.norm().item()
        if b < 1e-13 or j + 1 == steps:
            k = j + 1
            break
        T[j, j + 1] = T[j + 1, j] = b
        v = w / b
    e, Z = torch.linalg.eigh(T[:k, :k])
    x = V[:k].T @ Z[:, 0].cuda()
    return e[0].item(), x / x.norm()


def exact(case, seed):
    if case["kind"] == "heff":
        W, L, R, x = _site(case, seed)
        return _ref(_heff(W, L, R, x))
    if case["kind"] == "eig":
        W, L, R, x = _site(case, seed)
        shape = x.shape

        def apply(v):
            return _heff(W, L, R, v.reshape(shape)).reshape(-1)

        steps = min(x.numel(), 240)
        e, X = [], []
        for k in range(case["nev"]):
            def lifted(v):
                w = apply(v)
                return w + 40.0 * X[0] * (X[0] @ v) if X else w
            guess = x.reshape(-1) if k == 0 else torch.randn(x.numel(), dtype=torch.float64, device="cuda",
                                                            generator=_generator(seed + 1))
            ek, xk = _lowest(lifted, guess, steps)
            e.append(ek)
            X.append(xk)
        guess = _ref(x).cpu().numpy()
        return tuple([np.array(e)] + [_in_phase(_ref(v.reshape(shape)).cpu().numpy(), guess) for v in X])
    if case["kind"] == "expectation":
        F = torch.ones(1, 1, 1, dtype=torch.float64, device="cuda")
        for A, W in zip(_isometries(case, seed), models.xxz_mpo(case["L"], 0.5 * (case["d"] - 1))):
            D1, d, D2 = A.shape
            W = torch.from_numpy(W).cuda()
            T = (F.reshape(D1 * W.shape[0], D1) @ A.reshape(D1, d * D2)).reshape(D1, W.shape[0], d, D2)
            T = torch.einsum("awnb,wvmn->amvb", T, W).reshape(D1 * d, W.shape[1] * D2)
            F = (A.reshape(D1 * d, D2).T @ T).reshape(D2, W.shape[1], D2)
        return float(F[0, 0, 0])
    return None  # a sweep's state depends on every solve before it
