"""The work that a user has the engine do, through its public entry points.

A case is one whole call as a program makes it: a scheme built from a host
tensor and run to its norms and free energy, a run with the observables of
its last tensor, a batch of runs, or a list of requests through a server that
the program keeps.  The seed draws the temperatures, within 1e-3 (relative)
of the model's critical point, where renormalization runs are of use; the
number of steps stays below the one where such a run leaves the critical
point, so that every cut of a spectrum has a gap and the norms are functions
of the tensor.  The singular-vector basis of a scheme's tensor is not one
(each bond's basis is free), so a pass returns what does not depend on it:
every norm, the free energy, and spectra and ratios of the last tensor.
"""
import math

import numpy as np

import __graft_entry__

ISING_BETAC = math.log(1.0 + math.sqrt(2.0)) / 2.0
ISING3D_BETAC = 1.0 / 4.51152469
BAND = 1e-3
# couplings of the 3D model's three directions: with equal ones the cuts split
# eigenvalues that the cube's symmetry makes equal
ANISO = (1.0, 1.05, 0.95)
FIELD = 1e-3   # of the impurity runs, which measure a magnetisation
SCALE = {"TRG": 2.0, "BTRG": 2.0, "HOTRG": 4.0, "ATRG": 4.0, "HOTRG_3D": 8.0, "ImpurityHOTRG": 4.0}
# (scheme, model, chi) of a server's requests, in turn
MIX = (("BTRG", "ising_z2", 8), ("TRG", "ising", 16), ("BTRG", "potts3", 16), ("BTRG", "ising", 24),
       ("TRG", "ising_z2", 13), ("BTRG", "ising_z2", 32), ("TRG", "potts3", 27), ("BTRG", "ising", 32),
       ("HOTRG", "ising", 11), ("BTRG", "ising_z2", 48))


def listed():
    one = [
        # the smallest run: a few milliseconds of small launches
        ("trg_z2_chi8", "TRG", "ising_z2", 8, 20),
        # the documentation's example: BTRG, Z2 Ising, chi = 16
        ("btrg_z2_chi16", "BTRG", "ising_z2", 16, 20),
        # one run of the beta scan, alone
        ("btrg_chi32", "BTRG", "ising", 32, 20),
        # a large symmetric run: 2048 x 2048 blocks
        ("btrg_z2_chi64", "BTRG", "ising_z2", 64, 20),
        # HOTRG at the reference tests' size and at the larger one of its benchmark
        ("hotrg_chi16", "HOTRG", "ising", 16, 9),
        ("hotrg_chi32", "HOTRG", "ising", 32, 9),
        # the anisotropic method: three small truncations per half-step
        ("atrg_z2_chi16", "ATRG", "ising_z2", 16, 6),
        # 3D: six-leg tensors
        ("hotrg3d_z2_chi6", "HOTRG_3D", "ising3d_z2", 6, 6),
        # magnetisation: T and three impurity tensors, rows of four norms
        ("impurity_hotrg_chi16", "ImpurityHOTRG", "ising", 16, 8),
    ]
    cases = [dict(name=n, path="run", scheme=s, model=m, chi=c, steps=k) for n, s, m, c, k in one]
    # the conformal data of a fixed point, as after the reference tests' TRG chi = 24 run
    cases.append(dict(name="trg_chi24_observables", path="observables", scheme="TRG", model="ising", chi=24,
                      steps=10))
    # the beta scan: 128 runs in one batch
    cases.append(dict(name="batch_btrg_chi32_128", path="batch", scheme="BTRG", model="ising", chi=32, steps=20,
                      runs=128))
    # a server working off requests of mixed methods, models and sizes
    cases.append(dict(name="serve_mixed_40", path="serve", steps=12, runs=40))
    return cases


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(("btrg", "trg", "hotrg", "atrg", "hotrg3d", "impurity", "observables", "batch", "serve"))
    if kind in ("btrg", "trg"):
        model = rng.choice(("ising", "ising_z2"))
        return dict(path="run", scheme=kind.upper(), model=model, chi=_log_int(rng, 6, 40 if model == "ising" else 56),
                    steps=rng.randint(12, 20))
    if kind == "hotrg":
        return dict(path="run", scheme="HOTRG", model=rng.choice(("ising", "ising_z2")), chi=_log_int(rng, 8, 28),
                    steps=rng.randint(5, 9))
    if kind == "atrg":
        return dict(path="run", scheme="ATRG", model=rng.choice(("ising", "ising_z2")), chi=rng.randint(12, 16),
                    steps=rng.randint(3, 6))
    if kind == "hotrg3d":
        return dict(path="run", scheme="HOTRG_3D", model="ising3d_z2", chi=rng.randint(4, 6), steps=rng.randint(3, 6))
    if kind == "impurity":
        return dict(path="run", scheme="ImpurityHOTRG", model="ising", chi=_log_int(rng, 7, 18),
                    steps=rng.randint(4, 8))
    if kind == "observables":
        return dict(path="observables", scheme=rng.choice(("TRG", "BTRG")), model="ising", chi=_log_int(rng, 8, 32),
                    steps=rng.randint(6, 12))
    if kind == "batch":
        return dict(path="batch", scheme=rng.choice(("TRG", "BTRG")), model=rng.choice(("ising", "ising_z2")),
                    chi=_log_int(rng, 8, 32), steps=rng.randint(10, 20), runs=_log_int(rng, 3, 96))
    return dict(path="serve", steps=rng.randint(6, 12), runs=rng.randint(10, 40))


# ---------------------------------------------------------------- inputs
def _betac(model):
    return {"potts3": math.log(1.0 + math.sqrt(3.0)), "ising3d_z2": ISING3D_BETAC}.get(model, ISING_BETAC)


def _betas(case, seed):
    rng = np.random.default_rng(seed)
    models = [_request(case, i)[1] for i in range(case.get("runs", 1))]
    return [_betac(m) * (1.0 + BAND * rng.uniform(-1.0, 1.0)) for m in models]


def _request(case, i):
    """(scheme, model, chi, steps) of run i of the case."""
    if case["path"] != "serve":
        return case["scheme"], case["model"], case["chi"], case["steps"]
    scheme, model, chi = MIX[i % len(MIX)]
    # HOTRG squares the length that a TRG step doubles the area of
    return scheme, model, chi, case["steps"] // 2 if scheme == "HOTRG" else case["steps"]


def _ising3d_dense(beta):
    def w(b):
        x, y = math.sqrt(math.cosh(b)), math.sqrt(math.sinh(b))
        return np.array([[x, y], [x, -y]])
    z, y, x = (w(beta * a) for a in ANISO)
    return np.einsum("ai,aj,ak,al,am,an->ijklmn", z, z, y, x, y, x)


def _tensors(tk, scheme, model, beta):
    if scheme == "ImpurityHOTRG":
        T, I = tk.classical_ising(beta, "Trivial", FIELD), tk.classical_ising_impurity(beta, FIELD)
        return [T, I, I, T]
    if model == "ising3d_z2":
        return [tk.NTensor.from_dense(_ising3d_dense(beta), [[0, 1]] * 6, 2, 2)]
    if model == "potts3":
        return [tk.classical_potts(3, beta)]
    return [tk.classical_ising(beta, "Z2" if model == "ising_z2" else "Trivial")]


def prepare(case, seed):
    tk = __graft_entry__.package()
    betas = _betas(case, seed)
    state = {"tk": tk, "path": case["path"]}
    if case["path"] in ("run", "observables"):
        state.update(make=getattr(tk, case["scheme"]), T=_tensors(tk, case["scheme"], case["model"], betas[0]),
                     beta=betas[0], chi=tk.truncrank(case["chi"]), steps=tk.maxiter(case["steps"]),
                     scale=SCALE[case["scheme"]])
        return state
    reqs = []
    for i, beta in enumerate(betas):
        scheme, model, chi, steps = _request(case, i)
        reqs.append(tk.Request(scheme, _tensors(tk, scheme, model, beta), chi, steps))
    state["reqs"] = reqs
    if case["path"] == "serve":
        state["server"] = tk.Server(max_slots=64)
    return state


# ------------------------------------------------------------------ passes
def run(state):
    tk = state["tk"]
    if state["path"] == "batch":
        norms = tk.run_batch(state["reqs"])
        return {"first": norms[0], "others": np.array(norms[1:])}
    if state["path"] == "serve":
        server = state["server"]
        ids = [server.submit(r) for r in state["reqs"]]
        while server.pump():
            pass
        return [server.poll(i)[0] for i in ids]
    scheme = state["make"](*state["T"])
    norms = np.array(tk.run(scheme, state["chi"], state["steps"], verbosity=0))
    out = {"norms": norms,
           "f": tk.free_energy(norms if norms.ndim == 1 else norms[:, 0], state["beta"], state["scale"])}
    if state["path"] == "observables":
        spectrum = tk.transfer_spectrum(scheme)
        out.update(spectrum=spectrum, gsd=tk.ground_state_degeneracy(scheme), gu_wen=list(tk.gu_wen_ratio(scheme)))
    scheme.close()
    return out


def _run_flops(scheme, model, chi, steps):
    """The contractions of the method's networks in their cheapest pairwise
    order, and one product with each truncated matrix from either side; Z_N
    blocks divide a matrix product by N^2."""
    d, total = (3 if model == "potts3" else 2), 0.0
    for _ in range(steps):
        k = min(chi, d * d)
        cut = 4.0 * d ** 4 * k
        if scheme in ("TRG", "BTRG"):
            total += 2 * cut + 4.0 * d ** 2 * k ** 3 + 2.0 * d ** 2 * k ** 4
        elif scheme == "ATRG":
            total += 2 * (3 * cut + 4.0 * d ** 3 * k ** 2 + 2.0 * d ** 2 * k ** 4)
        elif scheme == "HOTRG_3D":
            total += 3 * (2.0 * d ** 9 * k ** 2 + 16.0 * d ** 8)
        else:
            nets = 9 if scheme == "ImpurityHOTRG" else 1
            total += 2 * (12.0 * d ** 6 + cut + nets * (2.0 * d ** 5 * k + 2.0 * d ** 6 * k + 2.0 * d ** 5 * k ** 2))
        d = k
    return total / {"ising": 1, "ising_z2": 4, "potts3": 9, "ising3d_z2": 4}[model]


def work(case):
    runs = case.get("runs", 1)
    flops = nbytes = 0.0
    for i in range(runs):
        scheme, model, chi, steps = _request(case, i)
        flops += _run_flops(scheme, model, chi, steps)
        rows = 4 if scheme == "ImpurityHOTRG" else 1
        nbytes += 8.0 * (rows * (64 if model == "ising3d_z2" else 16) + rows * (steps + 1))
    return {"bytes": nbytes, "flops": flops}


# ----------------------------------------------------- the same in 64 bits
# Dense numpy statements of the methods; a Z_N tensor is taken as the dense
# array of its model, whose singular values are those of its blocks together.
def _potts3_dense(beta):
    e = np.eye(3)
    return np.exp(beta * (e[:, :, None, None] + e[None, :, None, :] + e[None, None, :, :] + e[:, None, :, None]))


def _ising_dense(beta, h=0.0, impurity=False):
    w = np.array([math.sqrt(math.cosh(beta)), math.sqrt(math.sinh(beta))])
    odd = np.indices((2, 2, 2, 2)).sum(axis=0) % 2 == 1
    ch, sh = math.cosh(h * beta), math.sinh(h * beta)
    parity = np.where(odd, ch, sh) if impurity else np.where(odd, sh, ch)
    return 2.0 * parity * np.einsum("i,j,k,l->ijkl", w, w, w, w)


def _svd(T, perm, chi):
    """Top chi singular triplets of T, its legs in order `perm`, split in the middle."""
    T = T.transpose(perm)
    a, b, c, d = T.shape
    U, s, V = np.linalg.svd(T.reshape(a * b, c * d), full_matrices=False)
    k = min(chi, s.size)
    return U[:, :k].reshape(a, b, k), s[:k], V[:k].reshape(k, c, d)


def _dot(spec, *ops):
    return np.einsum(spec, *ops, optimize="optimal")


def _trg_step(st, chi):
    A, s, B = _svd(st["T"], (0, 1, 2, 3), chi)
    C, t, D = _svd(st["T"], (1, 3, 0, 2), chi)
    A, B, C, D = A * np.sqrt(s), B * np.sqrt(s)[:, None, None], C * np.sqrt(t), D * np.sqrt(t)[:, None, None]
    X = _dot("qae,pda->pqed", D, B)
    Y = _dot("dcr,ces->edrs", C, A)
    st["T"] = _dot("pqed,edrs->pqrs", X, Y)


def _power(s, a):
    small = s < np.finfo(np.float64).eps ** 0.75
    return np.where(small, s, np.where(small, 1.0, s) ** a)


def _btrg_step(st, chi):
    A, s, B = _svd(st["T"], (0, 1, 2, 3), chi)
    C, t, D = _svd(st["T"], (2, 0, 3, 1), chi)
    a, b = _power(s, 0.75), _power(t, 0.75)
    A, B, C, D = A * a, B * a[:, None, None], C * b, D * b[:, None, None]
    D, B = D * st["S1"], B * st["S2"]
    C, A = C * st["S1"][:, None, None], A * st["S2"][:, None, None]
    # D[p, 4, 1] B[q, 1, 2] C[5, 2, s] A[4, 5, r]
    X = _dot("pea,qac->pqec", D, B)
    Y = _dot("gcs,egr->cers", C, A)
    st["T"] = _dot("pqec,cers->pqrs", X, Y)
    st["S1"], st["S2"] = _power(s, -0.5), _power(t, -0.5)


def _atrg_half(T, chi):
    A, s, D = _svd(T, (0, 2, 1, 3), chi)
    B, C = D * s[:, None, None], A * s
    X, t, Y = _svd(_dot("cxd,axb->abcd", B, C), (0, 2, 1, 3), chi)
    X, Y = X * np.sqrt(t), Y * np.sqrt(t)[:, None, None]
    AX = _dot("abx,cxd->abcd", A, X)
    DY = _dot("xab,cxd->abcd", D, Y)
    H, u, G = _svd(_dot("xcyd,byax->abcd", AX, DY), (0, 1, 2, 3), chi)
    return _dot("acx,xbd->abcd", G * np.sqrt(u)[:, None, None], H * np.sqrt(u))


def _atrg_step(st, chi):
    T = _atrg_half(st["T"], chi).transpose(1, 3, 0, 2)
    st["T"] = _atrg_half(T, chi).transpose(2, 0, 3, 1)


def _eigh(M, shape, chi):
    """Top chi eigenvectors (by modulus) of the symmetrised M and the norm of what is cut."""
    lam, U = np.linalg.eigh(0.5 * (M + M.T))
    order = np.argsort(-np.abs(lam), kind="stable")
    k = min(chi, lam.size)
    return U[:, order[:k]].reshape(shape + (k,)), float(np.linalg.norm(lam[order[k:]]))


def _better(M, N, d, chi):
    U, e = _eigh(M.reshape(d * d, d * d), (d, d), chi)
    V, f = _eigh(N.reshape(d * d, d * d), (d, d), chi)
    return V if e > f else U


def _hotrg_x(T, chi):
    M = _dot("apbq,cpdq->acbd", _dot("apij,bqij->apbq", T, T), _dot("cipj,diqj->cpdq", T, T))
    N = _dot("paqb,pcqd->acbd", _dot("ipja,iqjb->paqb", T, T), _dot("ijpc,ijqd->pcqd", T, T))
    return _better(M, N, T.shape[0], chi)


def _hotrg_y(T, chi):
    M = _dot("apbq,pcqd->acbd", _dot("iajp,ibjq->apbq", T, T), _dot("pcij,qdij->pcqd", T, T))
    N = _dot("apbq,pcqd->acbd", _dot("ijap,ijbq->apbq", T, T), _dot("picj,qidj->pcqd", T, T))
    return _better(M, N, T.shape[1], chi)


def _apply_x(A, B, U):
    """A and B on top of each other, their left and right legs pairwise in U."""
    Q = _dot("bncxy,bdcr->nxydr", _dot("abn,acxy->bncxy", U, B), A)
    return _dot("nxydr,yrs->ndxs", Q, U)


def _apply_y(A, B, U):
    """A and B side by side, their bottom and top legs pairwise in U."""
    S = _dot("pxcbm,cbyr->pxmyr", _dot("paxc,abm->pxcbm", A, U), B)
    return _dot("pxmyr,xys->pmsr", S, U)


def _hotrg_step(st, chi):
    T = st["T"]
    T = _apply_x(T, T, _hotrg_x(T, chi))
    st["T"] = _apply_y(T, T, _hotrg_y(T, chi))


def _impurity_half(st, U, apply):
    T, I, J, K = st["T"], st["I"], st["J"], st["K"]
    st["T"] = apply(T, T, U)
    st["I"] = 0.5 * (apply(I, T, U) + apply(T, I, U))
    st["J"] = 0.5 * (apply(J, T, U) + apply(T, J, U))
    st["K"] = 0.25 * (apply(K, T, U) + apply(T, K, U) + apply(I, J, U) + apply(J, I, U))


def _impurity_step(st, chi):
    _impurity_half(st, _hotrg_y(st["T"], chi), _apply_y)
    _impurity_half(st, _hotrg_x(st["T"], chi), _apply_x)


def _hotrg3d_proj(T, chi):
    E = _dot("zijklx,wijkly->xzwy", T, T)
    F = _dot("izjklx,iwjkly->xzwy", T, T)
    M = _dot("bzwd,azwc->abcd", E, F)
    E = _dot("zijxkl,wijykl->xzwy", T, T)
    F = _dot("izjxkl,iwjykl->xzwy", T, T)
    N = _dot("bzwd,azwc->abcd", E, F)
    return _better(M, N, T.shape[5], chi)


def _hotrg3d_step(st, chi):
    T = st["T"]
    for _ in range(3):
        Ux = _hotrg3d_proj(T, chi)
        Uy = _hotrg3d_proj(T.transpose(0, 1, 3, 2, 5, 4), chi)
        B = _dot("azYXyx,XWn->azYyxWn", T, Ux)
        B = _dot("azYyxWn,xwm->azYyWnwm", B, Ux)
        B = _dot("azYyWnwm,zbVWvw->aYynmbVv", B, T)
        B = _dot("aYynmbVv,YVp->aynmbvp", B, Uy)
        T = _dot("aynmbvp,yvq->abpnqm", B, Uy)
        T = T.transpose(5, 3, 1, 2, 0, 4)
    st["T"] = T


_STEP = {"TRG": _trg_step, "BTRG": _btrg_step, "ATRG": _atrg_step, "HOTRG": _hotrg_step,
         "ImpurityHOTRG": _impurity_step, "HOTRG_3D": _hotrg3d_step}


def _finalize(scheme, st):
    if scheme == "HOTRG_3D":
        n = abs(_dot("aabcbc->", st["T"]))
    elif scheme == "BTRG":
        n = abs(np.einsum("abba,b,a->", st["T"], st["S1"], st["S2"]))
    else:
        n = abs(np.einsum("abba->", st["T"]))
    row = n
    if scheme == "ImpurityHOTRG":
        row = [n] + [abs(np.einsum("abba->", st[k])) for k in "IJK"]
        for k in "IJK":
            st[k] = st[k] / n
    st["T"] = st["T"] / n
    return row


def _exact_run(scheme, model, chi, steps, beta):
    if scheme == "HOTRG_3D":
        T = _ising3d_dense(beta)
    elif model == "potts3":
        T = _potts3_dense(beta)
    else:
        T = _ising_dense(beta, FIELD if scheme == "ImpurityHOTRG" else 0.0)
    st = {"T": T, "S1": np.ones(T.shape[1]), "S2": np.ones(T.shape[0])}
    if scheme == "ImpurityHOTRG":
        st.update(I=_ising_dense(beta, FIELD, True), J=_ising_dense(beta, FIELD, True), K=T)
    rows = [_finalize(scheme, st)]
    for _ in range(steps):
        _STEP[scheme](st, chi)
        rows.append(_finalize(scheme, st))
    return np.array(rows), st


def _free_energy(norms, beta, scale):
    return -sum(math.log(z) * scale ** -i for i, z in enumerate(norms)) / beta


def _observables(scheme, st):
    T = st["T"]
    if scheme == "BTRG":
        T = T * st["S2"][:, None, None, None] * st["S1"][None, :, None, None]
    v = np.linalg.eigvals(np.einsum("abca->bc", T))
    v = v[np.lexsort((-v.imag, -v.real, -np.abs(v)))]
    p = np.abs(v / v.sum())
    p = p[p > 0.0]
    P = np.einsum("abbc->ac", T)
    n = np.trace(P)
    return {"spectrum": v.astype(complex), "gsd": float(np.exp(-np.sum(p * np.log(p)))),
            "gu_wen": [float(n * n / np.trace(P @ P)), float(n * n / np.einsum("abcd,dcba->", T, T))]}


def _quick(scheme, model, chi, steps):
    """Whether numpy does the run within a few seconds."""
    if scheme in ("TRG", "BTRG"):
        return chi <= 32
    return chi <= (32 if scheme == "HOTRG" else 18)


def exact(case, seed):
    betas = _betas(case, seed)
    if case["path"] in ("run", "observables"):
        scheme, model, chi, steps = _request(case, 0)
        if not _quick(scheme, model, chi, steps):
            return None
        norms, st = _exact_run(scheme, model, chi, steps, betas[0])
        out = {"norms": norms, "f": _free_energy(norms if norms.ndim == 1 else norms[:, 0], betas[0], SCALE[scheme])}
        if case["path"] == "observables":
            out.update(_observables(scheme, st))
        return out
    if case["path"] == "batch":
        scheme, model, chi, steps = _request(case, 0)
        return {"first": _exact_run(scheme, model, chi, steps, betas[0])[0], "others": None}
    out = []
    for i, beta in enumerate(betas):
        scheme, model, chi, steps = _request(case, i)
        out.append(_exact_run(scheme, model, chi, steps, beta)[0] if chi <= 16 and i < len(MIX) else None)
    return out
