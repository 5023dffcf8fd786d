"""Performance cases: the calls a direct-SCF program makes of this library, over the range
of systems it makes them for.

Kinds of case
  build    one J/K build, P, J and K resident on the GPU (JKEngine.make_r_JK_device): the
           call of every SCF iteration.  n waters in a basis; FP64 or mixed precision,
           Cartesian or spherical, launched or replayed from a graph, the whole density or
           a density difference (the incremental iterations, at their tighter cutoffs).
  jonly    the allocation-free build of J alone, for callers that hold the scratch.
  uhf      one UHF build (make_u_JK_device) of a singly ionised cluster.
  batch    one build of many independent small clusters in the same launches (the learned
           guess's training data, conformer screens).
  setup    a new geometry: the context, S, T, V and the Schwarz table.
  train    forward, loss and backward of one minibatch of the learned guess's network.

Densities: every water's five lowest orbitals of T + V/2 on its own functions (screened
nuclei), orthogonalised over the cluster, P = 2 C (C^T S C)^-1 C^T.  Idempotent, with blocks
between the molecules that fall off as an SCF density's do: the builds then screen like
those of an SCF's densities (quartets within 20 %, times within 5 % on 8 to 32 waters).
"""
import math

import numpy as np
import torch

from tonto_amd.basis import Molecule, cart_components
from tonto_amd.geometry import water_cluster
from tonto_amd.gpu import JKEngine
from tonto_amd.mlp import DeviceNet, init_params

N_IN, NH = 273, 128  # the learned guess's network

# functions per water, and FLOPs of a build (tonto_amd.flops) over n^2.5 for n waters at the
# screening of an SCF (measured on 2 to 32 waters), per basis
BF = {"STO-3G": 7, "6-31G(d)": 19, "6-31G(d,p)": 25, "6-311G(d,p)": 31, "cc-pVDZ": 25,
      "aug-cc-pVDZ": 43, "cc-pVTZ": 65}
SPH_BF = {"cc-pVTZ": 58}
FLOPS = {"STO-3G": 4e6, "6-31G(d)": 2e7, "6-31G(d,p)": 3e7, "6-311G(d,p)": 3.6e7, "cc-pVDZ": 8e7,
         "aug-cc-pVDZ": 4.6e8, "cc-pVTZ": 5.6e8}


def _build(name, n, basis, schwarz=1e-9, mixed=False, spherical=False, graph=False, delta=False):
    c = dict(kind="build", n=n, basis=basis, schwarz=schwarz, mixed=mixed, spherical=spherical, graph=graph,
             delta=delta)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one molecule, as in most of the tests and in every atomic or monomer SCF: latency
        _build("water 6-31G(d)", 1, "6-31G(d)"),
        # an open-shell ion of the same size: three passes
        dict(name="water cation UHF", kind="uhf", n=1, basis="6-311G(d,p)", schwarz=1e-9),
        # a small cluster at tight screening, replayed from a graph as an SCF loop does
        _build("8 waters 6-31G(d) graph", 8, "6-31G(d)", schwarz=1e-12, graph=True),
        # spherical d and f functions, an odd number of molecules
        _build("5 waters cc-pVTZ spherical", 5, "cc-pVTZ", spherical=True),
        # Coulomb alone with diffuse functions (J-only engine of a pure functional)
        dict(name="7 waters aug-cc-pVDZ J", kind="jonly", n=7, basis="aug-cc-pVDZ", schwarz=1e-10),
        # an ordinary FP64 build with f functions
        _build("12 waters cc-pVTZ FP64", 12, "cc-pVTZ", schwarz=1e-11),
        # a difference build of an incremental mixed SCF
        _build("19 waters 6-311G(d,p) delta", 19, "6-311G(d,p)", schwarz=1e-10, mixed=True, delta=True),
        # a mixed build of a large cluster in a double-zeta class basis
        _build("32 waters 6-311G(d,p) mixed", 32, "6-311G(d,p)", mixed=True),
        # the largest: 2080 functions, every class of s to f shells
        _build("32 waters cc-pVTZ mixed", 32, "cc-pVTZ", schwarz=1e-11, mixed=True),
        # a batch of independent clusters of 1 to 13 waters
        dict(name="batch of 256 clusters", kind="batch", count=256, most=13, basis="6-31G(d,p)", graph=True),
        # every new geometry of an optimisation or a scan pays for this
        dict(name="setup 16 waters cc-pVTZ", kind="setup", n=16, basis="cc-pVTZ"),
        # a training minibatch for the O-O blocks of 6-31G(d)
        dict(name="guess training step", kind="train", rows=2048, n_out=225),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


# the most waters of a single-molecule build drawn in each basis
MOST = {"STO-3G": 24, "6-31G(d)": 30, "6-31G(d,p)": 28, "6-311G(d,p)": 32, "cc-pVDZ": 24, "aug-cc-pVDZ": 16,
        "cc-pVTZ": 20}


def draw(rng):
    kind = rng.choice(["build"] * 6 + ["jonly", "uhf", "batch", "setup", "train"])
    basis = rng.choice(sorted(MOST))
    schwarz = rng.choice([1e-9, 1e-10, 1e-11, 1e-12])
    if kind == "build":
        n = _log_int(rng, 1, MOST[basis])
        spherical = basis in SPH_BF and rng.random() < 0.3
        return _build(None, n, basis, schwarz, rng.random() < 0.5, spherical,
                      rng.random() < 0.3, not spherical and rng.random() < 0.25)
    if kind == "jonly":
        return dict(kind=kind, n=_log_int(rng, 1, min(14, MOST[basis])), basis=basis, schwarz=schwarz)
    if kind == "uhf":
        return dict(kind=kind, n=_log_int(rng, 1, min(10, MOST[basis])), basis=basis, schwarz=schwarz)
    if kind == "batch":
        return dict(kind=kind, count=_log_int(rng, 8, 200), most=rng.randint(2, 12),
                    basis=rng.choice(["STO-3G", "6-31G(d)", "6-31G(d,p)"]), graph=rng.random() < 0.5)
    if kind == "setup":
        return dict(kind=kind, n=_log_int(rng, 2, 20), basis=basis)
    return dict(kind=kind, rows=_log_int(rng, 65, 8192), n_out=rng.choice([4, 30, 225]))


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
def _monomers(mol):
    out = []
    for k in range(0, mol.n_atom, 3):
        m = Molecule(mol.symbols[k:k + 3], mol.coords[k:k + 3], mol.basis_name)
        m.build_shells()
        out.append(m)
    return out


def _one_electron(mols, spherical):
    """S, T, V of each molecule."""
    if not spherical:
        e = JKEngine(mols)
        S, T, V = e.one_electron()
        e.close()
        return list(zip(S, T, V)) if len(mols) > 1 else [(S, T, V)]
    out = []
    for m in mols:
        e = JKEngine(m, spherical=True)
        out.append(e.one_electron())
        e.close()
    return out


def _orbitals(monos, mats, screen):
    """The waters' five lowest orbitals each, as columns over the cluster's functions."""
    C = np.zeros((sum(s.shape[0] for s, _, _ in mats), 5 * len(monos)))
    row = 0
    for k, (s, t, v) in enumerate(mats):
        w, U = np.linalg.eigh(s)
        X = U / np.sqrt(w)
        c = X @ np.linalg.eigh(X.T @ (t + screen * v) @ X)[1]
        C[row:row + s.shape[0], 5 * k:5 * k + 5] = c[:, :5]
        row += s.shape[0]
    return C


def _projector(C, S):
    return C @ np.linalg.solve(C.T @ S @ C, C.T)


def _density(mol, S, spherical=False, delta=False):
    monos = _monomers(mol)
    mats = _one_electron(monos, spherical)
    P = 2.0 * _projector(_orbitals(monos, mats, 0.5), S)
    if delta:  # two successive densities of an SCF
        P = P - 2.0 * _projector(_orbitals(monos, mats, 0.51), S)
    return 0.5 * (P + P.T)


def _device(a):
    return torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        rng = np.random.default_rng(seed)
        net = DeviceNet(N_IN, NH, case["n_out"], init_params(N_IN, NH, case["n_out"], seed))
        X = rng.standard_normal((case["rows"], N_IN)).astype(np.float32)
        T = rng.standard_normal((case["rows"], case["n_out"])).astype(np.float32)
        return dict(case=case, net=net, X=torch.tensor(X, device="cuda"), T=torch.tensor(T, device="cuda"))
    if kind == "batch":
        # the sizes belong to the case, the geometries to the seed
        sizes = np.random.default_rng(case["most"]).integers(1, case["most"] + 1, case["count"])
        mols = [water_cluster(int(n), case["basis"], seed=seed * 4096 + i) for i, n in enumerate(sizes)]
        eng = JKEngine(mols)
        S = eng.one_electron()[0]
        monos = [m for mol in mols for m in _monomers(mol)]
        mats = _one_electron(monos, False)
        Ps, k = [], 0
        for mol, s in zip(mols, S):
            n = mol.n_atom // 3
            P = 2.0 * _projector(_orbitals(monos[k:k + n], mats[k:k + n], 0.5), s)
            Ps.append(0.5 * (P + P.T))
            k += n
        P = _device(eng.pack(Ps))
    elif kind == "setup":
        return dict(case=case, mol=water_cluster(case["n"], case["basis"], seed=seed))
    else:
        mol = water_cluster(case["n"], case["basis"], seed=seed)
        spherical = case.get("spherical", False)
        density_cutoff = 1e-12 if case.get("delta") else 1e-9
        eng = JKEngine(mol, schwarz=case["schwarz"], j_density=density_cutoff, k_density=density_cutoff,
                       spherical=spherical)
        S = eng.one_electron()[0]
        if kind == "uhf":  # the last water's highest orbital has lost its beta electron
            monos = _monomers(mol)
            C = _orbitals(monos, _one_electron(monos, False), 0.5)
            Pa, Pb = _projector(C, S), _projector(C[:, :-1], S)
            P = _device(0.5 * (Pa + Pa.T))
        else:
            P = _device(_density(mol, S, spherical, case.get("delta", False)))
    eng.schwarz()
    st = dict(case=case, eng=eng, P=P, J=torch.empty_like(P), K=torch.empty_like(P))
    if kind == "uhf":
        st.update(Pb=_device(0.5 * (Pb + Pb.T)), Jb=torch.empty_like(P), Kb=torch.empty_like(P))
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "train":
        loss = st["net"].loss_and_grad(st["X"], st["T"], 1.0 / st["T"].numel())
        return loss, st["net"].g
    if kind == "setup":
        eng = JKEngine(st["mol"])
        S, T, V = eng.one_electron()
        max_I = eng.schwarz()
        eng.close()
        return S, T, V, max_I
    eng, P, J, K = st["eng"], st["P"], st["J"], st["K"]
    eng.set_stream(torch.cuda.current_stream().cuda_stream)
    if kind == "uhf":
        eng.make_u_JK_device(P.data_ptr(), st["Pb"].data_ptr(), J.data_ptr(), st["Jb"].data_ptr(), K.data_ptr(),
                             st["Kb"].data_ptr())
        return J, st["Jb"], K, st["Kb"]
    if kind == "jonly":
        eng.make_r_JK_device_noalloc(P.data_ptr(), J.data_ptr(), K.data_ptr(), only="J")
        return J
    eng.make_r_JK_device(P.data_ptr(), J.data_ptr(), K.data_ptr(), mixed=case.get("mixed", False),
                         graph=case["graph"])
    return J, K


def work(case):
    kind = case["kind"]
    if kind == "train":
        per_row = N_IN * NH + NH * NH + NH * case["n_out"]
        n_par = per_row + 2 * NH + case["n_out"]
        return {"bytes": 4.0 * (case["rows"] * (N_IN + case["n_out"]) + 2 * n_par),
                "flops": 2.0 * case["rows"] * (3 * per_row - N_IN * NH)}
    n_bf, flops = BF[case["basis"]], FLOPS[case["basis"]]
    if kind == "batch":  # sizes 1 .. most equally likely
        sizes = range(1, case["most"] + 1)
        n2 = case["count"] * sum((n * n_bf) ** 2 for n in sizes) / len(sizes)
        return {"bytes": 8.0 * 3 * n2, "flops": case["count"] * sum(flops * n ** 2.5 for n in sizes) / len(sizes)}
    n = case["n"]
    if case.get("spherical"):
        n_bf = SPH_BF[case["basis"]]
    n2 = (n * n_bf) ** 2
    if kind == "setup":  # out: S, T, V and max_I (about n2 / 10 shell pairs); about 40 nuclei x 30 FLOPs an element
        return {"bytes": 8.0 * 3.1 * n2, "flops": 30.0 * 3 * n * n2}
    if kind == "uhf":
        return {"bytes": 8.0 * 6 * n2, "flops": 2 * flops * n ** 2.5}
    if kind == "jonly":
        return {"bytes": 8.0 * 2 * n2, "flops": 0.7 * flops * n ** 2.5}
    return {"bytes": 8.0 * 3 * n2, "flops": flops * n ** 2.5 * (0.5 if case["delta"] else 1.0)}


# ------------------------------------------------------------------------------------------
# the same results in plain 64-bit numpy: every integral of one molecule by the
# McMurchie-Davidson Hermite expansion (Helgaker, Jorgensen and Olsen, "Molecular
# Electronic-Structure Theory", ch. 9)
# ------------------------------------------------------------------------------------------
def _boys(m_max, T):
    """F_0 .. F_m_max(T): the series of the highest order and downward recursion, for large T
    the error function and upward recursion."""
    F = np.empty((m_max + 1,) + T.shape)
    big = T > 45.0
    t = np.where(big, 1.0, T)
    term = np.full(T.shape, 1.0 / (2 * m_max + 1))
    total = term.copy()
    e = np.exp(-t)
    for i in range(1, 190):
        term = term * (2.0 * t) / (2 * m_max + 2 * i + 1)
        total += term
    F[m_max] = e * total
    for m in range(m_max - 1, -1, -1):
        F[m] = (2.0 * t * F[m + 1] + e) / (2 * m + 1)
    if big.any():
        tb = T[big]
        f, eb = 0.5 * np.sqrt(math.pi / tb), np.exp(-tb)
        F[0][big] = f
        for m in range(m_max):
            f = ((2 * m + 1) * f - eb) / (2.0 * tb)
            F[m + 1][big] = f
    return F


def _hermite_1d(la, lb, a, b, d):
    """E[i][j][t] of one axis for arrays of primitive pairs (distance d between the centres)."""
    p = a + b
    pa, pb = -b / p * d, a / p * d
    E = {(0, 0): [np.exp(-a * b / p * d * d)]}

    def up(e, x):
        n = len(e)
        return [(e[t - 1] / (2 * p) if t else 0.0) + (x * e[t] if t < n else 0.0) +
                ((t + 1) * e[t + 1] if t + 1 < n else 0.0) for t in range(n + 1)]
    for i in range(la + 1):
        if i:
            E[i, 0] = up(E[i - 1, 0], pa)
        for j in range(1, lb + 1):
            E[i, j] = up(E[i, j - 1], pb)
    return E


def _hermites(L):
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


def _pair_lists(mol):
    """{(la, lb): (shell pairs, first primitive pair of each, p, P, E[primitive pair, functions, Hermites])}"""
    out = {}
    for x, a in enumerate(mol.shells):
        for y, b in enumerate(mol.shells):
            if (a.l, x) < (b.l, y):
                continue
            out.setdefault((a.l, b.l), []).append((a, b))
    lists = {}
    for (la, lb), prs in out.items():
        ea, eb, cc, d, P, first = [], [], [], [], [], []
        for a, b in prs:
            first.append(len(ea))
            for e1, c1 in zip(a.exps, a.coefs):
                for e2, c2 in zip(b.exps, b.coefs):
                    ea.append(e1)
                    eb.append(e2)
                    cc.append(c1 * c2)
                    A, B = np.array(a.center), np.array(b.center)
                    d.append(A - B)
                    P.append((e1 * A + e2 * B) / (e1 + e2))
        ea, eb, cc, d = np.array(ea), np.array(eb), np.array(cc), np.array(d)
        ax = [_hermite_1d(la, lb, ea, eb, d[:, k]) for k in range(3)]
        hs = _hermites(la + lb)
        ca, cb = cart_components(la), cart_components(lb)
        E = np.zeros((len(ea), len(ca) * len(cb), len(hs)))
        for i, x in enumerate(ca):
            for j, y in enumerate(cb):
                for h, (t, u, v) in enumerate(hs):
                    e = [ax[k][x[k], y[k]] for k in range(3)]
                    if t < len(e[0]) and u < len(e[1]) and v < len(e[2]):
                        E[:, i * len(cb) + j, h] = cc * e[0][t] * e[1][u] * e[2][v]
        lists[la, lb] = (prs, np.array(first), ea + eb, np.array(P), E)
    return lists


def _hermite_coulomb(L, alpha, d):
    """R_{tuv}, t + u + v <= L, of arrays of primitive quartets."""
    F = _boys(L, alpha * (d * d).sum(-1))
    R = {(0, 0, 0): [(-2.0 * alpha) ** n * F[n] for n in range(L + 1)]}
    for s in range(1, L + 1):
        for h in _hermites(s):
            if sum(h) != s:
                continue
            k = max(range(3), key=lambda i: h[i])
            one = tuple(h[i] - (i == k) for i in range(3))
            two = tuple(h[i] - 2 * (i == k) for i in range(3))
            R[h] = [d[..., k] * R[one][n + 1] + ((h[k] - 1) * R[two][n + 1] if h[k] > 1 else 0.0)
                    for n in range(L - s + 1)]
    return {h: r[0] for h, r in R.items()}


def _integrals(mol):
    """(ab|cd) over all functions."""
    n = mol.n_bf
    out = np.zeros((n, n, n, n))
    lists = _pair_lists(mol)
    for (la, lb), (pa, fa, p, P, Ea) in lists.items():
        for (lc, ld), (pc, fc, q, Q, Ec) in lists.items():
            ha, hc = _hermites(la + lb), _hermites(lc + ld)
            alpha = p[:, None] * q[None] / (p[:, None] + q[None])
            R = _hermite_coulomb(la + lb + lc + ld, alpha, P[:, None] - Q[None])
            pref = 2.0 * math.pi ** 2.5 / (p[:, None] * q[None] * np.sqrt(p[:, None] + q[None]))
            half = np.empty((len(p), len(ha), len(pc), Ec.shape[1]))
            for i, x in enumerate(ha):
                M = np.stack([(-1.0) ** sum(y) * R[tuple(np.add(x, y))] * pref for y in hc], -1)
                half[:, i] = np.add.reduceat(np.einsum("pqh,qfh->pqf", M, Ec), fc, axis=1)
            full = np.add.reduceat(np.einsum("phcf,pgh->pgcf", half, Ea), fa, axis=0)
            for i, (a, b) in enumerate(pa):
                for j, (c, d) in enumerate(pc):
                    s = [slice(t.first_bf, t.first_bf + t.n_comp) for t in (a, b, c, d)]
                    v = full[i, :, j].reshape(a.n_comp, b.n_comp, c.n_comp, d.n_comp)
                    for u, ab in ((v, s[:2]), (v.transpose(1, 0, 2, 3), s[1::-1])):
                        out[ab[0], ab[1], s[2], s[3]] = u
                        out[ab[0], ab[1], s[3], s[2]] = u.transpose(0, 1, 3, 2)
    return out


def _exact_train(case, seed):
    rows, n_out = case["rows"], case["n_out"]
    st_rng = np.random.default_rng(seed)
    X = st_rng.standard_normal((rows, N_IN)).astype(np.float32)
    T = st_rng.standard_normal((rows, n_out)).astype(np.float32)
    par = torch.tensor(init_params(N_IN, NH, n_out, seed), dtype=torch.float64, requires_grad=True)
    W, o = [], 0
    for shape in ((N_IN, NH), (NH,), (NH, NH), (NH,), (NH, n_out), (n_out,)):
        size = int(np.prod(shape))
        W.append(par[o:o + size].reshape(shape))
        o += size
    a = torch.tensor(X, dtype=torch.float64)
    a = torch.nn.functional.silu(a @ W[0] + W[1])
    a = torch.nn.functional.silu(a @ W[2] + W[3])
    y = a @ W[4] + W[5]
    loss = ((y - torch.tensor(T, dtype=torch.float64)) ** 2).sum() / T.size
    loss.backward()
    return loss.detach().reshape(1), par.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    # one water has atoms in common in every quartet, so no primitive pair is dropped there
    if kind not in ("build", "jonly", "uhf") or case["n"] > 1 or case["basis"] in ("cc-pVTZ", "aug-cc-pVDZ") or \
            case.get("delta"):
        return None
    st = prepare(case, seed)
    I = _integrals(water_cluster(1, case["basis"], seed=seed))
    J = lambda P: np.einsum("abcd,cd->ab", I, P)  # noqa: E731
    K = lambda P: np.einsum("acbd,cd->ab", I, P)  # noqa: E731
    P = st["P"].cpu().numpy()
    if kind == "uhf":  # Ja and Jb alone are split as Tonto's engine splits them
        return None, None, K(P), K(st["Pb"].cpu().numpy())
    if kind == "jonly":
        return J(P)
    return J(P), K(P)
