"""The lane form with each wavefront's own K rows in LDS (batches, short ket segments), against
the oracle: every class pair that has a lane form, part of the rows in LDS, and a batch with f
shells.  J and K to 1e-10 (FP64) and 1e-8 (mixed), the same quartets."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(autouse=True)
def torch_cuda():
    import torch  # before the library: torch brings its own HIP runtime
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible: GPU tests must run on an MI355X")


def _density(n, seed):
    A = np.random.default_rng(seed).standard_normal((n, n))
    return A @ A.T / n


def _lane_classes():
    from tonto_amd.build import class_list
    from tonto_amd.flops import class_pairs
    heavy = {tuple(c[:4]): c[4] for c in class_list()}
    return [k for k, cp in enumerate(class_pairs()) if not heavy[tuple(cp)]]


def _engine(monkeypatch, mol, budget=None, **options):
    """A context that takes no ket segment for the form with one bra pair per work-group."""
    from tonto_amd.gpu import JKEngine
    monkeypatch.setenv("TGPU_KROW_MIN_KETS", str(10 ** 9))
    if budget:
        monkeypatch.setenv("TGPU_KROW_BUDGET", str(budget))
    e = JKEngine(mol, **options)
    monkeypatch.undo()
    return e


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,seed", [(2, 0), (4, 2)])
def test_every_lane_class(monkeypatch, oracle_mod, mixed, n, seed):
    from tonto_amd.flops import class_pairs
    from tonto_amd.geometry import water_cluster
    mol = water_cluster(n, "cc-pVTZ", seed=seed)
    P = _density(mol.n_bf, 31)
    e = _engine(monkeypatch, mol, schwarz=1e-11)
    max_I = e.schwarz()
    Jo, Ko, so = oracle_mod.OracleSystem(mol).make_r_JK(P, schwarz=1e-11, max_I=max_I, return_stats=True)
    light = _lane_classes()
    for k in light:
        for kk in light:
            e.set_variant(kk, 1)
        e.set_variant(k, 0)
        J, K = e.make_r_JK(P, mixed=mixed)
        dJ, dK = np.max(np.abs(J - Jo)), np.max(np.abs(K - Ko))
        print(f"class {class_pairs()[k]} mixed={mixed}: dJ={dJ:.2e} dK={dK:.2e}")
        assert e.stats()["quartets"] == so["quartets"]
        assert max(dJ, dK) <= (1e-8 if mixed else 1e-10), class_pairs()[k]


@pytest.mark.parametrize("budget", [22016, 31200])
def test_part_of_the_rows(monkeypatch, oracle_mod, budget):
    """(H2O)8/6-31G(d): 56 s-type, 48 p-type, 48 d-type functions, so four rows (one of each
    wavefront) take 1792 B for (..|ss) and 3328 B for (..|ps).  22016 B leave, next to the 14848
    of the two-root classes, 4 of 6 rows of (pp|ss), 4 of 7 of (ds|ss), 2 of 4 of (ps|ps); 31200,
    next to the 22240 of the three-root classes, 5 of 12 of (dd|ss); (dp|ps), with
    room for 2 of 9, updates K globally."""
    from tonto_amd.geometry import water_cluster
    g = np.load(os.path.join(HERE, "golden", "w8_631gd.npz"))
    mol = water_cluster(8, "6-31G(d)", seed=int(g["seed"]))
    e = _engine(monkeypatch, mol, budget, schwarz=1e-12)
    max_I = e.schwarz()
    for k in _lane_classes():
        e.set_variant(k, 0)
    J, K = e.make_r_JK(g["P"])
    Jo, Ko = oracle_mod.OracleSystem(mol).make_r_JK(g["P"], schwarz=1e-12, max_I=max_I)
    assert max(np.max(np.abs(J - Jo)), np.max(np.abs(K - Ko))) <= 1e-10


@pytest.mark.parametrize("mixed", [False, True])
def test_batch_with_f_shells(oracle_mod, mixed):
    from tonto_amd.geometry import water_cluster
    from tonto_amd.gpu import JKEngine
    mols = [water_cluster(n, "cc-pVTZ", seed=50 + i) for i, n in enumerate((1, 3, 2, 1))]
    Ps = [_density(m.n_bf, i) for i, m in enumerate(mols)]
    e = JKEngine(mols, schwarz=1e-11)
    max_I = e.schwarz()
    Js, Ks = e.make_r_JK(Ps, mixed=mixed)
    quartets = 0
    for i, (m, P, J, K) in enumerate(zip(mols, Ps, Js, Ks)):
        Jo, Ko, so = oracle_mod.OracleSystem(m).make_r_JK(P, schwarz=1e-11, return_stats=True,
                                                          max_I=max_I[e.pair_off[i]:e.pair_off[i + 1]])
        quartets += so["quartets"]
        assert max(np.max(np.abs(J - Jo)), np.max(np.abs(K - Ko))) <= (1e-8 if mixed else 1e-10), i
    assert e.stats()["quartets"] == quartets
