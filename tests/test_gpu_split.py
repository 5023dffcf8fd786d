"""Lane-form quartets shared by several lanes (the last group of a bra pair, and every group
of small systems): the sizes where the groups fill differently, each against the oracle
(max |dF| <= 1e-10 Eh, the same quartets), with contracted kets of 1 to 64 primitives, alone
and as a batch; mixed builds with every quartet in FP32 (threshold above every bound) against
the oracle to the FP32 rounding of sums of terms below 20 Eh: 2^-24 x 20 x sqrt(4096) = 8e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def torch_cuda():
    import torch  # before the library: torch brings its own HIP runtime
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible: GPU tests must run on an MI355X")


CASES = [(1, "STO-3G"), (1, "6-31G(d)"), (1, "cc-pVDZ"), (2, "cc-pVDZ"), (3, "6-311G(d,p)"), (5, "STO-3G")]


def _density(n, seed):
    A = np.random.default_rng(seed).standard_normal((n, n))
    return 0.5 * A @ A.T / n


def _dF(J, K, Jo, Ko):
    return float(np.max(np.abs((J - 0.5 * K) - (Jo - 0.5 * Ko))))


@pytest.mark.parametrize("n,basis", CASES)
def test_against_oracle(oracle_mod, n, basis):
    from tonto_amd.geometry import water_cluster
    from tonto_amd.gpu import JKEngine
    mol = water_cluster(n, basis, seed=n)
    e = JKEngine(mol, schwarz=1e-12, fp32_threshold=1e30)
    max_I = e.schwarz()
    P = _density(mol.n_bf, n)
    o = oracle_mod.OracleSystem(mol)
    Jo, Ko = o.make_r_JK(P, schwarz=1e-12, max_I=max_I)
    J, K = e.make_r_JK(P)
    q = e.stats()
    assert _dF(J, K, Jo, Ko) <= 1e-10
    J, K = e.make_r_JK(P, mixed=True)
    assert e.stats()["quartets"] == q["quartets"] and e.stats()["prim_quartets"] == q["prim_quartets"]
    assert e.stats()["fp32_quartets"] == q["quartets"]
    assert _dF(J, K, Jo, Ko) <= 8e-5


def test_batch_against_singles():
    from tonto_amd.geometry import water_cluster
    from tonto_amd.gpu import JKEngine
    mols = [water_cluster(1 + i % 4, "cc-pVDZ", seed=40 + i) for i in range(9)]
    Ps = [_density(m.n_bf, i) for i, m in enumerate(mols)]
    e = JKEngine(mols, schwarz=1e-11)
    e.schwarz()
    Js, Ks = e.make_r_JK(Ps)
    total = 0
    for m, P, J, K in zip(mols, Ps, Js, Ks):
        s = JKEngine(m, schwarz=1e-11)
        s.schwarz()
        J1, K1 = s.make_r_JK(P)
        total += s.stats()["quartets"]
        assert _dF(J, K, J1, K1) <= 1e-11
    assert e.stats()["quartets"] == total
