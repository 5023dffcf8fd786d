"""Device memory of the wavefront-form workspace: sized by what the class launches can use, and
kept for the next context instead of freed and allocated with every set-up."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.fixture(autouse=True)
def torch_cuda():
    import torch  # before the library: torch brings its own HIP runtime
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible: GPU tests must run on an MI355X")


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _setup(n):
    from tonto_amd.geometry import water_cluster
    from tonto_amd.gpu import JKEngine
    mol = water_cluster(n, "cc-pVTZ", seed=n)
    e = JKEngine(mol, schwarz=1e-9)
    before = _free()
    e.schwarz()
    return mol, e, before - _free()


def test_small_systems_take_little():
    # the second context can't take a workspace that an earlier one left
    held = _setup(1)
    used = [_setup(1)[2], _setup(2)[2]]
    print("MiB allocated by the Schwarz step:", [u / MIB for u in used], held[2] / MIB)
    assert max(used) <= 64 * MIB


def test_next_context_takes_the_kept_workspace(oracle_mod):
    mol, e, _ = _setup(9)
    e.close()
    for _ in range(3):
        mol, e, used = _setup(9)
        assert used <= 64 * MIB
        e.close()
    # a smaller system in the kept buffer, still dirty, against the oracle
    mol, e, used = _setup(2)
    A = np.random.default_rng(1).standard_normal((mol.n_bf, mol.n_bf))
    P = 0.5 * A @ A.T / mol.n_bf
    J, K = e.make_r_JK(P)
    Jo, Ko = oracle_mod.OracleSystem(mol).make_r_JK(P, schwarz=1e-9, max_I=e.schwarz())
    assert used <= 64 * MIB
    assert np.max(np.abs((J - 0.5 * K) - (Jo - 0.5 * Ko))) <= 1e-10
    e.close()
