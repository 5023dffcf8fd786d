"""The allocating build captured by the caller, on a stream of its own that no build ran on before,
and replayed: each replay against a build outside.  J and K to 1e-12 (FP64 atomics in another
order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_build_captured_by_the_caller():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible: GPU tests must run on an MI355X")
    from tonto_amd.geometry import water_cluster
    from tonto_amd.gpu import JKEngine
    mol = water_cluster(2, "6-31G(d)", seed=21)
    e = JKEngine(mol, schwarz=1e-11)
    e.schwarz()
    A = np.random.default_rng(21).standard_normal((mol.n_bf, mol.n_bf))
    P = torch.tensor(0.5 * A @ A.T / mol.n_bf, device="cuda")
    J, K = torch.empty_like(P), torch.empty_like(P)
    e.set_stream(torch.cuda.current_stream().cuda_stream)
    e.make_r_JK_device(P.data_ptr(), J.data_ptr(), K.data_ptr())
    torch.cuda.synchronize()
    J0, K0 = J.clone(), K.clone()
    st, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        e.set_stream(st.cuda_stream)
        e.make_r_JK_device(P.data_ptr(), J.data_ptr(), K.data_ptr())
    for _ in range(3):
        J.fill_(float("nan"))
        K.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert float((J - J0).abs().max()) <= 1e-12 and float((K - K0).abs().max()) <= 1e-12
        # a build outside the graph between the replays
        e.set_stream(torch.cuda.current_stream().cuda_stream)
        e.make_r_JK_device(P.data_ptr(), J.data_ptr(), K.data_ptr())
        torch.cuda.synchronize()
        assert float((J - J0).abs().max()) <= 1e-12
