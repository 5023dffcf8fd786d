"""The network's kernel forms at the sizes where they can go wrong, against the numpy reference:
row blocks and tiles with remainders, a batch longer than one work-group's share of the
weight gradients, a net whose row block exceeds the LDS (general products).  FP32 sums of K
terms in another order: |error| <= 2^-24 (2 K)^(1/2) 8 max|result| with K the longest sum,
rounded up to 1e-4 relative to the largest entry, as for the other network tests."""
import numpy as np
import pytest

import oracle.mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,nh,n_out,M", [(1, 1, 1, 1), (273, 128, 225, 2047), (33, 31, 17, 16), (64, 48, 32, 17),
                                             (1000, 300, 900, 50), (9, 8, 5, 33000), (700, 16, 3, 200)])
def test_forms_against_reference(n_in, nh, n_out, M):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible: GPU tests must run on an MI355X")
    from tonto_amd.mlp import DeviceNet, init_params
    rng = np.random.default_rng(M)
    p = init_params(n_in, nh, n_out, 1)
    p = p + rng.standard_normal(p.size).astype(np.float32) * 0.01
    X = rng.standard_normal((M, n_in)).astype(np.float32)
    T = rng.standard_normal((M, n_out)).astype(np.float32)
    net = DeviceNet(n_in, nh, n_out, p)
    Xd, Td = torch.tensor(X, device="cuda"), torch.tensor(T, device="cuda")
    scale = 1.0 / (M * n_out)
    net.g.fill_(float("nan"))
    loss = float(net.loss_and_grad(Xd, Td, scale)[0])
    g = net.g.cpu().numpy()
    Y = net.forward(Xd).cpu().numpy()
    Yr, cache = R.forward(p, n_in, nh, n_out, X)
    lr, dY = R.mse(Yr, T, scale)
    gr = R.backward(p, n_in, nh, n_out, cache, dY)
    assert np.max(np.abs(Y - Yr)) <= 1e-4 * max(1.0, np.max(np.abs(Yr)))
    assert abs(loss - lr) <= 1e-4 * abs(lr)
    assert np.max(np.abs(g - gr)) <= 1e-4 * np.max(np.abs(gr))
