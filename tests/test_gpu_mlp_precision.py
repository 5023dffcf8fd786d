"""The weight gradients' sums over the batch: their error against 64 bits, for the operands that
the GPU had, is no larger than that of FP32 sums of 256 rows at a time, the blocks added up."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _blocked(A, B):
    total = np.zeros((A.shape[1], B.shape[1]), np.float32)
    for r0 in range(0, len(A), 256):
        acc = np.zeros_like(total)
        for a, b in zip(A[r0:r0 + 256], B[r0:r0 + 256]):
            acc += a[:, None] * b[None]
        total += acc
    return total


@pytest.mark.parametrize("M", [1500, 8192, 16384, 20000])
def test_sums_over_the_batch(M):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no HIP device visible: GPU tests must run on an MI355X")
    from tonto_amd.mlp import DeviceNet, init_params
    n_in, nh, n_out = 40, 32, 48
    rng = np.random.default_rng(M)
    net = DeviceNet(n_in, nh, n_out, init_params(n_in, nh, n_out, 2))
    X = torch.tensor(rng.standard_normal((M, n_in)).astype(np.float32), device="cuda")
    T = torch.tensor(rng.standard_normal((M, n_out)).astype(np.float32), device="cuda")
    net.loss_and_grad(X, T, 1.0 / (M * n_out))
    ws, ws2, _, dY = (t.cpu().numpy() for t in net._work(M))
    Z1, A1, Z2, A2 = ws[:4 * M * nh].reshape(4, M, nh)
    dZ1, dZ2 = ws2[:2 * M * nh].reshape(2, M, nh)
    g, at = net.g.cpu().numpy(), 0
    for A, B in ((X.cpu().numpy(), dZ1), (A1, dZ2), (A2, dY)):
        m, n = A.shape[1], B.shape[1]
        # the bias gradient as a column of ones
        got = np.vstack([g[at:at + m * n].reshape(m, n), g[at + m * n:at + (m + 1) * n]])
        at += (m + 1) * n
        A = np.hstack([A, np.ones((M, 1), np.float32)])
        exact = A.astype(np.float64).T @ B.astype(np.float64)
        rms = [np.sqrt(np.mean((x - exact) ** 2)) for x in (got, _blocked(A, B))]
        print(f"M={M} {m}x{n}: rms error {rms[0]:.3e}, of blocks of 256 rows {rms[1]:.3e}")
        assert rms[0] <= 1.1 * rms[1]
