"""getrs at the edges of its 64-row blocks and 256-row steps, on one work-group, step by step, and with many
right-hand sides (products on the matrix cores), single and batched, with padded leading dimensions.

Bar: normwise backward error |b - A x| / (|A| |x|) below 4 n eps, the bar of the LU tests; a right-hand side
solved in a batch of matrices equals the same one solved alone, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (15, 2), (64, 3), (65, 1), (200, 70), (256, 1), (257, 2), (320, 1), (513, 3),
                                    (600, 11), (1025, 1), (2048, 2), (2049, 1), (300, 1800), (1100, 481), (257, 2051)])
def test_getrs_steps(prec, n, nrhs):
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    print(f"[case] getrs n={n} nrhs={nrhs} {prec}", flush=True)
    dt, eps = (torch.float64, 2.3e-16) if prec == "f64" else (torch.float32, 1.2e-7)
    rng = np.random.default_rng(7 * n + nrhs)
    batch = 2
    As = [rng.standard_normal((n, n)) for _ in range(batch)]
    Bs = [rng.standard_normal((n, nrhs)) for _ in range(batch)]
    a = H.colmajor((n + 3, n, batch), dt)[:n]
    x = H.colmajor((n + 5, nrhs, batch), dt)[:n]
    for b in range(batch):
        a[:, :, b] = H.to_device(As[b], dt)
        x[:, :, b] = H.to_device(Bs[b], dt)
    ipiv = torch.zeros(n * batch, dtype=torch.int32, device="cuda")
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    H.getrf(a, ipiv, info)
    H.getrs(a, ipiv, x)
    assert (info == 0).all()
    for b in range(batch):
        A = H.to_device(As[b], dt).to(torch.float64)
        B = H.to_device(Bs[b], dt).to(torch.float64)
        X = x[:, :, b].to(torch.float64)
        res = float(torch.linalg.norm(A @ X - B) / (torch.linalg.norm(A) * torch.linalg.norm(X)))
        assert res < 4 * n * eps, res
    alone = H.colmajor((n, nrhs), dt)
    alone[:] = H.to_device(Bs[1], dt)
    H.getrs(a[:, :, 1], ipiv[n:], alone)
    assert torch.equal(alone, x[:, :, 1])
