"""getrf of matrices tall enough to be updated once per group of panels: sizes that end inside a group's reach
(a last group of ragged rows and columns below it), single and batched, against LAPACK.

Bars as for the other LU tests: LAPACK's pivots in FP64; normwise backward error of a solve below 4 n eps.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(6271, 1), (6272, 1), (6733, 2)])
def test_getrf_panel_groups(prec, n, batch):
    import scipy.linalg as sl
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    print(f"[case] getrf groups n={n} batch={batch} {prec}", flush=True)
    dt, eps = (torch.float64, 2.3e-16) if prec == "f64" else (torch.float32, 1.2e-7)
    rng = np.random.default_rng(n)
    As = [rng.standard_normal((n, n)) for _ in range(batch)]
    a = H.colmajor((n, n, batch), dt)
    x = H.colmajor((n, 1, batch), dt)
    b = rng.standard_normal((n, 1))
    for k in range(batch):
        a[:, :, k] = H.to_device(As[k], dt)
        x[:, :, k] = H.to_device(b, dt)
    ipiv = torch.zeros(n * batch, dtype=torch.int32, device="cuda")
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    H.getrf(a, ipiv, info)
    H.getrs(a, ipiv, x)
    assert (info == 0).all()
    for k in range(batch):
        X = x[:, :, k].to(torch.float64).cpu().numpy()
        res = np.linalg.norm(As[k] @ X - b) / (np.linalg.norm(As[k]) * np.linalg.norm(X))
        assert res < 4 * n * eps
    if prec == "f64":
        piv = ipiv.cpu().numpy().reshape(batch, n)[-1] - 1
        assert np.array_equal(piv, sl.lu_factor(As[-1], overwrite_a=True)[1])
