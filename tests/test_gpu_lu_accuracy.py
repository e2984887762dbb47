"""getrf on matrices whose factors have an ill-conditioned diagonal block although every multiplier is small:
two nearly dependent columns among 16 neighbours of a dominant diagonal.  LAPACK's pivots are the diagonal, so
nothing but the error of the factors tells how the multipliers were formed.

Bar, for any order of the sums: |A - L U| <= n eps |L| |U| in every element (elimination with each
multiplier and each entry of U rounded once per term).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _factor(As, npdt):
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    n, batch, dt = len(As[0]), len(As), torch.float64 if npdt == np.float64 else torch.float32
    a = H.colmajor((n, n, batch), dt)
    for b in range(batch):
        a[:, :, b] = H.to_device(As[b], dt)
    ipiv = torch.zeros(n * batch, dtype=torch.int32, device="cuda")
    info = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    H.getrf(a, ipiv, info)
    lu = [H.to_host(a[:, :, b]).astype(np.float64) for b in range(batch)]
    return lu, ipiv.cpu().numpy().reshape(batch, n) - 1, info.cpu().numpy()


def _worst(A, lu, eps):
    """max |A - L U| / (eps |L| |U|), A's rows already in pivot order."""
    L, U = np.tril(lu, -1) + np.eye(len(lu)), np.triu(lu)
    return np.max(np.abs(A - L @ U) / (np.abs(L) @ np.abs(U))) / eps


@pytest.mark.parametrize("npdt,gap", [(np.float64, g) for g in (1e-2, 1e-5, 1e-8, 1e-12)] +
                         [(np.float32, g) for g in (1e-2, 1e-3, 1e-5)])
@pytest.mark.parametrize("n,batch", [(81, 1), (192, 9), (1100, 1), (1100, 8)])
def test_nearly_dependent_columns(n, batch, npdt, gap):
    print(f"[case] dependent columns n={n} batch={batch} {npdt.__name__} gap={gap}", flush=True)
    rng = np.random.default_rng(n + batch)
    As = []
    for b in range(batch):
        A = rng.standard_normal((n, n)) / n ** 0.5 + 4.0 * np.eye(n)
        for j in (7, n // 2 // 16 * 16 + 9):  # in the first panel and in a later one
            A[:, j] = A[:, j - 4] + gap * A[:, j]
        As.append(A.astype(npdt))
    lus, pivs, info = _factor(As, npdt)
    for A, lu, piv, inf in zip(As, lus, pivs, info):
        assert inf == 0 and np.array_equal(piv, np.arange(n))
        assert _worst(A.astype(np.float64), lu, np.finfo(npdt).eps) <= n
