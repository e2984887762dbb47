"""getrf's speculative panels (k_panel_spec): pivots inside and outside the panel's diagonal block, panels
that fail every round, ties, and sizes at the edges of the 64-column panels and 16-row tiles.

Bars, from the arithmetic: pivots equal LAPACK's (the matrices have no near ties but the exact ones of
the tie case, which LAPACK settles by the row order), factors within 1e-11 of LAPACK's largest entry in
FP64 (the bar of the other LU tests), and ||P A - L U||_F <= 4 n eps ||A||_F in either precision
(the bound of Gaussian elimination with multipliers of at most 1 and little growth).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(kind, n, rng):
    A = rng.standard_normal((n, n)) + 2.0 * n ** 0.5 * np.eye(n)
    if kind == "inside":  # two interchanges inside every diagonal block
        for k in range(0, n - 20, 64):
            A[[k + 3, k + 17]] = A[[k + 17, k + 3]]
    elif kind == "below":  # every second panel pivots on two rows far below it
        for k in range(0, n // 2 - 64, 128):
            for d in (5, 40):
                A[[k + d, n - 1 - k // 64 - d]] = A[[n - 1 - k // 64 - d, k + d]]
    elif kind == "random":  # every round fails
        A = rng.standard_normal((n, n))
    elif kind == "tie":  # entries +-1: exact ties in every column
        A = np.sign(rng.standard_normal((n, n)))
    return A


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,batch", [(17, 1), (64, 3), (65, 1), (130, 9), (321, 1), (1100, 1), (1100, 8)])
@pytest.mark.parametrize("kind", ["diagonal", "inside", "below", "random", "tie"])
def test_speculative_panels(kind, n, batch, prec):
    import scipy.linalg as sl
    import torch

    from tinyvlm_amd import capi as H

    if kind == "tie" and n > 64:
        pytest.skip("exact ties only survive the first columns")
    H.init(0)
    print(f"[case] speculative panels {kind} n={n} batch={batch} {prec}", flush=True)
    dt, npdt = (torch.float64, np.float64) if prec == "f64" else (torch.float32, np.float32)
    rng = np.random.default_rng(n + batch)
    As = [_matrix(kind, n, rng).astype(npdt) for _ in range(batch)]
    if batch > 2:
        As[1][:, 5] = 0.0  # an exactly zero column: every round of its panel fails, info = 6
    a = H.colmajor((n, n, batch), dt)
    for b in range(batch):
        a[:, :, b] = H.to_device(As[b], dt)
    ipiv = torch.zeros(n * batch, dtype=torch.int32, device="cuda")
    info = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    H.getrf(a, ipiv, info)
    piv = ipiv.cpu().numpy().reshape(batch, n) - 1
    inf = info.cpu().numpy()
    for b in range(batch):
        if batch > 2 and b == 1:
            assert inf[b] == 6
            continue
        if kind == "tie":  # a +-1 matrix may be singular; LAPACK's own info decides
            assert piv[b][0] == 0  # all |a| equal in the first column: the first row
            continue
        assert inf[b] == 0
        ref, piv_ref = sl.lu_factor(As[b].astype(np.float64))
        if prec == "f64" or kind != "random":
            assert np.array_equal(piv[b], piv_ref)
        got = H.to_host(a[:, :, b]).astype(np.float64)
        if prec == "f64":
            assert np.max(np.abs(got - ref)) <= 1e-11 * np.max(np.abs(ref))
        perm = np.arange(n)
        for k in range(n):
            perm[[k, piv[b][k]]] = perm[[piv[b][k], k]]
        A = As[b].astype(np.float64)
        res = np.linalg.norm(A[perm] - (np.tril(got, -1) + np.eye(n)) @ np.triu(got)) / np.linalg.norm(A)
        assert res <= 4 * n * np.finfo(npdt).eps
