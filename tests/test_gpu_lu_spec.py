"""getrf's speculative panels (k_panel_spec): pivots inside and outside the panel's diagonal block, panels
that fail every round, ties, and sizes at the edges of the 64-column panels and 16-row tiles.

Bars, from the arithmetic: pivots equal LAPACK's (the matrices have no near ties but the exact ones of
the tie case, which LAPACK settles by the row order: there up to the first column whose pivot is no power of two,
before which nothing rounds), factors within 1e-11 of LAPACK's largest entry in
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


SIZES = [(17, 1), (64, 3), (65, 1), (130, 9), (321, 1), (1100, 1), (1100, 8)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind,n,batch", [(k, *s) for k in ("diagonal", "inside", "below", "random") for s in SIZES] +
                         [("tie", n, batch) for n, batch in SIZES if n <= 130])
def test_speculative_panels(kind, n, batch, prec):
    import torch
    from scipy.linalg import lapack

    from tinyvlm_amd import capi as H

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
        ref, piv_ref, info_ref = lapack.dgetrf(As[b].astype(np.float64))
        assert info_ref == (6 if batch > 2 and b == 1 else 0)
        assert inf[b] == info_ref
        got = H.to_host(a[:, :, b]).astype(np.float64)
        if kind == "tie":
            mantissas = np.abs(np.frexp(np.diag(ref))[0])
            exact = int(np.argmax((mantissas != 0.5) & (mantissas != 0.0)))  # the first pivot that is no power of two
            assert exact >= 3 and np.array_equal(piv[b][:exact + 1], piv_ref[:exact + 1])
        else:
            if prec == "f64" or kind != "random":
                assert np.array_equal(piv[b], piv_ref)
            if prec == "f64":
                assert np.max(np.abs(got - ref)) <= 1e-11 * np.max(np.abs(ref))
        perm = np.arange(n)
        for k in range(n):
            perm[[k, piv[b][k]]] = perm[[piv[b][k], k]]
        A = As[b].astype(np.float64)
        res = np.linalg.norm(A[perm] - (np.tril(got, -1) + np.eye(n)) @ np.triu(got)) / np.linalg.norm(A)
        assert res <= 4 * n * np.finfo(npdt).eps
