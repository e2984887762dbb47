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


@pytest.mark.parametrize("npdt", [np.float64, np.float32])
@pytest.mark.parametrize("row", [0, 20, 100])
def test_pivot_larger_by_an_ulp(row, npdt):
    """A row whose entry exceeds the diagonal's by one ulp is the pivot, also where their quotient rounds to 1
    (row 0: an exact tie instead, which the first row wins)."""
    print(f"[case] pivot by an ulp row={row} {npdt.__name__}", flush=True)
    n = 130
    rng = np.random.default_rng(row)
    d = rng.uniform(1.0, 2.0, 4096).astype(npdt)
    d = d[np.nextafter(d, npdt(3)) * (npdt(1) / d) <= 1][:8]
    assert len(d) == 8
    As = []
    for v in d:
        A = (rng.standard_normal((n, n)) / n + 4.0 * np.eye(n)).astype(npdt)
        A[0, 0], A[row if row else 100, 0] = v, -(np.nextafter(v, npdt(3)) if row else v)
        As.append(A)
    _, pivs, info = _factor(As, npdt)
    assert np.all(info == 0)
    assert np.array_equal(pivs[:, 0], np.full(8, row))


@pytest.mark.parametrize("npdt", [np.float64, np.float32])
@pytest.mark.parametrize("n,batch", [(70, 1), (192, 1), (192, 8), (1200, 1)])
def test_growing_inverse_of_l(n, batch, npdt):
    """U12 for panels whose L11 has diagonal blocks of large inverse (-0.97 below the diagonal): rows and columns
    of the first panel's U12, where every sum has at most 16 terms and one correction as many again."""
    print(f"[case] growing inverse n={n} batch={batch} {npdt.__name__}", flush=True)
    rng = np.random.default_rng(n)
    As = []
    for b in range(batch):
        L = np.eye(n)
        for k in range(0, 64, 16):
            L[k:k + 16, k:k + 16] -= 0.97 * np.tril(np.ones((16, 16)), -1)
        U = np.eye(n)
        U[:64, 64:] = rng.uniform(-1.0, 1.0, (64, n - 64))
        As.append((L @ U).astype(npdt))
    lus, pivs, info = _factor(As, npdt)
    for A, lu, piv, inf in zip(As, lus, pivs, info):
        assert inf == 0 and np.array_equal(piv, np.arange(n))
        L, U = np.tril(lu, -1) + np.eye(n), np.triu(lu)
        err = np.abs(A - L @ U)[:64, 64:] / (np.abs(L) @ np.abs(U))[:64, 64:]
        assert np.max(err) <= 4 * 16 * np.finfo(npdt).eps


@pytest.mark.parametrize("npdt", [np.float64, np.float32])
@pytest.mark.parametrize("n,batch", [(32, 3), (33, 3), (40, 300), (49, 300), (65, 2), (128, 2), (129, 2), (193, 1), (257, 9)])
def test_no_dominant_diagonal(n, batch, npdt):
    """Matrices whose pivots lie anywhere, at the sizes where the rounds of a panel begin, take all rows as
    candidates, or give up: LAPACK's pivots (FP64; FP32 sums may order near ties otherwise) and factors."""
    import scipy.linalg as sl

    print(f"[case] no dominant diagonal n={n} batch={batch} {npdt.__name__}", flush=True)
    rng = np.random.default_rng(n)
    As = [rng.standard_normal((n, n)).astype(npdt) for _ in range(batch)]
    lus, pivs, info = _factor(As, npdt)
    for b in range(0, batch, max(1, batch // 7)):
        A, lu, piv = As[b].astype(np.float64), lus[b], pivs[b]
        assert info[b] == 0
        if npdt == np.float64:
            assert np.array_equal(piv, sl.lu_factor(A)[1])
        assert np.max(np.abs(np.tril(lu, -1))) <= 1 + 4 * np.finfo(npdt).eps
        for k in range(n):
            A[[k, piv[k]]] = A[[piv[k], k]]
        assert _worst(A, lu, np.finfo(npdt).eps) <= n


def test_scratch_of_a_large_batch_of_small_matrices():
    """65535 FP32 matrices of 16 x 16 (67 MB): what the factorisation keeps is its interchange lists (2056 bytes a
    matrix, with a quarter more than asked for), not room for panels that these matrices do not have."""
    import torch

    from tinyvlm_amd import capi as H
    from tinyvlm_amd.serve import stream_create, stream_destroy

    H.init(0)
    n, batch = 16, 65535
    print(f"[case] scratch n={n} batch={batch}", flush=True)
    a = torch.randn(batch, n, n, device="cuda").permute(2, 1, 0)
    ipiv = torch.zeros(n * batch, dtype=torch.int32, device="cuda")
    info = torch.full((batch,), -1, dtype=torch.int32, device="cuda")
    st = stream_create()  # a stream without any scratch yet
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    H.getrf(a, ipiv, info, stream=st)
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    stream_destroy(st)
    assert info.cpu().abs().max() == 0
    assert used <= 1.5 * 2056 * batch
