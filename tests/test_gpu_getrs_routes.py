"""getrs on either side of the lines between its routes (a work-group per right-hand side, steps of 256 rows,
steps of 64 rows, products over many right-hand sides) and at the edges of the 64-row blocks each of them walks.

Bar: normwise backward error |b - A x| / (|A| |x|) below 4 n eps, the bar of the other LU tests.  Where the route
does not depend on the number of matrices a right-hand side solved in a batch equals the same one alone.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,nrhs,batch", [
    (257, 1, 3), (320, 2, 2), (321, 2, 2), (577, 64, 2), (641, 65, 2), (641, 200, 1), (513, 512, 1), (897, 200, 1),
    (700, 11, 24), (1000, 8, 32), (1024, 200, 1), (1025, 257, 2),   # a work-group per right-hand side, and beside it
    (1400, 96, 2), (2049, 64, 2), (3072, 126, 1), (4100, 32, 1),     # steps of 64 rows
    (300, 3500, 1), (900, 1020, 2), (2049, 450, 1)])                 # products
def test_getrs_routes(prec, n, nrhs, batch):
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    print(f"[case] getrs routes n={n} nrhs={nrhs} batch={batch} {prec}", flush=True)
    dt, eps = (torch.float64, 2.3e-16) if prec == "f64" else (torch.float32, 1.2e-7)
    g = torch.Generator(device="cuda").manual_seed(n + nrhs)
    A = torch.randn(batch, n, n + 3, generator=g, dtype=dt, device="cuda")  # column-major, leading dimension n + 3
    B = torch.randn(batch, nrhs, n + 5, generator=g, dtype=dt, device="cuda")
    a, x = A.clone().permute(2, 1, 0)[:n], B.clone().permute(2, 1, 0)[:n]
    ipiv = torch.zeros(n * batch, dtype=torch.int32, device="cuda")
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    H.getrf(a, ipiv, info)
    H.getrs(a, ipiv, x)
    assert (info == 0).all()
    for b in range(batch):
        Ab, Bb, Xb = (t.t().to(torch.float64).contiguous() for t in (A[b][:, :n], B[b][:, :n], x[:, :, b].t()))
        res = float(torch.linalg.norm(Ab @ Xb - Bb) / (torch.linalg.norm(Ab) * torch.linalg.norm(Xb)))
        assert res < 4 * n * eps, res
    if batch < 8:
        one = B[batch - 1:].clone().permute(2, 1, 0)[:n]
        H.getrs(a[:, :, batch - 1:], ipiv[(batch - 1) * n:], one)
        assert torch.equal(one[:, :, 0], x[:, :, batch - 1])
