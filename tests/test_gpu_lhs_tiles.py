"""lhs_assemble over its tile shapes (lhs_tile_shape) and wake rows: edges of the row and span tiles, one
and several wake rows, the core model, and every precision form, against the oracle.

Bars: FP64 exact and seeded within 1e-12 of the largest entry (each entry sums eight terms of at most
about a hundred times its size, each good to a few ulp); FP32 no worse than 3x the FP32 oracle's own
error against FP64 on the same inputs (the bar of the FP32 wake tests).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,nc", [(1, 1), (1, 5), (5, 1), (17, 9), (65, 3), (33, 21), (130, 7)])
@pytest.mark.parametrize("iteration,sigma", [(0, 0.0), (1, 0.0), (6, 0.0), (1, 1e-3)])
def test_lhs_tile_shapes(oracle, ns, nc, iteration, sigma):
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    print(f"[case] lhs tiles {ns}x{nc} it={iteration} sigma={sigma}", flush=True)
    rng = np.random.default_rng(100 * ns + nc)
    v = oracle.rectangular_wing(ns, nc, chord=1.0, half_span=3.0, sweep_deg=20.0)
    v[:, :, 2] += 0.02 * rng.standard_normal(v.shape[:2])
    w = np.zeros((ns + 1, 8, 4), order="F")
    for r in range(8):
        w[:, 7 - r] = v[:, -1] + [0.3 * r, 0.0, 0.02 * r, 0.0]

    def surf(dtype):
        a, b = (np.asfortranarray(x.astype(np.float32).astype(dtype)) for x in (v, w))
        s = oracle.Surface(verts=a, verts_wake=b)
        oracle.mesh_metrics(0.05, [s])
        return s

    def gpu(s, dt, f):
        lhs = H.colmajor((ns * nc, ns * nc), dt)
        f(lhs, *[[H.to_device(x, dt)] for x in (s.colloc, s.normals, s.verts, s.verts_wake)], iteration)
        return H.to_host(lhs)

    s64 = surf(np.float64)
    ref = oracle.lhs_assemble([s64], iteration, sigma=sigma)
    top = np.max(np.abs(ref))
    got = gpu(s64, torch.float64, lambda *a: H.lhs_assemble(*a, sigma=sigma))
    assert np.max(np.abs(got - ref)) <= 1e-12 * top
    if sigma == 0.0:
        assert np.max(np.abs(gpu(s64, torch.float64, H.lhs_assemble_seeded) - ref)) <= 1e-12 * top
    s32 = surf(np.float32)
    up = oracle.Surface(verts=s32.verts.astype(np.float64), verts_wake=s32.verts_wake.astype(np.float64))
    up.colloc, up.normals = (np.asfortranarray(x.astype(np.float64)) for x in (s32.colloc, s32.normals))
    ref32 = oracle.lhs_assemble([up], iteration, sigma=sigma)
    e_orc = np.linalg.norm(oracle.lhs_assemble([s32], iteration, sigma=sigma) - ref32) / np.linalg.norm(ref32)
    e_gpu = np.linalg.norm(gpu(s32, torch.float32, lambda *a: H.lhs_assemble(*a, sigma=sigma)) - ref32) / np.linalg.norm(ref32)
    assert e_gpu <= max(3 * e_orc, 1e-6)
