"""The steady plan's per-request kernels (geometry and rhs; circulation differences, forces and coefficient
sums) at the edges of their grids: one panel, several ragged surfaces, more panels than the post kernel has
threads; a partial batch, and results that do not depend on the batch they were computed in.

Bars as for the plan's full-size meshes: plain FP64 within 1e-12 of the oracle's VLM run, served within 1e-10.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,bar", [(0, 1e-12), (1, 1e-10)])
@pytest.mark.parametrize("dims", [[(1, 1)], [(3, 17), (1, 1), (5, 2)], [(70, 16), (2, 3)]])
def test_batched_requests(oracle, dims, mode, bar):
    from tinyvlm_amd import capi as H
    from tinyvlm_amd.steady_plan import SteadyPlan

    H.init(0)
    print(f"[case] steady batch {dims} mode {mode}", flush=True)
    meshes = []
    for k, (ns, nc) in enumerate(dims):
        v = oracle.rectangular_wing(ns, nc, chord=1.0 + 0.2 * k, half_span=2.0, sweep_deg=10.0)
        v[:, :, 1] += 4.5 * k
        meshes.append(v)
    alphas = [0.03, -0.05, 0.1]
    p = SteadyPlan(meshes, 4, mode=mode)
    p.solve(alphas)
    r = p.results()
    for b, a in enumerate(alphas):
        g, cl, cm, _ = oracle.vlm_run(meshes, a)
        assert np.max(np.abs(r["gamma"][b] - g)) <= bar * np.max(np.abs(g))
        assert abs(r["cl"][b] - cl) <= bar * abs(cl)
        assert np.max(np.abs(r["cm"][b] - cm)) <= bar * np.max(np.abs(cm))
    p.solve(alphas[1:2])
    one = p.results()
    p.close()
    assert np.array_equal(one["gamma"][0], r["gamma"][1]) and one["cl"][0] == r["cl"][1]
