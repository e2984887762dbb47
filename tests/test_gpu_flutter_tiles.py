"""The flutter sweep's circulation product (k_fl_gemm) at the edges of its 16 x 16 tiles and 512-column
blocks: panel counts and airspeed counts that are no multiple of the tile, a column block of a few
columns, a wave without columns.  Against the oracle to the sweep's bar (1e-9 of each result's scale),
and each airspeed alone bit for bit as in the batch.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C5 = dict(mu=20.0, omega=0.5, a_h=-0.3, x_a=0.25, r_a=0.5)


@pytest.mark.parametrize("ns,nc,n_air", [(1, 2, 1), (5, 3, 17), (23, 23, 18), (33, 16, 16)])
def test_flutter_product_tiles(oracle, ns, nc, n_air):
    from oracle import two_dof as O

    from tinyvlm_amd import capi as H
    from tinyvlm_amd import flutter_plan as F

    H.init(0)
    print(f"[case] flutter tiles {ns}x{nc} {n_air} airspeeds", flush=True)
    v = oracle.rectangular_wing(ns, nc, chord=1.0, half_span=3.0)
    air = list(np.linspace(0.5, 2.0, n_air))
    steps, R = 3, 10

    def run(a):
        plan = F.FlutterPlan(v, a, F.params(**C5), wake_rows=R, max_steps=steps)
        plan.run(steps)
        r = plan.results()
        plan.close()
        return r

    res = run(air)
    for b in {0, n_air // 2, n_air - 1}:
        one = run([air[b]])
        dt = one["dt"]
        o = O.run([(v, True)], O.Vars(U_a=air[b], **C5), t_final_nd=(steps + 2) * dt + 0.5 * dt, dtype=np.float64,
                  wake_rows=R)
        assert np.array_equal(res["iters"][:, b], o["iters"])
        for key in ("u", "v", "F"):
            assert np.array_equal(res[key][:, b, :], one[key][:, 0, :]), key
            ref = o[key]
            assert np.max(np.abs(res[key][:, b, :].T - ref)) <= 1e-9 * max(np.max(np.abs(ref)), 1e-30), key
