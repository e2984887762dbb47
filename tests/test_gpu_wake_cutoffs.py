"""The wake lattice's walk without cutoffs and its second walk with them (lattice_chunk): receivers on a
wake vertex, on a segment, on its extension and just above the cutoff distance, inputs that are not
finite and wings of small chord, against the exact form.

Bar: 2e-12 of the largest entry, the bar of the lattice form against the exact one (its reciprocals'
few ulp, amplified near the extension of a segment).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,ns", [(1, 1), (2, 9), (5, 40), (30, 65)])
@pytest.mark.parametrize("bad", [None, "nan", "inf", "1e39"])
def test_lattice_near_cutoffs(rows, ns, bad):
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    print(f"[case] lattice cutoffs rows={rows} ns={ns} {bad}", flush=True)
    rng = np.random.default_rng(rows + ns)
    ys, xs = np.linspace(0.0, 2.0, ns + 1), np.linspace(0.0, 0.1 * rows, rows + 1)
    w = np.zeros((ns + 1, rows + 1, 4))
    w[:, :, 0], w[:, :, 1], w[:, :, 3] = xs[None, :], ys[:, None], 1.0
    w[:, :, 2] = 0.05 * np.sin(xs)[None, :]
    g = rng.standard_normal((ns, rows))
    c = rng.standard_normal((70, 1, 3)) * [0.3, 0.8, 0.2] + [0.05 * rows, 1.0, 0.3]
    a, b, d = w[0, 0, :3], w[1, 0, :3], w[0, 1, :3]
    for k, p in enumerate((a, b, 0.5 * (a + b), 0.5 * (a + d), b + 3 * (b - a), d + 2 * (d - a), 0.5 * (a + b) + [0, 0, 1e-7],
                           0.5 * (a + b) + [0, 0, 1e-3], a + [1e-12, 0, 0])):
        c[7 * k, 0] = p
    n = rng.standard_normal(c.shape)
    # surface 0 sheds the wake (its receivers stand clear of it), surface 1 holds the receivers above
    c0 = np.zeros((ns, 1, 3)) + [-0.3, 1.0, 0.4]
    wakes, gammas = [w, np.zeros((71, rows + 1, 4))], [g, np.zeros((70, rows))]
    if bad:
        w[-1, -1, 2] = float(bad)
    t = lambda x: H.to_device(x, torch.float64)  # noqa: E731
    out = []
    for f in (H.rhs_assemble_wake_influence, H.rhs_assemble_wake_influence_lattice):
        rhs = torch.zeros(ns + 70, dtype=torch.float64, device="cuda")
        f(rhs, [t(x) for x in gammas], [t(c0), t(c)], [t(c0), t(n)], [t(x) for x in wakes], [True, False], rows)
        out.append(rhs.cpu().numpy())
    # a vertex that is not finite reaches every receiver, in either form; one at 1e39 overflows the walk without
    # cutoffs alone, whose second walk then gives the value
    finite = np.full(ns + 70, bad not in ("nan", "inf"))
    assert np.array_equal(np.isfinite(out[0]), finite) and np.array_equal(np.isfinite(out[1]), finite)
    out = [x[finite] for x in out]
    if not len(out[0]):
        return
    assert np.max(np.abs(out[0] - out[1])) <= 2e-12 * np.max(np.abs(out[0]))


@pytest.mark.parametrize("chord", [1.0, 0.05, 0.02, 0.005])
@pytest.mark.parametrize("rows,ns,nc", [(1, 5, 3), (7, 40, 10), (30, 65, 4)])
def test_small_wing_at_the_cutoffs(rows, ns, nc, chord):
    """A wing right in front of its wake, down to chords at which the absolute cutoffs meet most of its
    segments: tiles walked without the cutoffs, twice, and with them from the start."""
    import torch

    from tinyvlm_amd import capi as H

    H.init(0)
    print(f"[case] lattice columns chord={chord} rows={rows} ns={ns} nc={nc}", flush=True)
    rng = np.random.default_rng(ns)
    d = chord / nc
    ys = np.linspace(0.0, 2.0 * chord, ns + 1)
    w = np.zeros((ns + 1, rows + 1, 4))
    w[:, :, 0], w[:, :, 1], w[:, :, 3] = chord + d * np.arange(rows + 1)[None, :], ys[:, None], 1.0
    w[:, :, 2] = 0.1 * chord * np.sin(np.arange(rows + 1))[None, :]
    g = rng.standard_normal((ns, rows))
    c = np.zeros((ns, nc, 3))
    c[:, :, 0], c[:, :, 1] = d * (np.arange(nc) + 0.75)[None, :], 0.5 * (ys[1:] + ys[:-1])[:, None]
    n = np.zeros((ns, nc, 3)) + [0.1, 0.05, 1.0]
    t = lambda x: [H.to_device(x, torch.float64)]  # noqa: E731
    out = []
    for f in (H.rhs_assemble_wake_influence, H.rhs_assemble_wake_influence_lattice):
        rhs = torch.zeros(ns * nc, dtype=torch.float64, device="cuda")
        f(rhs, t(g), t(c), t(n), t(w), [True], rows)
        out.append(rhs.cpu().numpy())
    assert np.all(np.isfinite(out[1]))
    assert np.max(np.abs(out[0] - out[1])) <= 2e-12 * np.max(np.abs(out[0]))
