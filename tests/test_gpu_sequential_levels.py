"""Sequential sweeps run level by level: the regrouped launches must give what one update
after the other gives.  The reference is the engine's own single-message update
(`update_slot`) applied in order, and the oracle; schedules with repeated slots, partial
schedules and reversed ones have dependences the forest cover does not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _orders(pkg, g, t):
    forest = [t.slot(*e) for e in pkg.forest_cover_edge_sequence(g)]
    rng = np.random.default_rng(3)
    shuffled = list(rng.permutation(t.nports))
    return {"forest": forest, "reversed": forest[::-1], "shuffled": shuffled,
            "repeated": shuffled[:7] * 3 + forest + shuffled[:5], "partial": forest[::3],
            "one": [forest[0]] * 4}


@pytest.mark.parametrize("dtype,D", [("f64", 3), ("f64", 9), ("f32", 4), ("bf16", 3), ("c128", 2)])
def test_levels_match_single_updates(pkg, orc, dtype, D):
    shape = (2, 3) if D > 8 else (4, 5)
    g = pkg.named_grid(shape)
    t = pkg.build_topology(g, D, 2)
    s = pkg.peps.random_sites(t, 12, scale=pkg.peps.peps_scale(2, D))
    if dtype == "c128":
        s = s + 1j * s[::-1]
    m0 = pkg.peps.random_messages(t, 13)
    # FP64: the pair kernel against the generic one, sums in another order; FP32, BF16 and
    # bond dimension 9 run the same kernel on the same inputs either way
    tol = {"f64": 1e-12, "c128": 1e-12}.get(dtype, 0.0) if D <= 8 else 0.0
    for name, order in _orders(pkg, g, t).items():
        print(f"case levels {dtype} D={D} {name}", flush=True)
        with pkg.Engine(t, s, dtype=dtype) as e:
            e.set_messages(m0)
            r = e.run_sequential(order, maxiter=2)
            got = e.messages()
        assert r.sweeps[0] == 2
        with pkg.Engine(t, s, dtype=dtype) as e:
            e.set_messages(m0)
            for q in list(order) * 2:
                e.update_slot(q)
            want = e.messages()
        assert np.max(np.abs(got - want)) <= tol * np.max(np.abs(want))
        if dtype == "f64":
            ref = orc.sweep_sequential(t, s, m0, order)
            ref = orc.sweep_sequential(t, s, ref[0] if isinstance(ref, tuple) else ref, order)
            ref = ref[0] if isinstance(ref, tuple) else ref
            np.testing.assert_allclose(got, ref, rtol=1e-11, atol=1e-14)
