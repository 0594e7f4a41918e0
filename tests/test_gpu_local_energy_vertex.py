"""Local energies with operator matrices on the FP32 dual-number kernels against the generic
kernels (FP64 context, which run one override and operator at a time) and the oracle: physical
dimensions 1..4 (a launch per bra-ket slice offset), non-symmetric operators (bra and ket sides
differ), padded bonds and degrees, vertex or edge terms alone, larger operator blocks.

FP32 contractions of d D^k terms against FP64 at FP32-converged messages: 1e-4 of the largest
gradient entry (the FP32 TFIM gradients are within 1e-6 on the same lattices)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,D,d,terms,ld", [((3, 4), 5, 2, "ve", 2), ((4, 3), 6, 2, "e", 3),
                                                ((3, 3), 8, 2, "v", 2), ((3, 3), 6, 3, "ve", 3),
                                                ((2, 3), 7, 4, "ve", 4), ((1, 4), 6, 2, "ve", 2),
                                                ((3, 3), 5, 1, "ve", 2)])
def test_against_fp64(pkg, orc, shape, D, d, terms, ld):
    print(f"case local vertex {shape} D={D} d={d} {terms} ld={ld}", flush=True)
    t = pkg.build_topology(pkg.named_grid(shape), D, d)
    s = pkg.peps.random_sites(t, 31, scale=pkg.peps.peps_scale(d, D))
    s = s.astype(np.float32).astype(np.float64)
    rng = np.random.default_rng(32)
    ov = rng.standard_normal((t.nv, ld, ld)) if "v" in terms else None
    oa = rng.standard_normal((t.ne, ld, ld)) if "e" in terms else None
    ob = rng.standard_normal((t.ne, ld, ld)) if "e" in terms else None
    out = {}
    for dtype, tol in (("f32", 1e-13), ("f64", 1e-15)):
        with pkg.Engine(t, s, dtype=dtype) as e:
            e.init_messages("identity")
            e.run(maxiter=300, tol=tol)
            assert dtype == "f64" or e.path() == "vertex"
            E0 = e.local_energy(ov, oa, ob)
            E, g, it, res = e.local_energy(ov, oa, ob, grad=True, adj_tol=1e-6, adj_maxiter=300)
            dev = None
            if dtype == "f32":
                dev = e.local_energy(ov, oa, ob, grad=True, adj_tol=1e-6, adj_maxiter=300,
                                     device=True)[1].numpy()
        assert E == E0
        out[dtype] = (E, g, dev)
    E, g, dev = out["f32"]
    Ew, gw, _ = out["f64"]
    # at d = 1 the expectation values do not depend on the tensors: terms of order |O| / |A|,
    # above 1 on these sites, cancel to zero
    scale = max(np.max(np.abs(gw)), 1.0 if d == 1 else 0.0)
    assert np.max(np.abs(g - gw)) < 1e-4 * scale
    np.testing.assert_array_equal(dev, g.astype(np.float32))
    assert abs(E - Ew) < 1e-4 * max(abs(Ew), 1.0)


@pytest.mark.parametrize("shape,D,d", [((4, 4), 5, 2), ((3, 4), 6, 3), ((3, 3), 8, 2), ((1, 4), 6, 2)])
def test_multiples_of_the_identity(pkg, shape, D, d):
    """O_v = c, A_e B_e = c: the energy is c per term and its gradient zero whatever the tensors
    are, so what is left is the rounding of operators, coefficients and sums over slices.  In
    FP64 that is some 1e-15 of c (sums of at most 64 d terms of the same FP32 products above and
    below the fraction; 1e-12 is asserted), with c rounded to FP32 1e-8 of it."""
    print(f"case local identity {shape} D={D} d={d}", flush=True)
    t = pkg.build_topology(pkg.named_grid(shape), D, d)
    s = pkg.peps.random_sites(t, 33, scale=pkg.peps.peps_scale(d, D))
    c = 1000.1
    one = lambda n, x: np.broadcast_to(x * np.eye(d), (n, d, d)).copy()  # noqa: E731
    with pkg.Engine(t, s, dtype="f32") as e:
        e.init_messages("identity")
        e.run(maxiter=300, tol=1e-13)
        assert e.path() == "vertex"
        kw = {"grad": True, "adj_tol": 1e-6, "adj_maxiter": 50}
        Ev, gv, _, _ = e.local_energy(one(t.nv, c), **kw)
        Ee, ge, _, _ = e.local_energy(None, one(t.ne, c), one(t.ne, 1.0), **kw)
        h = np.random.default_rng(34).standard_normal((t.nv, d, d))
        size = np.max(np.abs(e.local_energy(h, **kw)[1])) if d > 1 else 1.0
    assert abs(Ev - c * t.nv) <= 1e-12 * c * t.nv
    assert abs(Ee - c * t.ne) <= 1e-12 * c * t.ne
    assert np.max(np.abs(gv)) <= 1e-10 * c * size
    assert np.max(np.abs(ge)) <= 1e-10 * c * size
