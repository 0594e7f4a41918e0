"""Reductions over whole networks: the stopping rule (folded into the small-bond sweep, on many
workgroups, on one), the log-norm on one and on many workgroups, vertex scalars of every FP32
bucket, edge scalars.

Networks of more than 4 x 4096 message slots take the many-workgroup reduction; of more than
2 x 4096 terms the many-workgroup log-norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(pkg, shape, D, d=2, seed=1, hexa=False):
    g = pkg.heavy_hex_lattice(*shape) if hexa else pkg.named_grid(shape)
    t = pkg.build_topology(g, D, d)
    return t, pkg.peps.random_sites(t, seed, scale=pkg.peps.peps_scale(d, D))


@pytest.mark.parametrize("shape,D,d", [((1, 2), 2, 2), ((3, 3), 2, 3), ((9, 7), 3, 2), ((5, 5), 4, 4),
                                       ((70, 65), 2, 2), ((66, 66), 3, 2), ((1, 300), 4, 1)])
def test_folded_small_bond_run(pkg, shape, D, d):
    print(f"case small-bond fold {shape} D={D} d={d}", flush=True)
    t, s = _net(pkg, shape, D, d)
    for kw in ({"maxiter": 50, "tol": 1e-7}, {"maxiter": 50, "tol": 1e-4, "criterion": "maxabs"},
               {"maxiter": 5, "tol": 1e-9}, {"maxiter": 19}):
        got = []
        for fold, graph in ((1, True), (0, True), (1, False)):
            with pkg.Engine(t, s, dtype="f32") as e:
                e.set_option("fold_bookkeeping", fold)
                for _ in range(2):
                    e.init_messages("identity")
                    r = e.run(use_graph=graph, **kw)
                fid, mab = e.residuals()
                got.append((e.messages(), r.sweeps, r.delta, r.at_iteration))
            if r.at_iteration[0] < 0:  # the last sweep ran: its residuals are the slots' own
                res = mab if kw.get("criterion") == "maxabs" else fid
                assert r.delta[0] == max(0.0, res.max())
        for x in got[1:]:
            for u, v in zip(got[0], x):
                np.testing.assert_array_equal(u, v)


def test_batch_with_a_large_network(pkg):
    """Two networks, one above the many-workgroup line: each stops where it stops alone."""
    print("case batch reduction", flush=True)
    parts = [_net(pkg, (70, 65), 2, seed=3), _net(pkg, (3, 3), 3, seed=4)]
    b = pkg.concat_topologies([t for t, _ in parts])
    with pkg.Engine(b, np.concatenate([s for _, s in parts]), dtype="f32") as e:
        e.init_messages("identity")
        r = e.run(maxiter=80, tol=1e-8)
        m, ln = e.messages(), e.lognorms()
    off = 0
    for i, (t, s) in enumerate(parts):
        with pkg.Engine(t, s, dtype="f32") as e:
            e.init_messages("identity")
            q = e.run(maxiter=80, tol=1e-8)
            assert (q.sweeps[0], q.at_iteration[0], q.delta[0]) == (
                r.sweeps[i], r.at_iteration[i], r.delta[i])
            n = int(t.msg_off[-1])
            np.testing.assert_array_equal(e.messages(), m[off:off + n])
            off += n
            # the same terms in another order, compensated
            assert ln[i] == pytest.approx(e.lognorm(), rel=1e-14)


BUCKETS = [((4, 5), 1, 2, False), ((4, 5), 2, 2, False), ((5, 4), 2, 1, False), ((4, 4), 3, 3, False),
           ((4, 5), 4, 2, False), ((4, 4), 6, 2, False), ((3, 6), 8, 2, True), ((3, 4), 10, 2, False),
           ((3, 4), 12, 2, False), ((2, 5), 11, 2, True), ((1, 6), 3, 2, False)]


@pytest.mark.parametrize("shape,D,d,hexa", BUCKETS)
def test_fp32_scalars(pkg, orc, shape, D, d, hexa):
    """Z_v is a sum of n = d D^(2k) positive-dominated products in FP32: 1e-5 relative, as the
    generic FP32 kernel's."""
    print(f"case scalars {shape} D={D} d={d} hex={hexa}", flush=True)
    t, s = _net(pkg, shape, D, d, seed=5, hexa=hexa)
    m = pkg.peps.random_messages(t, 6)
    with pkg.Engine(t, s, dtype="f32") as e:
        e.set_messages(m)
        got, ze, ln, after = e.vertex_scalars(), e.edge_scalars(), e.lognorms()[0], e.messages()
    m32 = m.astype(np.float32).astype(np.float64)
    np.testing.assert_array_equal(after, m32)
    want = orc.vertex_scalars(t, s, m32)
    scale = orc.vertex_scalars(t, np.abs(s), m32)  # cancellation: against the absolute sums
    assert np.max(np.abs(got - want) / scale) < 1e-5
    np.testing.assert_allclose(ze, orc.edge_scalars(t, m32), rtol=1e-12)
    # the log-norm of the engine's own terms, its imaginary part counting the negative ones
    z = np.sum(np.log(np.abs(got))) - np.sum(np.log(np.abs(ze)))
    assert np.real(ln) == pytest.approx(z, rel=1e-12, abs=1e-12)
    assert np.imag(ln) == pytest.approx(np.pi * (np.sum(got < 0) - np.sum(ze < 0)))


def test_fp32_scalars_of_a_mixed_batch(pkg, orc):
    """Every FP32 bucket in one engine, beside an isolated vertex's network."""
    print("case scalars batch", flush=True)
    nets = [_net(pkg, sh, D, seed=7 + i, hexa=h) for i, (sh, D, h) in enumerate(
        [((3, 3), 2, False), ((3, 4), 4, False), ((3, 3), 6, False), ((2, 4), 8, True),
         ((3, 3), 10, False), ((3, 3), 12, False), ((2, 4), 12, True)])]
    one = pkg.build_topology(pkg.NamedGraph(vertices=["a"], edges=[]), 2, 2)
    for extra in ([], [(one, np.array([0.5, -2.0]))]):
        all_ = nets + extra
        b, s = pkg.concat_topologies([t for t, _ in all_]), np.concatenate([s for _, s in all_])
        with pkg.Engine(b, s, dtype="f32") as e:
            e.init_messages("identity")
            e.run(maxiter=3)
            m = e.messages()
            got = e.vertex_scalars()
        np.testing.assert_allclose(got, orc.vertex_scalars(b, s, m), rtol=1e-5)


@pytest.mark.parametrize("dtype", ["f64", "c128"])
@pytest.mark.parametrize("shape,D", [((1, 2), 2), ((3, 4), 3), ((3, 3), 5), ((64, 40), 2)])
def test_fp64_lognorm(pkg, orc, shape, D, dtype):
    from oracle import complex_oracle as co
    print(f"case lognorm {dtype} {shape} D={D}", flush=True)
    t, s = _net(pkg, shape, D, seed=9)
    m = pkg.peps.random_messages(t, 10)
    if dtype == "c128":
        s, m = s + 1j * s[::-1], m + 0.3j * m[::-1]
        if t.nv > 100:
            pytest.skip("the complex restatement loops in Python")
    with pkg.Engine(t, s, dtype=dtype) as e:
        e.set_messages(m)
        zv, ln = e.vertex_scalars(), e.lognorms()[0]
    if dtype == "f64":
        want = orc.vertex_scalars(t, s, m)
        scale = orc.vertex_scalars(t, np.abs(s), m)
        assert np.max(np.abs(zv - want) / scale) < 1e-13
        assert np.real(ln) == pytest.approx(np.real(orc.bethe_free_energy(t, s, m)), rel=1e-11)
    else:
        want = np.asarray(co.vertex_scalars(t, s, m))
        np.testing.assert_allclose(zv, want, rtol=1e-11, atol=1e-12 * np.max(np.abs(want)))
        ref = co.bethe_free_energy(t, s, m)
        assert ln.real == pytest.approx(ref.real, rel=1e-11)
        assert ln.imag == pytest.approx(ref.imag, abs=1e-9)
