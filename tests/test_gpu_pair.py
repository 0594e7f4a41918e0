"""The pair-environment sweep kernel (csrc/pair.hip) of FP64 and complex contexts against the
oracle: one Jacobi sweep from random non-symmetric messages, at every degree 0..4, at pair
sides around the 16-wide tiles (1, 4, 9, 15, 16, 18, 25, 32, 49, 64), several physical
dimensions (slices staged in chunks), vertices it does not take, and the stopping rule folded
into it.

Tolerance: an entry is a sum of at most n = d D^(k+1) <= 4 * 8^5 products of five factors; the
inputs are of one sign in the messages and random in the sites, so the rounding error stays
near sqrt(n) eps of the largest entry, 1e-13; 1e-12 is asserted."""
import numpy as np
import pytest

from oracle import complex_oracle as co

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(b))) / np.max(np.abs(b)))


def _grid_dims(pkg, shape, dims):
    g = pkg.named_grid(shape)
    return g, {e: dims[i % len(dims)] for i, e in enumerate(g.edges())}


CASES = [  # lattice shape, bond dimensions (cycled over the edges), physical dimension
    ((1, 2), (3,), 2), ((1, 5), (8,), 2), ((2, 2), (2,), 2), ((3, 4), (1,), 2), ((4, 4), (2,), 3),
    ((5, 4), (3,), 2), ((4, 5), (4,), 2), ((4, 4), (4,), 5), ((5, 5), (5,), 2), ((4, 4), (6,), 1),
    ((3, 4), (7,), 2), ((4, 4), (8,), 2), ((3, 3), (8,), 4), ((5, 5), (1, 2, 3, 5, 8), 2),
    ((4, 5), (3, 5, 6), 2), ((4, 4), (2, 9, 3), 2), ((4, 4), (2, 8, 4, 4), 3),
]


@pytest.mark.parametrize("shape,dims,d", CASES)
def test_one_sweep_fp64(pkg, orc, shape, dims, d):
    print(f"case pair fp64 {shape} {dims} d={d}", flush=True)
    g, bond = _grid_dims(pkg, shape, dims)
    t = pkg.build_topology(g, bond, d)
    s = pkg.peps.random_sites(t, 5, scale=pkg.peps.peps_scale(d, max(dims)))
    m = pkg.peps.random_messages(t, 6)
    want, fid, mab = orc.sweep_jacobi(t, s, m)
    with pkg.Engine(t, s, dtype="f64") as e:
        e.set_option("vertex_bond_mask", 0)  # bond dimensions 6..8 too, without the mask's choice
        e.set_messages(m)
        e.sweep()
        got = e.messages()
        gfid, gmab = e.residuals()
    np.testing.assert_allclose(got, want, rtol=1e-12, atol=1e-15 * np.max(np.abs(want)))
    np.testing.assert_allclose(gfid, fid, atol=1e-12)
    np.testing.assert_allclose(gmab, mab, rtol=1e-9, atol=1e-15)


@pytest.mark.parametrize("shape,dims,d", [((2, 2), (2,), 2), ((4, 3), (4,), 3), ((3, 4), (5,), 2),
                                          ((3, 3), (1, 3, 5), 1), ((3, 3), (2, 6), 2)])
def test_one_sweep_complex(pkg, shape, dims, d):
    print(f"case pair c128 {shape} {dims} d={d}", flush=True)
    g, bond = _grid_dims(pkg, shape, dims)
    t = pkg.build_topology(g, bond, d)
    rng = np.random.default_rng(7)
    cx = lambda n: rng.standard_normal(n) + 1j * rng.standard_normal(n)  # noqa: E731
    s, m = cx(int(t.site_off[-1])) / max(dims) ** 2, cx(int(t.msg_off[-1]))
    with pkg.Engine(t, s, dtype="c128") as e:
        e.set_messages(m)
        e.sweep()
        got = e.messages()
    assert _rel(got, co.sweep_jacobi(t, s, m)) < 1e-12


def test_vertices_outside_the_kernel(pkg, orc):
    """A degree-5 vertex and an isolated one beside qualifying vertices."""
    print("case pair rest", flush=True)
    edges = [("c", i) for i in range(5)] + [(0, 1), (1, 2)]
    g = pkg.NamedGraph(vertices=["alone"], edges=edges)
    t = pkg.build_topology(g, 3, 2)
    s = pkg.peps.random_sites(t, 8)
    m = pkg.peps.random_messages(t, 9)
    want, _, _ = orc.sweep_jacobi(t, s, m)
    with pkg.Engine(t, s, dtype="f64") as e:
        e.set_messages(m)
        e.sweep()
        np.testing.assert_allclose(e.messages(), want, rtol=1e-12,
                                   atol=1e-15 * np.max(np.abs(want)))


@pytest.mark.parametrize("dtype", ["f64", "c128"])
def test_folded_stopping_rule(pkg, dtype):
    """Networks that stop at different sweeps, inside a 16-sweep graph and at maxiter: the
    folded rule, the separate reduction and eager launches agree bit for bit."""
    print(f"case pair fold {dtype}", flush=True)
    tops = [pkg.build_topology(pkg.named_grid(sh), D, 2)
            for sh, D in (((3, 3), 2), ((4, 5), 4), ((1, 6), 3), ((5, 3), 5))]
    b = pkg.concat_topologies(tops)
    rng = np.random.default_rng(11)
    s = rng.standard_normal(int(b.site_off[-1])) / 4
    if dtype == "c128":
        s = s + 1j * rng.standard_normal(s.size) / 4
    for kw in ({"maxiter": 60, "tol": 1e-9}, {"maxiter": 60, "tol": 1e-9, "criterion": "maxabs"},
               {"maxiter": 7, "tol": 1e-9}, {"maxiter": 21}):
        got = []
        for fold, graph in ((1, True), (0, True), (1, False)):
            with pkg.Engine(b, s, dtype=dtype) as e:
                e.set_option("fold_bookkeeping", fold)
                for _ in range(2):  # the second run replays the captured graph
                    e.init_messages("identity")
                    r = e.run(use_graph=graph, **kw)
                got.append((e.messages(), r.sweeps, r.delta, r.at_iteration))
        for x in got[1:]:
            for u, v in zip(got[0], x):
                np.testing.assert_array_equal(u, v)
