"""Runs on the pair kernel's many-sweep launches (csrc/pair.hip, k_pair_run) against the same
runs launch by launch (option "pair_run" 0).  The arithmetic of a sweep is the same code, so a
Jacobi run agrees bit for bit: messages, sweeps, delta, the stopping sweep and the residuals.
A sequential run launch by launch takes its residuals from another kernel, which sums in
another order: those agree to rounding.  Lattices with leaves, isolated edges, sides around
the 16-wide tiles, sweep counts around the look-back of the stopping rule and of one launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(pkg, g, D, d, dtype, seed=3):
    t = pkg.build_topology(g, D, d)
    rng = np.random.default_rng(seed)
    s = rng.standard_normal(int(t.site_off[-1])) * pkg.peps.peps_scale(d, max(2, int(t.edge_dim.max())))
    m = rng.random(int(t.msg_off[-1])) + 0.1
    if dtype == "c128":
        s = s + 1j * rng.standard_normal(s.size) / 4
        m = m + 0.1j * rng.standard_normal(m.size)
    return t, s, m


def _run(pkg, t, s, m, dtype, option, order=None, **kw):
    with pkg.Engine(t, s, dtype=dtype) as e:
        e.set_option("pair_run", option)
        out = []
        for _ in range(2):  # the second run starts on buffers the first one has used
            e.set_messages(m)
            r = e.run(**kw) if order is None else e.run_sequential(order, **kw)
            out.append((e.messages(), np.array(r.sweeps), np.array(r.at_iteration),
                        np.array(r.delta), *e.residuals()))
        for x, y in zip(*out):
            np.testing.assert_array_equal(x, y)
        return out[0]


LATTICES = {"4x4": ((4, 4), 2), "1x2": ((1, 2), 3), "1x7": ((1, 7), 8), "5x3": ((5, 3), 4),
            "6x5": ((6, 5), 5), "4x3": ((4, 3), 6), "13x11": ((13, 11), 3), "16x16": ((16, 16), 6)}


@pytest.mark.parametrize("dtype", ["f64", "c128"])
@pytest.mark.parametrize("name", list(LATTICES) + ["hex"])
def test_jacobi_runs(pkg, name, dtype):
    if name == "hex":
        g, D = pkg.heavy_hex_lattice(3, 6), 4
    else:
        shape, D = LATTICES[name]
        g = pkg.named_grid(shape)
    if dtype == "c128":
        D = min(D, 5)
    t, s, m = _net(pkg, g, D, 1 if name == "5x3" else 2, dtype)
    for kw in ({"maxiter": 100, "tol": 1e-8}, {"maxiter": 100, "tol": 1e-10, "criterion": "maxabs"},
               {"maxiter": 4}, {"maxiter": 5, "tol": 0.0}, {"maxiter": 9, "tol": 1e-30},
               {"maxiter": 60, "tol": 0.9}, {"maxiter": 6, "tol": 1e-2}, {"tol": 1e-6}):
        print(f"case pair run {name} {dtype} {kw}", flush=True)
        for x, y in zip(_run(pkg, t, s, m, dtype, 250000, **kw), _run(pkg, t, s, m, dtype, 0, **kw)):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("maxiter", [255, 256, 257, 513])
def test_several_launches(pkg, maxiter):
    print(f"case pair run launches {maxiter}", flush=True)
    t, s, m = _net(pkg, pkg.named_grid((3, 4)), 2, 2, "f64")
    for kw in ({"maxiter": maxiter}, {"maxiter": maxiter, "tol": 0.0}):
        for x, y in zip(_run(pkg, t, s, m, "f64", 250000, **kw), _run(pkg, t, s, m, "f64", 0, **kw)):
            np.testing.assert_array_equal(x, y)


def test_invalid_numbers(pkg):
    """NaN (quiet, signalling with any payload) and infinite messages end at the same sweep."""
    t, s, m = _net(pkg, pkg.named_grid((4, 3)), 3, 2, "f64")
    bits = m.copy().view(np.uint64)
    bits[5], bits[40] = 0x7FF4DEADBEEF0001, 0x7FF0000000000000
    for k, x in enumerate((m * 0, bits.view(np.float64))):
        print(f"case pair run invalid {k}", flush=True)
        a, b = (_run(pkg, t, s, x, "f64", o, maxiter=12, tol=1e-9) for o in (250000, 0))
        for u, v in zip(a, b):
            np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("dtype", ["f64", "c128"])
@pytest.mark.parametrize("shape,D", [((4, 4), 2), ((1, 5), 3), ((5, 7), 4), ((10, 10), 3), ((4, 3), 5)])
def test_sequential_runs(pkg, shape, D, dtype):
    g = pkg.named_grid(shape)
    t, s, m = _net(pkg, g, D, 2, dtype)
    forest = [t.slot(*e) for e in pkg.forest_cover_edge_sequence(g)]
    shuffled = [int(q) for q in np.random.default_rng(5).permutation(t.nports)]
    for name, order in (("forest", forest), ("reversed", forest[::-1]), ("shuffled", shuffled),
                        ("sorted", sorted(forest))):
        for kw in ({"maxiter": 60, "tol": 1e-9}, {"maxiter": 1}, {"maxiter": 1, "tol": 1e-9},
                   {"maxiter": 2}, {"maxiter": 7, "tol": 1e-30},
                   {"maxiter": 60, "tol": 1e-8, "criterion": "maxabs"}):
            print(f"case pair run sequential {shape} D={D} {dtype} {name} {kw}", flush=True)
            a, b = (_run(pkg, t, s, m, dtype, o, order=order, **kw) for o in (250000, 0))
            np.testing.assert_array_equal(a[0], b[0])
            np.testing.assert_array_equal(a[1], b[1])
            np.testing.assert_array_equal(a[2], b[2])
            np.testing.assert_allclose(a[3], b[3], rtol=1e-6, atol=1e-13)


def test_waits_cut_short(pkg):
    """A wait limit of 1 us: most launches give up, and the run is repeated launch by launch."""
    t, s, m = _net(pkg, pkg.named_grid((12, 12)), 4, 2, "f64")
    g = pkg.named_grid((12, 12))
    forest = [t.slot(*e) for e in pkg.forest_cover_edge_sequence(g)]
    for order in (None, forest):
        print(f"case pair run cut short {order is not None}", flush=True)
        kw = {"maxiter": 80, "tol": 1e-9}
        a, b = (_run(pkg, t, s, m, "f64", o, order=order, **kw) for o in (1, 0))
        for u, v in zip(a[:3], b[:3]):
            np.testing.assert_array_equal(u, v)
        with pkg.Engine(t, s, dtype="f64") as e:
            e.set_option("pair_run", 1)
            e.set_messages(m)
            e.run(**kw) if order is None else e.run_sequential(order, **kw)
            assert e.get_option("pair_run_gave_up") == 1


@pytest.mark.parametrize("order", ["jacobi", "sequential"])
@pytest.mark.parametrize("launch,maxiter", [(1, 80), (2, 300), (2, 600), (3, 600)])
def test_a_later_launch_gives_up(pkg, order, launch, maxiter):
    """The run goes on launch by launch behind the launches that came to their end."""
    print(f"case pair run gives up {order} launch {launch} of {maxiter} sweeps", flush=True)
    g = pkg.named_grid((4, 3))
    t, s, m = _net(pkg, g, 2, 2, "f64")
    seq = None if order == "jacobi" else [t.slot(*x) for x in pkg.forest_cover_edge_sequence(g)]
    for kw in ({"maxiter": maxiter}, {"maxiter": maxiter, "tol": 0.0},
               {"maxiter": maxiter, "tol": 0.0, "criterion": "maxabs"}):
        want = _run(pkg, t, s, m, "f64", 0, order=seq, **kw)
        with pkg.Engine(t, s, dtype="f64") as e:
            e.set_option("pair_run_give_up", launch)
            e.set_messages(m)
            r = e.run(**kw) if seq is None else e.run_sequential(seq, **kw)
            got = (e.messages(), np.array(r.sweeps), np.array(r.at_iteration), np.array(r.delta),
                   *e.residuals())
            assert e.get_option("pair_run_gave_up") == 1
        for x, y in zip(got, want):
            np.testing.assert_array_equal(x, y)


def test_runs_after_one_that_gave_up(pkg):
    """The next run goes launch by launch, the one after it tries again; given up again, two do;
    after a run that ends, the count starts anew."""
    print("case pair run tries again", flush=True)
    t, s, m = _net(pkg, pkg.named_grid((4, 3)), 2, 2, "f64")
    with pkg.Engine(t, s, dtype="f64") as e:
        def run():
            e.set_messages(m)
            e.run(maxiter=20)
            return e.get_option("pair_run_gave_up")
        e.set_option("pair_run_give_up", 1)
        assert [run() for _ in range(8)] == [1, 1, 2, 2, 2, 3, 3, 3]
        e.set_option("pair_run_give_up", 0)
        assert [run() for _ in range(3)] == [3, 3, 3]  # left out twice more, then a whole run
        e.set_option("pair_run_give_up", 1)
        assert [run() for _ in range(3)] == [4, 4, 5]
