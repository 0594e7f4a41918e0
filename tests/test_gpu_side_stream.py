"""FP32 engines with a large-bond bucket (9..12) beside one of bond dimensions 5..8 sweep them on
two streams (a fork and a join in every sweep, captured or not), whatever their sizes.  Every
network runs the same kernels as in an engine of its own, which has one bucket and one stream:
the messages, sweeps and deltas agree bit for bit, run after run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("size", ["large", "small", "with D = 3"])
def test_two_buckets_match_each_alone(pkg, size, use_graph):
    print(f"case side stream {size} graph={use_graph}", flush=True)
    nets = [(pkg.named_grid((16, 17)), 10), (pkg.named_grid((18, 16)), 6),
            (pkg.heavy_hex_lattice(5, 12), 12), (pkg.heavy_hex_lattice(4, 8), 8)]
    if size != "large":
        nets = [(pkg.named_grid((2, 2)), 9), (pkg.named_grid((1, 3)), 12), (pkg.named_grid((3, 2)), 5)]
    if size == "with D = 3":
        nets.append((pkg.named_grid((4, 4)), 3))
    tops = [pkg.build_topology(g, D, 2) for g, D in nets]
    sites = [pkg.peps.random_sites(t, 3 + i, scale=pkg.peps.peps_scale(2, D))
             for i, (t, (_, D)) in enumerate(zip(tops, nets))]
    kw = {"maxiter": 37, "tol": 1e-5, "use_graph": use_graph}
    alone = []
    for t, s in zip(tops, sites):
        with pkg.Engine(t, s, dtype="f32") as e:
            e.init_messages("identity")
            r = e.run(**kw)
            alone.append((e.messages(), r.sweeps[0], r.delta[0]))
    with pkg.Engine(pkg.concat_topologies(tops), np.concatenate(sites), dtype="f32") as e:
        for _ in range(3):
            e.init_messages("identity")
            r = e.run(**kw)
            np.testing.assert_array_equal(e.messages(), np.concatenate([a[0] for a in alone]))
            np.testing.assert_array_equal(r.sweeps, [a[1] for a in alone])
            np.testing.assert_array_equal(r.delta, [a[2] for a in alone])
