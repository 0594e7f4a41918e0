"""FP32 vertex scalars on every bucket's kernel, alone and beside the others in one engine: ports
absorbed in FP32, the last contraction <E, A> in FP64, as the generic kernel has it, so that
their distance from FP64 (the same FP32 inputs in an FP64 engine) is no larger than the generic
kernel's.  Compared as root mean squares over the vertices of a network at its fixed point:
100 or more independent errors give each to 7%, and 1.4 is four times the uncertainty of the
ratio.  The last contraction in FP32, rounded at the size of the scalar instead of its terms',
is 2 to 6 times further off."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NETS = [((24, 24), 2, False), ((20, 20), 3, False), ((16, 16), 4, False), ((6, 12), 6, True),
        ((11, 12), 7, False), ((10, 11), 8, False), ((10, 10), 10, False), ((10, 10), 12, False),
        ((5, 12), 11, True)]


def _net(pkg, net, d, seed):
    shape, D, hexa = net
    t = pkg.build_topology(pkg.heavy_hex_lattice(*shape) if hexa else pkg.named_grid(shape), D, d)
    s = pkg.peps.random_sites(t, seed, scale=pkg.peps.peps_scale(d, D))
    return t, s.astype(np.float32).astype(np.float64)


def _scalars(pkg, t, s):
    """FP64, FP32 and FP32 generic scalars at the FP32 messages of a converged run."""
    with pkg.Engine(t, s, dtype="f64") as e:
        e.init_messages("identity")
        e.run(maxiter=40, tol=1e-12)
        m = e.messages().astype(np.float32).astype(np.float64)
        e.set_messages(m)
        out = [e.vertex_scalars()]
    for path in ("auto", "generic"):
        with pkg.Engine(t, s, dtype="f32") as e:
            e.set_path(path)
            e.set_messages(m)
            out.append(e.vertex_scalars())
    return out


def _check(want, got, generic):
    rms = lambda x: float(np.sqrt(np.mean((x / want - 1.0) ** 2)))  # noqa: E731
    print(f"rms {rms(got):.2e}, generic {rms(generic):.2e}", flush=True)
    assert rms(got) <= 1.4 * rms(generic)


@pytest.mark.parametrize("net", range(len(NETS)))
def test_alone(pkg, net):
    print(f"case scalar precision {NETS[net]}", flush=True)
    _check(*_scalars(pkg, *_net(pkg, NETS[net], 2, 21)))


@pytest.mark.parametrize("d", [1, 3])
@pytest.mark.parametrize("net", [0, 2, 4])
def test_other_physical_dimensions(pkg, net, d):
    print(f"case scalar precision {NETS[net]} d={d}", flush=True)
    _check(*_scalars(pkg, *_net(pkg, NETS[net], d, 22)))


def test_beside_others(pkg):
    """Every bucket in one engine, with an isolated vertex or without."""
    nets = [_net(pkg, n, 2, 23 + i) for i, n in enumerate(NETS)]
    one = pkg.build_topology(pkg.NamedGraph(vertices=["a"], edges=[]), 2, 2)
    for extra in ([], [(one, np.array([0.5, -2.0]))]):
        all_ = nets + extra
        b, s = pkg.concat_topologies([t for t, _ in all_]), np.concatenate([s for _, s in all_])
        out = _scalars(pkg, b, s)
        at = 0
        for t, _ in nets:
            print(f"case scalar precision batch {t.nv} vertices", flush=True)
            _check(*(x[at:at + t.nv] for x in out))
            at += t.nv
        if extra:
            np.testing.assert_allclose(out[1][at:], [4.25], rtol=1e-15)
