"""Two streaming products in one pass (csrc/contract.h, k_cn_pair): A with B1, the result with
B2, over label positions in every arrangement, extents of 1, odd extents, row counts around a
block's, and the output widths 4, 9 and 16 with remainders, against numpy einsum.  An entry is
a sum of U V S products of three normal factors: the error stays near sqrt(U V S) eps of the
largest entry, below 1e-14 here; 1e-12 is asserted.  A longer network compares the fused
steps with each other through a chain."""
import string

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# row extents of A, then the extents shared by (A, B1), (A, B2), (B1, B2), kept by B1 and B2
CASES = [((17, 31), (3, 2), (3,), (2,), (3,), (3, 3)), ((256,), (4,), (4,), (2,), (2, 2), (4,)),
         ((7, 5, 9), (), (3,), (2,), (5,), (2,)), ((300,), (3,), (), (2,), (), (3,)),
         ((1000,), (2, 2), (2,), (), (4,), (5, 2)), ((29,), (9,), (9,), (2,), (9,), (9,)),
         ((28,), (9,), (9,), (2,), (9,), (9,)), ((57,), (9,), (9,), (2,), (9,), (9,)),
         ((64, 3), (16,), (16,), (2,), (16,), (16,)), ((100,), (5,), (5,), (3,), (5,), (17,)),
         ((2049,), (1,), (1,), (1,), (1,), (1,)), ((40,), (25,), (2,), (2,), (25,), (3,))]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("seed", [0, 1])
def test_three_tensors(pkg, case, seed):
    print(f"case contract pair {CASES[case]} seed {seed}", flush=True)
    rng = np.random.default_rng([case, seed])
    letters = iter(string.ascii_letters)
    groups = [[(next(letters), d) for d in dims] for dims in CASES[case]]
    f, u, v, s, o, n = groups
    tensors, terms = [], []
    for labs in (f + u + v, u + s + o, v + s + n):
        labs = [labs[i] for i in rng.permutation(len(labs))]
        terms.append("".join(x for x, _ in labs))
        tensors.append(rng.standard_normal([d for _, d in labs]))
    idx = {x: pkg.Index(d) for g in groups for x, d in g}
    its = [pkg.ITensor(t, [idx[x] for x in term]) for t, term in zip(tensors, terms)]
    r = pkg.contract_network(its, alg=pkg.Exact(order=((0, 1), 2)))
    name = {i: x for x, i in idx.items()}
    out = "".join(name[i] for i in r.inds)
    want = np.einsum(",".join(terms) + "->" + out, *tensors, optimize=True)
    assert sorted(out) == sorted(x for g in (f, o, n) for x, _ in g)
    assert np.max(np.abs(r.data - want)) <= 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("shape,D,d", [((3, 3), 2, 2), ((4, 3), 3, 2), ((3, 5), 2, 3), ((3, 3), 4, 1)])
def test_peps_norm(pkg, orc, shape, D, d):
    """Site, conjugate site, site by site: every step but the first pairs is a fused one."""
    print(f"case contract pair norm {shape} D={D} d={d}", flush=True)
    t = pkg.build_topology(pkg.named_grid(shape), D, d)
    s = pkg.peps.random_sites(t, 4, scale=pkg.peps.peps_scale(d, D))
    idx = {}
    its, ops = [], []
    for w in range(t.nv):
        a = s[t.site_off[w]:t.site_off[w + 1]].reshape(t.site_shape(w))
        edges = [int(t.port_edge[q]) for q in range(t.port_off[w], t.port_off[w + 1])]
        for side in "kb":
            labs = [("s", w)] + [(side, e) for e in edges]
            for x, m in zip(labs, a.shape):
                idx.setdefault(x, pkg.Index(int(m)))
            its.append(pkg.ITensor(a, [idx[x] for x in labs]))
            ops.append((a, labs))
    n = len(its)
    order = 0
    for k in range(1, n):
        order = (order, k)
    got = float(pkg.contract_network(its, alg=pkg.Exact(order=order)).data)
    want, have = ops[0]
    for a, labs in ops[1:]:
        shared = [x for x in have if x in labs]
        want = np.tensordot(want, a, ([have.index(x) for x in shared],
                                      [labs.index(x) for x in shared]))
        have = [x for x in have + labs if x not in shared]
    want = float(want)
    assert abs(got - want) <= 1e-12 * abs(want)


def test_plan_figures(pkg):
    """A fused pair's bytes: three operands and the result; FLOPs of both products.  Beyond the
    fused kernel's extents (17 labels shared by A and B1) the product between counts twice."""
    print("case contract pair figures", flush=True)
    m, v, s, o, n = 300, 3, 2, 3, 9
    for u, between in ((9, 0), (17, 2)):
        size = {"m": m, "u": u, "v": v, "s": s, "o": o, "n": n}
        labels = ["muv", "uso", "vsn"]
        plan = pkg.ContractionPlan([tuple(size[x] for x in t) for t in labels],
                                   [tuple(t) for t in labels], order=(0, 1, 3, 2))
        moved = m * u * v + u * s * o + v * s * n + m * o * n + between * m * v * s * o
        assert plan.bytes == 8.0 * moved
        assert plan.flops == 2.0 * (m * v * u * s * o + m * o * v * s * n)
        plan.close()
