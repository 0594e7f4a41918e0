"""Memory that a context keeps between calls: bounded by the option "keep_workspace", given back
when it is lowered, and without any of it (0: pageable copies, as where no memory can be
pinned) every result is the same."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _free():
    """Free device memory, from the HIP runtime that the library links."""
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _layer(t):
    idx = {v: i for i, v in enumerate(t.vertices)}
    slots = []
    for (i, j) in t.vertices:
        if j % 2 == 1 and (i, j + 1) in idx:
            u, w = idx[(i, j)], idx[(i, j + 1)]
            slots.append(next(q for q in range(t.port_off[u], t.port_off[u + 1])
                              if int(t.port_nbr[q]) == w))
    return slots


def _gates(pkg, e, t, D):
    rng = np.random.default_rng(3)
    slots = _layer(t)
    return e.apply_gates([2] * len(slots), slots, list(rng.standard_normal((len(slots), 4, 4))),
                         normalize=True, maxdim=D)


def test_gate_workspace(pkg):
    print("case kept workspace gates", flush=True)
    t = pkg.build_topology(pkg.named_grid((16, 16)), 6, 2)
    s = pkg.peps.random_sites(t, 5, scale=pkg.peps.peps_scale(2, 6))
    out = []
    # the first pass also has the runtime set aside the kernels' scratch memory
    for keep in ("first", None, 0, 1):
        with pkg.Engine(t, s, dtype="f64") as e:
            assert e.get_option("keep_workspace") == 512
            if keep in (0, 1):
                e.set_option("keep_workspace", keep)
            e.init_messages("identity")
            e.run(maxiter=3)
            before = _free()
            for _ in range(2):
                e.set_sites(s)
                chi, sv = _gates(pkg, e, t, 6)
            kept = before - _free()
            if keep is None:  # 112 gates: 30 MiB
                assert kept >= 16 * MIB
                e.set_option("keep_workspace", 0)
                assert before - _free() <= 4 * MIB
            elif keep != "first":
                assert kept <= 4 * MIB
            out.append((np.array(chi), np.array(sv), e.messages(), e.sites()))
    for x in out[1:]:
        for u, v in zip(out[0], x):
            np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("dtype,shape,D", [("f32", (48, 41), 3), ("f32", (90, 91), 4), ("f64", (70, 71), 4),
                                           ("f64", (130, 129), 4), ("c128", (60, 61), 4)])
def test_message_download(pkg, dtype, shape, D):
    """Messages of one, two and several chunks, through pinned staging and without it."""
    print(f"case kept workspace messages {dtype} {shape}", flush=True)
    t = pkg.build_topology(pkg.named_grid(shape), D, 1)
    rng = np.random.default_rng(6)
    s, m = rng.standard_normal(int(t.site_off[-1])), rng.standard_normal(int(t.msg_off[-1]))
    if dtype == "c128":
        s, m = s + 0j, m + 1j * m[::-1]
    with pkg.Engine(t, s, dtype=dtype) as e:
        e.set_messages(m)
        want = m.astype(np.float32).astype(np.float64) if dtype == "f32" else m
        for keep in (512, 0, 512):
            e.set_option("keep_workspace", keep)
            np.testing.assert_array_equal(e.messages(), want)


def test_refuses_a_negative_size(pkg):
    t = pkg.build_topology(pkg.named_grid((2, 2)), 2, 2)
    with pkg.Engine(t, pkg.peps.random_sites(t, 1), dtype="f64") as e:
        with pytest.raises(Exception, match="keep_workspace"):
            e.set_option("keep_workspace", -1)
