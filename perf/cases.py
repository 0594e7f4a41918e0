"""The workloads whose speed matters to users of this framework, each through its public entry
points (`Engine`, `ContractionPlan`), over the sizes, lattices, data types and options that
the repository's own benchmark, tests and configurations run.

Paths ("path" of a case):
  jacobi      messages reset, Jacobi sweeps to a tolerance or a count (FP32, BF16, FP64,
              complex FP64; one network or a batch of uneven ones), optional FP64 polishing
              sweeps, messages and log-norm out
  sequential  the reference's default schedule: one message at a time over the forest cover
  tfim        BP, then the transverse-field Ising energy and its gradient (fixed-point adjoint)
  local       BP, then a general local energy and its gradient
  contract    exact <psi|psi> of a small PEPS on a kept plan
  gates       one simple-update step: two-site gates on every bond, in four layers of
              disjoint bonds, on a resident network
"""
import functools
import math

import numpy as np
import torch

from __graft_entry__ import import_package

pkg = import_package()
DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ------------------------------------------------------------------ the cases

def _jacobi(name, lattice, rows, cols, bond, dtype, maxiter, tol=-1.0, polish=0, phys=2):
    c = {"path": "jacobi", "lattice": lattice, "rows": rows, "cols": cols, "bond": bond,
         "phys": phys, "dtype": dtype, "maxiter": maxiter, "tol": tol, "polish": polish}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a 4x4 solve in the default data type, where launches and host
        # round trips are all of the time
        _jacobi("jacobi_4x4_D2_f64", "square", 4, 4, 2, "f64", 100, 1e-10),
        # the headline network, 20 sweeps as a time-evolution step warm-starts them
        _jacobi("jacobi_32x32_D8_f32", "square", 32, 32, 8, "f32", 20),
        # an ordinary FP64 run (the reference's only type) at an odd size and bond dimension
        _jacobi("jacobi_23x17_D5_f64", "square", 23, 17, 5, "f64", 200, 1e-10),
        # complex states (real-time evolution)
        _jacobi("jacobi_10x10_D4_c128", "square", 10, 10, 4, "c128", 200, 1e-10),
        # a very large lattice of small tensors, where memory traffic counts
        _jacobi("jacobi_256x256_D3_f32", "square", 256, 256, 3, "f32", 64),
        # large tensors in mixed precision: BF16 sweeps, then FP64 polishing
        _jacobi("jacobi_24x24_D16_bf16", "square", 24, 24, 16, "bf16", 6, polish=3),
        # many independent networks of uneven size, bond dimension and lattice in one engine
        {"name": "batch_16_uneven_f32", "path": "jacobi", "lattice": "batch", "rows": 16,
         "cols": 48, "bond": 12, "phys": 2, "dtype": "f32", "maxiter": 200, "tol": 1e-7,
         "polish": 0},
        # the default of `beliefpropagation`: sequential updates over the forest cover
        {"name": "sequential_10x10_D4_f64", "path": "sequential", "rows": 10, "cols": 10,
         "bond": 4, "dtype": "f64", "maxiter": 100, "tol": 1e-10},
        # variational optimisation: energy and gradient of the Ising model in a field
        {"name": "tfim_16x16_D6_f32", "path": "tfim", "rows": 16, "cols": 16, "bond": 6,
         "dtype": "f32"},
        # the same for a general Hamiltonian of one- and two-site terms
        {"name": "local_16x16_D6_f32", "path": "local", "rows": 16, "cols": 16, "bond": 6,
         "dtype": "f32"},
        # exact norm of a small state, the check of a BP result
        {"name": "contract_6x6_D3", "path": "contract", "rows": 6, "cols": 6, "bond": 3},
        # one Trotter step of imaginary-time evolution
        {"name": "gates_16x16_D6_f64", "path": "gates", "rows": 16, "cols": 16, "bond": 6,
         "dtype": "f64"},
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["jacobi"] * 6 + ["sequential", "tfim", "local", "contract", "gates"])
    if path == "jacobi":
        dtype = rng.choice(["f32", "f32", "f32", "f64", "f64", "bf16", "c128"])
        bond = {"f32": lambda: rng.randint(2, 12), "f64": lambda: rng.randint(2, 10),
                "bf16": lambda: rng.randint(6, 16), "c128": lambda: rng.randint(2, 5)}[dtype]()
        # the lattice fills at most 2^24 tensor entries, and 256 x 256 sites
        most = min(256, int(math.sqrt(2 ** 24 / (2 * bond ** 4)))) if dtype != "c128" else 14
        if dtype == "f64" and bond < 6:
            most = min(most, 40)
        rows, cols = _logint(rng, 4, max(5, most)), _logint(rng, 4, max(5, most))
        lattice = rng.choice(["square", "square", "hex"])
        if dtype == "bf16":
            return _jacobi(None, lattice, rows, cols, bond, dtype, rng.randint(4, 20),
                           polish=rng.randint(0, 3))
        if dtype == "f32":
            return _jacobi(None, lattice, rows, cols, bond, dtype, rng.randint(8, 64))
        return _jacobi(None, lattice, rows, cols, bond, dtype, 200, 1e-10)
    if path == "sequential":
        return {"path": path, "rows": _logint(rng, 3, 14), "cols": _logint(rng, 3, 14),
                "bond": rng.randint(2, 6), "dtype": rng.choice(["f64", "f64", "f32"]),
                "maxiter": 100, "tol": 1e-10}
    if path in ("tfim", "local"):
        return {"path": path, "rows": _logint(rng, 4, 20), "cols": _logint(rng, 4, 20),
                "bond": rng.randint(5, 8), "dtype": "f32"}
    if path == "contract":
        bond = rng.randint(2, 4)
        cols = rng.randint(3, {2: 8, 3: 6, 4: 5}[bond])
        return {"path": path, "rows": rng.randint(3, 9), "cols": cols, "bond": bond}
    return {"path": path, "rows": _logint(rng, 4, 20), "cols": _logint(rng, 4, 20),
            "bond": rng.randint(3, 8), "dtype": rng.choice(["f64", "f32"])}


# ------------------------------------------------------------------ networks and inputs

@functools.lru_cache(maxsize=64)
def _topology(lattice, rows, cols, bond, phys):
    """Topologies of one lattice, or of a batch: `rows` networks with sides up to `cols` and
    bond dimensions up to `bond`, as the uneven workload draws them."""
    if lattice != "batch":
        g = (pkg.heavy_hex_lattice(max(2, rows // 2), max(cols, 4)) if lattice == "hex"
             else pkg.named_grid((rows, cols)))
        return (pkg.build_topology(g, bond, phys),)
    rng = np.random.default_rng(20)
    tops = []
    for n in range(rows):
        L = int(rng.integers(8, cols + 1))
        D = (4, 6, 8, 10, 12)[n % 5] if n < 10 else int(rng.choice([4, 6, 8, 10, 12]))
        D = min(D, bond)
        hex_ = bool(rng.integers(0, 2))
        g = pkg.heavy_hex_lattice(max(2, L // 2), L) if hex_ else pkg.named_grid((L, L))
        tops.append(pkg.build_topology(g, D, phys))
    return tuple(tops)


def _topologies(case):
    return _topology(case.get("lattice", "square"), case["rows"], case["cols"], case["bond"],
                     case.get("phys", 2))


@functools.lru_cache(maxsize=8)
def _joined(*key):
    tops = _topology(*key)
    return tops[0] if len(tops) == 1 else pkg.concat_topologies(tops)


def _sites(case, seed):
    """Site tensors of every network: iid normal entries over sqrt(d D^4)."""
    gen = torch.Generator(device=DEV)
    out = []
    for n, t in enumerate(_topologies(case)):
        gen.manual_seed(int(seed) * 1000003 + n)
        D = int(t.edge_dim.max())
        k = 2 if case.get("dtype") == "c128" else 1
        x = torch.randn(k * int(t.site_off[-1]), generator=gen, device=DEV, dtype=torch.float64)
        x = (x * pkg.peps.peps_scale(case.get("phys", 2), D)).cpu().numpy()
        out.append(x.view(np.complex128) if k == 2 else x)
    return out[0] if len(out) == 1 else np.concatenate(out)


def _slots(t, layer):
    """The message slots (owner = first site) of one layer of disjoint square-lattice bonds:
    layer 0, 1 bonds along the columns' direction, 2, 3 along the rows'."""
    out = []
    idx = {v: i for i, v in enumerate(t.vertices)}
    for (i, j) in t.vertices:
        w = (i, j + 1) if layer < 2 else (i + 1, j)
        if w in idx and (j if layer < 2 else i) % 2 == (1 + layer) % 2:
            u = idx[(i, j)]
            out.append(next(q for q in range(t.port_off[u], t.port_off[u + 1])
                            if int(t.port_nbr[q]) == idx[w]))
    return out


def _gates(t, seed):
    """exp(-0.1 h) with a random symmetric bond term h for every bond, layer by layer."""
    rng = np.random.default_rng([int(seed), 3])
    layers = []
    for layer in range(4):
        slots = _slots(t, layer)
        mats = []
        for _ in slots:
            h = rng.standard_normal((4, 4))
            w, v = np.linalg.eigh(0.5 * (h + h.T))
            mats.append((v * np.exp(-0.1 * w)) @ v.T)
        if slots:
            layers.append((slots, mats))
    return layers


def _operators(t, seed):
    """Random symmetric one-site terms and nearest-neighbour products."""
    rng = np.random.default_rng([int(seed), 4])
    sym = lambda n: (lambda x: 0.5 * (x + x.transpose(0, 2, 1)))(rng.standard_normal((n, 2, 2)))  # noqa: E731
    return sym(t.nv), sym(t.ne), sym(t.ne)


def _norm_network(t, s):
    tensors, labels = [], []
    for u in range(t.nv):
        a = s[t.site_off[u]:t.site_off[u + 1]].reshape(t.site_shape(u))
        edges = [int(t.port_edge[q]) for q in range(t.port_off[u], t.port_off[u + 1])]
        tensors += [a, a]
        labels += [(("s", u),) + tuple(("k", e) for e in edges),
                   (("s", u),) + tuple(("b", e) for e in edges)]
    return tensors, labels


def prepare(case, seed):
    s = _sites(case, seed)
    t = _joined(case.get("lattice", "square"), case["rows"], case["cols"], case["bond"],
                case.get("phys", 2))
    if case["path"] == "contract":
        tensors, labels = _norm_network(t, s)
        plan = pkg.ContractionPlan([x.shape for x in tensors], labels, order_alg="cheapest")
        flat = np.concatenate([x.ravel() for x in tensors])
        src = pkg._lib.DeviceArray(flat.size, np.float64)
        dst = pkg._lib.DeviceArray(1, np.float64)
        src.upload(flat)
        return {"case": case, "plan": plan, "src": src, "dst": dst}
    st = {"case": case, "topo": t, "engine": pkg.Engine(t, s, dtype=case["dtype"])}
    e = st["engine"]
    e.init_messages("identity")
    if case["path"] == "sequential":
        g = pkg.named_grid((case["rows"], case["cols"]))
        st["order"] = np.array([t.slot(*uv) for uv in pkg.forest_cover_edge_sequence(g)],
                               dtype=np.int32)
    elif case["path"] == "local":
        st["ops"] = _operators(t, seed)
    elif case["path"] == "gates":
        st["layers"] = _gates(t, seed)
        st["sites"] = s
        z = np.diag([1.0, -1.0])
        st["z"] = np.broadcast_to(z, (t.nv, 2, 2)).copy()
    return st


# ------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    if case["path"] == "contract":
        state["plan"].execute_device(state["src"], state["dst"])
        return state["dst"].numpy()
    e = state["engine"]
    if case["path"] == "jacobi":
        e.init_messages("identity")
        e.run(maxiter=case["maxiter"], tol=case["tol"] if case["tol"] > 0 else None)
        if case["polish"]:
            e.polish_fp64(case["polish"])
        return {"messages": e.messages(), "lognorm": e.lognorms()}
    if case["path"] == "sequential":
        e.init_messages("identity")
        e.run_sequential(state["order"], maxiter=case["maxiter"], tol=case["tol"])
        return {"messages": e.messages(), "lognorm": e.lognorms()}
    if case["path"] in ("tfim", "local"):
        e.init_messages("identity")
        e.run(maxiter=200, tol=1e-11)
        if case["path"] == "tfim":
            energy, grad, _, _ = e.tfim_energy(1.0, 3.0, grad=True, adj_tol=1e-6,
                                               adj_maxiter=500)
        else:
            energy, grad, _, _ = e.local_energy(*state["ops"], grad=True, adj_tol=1e-6,
                                                adj_maxiter=500)
        return {"energy": energy, "gradient": grad}
    # gates: a fresh state, converged messages, one gate on every bond, <Z> of every site.
    # The site tensors themselves are fixed only up to a sign per bond index; the singular
    # values, the new messages and the expectation values are not.
    e.set_sites(state["sites"])
    e.init_messages("identity")
    e.run(maxiter=12)
    sing = []
    for slots, mats in state["layers"]:
        _, sv = e.apply_gates([2] * len(slots), slots, mats, normalize=True,
                              maxdim=case["bond"])
        sing.append(sv)
    return {"singular_values": sing, "messages": e.messages(), "z": e.expect_vertex(state["z"])}


# ------------------------------------------------------------------ what a pass cannot do without

def _sweep_flops(t):
    """One Jacobi sweep with the partial products of a vertex shared between its outgoing
    messages: mode products and open contractions of 2 d D^(k+1) each."""
    n = {0: 0, 1: 1, 2: 4, 3: 8, 4: 12}
    tot = 0.0
    for u in range(t.nv):
        size, D = 1.0, 1
        k = int(t.port_off[u + 1] - t.port_off[u])
        if k:
            D = int(t.edge_dim[t.port_edge[t.port_off[u]]])
        size = float(t.phys_dim[u]) * float(D) ** k
        tot += 2.0 * n[k] * size * D
    return tot


def work(case):
    t = _joined(case.get("lattice", "square"), case["rows"], case["cols"], case["bond"],
                case.get("phys", 2))
    dtype = case.get("dtype", "f64")
    elt = {"f64": 8, "f32": 4, "bf16": 2, "c128": 16}[dtype]
    ns, nm, f = float(t.site_off[-1]), float(t.msg_off[-1]), _sweep_flops(t)
    f *= 4.0 if dtype == "c128" else 1.0
    sweep = elt * ns + 2.0 * (4 if dtype == "bf16" else elt) * nm
    if case["path"] == "jacobi":
        # sweeps to fidelity 1e-10 from the identity: about 14 on these networks
        n = min(case["maxiter"], 14) if case["tol"] > 0 else case["maxiter"]
        p = case["polish"]
        return {"bytes": n * sweep + p * 8.0 * (ns + 2 * nm) + 8.0 * nm, "flops": (n + p) * f}
    if case["path"] == "sequential":
        n = 10
        return {"bytes": n * sweep, "flops": n * f}
    if case["path"] in ("tfim", "local"):
        # 12 forward sweeps, 14 adjoint sweeps (products in value and tangent: twice), the
        # energy's and the gradient's own contractions
        return {"bytes": 12 * sweep + 14 * sweep + 6 * elt * ns + 8.0 * ns,
                "flops": (12 + 2 * 14 + 8) * f}
    if case["path"] == "contract":
        D2, rows, cols = case["bond"] ** 2, case["rows"], case["cols"]
        # boundary contraction, site by site, ket and bra absorbed one after the other
        per = 2.0 * 2.0 * 2 * case["bond"] * float(D2) ** min(rows, cols)
        return {"bytes": 8.0 * 2 * (rows - 1) * cols * float(D2) ** (min(rows, cols) - 1),
                "flops": rows * cols * per * case["bond"]}
    # gates: both sites of every bond read and written, gauge, QR, SVD and rebuild as about 12
    # products of a site with a bond matrix
    D = case["bond"]
    return {"bytes": 12 * sweep + 2.0 * 8.0 * 4.0 * ns, "flops": 12 * f + 4 * 12 * 2.0 * ns * 2 * D}


def tolerance(case):
    # About four times what implementations at the same precision show against 64 bits: FP32
    # 5e-8 to 2e-7 on square lattices and up to 9e-6 on slowly converging heavy-hex ones,
    # FP64 2e-16 to 1e-15 (with the same slow lattices allowed for), BF16 3e-3 before the
    # polishing sweeps contract it.  The stopping tolerances are far above the rounding noise
    # of a residual, so another correct implementation stops at the same sweep; the adjoint
    # sweeps stop at 1e-6.
    p, f32 = case["path"], case.get("dtype") == "f32"
    if p == "jacobi" and case["dtype"] == "bf16":
        return {"rel": 1.2e-2 * 0.7 ** case["polish"], "max": 2e-1}
    if p in ("jacobi", "sequential"):
        return {"rel": 4e-5 if f32 else 1e-12}
    if p in ("tfim", "local"):
        return {"rel": 1e-5}
    if p == "contract":
        return {"rel": 1e-13}
    return {"rel": 1e-5 if f32 else 1e-11}


# ------------------------------------------------------------------ the same in 64 bits

class _Net64:
    """One network in plain torch at 64 bits: vertices grouped by degree, messages as one
    (slots, D, D) tensor (one bond dimension per network)."""

    def __init__(self, t, sites, cplx=False):
        self.t, self.D, self.d = t, int(t.edge_dim.max()), int(t.phys_dim[0])
        self.dt = torch.complex128 if cplx else torch.float64
        own = t.port_owner()
        deg = np.diff(t.port_off)
        rev = torch.as_tensor(np.asarray(t.port_rev, dtype=np.int64), device=DEV)
        self.rev, self.groups = rev, []
        S = torch.as_tensor(sites, device=DEV).to(self.dt)
        for k in sorted(set(int(x) for x in deg)):
            us = np.nonzero(deg == k)[0]
            n = self.d * self.D ** k
            idx = np.asarray(t.site_off)[us][:, None] + np.arange(n)[None]
            idx = torch.as_tensor(idx, device=DEV)
            ports = torch.as_tensor(np.asarray(t.port_off)[us][:, None] + np.arange(k)[None],
                                    device=DEV)
            self.groups.append((k, torch.as_tensor(us, device=DEV), idx, ports))
        self.S = S
        del own

    def identity(self):
        e = torch.eye(self.D, device=DEV, dtype=self.dt)
        return e.expand(self.t.nports, self.D, self.D).clone()

    def site(self, g, S=None):
        return (self.S if S is None else S)[g[2]]

    def absorb(self, A, k, j, M):
        """A (n, d D^k) with its ket port j contracted with M (n, D, D) [ket][bra]."""
        n, D = A.shape[0], self.D
        x = A.reshape(n, self.d * D ** j, D, D ** (k - 1 - j))
        return torch.matmul(M.transpose(1, 2).contiguous()[:, None], x).reshape(n, -1)

    def opened(self, A, B, k, j):
        n, D = A.shape[0], self.D
        x = A.reshape(n, self.d * D ** j, D, -1).transpose(1, 2).reshape(n, D, -1)
        y = B.reshape(n, self.d * D ** j, D, -1).transpose(1, 2).reshape(n, D, -1)
        return torch.matmul(x, y.transpose(1, 2).conj())

    def op(self, A, O):
        """O (n, d, d) or (d, d) on the physical index of A (n, d D^k)."""
        return torch.matmul(O, A.reshape(A.shape[0], self.d, -1)).reshape(A.shape)

    def vertex(self, g, m, S=None, ket=None):
        """The unnormalised outgoing messages of group g (n, k, D, D)."""
        k, _, _, ports = g
        A = self.site(g, S)
        K = A if ket is None else ket
        min_ = m[self.rev[ports]]
        out = []
        for j in range(k):
            x = K
            for i in range(k):
                if i != j:
                    x = self.absorb(x, k, i, min_[:, i])
            out.append(self.opened(x, A, k, j))
        return torch.stack(out, 1)

    def sweep(self, m, S=None):
        new = torch.empty_like(m)
        for g in self.groups:
            if g[0]:
                o = self.vertex(g, m, S)
                s = o.sum((2, 3), keepdim=True)
                new = new.index_copy(0, g[3].reshape(-1),
                                     (o / torch.where(s == 0, torch.ones_like(s), s))
                                     .reshape(-1, self.D, self.D))
        return new

    def fidelity(self, new, old):
        a, b = new.reshape(len(new), -1), old.reshape(len(old), -1)
        c = (a.conj() * b).sum(1) / torch.sqrt((a.conj() * a).sum(1) * (b.conj() * b).sum(1))
        return float((1 - c.abs() ** 2).max())

    def solve(self, maxiter, tol):
        m = self.identity()
        for _ in range(maxiter):
            new = self.sweep(m)
            stop = tol > 0 and self.fidelity(new, m) < tol
            m = new
            if stop:
                break
        return m

    def zv(self, m, S=None, O=None):
        z = torch.empty(self.t.nv, device=DEV, dtype=self.dt)
        for g in self.groups:
            A = self.site(g, S)
            x = A if O is None else self.op(A, O[g[1]] if O.dim() == 3 else O)
            for i in range(g[0]):
                x = self.absorb(x, g[0], i, m[self.rev[g[3]]][:, i])
            z = z.index_copy(0, g[1], (x * A.conj()).sum(1))
        return z

    def lognorm(self, m):
        z, q = self.zv(m), torch.arange(self.t.nports, device=DEV)
        pair = q < self.rev
        ze = (m[q[pair]] * m[self.rev[pair]]).sum((1, 2))
        if self.dt == torch.complex128:
            return complex((torch.log(z).sum() - torch.log(ze).sum()).item())
        return float(torch.log(z.abs()).sum() - torch.log(ze.abs()).sum())

    def edges(self, m, ops, S=None):
        """<A_e B_e> of every edge: ops = (first, second), (ne, d, d) or (d, d)."""
        q = torch.arange(self.t.nports, device=DEV)
        lower = q < self.rev
        edge = torch.as_tensor(np.asarray(self.t.port_edge, dtype=np.int64), device=DEV)
        plain, with_op = torch.empty_like(m), torch.empty_like(m)
        for g in self.groups:
            k, _, _, ports = g
            A = self.site(g, S)
            plain = plain.index_copy(0, ports.reshape(-1),
                                     self.vertex(g, m, S).reshape(-1, self.D, self.D))
            for j in range(k):
                p = ports[:, j]
                if ops[0].dim() == 2:
                    O = ops[0]
                else:
                    O = torch.where(lower[p][:, None, None], ops[0][edge[p]], ops[1][edge[p]])
                o = self.vertex(g, m, S, ket=self.op(A, O))[:, j]
                with_op = with_op.index_copy(0, p, o)
        a = (with_op[q[lower]] * with_op[self.rev[lower]]).sum((1, 2))
        b = (plain[q[lower]] * plain[self.rev[lower]]).sum((1, 2))
        return a / b

    def energy(self, m, S, ops_v, ops_e, cv, ce):
        v = (self.zv(m, S, ops_v) / self.zv(m, S)).sum()
        return cv * v + ce * self.edges(m, ops_e, S).sum()

    def energy_and_gradient(self, m, ops_v, ops_e, cv, ce):
        """Energy at the fixed point m and its gradient through the fixed point."""
        S = self.S.clone().requires_grad_(True)
        mm = m.clone().requires_grad_(True)
        E = self.energy(mm, S, ops_v, ops_e, cv, ce)
        gS, gm = torch.autograd.grad(E, (S, mm))
        F = self.sweep(mm, S)
        lam = gm
        for _ in range(300):
            new = torch.autograd.grad(F, mm, lam, retain_graph=True)[0] + gm
            done = float((new - lam).abs().max()) < 1e-13 * float(new.abs().max())
            lam = new
            if done:
                break
        gS = gS + torch.autograd.grad(F, S, lam)[0]
        return float(E.detach()), gS.cpu().numpy()


def _gauge(M):
    w, V = np.linalg.eigh(0.5 * (M + M.T))
    w = np.where(w > 1e-13 * w.max(), w, 0.0)
    r = np.sqrt(w)
    return V * r, np.where(r > 0, V / np.where(r > 0, r, 1.0), 0.0).T


def _on_port(A, j, M):
    return np.moveaxis(np.tensordot(A, M, axes=(j + 1, 0)), -1, j + 1)


def _exact_gates(case, seed, t, s):
    D = case["bond"]
    net = _Net64(t, s)
    m = net.solve(12, -1.0).cpu().numpy()
    A = [s[t.site_off[u]:t.site_off[u + 1]].reshape(t.site_shape(u)) for u in range(t.nv)]
    own, rev, off = t.port_owner(), t.port_rev, t.port_off
    sing = []
    for slots, mats in _gates(t, seed):
        rows = np.zeros((len(slots), D))
        for g, (q, G) in enumerate(zip(slots, mats)):
            Q, R, back = [], [], []
            for u, p in ((own[q], q - off[own[q]]), (own[rev[q]], rev[q] - off[own[rev[q]]])):
                k = A[u].ndim - 1
                others = [j for j in range(k) if j != p]
                X = {j: _gauge(m[rev[off[u] + j]]) for j in others}
                B = A[u]
                for j in others:
                    B = _on_port(B, j, X[j][0])
                B = np.transpose(B, [1 + j for j in others] + [0, 1 + p])
                qq, rr = np.linalg.qr(B.reshape(-1, 2 * D))
                Q.append(qq)
                R.append(rr.reshape(-1, 2, D))
                back.append((u, p, k, others, X))
            th = np.einsum("iab,jcb->iajc", R[0], R[1], optimize=True)
            th = np.einsum("xyac,iajc->ixjy", G.reshape(2, 2, 2, 2), th, optimize=True)
            r1, r2 = len(R[0]), len(R[1])
            U, sv, Vt = np.linalg.svd(th.reshape(2 * r1, 2 * r2), full_matrices=False)
            n = min(D, len(sv))
            sv = sv[:n] / np.linalg.norm(sv[:n])
            rows[g, :n] = sv
            for (u, p, k, others, X), qq, W in zip(back, Q, (U[:, :n], Vt[:n].T)):
                W = np.pad(W * np.sqrt(sv), ((0, 0), (0, D - n)))
                N = (qq @ W.reshape(qq.shape[1], -1)).reshape([D] * len(others) + [2, D])
                perm = [len(others)] + [0] * k
                for a, j in enumerate(others):
                    perm[1 + j] = a
                perm[1 + p] = len(others) + 1
                N = np.transpose(N, perm)
                for j in others:
                    N = _on_port(N, j, X[j][1])
                A[u] = N
            m[q] = m[rev[q]] = np.diag(np.pad(sv, (0, D - n)))
        sing.append(rows)
    net = _Net64(t, np.concatenate([a.ravel() for a in A]))
    mt = torch.as_tensor(m, device=DEV)
    z = torch.tensor([[1.0, 0.0], [0.0, -1.0]], device=DEV, dtype=torch.float64)
    zz = net.zv(mt, O=z) / net.zv(mt)
    return {"singular_values": sing, "messages": m.ravel(), "z": zz.cpu().numpy()}


def _exact_contract(t, s, rows, cols):
    """<psi|psi> site by site: the boundary holds one (ket, bra) pair of indices per cut bond."""
    S = torch.as_tensor(s, device=DEV)
    idx = {v: i for i, v in enumerate(t.vertices)}
    # open bonds of the boundary, in order; state tensor with one axis of size D^2 per bond
    order, state = [], torch.ones((), device=DEV, dtype=torch.float64)
    for v in [(i, j) for i in range(1, rows + 1) for j in range(1, cols + 1)]:
        u = idx[v]
        A = S[t.site_off[u]:t.site_off[u + 1]].reshape(t.site_shape(u))
        k = A.dim() - 1
        E = torch.tensordot(A, A, dims=([0], [0]))
        E = E.permute([x for j in range(k) for x in (j, k + j)])
        E = E.reshape([A.shape[1 + j] ** 2 for j in range(k)])
        edges = [int(t.port_edge[q]) for q in range(t.port_off[u], t.port_off[u + 1])]
        have = [e for e in edges if e in order]
        state = torch.tensordot(state, E, dims=([order.index(e) for e in have],
                                                [edges.index(e) for e in have]))
        order = [e for e in order if e not in have] + [e for e in edges if e not in have]
    return state.reshape(1).cpu().numpy()


def exact(case, seed):
    s = _sites(case, seed)
    tops = _topologies(case)
    t = tops[0]
    if case["path"] == "contract":
        return _exact_contract(t, s, case["rows"], case["cols"])
    if case["path"] == "gates":
        return _exact_gates(case, seed, t, s)
    if case["path"] == "jacobi":
        msgs, logs, off = [], [], 0
        for n in tops:
            net = _Net64(n, s[off:off + int(n.site_off[-1])], case["dtype"] == "c128")
            off += int(n.site_off[-1])
            m = net.solve(case["maxiter"], case["tol"])
            for _ in range(case["polish"]):
                m = net.sweep(m)
            msgs.append(m.reshape(-1).cpu().numpy())
            logs.append(net.lognorm(m))
        return {"messages": np.concatenate(msgs), "lognorm": np.array(logs)}
    net = _Net64(t, s)
    if case["path"] == "sequential":
        A = [s[t.site_off[u]:t.site_off[u + 1]].reshape(t.site_shape(u)) for u in range(t.nv)]
        g = pkg.named_grid((case["rows"], case["cols"]))
        own = t.port_owner()
        m = np.tile(np.eye(case["bond"]), (t.nports, 1, 1))
        for _ in range(case["maxiter"]):
            old = m.copy()
            for uv in pkg.forest_cover_edge_sequence(g):
                q = t.slot(*uv)
                u = own[q]
                p = q - t.port_off[u]
                x = A[u]
                for j in range(x.ndim - 1):
                    if j != p:
                        x = _on_port(x, j, m[t.port_rev[t.port_off[u] + j]])
                axes = [a for a in range(x.ndim) if a != p + 1]
                o = np.tensordot(x, A[u], axes=(axes, axes))
                m[q] = o / o.sum()
            if net.fidelity(torch.as_tensor(m), torch.as_tensor(old)) < case["tol"]:
                break
        mt = torch.as_tensor(m, device=DEV)
        return {"messages": m.ravel(), "lognorm": np.array([net.lognorm(mt)])}
    # tfim, local: the fixed point of the 64-bit map
    m = net.solve(200, 1e-24)
    f = lambda a: torch.as_tensor(a, device=DEV, dtype=torch.float64)  # noqa: E731
    if case["path"] == "tfim":
        z, x = f([[1.0, 0.0], [0.0, -1.0]]), f([[0.0, 1.0], [1.0, 0.0]])
        E, g = net.energy_and_gradient(m, x, (z, z), -3.0, -1.0)
    else:
        ov, oa, ob = (f(a) for a in _operators(t, seed))
        E, g = net.energy_and_gradient(m, ov, (oa, ob), 1.0, 1.0)
    return {"energy": E, "gradient": g}
