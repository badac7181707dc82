"""Performance cases: the calls that programs make on this solver, with inputs
made from a seed, the work that each cannot do without, and 64-bit references
that use nothing of the package.

A case names a structured box (HEXA8 elasticity or heat) cut into subdomains
and one call on it:

  project     P x on device vectors (allocation-free entry point)
  apply_F     the dual operator on host vectors
  apply_prec  the preconditioner on host vectors
  resolve     new nodal loads on a set-up instance: PCG and primal recovery
  block       several nodal load cases solved together on a set-up instance
  reassemble  new element materials on a loaded instance: set-up and solve
  cold        a new instance from the problem description to the solution
  gradient    compliance and its gradient through torch.autograd

Geometry fields: ``domains`` subdomains per direction ("10x10x20"), gathered in
clusters of ``cluster``^3 for the hybrid method, ``elements`` per subdomain and
direction ("10", or "4-14" for boxes of uneven sizes drawn per slab).
"""
import math

import numpy as np
import torch

from espreso_amd import autograd, core

DEV = "cuda" if torch.cuda.is_available() else "cpu"
CORNER = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
POISSON, DENSITY = 0.3, 7850.0


def case(call, physics, domains, elements, method="total", cluster=1, prec="dirichlet", f_store="fp64", sd_store="fp64",
         loads=1):
    return dict(call=call, physics=physics, domains=domains, elements=elements, method=method, cluster=cluster,
                prec=prec, f_store=f_store, sd_store=sd_store, loads=loads)


def listed():
    return [
        # one projector call inside a user's own iteration on a small problem: the smallest call, latency only
        dict(case("project", "elasticity", "4x4x4", "5"), name="project_64x5"),
        # interactive or time-stepping use of a small structure: a new load every call (64 subdomains of 5^3, lumped)
        dict(case("resolve", "elasticity", "4x4x4", "5", prec="lumped"), name="resolve_64x5_lumped"),
        # one solve of a small problem from its description, host preparation included
        dict(case("cold", "elasticity", "4x4x4", "5", prec="lumped"), name="cold_64x5_lumped"),
        # the dual operator called from a program that runs its own Krylov method (512 subdomains of 10^3, hybrid)
        dict(case("apply_F", "elasticity", "8x8x8", "10", "hybrid", 2), name="apply_F_512x10_hybrid"),
        # the next load step of a large structure, hybrid, FP64 operators
        dict(case("resolve", "elasticity", "8x8x8", "10", "hybrid", 2), name="resolve_512x10_hybrid"),
        # the same with the operators kept in FP32 and BF16 (FP64 refinement)
        dict(case("resolve", "elasticity", "8x8x8", "10", "hybrid", 2, f_store="fp32", sd_store="bf16"),
             name="resolve_512x10_mixed"),
        # one source term of a large heat problem with uneven subdomains
        dict(case("resolve", "heat", "10x10x20", "4-14"), name="resolve_heat_2000"),
        # a load-case study: 16 sources on the same heat problem
        dict(case("block", "heat", "10x10x20", "4-14", loads=16), name="block16_heat_2000"),
        # a few load cases on uneven elasticity, an odd number of them
        dict(case("block", "elasticity", "8x8x8", "4-9", loads=5), name="block5_elasticity_512"),
        # material update of a nonlinear or optimisation loop: everything is assembled again (216 subdomains of 12^3)
        dict(case("reassemble", "elasticity", "6x6x6", "12"), name="reassemble_216x12"),
        # the same with uneven subdomains in hybrid clusters
        dict(case("reassemble", "elasticity", "8x8x8", "4-11", "hybrid", 2), name="reassemble_uneven_512"),
        # a design gradient: solve, adjoint solve, element sensitivities (40^3 elements in 64 subdomains)
        dict(case("gradient", "elasticity", "4x4x4", "10"), name="gradient_64x10"),
    ]


def draw(rng):
    call = rng.choice(["project", "apply_F", "apply_prec", "resolve", "resolve", "block", "block", "reassemble",
                       "reassemble", "cold", "gradient"])
    physics = "elasticity" if call == "gradient" or rng.random() < 0.65 else "heat"
    n = round(math.exp(rng.uniform(math.log(2), math.log(8))))  # subdomains per direction, 8 to 512 in all
    dom = [n, max(2, n - rng.randrange(2)), n]
    top = 11 if physics == "elasticity" else 14
    if call in ("cold", "gradient"):
        top = 8  # host preparation included: kept to what is solved interactively
    lo = rng.randint(3, top)
    elements = "%d" % lo if rng.random() < 0.5 else "%d-%d" % (max(3, lo - 4), lo)
    method, cluster = "total", 1
    if call != "gradient" and n % 2 == 0 and dom[1] % 2 == 0 and rng.random() < 0.4:
        method, cluster = "hybrid", 2
    prec = rng.choice(["dirichlet", "dirichlet", "lumped"])
    f_store, sd_store = "fp64", "fp64"
    if call == "resolve" and rng.random() < 0.3:
        f_store, sd_store = rng.choice([("fp32", "bf16"), ("fp32", "fp64"), ("fp64", "bf16")])
    loads = rng.randint(2, 16) if call == "block" else 1
    return case(call, physics, "%dx%dx%d" % tuple(dom), elements, method, cluster, prec, f_store, sd_store, loads)


# ---------------------------------------------------------------- problems ----
def domains_of(c):
    return [int(v) for v in c["domains"].split("x")]


def slabs_of(c):
    """Elements of every subdomain slab per direction (the uneven ones from a fixed seed: part of the case)."""
    ends = [int(v) for v in c["elements"].split("-")]
    rng = np.random.default_rng(20261203)
    return [[int(v) for v in rng.integers(ends[0], ends[-1] + 1, size=n)] for n in domains_of(c)]


def lengths_of(c):
    dom = domains_of(c)
    return tuple(n / dom[0] for n in dom)


def material_of(c, seed):
    """Per-element modulus (scatter of 10 % around steel) or conductivity (0.1 to 10 per subdomain), x fastest."""
    rng = np.random.default_rng([seed, 1])
    sl = slabs_of(c)
    if c["physics"] == "elasticity":
        return 2.1e11 * np.exp(0.1 * rng.standard_normal(int(np.prod([sum(v) for v in sl]))))
    k = 10.0 ** rng.uniform(-1.0, 1.0, size=[len(v) for v in sl[::-1]])
    for axis, v in enumerate(sl[::-1]):
        k = np.repeat(k, v, axis=axis)
    return np.ascontiguousarray(k).reshape(-1)


def accel_of(seed):
    rng = np.random.default_rng([seed, 2])
    return tuple(float(v) for v in rng.uniform(-1.0, 1.0, 3) + (0.0, 0.0, -9.81))


def spec_of(c, seed):
    dom, k = domains_of(c), c["cluster"]
    spec = dict(physics=0 if c["physics"] == "elasticity" else 1, clusters=tuple(n // k for n in dom),
                domains=(k, k, k), elements=(1, 1, 1), slab_elements=tuple(tuple(v) for v in slabs_of(c)),
                length=lengths_of(c), poisson=POISSON, density=DENSITY, heat_source=1.0,
                material_elem=material_of(c, seed))
    if c["physics"] == "elasticity":
        spec.update(fixed=(0, 0, 0, 0, 7, 0), accel=accel_of(seed))
    else:
        spec.update(fixed=(0, 0, 0, 0, 1, 0))
    return spec


def options_of(c):
    # solved to 1e-10, so that the solutions are good for the nine digits that programs compare them to
    return dict(method=c["method"], preconditioner=c["prec"], sc_precision=c["f_store"], sd_precision=c["sd_store"],
                precision=1e-10, max_iterations=1000)


def loads_of(c, seed):
    """Nodal load cases, U(-1, 1) (loads, nodes, components)."""
    nn = np.prod([sum(v) + 1 for v in slabs_of(c)])
    nd = 3 if c["physics"] == "elasticity" else 1
    return np.random.default_rng([seed, 3]).uniform(-1.0, 1.0, size=(c["loads"], int(nn), nd))


def prepare(c, seed):
    call = c["call"]
    if call == "cold":
        return dict(call=call, spec=spec_of(c, seed), options=options_of(c))
    if call == "gradient":
        spec = spec_of(c, seed)
        young = torch.from_numpy(spec.pop("material_elem")).to(DEV).requires_grad_(True)
        return dict(call=call, spec=spec, options=options_of(c), young=young)
    solver = core.GridFETI(spec_of(c, seed), **options_of(c))
    solver.setup()
    state = dict(call=call, solver=solver)
    if call == "project":
        x = np.random.default_rng([seed, 4]).standard_normal(solver.n_lambda)
        state.update(x=torch.from_numpy(x).to(DEV), y=torch.empty(solver.n_lambda, dtype=torch.float64, device=DEV))
    elif call in ("apply_F", "apply_prec"):
        state.update(x=np.random.default_rng([seed, 4]).standard_normal(solver.n_lambda))
    elif call in ("resolve", "block"):
        state.update(loads=loads_of(c, seed))
    elif call == "reassemble":
        state.update(material=material_of(c, seed + 7919))
    return state


def run(state):
    call = state["call"]
    if call == "cold":
        with core.GridFETI(state["spec"], **state["options"]) as solver:
            solver.setup()
            solver.solve()
            return solver.nodal_solution()
    if call == "gradient":
        young = state["young"]
        young.grad = None
        value = autograd.compliance(young, dict(state["spec"]), **state["options"])
        value.backward()
        return value.detach(), young.grad
    solver = state["solver"]
    if call == "project":
        solver.project_device(state["x"].data_ptr(), state["y"].data_ptr())
        return state["y"]
    if call == "apply_F":
        return solver.apply_F(state["x"])
    if call == "apply_prec":
        return solver.apply_prec(state["x"])
    if call == "resolve":
        solver.set_nodal_rhs(state["loads"][0])
        solver.resolve()
        return solver.nodal_solution()
    if call == "block":
        u, _, _ = solver.resolve_block_nodal(state["loads"])
        return list(u)
    solver.update_material(state["material"])
    solver.setup()
    solver.solve()
    return solver.nodal_solution()


# -------------------------------------------------------------------- work ----
def sizes_of(c):
    """(interface DOFs m, interior DOFs n, entries of K) of every subdomain: the interface is what touches another
    subdomain or the fixed face z = 0."""
    nd = 3 if c["physics"] == "elasticity" else 1
    sl = slabs_of(c)
    out = []
    for z, ez in enumerate(sl[2]):
        for y, ey in enumerate(sl[1]):
            for x, ex in enumerate(sl[0]):
                e, at, n = (ex, ey, ez), (x, y, z), [len(v) for v in sl]
                free = 1
                for d in range(3):
                    free *= max(0, e[d] + 1 - (at[d] > 0 or d == 2) - (at[d] < n[d] - 1))
                nodes = np.prod([v + 1 for v in e])
                out.append((nd * int(nodes - free), nd * free, nd * nd * int(np.prod([3 * v + 1 for v in e])),
                            nd * (min(e[0], e[1], e[2]) + 1) ** 2))
    return out


def work(c):
    store = {"fp64": 8, "fp32": 4, "bf16": 2}
    s = sizes_of(c)
    tri = sum(m * (m + 1) / 2 for m, _, _, _ in s)
    f_bytes = tri * store[c["f_store"]]
    p_bytes = tri * store[c["sd_store"]] if c["prec"] == "dirichlet" else 12 * 27 * sum(m for m, _, _, _ in s)
    lam = 1.2 * sum(m for m, _, _, _ in s) / 2  # multipliers: a little over one per pair of interface DOFs
    dofs = sum(m + n for m, n, _, _ in s)
    k_bytes = 8 * sum(k for _, _, k, _ in s) / 2  # K is symmetric: one triangle
    # iterations of the stop test as met in earnest (they grow with the clusters' coarseness, not with the size)
    iters = 110 if c["method"] == "hybrid" else 45
    nc = len(s) * (6 if c["physics"] == "elasticity" else 1) / c["cluster"] ** 3
    band = sum(8 * n * b for _, n, _, b in s)  # the factor of K_ii
    solve = iters * (f_bytes + p_bytes + 8 * nc * nc) + 2 * band + 8 * 4 * dofs
    # banded Cholesky, its substitution, S, the inverse of S
    asm_flops = sum(n * b * b + 2 * n * b * m + n * m * m + float(m) ** 3 for m, n, _, b in s)
    asm_bytes = k_bytes + 8 * tri + (f_bytes if c["f_store"] != "fp64" else 0) + p_bytes + band
    flops_solve = iters * 4 * tri * (2 if c["prec"] == "dirichlet" else 1)
    call = c["call"]
    if call == "project":
        return dict(bytes=8 * (2 * lam + nc * nc + sum(m for m, _, _, _ in s) * (6 if c["physics"] == "elasticity" else 1)),
                    flops=2 * nc * nc)
    if call == "apply_F":
        return dict(bytes=f_bytes + 16 * lam, flops=4 * tri)
    if call == "apply_prec":
        return dict(bytes=p_bytes + 16 * lam, flops=4 * tri)
    if call == "resolve":
        return dict(bytes=solve, flops=flops_solve)
    if call == "block":
        k = c["loads"]
        return dict(bytes=solve + k * 8 * (iters * 2 * lam + 4 * dofs), flops=k * flops_solve)
    if call == "gradient":
        return dict(bytes=asm_bytes + 2 * solve, flops=asm_flops + 2 * flops_solve)
    return dict(bytes=asm_bytes + solve, flops=asm_flops + flops_solve)


# ------------------------------------------------------------------- exact ----
def unit_element(c):
    """Element matrix for a modulus or conductivity of 1, 2 x 2 x 2 Gauss points (node-major, corner order CORNER)."""
    h = [length / sum(v) for length, v in zip(lengths_of(c), slabs_of(c))]
    g = 0.5 / math.sqrt(3.0)
    nd = 3 if c["physics"] == "elasticity" else 1
    K = np.zeros((8 * nd, 8 * nd))
    lam, mu = POISSON / ((1 + POISSON) * (1 - 2 * POISSON)), 0.5 / (1 + POISSON)
    D = np.zeros((6, 6))
    D[:3, :3] = lam
    D += np.diag([2 * mu] * 3 + [mu] * 3)
    for q in np.ndindex(2, 2, 2):
        t = [0.5 - g + 2 * g * v for v in q]
        dN = np.zeros((3, 8))
        for a, corner in enumerate(CORNER):
            N = [t[d] if corner[d] else 1 - t[d] for d in range(3)]
            for d in range(3):
                dN[d, a] = np.prod([N[e] for e in range(3) if e != d]) * (1 if corner[d] else -1) / h[d]
        if nd == 1:
            K += dN.T @ dN * np.prod(h) / 8
            continue
        B = np.zeros((6, 24))
        for d in range(3):
            B[d, d::3] = dN[d]
        for row, (i, j) in enumerate(((0, 1), (1, 2), (0, 2))):
            B[3 + row, i::3], B[3 + row, j::3] = dN[j], dN[i]
        K += B.T @ D @ B * np.prod(h) / 8
    return torch.from_numpy(K).to(DEV)


class Mesh:
    """The undecomposed problem: K u by elements and a Jacobi-preconditioned CG."""

    def __init__(self, c, material):
        self.ne = [sum(v) for v in slabs_of(c)][::-1]  # z, y, x
        self.nd = 3 if c["physics"] == "elasticity" else 1
        self.K = unit_element(c)
        self.E = torch.from_numpy(np.ascontiguousarray(material)).to(DEV)
        one = self.scatter(self.E * torch.diagonal(self.K)[:, None])
        self.free = torch.ones_like(one)
        self.free[:, 0] = 0.0  # the face z = 0 is held
        self.jacobi = self.free / one

    def corner(self, u, a):
        x, y, z = CORNER[a]
        nz, ny, nx = self.ne
        return u[:, z:z + nz, y:y + ny, x:x + nx]

    def gather(self, u):
        return torch.stack([self.corner(u, a)[i].reshape(-1) for a in range(8) for i in range(self.nd)])

    def scatter(self, v):
        out = torch.zeros([self.nd] + [n + 1 for n in self.ne], dtype=torch.float64, device=DEV)
        v = v.reshape([8, self.nd] + self.ne)
        for a in range(8):
            self.corner(out, a).add_(v[a])
        return out

    def apply(self, u):
        return self.free * self.scatter((self.K @ self.gather(u)).mul_(self.E))

    def solve(self, f, digits=1e-13):
        """f and the result as (nd, z, y, x) fields."""
        r = self.free * f
        x, z = torch.zeros_like(r), self.jacobi * r
        p, rz, stop = z.clone(), (r * z).sum(), digits * r.norm()
        for i in range(20000):
            q = self.apply(p)
            alpha = rz / (p * q).sum()
            x.add_(alpha * p)
            r.sub_(alpha * q)
            if i % 16 == 15 and r.norm() < stop:
                break
            z = self.jacobi * r
            old, rz = rz, (r * z).sum()
            p = z + (rz / old) * p
        return x

    def field(self, nodal):
        """(nodes, nd), x fastest, to a field."""
        return torch.from_numpy(nodal).to(DEV).reshape([n + 1 for n in self.ne] + [self.nd]).permute(3, 0, 1, 2)

    def nodal(self, u):
        return u.permute(1, 2, 3, 0).reshape(-1, self.nd)


def body_load(c, mesh, seed):
    h = [length / sum(v) for length, v in zip(lengths_of(c), slabs_of(c))]
    per_node = float(np.prod(h)) / 8
    force = [DENSITY * a for a in accel_of(seed)] if mesh.nd == 3 else [1.0]
    one = torch.tensor(force * 8, dtype=torch.float64, device=DEV) * per_node
    return mesh.scatter(one[:, None].expand(-1, mesh.E.numel()))


def exact_projection(c, seed):
    """P x for one coarse block per subdomain: G from the multiplier rows (held DOFs by global DOF, then the redundant
    gluing rows by global DOF and pair of subdomains) and the rigid motions at the nodes."""
    sl, dom = slabs_of(c), domains_of(c)
    off = [np.concatenate([[0], np.cumsum(v)]) for v in sl]
    h = [length / sum(v) for length, v in zip(lengths_of(c), sl)]
    nd = 3 if c["physics"] == "elasticity" else 1
    own = [[[i for i in range(len(v)) if o[i] <= g <= o[i + 1]] for g in range(o[-1] + 1)] for v, o in zip(sl, off)]
    first, second = [], []  # rows: (subdomain, node, component, sign) per entry
    for gz in range(off[2][-1] + 1):
        for gy in range(off[1][-1] + 1):
            for gx in range(off[0][-1] + 1):
                subs = [x + dom[0] * (y + dom[1] * z) for z in own[2][gz] for y in own[1][gy] for x in own[0][gx]]
                at = (gx, gy, gz)
                if gz == 0:
                    first += [[(s, at, i, 1.0)] for i in range(nd) for s in subs]
                elif len(subs) > 1:
                    second += [[(a, at, i, 1.0), (b, at, i, -1.0)] for i in range(nd) for k, a in enumerate(subs)
                               for b in subs[k + 1:]]
    rows = first + second
    k = 6 if nd == 3 else 1
    G = np.zeros((len(rows), k * int(np.prod(dom))))
    for row, entries in enumerate(rows):
        for s, at, i, sign in entries:
            S = (s % dom[0], s // dom[0] % dom[1], s // (dom[0] * dom[1]))
            X = [(at[d] - 0.5 * (off[d][S[d]] + off[d][S[d] + 1])) * h[d] * dom[d] for d in range(3)]
            modes = [1.0] if nd == 1 else [float(i == 0), float(i == 1), float(i == 2), (-X[1], X[0], 0.0)[i],
                                           (-X[2], 0.0, X[0])[i], (0.0, -X[2], X[1])[i]]
            G[row, k * s:k * s + k] += sign * np.array(modes)
    x = np.random.default_rng([seed, 4]).standard_normal(len(rows))
    Q, _ = np.linalg.qr(G)
    return x - Q @ (Q.T @ x)


def exact(c, seed):
    call = c["call"]
    if call in ("apply_F", "apply_prec"):
        return None  # F depends on the generalised inverse that is taken, the preconditioner on its storage
    if call == "project":
        small = sum(m for m, _, _, _ in sizes_of(c)) < 40000 and len(sizes_of(c)) <= 64
        return exact_projection(c, seed) if small and c["method"] == "total" else None
    mesh = Mesh(c, material_of(c, seed + 7919 if call == "reassemble" else seed))
    if call in ("resolve", "block"):
        loads = loads_of(c, seed)
        known = 2 if call == "block" else 1  # of a block, two load cases: a CG for each takes its time
        u = [mesh.nodal(mesh.solve(mesh.field(g))) for g in loads[:known]]
        return u[0] if call == "resolve" else u + [None] * (len(loads) - known)
    f = body_load(c, mesh, seed)
    u = mesh.solve(f)
    if call == "gradient":
        ue = mesh.gather(u)
        return (f * u).sum(), -((mesh.K @ ue) * ue).sum(0)
    return mesh.nodal(u)
