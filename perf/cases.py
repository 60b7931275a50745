"""Performance cases: the work a user of this library has it do, through its
public entry points, and the same results in plain 64-bit torch.

A case names what is called ("call"), the formulation, the cell type, the H1
order k and test degree kt of the cells, the mesh, and how the caller's
program uses the library: `tuned` programs assemble the same mesh over and
over (they autotune the plan once and keep the output buffers, as the
benchmark does), the others take a plan as it comes.

  assemble   local_stiffness_and_rhs: K, rhs, Schur complement (and G)
  gradient   the forward assembly with the factorisation kept, then the energy
             error and its gradient in the cells' coefficients
  graph      all element types of an hp mesh in one captured launch
  eta        the energy error of a given solution
  recover    the field unknowns from a condensed solution
  solve      the condensed global system: assembly and block-Jacobi CG
"""
import math

import numpy as np
import torch

from camellia2_amd import capi, dpg

TOPOLOGY = {"quad": capi.QUAD, "hex": capi.HEX, "tri": capi.TRI}
DEV = "cuda:0"
GIB = 2.0 ** 30


def _mesh_case(name, call, form, cells, k, kt, **options):
    return dict(name=name, call=call, form=form, cells="x".join(map(str, cells)), k=k, kt=kt, tuned=False, gram=False,
                **options)


def listed():
    tuned = lambda c: dict(c, tuned=True)  # noqa: E731
    return [
        # a handful of cells (the unrefined mesh a program starts from, a smoke test): latency
        _mesh_case("poisson2d 4x4 p2", "assemble", "poisson2d", (4, 4), 3, 4),
        # the 16 x 16 Poisson workload of the benchmark, with the Gram matrix as an output
        dict(_mesh_case("poisson2d 16x16 p2 gram", "assemble", "poisson2d", (16, 16), 3, 4), gram=True),
        # a small 3D mesh of odd sizes, between latency and throughput
        _mesh_case("poisson3d 5x4x3 p2", "assemble", "poisson3d", (5, 4, 3), 3, 4),
        # the Stokes workload of the benchmark (p = 3, test degree 5) on a quarter of its mesh
        tuned(_mesh_case("stokes2d 64x64 p3", "assemble", "stokes2d", (64, 64), 4, 5)),
        # the 3D Poisson workload of the benchmark (p = 3, test degree 5) on an eighth of its mesh
        tuned(_mesh_case("poisson3d 16x16x16 p3", "assemble", "poisson3d", (16, 16, 16), 4, 5)),
        # the differentiation workload: per-cell coefficients, forward, energy error and gradient
        tuned(_mesh_case("cdr2d 64x64 p2 gradient", "gradient", "cdr2d", (64, 64), 3, 4)),
        # an adaptive mesh: quads and triangles, p = 1..6, test degree p+1..p+3, 36 element types (graded
        # less than the benchmark's, whose finest cells leave no digits to compare in 64 bits)
        dict(name="hp convection 1500 cells", call="graph", form="cd2d", ncells=1500, levels=1, pmax=6, dpmax=3),
        # error estimation after a solve on a 3D mesh
        _mesh_case("eta poisson3d 9x8x7 p2", "eta", "poisson3d", (9, 8, 7), 3, 4),
        # the fields of a condensed 3D solution
        _mesh_case("recover poisson3d 11x10x9 p2", "recover", "poisson3d", (11, 10, 9), 3, 4),
        # the global condensed system of a 2D mesh: assembly and solve to 1e-10
        _mesh_case("solve poisson2d 48x41 p2", "solve", "poisson2d", (48, 41), 3, 4),
    ]


def draw(rng):
    largest = max((work(c) for c in listed()), key=lambda w: w["flops"])
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= largest["flops"] and w["bytes"] <= largest["bytes"]:
            return case


def _draw(rng):
    spread = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    call = rng.choice(["assemble", "assemble", "assemble", "gradient", "graph", "eta", "recover", "solve"])
    if call == "graph":
        return dict(call=call, form="cd2d", ncells=spread(150, 3000), levels=rng.randint(0, 1), pmax=rng.randint(3, 6),
                    dpmax=rng.randint(2, 3))
    forms = {"assemble": ["poisson2d", "stokes2d", "poisson3d", "cdr2d"], "gradient": ["cdr2d"],
             "solve": ["poisson2d"]}.get(call, ["poisson2d", "poisson3d", "stokes2d"])
    form = rng.choice(forms)
    if form == "poisson3d":
        k = rng.randint(2, 4)
        cells = [spread(2, 16) for _ in range(3)]
    else:
        k = rng.randint(2, 4 if call in ("gradient", "solve") else 5)
        cells = [spread(*((12, 64) if call == "solve" else (3, 64))) for _ in range(2)]
    kt = k + rng.randint(1, 2 if form != "poisson3d" and call != "gradient" else 1)
    c = _mesh_case("", call, form, cells, k, kt)
    del c["name"]
    if call in ("assemble", "gradient"):
        c["tuned"] = rng.random() < 0.5
        c["gram"] = call == "assemble" and not c["tuned"] and rng.random() < 0.25
    return c


# ------------------------------------------------------------------------- sizes
# (kind, components) of the trial variables, test spaces, all in order
SPACES = {
    "poisson2d": (2, ["field", "vector", "trace", "flux"], ["grad", "div"]),
    "poisson3d": (3, ["field", "vector", "trace", "flux"], ["grad", "div"]),
    "cdr2d": (2, ["field", "vector", "trace", "flux"], ["grad", "div"]),
    "cd2d": (2, ["field", "vector", "trace", "flux"], ["grad", "div"]),
    "stokes2d": (2, ["field"] * 7 + ["trace"] * 2 + ["flux"] * 2, ["grad", "grad", "div", "div", "grad"]),
}
NCOEFS = {"cdr2d": 4, "cd2d": 3}


def sizes(form, topology, k, kt):
    """(test dofs N, trial dofs M, of them field dofs F) of one cell."""
    dim, trial, test = SPACES[form]
    nsides = {"quad": 4, "hex": 6, "tri": 3}[topology]
    tri = topology == "tri"
    nf = k * (k + 1) // 2 if tri else k ** dim
    F = sum(nf * (dim if t == "vector" else 1) for t in trial if t in ("field", "vector"))
    T = nsides * sum((k + 1) ** (dim - 1) if t == "trace" else k ** (dim - 1) for t in trial if t in ("trace", "flux"))
    grad = (kt + 1) * (kt + 2) // 2 if tri else (kt + 1) ** dim
    div = kt * (kt + 2) if tri else dim * (kt + 1) * kt ** (dim - 1)
    return sum(grad if t == "grad" else div for t in test), F + T, F


def work(case):
    """Inputs read and outputs written once; the factorisations and triangular
    solves, and for every entry of G (lower) and B one sum over the points of one
    direction (the last step of a sum-factorised contraction)."""
    call, form = case["call"], case["form"]
    nc = NCOEFS.get(form, 0)
    if call == "graph":
        groups = [(g["topology"], g["k"], g["kt"], g["ncells"]) for g in _hp_types(case, 1)]
    else:
        topology = "hex" if form == "poisson3d" else "quad"
        groups = [(topology, case["k"], case["kt"], int(np.prod(_shape(case))))]
    total = {"bytes": 0.0, "flops": 0.0}
    for topology, k, kt, C in groups:
        N, M, F = sizes(form, topology, k, kt)
        T = M - F
        nverts, nsides, dim = {"quad": (4, 4, 2), "hex": (8, 6, 3), "tri": (3, 3, 2)}[topology]
        inputs = 8 * (nverts * dim + nc) + nsides
        contract = (kt + 1) * N * (N + 1) + 2 * (kt + 1) * N * (M + 1)
        factor, solve = N ** 3 / 3, N * N * (M + 1)
        schur = F ** 3 / 3 + F * F * (T + 1) + F * T * (T + 1)
        if call in ("assemble", "graph", "gradient"):
            b = inputs + 8 * (M * M + M + T * T + T + (N * N if case.get("gram") else 0))
            fl = contract + factor + solve + N * M * (M + 1) + schur
            if call == "gradient":  # the residual, one back solve, the sums over the points; u, eta, gradient
                b += 8 * (M + 1 + nc)
                fl += 2 * N * M + N * N + 2 * N * M
        elif call == "eta":
            b = inputs + 8 * (M + 1)
            fl = contract + factor + 2 * N * M + N * N
        elif call == "recover":
            b = 8 * (M * F + F + M + F)
            fl = F ** 3 / 3 + 2 * F * F + 2 * F * T
        else:  # the blocks in, the matrix and the vectors out, one product with the matrix
            b = 8 * (2 * T * T + 3 * T)
            fl = 3 * T * T
        total["bytes"] += float(C * b)
        total["flops"] += float(C * fl)
    return total


# ------------------------------------------------------------------------ inputs
def _shape(case):
    return [int(n) for n in case["cells"].split("x")]


def _grid(shape, jitter, rng):
    """Vertices (C, V, d) and side parities (C, S) of a jittered grid of quads or
    hexes in the unit box, cells x fastest; +1 on the boundary and on the side of
    the lower cell."""
    dim = len(shape)
    axes = [np.arange(n + 1) / n for n in shape]
    X = np.stack(np.meshgrid(*axes, indexing="ij"), axis=-1)
    inner = (slice(1, -1),) * dim
    X[inner] += rng.uniform(-jitter, jitter, X[inner].shape) / np.array(shape)
    corner = {2: [(0, 0), (1, 0), (1, 1), (0, 1)],
              3: [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]}[dim]
    order = tuple(reversed(range(dim)))  # x fastest
    nodes = np.stack([X[tuple(slice(o, o + n) for o, n in zip(c, shape))].transpose(order + (dim,)).reshape(-1, dim)
                      for c in corner], axis=1)
    index = np.stack(np.meshgrid(*[np.arange(n) for n in shape], indexing="ij"), axis=-1)
    index = index.transpose(order + (dim,)).reshape(-1, dim)
    low = np.where(index == 0, 1, -1)  # parity of the low side of each direction; the high sides are +1
    one = np.ones(len(index), dtype=int)
    sides = [low[:, 1], one, one, low[:, 0]] + ([low[:, 2], one] if dim == 3 else [])
    return np.ascontiguousarray(nodes), np.stack(sides, axis=1).astype(np.int8)


def _load(dim, ncomp, nmodes, rng):
    """Sine modes: amplitudes N(0, 1), wave numbers 1..6, per load component."""
    return [(rng.standard_normal(nmodes), rng.integers(1, 7, (nmodes, dim))) for _ in range(ncomp)]


def _load_desc(load):
    d = capi.LoadDesc()
    d.ncomp = len(load)
    for c, (amp, waves) in enumerate(load):
        d.nmodes[c] = len(amp)
        for m in range(len(amp)):
            d.amp[c][m] = float(amp[m])
            for e in range(waves.shape[1]):
                d.k[c][m][e] = int(waves[m, e])
    return d


def _coefs(form, C, rng):
    """Per-cell coefficients of the benchmark's workloads: diffusion log-uniform,
    one convection direction for the mesh (with reaction: its size per cell)."""
    if form not in NCOEFS:
        return None
    angle = rng.uniform(0.0, 2.0 * np.pi)
    if form == "cdr2d":
        eps, size = 10.0 ** rng.uniform(-3.0, 0.0, C), rng.uniform(0.5, 2.0, C)
        return np.stack([eps, size * np.cos(angle), size * np.sin(angle), rng.uniform(0.0, 1.0, C)], axis=1)
    eps = 10.0 ** rng.uniform(-4.0, -2.0, C)
    return np.stack([eps, np.full(C, np.cos(angle)), np.full(C, np.sin(angle))], axis=1)


def _hp_types(case, seed):
    """The element types of an hp mesh graded toward one side (cells of level l
    have edge 2^-l / 16, each level twice as many as the one before; one cell in
    eight is two triangles) with a degree and an enrichment per cell: dicts with
    the type and its cells' arrays, most work per cell first."""
    C = case["ncells"]
    kinds = np.random.default_rng(C)  # the types and their sizes are the case's, the cells the seed's
    p, dp = kinds.integers(1, case["pmax"] + 1, C), kinds.integers(1, case["dpmax"] + 1, C)
    split = kinds.uniform(size=C) < 0.125
    rng = np.random.default_rng([seed, 3])
    share = 2.0 ** np.arange(case["levels"] + 1)
    level = rng.choice(len(share), C, p=share / share.sum())
    h = 2.0 ** -level / 16
    at = np.floor(rng.uniform(0.0, 1.0, (C, 2)) / h[:, None]) * h[:, None]
    corner = np.array([(0, 0), (1, 0), (1, 1), (0, 1)]) + rng.uniform(-0.05, 0.05, (C, 4, 2))
    nodes = at[:, None, :] + h[:, None, None] * corner
    par = rng.choice(np.array([-1, 1], dtype=np.int8), (C, 4))
    coefs = _coefs("cd2d", C, rng)
    types = []
    for topology, mine in (("quad", ~split), ("tri", split)):
        for a, b in sorted(set(zip(p[mine].tolist(), dp[mine].tolist()))):
            i = np.flatnonzero(mine & (p == a) & (dp == b))
            n, q, c = nodes[i], par[i], coefs[i]
            if topology == "tri":
                one = np.ones(len(i), dtype=np.int8)
                n = np.concatenate([n[:, [0, 1, 2]], n[:, [0, 2, 3]]])
                q = np.concatenate([np.stack([q[:, 0], q[:, 1], one], 1), np.stack([-one, q[:, 2], q[:, 3]], 1)])
                c = np.concatenate([c, c])
            types.append(dict(topology=topology, k=a + 1, kt=a + b, nodes=n, parities=q, coefs=c, ncells=len(n)))
    types.sort(key=lambda t: (-(t["kt"] + t["k"]), -t["k"], t["topology"]))
    return types


def _inputs(case, seed):
    """Host arrays of a mesh case."""
    form = case["form"]
    rng = np.random.default_rng([seed, 1])
    shape = _shape(case)
    nodes, par = _grid(shape, 0.05 if len(shape) == 3 else 0.10, rng)
    C = len(nodes)
    load = _load(len(shape), 2 if form == "stokes2d" else 1, 16 if len(shape) == 3 else 8, rng)
    _, M, _ = sizes(form, "hex" if len(shape) == 3 else "quad", case["k"], case["kt"])
    u = rng.standard_normal((C, M)) if case["call"] in ("gradient", "eta", "recover") else None
    return nodes, par, _coefs(form, C, rng), load, u


# ------------------------------------------------------- what a user's program does
LIBRARY_FORM = {"poisson2d": ("poisson", 2), "poisson3d": ("poisson", 3), "stokes2d": ("stokes", 2),
                "cdr2d": ("cdr", 2), "cd2d": ("cd", 2)}


def _dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _arena(types):
    """The outputs of all types of one topology in one buffer each, and the types' parts of them."""
    views = []
    for t in types:
        N, M, F = sizes("cd2d", t["topology"], t["k"], t["kt"])
        T, C = M - F, t["ncells"]
        views.append({"K": (C, M, M), "rhs": (C, M), "schur": (C, T, T), "schur_rhs": (C, T), "info": (C,)})
    arena = {}
    for topology in sorted({t["topology"] for t in types}):
        mine = [v for t, v in zip(types, views) if t["topology"] == topology]
        arena[topology] = {}
        for key in ("K", "rhs", "schur", "schur_rhs", "info"):
            counts = [math.prod(v[key]) for v in mine]
            buffer = torch.zeros(sum(counts), dtype=torch.int32 if key == "info" else torch.float64, device=DEV)
            arena[topology][key] = buffer
            for v, part in zip(mine, buffer.split(counts)):
                v[key] = part.view(v[key])
    return arena, views


def prepare(case, seed):
    form = dpg.form(*LIBRARY_FORM[case["form"]])
    if case["call"] == "graph":
        types = _hp_types(case, seed)
        load = _load_desc(_load(2, 1, 8, np.random.default_rng([seed, 2])))
        A = dpg.LocalAssembler(form, [dpg.bucket(TOPOLOGY[t["topology"]], t["k"], t["kt"]) for t in types])
        arena, views = _arena(types)
        items = []
        for b, t in enumerate(types):
            n, p, c = _dev(t["nodes"]), _dev(t["parities"]), _dev(t["coefs"])
            A.autotune(b, n, p, c, load, sample=512)
            items.append(dict(bucket=b, nodes=n, parities=p, coefs=c, load=load, want_schur=True, out=views[b]))
        return dict(case=case, assembler=A, graph=dpg.AssemblyGraph(A, items, lanes=4), arena=arena)
    nodes, par, coefs, load, u = _inputs(case, seed)
    bucket = dpg.bucket(capi.HEX if len(_shape(case)) == 3 else capi.QUAD, case["k"], case["kt"])
    s = dict(case=case, nodes=_dev(nodes), par=_dev(par), coefs=_dev(coefs), load=_load_desc(load), u=_dev(u), out=None)
    if case["call"] == "solve":
        # the blocks a local assembly hands over, here from the plain evaluation below
        ref = _reference(case["form"], case["k"], case["kt"], nodes, par, coefs, load)
        ids = dpg.vertex_ids(nodes)
        gdof, n = dpg.skeleton_numbering(form, bucket, ids)
        s["system"] = dpg.CondensedSystem(gdof, n)
        entity, count = dpg.skeleton_entities(form, bucket, ids, n)
        s["system"].set_blocks(entity, count)
        s["fixed"] = _dev(dpg.boundary_trace_mask(form, bucket, gdof, ids, n))
        s["schur"], s["schur_rhs"] = ref["schur"].contiguous(), ref["schur_rhs"].contiguous()
        return s
    s["assembler"] = A = dpg.LocalAssembler(form, [bucket], workspace_bytes=32 * GIB if case["tuned"] else 0.0)
    if case["call"] == "recover":
        ref = _reference(case["form"], case["k"], case["kt"], nodes, par, coefs, load)
        s["K"], s["rhs"] = ref["K"].contiguous(), ref["rhs"].contiguous()
    if case["tuned"]:
        A.autotune(0, s["nodes"], s["par"], s["coefs"], s["load"], sample=min(len(nodes), 512))
        s["out"] = {}
    return s


def run(state):
    case, A = state["case"], state.get("assembler")
    call = case["call"]
    if call == "graph":
        state["graph"].launch()
        return state["arena"]
    if call == "solve":
        S = state["system"]
        values, rhs = S.assemble(state["schur"], state["schur_rhs"])
        x = torch.zeros(S.nglobal, dtype=torch.float64, device=DEV)
        S.solve(values, rhs, state["fixed"], x, tol=1e-10, maxit=8000)
        return {"values": values, "rhs": rhs, "x": x}
    if call == "recover":
        u = state["u"].clone()  # the condensed solution; its field part is written
        A.recover_fields(0, state["K"], state["rhs"], u)
        return u
    mesh = (0, state["nodes"], state["par"])
    if call == "eta":
        return A.energy_error(*mesh, state["u"], state["coefs"], state["load"])
    gradient = call == "gradient"
    out, _ = A.local_stiffness_and_rhs(*mesh, state["coefs"], state["load"], want_G=case["gram"], want_schur=True,
                                       want_info=not case["tuned"], out=state["out"], want_factor=gradient)
    result = {k: out[k] for k in ("K", "rhs", "schur", "schur_rhs") + (("G",) if case["gram"] else ())}
    if gradient:
        result["eta2"], result["grad"] = A.adjoint(*mesh, state["coefs"], state["load"], u=state["u"],
                                                   factor=out["factor"], factor_scale=out["factor_scale"],
                                                   want_eta2=True)
    return result


# -------------------------------------------------------- the same in plain torch
def exact(case, seed):
    call = case["call"]
    if call == "solve":
        return None  # the order of the global unknowns and of the matrix entries is the library's own
    if call == "graph":
        load = _load(2, 1, 8, np.random.default_rng([seed, 2]))
        keys = ("K", "rhs", "schur", "schur_rhs")
        types = _hp_types(case, seed)
        quads = [_reference("cd2d", t["k"], t["kt"], t["nodes"], t["parities"], t["coefs"], load)
                 for t in types if t["topology"] == "quad"]
        # the nodes of the triangles' basis are the library's own choice
        result = {t: dict.fromkeys(keys + ("info",)) for t in sorted({t["topology"] for t in types})}
        result["quad"].update({k: torch.cat([r[k].reshape(-1) for r in quads]) for k in keys})
        return result
    nodes, par, coefs, load, u = _inputs(case, seed)
    r = _reference(case["form"], case["k"], case["kt"], nodes, par, coefs, load,
                   u if call in ("gradient", "eta") else None, gradient=call == "gradient", gram=case["gram"])
    if call == "eta":
        return r["eta2"]
    if call == "recover":
        _, _, F = sizes(case["form"], "hex" if len(_shape(case)) == 3 else "quad", case["k"], case["kt"])
        x = _dev(u)
        b = r["rhs"][:, :F, None] - r["K"][:, :F, F:].contiguous() @ x[:, F:, None]
        x[:, :F] = torch.cholesky_solve(b, torch.linalg.cholesky(r["K"][:, :F, :F].contiguous()))[:, :, 0]
        return x
    keys = ("K", "rhs", "schur", "schur_rhs") + (("G",) if case["gram"] else ())
    return {k: r[k] for k in keys + (("eta2", "grad") if call == "gradient" else ())}


def _terms(form):
    """Bilinear terms (trial variable, component, test variable, test operator,
    coefficient) with operators 'v', ('d', i), ('c', i), 'div', 'n' (normal trace)
    and coefficient(c, n) of the cells' coefficients c (C, 1, .) and the normal n."""
    one, neg = lambda c, n: 1.0, lambda c, n: -1.0  # noqa: E731
    if form == "stokes2d":  # u1 u2 p s11 s12 s21 s22 | u^ t^ ; v1 v2 tau1 tau2 q
        t = []
        for i in range(2):
            t.append((i, 0, 2 + i, "div", one))
            t += [(3 + 2 * i + j, 0, 2 + i, ("c", j), one) for j in range(2)]
            t.append((7 + i, 0, 2 + i, "n", neg))
            t += [(3 + 2 * i + j, 0, i, ("d", j), one) for j in range(2)]
            t.append((2, 0, i, ("d", i), neg))
            t.append((9 + i, 0, i, "v", one))
            t.append((i, 0, 4, ("d", i), neg))
            t.append((7 + i, 0, 4, "v", lambda c, n, i=i: n[..., i]))
        return t
    dim = SPACES[form][0]
    if form.startswith("poisson"):
        return ([(0, 0, 1, "div", one), (2, 0, 1, "n", neg), (3, 0, 0, "v", one)]
                + [(1, d, 1, ("c", d), one) for d in range(dim)] + [(1, d, 0, ("d", d), neg) for d in range(dim)])
    beta = [(0, 0, 0, ("d", d), lambda c, n, d=d: -c[..., 1 + d]) for d in range(dim)]
    if form == "cdr2d":
        root = lambda c, n: torch.sqrt(c[..., 0])  # noqa: E731
        return ([(1, d, 1, ("c", d), one) for d in range(dim)] + [(1, d, 0, ("d", d), root) for d in range(dim)] + beta
                + [(0, 0, 1, "div", root), (2, 0, 1, "n", lambda c, n: -torch.sqrt(c[..., 0])), (3, 0, 0, "v", neg),
                   (0, 0, 0, "v", lambda c, n: c[..., 1 + dim])])
    return ([(1, d, 1, ("c", d), lambda c, n: 1.0 / c[..., 0]) for d in range(dim)]
            + [(1, d, 0, ("d", d), one) for d in range(dim)] + beta
            + [(0, 0, 1, "div", one), (2, 0, 1, "n", neg), (3, 0, 0, "v", one)])


def _gll(n):
    """The n + 1 Gauss-Lobatto points of degree n."""
    inner = np.polynomial.legendre.Legendre.basis(n).deriv().roots() if n > 1 else []
    return np.concatenate([[-1.0], np.sort(np.real(inner)), [1.0]])


def _lagrange(points, x):
    """Values and derivatives (len(x), len(points)) of the nodal basis at x."""
    n = len(points)
    v, d = np.ones((len(x), n)), np.zeros((len(x), n))
    for i in range(n):
        for j in range(n):
            if j == i:
                continue
            f = 1.0 / (points[i] - points[j])
            d[:, i] = d[:, i] * (x - points[j]) * f + v[:, i] * f
            v[:, i] *= (x - points[j]) * f
    return v, d


def _outer(tables):
    """(Q, n) product of per-direction tables (Q, n_d), the first direction fastest."""
    out = tables[0]
    for t in tables[1:]:
        out = (t[:, :, None] * out[:, None, :]).reshape(len(out), -1)
    return out


def _test_tables(space, dim, kt, xi):
    """(dim + 1, Q, n): value and reference gradient, or components and divergence."""
    c = [_lagrange(_gll(kt), xi[:, d]) for d in range(dim)]
    if space == "grad":
        return np.stack([_outer([v for v, _ in c])] +
                        [_outer([c[d][1 if d == e else 0] for d in range(dim)]) for e in range(dim)])
    o = [_lagrange(np.polynomial.legendre.leggauss(kt)[0], xi[:, d])[0] for d in range(dim)]
    parts = []
    for e in range(dim):
        value = _outer([c[d][0] if d == e else o[d] for d in range(dim)])
        t = np.zeros((dim + 1,) + value.shape)
        t[e], t[dim] = value, _outer([c[d][1] if d == e else o[d] for d in range(dim)])
        parts.append(t)
    return np.concatenate(parts, axis=2)


REF_VERTICES = {2: np.array([(-1, -1), (1, -1), (1, 1), (-1, 1)], float),
                3: np.array([(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1),
                             (-1, 1, 1)], float)}
SIDE_NODES = {2: [(0, 1), (1, 2), (2, 3), (3, 0)],
              3: [(0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (0, 4, 7, 3), (0, 3, 2, 1), (4, 5, 6, 7)]}


class _Points:
    """Geometry and operator values at reference points xi (Q, dim) of cells X (C, V, dim)."""

    def __init__(self, X, xi, spaces, kt):
        C, dim = X.shape[0], X.shape[2]
        ref = REF_VERTICES[dim]
        fac = 0.5 * (1.0 + ref[None] * xi[:, None, :])  # (Q, V, dim)
        dN = np.stack([0.5 * ref[:, e] * np.prod(np.delete(fac, e, axis=2), axis=2) for e in range(dim)], axis=2)
        self.x = torch.einsum("cvd,qv->cqd", X, _dev(np.prod(fac, axis=2)))
        self.J = torch.einsum("cvd,qve->cqde", X, _dev(dN))
        self.det, self.inv = torch.linalg.det(self.J), torch.linalg.inv(self.J)
        tables = {s: _dev(_test_tables(s, dim, kt, xi)) for s in set(spaces)}
        self.tables = [tables[s] for s in spaces]
        self.dim, self.shape, self.normal = dim, (C, len(xi)), None

    def op(self, var, op):
        """(C, Q, n) values of an operator on the test functions of a variable."""
        R = self.tables[var]
        if op == "v":
            return R[0].expand(self.shape[0], -1, -1)
        if op == "div":
            return R[self.dim] / self.det[..., None]
        if op == "n":
            return sum(self.normal[..., i, None] * self.op(var, ("c", i)) for i in range(self.dim))
        kind, i = op
        if kind == "d":
            return sum(self.inv[..., e, i, None] * R[1 + e] for e in range(self.dim))
        return sum((self.J[..., i, e] / self.det)[..., None] * R[e] for e in range(self.dim))


def _cells(form, k, kt, X, par, coefs, load):
    """G (C, N, N), B (C, M, N), l (C, N) of a few cells."""
    dim, trial, test = SPACES[form]
    terms = _terms(form)
    C = X.shape[0]
    N, M, F = sizes(form, "hex" if dim == 3 else "quad", k, kt)
    ntest = [(kt + 1) ** dim if s == "grad" else dim * (kt + 1) * kt ** (dim - 1) for s in test]
    toff = np.cumsum([0] + ntest)
    f64 = dict(dtype=torch.float64, device=DEV)
    cc = None if coefs is None else coefs[:, None, :]

    def rule(degree, d):
        x, w = np.polynomial.legendre.leggauss(degree // 2 + 1)
        pts = np.stack([a.reshape(-1, order="F") for a in np.meshgrid(*[x] * d, indexing="ij")], axis=1)
        return pts, np.prod(np.stack([a.reshape(-1, order="F") for a in np.meshgrid(*[w] * d, indexing="ij")]), axis=0)

    def scaled(a, values):  # coefficient (number or (C, Q) or (C, 1)) times values (C, Q, n)
        return values * (a[..., None] if torch.is_tensor(a) else a)

    # the graph norm: the test functions' adjoint values per field component, then their L2 parts
    xi, w = rule(2 * kt, dim)
    P = _Points(X, xi, test, kt)
    W = _dev(w) * P.det
    norm = {}
    for v, comp, tv, op, a in terms:
        if trial[v] in ("field", "vector"):
            norm.setdefault((v, comp), []).append((tv, op, a))
    norm = list(norm.values())
    for tv, s in enumerate(test):
        norm += [[(tv, op, lambda c, n: 1.0)] for op in (["v"] if s == "grad" else [("c", d) for d in range(dim)])]
    G = torch.zeros((C, N, N), **f64)
    for lt in norm:
        value = [None] * len(test)
        for tv, op, a in lt:
            one = scaled(a(cc, None), P.op(tv, op))
            value[tv] = one if value[tv] is None else value[tv] + one
        use = [i for i, x in enumerate(value) if x is not None]
        for i in use:
            left = (value[i] * W[..., None]).transpose(1, 2).contiguous()
            for j in use:
                block = left @ value[j].contiguous()
                G = G + torch.nn.functional.pad(block, (int(toff[j]), int(N - toff[j + 1]), int(toff[i]),
                                                        int(N - toff[i + 1])))
    # volume part of B and the load
    xi, w = rule(k + kt, dim)
    P = _Points(X, xi, test, kt)
    W = _dev(w) * P.det
    phi = _dev(_outer([_lagrange(_gll(k - 1), xi[:, d])[0] for d in range(dim)]))
    rows = [torch.zeros((C, 0, N), **f64)]

    def wide(block, tv):
        return torch.nn.functional.pad(block, (int(toff[tv]), int(N - toff[tv + 1])))

    for v, kind in enumerate(trial):
        for comp in range(dim if kind == "vector" else 1) if kind in ("field", "vector") else ():
            block = torch.zeros((C, phi.shape[1], N), **f64)
            for tv, op, a in [t[2:] for t in terms if t[:2] == (v, comp)]:
                block = block + wide((phi * W[..., None]).transpose(1, 2).contiguous()
                                     @ scaled(a(cc, None), P.op(tv, op)).contiguous(), tv)
            rows.append(block)
    ell = torch.zeros((C, N), **f64)
    for comp, (amp, waves) in enumerate(load):
        tv = comp  # the load component tests the HGRAD variable of the same number
        f = sum(float(amp[m]) * torch.prod(torch.sin(math.pi * _dev(waves[m].astype(float)) * P.x), dim=2)
                for m in range(len(amp)))
        ell = ell + torch.nn.functional.pad(torch.einsum("cq,cqn->cn", W * f, P.op(tv, "v")),
                                            (int(toff[tv]), int(N - toff[tv + 1])))
    # sides
    s, ws = rule(k + kt, dim - 1)
    bases = {"trace": _dev(_outer([_lagrange(_gll(k), s[:, d])[0] for d in range(dim - 1)])),
             "flux": _dev(_outer([_lagrange(_gll(k - 1), s[:, d])[0] for d in range(dim - 1)]))}
    side = []
    for nodes in SIDE_NODES[dim]:
        r = REF_VERTICES[dim][list(nodes)]
        if dim == 2:
            mid, tangents = r.mean(axis=0), [(r[1] - r[0]) / 2]
        else:
            mid, tangents = r.mean(axis=0), [(r[1] + r[2] - r[0] - r[3]) / 4, (r[2] + r[3] - r[0] - r[1]) / 4]
        P = _Points(X, mid + sum(s[:, a, None] * t for a, t in enumerate(tangents)), test, kt)
        t = [torch.einsum("cqde,e->cqd", P.J, _dev(x)) for x in tangents]
        n = torch.stack([t[0][..., 1], -t[0][..., 0]], dim=2) if dim == 2 else torch.linalg.cross(t[0], t[1])
        length = torch.linalg.norm(n, dim=2)
        P.normal = n / length[..., None]
        side.append((P, _dev(ws) * length))
    for v, kind in enumerate(trial):
        if kind not in bases:
            continue
        for j, (P, W) in enumerate(side):
            weight = W * par[:, j, None] if kind == "flux" else W
            block = torch.zeros((C, bases[kind].shape[1], N), **f64)
            for tv, op, a in [t[2:] for t in terms if t[0] == v]:
                block = block + wide((bases[kind] * weight[..., None]).transpose(1, 2).contiguous()
                                     @ scaled(a(cc, P.normal), P.op(tv, op)).contiguous(), tv)
            rows.append(block)
    return G, torch.cat(rows, dim=1), ell


def _reference(form, k, kt, nodes, par, coefs, load, u=None, gradient=False, gram=False):
    """K = B G^-1 B^T and rhs, the Schur complement on the trace unknowns, and with
    u the energy error r^T G^-1 r, r = l - B^T u, and its gradient in the coefficients."""
    dim = SPACES[form][0]
    N, M, F = sizes(form, "hex" if dim == 3 else "quad", k, kt)
    step = max(1, min(64, int(3e9 / (8.0 * N * (kt + 1) ** dim * 8))))
    parts = []
    for i in range(0, len(nodes), step):
        X, p = _dev(nodes[i:i + step]), _dev(par[i:i + step]).double()
        c = None if coefs is None else _dev(coefs[i:i + step]).requires_grad_(gradient)
        G, B, ell = _cells(form, k, kt, X, p, c, load)
        s = torch.rsqrt(torch.diagonal(G, dim1=1, dim2=2)).detach()
        L = torch.linalg.cholesky((s[:, :, None] * G * s[:, None, :]).detach())
        part = {}
        if u is not None:
            r = ell - (_dev(u[i:i + step])[:, None, :] @ B)[:, 0]
            y = torch.linalg.solve_triangular(L, (s * r).detach()[:, :, None], upper=False)
            part["eta2"] = y.square().sum(dim=(1, 2))
            if gradient:  # of 2 e.r - e.G e at e = G^-1 r, where it is stationary in e
                e = s * torch.linalg.solve_triangular(L.transpose(1, 2).contiguous(), y, upper=True)[:, :, 0]
                (part["grad"],) = torch.autograd.grad((2 * e * r - e * (G @ e[:, :, None])[:, :, 0]).sum(), c)
        with torch.no_grad():
            Y = torch.linalg.solve_triangular(
                L, torch.cat([(s[:, None, :] * B).transpose(1, 2), (s * ell)[:, :, None]], dim=2).contiguous(),
                upper=False)
            Yt = Y.transpose(1, 2).contiguous()
            A = Yt @ Y  # [K rhs; rhs' .]
            part["K"], part["rhs"] = A[:, :M, :M], A[:, :M, M]
            Lf = torch.linalg.cholesky(A[:, :F, :F].contiguous())
            Z = torch.linalg.solve_triangular(Lf, A[:, :F, F:].contiguous(), upper=False)
            S = A[:, F:, F:] - Z.transpose(1, 2).contiguous() @ Z
            part["schur"], part["schur_rhs"] = S[:, :M - F, :M - F], S[:, :M - F, M - F]
            if gram:
                part["G"] = G
        parts.append({key: x.detach() for key, x in part.items()})
    return {key: torch.cat([q[key] for q in parts]) for key in parts[0]}
