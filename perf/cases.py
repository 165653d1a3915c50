"""The work that a user of fem_2d_amd has it do, as cases whose time can be measured.

A program that uses the framework refines a Mesh, turns it into a Domain, assembles the
Galerkin eigenproblem (GEP) of that Domain, solves it for one eigenpair and evaluates the
fields of the eigenvector. The cases cover each of these steps through the entry points that
such a program calls, on the workload families of ``fem_2d_amd.workloads``, from about a
thousand DoFs to 1.8 million.
"""

from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import fem_2d_amd as F
from fem_2d_amd import _native as N
from fem_2d_amd import workloads as W

BASES = {"hier": F.HierPoly, "kol": F.KOLShapeFn}
PRECISIONS = {"f64": F.FP64, "f32": F.FP32, "f32r": F.FP32R}
ENTRY_BYTES = {"f64": 20, "f32": 12, "f32r": 16}


def listed():
    return [
        # The smallest call in use: the 1 096-DoF waveguide that the documentation and the
        # tests start from, assembled again and again (a sweep over Gauss points or bases).
        dict(name="assemble_small", kind="assemble", mesh="small", order=4, glq=8, basis="hier", precision="f64"),
        # Few Elems of high order, stored in FP32 plus residual: the precision study.
        dict(name="assemble_precision", kind="assemble", mesh="small", order=8, glq=12, basis="hier",
             precision="f32r"),
        # The benchmark: a 64 x 32 waveguide, orders (6, 6), two levels of refinement on a
        # random quarter of the leaves (445 380 DoFs).
        dict(name="assemble_waveguide", kind="assemble", mesh="waveguide", nx=64, ny=32, order=6, glq=8, basis="hier",
             precision="f64"),
        # The same with the values stored in FP32 (a preconditioner's matrices).
        dict(name="assemble_waveguide_f32", kind="assemble", mesh="waveguide", nx=64, ny=32, order=6, glq=8,
             basis="hier", precision="f32"),
        # The largest: anisotropic orders 1..8 per Elem, three levels of T / U / V refinement,
        # the Legendre space (1.8 M DoFs): the mesh an hp-adaptive run ends with.
        dict(name="assemble_hp", kind="assemble", mesh="hp", nx=128, ny=64, glq=10, basis="kol", precision="f64"),
        # 256 independent guides of random sizes and orders in one Mesh: a design sweep.
        dict(name="assemble_many", kind="assemble", mesh="many", count=256, glq=8, basis="hier", precision="f64"),
        # One step of an adaptive loop: the Mesh was just refined, its Domain is built on the
        # GPU and assembled once (the next step has another Mesh).
        dict(name="adaptive_step", kind="adaptive", mesh="hp", nx=32, ny=16, glq=10, basis="kol", precision="f64"),
        # The drop-in call on host data: Domain in, GEP out, as a host solver wants it.
        dict(name="drop_in", kind="drop_in", mesh="waveguide", nx=16, ny=8, order=5, glq=8, basis="hier",
             precision="f64"),
        # The x and y fields of a solution on a 12 x 12 grid over every leaf (plots, error
        # indicators), Domain, solution and fields in HBM.
        dict(name="fields", kind="fields", mesh="waveguide", nx=64, ny=32, order=6, density=12, basis="hier"),
        # slepc_solve_gep near the lowest cutoff, as it runs on a small GEP (dense) ...
        dict(name="solve_dense", kind="solve", mesh="small", order=4, glq=8, basis="hier", target=10.0),
        # ... and on a larger one (sparse).
        dict(name="solve_sparse", kind="solve", mesh="hp", nx=12, ny=6, glq=10, basis="kol", target=5.0),
    ]


def draw(rng):
    """One more case of the same ranges."""

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["assemble"] * 6 + ["adaptive", "drop_in", "fields", "solve"])
    case = dict(kind=kind, basis=rng.choice(["hier", "kol"]))
    if kind == "solve":
        if rng.random() < 0.5:
            return dict(case, mesh="small", order=rng.randint(3, 5), glq=8, target=round(rng.uniform(8.0, 12.0), 2))
        nx = rng.randint(5, 12)
        return dict(case, mesh="hp", nx=nx, ny=max(2, nx // 2), glq=10, target=5.0, layout=rng.randrange(1000))
    mesh = rng.choice(["small", "waveguide", "hp", "many"]) if kind == "assemble" else rng.choice(["waveguide", "hp"])
    case["mesh"] = mesh
    if mesh != "small":
        case["layout"] = rng.randrange(1000)
    top = {"assemble": 64, "adaptive": 40, "drop_in": 24, "fields": 64}[kind]
    if mesh == "small":
        case["order"] = rng.randint(2, 8)
    elif mesh == "waveguide":
        nx = log_int(4, top)
        case.update(nx=nx, ny=max(1, nx // rng.choice([1, 2, 2, 3])), order=rng.randint(2, 7))
    elif mesh == "hp":
        nx = log_int(4, 2 * top if kind == "assemble" else top)
        case.update(nx=nx, ny=max(1, nx // rng.choice([2, 2, 3])))
    else:
        case["count"] = log_int(4, 256)
    if kind == "fields":
        return dict(case, density=rng.randint(3, 16))
    return dict(case, glq=rng.choice([8, 9, 10, 12]), precision=rng.choice(["f64", "f64", "f32", "f32r"]))


def _filling(elements, kind, seed):
    """Per element (eps_r, mu_r): air in the guides that are solved for a cutoff, a dielectric
    drawn from the seed elsewhere."""
    mats = np.tile([1.0, 0.0, 1.0, 0.0], (elements, 1))
    if kind != "solve":
        r = np.random.default_rng(seed)
        mats[:, 0] += 2.0 * r.random(elements)
        mats[:, 2] += 0.2 * r.random(elements)
    return mats


def _guide(nx, ny, x0, width, height, first=0):
    """Points and the elements' corner ids of one nx-by-ny guide."""
    px, py = np.meshgrid(np.linspace(x0, x0 + width, nx + 1), np.linspace(0.0, height, ny + 1))
    i, j = np.meshgrid(np.arange(nx), np.arange(ny))
    low = (first + j * (nx + 1) + i).reshape(-1, 1)
    return np.stack([px.ravel(), py.ravel()], 1), low + np.array([0, 1, nx + 1, nx + 2])


def _refine(mesh, rng, levels, pick):
    for _ in range(levels):
        leaves = [e for e in range(mesh.num_elems) if mesh.elem_is_h_refineable(e)]
        picked = [(e, pick(rng.uniform())) for e in leaves]
        mesh.execute_h_refinements([(e, h) for e, h in picked if h is not None])


def _mesh(case, seed):
    """The case's Mesh: its refinement and orders are the case's (the families of
    fem_2d_amd.workloads, with their own seeds), its size and filling the seed's."""
    kind, r = case["mesh"], np.random.default_rng(seed)
    width, height = 1.0 + 0.25 * r.random(), 0.5 + 0.1 * r.random()
    rng = W.SplitMix64(case.get("layout", {"waveguide": 0, "hp": 1, "many": 2}.get(kind, 0)))
    if kind == "many":
        points, corners, orders, x0 = [], [], [], 0.0
        for _ in range(case["count"]):
            a, nx = 1.0 + rng.uniform(), rng.randint(4, 16)
            p = rng.randint(2, 6)
            pts, ids = _guide(nx, nx // 2, x0, a * width, height, sum(map(len, points)))
            points.append(pts)
            corners.append(ids)
            orders += [F.Orders(p, p)] * len(ids)
            x0 += a * width + 0.5
        points, corners = np.concatenate(points), np.concatenate(corners)
    else:
        nx, ny = (4, 2) if kind == "small" else (case["nx"], case["ny"])
        points, corners = _guide(nx, ny, 0.0, 2.0 * width if kind == "hp" else width,
                                 2.0 * height if kind == "hp" else height)
        if kind == "hp":
            orders = [F.Orders(rng.randint(1, 8), rng.randint(1, 8)) for _ in range(nx * ny)]
        else:
            orders = [F.Orders(case["order"], case["order"])] * (nx * ny)
    mesh = F.Mesh.from_parts(points, corners.astype(np.int32), _filling(len(corners), case["kind"], seed))
    mesh.set_expansion_orders(list(enumerate(orders)))
    if kind == "small":
        mesh.global_h_refinement(F.HRef.T)
        centre = 7  # the middle node of the coarse grid
        mesh.h_refine_with_filter(lambda e: F.HRef.u() if centre in e.nodes else None)
    elif kind == "waveguide":
        _refine(mesh, rng, 2, lambda u: F.HRef.T if u < 0.25 else None)
    elif kind == "many":
        _refine(mesh, rng, 1, lambda u: F.HRef.T if u < 0.3 else None)
    else:
        _refine(mesh, rng, 3, lambda u: F.HRef.T if u < 0.2 else F.HRef.u() if u < 0.3 else
                F.HRef.v() if u < 0.4 else None)
    return mesh


class _Span:
    """Device memory of a context as torch takes it in. The tensor made of it keeps this object,
    and so the context whose buffers it shows, alive."""

    def __init__(self, ctx, ptr, count, typestr):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "version": 3,
                                         "data": (C.cast(ptr, C.c_void_p).value, False)}


def _views(ctx, g, precision):
    """A device GEP's arrays as tensors."""

    def tensor(ptr, count, typestr):
        return torch.as_tensor(_Span(ctx, ptr, count, typestr), device="cuda")

    out = {"row_ptr": tensor(g.row_ptr, g.n + 1, "<i8"), "col": tensor(g.col, g.nnz, "<i4")}
    if precision == "f64":
        out["a"], out["b"] = tensor(g.a_val, g.nnz, "<f8"), tensor(g.b_val, g.nnz, "<f8")
    else:
        out["a"], out["b"] = tensor(g.a_val32, g.nnz, "<f4"), tensor(g.b_val32, g.nnz, "<f4")
    if precision == "f32r":
        out["res"] = tensor(g.res16, g.nnz, "<i4")
    return out


class _Assemble:
    """A Domain in HBM, assembled again and again on a context of its own."""

    def __init__(self, case, seed):
        self.ctx = F.Context(0)
        self.dd = F.DeviceDomain.from_mesh(_mesh(case, seed), ctx=self.ctx)
        self.precision = case["precision"]
        self.step = self.dd.assembler((case["glq"], case["glq"]), BASES[case["basis"]],
                                      precision=PRECISIONS[self.precision])
        self.at, self.views = None, None

    def run(self):
        g = self.step()
        # the arrays stay where they are while they are large enough
        at = bytes(g)[:N.GepDevice.generation.offset]
        if at != self.at:
            self.at, self.views = at, _views(self.ctx, g, self.precision)
        return self.views


class _Adaptive:
    def __init__(self, case, seed):
        self.ctx = F.Context(0)
        self.mesh = _mesh(case, seed)
        self.glq, self.basis, self.precision = (case["glq"],) * 2, BASES[case["basis"]], case["precision"]

    def run(self):
        dd = F.DeviceDomain.from_mesh(self.mesh, ctx=self.ctx)
        return _views(self.ctx, dd.assemble(self.glq, self.basis, precision=PRECISIONS[self.precision]), self.precision)


class _DropIn:
    def __init__(self, case, seed):
        self.ctx = F.Context(0)
        self.domain = F.Domain.from_mesh(_mesh(case, seed))
        self.domain.view()
        self.glq, self.basis, self.precision = (case["glq"],) * 2, BASES[case["basis"]], case["precision"]

    def run(self):
        g = F.galerkin_sample_gep_hcurl(self.domain, self.glq, self.basis, ctx=self.ctx,
                                        precision=PRECISIONS[self.precision])
        return {"row_ptr": g.row_ptr, "col": g.col, "a": g.a_val, "b": g.b_val}


class _Fields:
    def __init__(self, case, seed):
        self.ctx = F.Context(0)
        self.dd = F.DeviceDomain.from_mesh(_mesh(case, seed), ctx=self.ctx)
        n = C.c_int64()
        self.lib = N.load()
        F.errors.check(self.lib.fem2d_device_domain_num_leaves(self.dd._h, C.byref(n)))
        self.d, self.basis = case["density"], BASES[case["basis"]].code
        self.solution = torch.from_numpy(_solution(self.dd.n_dofs, seed)).cuda()
        self.x = torch.empty((n.value, self.d, self.d), dtype=torch.float64, device="cuda")
        self.y = torch.empty_like(self.x)

    def run(self):
        F.errors.check(self.lib.fem2d_device_xy_fields(
            self.ctx._h, self.dd._h, self.basis, self.d, self.d, self.solution.data_ptr(), self.solution.numel(),
            self.x.data_ptr(), self.y.data_ptr()))
        return {"x": self.x, "y": self.y}


class _Solve:
    def __init__(self, case, seed):
        self.ctx = F.Context(0)
        self.dd = F.DeviceDomain.from_mesh(_mesh(case, seed), ctx=self.ctx)
        self.gep = self.dd.assemble((case["glq"],) * 2, BASES[case["basis"]])
        self.target = case["target"]

    def run(self):
        pair = F.slepc_solve_gep(self.gep, self.target, ctx=self.ctx)
        return {"value": pair.value, "vector": pair.vector}


_KINDS = {"assemble": _Assemble, "adaptive": _Adaptive, "drop_in": _DropIn, "fields": _Fields, "solve": _Solve}


def _solution(n, seed):
    return np.random.default_rng(seed).standard_normal(n)


def prepare(case, seed):
    state = _KINDS[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return state.run()


def work(case):
    """Inputs read once, outputs written once. A Domain is its view's arrays: 54 bytes an Elem
    (parent, location, box, materials, offset) and 7 a basis spec."""
    a = F.Domain.from_mesh(_mesh(case, 0)).arrays()
    n, specs, elems = a["n_dofs"], a["bs_dof"].size, a["n_elems"]
    domain = 54 * elems + 7 * specs
    if case["kind"] == "fields":
        leaves = elems - np.unique(a["parent"][a["parent"] >= 0]).size
        points = leaves * case["density"] ** 2
        return {"bytes": domain + 8 * n + 16 * points, "flops": 8.0 * case["density"] ** 2 * _nested_specs(a)}
    pairs = _pairs(a)
    if case["kind"] == "solve":
        # a dense solve: the two factorisations; a sparse one: the matrices are read
        return {"bytes": 20 * pairs, "flops": 1.0 * n ** 3 if n <= F.linalg.SLEPC_DENSE_LIMIT else 0.0}
    entry = 20 if case["kind"] == "drop_in" else ENTRY_BYTES[case["precision"]]
    return {"bytes": domain + 8 * n + entry * pairs, "flops": 6.0 * pairs}


def _chain(parent, e):
    while e >= 0:
        yield e
        e = parent[e]


def _nested_specs(a):
    """Specs of every leaf and its ancestors, summed over the leaves."""
    parent, count = a["parent"], np.diff(a["bs_offsets"])
    inner = np.zeros(a["n_elems"], bool)
    inner[parent[parent >= 0]] = True
    return int(sum(count[x] for e in np.flatnonzero(~inner) for x in _chain(parent, e)))


def _pairs(a):
    """Pairs of basis specs of one Elem or of an Elem and its ancestor: the terms of the GEP
    (a few per cent of its entries have two)."""
    parent, count = a["parent"], np.diff(a["bs_offsets"])
    total = 0
    for e in range(a["n_elems"]):
        k = int(count[e])
        total += k * (k + 1) // 2 + k * sum(int(count[x]) for x in _chain(parent, e) if x != e)
    return total


# -- the same results in 64 bits, from the Domain's lists alone ---------------------------------


def _shapes(basis, orders, x):
    """N, N', T, T' of orders 0..orders-1 at the points x: arrays [4][orders][points]."""
    out = np.zeros((4, orders, x.size))
    legendre = np.polynomial.legendre
    norms = {2: 0.968246, 3: 2.561738, 4: 0.838525, 5: 4.248161, 6: 0.816397, 7: 5.882766, 8: 0.808509}
    for n in range(orders):
        if basis == "hier":
            f, df = x ** n, n * x ** max(n - 1, 0)
            bubble, dbubble = (f - 1.0, df) if n % 2 == 0 else (f - x, df - 1.0)
        else:
            c = np.zeros(n + 1)
            c[n] = 1.0
            f, df = legendre.legval(x, c), legendre.legval(x, legendre.legder(c))
            if n >= 2:
                # T_n = c_n (L_n - L'_(n-1) / (n (n - 1) / 2))
                low = np.zeros(n)
                low[n - 1] = 1.0
                t = np.append(np.zeros(n), 1.0)
                d = legendre.legder(low) / (n * (n - 1) / 2)
                t[:d.size] -= d
                t *= norms.get(n, 1.0)
                bubble, dbubble = legendre.legval(x, t), legendre.legval(x, legendre.legder(t))
        out[0, n], out[1, n] = f, df
        if n == 0:
            out[2, n], out[3, n] = 1.0 - x, -1.0
        elif n == 1:
            out[2, n], out[3, n] = 1.0 + x, 1.0
        else:
            out[2, n], out[3, n] = bubble, dbubble
    return out


def _places(a):
    """Per Elem its place inside its base Elem, (halvings, index) per axis, and its half extents."""
    place = np.zeros((a["n_elems"], 4), np.int64)
    half = np.zeros((a["n_elems"], 2))
    for e in range(a["n_elems"]):
        p = a["parent"][e]
        if p >= 0:
            loc = int(a["loc"][e])  # SW SE NW NE W E S N
            du, iu, dv, iv = place[p]
            if loc < 6:
                du, iu = du + 1, 2 * iu + (loc in (1, 3, 5))
            if loc < 4 or loc >= 6:
                dv, iv = dv + 1, 2 * iv + (loc in (2, 3, 7))
            place[e] = du, iu, dv, iv
        x0, y0, x1, y1 = a["element_box"][e]
        half[e] = (x1 - x0) / 2.0 / 2.0 ** place[e][0], (y1 - y0) / 2.0 / 2.0 ** place[e][2]
    return place, half


def _inside(place, axis, e, anc):
    """(scale, offset) that take a coordinate of Elem e to its ancestor's, on one axis."""
    d = int(place[e][2 * axis] - place[anc][2 * axis])
    i = int(place[e][2 * axis + 1] - (place[anc][2 * axis + 1] << d))
    s = 0.5 ** d
    return s, -1.0 + (2 * i + 1) * s


def _exact_gep(a, basis, glq):
    place, half = _places(a)
    orders = int(max(a["bs_i"].max(), a["bs_j"].max())) + 1
    x, w = np.polynomial.legendre.leggauss(glq)
    own = _shapes(basis, orders, x)
    grams = {}

    def gram(s, c):
        # [4][4][orders][orders]: the ancestor's function at the mapped points, the Elem's at its own
        if (s, c) not in grams:
            grams[s, c] = np.einsum("fam,gbm->fgab", _shapes(basis, orders, s * x + c) * w, own)
        return grams[s, c]

    off, n = a["bs_offsets"], a["n_dofs"]
    keys, va, vb = [], [], []
    for e in range(a["n_elems"]):
        q = slice(off[e], off[e + 1])
        qd, qi, qj = (a[k][q].astype(np.int64) for k in ("bs_dir", "bs_i", "bs_j"))
        for p_elem in _chain(a["parent"], e):
            p = slice(off[p_elem], off[p_elem + 1])
            pd, pi, pj = (a[k][p].astype(np.int64)[:, None] for k in ("bs_dir", "bs_i", "bs_j"))
            (su, cu), (sv, cv) = (_inside(place, ax, e, p_elem) for ax in (0, 1))
            gx, gy = gram(su, cu), gram(sv, cv)
            eps, mu = a["materials"][p_elem]
            (ap, bp), (aq, bq) = half[p_elem], half[e]
            big = half[p_elem] if ap * bp >= aq * bq else half[e]
            same = pd == qd
            # the curl of a U spec is -N_i(x) T'_j(y) / a, of a V spec T'_i(x) N_j(y) / b
            scale = np.where(pd == 0, -1.0 / ap, 1.0 / bp) * np.where(qd == 0, -su / aq, sv / bq) / mu
            scale = scale * np.where(same, np.where(pd == 0, big[0] / big[1], big[1] / big[0]), 1.0)
            cc = scale * gx[3 * pd, 3 * qd, pi, qi] * gy[3 * (1 - pd), 3 * (1 - qd), pj, qj]
            s2 = eps * su * sv * max(ap * bp, aq * bq) * np.where(pd == 0, 1.0 / (ap * aq), 1.0 / (bp * bq))
            l2 = np.where(same, s2 * gx[2 * pd, 2 * qd, pi, qi] * gy[2 * (1 - pd), 2 * (1 - qd), pj, qj], 0.0)
            r, c = np.broadcast_arrays(a["bs_dof"][p].astype(np.int64)[:, None], a["bs_dof"][q].astype(np.int64))
            take = np.triu(np.ones(r.shape, bool)) if p_elem == e else np.ones(r.shape, bool)
            keys.append((np.minimum(r, c) * n + np.maximum(r, c))[take])
            va.append(cc[take])
            vb.append(l2[take])
    keys, va, vb = np.concatenate(keys), np.concatenate(va), np.concatenate(vb)
    order = np.argsort(keys, kind="stable")
    keys = keys[order]
    first = np.flatnonzero(np.concatenate([[True], keys[1:] != keys[:-1]]))
    return keys[first] // n, keys[first] % n, np.add.reduceat(va[order], first), np.add.reduceat(vb[order], first)


def _exact_fields(a, basis, density, solution):
    place, half = _places(a)
    orders = int(max(a["bs_i"].max(), a["bs_j"].max())) + 1
    grid = -1.0 + 2.0 * np.arange(density) / (density - 1)
    shapes = {}

    def at(s, c):
        if (s, c) not in shapes:
            shapes[s, c] = _shapes(basis, orders, s * grid + c)
        return shapes[s, c]

    off = a["bs_offsets"]
    inner = np.zeros(a["n_elems"], bool)
    inner[a["parent"][a["parent"] >= 0]] = True
    xs, ys = [], []
    for e in np.flatnonzero(~inner):
        fx, fy = np.zeros((density, density)), np.zeros((density, density))
        for p in _chain(a["parent"], e):
            u, v = at(*_inside(place, 0, e, p)), at(*_inside(place, 1, e, p))
            t = slice(off[p], off[p + 1])
            d, i, j = a["bs_dir"][t], a["bs_i"][t], a["bs_j"][t]
            s = solution[a["bs_dof"][t]]
            k = d == 0
            fx += (u[0][i[k]] * (s[k] / half[p][0])[:, None]).T @ v[2][j[k]]
            k = d == 1
            fy += (u[2][i[k]] * (s[k] / half[p][1])[:, None]).T @ v[0][j[k]]
        xs.append(fx)
        ys.append(fy)
    return np.array(xs), np.array(ys)


def exact(case, seed):
    kind = case["kind"]
    # the largest would take minutes here
    if case["mesh"] == "hp" and case["nx"] > 64 or case["mesh"] == "many" and case["count"] > 160:
        return None
    if kind == "solve" and case["mesh"] == "hp":
        return None
    a = F.Domain.from_mesh(_mesh(case, seed)).arrays()
    if kind == "fields":
        x, y = _exact_fields(a, case["basis"], case["density"], _solution(a["n_dofs"], seed))
        return {"x": x, "y": y}
    rows, cols, va, vb = _exact_gep(a, case["basis"], case["glq"])
    if kind == "solve":
        m = np.zeros((2, a["n_dofs"], a["n_dofs"]))
        for k, v in enumerate((va, vb)):
            m[k, rows, cols] = m[k, cols, rows] = v
        low = np.linalg.cholesky(m[1])
        half = np.linalg.solve(low, m[0])
        values = np.linalg.eigvalsh(np.linalg.solve(low, half.T))
        # the sign of an eigenvector is free
        return {"value": float(values[np.argmin(np.abs(values - case["target"]))]), "vector": None}
    out = {"row_ptr": None, "col": None, "a": va, "b": vb}
    if case.get("precision") == "f32r" and kind != "drop_in":
        out["res"] = None
    return out
